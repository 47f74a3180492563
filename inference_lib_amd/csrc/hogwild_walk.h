// The way of one workgroup of a launch in whole row groups and runs (KH_STREAM), for the kernel and for the check of it on the CPU.
#pragma once

#ifdef __HIPCC__
#define HW_BOTH __host__ __device__ __forceinline__
#else
#define HW_BOTH inline
#endif

namespace hw {

struct Walk {
    int begin, end;      // the workgroup's run: tiles, counted through the row groups 0 .. split - 1
    int tiles;           // tiles of a row group
    int split, groups;   // row groups split .. groups - 1 are dealt whole, every wgs-th to one workgroup
    int wgs;
};

// Workgroup g: does it begin with a whole row group?  The first one it opens, if any.
HW_BOTH bool walk_whole(const Walk& w, int g) { return w.split + g < w.groups; }
HW_BOTH int walk_first(const Walk& w, int g) { return walk_whole(w, g) ? w.split + g : w.begin / w.tiles; }
// Whether it opens any: the first row group of an empty run may lie behind the last one there is.
HW_BOTH bool walk_opens(const Walk& w, bool whole) { return whole || w.begin < w.end; }
// Its tiles of row group `group`.
HW_BOTH int walk_from(const Walk& w, bool whole, int group) {
    const int t = whole ? 0 : w.begin - group * w.tiles;
    return t > 0 ? t : 0;
}
HW_BOTH int walk_to(const Walk& w, bool whole, int group) {
    const int t = whole ? w.tiles : w.end - group * w.tiles;
    return t < w.tiles ? t : w.tiles;
}
// The row group behind `group`, or -1; below w.split it is part of the run.
HW_BOTH int walk_next(const Walk& w, bool whole, int group) {
    const int next = whole ? group + w.wgs : group + 1;
    if (whole && next < w.groups) return next;
    const int run = whole ? w.begin / w.tiles : next;
    const int from = w.begin > run * w.tiles ? w.begin : run * w.tiles;
    return from < w.end ? run : -1;
}

}  // namespace hw
