// LDS layout of the exhaustive matchers, one description for the kernels, the
// launches and the limits (plain functions of StageDesc, host and device).
#pragma once

#include "common.h"

namespace vnlbhip {

constexpr int kMatchThreads = 256;

// Dynamic LDS of match_kernel: 160 KB less its static arrays (1.6 KB) and
// room to spare.  Stages whose narrow rows, candidate distances and
// selection scratch exceed kMatchBudget / kGuidedMatchBudget are refused.
constexpr size_t kMatchLds = 156 * 1024;
constexpr size_t kMatchBudget = 108 * 1024;
constexpr size_t kGuidedMatchBudget = 152 * 1024;

// Unguided: the scheduled frames share one window, frames t_low ..
// t_high + Pt - 1.  Guided: every scheduled frame has its own window, so
// each (frame, patch frame) pair has its own plane.
__host__ __device__ inline int region_floats(int window, int patch, int temporal, int patch_time,
                                             bool guided) {
    const int side = window + patch - 1;
    return (guided ? temporal * patch_time : temporal + patch_time - 1) * side * side + 8;
}

// The exhaustive matcher's region: wide rows of a 16-byte multiple that hold
// the four samples past the last group of four candidates, or rows as narrow
// as region_floats has them; and one row more (the second of a pair of
// candidate rows may lie past the window).
__host__ __device__ inline int region_pitch(int window, int patch, bool wide) {
    return wide ? (window + 3) / 4 * 4 + (patch + 3 + 3) / 4 * 4 - 4 : window + patch - 1;
}
__host__ __device__ inline int match_region_floats(int window, int patch, int temporal, int patch_time, bool guided,
                                                   bool wide) {
    const int rows = (guided ? temporal * patch_time : temporal + patch_time - 1) * (window + patch - 1);
    return wide ? ((rows + 1) * region_pitch(window, patch, true) + 3) / 4 * 4
                : region_floats(window, patch, temporal, patch_time, guided) + window + patch - 1;
}

// Candidate distances of a full window: window^2 per scheduled frame.
__host__ __device__ inline int window_candidates(const StageDesc& d) {
    return d.search_window * d.search_window * (d.search_bwd + d.search_fwd + 1);
}

// Entries of each of the three selection arrays after the distances: the
// selected list (at most the cap) and the short path's candidate list (at
// most one per thread).
__host__ __device__ inline int selection_entries(const StageDesc& d) {
    return d.cap > kMatchThreads ? d.cap : kMatchThreads;
}

// match_kernel's dynamic LDS, in words from its start (the region is at 0).
struct MatchLayout {
    int dist;   // candidate distances
    int sel;    // three selection arrays
    int ref;    // the reference patch (16-byte aligned)
    int words;
};

__host__ __device__ inline MatchLayout match_layout(const StageDesc& d, int patch, bool guided, bool wide) {
    MatchLayout L{};
    L.dist = match_region_floats(d.search_window, patch, d.search_bwd + d.search_fwd + 1, d.patch_time, guided, wide);
    L.sel = L.dist + window_candidates(d);
    L.ref = (L.sel + 3 * selection_entries(d) + 3) / 4 * 4;
    L.words = L.ref + d.dim;
    return L;
}

// Wide rows wherever they fit the LDS, else narrow ones.  For small patches and
// windows a wide row takes several times a narrow one (16 floats for 10 with
// 2x2 patches in 9x9 windows), so long patches or many scheduled frames may
// not fit within the budgets above: unguided only 2x2 patches in 9x9 windows,
// from 138 patch frames on.
__host__ __device__ inline bool match_wide_rows(const StageDesc& d, bool guided) {
    return match_layout(d, d.patch, guided, true).words * sizeof(float) <= kMatchLds;
}

// Whether a thread takes two candidate rows: where one row each (four
// candidates) would fill the workgroup more than once.  Every anchor's window
// is shifted inside the clip, so all have the same size.  Measured with one
// and with two rows (8x8 patches of a 200x150 grey clip, matching of both
// stages): 15x15x3 windows, 180 threads of one row, 0.350 and 0.387 ms;
// 19x19x3, 285, 0.384 and 0.374 ms; 21x21x3, 378, 0.441 and 0.388 ms; 25x25x5,
// 875, 1.109 and 0.991 ms.
__host__ __device__ inline bool match_paired_rows(const StageDesc& d) {
    const auto least = [](int a, int b) { return a < b ? a : b; };
    const int nx = least(d.search_window, d.width - d.patch + 1);
    const int ny = least(d.search_window, d.height - d.patch + 1);
    const int nt = least(d.search_bwd + d.search_fwd + 1, d.total_frames - d.patch_time + 1);
    return nt * ny * ((nx + 3) / 4) > kMatchThreads;
}

// Patches whose unguided stages within kMatchBudget may need narrow rows: the
// only ones match_kernel is built for them.
constexpr bool narrow_unguided_patch(int patch) { return patch == 2; }

}  // namespace vnlbhip
