// Walks every shape that the exhaustive matcher is launched for (window,
// patch, patch frames, scheduled frames, channels, cap; both kinds of search)
// and checks that its LDS allocation covers what the chosen kernel touches.
// Prints the shapes that take narrow rows, unguided and guided, by patch size.
#include "match_layout.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>

using namespace vnlbhip;

namespace {

void fail(const char* what, const StageDesc& d, bool guided) {
    std::printf("%s: patch %d x %d, window %d, %d scheduled frames, %d channels, cap %d, guided %d\n", what, d.patch,
                d.patch_time, d.search_window, d.search_bwd + d.search_fwd + 1, d.channels, d.cap, guided);
    std::exit(1);
}

// Last word of the region that a pair of candidate rows reads, as the kernel
// addresses it: the last plane, the last pair of rows, the last group of four
// candidates; wide rows are read in fours.
long long last_read(const StageDesc& d, bool guided, bool wide) {
    const int side = d.search_window + d.patch - 1;
    const int temporal = d.search_bwd + d.search_fwd + 1;
    const long long planes = guided ? temporal * d.patch_time : temporal + d.patch_time - 1;
    const int pitch = region_pitch(d.search_window, d.patch, wide);
    const int row = (d.search_window + 1) / 2 * 2 - 2 + d.patch;  // the second row's last patch row
    const int column = (d.search_window + 3) / 4 * 4 - 4 + (wide ? (d.patch + 6) / 4 * 4 : d.patch + 3) - 1;
    return (planes - 1) * side * pitch + static_cast<long long>(row) * pitch + column;
}

}  // namespace

int main() {
    constexpr size_t kStatic = 2048;  // match_kernel's static arrays, rounded up
    long long narrow[2][kMaxPatch + 1] = {};
    long long shapes = 0;
    double widest = 0.0;
    StageDesc d{};
    for (int channels = 1; channels <= 3; channels += 2) {
        for (int patch = 1; patch <= kMaxPatch; ++patch) {
            for (int frames = 1; frames <= kMaxFrames && channels * frames * patch * patch <= kMaxDim; ++frames) {
                for (int window = 1; window * window <= kMaxCandidates; window += 2) {
                    // Either radius is at most the frames in device memory less the patch's.
                    const int scheduled = std::min(kMaxTemporal, 2 * (kMaxFrames - frames) + 1);
                    for (int temporal = 1; temporal <= scheduled; ++temporal) {
                        if (window * window * temporal > kMaxCandidates) {
                            break;
                        }
                        for (int cap = kMatchThreads; cap <= kMaxCap; cap += 64) {
                            d.channels = channels;
                            d.patch = patch;
                            d.patch_time = frames;
                            d.dim = channels * frames * patch * patch;
                            d.search_window = window;
                            d.search_bwd = temporal - 1;
                            d.cap = cap;
                            const size_t others =
                                sizeof(float) * (window_candidates(d) + 3ULL * selection_entries(d));
                            for (int guided = 0; guided < 2; ++guided) {
                                const size_t budget = guided ? kGuidedMatchBudget : kMatchBudget;
                                const size_t counted =
                                    others + sizeof(float) * region_floats(window, patch, temporal, frames, guided);
                                if (counted > budget) {
                                    continue;
                                }
                                ++shapes;
                                const bool wide = match_wide_rows(d, guided);
                                const MatchLayout L = match_layout(d, patch, guided, wide);
                                if (L.words * sizeof(float) + kStatic > 160 * 1024) {
                                    fail("allocation past the LDS", d, guided);
                                }
                                if (last_read(d, guided, wide) >= L.dist || L.sel < L.dist + window_candidates(d) ||
                                    L.ref < L.sel + 3 * selection_entries(d) || L.words < L.ref + d.dim) {
                                    fail("arrays overlap", d, guided);
                                }
                                if (wide && (L.dist % 4 != 0 || region_pitch(window, patch, true) % 4 != 0)) {
                                    fail("wide rows off their alignment", d, guided);
                                }
                                const int pitch = region_pitch(window, patch, true);
                                widest = std::max(widest, pitch / double(region_pitch(window, patch, false)));
                                if (!wide) {
                                    ++narrow[guided][patch];
                                    if (!guided && !narrow_unguided_patch(patch)) {
                                        fail("no kernel for narrow rows", d, guided);
                                    }
                                }
                            }
                        }
                    }
                }
            }
        }
    }
    std::printf("%lld shapes, wide rows at most %.2f times the narrow ones\n", shapes, widest);
    for (int guided = 0; guided < 2; ++guided) {
        for (int patch = 1; patch <= kMaxPatch; ++patch) {
            if (narrow[guided][patch] > 0) {
                std::printf("%s %d: %lld\n", guided ? "guided" : "unguided", patch, narrow[guided][patch]);
            }
        }
    }
    return 0;
}
