// Filter stage of a group: dual-basis map, Wiener coefficients, aggregation
// weights, reconstruction and the weighted scatter of every sample into the
// per-output-frame double accumulators.
//
// Semantics follow the reference's filter path (src/core/core.cpp:184-871,
// src/linalg/linalg.cpp:153-595) with the 16-lane summation order of the CPU
// restatement: a dot product is 16 lane-wise fma chains over the vector part
// of the row, a halving tree over the lanes, then the scalar tail in order.
//
// Slot layout.  Lane l of a 16-lane team owns the elements e = 16 k + l of a
// model row: slots k < chunks are the vector part, slot k == chunks (lanes
// l < tail) the scalar tail.  Per-element tables, the group means and the
// basis live in LDS per lane with a padded pitch, so a lane reads its slots
// with 128-bit loads and the 16 lanes of a team hit distinct banks; the four
// teams of a wavefront read the same basis words (broadcast).  Sample rows
// never go through LDS: a team loads its row straight into registers.
//
// Workgroups are persistent: each builds the stage-constant tables once and
// then walks the groups with a stride coprime with their count, so that
// concurrently running groups scatter into distant parts of the clip.
//
// Aggregation.  The GPU executes about 20 G memory-side atomic operations per
// second and 64-byte line touched; a patch row of 8 doubles touches two lines
// as often as one, and adding each sample's rows straight into the
// accumulators (2 k line operations per 16-sample group of a YUV clip) took
// the kernel exactly that long.  A group's patches overlap, so for 8x8
// patches (kTile) its workgroup first adds them up in an LDS tile of doubles
// and flushes each touched cell once, 8 rows x 8 line-aligned pixels per
// wavefront instruction.  The addends are floats and the sums doubles as
// before.  What bounds the rest is the latency of a group's phases (vector
// units 45 % busy at three workgroups per compute unit), so loads are issued
// in batches and basis rows are taken in pairs.  Measured against per-sample
// atomics, a load at a time: 188 k groups of 16 YUV samples, rank 16, 18.4 ->
// 10.7 ms (15.3 with the tile alone), 50 k grey ones 2.29 -> 1.27 ms.
#include "common.h"
#include "device_util.h"
#include "group.h"
#include "kernels.h"

#include <float.h>

#include <algorithm>

namespace vnlbhip {
namespace {

// LDS layout of the filter kernel in 4-byte words (host computed).
struct FilterLayout {
    int pitch;       // words per lane slot row (>= template slots, 16-byte multiple)
    int row;         // 16 * pitch: words per model row
    int chunks;      // vector slots per lane
    int tail;        // lanes holding a tail element
    int u_pitch;     // words per dual-eigenvector sample row (multiple of 4)
    int tab_in;      // [models][row] input offsets from the patch origin
    int tab_acc;     // [models][row] accumulator offsets from the patch's cell
    int tab_meta;    // [models][row] t | c << 8 | fused << 16 | valid << 17
    int tab_win;     // [models][row] aggregation window weight
    int mean_n;      // [models][row] noisy mean
    int mean_b;      // [models][row] basic mean (Final)
    int basis;       // [models][rank][row]
    int u;           // [models][max_rows][u_pitch] dual eigenvectors, sample-major
    int proj;        // [cap][models][rank] projections kept between the passes
    int terms;       // 6 x [models][rank]: eigenvalues and what follows from them
    int base;        // [cap] 64-bit offsets of the sample patches in the videos
    int pos;         // [cap] packed sample positions
    int logw;        // [cap]
    int w;           // [cap]
    int score;       // [models][cap]
    int box;         // [slots] boxes of the output frames (TileBox), then the batch count
    int tile;        // [tile_words] doubles of the planes of one or more boxes
    int tile_words;  // 0: every contribution goes straight to the accumulators
    int tile_alias;  // the tile overlays the basis: groups of one round only
    int proj_cache;  // Basic: scores and reconstruction share the projections
    int words;
};

// LDS tile of the aggregation: doubles for the planes (the model's channels
// and the weights) of at least one box of search_window + 7 pixels squared,
// which holds the patches of one output frame (the windows of a scheduled
// frame, guided or not, are its candidates' origins; the patch times of two
// differently guided frames may widen a box, such a one is added directly).
struct TileBox {
    int x0, y0;
    int width, height;  // 0: no patch
    int cell;           // first of its width * height cells, per plane, in the batch
    int batch;          // boxes are added up and flushed in batches that fill the tile; -1: direct
};

// Planes that one model's pass writes.
int filter_tile_planes(const StageDesc& d) {
    return (d.coupled ? d.channels : 1) + 1;
}

// Words of the tile, 0 where the kernel has none: the tile needs rows of whole
// 16-element slots and 8x8 patches, and 40 KB at most.
int filter_tile_words(const StageDesc& d) {
    const int side = d.search_window + d.patch - 1;
    const bool exact = d.model_dim == kLanes * template_slots(d.model_dim);
    const long long words = 2LL * side * side * filter_tile_planes(d);
    return exact && d.patch == 8 && words <= 10240 ? static_cast<int>(words) : 0;
}

// Template slot count chosen for a stage (register array length).
int filter_template_slots(const StageDesc& d) {
    return template_slots(d.model_dim);
}

FilterLayout filter_layout(const StageDesc& d, int tile_words, bool alias) {
    FilterLayout L{};
    L.pitch = slot_pitch(d.model_dim);
    L.row = kLanes * L.pitch;
    L.chunks = d.model_dim / kLanes;
    L.tail = d.model_dim % kLanes;
    L.u_pitch = (d.rank + 3) / 4 * 4;
    const int models = d.models;
    int at = 0;
    const auto take = [&at](int words) {
        const int start = at;
        at += (words + 3) / 4 * 4;
        return start;
    };
    const int basis_words = models * d.rank * L.row;
    L.tile_alias = tile_words > 0 && alias ? 1 : 0;
    L.tile_words = L.tile_alias ? std::max(tile_words, basis_words) : tile_words;
    L.tile = take(L.tile_alias ? 0 : tile_words);
    L.box = take(tile_words > 0 ? static_cast<int>(sizeof(TileBox) / 4) * d.slots + 1 : 0);
    L.tab_in = take(models * L.row);
    L.tab_acc = take(tile_words > 0 ? 0 : models * L.row);
    L.tab_meta = take(tile_words > 0 ? 0 : models * L.row);
    L.tab_win = take(models * L.row);
    L.mean_n = take(models * L.row);
    L.mean_b = take(models * L.row);
    L.basis = take(L.tile_alias ? L.tile_words : basis_words);
    if (L.tile_alias) {
        L.tile = L.basis;
    }
    // Any group with fewer rows than a model dimension of at least 64 is dual.
    L.u = take(d.model_dim >= 64 ? models * d.max_rows * L.u_pitch : 0);
    const int proj_words = d.cap * models * d.rank;
    L.proj_cache = (d.stage == kBasic && proj_words <= 4096) ? 1 : 0;
    L.proj = take(L.proj_cache ? proj_words : 0);
    L.terms = take(6 * models * d.rank);
    L.base = take(2 * d.cap);
    L.pos = take(d.cap);
    L.logw = take(d.cap);
    L.w = take(d.cap);
    L.score = take(models * d.cap);
    L.words = at;
    return L;
}

// The layout a stage runs with: a tile of its own where four workgroups still
// fit a compute unit, or where its groups always take several rounds of
// samples (more than a sample per team); else over the basis, which a group
// of one round no longer needs once its rows are filtered (larger groups of
// such a stage are added directly); none where the model leaves no room.
// Groups of several rounds pay for the tile with a workgroup or two per compute
// unit and gain all the same: Basic of a 640x360x6 clip, coupled YUV, rank 16,
// 17 samples 6.6 ms without a tile, 5.4 with it, 24 samples 8.1 and 5.5, 40
// samples 11.1 and 7.0; rank 4, 24 samples 8.0 and 2.9; one model per channel,
// 24 samples 8.1 and 4.6; grey, 24 samples 4.1 and 2.0, 64 samples 6.8 and 3.7.
constexpr size_t kFilterSharedLimit = 112 * 1024;
FilterLayout filter_layout(const StageDesc& d) {
    const auto fits = [](const FilterLayout& L, size_t limit) {
        return L.tile_words > 0 && L.words * sizeof(float) <= limit;
    };
    const FilterLayout own = filter_layout(d, filter_tile_words(d), false);
    if (fits(own, 40 * 1024) || (d.similar > kTeams && fits(own, kFilterSharedLimit))) {
        return own;
    }
    const FilterLayout over = filter_layout(d, filter_tile_words(d), true);
    if (d.models == 1 && d.similar <= kTeams && fits(over, kFilterSharedLimit)) {
        return over;
    }
    return fits(own, kFilterSharedLimit) ? own : filter_layout(d, 0, false);
}

// Loads a lane's slots of an LDS row (slot layout) into registers with
// 128-bit reads; bt receives the tail slot.
template <int kS>
__device__ inline void load_slots(float (&b)[kS], float& bt, const float* row, int chunks,
                                  bool tail_lane) {
    const float4* b4 = reinterpret_cast<const float4*>(row);
#pragma unroll
    for (int q = 0; q < kS / 4; ++q) {
        if (4 * q < chunks) {
            const float4 v = b4[q];
            b[4 * q + 0] = v.x;
            b[4 * q + 1] = v.y;
            b[4 * q + 2] = v.z;
            b[4 * q + 3] = v.w;
        } else {
            b[4 * q + 0] = 0.0F;
            b[4 * q + 1] = 0.0F;
            b[4 * q + 2] = 0.0F;
            b[4 * q + 3] = 0.0F;
        }
    }
    bt = tail_lane ? row[chunks] : 0.0F;
}

// Dot product of two register row slices in the 16-lane order
// (dot_contiguous_highway, kernels_highway.hpp:12-44): lane-wise fma chains
// over the vector slots, a halving tree over the team, then the tail
// elements one by one.
template <int kS>
__device__ inline float team_dot(const float (&x)[kS], float xt, const float (&b)[kS], float bt,
                                 int chunks, int tail, int lane) {
    float part = 0.0F;
#pragma unroll
    for (int k = 0; k < kS; ++k) {
        if (k < chunks) {
            part = fmaf(x[k], b[k], part);
        }
    }
    float total = segment16_sum(part);
    if (tail > 0) {
        const float product = lane < tail ? xt * bt : 0.0F;
        for (int i = 0; i < tail; ++i) {
            total = total + __shfl(product, i, kLanes);
        }
    }
    return total;
}

// Squared norm of a register row slice in the same order.
template <int kS>
__device__ inline float team_norm2(const float (&x)[kS], float xt, int chunks, int tail,
                                   int lane) {
    float part = 0.0F;
#pragma unroll
    for (int k = 0; k < kS; ++k) {
        if (k < chunks) {
            part = fmaf(x[k], x[k], part);
        }
    }
    float total = segment16_sum(part);
    if (tail > 0) {
        const float product = lane < tail ? xt * xt : 0.0F;
        for (int i = 0; i < tail; ++i) {
            total = total + __shfl(product, i, kLanes);
        }
    }
    return total;
}

// Loads a lane's slots of one sample row, centered by an LDS mean in slot
// layout.  Slots outside the row stay zero.
template <int kS>
__device__ inline void load_centered(float (&x)[kS], float& xt, const float* __restrict__ video,
                                     size_t base, const int* tab_in, const float* mean,
                                     int chunks, bool tail_lane) {
#pragma unroll
    for (int k = 0; k < kS; ++k) {
        x[k] = 0.0F;
        if (k < chunks) {
            x[k] = video[base + tab_in[k]] - mean[k];
        }
    }
    xt = 0.0F;
    if (tail_lane) {
        xt = video[base + tab_in[chunks]] - mean[chunks];
    }
}

// The output frames' boxes of a group and their batches: a box takes `cell`
// to `cell + width * height` of every plane's tile cells.  One wavefront
// (lane 0 .. 63), lane = output frame, 64 of them at a time; complete after
// the caller's next barrier.
__device__ __forceinline__ void plan_boxes(const StageDesc& d, const uint32_t* __restrict__ s_pos, int similar,
                                           int af, int cells, TileBox* __restrict__ boxes, int* __restrict__ batches,
                                           int lane) {
    int batch = 0;
    int used = 0;
    for (int first = 0; first < d.slots; first += 64) {
        const int slot = first + lane;
        const int f = af + slot - d.search_bwd;
        int x0 = kMaxSide;
        int y0 = kMaxSide;
        int x1 = 0;
        int y1 = 0;
#pragma unroll 4
        for (int r = 0; r < similar; ++r) {
            const uint32_t p = s_pos[r];
            const int t = f - position_frame(p);
            const bool in = t >= 0 && t < d.patch_time;
            x0 = in ? min(x0, position_x(p)) : x0;
            y0 = in ? min(y0, position_y(p)) : y0;
            x1 = in ? max(x1, position_x(p) + 8) : x1;
            y1 = in ? max(y1, position_y(p) + 8) : y1;
        }
        const bool any = x1 > x0;
        TileBox box{x0, y0, any ? x1 - x0 : 0, any ? y1 - y0 : 0, 0, -1};
        const int size = slot < d.slots ? box.width * box.height : 0;
        const int here = min(d.slots - first, 64);
        for (int i = 0; i < here; ++i) {
            const int next = __builtin_amdgcn_readlane(size, i);
            if (next == 0 || next > cells) {
                continue;
            }
            if (used + next > cells) {
                ++batch;
                used = 0;
            }
            if (lane == i) {
                box.cell = used;
                box.batch = batch;
            }
            used += next;
        }
        if (slot < d.slots) {
            boxes[slot] = box;
        }
    }
    if (lane == 0) {
        *batches = batch + 1;
    }
}

// Sums in LDS and in device memory, by the pointer's type: through plain
// pointers the compiler joins the two into FLAT atomics.
using LdsDouble = __attribute__((address_space(3))) double;
using GlobalDouble = __attribute__((address_space(1))) double;
__device__ inline void add_double(LdsDouble* p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline void add_double(GlobalDouble* p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One round of samples (one per team, position p, weight w, the filtered row
// of model m in `out`; teams without a sample have held false) into the
// accumulators, through the tile.  Slots 4 q + i of a row are the 64 pixels
// of channel q / patch_time and patch time q % patch_time: lane l of the team
// holds pixel (l & 7, 2 i + (l >> 3)).  The weight of a sample's pixels is
// added once, with model 0.  Uniform over the workgroup but for the sample;
// `cells` cells per plane, zero before and after.
template <int kS>
__device__ __forceinline__ void aggregate_tile(const StageDesc& d, double* __restrict__ tile,
                                               const TileBox* __restrict__ boxes, int batches, int cells,
                                               double* __restrict__ acc, int af, uint32_t p, bool held, int m,
                                               float w, const float* __restrict__ t_win, const float (&out)[kS],
                                               int tid) {
    const int lane = tid % kLanes;
    float cw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        cw[i] = w * t_win[i];
    }
    const int px = position_x(p) + (lane & 7);
    const int py = position_y(p) + (lane >> 3);
    const int slot_base = position_frame(p) - af + d.search_bwd;
    const int c_first = d.coupled ? 0 : m;
    const int channels = d.coupled ? d.channels : 1;
    const size_t plane = static_cast<size_t>(d.height) * d.width;
    // Adds the sample's pixels of patch time t: value plane by value plane
    // from `cell` (plane_step apart), the weights into `weight`.
    const auto add = [&](int t, auto* cell, size_t plane_step, int row_step, auto* weight) {
        int next = t;
#pragma unroll
        for (int q = 0; q < kS / 4; ++q) {
            if (q == next) {  // uniform
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    add_double(cell + 2 * i * row_step, static_cast<double>(cw[i] * pinned(out[4 * q + i])));
                }
                cell += plane_step;
                next += d.patch_time;
            }
        }
        if (m == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                add_double(weight + 2 * i * row_step, static_cast<double>(cw[i]));
            }
        }
    };
#pragma nounroll
    for (int batch = 0; batch < batches; ++batch) {
#pragma nounroll
        for (int t = 0; t < d.patch_time; ++t) {
            const int slot = slot_base + t;
            if (held && slot >= 0 && slot < d.slots) {
                const TileBox box = boxes[slot];
                if (box.batch == batch) {
                    LdsDouble* cell = (LdsDouble*)tile + box.cell + (py - box.y0) * box.width + px - box.x0;
                    add(t, cell, cells, box.width, cell + channels * cells);
                } else if (batch == 0 && box.batch < 0) {
                    // Boxes too large for the tile.
                    GlobalDouble* frame = (GlobalDouble*)acc +
                                          static_cast<size_t>(af + slot - d.search_bwd) * (d.channels + 1) * plane +
                                          static_cast<size_t>(py) * d.width + px;
                    add(t, frame + c_first * plane, plane, d.width, frame + d.channels * plane);
                }
            }
        }
        __syncthreads();
        // Flush: a wavefront takes one plane of one box at a time, lane l
        // pixel l & 7 of a memory line in row l >> 3 of 8; lines count per
        // row from the one that holds the box's first pixel.
        int item = 0;
#pragma nounroll
        for (int slot = 0; slot < d.slots; ++slot) {
            const TileBox box = boxes[slot];
            if (__builtin_amdgcn_readfirstlane(box.batch) != batch) {
                continue;
            }
            const size_t f = static_cast<size_t>(af + slot - d.search_bwd) * (d.channels + 1);
            const int planes = channels + (m == 0 ? 1 : 0);
#pragma nounroll
            for (int k = 0; k < planes; ++k, ++item) {
                if ((item & (kModelThreads / 64 - 1)) != __builtin_amdgcn_readfirstlane(tid >> 6)) {
                    continue;
                }
                const size_t first = (f + (k < channels ? c_first + k : d.channels)) * plane +
                                     static_cast<size_t>(box.y0) * d.width + box.x0;
                double* sums = tile + k * cells + box.cell;
#pragma nounroll
                for (int y = (tid & 63) >> 3; y < box.height; y += 8) {
                    const size_t at = first + static_cast<size_t>(y) * d.width;
                    double* row = sums + y * box.width;
                    double* out_row = acc + at;
                    for (int x = (tid & 7) - static_cast<int>(at & 7); x < box.width; x += 8) {
                        if (x >= 0) {
                            const double sum = row[x];
                            if (sum != 0.0) {
                                row[x] = 0.0;
                                unsafeAtomicAdd(out_row + x, sum);
                            }
                        }
                    }
                }
            }
        }
        __syncthreads();
    }
}

// kExact: the model row is exactly 16 * kS elements (no tail, no slot
// guards at run time).  kTile (kExact and 8x8 patches): aggregation through
// the LDS tile.
template <int kS, bool kExact, bool kTile>
__global__ __launch_bounds__(kModelThreads, kS <= 8 ? 4 : (kS <= 24 ? 3 : 1)) void filter_kernel(
    StageDesc d, FilterLayout L, const float* __restrict__ noisy,
    const float* __restrict__ basic, GroupRefs refs, const int* __restrict__ group_count_dev,
    int problem_stride, const int* __restrict__ group_flags, const float* __restrict__ means,
    const float* __restrict__ eigenvalues, const float* __restrict__ vectors, Accumulators acc,
    float* __restrict__ weights_out, int* __restrict__ work_counter) {
    extern __shared__ float4 s_dyn4[];
    float* s_dyn = reinterpret_cast<float*>(s_dyn4);
    __shared__ float s_scalar[4 * kMaxChannels];
    __shared__ float s_red[kMaxChannels][kModelThreads / 64];

    int* tab_in = reinterpret_cast<int*>(s_dyn + L.tab_in);
    int* tab_acc = reinterpret_cast<int*>(s_dyn + L.tab_acc);
    int* tab_meta = reinterpret_cast<int*>(s_dyn + L.tab_meta);
    float* tab_win = s_dyn + L.tab_win;
    float* s_mean_n = s_dyn + L.mean_n;
    float* s_mean_b = s_dyn + L.mean_b;
    float* s_basis = s_dyn + L.basis;
    float* s_u = s_dyn + L.u;
    float* s_proj = s_dyn + L.proj;
    uint32_t* s_pos = reinterpret_cast<uint32_t*>(s_dyn + L.pos);
    float* s_logw = s_dyn + L.logw;
    float* s_w = s_dyn + L.w;
    float* s_score = s_dyn + L.score;

    // Basis rows taken together by a team (registers allowing): the dot
    // products' serial chains run side by side.
    constexpr int kAhead = kS <= 8 ? 4 : (kS <= 24 ? 2 : 1);

    const int tid = threadIdx.x;
    const int team = tid / kLanes;
    const int lane = tid % kLanes;
    const int models = d.models;
    const int md = d.model_dim;
    const int R = d.rank;
    const int row = L.row;
    const int pitch = L.pitch;
    const int chunks = kExact ? kS : L.chunks;
    const int tail = kExact ? 0 : L.tail;
    const bool tail_lane = lane < tail;
    const bool final_stage = d.stage == kFinal;
    float* s_lambda = s_dyn + L.terms;  // [models][R] each
    float* s_inv_sqrt = s_lambda + models * R;
    float* s_coef = s_inv_sqrt + models * R;
    float* s_lhat = s_coef + models * R;
    float* s_trace_term = s_lhat + models * R;
    float* s_volume_term = s_trace_term + models * R;
    size_t* s_base = reinterpret_cast<size_t*>(s_dyn + L.base);
    double* s_tile = reinterpret_cast<double*>(s_dyn + L.tile);
    TileBox* s_box = reinterpret_cast<TileBox*>(s_dyn + L.box);
    int* s_batches = reinterpret_cast<int*>(s_box + d.slots);
    const int cells = kTile ? L.tile_words / 2 / ((d.coupled ? d.channels : 1) + 1) : 0;
    if (kTile && L.tile_alias == 0) {
        for (int i = tid; i < L.tile_words / 2; i += kModelThreads) {
            s_tile[i] = 0.0;
        }
    }

    // Stage-constant element tables in slot layout.
    for (int i = tid; i < models * row; i += kModelThreads) {
        const int m = i / row;
        const int rem = i - m * row;
        const int l = rem / pitch;
        const int k = rem - l * pitch;
        const bool valid = k < chunks || (k == chunks && l < tail);
        int in_off = 0;
        int acc_off = 0;
        int meta = 0;
        float win = 0.0F;
        if (valid) {
            const int e = (d.coupled ? 0 : m * d.patch_dim) + kLanes * k + l;
            const int c = e / d.patch_dim;
            const int wi = e - c * d.patch_dim;
            const int t = wi / d.patch_area;
            const int yx = wi - t * d.patch_area;
            const int y = yx / d.patch;
            const int x = yx - y * d.patch;
            in_off = ((t * d.channels + c) * d.height + y) * d.width + x;
            acc_off = ((t * (d.channels + 1) + c) * d.height + y) * d.width + x;
            meta = t | (c << 8) | (x < d.fused_width ? kMetaFused : 0) | kMetaValid;
            win = d.window[yx];
        }
        tab_in[i] = in_off;
        if constexpr (!kTile) {
            tab_acc[i] = acc_off;
            tab_meta[i] = meta;
        }
        tab_win[i] = win;
    }

    const float sigma = d.sigma;
    const float beta = d.beta;
    const float sigma2 = (beta * sigma) * sigma;
    const float model_noise2 = final_stage ? (beta * d.sigma_basic) * d.sigma_basic : sigma2;
    const float estimate_noise2 = sigma2;
    const float match_sigma = final_stage ? d.sigma_basic : sigma;
    const float match_noise2 = match_sigma * match_sigma;
    const float floor_noise2 = (d.membership_noise_floor * sigma) * sigma;
    const float membership_noise2 = match_noise2 > floor_noise2 ? match_noise2 : floor_noise2;
    const float dual_floor = 128.0F * FLT_EPSILON;
    const float* member_video = final_stage ? basic : noisy;
    const float* member_mean_all = final_stage ? s_mean_b : s_mean_n;

    // Group indices are taken in order from the work counter (the next one
    // requested while the current group is processed) and spread over the
    // list by the largest odd stride near 0.618 * count coprime with the
    // count (uniform: every thread computes it from the device count).
    const int group_count = *group_count_dev;
    unsigned group_stride = static_cast<unsigned>(static_cast<double>(group_count) * 0.6180339887) | 1u;
    while (group_stride > 1) {
        unsigned x = group_stride;
        unsigned y = static_cast<unsigned>(group_count);
        while (y != 0) {
            const unsigned r = x % y;
            x = y;
            y = r;
        }
        if (x == 1) {
            break;
        }
        group_stride -= 2;
    }
    if (group_stride == 0) {
        group_stride = 1;
    }
    __shared__ int s_next;
    if (threadIdx.x == 0) {
        s_next = atomicAdd(work_counter, 1);
    }
    int following = 0;
    const auto advance = [&]() {
        __syncthreads();  // the group is done with the LDS and s_next
        if (threadIdx.x == 0) {
            s_next = following;
        }
        __syncthreads();
        return s_next;
    };
    __syncthreads();
    for (int gi = s_next; gi < group_count; gi = advance()) {
        if (threadIdx.x == 0) {
            following = atomicAdd(work_counter, 1);
        }
        const int g = static_cast<int>((static_cast<unsigned long long>(gi) * group_stride) %
                                       static_cast<unsigned>(group_count));
        const int a = refs.group_list[g];
        const int af = position_frame(refs.anchors[a]);
        const int similar = refs.counts[a];
        const size_t list = static_cast<size_t>(a) * d.cap;
        const int flags = group_flags[g];
        const bool equal = (flags & kFlagEqual) != 0;
        const bool flat = (flags & kFlagFlat) != 0;
        const bool modelled = (flags & kFlagModelled) != 0;
        const int rows = model_rows_of(d, similar);
        const bool dual = group_uses_dual(d, rows);
        const bool fit = modelled && !equal;

        for (int r = tid; r < similar; r += kModelThreads) {
            const uint32_t p = refs.positions[list + r];
            s_pos[r] = p;
            s_base[r] = patch_base(d, p);
            s_logw[r] = 0.0F;
            s_w[r] = 1.0F;
        }
        const float* g_mean = means + static_cast<size_t>(g) * 2 * d.dim;
        for (int m = 0; m < models; ++m) {
            for (int i = tid; i < md; i += kModelThreads) {
                const int slot = m * row + (i % kLanes) * pitch + i / kLanes;
                const int e = (d.coupled ? 0 : m * d.patch_dim) + i;
                s_mean_n[slot] = g_mean[e];
                s_mean_b[slot] = final_stage ? g_mean[d.dim + e] : 0.0F;
            }
        }
        if (fit) {
            // Eigenvalues, compute_filter_coefficients (core.cpp:616-636) and
            // the per-component terms of accumulate_aggregation_model
            // (core.cpp:326-412), by the last threads: they have the least to
            // do in the basis map below.
            const float sigma_basic2 = final_stage ? (beta * d.sigma_basic) * d.sigma_basic : sigma2;
            const float threshold = d.variance_threshold * sigma2;
            for (int i = kModelThreads - 1 - tid; i < models * R; i += kModelThreads) {
                const float lambda = eigenvalues[static_cast<size_t>(g) * models * R + i];
                float variance = lambda;
                if (sigma_basic2 > 0.0F) {
                    variance = variance - fminf(variance, sigma_basic2);
                }
                const float lhat_raw = lambda - model_noise2;
                const float lhat = lhat_raw > 0.0F ? lhat_raw : 0.0F;
                s_lambda[i] = lambda;
                s_inv_sqrt[i] = !(lambda <= dual_floor) ? 1.0F / sqrtf(lambda) : 0.0F;
                s_coef[i] = variance > threshold ? 1.0F / (1.0F + (sigma2 / variance)) : 0.0F;
                s_lhat[i] = lhat;
                s_trace_term[i] = lhat > 0.0F ? lhat / (lhat + estimate_noise2) : 0.0F;
                s_volume_term[i] = lhat > 0.0F ? log1p_via_double(lhat / membership_noise2) : 0.0F;
            }
            if (dual) {
                // Eigenvectors of the Gram matrix, sample-major: u[m][s][j].
                for (int q = team; q < models * R; q += kTeams) {
                    const int m = models == 1 ? 0 : q / R;
                    const int j = q - m * R;
                    const float* vector = vectors + static_cast<size_t>(g * models * R + q) * problem_stride;
                    for (int s = lane; s < rows; s += kLanes) {
                        s_u[(m * d.max_rows + s) * L.u_pitch + j] = vector[s];
                    }
                }
            } else {
                // Covariance eigenvectors are the basis itself.
                for (int q = team; q < models * R; q += kTeams) {
                    const float* vector = vectors + static_cast<size_t>(g * models * R + q) * problem_stride;
                    for (int e = lane; e < md; e += kLanes) {
                        s_basis[q * row + lane * pitch + e / kLanes] = vector[e];
                    }
                }
            }
        }
        __syncthreads();

        // The group's precision and volume terms, beside the basis map.
        if (!equal && tid >= kModelThreads - models) {
            const int m = kModelThreads - 1 - tid;
            const int rank_used = modelled ? R : 0;
            float trace = 0.0F;
            float volume = 0.0F;
            for (int j = 0; j < rank_used; ++j) {
                if (s_lhat[m * R + j] > 0.0F) {
                    trace = trace + s_trace_term[m * R + j];
                    volume = volume + s_volume_term[m * R + j];
                }
            }
            const float mean_term = static_cast<float>(md) / static_cast<float>(rows);
            const float tau = (d.weight_epsilon + mean_term) + trace;
            s_scalar[4 * m + 0] = d.weight_alpha == 0.0F ? 0.0F : -d.weight_alpha * log_via_double(tau);
            s_scalar[4 * m + 1] = volume / static_cast<float>(md);
        }
        if (fit && dual) {
            // map_dual_eigenvectors_to_basis (linalg.cpp:552-595): basis row j
            // is sum_s u[s][j] (x_s - mean) / sqrt(lambda_j), then normalized.
            for (int i = tid; i < models * md; i += kModelThreads) {
                const int m = i / md;
                const int e = i - m * md;
                const int k = e / kLanes;
                const int slot = m * row + (e % kLanes) * pitch + k;
                const bool fused = k < chunks;
                const int in_off = tab_in[slot];
                const float mean_e = member_mean_all[slot];
                for (int j0 = 0; j0 < R; j0 += 16) {
                    float accs[16];
#pragma unroll
                    for (int jj = 0; jj < 16; ++jj) {
                        accs[jj] = 0.0F;
                    }
                    // (Eight samples' loads at a time, then their products in
                    // sample order: the loop would wait for each load.)
                    for (int s0 = 0; s0 < rows; s0 += 8) {
                        float x[8];
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            x[i] = member_video[s_base[min(s0 + i, rows - 1)] + in_off];
                        }
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            if (s0 + i >= rows) {
                                break;
                            }
                            const float xi = x[i] - mean_e;
                            const float4* u4 = reinterpret_cast<const float4*>(
                                s_u + (m * d.max_rows + s0 + i) * L.u_pitch + j0);
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                if (j0 + 4 * q < R) {
                                    const float4 u = u4[q];
                                    const float uu[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                                    for (int h = 0; h < 4; ++h) {
                                        // (Products past R are never stored.)
                                        const int jj = 4 * q + h;
                                        if (kExact || fused) {
                                            accs[jj] = fmaf(uu[h], xi, accs[jj]);
                                        } else {
                                            const float product = uu[h] * xi;
                                            accs[jj] = accs[jj] + product;
                                        }
                                    }
                                }
                            }
                        }
                    }
#pragma unroll
                    for (int jj = 0; jj < 16; ++jj) {
                        const int j = j0 + jj;
                        if (j < R) {
                            const float value =
                                !(s_lambda[m * R + j] <= dual_floor) ? accs[jj] * s_inv_sqrt[m * R + j] : 0.0F;
                            s_basis[(m * R + j) * row + slot - m * row] = value;
                        }
                    }
                }
            }
            __syncthreads();
            // normalize_or_zero (linalg.cpp:235-246).
            for (int q = team; q < models * R; q += kTeams) {
                const int m = q / R;
                const int j = q - m * R;
                if (s_lambda[m * R + j] <= dual_floor) {
                    continue;
                }
                float* brow = s_basis + q * row + lane * pitch;
                float v[kS];
#pragma unroll
                for (int k = 0; k < kS; ++k) {
                    v[k] = k < chunks ? brow[k] : 0.0F;
                }
                const float vt = tail_lane ? brow[chunks] : 0.0F;
                const float norm2 = team_norm2(v, vt, chunks, tail, lane);
                const bool zero = norm2 <= dual_floor;
                const float scale = zero ? 0.0F : 1.0F / sqrtf(norm2);
#pragma unroll
                for (int k = 0; k < kS; ++k) {
                    if (k < chunks) {
                        brow[k] = zero ? 0.0F : v[k] * scale;
                    }
                }
                if (tail_lane) {
                    brow[chunks] = zero ? 0.0F : vt * scale;
                }
            }
        }

        __syncthreads();

        // Aggregation weights (accumulate_aggregation_model core.cpp:326-412,
        // finalize_aggregation_weights :276-294).
        const bool weights_need_scores = !equal && d.weight_beta != 0.0F;
        const bool cached = L.proj_cache != 0 && weights_need_scores && modelled;
        int model_count = 0;
        if (!equal) {
            if (d.weight_alpha == 0.0F && d.weight_beta == 0.0F) {
                model_count = models;
            } else if (!weights_need_scores) {
                for (int r = tid; r < similar; r += kModelThreads) {
                    float lw = s_logw[r];
                    for (int m = 0; m < models; ++m) {
                        lw = lw + s_scalar[4 * m + 0];
                    }
                    s_logw[r] = lw;
                }
                model_count = models;
            } else {
                const int rank_used = modelled ? R : 0;
                const float score_scale = sqrtf(2.0F * static_cast<float>(md));
                float local_min[kMaxChannels];
#pragma unroll
                for (int m = 0; m < kMaxChannels; ++m) {
                    local_min[m] = INFINITY;
                }
                for (int r = team; r < similar; r += kTeams) {
                    const size_t base = s_base[r];
                    for (int m = 0; m < models; ++m) {
                        const int lane_slot = m * row + lane * pitch;
                        float x[kS];
                        float xt;
                        load_centered(x, xt, member_video, base, tab_in + lane_slot,
                                      member_mean_all + lane_slot, chunks, tail_lane);
                        const float norm2 = team_norm2(x, xt, chunks, tail, lane);
                        float distance = 0.0F;
                        float projected = 0.0F;
                        for (int j0 = 0; j0 < rank_used; j0 += kAhead) {
                            float b[kAhead][kS];
                            float bt[kAhead];
#pragma unroll
                            for (int i = 0; i < kAhead; ++i) {
                                const int j = min(j0 + i, rank_used - 1);
                                load_slots(b[i], bt[i], s_basis + (m * R + j) * row + lane * pitch, chunks,
                                           tail_lane);
                            }
                            float projection[kAhead];
#pragma unroll
                            for (int i = 0; i < kAhead; ++i) {
                                projection[i] = team_dot(x, xt, b[i], bt[i], chunks, tail, lane);
                            }
#pragma unroll
                            for (int i = 0; i < kAhead; ++i) {
                                const int j = j0 + i;
                                if (j < rank_used) {
                                    if (cached && lane == 0) {
                                        s_proj[(r * models + m) * R + j] = projection[i];
                                    }
                                    const float projection2 = projection[i] * projection[i];
                                    distance = distance + projection2 / (s_lhat[m * R + j] + membership_noise2);
                                    projected = projected + projection2;
                                }
                            }
                        }
                        const float residual = norm2 - projected > 0.0F ? norm2 - projected : 0.0F;
                        distance = distance + residual / membership_noise2;
                        const float score = (distance - static_cast<float>(md)) / score_scale;
                        if (lane == 0) {
                            s_score[m * d.cap + r] = score;
                        }
#pragma unroll
                        for (int mm = 0; mm < kMaxChannels; ++mm) {
                            if (mm == m) {
                                local_min[mm] = fminf(local_min[mm], score);
                            }
                        }
                    }
                }
#pragma unroll
                for (int m = 0; m < kMaxChannels; ++m) {
                    if (m < models) {
                        const float v = wave_min(local_min[m]);
                        if ((tid & 63) == 0) {
                            s_red[m][tid >> 6] = v;
                        }
                    }
                }
                __syncthreads();
                for (int r = tid; r < similar; r += kModelThreads) {
                    float lw = s_logw[r];
                    for (int m = 0; m < models; ++m) {
                        float min_score = s_red[m][0];
                        for (int w = 1; w < kModelThreads / 64; ++w) {
                            min_score = fminf(min_score, s_red[m][w]);
                        }
                        const float excess = s_score[m * d.cap + r] - min_score;
                        const float membership = (excess > 0.0F ? excess : 0.0F) + s_scalar[4 * m + 1];
                        const float delta = s_scalar[4 * m + 0] - (d.weight_beta * membership);
                        lw = lw + delta;
                    }
                    s_logw[r] = lw;
                }
                model_count = models;
            }
        }
        if (d.weights_enabled) {
            if (model_count == 0) {
                const float tau = d.weight_epsilon + (static_cast<float>(md) / static_cast<float>(rows));
                const float log_group = d.weight_alpha == 0.0F ? 0.0F : -d.weight_alpha * log_via_double(tau);
                for (int r = tid; r < similar; r += kModelThreads) {
                    s_logw[r] = s_logw[r] + log_group;
                }
                model_count = 1;
            }
            const float inv_models = 1.0F / static_cast<float>(model_count);
            for (int r = tid; r < similar; r += kModelThreads) {
                float value = s_logw[r] * inv_models;
                value = value < -80.0F ? -80.0F : (value > 80.0F ? 80.0F : value);
                s_w[r] = exp_via_double(value);
            }
        }
        if constexpr (kTile) {
            // (Several rounds need the basis until the last: no tile over it.)
            // The last wavefront: the first takes the samples' weights.
            if (tid >= kModelThreads - 64) {
                const bool no_tile = L.tile_alias != 0 && similar > kTeams;
                plan_boxes(d, s_pos, similar, af, no_tile ? 0 : cells, s_box, s_batches, tid & 63);
            }
        }
        __syncthreads();
        if (weights_out != nullptr) {
            for (int r = tid; r < similar; r += kModelThreads) {
                weights_out[list + r] = s_w[r];
            }
        }

        // Reconstruction (project_bayes_estimate core.cpp:578-614) and the
        // weighted scatter of every sample.
        const float* center_all = (final_stage && flat) ? s_mean_b : s_mean_n;
        // (With the tile, the workgroup's teams stay together through a round
        // of samples: teams past the last sample join its barriers.)
        const int rounds_end = kTile ? (similar + kTeams - 1) / kTeams * kTeams : similar;
        for (int r = team; r < rounds_end; r += kTeams) {
            const bool held = !kTile || r < similar;
            const float w = held ? s_w[r] : 0.0F;
            const uint32_t p = held ? s_pos[r] : s_pos[0];
            const int pf = position_frame(p);
            const size_t base = s_base[held ? r : 0];
            double* cell_base =
                acc.data + (static_cast<size_t>(pf) * (d.channels + 1) * d.height + position_y(p)) * d.width +
                position_x(p);
            const int slot_base = pf - af + d.search_bwd;
            for (int m = 0; m < models; ++m) {
                const int lane_slot = m * row + lane * pitch;
                const int* t_in = tab_in + lane_slot;
                const int* t_acc = tab_acc + lane_slot;
                const int* t_meta = tab_meta + lane_slot;
                const float* t_win = tab_win + lane_slot;
                const float* center = center_all + lane_slot;
                float out[kS];
                float out_t = 0.0F;
                if (!held) {
#pragma unroll
                    for (int k = 0; k < kS; ++k) {
                        out[k] = 0.0F;
                    }
                } else if (equal) {
#pragma unroll
                    for (int k = 0; k < kS; ++k) {
                        out[k] = k < chunks ? noisy[base + t_in[k]] : 0.0F;
                    }
                    if (tail_lane) {
                        out_t = noisy[base + t_in[chunks]];
                    }
                } else if (!modelled) {
#pragma unroll
                    for (int k = 0; k < kS; ++k) {
                        out[k] = k < chunks ? center[k] : 0.0F;
                    }
                    if (tail_lane) {
                        out_t = center[chunks];
                    }
                } else {
                    float y[kS] = {};
                    float yt = 0.0F;
                    if (!cached) {
                        load_centered(y, yt, noisy, base, t_in, center, chunks, tail_lane);
                    }
#pragma unroll
                    for (int k = 0; k < kS; ++k) {
                        out[k] = 0.0F;
                    }
                    // Per element the terms arrive in basis order, fused over
                    // the vector slots and rounded product-then-sum in the tail.
                    for (int j0 = 0; j0 < R; j0 += kAhead) {
                        float b[kAhead][kS];
                        float bt[kAhead];
                        float projection[kAhead];
                        float coefficient[kAhead];
#pragma unroll
                        for (int i = 0; i < kAhead; ++i) {
                            const int j = min(j0 + i, R - 1);
                            coefficient[i] = j0 + i < R ? s_coef[m * R + j] : 0.0F;
                            load_slots(b[i], bt[i], s_basis + (m * R + j) * row + lane * pitch, chunks, tail_lane);
                            projection[i] = cached ? s_proj[(r * models + m) * R + j] : 0.0F;
                        }
                        if (!cached) {
#pragma unroll
                            for (int i = 0; i < kAhead; ++i) {
                                projection[i] = team_dot(y, yt, b[i], bt[i], chunks, tail, lane);
                            }
                        }
#pragma unroll
                        for (int i = 0; i < kAhead; ++i) {
                            if (coefficient[i] == 0.0F) {
                                continue;
                            }
                            const float sp = coefficient[i] * projection[i];
#pragma unroll
                            for (int k = 0; k < kS; ++k) {
                                if (k < chunks) {
                                    out[k] = fmaf(sp, b[i][k], out[k]);
                                }
                            }
                            if (tail_lane) {
                                const float product = sp * bt[i];
                                out_t = out_t + product;
                            }
                        }
                    }
#pragma unroll
                    for (int k = 0; k < kS; ++k) {
                        if (k < chunks) {
                            out[k] = out[k] + center[k];
                        }
                    }
                    if (tail_lane) {
                        out_t = out_t + center[chunks];
                    }
                }
                if constexpr (kTile) {
                    if (L.tile_alias != 0 && similar <= kTeams) {
                        // The basis gives way to the tile.
                        __syncthreads();
                        for (int i = tid; i < L.tile_words / 2; i += kModelThreads) {
                            s_tile[i] = 0.0;
                        }
                        __syncthreads();
                    }
                    aggregate_tile<kS>(d, s_tile, s_box, *s_batches, cells, acc.data, af, p, held, m, w, t_win, out,
                                       tid);
                    continue;
                }
#pragma unroll
                for (int k = 0; k < kS; ++k) {
                    if (k < chunks) {
                        scatter(d, cell_base, slot_base, t_meta[k], t_acc[k], t_win[k], out[k], w);
                    }
                }
                if (tail_lane) {
                    scatter(d, cell_base, slot_base, t_meta[chunks], t_acc[chunks], t_win[chunks], out_t, w);
                }
            }
        }
    }
}

}  // namespace

size_t filter_shared_bytes(const StageDesc& d) {
    // The stage limit counts what grows with the patch and the model; the
    // component terms and the sample offsets are on top of it, and the tile
    // gives way (filter_layout).
    const int extra = (6 * d.models * d.rank + 3) / 4 * 4 + (2 * d.cap + 3) / 4 * 4;
    return static_cast<size_t>(filter_layout(d, 0, false).words - extra) * sizeof(float);
}

hipError_t launch_filter(const StageDesc& d, const float* noisy, const float* basic,
                         const uint32_t* anchors, const int* counts,
                         const uint32_t* positions, const int* group_list,
                         const int* group_count_dev, int group_capacity,
                         int problem_stride, const int* group_flags, const int* problem_dims,
                         const float* means, const float* eigenvalues, const float* vectors,
                         double* accumulators, float* weights_out, int* work_counter,
                         hipStream_t stream) {
    (void)problem_dims;
    if (group_capacity <= 0) {
        return hipSuccess;
    }
    const GroupRefs refs{anchors, counts, positions, group_list};
    const Accumulators acc{accumulators};
    const FilterLayout L = filter_layout(d);
    const size_t shared = static_cast<size_t>(L.words) * sizeof(float);
    int device = 0;
    int units = 0;
    hipError_t status = hipGetDevice(&device);
    if (status == hipSuccess) {
        status = hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device);
    }
    if (status != hipSuccess) {
        return status;
    }
    const int slots = filter_template_slots(d);
    const bool exact = d.model_dim == kLanes * slots;
#define VNLBHIP_FILTER(KS, EXACT, TILE)                                                           \
    do {                                                                                          \
        int per_unit = 0;                                                                         \
        status = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_unit, (filter_kernel<KS, EXACT, TILE>), \
                                                              kModelThreads, shared);             \
        if (status != hipSuccess) {                                                               \
            return status;                                                                        \
        }                                                                                         \
        const long long resident = static_cast<long long>(per_unit > 0 ? per_unit : 1) * units;   \
        const unsigned blocks =                                                                   \
            static_cast<unsigned>(resident < group_capacity ? resident : group_capacity);         \
        hipLaunchKernelGGL((filter_kernel<KS, EXACT, TILE>), dim3(blocks), dim3(kModelThreads), shared, \
                           stream, d, L, noisy, basic, refs, group_count_dev,                     \
                           problem_stride, group_flags, means, eigenvalues, vectors, acc,         \
                           weights_out, work_counter);                                            \
    } while (0)
#define VNLBHIP_FILTER_SLOTS(KS)          \
    if (L.tile_words > 0) {               \
        VNLBHIP_FILTER(KS, true, true);   \
    } else if (exact) {                   \
        VNLBHIP_FILTER(KS, true, false);  \
    } else {                              \
        VNLBHIP_FILTER(KS, false, false); \
    }
    switch (slots) {
        case 4: VNLBHIP_FILTER_SLOTS(4); break;
        case 8: VNLBHIP_FILTER_SLOTS(8); break;
        case 16: VNLBHIP_FILTER_SLOTS(16); break;
        case 24: VNLBHIP_FILTER_SLOTS(24); break;
        case 32: VNLBHIP_FILTER_SLOTS(32); break;
        default: VNLBHIP_FILTER_SLOTS(64); break;
    }
#undef VNLBHIP_FILTER_SLOTS
#undef VNLBHIP_FILTER
    return hipGetLastError();
}

}  // namespace vnlbhip
