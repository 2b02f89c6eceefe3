// Batched cyclic Jacobi eigen solve of the group models, several small
// problems per wavefront.
//
// Semantics follow filter_vnlb_samples and its callees in the reference
// (src/core/core.cpp:184-871, src/linalg/linalg.cpp:153-595) with the
// 16-lane summation order of the CPU restatement.
#include "common.h"
#include "device_util.h"
#include "eigen_order.h"
#include "group.h"
#include "kernels.h"

#include <float.h>

#include <utility>

namespace vnlbhip {
namespace {

// ---------------------------------------------------------------------------
// jacobi
// ---------------------------------------------------------------------------

// topk_symmetric_eigen_jacobi (linalg.cpp:447-519): cyclic row-by-row
// rotations above threshold = max(0, 64 eps max(1, max|A|)), at most
// max_sweeps sweeps, "converged" also when the off-diagonal is below
// 8 * threshold; eigenpairs sorted descending (stable) and each vector made
// unit length with its largest-magnitude entry positive
// (canonicalize_vector_row :204-233).
//
// Both kernels below apply the rotations in the reference's order with its
// operations, so their results are the reference's bit for bit.  They share
// one observation: while the rotations (p, p + 1), (p, p + 2), ... of row p
// run, row r only needs its running entry A[r][p], its entry A[r][q] of the
// current column and the same two of V; what the symmetric copies of row p
// hold is read by nobody until the row is finished.

// jacobi_rotate (linalg.cpp:153-202): the rotation of pivot apq between the
// diagonal entries app and aqq, and the new diagonal.
struct Rotation {
    float c;
    float s;
    float new_pp;
    float new_qq;
};

// Square root and reciprocal of x >= 1, correctly rounded: the hardware's
// approximation and one Newton step on its residual.  Compared with sqrtf
// and 1.0F / x for every float in [1, 2^52): no difference.  Without the
// general case's scaling and special values they are 4 and 3 dependent
// instructions instead of 15 and 11.
__device__ __forceinline__ float sqrt_from_one(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    const float s = x * y;
    return fmaf(fmaf(-s, s, x), 0.5F * y, s);
}
__device__ __forceinline__ float reciprocal_from_one(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(fmaf(-x, r, 1.0F), r, r);
}

// A rotating pivot is above 64 float epsilons (2^-17) of max |A| and the
// diagonal at most n max |A| = 128 max |A| in magnitude, so |tau| is at most
// 2^24: the first root's argument is at most 1 + 2^48, its reciprocal's 2^25
// and the second pair's 2, all within the range compared above.
__device__ __forceinline__ Rotation rotation_of(float app, float aqq, float apq) {
    Rotation o;
    const float tau = (aqq - app) / (2.0F * apq);
    const float tau_abs = fabsf(tau);
    const float t_abs = reciprocal_from_one(tau_abs + sqrt_from_one(1.0F + (tau * tau)));
    const float t = tau < 0.0F ? -t_abs : t_abs;
    o.c = reciprocal_from_one(sqrt_from_one(1.0F + (t * t)));
    o.s = t * o.c;
    const float cc = o.c * o.c;
    const float ss = o.s * o.s;
    const float two_cs = 2.0F * (o.c * o.s);
    o.new_pp = ((cc * app) - (two_cs * apq)) + (ss * aqq);
    o.new_qq = ((ss * app) + (two_cs * apq)) + (cc * aqq);
    return o;
}

__device__ inline void rotate_pair(const Rotation& o, float& left, float& right) {
    const float l = left;
    const float r = right;
    left = (o.c * l) - (o.s * r);
    right = (o.s * l) + (o.c * r);
}

// The canonical vector of column col of V (rows of `stride` floats in LDS),
// read in row order.
__device__ inline void write_eigenvector(const float* __restrict__ v, int stride, int n, int col,
                                         float* __restrict__ out) {
    float norm_squared = 0.0F;
    float max_abs = 0.0F;
    int pivot = 0;
    for (int i = 0; i < n; ++i) {
        const float value = v[i * stride + col];
        const float square = value * value;
        norm_squared = norm_squared + square;
        const float value_abs = fabsf(value);
        if (value_abs > max_abs) {
            max_abs = value_abs;
            pivot = i;
        }
    }
    float scale = 1.0F;
    const bool rescale = norm_squared > FLT_MIN;
    if (rescale) {
        scale = 1.0F / sqrtf(norm_squared);
        if (v[pivot * stride + col] < 0.0F) {
            scale = -scale;
        }
    }
    for (int i = 0; i < n; ++i) {
        const float value = v[i * stride + col];
        out[i] = rescale ? value * scale : value;
    }
}

// v of lane kLane of the same four lanes.
template <int kLane> __device__ inline float quad_lane(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), kLane * 0x55, 0xF, 0xF, true));
}

// Problems of at most 4 kSlots (<= 16) rows: four lanes per problem, sixteen
// problems per wavefront, A and V in registers; lane l holds the rows
// l, l + 4, ... (slot k is row 4 k + l).  Bound by instruction issue: a
// rotation's divide, roots and reciprocals (about 50 instructions) cost the
// wavefront the same whether 4 or 16 problems share it, so four lanes per
// problem beat sixteen; one lane per problem would need A and V of 16 rows in
// 392 registers.  Measured against sixteen lanes per problem with A and V in
// LDS, half a stage each: 188 k problems of 16 rows 4.60 -> 1.67 ms, 83 k of
// 12 rows 1.24 -> 0.38 ms, 2.6 k of 8 rows 79 -> 46 us (a wavefront's serial
// chain).
template <int kSlots, int kP>
__device__ __forceinline__ void quad_load_row(const float (&a)[kSlots][4 * kSlots], const float (&v)[kSlots][4 * kSlots],
                                     int p, float (&rp)[kSlots], float (&vp)[kSlots], float& app) {
    if (p == kP) {
#pragma unroll
        for (int k = 0; k < kSlots; ++k) {
            rp[k] = pinned(a[k][kP]);
            vp[k] = pinned(v[k][kP]);
        }
        app = quad_lane<kP % 4>(pinned(a[kP / 4][kP]));
    }
}

// Row p finished: column p and row p of A (entries rp, diagonal app).
template <int kSlots, int kP, int... kX>
__device__ __forceinline__ void quad_store_row(float (&a)[kSlots][4 * kSlots], float (&v)[kSlots][4 * kSlots], int l, int p,
                                      const float (&rp)[kSlots], const float (&vp)[kSlots], float app,
                                      std::integer_sequence<int, kX...>) {
    if (p == kP) {
#pragma unroll
        for (int k = 0; k < kSlots; ++k) {
            a[k][kP] = pinned(rp[k]);
            v[k][kP] = pinned(vp[k]);
        }
        // (The lane exchanges run in all lanes of the four, the selects after them.)
        const bool own = l == kP % 4;
        const auto take = [&](float& entry, float value) { entry = own ? value : entry; };
        (take(a[kP / 4][kX], quad_lane<kX % 4>(rp[kX / 4])), ...);
        a[kP / 4][kP] = own ? app : a[kP / 4][kP];
    }
}

// Rotation (p, kQ).  The lane of row kQ takes the new column's entries as
// its row; row p's entries are junk until quad_store_row.
template <int kSlots, int kQ, int... kX>
__device__ __forceinline__ void quad_rotate(float (&a)[kSlots][4 * kSlots], float (&v)[kSlots][4 * kSlots], int l, int p,
                                   bool active, float threshold, float (&rp)[kSlots], float (&vp)[kSlots],
                                   float& app, std::integer_sequence<int, kX...>) {
    if (kQ <= p) {
        return;  // uniform
    }
    const float apq = quad_lane<kQ % 4>(rp[kQ / 4]);
    if (active && fabsf(apq) > threshold) {
        const float aqq = quad_lane<kQ % 4>(a[kQ / 4][kQ]);
        const Rotation o = rotation_of(app, aqq, apq);
        app = o.new_pp;
#pragma unroll
        for (int k = 0; k < kSlots; ++k) {
            rotate_pair(o, rp[k], a[k][kQ]);
            rotate_pair(o, vp[k], v[k][kQ]);
        }
        const bool own = l == kQ % 4;
        rp[kQ / 4] = own ? 0.0F : rp[kQ / 4];
        const auto take = [&](float& entry, float value) { entry = own ? value : entry; };
        (take(a[kQ / 4][kX], quad_lane<kX % 4>(a[kX / 4][kQ])), ...);
        a[kQ / 4][kQ] = own ? o.new_qq : a[kQ / 4][kQ];
    }
    // One rotation at a time (bounded register use).
    __builtin_amdgcn_sched_barrier(0);
}

template <int kSlots, int... kI>
__device__ __forceinline__ void quad_sweep(float (&a)[kSlots][4 * kSlots], float (&v)[kSlots][4 * kSlots], int l, bool active,
                                  float threshold, std::integer_sequence<int, kI...> all) {
#pragma nounroll
    for (int p = 0; p + 1 < 4 * kSlots; ++p) {
        float rp[kSlots];
        float vp[kSlots];
        float app = 0.0F;
        (quad_load_row<kSlots, kI>(a, v, p, rp, vp, app), ...);
        (quad_rotate<kSlots, kI>(a, v, l, p, active, threshold, rp, vp, app, all), ...);
        (quad_store_row<kSlots, kI>(a, v, l, p, rp, vp, app, all), ...);
    }
}

// Eigenpairs in the stable descending order of the diagonal.  Every lane
// walks a column of V in row order (the lane exchanges bring the other
// lanes' rows), then writes its own rows of the canonical vector: a few
// percent of the solver's instructions, and no LDS, whose staging of 16
// problems would halve the wavefronts per compute unit.
template <int kSlots, int kC, int... kI>
__device__ __forceinline__ void quad_output_column(const float (&v)[kSlots][4 * kSlots],
                                                   const float (&diag)[4 * kSlots],
                                                   const float (&keys)[4 * kSlots], int l, bool valid, int n, int rank_limit, int stride,
                                                   float* __restrict__ vectors, float* __restrict__ values,
                                                   std::integer_sequence<int, kI...>) {
    const float dr = diag[kC];
    int rank = 0;
    ((rank += kI < n && kI != kC && ordered_before(keys[kI], keys[kC], kI < kC) ? 1 : 0), ...);
    float norm_squared = 0.0F;
    float max_abs = 0.0F;
    float pivot = quad_lane<0>(v[0][kC]);
    const auto add = [&](float value, bool held) {
        if (held) {
            norm_squared = norm_squared + value * value;
            const float value_abs = fabsf(value);
            if (value_abs > max_abs) {
                max_abs = value_abs;
                pivot = value;
            }
        }
    };
    (add(quad_lane<kI % 4>(v[kI / 4][kC]), kI < n), ...);
    float scale = 1.0F;
    const bool rescale = norm_squared > FLT_MIN;
    if (rescale) {
        scale = 1.0F / sqrtf(norm_squared);
        if (pivot < 0.0F) {
            scale = -scale;
        }
    }
    if (valid && kC < n && rank < rank_limit) {
#pragma unroll
        for (int k = 0; k < kSlots; ++k) {
            const int r = 4 * k + l;
            if (r < n) {
                vectors[static_cast<size_t>(rank) * stride + r] = rescale ? v[k][kC] * scale : v[k][kC];
            }
        }
        if (l == 0) {
            values[rank] = dr;
        }
    }
}

template <int kSlots, int... kI>
__device__ __forceinline__ void quad_output(const float (&a)[kSlots][4 * kSlots],
                                            const float (&v)[kSlots][4 * kSlots], int l, bool valid, int n,
                                            int rank_limit, int stride, float* __restrict__ vectors,
                                            float* __restrict__ values, std::integer_sequence<int, kI...> all) {
    const float diag[] = {quad_lane<kI % 4>(a[kI / 4][kI])...};
    const float keys[] = {order_key(diag[kI])...};
    (quad_output_column<kSlots, kI>(v, diag, keys, l, valid, n, rank_limit, stride, vectors, values, all), ...);
}

template <int kSlots>
__global__ __launch_bounds__(64) void jacobi_quad_kernel(
    StageDesc d, const int* __restrict__ group_count_dev, int problem_stride,
    const int* __restrict__ group_flags, const int* __restrict__ problem_dims,
    const float* __restrict__ problems, float* __restrict__ eigenvalues,
    float* __restrict__ vectors, int* __restrict__ status) {
    constexpr int kN = 4 * kSlots;
    constexpr int kPerWave = 16;
    const int problem_count = *group_count_dev * d.models;
    if (static_cast<int>(blockIdx.x) * kPerWave >= problem_count) {
        return;
    }
    const int sub = threadIdx.x / 4;
    const int l = threadIdx.x % 4;
    const int problem = blockIdx.x * kPerWave + sub;
    const int group = problem / d.models;
    bool valid = problem < problem_count;
    int n = 0;
    if (valid) {
        valid = (group_flags[group] & kFlagModelled) != 0;
        n = problem_dims[group];
    }
    const float* in = problems + static_cast<size_t>(problem) * problem_stride * problem_stride;
    float a[kSlots][kN];
    float v[kSlots][kN];
    float scale = 0.0F;
#pragma unroll
    for (int k = 0; k < kSlots; ++k) {
        const int r = 4 * k + l;
#pragma unroll
        for (int c = 0; c < kN; ++c) {
            float value = 0.0F;
            if (valid && r < n && c < n) {
                value = in[r * problem_stride + c];
                scale = fmaxf(scale, fabsf(value));
            }
            a[k][c] = value;
            v[k][c] = r == c ? 1.0F : 0.0F;
        }
    }
    scale = fmaxf(scale, xor16<1>(scale));
    scale = fmaxf(scale, xor16<2>(scale));
    const float threshold = (64.0F * FLT_EPSILON) * (scale > 1.0F ? scale : 1.0F);
    const auto offdiag_max = [&]() {
        float value = 0.0F;
#pragma unroll
        for (int k = 0; k < kSlots; ++k) {
#pragma unroll
            for (int c = 0; c < kN; ++c) {
                if (c / 4 == k) {
                    value = fmaxf(value, l == c % 4 ? 0.0F : fabsf(a[k][c]));
                } else {
                    value = fmaxf(value, fabsf(a[k][c]));
                }
            }
        }
        value = fmaxf(value, xor16<1>(value));
        return fmaxf(value, xor16<2>(value));
    };
    bool done = !valid || n <= 1;
    bool converged = true;
    int sweeps = 0;
#pragma nounroll
    for (int sweep = 0; sweep < d.max_sweeps; ++sweep) {
        if (!done) {
            sweeps = sweep + 1;
        }
        const float off = offdiag_max();
        if (!done && off <= threshold) {
            done = true;
        }
        if (__all(done)) {
            break;
        }
        quad_sweep<kSlots>(a, v, l, !done, threshold, std::make_integer_sequence<int, kN>{});
    }
    const float final_off = offdiag_max();
    if (!done) {
        sweeps = d.max_sweeps;
        converged = final_off <= 8.0F * threshold;
    }
    quad_output<kSlots>(a, v, l, valid, n, d.rank, problem_stride,
                        vectors + static_cast<size_t>(problem) * d.rank * problem_stride,
                        eigenvalues + static_cast<size_t>(problem) * d.rank,
                        std::make_integer_sequence<int, kN>{});
    if (valid && l == 0) {
        status[problem] = sweeps | (converged ? 0 : (1 << 16));
    }
}

// Larger problems, 64 / kLP per wavefront: lane x holds rows x (and x + 64,
// kRows = 2).  A lives in LDS, both symmetric copies of an entry kept equal;
// the running entries A[r][p], the diagonal and V stay in registers.  The
// next column's entries are read one rotation ahead (only the row of the
// current q changes in between, and its entry comes from the lane of row
// q + 1), so a rotation waits for its pivot and its arithmetic only: no
// barriers, no LDS round trip.  V takes a row's rotations after the row is
// finished, from a log (lane q holds rotation (p, q)), so that every register
// index is a constant.  Entries of row p are junk while it runs (see above);
// rows and columns past n are zero and never rotate.  LDS holds A alone: a
// 100-row problem takes 40400 bytes, four per compute unit.  Bound by the
// chain of a rotation (pivot, divide, roots, pivot).  Measured against one
// workgroup of a lane per row with A and V in LDS and two barriers a
// rotation: 983 problems of 100 rows 57.5 -> 16.5 ms, 1.4 k of 60 rows 8.95
// -> 4.50 ms, 62 k of 17 rows 8.3 -> 3.9 ms, 53 k of 32 rows 18.3 -> 12.6 ms.
constexpr float kNoRotation = 2.0F;  // log entry: a rotation's c is at most 1

__host__ __device__ inline int jacobi_row_stride(int problem_stride) { return problem_stride | 1; }
__host__ __device__ inline size_t jacobi_problem_floats(int problem_stride) {
    return static_cast<size_t>(problem_stride) * jacobi_row_stride(problem_stride);
}

// LDS accesses of one wavefront stay in program order; the compiler has to
// keep them there.
__device__ inline void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Value of row q (uniform) of the problem, one register per row.
template <int kLP, int kRows> __device__ inline float row_value(const float (&v)[kRows], int q, bool upper) {
    if constexpr (kLP == 32) {
        const int lo = __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[0]), q);
        const int hi = __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[0]), 32 + q);
        return __builtin_bit_cast(float, upper ? hi : lo);
    } else if constexpr (kRows == 2) {
        const int lo = __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[0]), q & 63);
        const int hi = __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[1]), q & 63);
        return __builtin_bit_cast(float, q < 64 ? lo : hi);
    } else {
        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v[0]), q));
    }
}

template <int kLP, int kRows>
__global__ __launch_bounds__(64) void jacobi_wave_kernel(
    StageDesc d, const int* __restrict__ group_count_dev, int problem_stride,
    const int* __restrict__ group_flags, const int* __restrict__ problem_dims,
    const float* __restrict__ problems, float* __restrict__ eigenvalues,
    float* __restrict__ vectors, int* __restrict__ status) {
    constexpr int kN = kLP * kRows;
    constexpr int kPerWave = 64 / kLP;
    extern __shared__ __attribute__((aligned(16))) float s_jacobi[];
    const int problem_count = *group_count_dev * d.models;
    if (static_cast<int>(blockIdx.x) * kPerWave >= problem_count) {
        return;
    }
    const int sub = threadIdx.x / kLP;
    const bool upper = sub != 0;
    const int lane = threadIdx.x % kLP;
    const int problem = blockIdx.x * kPerWave + sub;
    const int group = problem / d.models;
    bool valid = problem < problem_count;
    int n = 0;
    if (valid) {
        valid = (group_flags[group] & kFlagModelled) != 0;
        n = problem_dims[group];
    }
    const int stride = jacobi_row_stride(problem_stride);
    float* m = s_jacobi + sub * jacobi_problem_floats(problem_stride);
    const float* in = problems + static_cast<size_t>(problem) * problem_stride * problem_stride;
    // Rows past the matrix (lanes x >= problem_stride) read row 0 and never
    // write.
    int row[kRows];
    bool in_matrix[kRows];
    float* mine[kRows];
    float diag[kRows];
    float v[kRows][kN];
    float scale = 0.0F;
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        row[k] = lane + k * 64;
        in_matrix[k] = row[k] < problem_stride;
        mine[k] = m + (in_matrix[k] ? row[k] : 0) * stride;
        diag[k] = 0.0F;
#pragma unroll
        for (int c = 0; c < kN; ++c) {
            v[k][c] = row[k] == c ? 1.0F : 0.0F;
        }
    }
    // Rows of the input are read by the whole problem's lanes.
    for (int r = 0; r < problem_stride; ++r) {
        for (int c = lane; c < problem_stride; c += kLP) {
            float value = 0.0F;
            if (valid && r < n && c < n) {
                value = in[r * problem_stride + c];
                scale = fmaxf(scale, fabsf(value));
            }
            m[r * stride + c] = value;
        }
    }
    for (int offset = kLP / 2; offset >= 1; offset >>= 1) {
        scale = fmaxf(scale, __shfl_xor(scale, offset, kLP));
    }
    const float threshold = (64.0F * FLT_EPSILON) * (scale > 1.0F ? scale : 1.0F);
    wave_lds_order();
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        if (in_matrix[k]) {
            diag[k] = mine[k][row[k]];
        }
    }
    const int rows_max = __builtin_amdgcn_readfirstlane(wave_max_int(n));
    const auto offdiag_max = [&]() {
        float value = 0.0F;
        wave_lds_order();
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if (row[k] < n) {
                for (int c = 0; c < n; ++c) {
                    value = fmaxf(value, c != row[k] ? fabsf(mine[k][c]) : 0.0F);
                }
            }
        }
        for (int offset = kLP / 2; offset >= 1; offset >>= 1) {
            value = fmaxf(value, __shfl_xor(value, offset, kLP));
        }
        return value;
    };
    bool done = !valid || n <= 1;
    bool converged = true;
    int sweeps = 0;
#pragma nounroll
    for (int sweep = 0; sweep < d.max_sweeps; ++sweep) {
        if (!done) {
            sweeps = sweep + 1;
        }
        const float off = offdiag_max();
        if (!done && off <= threshold) {
            done = true;
        }
        if (__all(done)) {
            break;
        }
#pragma nounroll
        for (int p = 0; p + 1 < rows_max; ++p) {
            float rp[kRows];
            float column[kRows];
            float log_c[kRows];
            float log_s[kRows];
#pragma unroll
            for (int k = 0; k < kRows; ++k) {
                rp[k] = mine[k][p];
                column[k] = mine[k][p + 1];
                log_c[k] = kNoRotation;
                log_s[k] = 0.0F;
            }
            wave_lds_order();
            float app = row_value<kLP, kRows>(diag, p, upper);
            bool any = false;
#pragma nounroll
            for (int q = p + 1; q < rows_max; ++q) {
                const int ahead = q + 1 < rows_max ? q + 1 : q;
                float next[kRows];
#pragma unroll
                for (int k = 0; k < kRows; ++k) {
                    next[k] = mine[k][ahead];
                }
                wave_lds_order();
                const float apq = row_value<kLP, kRows>(rp, q, upper);
                const float aqq = row_value<kLP, kRows>(diag, q, upper);
                const bool rotate = !done && fabsf(apq) > threshold;
                if (rotate) {
                    any = true;
                    const Rotation o = rotation_of(app, aqq, apq);
                    app = o.new_pp;
#pragma unroll
                    for (int k = 0; k < kRows; ++k) {
                        rotate_pair(o, rp[k], column[k]);
                        if (in_matrix[k]) {
                            mine[k][q] = column[k];
                            m[q * stride + row[k]] = column[k];
                        }
                        const bool own = row[k] == q;
                        rp[k] = own ? 0.0F : rp[k];
                        diag[k] = own ? o.new_qq : diag[k];
                        log_c[k] = own ? o.c : log_c[k];
                        log_s[k] = own ? o.s : log_s[k];
                    }
                }
                // Row q's entry of the next column is the one row q + 1 has
                // just taken (the same value where nothing rotated).
                const float fresh = row_value<kLP, kRows>(column, ahead, upper);
#pragma unroll
                for (int k = 0; k < kRows; ++k) {
                    column[k] = row[k] == q && rotate ? fresh : next[k];
                }
                wave_lds_order();
            }
            // Row and column p.
#pragma unroll
            for (int k = 0; k < kRows; ++k) {
                if (row[k] == p) {
                    diag[k] = app;
                } else if (in_matrix[k]) {
                    mine[k][p] = rp[k];
                    m[p * stride + row[k]] = rp[k];
                }
            }
            wave_lds_order();
            if (!__any(any)) {
                continue;
            }
            float vp[kRows];
#pragma unroll
            for (int c = 0; c < kN; ++c) {
                if (c == p) {
#pragma unroll
                    for (int k = 0; k < kRows; ++k) {
                        vp[k] = pinned(v[k][c]);
                    }
                }
            }
#pragma unroll
            for (int c = 1; c < kN; ++c) {
                const Rotation o{row_value<kLP, kRows>(log_c, c, upper), row_value<kLP, kRows>(log_s, c, upper),
                                 0.0F, 0.0F};
                if (o.c != kNoRotation) {
#pragma unroll
                    for (int k = 0; k < kRows; ++k) {
                        rotate_pair(o, vp[k], v[k][c]);
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < kN; ++c) {
                if (c == p) {
#pragma unroll
                    for (int k = 0; k < kRows; ++k) {
                        v[k][c] = pinned(vp[k]);
                    }
                }
            }
            wave_lds_order();
        }
    }
    const float final_off = offdiag_max();
    if (!done) {
        sweeps = d.max_sweeps;
        converged = final_off <= 8.0F * threshold;
    }
    // Stable descending order of the diagonal, then V, in A's place.  Lane x
    // writes eigenpair x (the rank is at most 64, and at most n).
    float* diagonal = m;
    int* order = reinterpret_cast<int*>(m + problem_stride);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        if (in_matrix[k]) {
            diagonal[row[k]] = diag[k];
        }
    }
    __syncthreads();
    for (int r = lane; valid && r < n; r += kLP) {
        order[descending_place(diagonal, n, r)] = r;
    }
    __syncthreads();
    const bool writes = valid && lane < d.rank && lane < n;
    const int col = writes ? order[lane] : 0;
    const float value = writes ? diagonal[col] : 0.0F;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        if (in_matrix[k]) {
#pragma unroll
            for (int c = 0; c < kN; ++c) {
                if (c < problem_stride) {
                    mine[k][c] = v[k][c];
                }
            }
        }
    }
    __syncthreads();
    if (writes) {
        write_eigenvector(m, stride, n, col,
                          vectors + (static_cast<size_t>(problem) * d.rank + lane) * problem_stride);
        eigenvalues[static_cast<size_t>(problem) * d.rank + lane] = value;
    }
    if (valid && lane == 0) {
        status[problem] = sweeps | (converged ? 0 : (1 << 16));
    }
}

// ---------------------------------------------------------------------------
// parallel-order Jacobi (FAST form)
// ---------------------------------------------------------------------------

// Column pair (j, j ^ k) of the relative row: column x = r ^ j pairs with
// x ^ k and takes the rotation of lane x.  Both lanes of a pair hold the
// same c and opposite sigma, so lane x ^ k's values are c and -sigma of lane
// x: one exchange per column pair instead of two.
template <int kK, int kJ>
__device__ inline void rotate_columns(float (&a)[16], float (&v)[16], const float (&b)[16], float c,
                                      float sigma) {
    constexpr int kHigh = kK >= 8 ? 8 : (kK >= 4 ? 4 : (kK >= 2 ? 2 : 1));
    if constexpr ((kJ & kHigh) == 0) {
        constexpr int kJJ = kJ ^ kK;
        const float c0 = xor16<kJ>(c);
        const float s0 = xor16<kJ>(sigma);
        const float c1 = c0;
        const float s1 = -s0;
        const float v0 = v[kJ];
        const float v1 = v[kJJ];
        a[kJ] = fmaf(s0, b[kJJ], c0 * b[kJ]);
        a[kJJ] = fmaf(s1, b[kJ], c1 * b[kJJ]);
        v[kJ] = fmaf(s0, v1, c0 * v0);
        v[kJJ] = fmaf(s1, v0, c1 * v1);
    }
}

template <int kK, int... kJ>
__device__ inline void rotate_rows_and_columns(float (&a)[16], float (&v)[16], float c, float sigma,
                                               std::integer_sequence<int, kJ...>) {
    // Rows: B[r][.] = c A[r][.] + sigma A[r ^ k][.]; the partner's
    // A[r ^ k][r ^ j] is its a[j ^ k].
    float b[16];
    ((b[kJ] = fmaf(sigma, xor16<kK>(a[kJ ^ kK]), c * a[kJ])), ...);
    (rotate_columns<kK, kJ>(a, v, b, c, sigma), ...);
}

// One rotation round of the parallel ordering for problems of at most 16
// rows: in round k every index r is paired with r ^ k (rounds 1..15 cover
// each pair exactly once per sweep), and the eight disjoint rotations of a
// problem are applied together as A <- J^T A J, V <- V J.  Lane r of a
// 16-lane row holds row r of A and V in relative order, a[j] = A[r][r ^ j],
// so the diagonal is a[0], the pivot A[r][r ^ k] is a[k] and every register
// index and lane exchange is a compile-time constant.  The rotation is that
// of the cyclic solver (jacobi_rotate, linalg.cpp:153-202) with hardware
// reciprocal and square-root approximations; both lanes of a pair compute it
// from the lower index's values, so they agree bit for bit.  Rounds in which
// no problem of the wavefront rotates are skipped.
template <int kK>
__device__ inline void parallel_round(float (&a)[16], float (&v)[16], int r, bool active,
                                      float threshold) {
    constexpr int kHigh = kK >= 8 ? 8 : (kK >= 4 ? 4 : (kK >= 2 ? 2 : 1));
    const bool is_p = (r & kHigh) == 0;  // r is the lower index of its pair
    const float own_diag = a[0];
    const float own_off = a[kK];
    const float partner_diag = xor16<kK>(own_diag);
    const float partner_off = xor16<kK>(own_off);
    const float app = is_p ? own_diag : partner_diag;
    const float aqq = is_p ? partner_diag : own_diag;
    const float apq = is_p ? own_off : partner_off;
    const bool rotate = active && fabsf(apq) > threshold;
    if (!__any(rotate)) {
        return;
    }
    // Branch-free: every lane evaluates the rotation (apq is replaced by 1
    // where no rotation happens), then selects.
    const float safe_apq = rotate ? apq : 1.0F;
    const float tau = (aqq - app) * __builtin_amdgcn_rcpf(2.0F * safe_apq);
    const float tau_abs = fabsf(tau);
    const float t_abs = __builtin_amdgcn_rcpf(tau_abs + __builtin_amdgcn_sqrtf(1.0F + (tau * tau)));
    const float t = tau < 0.0F ? -t_abs : t_abs;
    const float c_rot = __builtin_amdgcn_rsqf(1.0F + (t * t));
    const float s_rot = t * c_rot;
    const float cc = c_rot * c_rot;
    const float ss = s_rot * s_rot;
    const float two_cs = 2.0F * (c_rot * s_rot);
    const float new_pp = ((cc * app) - (two_cs * apq)) + (ss * aqq);
    const float new_qq = ((ss * app) + (two_cs * apq)) + (cc * aqq);
    const float c = rotate ? c_rot : 1.0F;
    // -s for the lower index, +s for the upper one.
    const float sigma = rotate ? (is_p ? -s_rot : s_rot) : 0.0F;
    const float new_diag = is_p ? new_pp : new_qq;
    rotate_rows_and_columns<kK>(a, v, c, sigma, std::make_integer_sequence<int, 16>{});
    a[0] = rotate ? new_diag : a[0];
    a[kK] = rotate ? 0.0F : a[kK];
    // Rounds are scheduled one after the other (bounded register use).
    __builtin_amdgcn_sched_barrier(0);
}

template <int... kKs>
__device__ inline void parallel_sweep(float (&a)[16], float (&v)[16], int r, bool active,
                                      float threshold) {
    (parallel_round<kKs>(a, v, r, active, threshold), ...);
}

// Same sweep structure and canonical vectors as the cyclic kernels above, with the
// parallel ordering above: 16 lanes per problem, four per wavefront.  The
// sweeps stop once every off-diagonal entry is at most 2^-14 of
// max(1, max |A|) (the exact form stops at 64 float epsilons, about 2^-17):
// the sweeps this saves (7 % of the solver's time on 16-row models) only
// refine eigenpairs already within the fast form's tolerance (eigenvalues
// within 1e-3 of the largest, checked against the fp64 oracle).
__global__ __launch_bounds__(64) void jacobi_parallel_kernel(
    StageDesc d, const int* __restrict__ group_count_dev, int problem_stride,
    const int* __restrict__ group_flags, const int* __restrict__ problem_dims,
    const float* __restrict__ problems, float* __restrict__ eigenvalues, float* __restrict__ vectors,
    int* __restrict__ status, float refine_gap, int* __restrict__ refine_list,
    int* __restrict__ refine_count) {
    const int problem_count = *group_count_dev * d.models;
    constexpr int kPerWave = 4;
    constexpr int kStride = 17;
    __shared__ float s_v[kPerWave][16 * kStride];
    __shared__ float s_diag[kPerWave][16];
    __shared__ int s_order[kPerWave][16];

    const int sub = threadIdx.x / 16;
    const int r = threadIdx.x % 16;
    const int problem = blockIdx.x * kPerWave + sub;
    const int group = problem / d.models;
    bool valid = problem < problem_count;
    int n = 0;
    if (valid) {
        valid = (group_flags[group] & kFlagModelled) != 0;
        n = problem_dims[group];
    }
    const float* in = problems + static_cast<size_t>(problem) * problem_stride * problem_stride;
    float a[16];
    float v[16];
    float row_max = 0.0F;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int col = r ^ j;
        float value = 0.0F;
        if (valid && r < n && col < n) {
            value = in[r * problem_stride + col];
            row_max = fmaxf(row_max, fabsf(value));
        }
        a[j] = value;
        v[j] = j == 0 ? 1.0F : 0.0F;
    }
    row_max = fmaxf(row_max, xor16<8>(row_max));
    row_max = fmaxf(row_max, xor16<4>(row_max));
    row_max = fmaxf(row_max, xor16<2>(row_max));
    row_max = fmaxf(row_max, xor16<1>(row_max));
    const float matrix_scale = row_max > 1.0F ? row_max : 1.0F;
    const float threshold = 0x1p-14F * matrix_scale;

    const auto offdiag_max = [&]() {
        float value = 0.0F;
#pragma unroll
        for (int j = 1; j < 16; ++j) {
            value = fmaxf(value, fabsf(a[j]));
        }
        value = fmaxf(value, xor16<8>(value));
        value = fmaxf(value, xor16<4>(value));
        value = fmaxf(value, xor16<2>(value));
        value = fmaxf(value, xor16<1>(value));
        return value;
    };

    bool done = !valid || n <= 1;
    bool converged = true;
    int sweeps = 0;
#pragma nounroll
    for (int sweep = 0; sweep < d.max_sweeps; ++sweep) {
        if (!done) {
            sweeps = sweep + 1;
        }
        const float off = offdiag_max();
        if (!done && off <= threshold) {
            done = true;
        }
        if (__all(done)) {
            break;
        }
        parallel_sweep<1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15>(a, v, r, !done, threshold);
    }
    const float final_off = offdiag_max();
    if (!done) {
        sweeps = d.max_sweeps;
        converged = final_off <= 8.0F * threshold;
    }

    // V[r][r ^ j] = v[j] into LDS; the diagonal in row order.
    float* vs = s_v[sub];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        vs[r * kStride + (r ^ j)] = v[j];
    }
    s_diag[sub][r] = a[0];
    __syncthreads();
    if (valid && r < n) {
        s_order[sub][descending_place(s_diag[sub], n, r)] = r;
    }
    __syncthreads();
    if (valid && r < d.rank && r < n) {
        const int col = s_order[sub][r];
        float* vec_out = vectors + (static_cast<size_t>(problem) * d.rank + r) * problem_stride;
        float norm_squared = 0.0F;
        float max_abs = 0.0F;
        int pivot = 0;
        for (int i = 0; i < n; ++i) {
            const float value = vs[i * kStride + col];
            norm_squared = norm_squared + value * value;
            const float value_abs = fabsf(value);
            if (value_abs > max_abs) {
                max_abs = value_abs;
                pivot = i;
            }
        }
        float scale = 1.0F;
        const bool rescale = norm_squared > FLT_MIN;
        if (rescale) {
            scale = 1.0F / sqrtf(norm_squared);
            if (vs[pivot * kStride + col] < 0.0F) {
                scale = -scale;
            }
        }
        for (int i = 0; i < n; ++i) {
            const float value = vs[i * kStride + col];
            vec_out[i] = rescale ? value * scale : value;
        }
        eigenvalues[static_cast<size_t>(problem) * d.rank + r] = s_diag[sub][col];
    }
    if (valid && r == 0) {
        status[problem] = sweeps | (converged ? 0 : (1 << 16));
        // A rank cutoff inside the spectrum whose gap is small against the
        // largest eigenvalue: the kept subspace is re-solved in fp64.
        const int rank = d.rank;
        if (rank < n && rank > 0 && refine_list != nullptr) {
            const float top = fabsf(s_diag[sub][s_order[sub][0]]);
            const float gap = s_diag[sub][s_order[sub][rank - 1]] - s_diag[sub][s_order[sub][rank]];
            if (!(gap >= refine_gap * fmaxf(top, FLT_MIN))) {
                refine_list[atomicAdd(refine_count, 1)] = problem;
            }
        }
    }
}

// The parallel ordering in double with the full-precision operations, for
// the re-solve below (same layout and rounds as parallel_round).
template <int kK, int kJ>
__device__ __forceinline__ void rotate_columns_double(double (&a)[16], double (&v)[16], const double (&b)[16],
                                                      double c, double sigma) {
    constexpr int kHigh = kK >= 8 ? 8 : (kK >= 4 ? 4 : (kK >= 2 ? 2 : 1));
    if constexpr ((kJ & kHigh) == 0) {
        constexpr int kJJ = kJ ^ kK;
        const double c0 = xor16<kJ>(c);
        const double s0 = xor16<kJ>(sigma);
        const double v0 = v[kJ];
        const double v1 = v[kJJ];
        a[kJ] = fma(s0, b[kJJ], c0 * b[kJ]);
        a[kJJ] = fma(-s0, b[kJ], c0 * b[kJJ]);
        v[kJ] = fma(s0, v1, c0 * v0);
        v[kJJ] = fma(-s0, v0, c0 * v1);
    }
}

template <int kK, int... kJ>
__device__ __forceinline__ void parallel_round_double(double (&a)[16], double (&v)[16], int r, bool active,
                                                      double threshold, std::integer_sequence<int, kJ...>) {
    constexpr int kHigh = kK >= 8 ? 8 : (kK >= 4 ? 4 : (kK >= 2 ? 2 : 1));
    const bool is_p = (r & kHigh) == 0;
    const double partner_diag = xor16<kK>(a[0]);
    const double partner_off = xor16<kK>(a[kK]);
    const double app = is_p ? a[0] : partner_diag;
    const double aqq = is_p ? partner_diag : a[0];
    const double apq = is_p ? a[kK] : partner_off;
    const bool rotate = active && fabs(apq) > threshold;
    if (!__any(rotate)) {
        return;
    }
    const double tau = (aqq - app) / (2.0 * (rotate ? apq : 1.0));
    const double t_abs = 1.0 / (fabs(tau) + sqrt(1.0 + tau * tau));
    const double t = tau < 0.0 ? -t_abs : t_abs;
    const double c_rot = 1.0 / sqrt(1.0 + t * t);
    const double s_rot = t * c_rot;
    const double cc = c_rot * c_rot;
    const double ss = s_rot * s_rot;
    const double two_cs = 2.0 * (c_rot * s_rot);
    const double new_pp = ((cc * app) - (two_cs * apq)) + (ss * aqq);
    const double new_qq = ((ss * app) + (two_cs * apq)) + (cc * aqq);
    const double c = rotate ? c_rot : 1.0;
    const double sigma = rotate ? (is_p ? -s_rot : s_rot) : 0.0;
    double b[16];
    ((b[kJ] = fma(sigma, xor16<kK>(a[kJ ^ kK]), c * a[kJ])), ...);
    (rotate_columns_double<kK, kJ>(a, v, b, c, sigma), ...);
    a[0] = rotate ? (is_p ? new_pp : new_qq) : a[0];
    a[kK] = rotate ? 0.0 : a[kK];
    __builtin_amdgcn_sched_barrier(0);
}

template <int... kKs>
__device__ __forceinline__ void parallel_sweep_double(double (&a)[16], double (&v)[16], int r, bool active,
                                                      double threshold) {
    (parallel_round_double<kKs>(a, v, r, active, threshold, std::make_integer_sequence<int, 16>{}), ...);
}

// fp64 re-solve of the flagged problems (Jacobi in double, the reference's
// solver at its double instantiation, linalg.cpp:447-550: same rotation,
// threshold 64 eps max(1, max|A|) with the double eps, stopping rule, ordering
// and canonical vectors; the pairs in the parallel order), results rounded to
// float.  Sixteen lanes per problem, four problems per wavefront at a time,
// A and V in registers; the list length is read on the device, so no host
// round trip is needed.  Bound by double-precision issue: the eight
// rotations of a round share one divide and root chain.  Measured against
// one problem per wavefront in the cyclic order with A and V in LDS: a
// 501x283x6 YUV clip at rank 4, 443 us per half stage -> 76 us per stage.
__global__ __launch_bounds__(64) void jacobi_refine_kernel(
    StageDesc d, int problem_stride, const int* __restrict__ problem_dims,
    const float* __restrict__ problems, const int* __restrict__ refine_list,
    const int* __restrict__ refine_count, float* __restrict__ eigenvalues,
    float* __restrict__ vectors, int* __restrict__ refined_total) {
    constexpr int kN = 16;
    constexpr int kPerWave = 4;
    constexpr int kStride = kN + 1;
    __shared__ double s_v[kPerWave][kN * kStride];
    __shared__ double s_diag[kPerWave][kN];
    __shared__ int s_order[kPerWave][kN];
    const int sub = threadIdx.x / kN;
    const int r = threadIdx.x % kN;
    const int total = *refine_count;
    if (blockIdx.x == 0 && threadIdx.x == 0 && refined_total != nullptr) {
        atomicAdd(refined_total, total);
    }
    for (int first = blockIdx.x * kPerWave; first < total; first += gridDim.x * kPerWave) {
        const bool valid = first + sub < total;
        const int problem = refine_list[valid ? first + sub : first];
        const int n = problem_dims[problem / d.models];
        const float* in = problems + static_cast<size_t>(problem) * problem_stride * problem_stride;
        double a[kN];
        double v[kN];
        double scale = 0.0;
#pragma unroll
        for (int j = 0; j < kN; ++j) {
            const int col = r ^ j;
            double value = 0.0;
            if (r < n && col < n) {
                value = static_cast<double>(in[r * problem_stride + col]);
                scale = fmax(scale, fabs(value));
            }
            a[j] = value;
            v[j] = j == 0 ? 1.0 : 0.0;
        }
        const auto problem_max = [](double value) {
            value = fmax(value, xor16<8>(value));
            value = fmax(value, xor16<4>(value));
            value = fmax(value, xor16<2>(value));
            return fmax(value, xor16<1>(value));
        };
        scale = problem_max(scale);
        const double threshold = (64.0 * DBL_EPSILON) * (scale > 1.0 ? scale : 1.0);
        bool done = !valid || n <= 1;
#pragma nounroll
        for (int sweep = 0; sweep < d.max_sweeps; ++sweep) {
            double off = 0.0;
#pragma unroll
            for (int j = 1; j < kN; ++j) {
                off = fmax(off, fabs(a[j]));
            }
            done = done || problem_max(off) <= threshold;
            if (__all(done)) {
                break;
            }
            parallel_sweep_double<1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15>(a, v, r, !done, threshold);
        }
        __syncthreads();  // the previous problems' vectors are written
#pragma unroll
        for (int j = 0; j < kN; ++j) {
            s_v[sub][r * kStride + (r ^ j)] = v[j];
        }
        s_diag[sub][r] = a[0];
        __syncthreads();
        if (valid && r < n) {
            s_order[sub][descending_place(s_diag[sub], n, r)] = r;
        }
        __syncthreads();
        if (valid && r < d.rank && r < n) {
            const int col = s_order[sub][r];
            const double* vs = s_v[sub];
            float* vec_out = vectors + (static_cast<size_t>(problem) * d.rank + r) * problem_stride;
            double norm_squared = 0.0;
            double max_abs = 0.0;
            int pivot = 0;
            for (int i = 0; i < n; ++i) {
                const double value = vs[i * kStride + col];
                norm_squared += value * value;
                if (fabs(value) > max_abs) {
                    max_abs = fabs(value);
                    pivot = i;
                }
            }
            double scale_out = 1.0;
            const bool rescale = norm_squared > DBL_MIN;
            if (rescale) {
                scale_out = 1.0 / sqrt(norm_squared);
                if (vs[pivot * kStride + col] < 0.0) {
                    scale_out = -scale_out;
                }
            }
            for (int i = 0; i < n; ++i) {
                const double value = vs[i * kStride + col];
                vec_out[i] = static_cast<float>(rescale ? value * scale_out : value);
            }
            eigenvalues[static_cast<size_t>(problem) * d.rank + r] = static_cast<float>(s_diag[sub][col]);
        }
    }
}

}  // namespace

hipError_t launch_jacobi(const StageDesc& d, const int* group_count_dev, int problem_capacity,
                         int problem_stride, const int* group_flags, const int* problem_dims,
                         const float* problems, float* eigenvalues, float* vectors,
                         int* status, hipStream_t stream) {
    if (problem_capacity <= 0) {
        return hipSuccess;
    }
    const int n = problem_stride;
#define VNLBHIP_JACOBI(KERNEL, PER, SHARED)                                                     \
    hipLaunchKernelGGL((KERNEL), dim3(static_cast<unsigned>((problem_capacity + PER - 1) / PER)), \
                       dim3(64), SHARED, stream, d, group_count_dev, problem_stride,            \
                       group_flags, problem_dims, problems, eigenvalues, vectors, status)
    if (n > 128) {
        return hipErrorInvalidValue;
    }
    // Up to 16 rows the wavefront's rotations are bound by issue, and four
    // lanes per problem share them among 16 problems (128 registers of A and
    // V a lane at 16 rows; 32 rows would take 512): see the figures at
    // jacobi_quad_kernel.  Above, one or two problems per wavefront with A in
    // LDS (figures at jacobi_wave_kernel's comment).
    const size_t shared = jacobi_problem_floats(n) * sizeof(float);
    if (n <= 4) {
        VNLBHIP_JACOBI(jacobi_quad_kernel<1>, 16, 0);
    } else if (n <= 8) {
        VNLBHIP_JACOBI(jacobi_quad_kernel<2>, 16, 0);
    } else if (n <= 12) {
        VNLBHIP_JACOBI(jacobi_quad_kernel<3>, 16, 0);
    } else if (n <= 16) {
        VNLBHIP_JACOBI(jacobi_quad_kernel<4>, 16, 0);
    } else if (n <= 32) {
        VNLBHIP_JACOBI((jacobi_wave_kernel<32, 1>), 2, 2 * shared);
    } else if (n <= 64) {
        VNLBHIP_JACOBI((jacobi_wave_kernel<64, 1>), 1, shared);
    } else {
        VNLBHIP_JACOBI((jacobi_wave_kernel<64, 2>), 1, shared);
    }
#undef VNLBHIP_JACOBI
    return hipGetLastError();
}

}  // namespace vnlbhip

namespace vnlbhip {

bool jacobi_parallel_supported(int problem_stride) {
    return problem_stride <= 16;
}

hipError_t launch_jacobi_parallel(const StageDesc& d, const int* group_count_dev, int problem_capacity,
                                  int problem_stride, const int* group_flags, const int* problem_dims,
                                  const float* problems, float* eigenvalues, float* vectors,
                                  int* status, float refine_gap, int* refine_list, int* refine_count,
                                  int* refined_total, hipStream_t stream) {
    if (problem_capacity <= 0) {
        return hipSuccess;
    }
    if (!jacobi_parallel_supported(problem_stride)) {
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(jacobi_parallel_kernel, dim3(static_cast<unsigned>((problem_capacity + 3) / 4)),
                       dim3(64), 0, stream, d, group_count_dev, problem_stride, group_flags,
                       problem_dims, problems, eigenvalues, vectors, status, refine_gap, refine_list,
                       refine_count);
    if (refine_list != nullptr && d.rank > 0) {
        const int blocks = problem_capacity < 2048 ? problem_capacity : 2048;
        hipLaunchKernelGGL(jacobi_refine_kernel, dim3(static_cast<unsigned>(blocks)), dim3(64), 0, stream, d,
                           problem_stride, problem_dims, problems, refine_list, refine_count, eigenvalues,
                           vectors, refined_total);
    }
    return hipGetLastError();
}

}  // namespace vnlbhip
