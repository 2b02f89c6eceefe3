// Training and scoring kernels of the learned candidate proposer (the network
// and its features are described in proposer.h).
//
// Training minimises, over groups of rows (one anchor's candidates each),
// the listwise loss -sum_r t_r log softmax(s)_r with targets t summing to 1
// per group (the exact k nearest of the plain matcher share the mass).
// Matrix products run on the matrix cores (v_mfma_f32_16x16x32_bf16: bf16
// operands, fp32 accumulation) in one generic tiled kernel; the fp32 master
// weights take Adam steps and are copied to bf16 for the products.
#include <algorithm>
#include <cfloat>

#include "kernels.h"
#include "proposer.h"

namespace vnlbhip {
namespace {

constexpr int kGemmTile = 64;
constexpr int kGemmK = 32;
constexpr int kGemmPitch = kGemmK + 8;  // bf16 per staged row (16-byte pad)

__device__ inline uint64_t splitmix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// He-uniform weights (limit sqrt(6 / fan_in)), zero biases; the output
// weights at a tenth of that so the first scores are small.
__global__ void init_kernel(float* __restrict__ params, uint64_t seed) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= kPropParams) {
        return;
    }
    const double u = static_cast<double>(splitmix64(seed ^ (0xA24BAED4963EE407ull * (i + 1))) >> 11) *
                     (1.0 / 9007199254740992.0);
    float limit = 0.0F;
    if (i < kOffB1) {
        limit = sqrtf(6.0F / kPropIn);
    } else if (i >= kOffW2 && i < kOffB2) {
        limit = sqrtf(6.0F / kPropHidden);
    } else if (i >= kOffW3 && i < kOffB3) {
        limit = 0.1F * sqrtf(6.0F / kPropHidden);
    }
    params[i] = static_cast<float>((2.0 * u - 1.0) * limit);
}

__global__ void to_bf16_kernel(const float* __restrict__ src, __bf16* __restrict__ dst, int count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) {
        dst[i] = static_cast<__bf16>(src[i]);
    }
}

// One input row per thread from global memory (channel 0 of the clip).
__global__ void features_kernel(const float* __restrict__ clip, int width, int height, int channels,
                                int patch_time, const uint32_t* __restrict__ anchors,
                                const uint32_t* __restrict__ candidates, int rows, __bf16* __restrict__ out) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) {
        return;
    }
    const uint32_t a = anchors[r];
    const uint32_t c = candidates[r];
    const size_t plane = static_cast<size_t>(width) * height;
    float am[kPropBoxes];
    float cm[kPropBoxes];
    for (int t = 0; t < patch_time; ++t) {
        const float* ap = clip + (static_cast<size_t>(position_frame(a) + t) * channels) * plane +
                          static_cast<size_t>(position_y(a)) * width + position_x(a);
        const float* cp = clip + (static_cast<size_t>(position_frame(c) + t) * channels) * plane +
                          static_cast<size_t>(position_y(c)) * width + position_x(c);
        patch_box_means(ap, width, am + 16 * t);
        patch_box_means(cp, width, cm + 16 * t);
    }
    float x[kPropIn];
    proposer_features(am, cm, 16 * patch_time, position_x(c) - position_x(a), position_y(c) - position_y(a),
                      position_frame(c) - position_frame(a), x);
    __bf16* row = out + static_cast<size_t>(r) * kPropIn;
    for (int k = 0; k < kPropIn; ++k) {
        row[k] = static_cast<__bf16>(x[k]);
    }
}

// Eight consecutive operand elements as bf16 (fp32 ones rounded to nearest
// even), from a 16-byte aligned address.
__device__ inline prop_bf16x8 load8(const __bf16* p) { return *reinterpret_cast<const prop_bf16x8*>(p); }
__device__ inline prop_bf16x8 load8(const float* p) {
    const prop_floatx4 lo = *reinterpret_cast<const prop_floatx4*>(p);
    const prop_floatx4 hi = *reinterpret_cast<const prop_floatx4*>(p + 4);
    prop_bf16x8 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        out[i] = static_cast<__bf16>(lo[i]);
        out[4 + i] = static_cast<__bf16>(hi[i]);
    }
    return out;
}

// This thread's eight elements of a staged 64 x 32 operand tile (rows
// i0 .. i0 + 63, k0 .. k0 + 31).  kAlongK: the operand is [i][k] with k
// contiguous (extent k_end a multiple of 32, rows past `extent` are zero);
// else it is [k][i] with i contiguous (extent a multiple of 64, k past k_end
// is zero).
template <bool kAlongK, class T>
__device__ inline prop_bf16x8 tile_load(const T* __restrict__ p, int ld, int i0, int extent, int k0, int k_end) {
    const int i = kAlongK ? i0 + (threadIdx.x >> 2) : i0 + (threadIdx.x & 7) * 8;
    const int k = kAlongK ? k0 + (threadIdx.x & 3) * 8 : k0 + (threadIdx.x >> 3);
    prop_bf16x8 zero{};
    if (kAlongK) {
        return i < extent ? load8(p + static_cast<size_t>(i) * ld + k) : zero;
    }
    return k < k_end ? load8(p + static_cast<size_t>(k) * ld + i) : zero;
}

template <bool kAlongK>
__device__ inline void tile_store(__bf16* __restrict__ s, const prop_bf16x8& v) {
    if constexpr (kAlongK) {
        *reinterpret_cast<prop_bf16x8*>(s + (threadIdx.x >> 2) * kGemmPitch + (threadIdx.x & 3) * 8) = v;
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            s[((threadIdx.x & 7) * 8 + j) * kGemmPitch + (threadIdx.x >> 3)] = v[j];
        }
    }
}

// C[m][n] = sum_k A(m, k) B(k, n), operands rounded to bf16 when staged;
// kAK: A is [m][k], else [k][m]; kBK: B is [n][k], else [k][n] (leading
// dimensions lda, ldb; see tile_load for the extents).  64 x 64 output
// tiles, four waves of 32 x 32; the next k step's operands are loaded (16
// bytes per load) while this one is on the matrix cores.  Epilogue: +
// bias[n] when given, zero where mask[m][n] <= 0 when given; fp32 result to
// c32 (ldc) and/or relu(result) as bf16 to c16.
//
// Split K: workgroup z sums k in [z per_split, (z + 1) per_split) into
// c32 + z M ldc.  The weight gradients contract over the batch's rows (8192
// for 64 anchors) into 256 x 256 and 256 x 128 results, 16 and 8 tiles for
// 256 compute units: unsplit, each of them took 1.3 ms of latency-bound
// steps; with 32 splits and the step pipeline the two average 14 us.
template <bool kAK, bool kBK, class TA, class TB>
__global__ __launch_bounds__(256) void gemm_kernel(int M, int N, int K, int per_split, const TA* __restrict__ a,
                                                   int lda, const TB* __restrict__ b, int ldb,
                                                   const float* __restrict__ bias, const float* __restrict__ mask,
                                                   float* __restrict__ c32, __bf16* __restrict__ c16, int ldc) {
    __shared__ __attribute__((aligned(16))) __bf16 s_a[kGemmTile * kGemmPitch];
    __shared__ __attribute__((aligned(16))) __bf16 s_b[kGemmTile * kGemmPitch];
    const int m0 = blockIdx.y * kGemmTile;
    const int n0 = blockIdx.x * kGemmTile;
    const int k_begin = blockIdx.z * per_split;
    const int k_end = min(K, k_begin + per_split);
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int col = lane & 15;
    const int kb = lane >> 4;
    const int wm = (wave >> 1) * 32;
    const int wn = (wave & 1) * 32;
    prop_floatx4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            acc[i][j] = prop_floatx4{0.0F, 0.0F, 0.0F, 0.0F};
        }
    }
    prop_bf16x8 ra{};
    prop_bf16x8 rb{};
    if (k_begin < k_end) {
        ra = tile_load<kAK>(a, lda, m0, M, k_begin, k_end);
        rb = tile_load<kBK>(b, ldb, n0, N, k_begin, k_end);
    }
    for (int k0 = k_begin; k0 < k_end; k0 += kGemmK) {
        tile_store<kAK>(s_a, ra);
        tile_store<kBK>(s_b, rb);
        __syncthreads();
        if (k0 + kGemmK < k_end) {
            ra = tile_load<kAK>(a, lda, m0, M, k0 + kGemmK, k_end);
            rb = tile_load<kBK>(b, ldb, n0, N, k0 + kGemmK, k_end);
        }
        prop_bf16x8 av[2];
        prop_bf16x8 bv[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            av[i] = *reinterpret_cast<const prop_bf16x8*>(s_a + (wm + 16 * i + col) * kGemmPitch + 8 * kb);
            bv[i] = *reinterpret_cast<const prop_bf16x8*>(s_b + (wn + 16 * i + col) * kGemmPitch + 8 * kb);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    float* __restrict__ out32 = c32 + static_cast<size_t>(blockIdx.z) * M * ldc;
    // acc[i][j][v] = C[wm + 16 i + 4 kb + v][wn + 16 j + col]
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + wn + 16 * j + col;
        if (n >= N) {
            continue;
        }
        const float add = bias != nullptr ? bias[n] : 0.0F;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = m0 + wm + 16 * i + 4 * kb + v;
                if (m < M) {
                    const size_t at = static_cast<size_t>(m) * ldc + n;
                    float z = acc[i][j][v] + add;
                    if (mask != nullptr && !(mask[at] > 0.0F)) {
                        z = 0.0F;
                    }
                    out32[at] = z;
                    if (c16 != nullptr) {
                        c16[at] = static_cast<__bf16>(z > 0.0F ? z : 0.0F);
                    }
                }
            }
        }
    }
}

// s[m] = sum_n relu(z2[m][n]) w3[n] + b3 (one wave per row; lane l sums
// units 4 l .. 4 l + 3 in order, then a butterfly over the wave).
__global__ void output_kernel(const float* __restrict__ z2, const float* __restrict__ params, int rows,
                              float* __restrict__ s) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= rows) {
        return;
    }
    const float* w3 = params + kOffW3;
    float sum = 0.0F;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int n = 4 * lane + q;
        const float z = z2[static_cast<size_t>(r) * kPropHidden + n];
        sum = sum + (z > 0.0F ? z : 0.0F) * w3[n];
    }
    for (int offset = 32; offset >= 1; offset >>= 1) {
        sum = sum + __shfl_xor(sum, offset, 64);
    }
    if (lane == 0) {
        s[r] = sum + params[kOffB3];
    }
}

// Listwise loss per group (one wave per group): ds = (softmax(s) - t) / G,
// loss_out[g] = -sum t log softmax(s).
__global__ void loss_kernel(const float* __restrict__ s, const float* __restrict__ targets, int groups,
                            int group, float* __restrict__ ds, float* __restrict__ loss_out) {
    const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (g >= groups) {
        return;
    }
    const float* sg = s + static_cast<size_t>(g) * group;
    const float* tg = targets + static_cast<size_t>(g) * group;
    float mx = -FLT_MAX;
    for (int r = lane; r < group; r += 64) {
        mx = fmaxf(mx, sg[r]);
    }
    mx = wave_max(mx);
    float z = 0.0F;
    for (int r = lane; r < group; r += 64) {
        z = z + expf(sg[r] - mx);
    }
    for (int offset = 32; offset >= 1; offset >>= 1) {
        z = z + __shfl_xor(z, offset, 64);
    }
    const float log_z = logf(z);
    const float inv_groups = 1.0F / static_cast<float>(groups);
    float loss = 0.0F;
    for (int r = lane; r < group; r += 64) {
        const float logp = sg[r] - mx - log_z;
        const float t = tg[r];
        ds[static_cast<size_t>(g) * group + r] = (expf(logp) - t) * inv_groups;
        loss = loss - t * logp;
    }
    for (int offset = 32; offset >= 1; offset >>= 1) {
        loss = loss + __shfl_xor(loss, offset, 64);
    }
    if (lane == 0) {
        loss_out[g] = loss;
    }
}

// Column sums over the batch's rows go through partial sums of row chunks, in
// row order within a chunk; reduce_kernel adds the chunks.
constexpr int kColChunkRows = 32;
constexpr int kColMaxChunks = 512;

__host__ __device__ inline int column_chunk_rows(int rows) {
    const int per = (rows + kColMaxChunks - 1) / kColMaxChunks;
    return per > kColChunkRows ? per : kColChunkRows;
}

// Output layer's backward: dz2[m][n] = ds[m] w3[n] (z2 > 0), and the chunk's
// partial sums of dw3[n] = sum relu(z2) ds and db2[n] = sum dz2 (thread n,
// one workgroup per row chunk).
__global__ __launch_bounds__(kPropHidden) void output_grad_kernel(const float* __restrict__ z2,
                                                                  const float* __restrict__ ds,
                                                                  const float* __restrict__ params, int rows,
                                                                  float* __restrict__ dz2,
                                                                  float* __restrict__ part_w3,
                                                                  float* __restrict__ part_b2) {
    const int n = threadIdx.x;
    const int per = column_chunk_rows(rows);
    const int lo = blockIdx.x * per;
    const int hi = min(rows, lo + per);
    const float w3 = params[kOffW3 + n];
    float sum_w3 = 0.0F;
    float sum_b2 = 0.0F;
#pragma unroll 8
    for (int m = lo; m < hi; ++m) {
        const float z = z2[static_cast<size_t>(m) * kPropHidden + n];
        const float g = ds[m];
        const float d = z > 0.0F ? g * w3 : 0.0F;
        sum_w3 = sum_w3 + (z > 0.0F ? z : 0.0F) * g;
        sum_b2 = sum_b2 + d;
        dz2[static_cast<size_t>(m) * kPropHidden + n] = d;
    }
    part_w3[static_cast<size_t>(blockIdx.x) * kPropHidden + n] = sum_w3;
    part_b2[static_cast<size_t>(blockIdx.x) * kPropHidden + n] = sum_b2;
}

// The chunk's partial sums of db1[n] = sum dz1.
__global__ __launch_bounds__(kPropHidden) void column_partial_kernel(const float* __restrict__ a, int rows,
                                                                     float* __restrict__ part) {
    const int n = threadIdx.x;
    const int per = column_chunk_rows(rows);
    const int lo = blockIdx.x * per;
    const int hi = min(rows, lo + per);
    float sum = 0.0F;
#pragma unroll 8
    for (int m = lo; m < hi; ++m) {
        sum = sum + a[static_cast<size_t>(m) * kPropHidden + n];
    }
    part[static_cast<size_t>(blockIdx.x) * kPropHidden + n] = sum;
}

// Adds the partial results of a batch into the flat gradient, every sum in a
// fixed order: the splits of dW2 and dW1 (one element per thread), the row
// chunks of dw3, db2 and db1 (16 columns x 16 chunk runs per workgroup) and
// db3 = sum ds (the last workgroup).
constexpr int kReduceWeightBlocks = kPropHidden * (kPropHidden + kPropIn) / 256;
constexpr int kReduceColumnBlocks = 3 * kPropHidden / 16;
__global__ __launch_bounds__(256) void reduce_kernel(const float* __restrict__ part_weights, int splits,
                                                     const float* __restrict__ part_columns, int chunks,
                                                     const float* __restrict__ ds, int rows,
                                                     float* __restrict__ grads) {
    __shared__ float s_part[256];
    const int block = blockIdx.x;
    if (block < kReduceWeightBlocks) {
        int e = block * 256 + threadIdx.x;
        const bool second = e < kPropHidden * kPropHidden;
        const int size = kPropHidden * (second ? kPropHidden : kPropIn);
        const float* p = part_weights;
        if (!second) {
            e -= kPropHidden * kPropHidden;
            p += static_cast<size_t>(splits) * kPropHidden * kPropHidden;
        }
        float sum = 0.0F;
#pragma unroll 8
        for (int z = 0; z < splits; ++z) {
            sum = sum + p[static_cast<size_t>(z) * size + e];
        }
        grads[(second ? kOffW2 : kOffW1) + e] = sum;
        return;
    }
    float sum = 0.0F;
    if (block < kReduceWeightBlocks + kReduceColumnBlocks) {
        const int column = (block - kReduceWeightBlocks) * 16 + (threadIdx.x & 15);
        const int which = column / kPropHidden;
        const int n = column % kPropHidden;
        const float* p = part_columns + static_cast<size_t>(which) * chunks * kPropHidden + n;
#pragma unroll 4
        for (int c = threadIdx.x >> 4; c < chunks; c += 16) {
            sum = sum + p[static_cast<size_t>(c) * kPropHidden];
        }
        s_part[threadIdx.x] = sum;
        __syncthreads();
        if (threadIdx.x < 16) {
            float total = 0.0F;
            for (int g = 0; g < 16; ++g) {
                total = total + s_part[16 * g + threadIdx.x];
            }
            grads[(which == 0 ? kOffW3 : (which == 1 ? kOffB2 : kOffB1)) + n] = total;
        }
        return;
    }
    for (int i = threadIdx.x; i < rows; i += 256) {
        sum = sum + ds[i];
    }
    s_part[threadIdx.x] = sum;
    __syncthreads();
    for (int width = 128; width >= 1; width >>= 1) {
        if (static_cast<int>(threadIdx.x) < width) {
            s_part[threadIdx.x] = s_part[threadIdx.x] + s_part[threadIdx.x + width];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        grads[kOffB3] = s_part[0];
    }
}

__global__ void adam_kernel(float* __restrict__ params, const float* __restrict__ grads, float* __restrict__ m,
                            float* __restrict__ v, int count, float lr, float beta1, float beta2, float eps,
                            float correction1, float correction2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) {
        return;
    }
    const float g = grads[i];
    const float mi = beta1 * m[i] + (1.0F - beta1) * g;
    const float vi = beta2 * v[i] + (1.0F - beta2) * g * g;
    m[i] = mi;
    v[i] = vi;
    params[i] = params[i] - lr * (mi / correction1) / (sqrtf(vi / correction2) + eps);
}

// Scores of rows of inputs with the inference tile (the matcher's code).
template <bool kFp8>
__global__ __launch_bounds__(256) void scores_kernel(const __bf16* __restrict__ x, int rows, ProposerWeights wt,
                                                     float* __restrict__ scores) {
    __shared__ __attribute__((aligned(16))) __bf16 s_x[kPropTile * kPropXPitch];
    __shared__ __attribute__((aligned(16))) __bf16 s_h[kPropTile * kPropHPitch];
    __shared__ float s_partial[4 * 64];
    __shared__ float s_scores[kPropTile];
    const int r0 = blockIdx.x * kPropTile;
    {
        // Thread (r, q) stages inputs 32 q .. 32 q + 31 of row r.
        const int r = threadIdx.x >> 2;
        const int q = threadIdx.x & 3;
        float v[32];
        for (int k = 0; k < 32; ++k) {
            v[k] = r0 + r < rows ? static_cast<float>(x[static_cast<size_t>(r0 + r) * kPropIn + 32 * q + k]) : 0.0F;
        }
        store_features32<kFp8>(s_x, r, 32 * q, v, kFp8 ? wt.fp8.scales + kPropScaleX : nullptr);
    }
    __syncthreads();
    if constexpr (kFp8) {
        proposer_tile_scores_fp8(reinterpret_cast<const uint8_t*>(s_x), reinterpret_cast<uint8_t*>(s_h), s_partial,
                                 s_scores, wt);
    } else {
        proposer_tile_scores(s_x, s_h, s_partial, s_scores, wt);
    }
    if (threadIdx.x < kPropTile && r0 + static_cast<int>(threadIdx.x) < rows) {
        scores[r0 + threadIdx.x] = s_scores[threadIdx.x];
    }
}

// ---- FP8 calibration ----

// x_scale[k] = 224 / max_r |x[r][k]| (1 where the column is zero): half the
// format's range, room for inputs beyond the sample.
__global__ void input_scale_kernel(const __bf16* __restrict__ x, int rows, float* __restrict__ scales) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= kPropIn) {
        return;
    }
    float mx = 0.0F;
    for (int r = 0; r < rows; ++r) {
        mx = fmaxf(mx, fabsf(static_cast<float>(x[static_cast<size_t>(r) * kPropIn + k])));
    }
    scales[kPropScaleX + k] = mx > 0.0F ? 0.5F * kFp8Max / mx : 1.0F;
}

// One row of a weight matrix per block: w'[k] = w[n][k] * fold[k] (fold:
// 1 / x_scale, or none), row scale r = 448 / max |w'| (1 for a zero row),
// out[n][k] = fp8(w'[k] r), inv[n] = 1 / (r * extra) with extra = h_scale
// for W2 (read from scales) or 1.
__global__ __launch_bounds__(256) void quantize_rows_kernel(const float* __restrict__ w, int cols,
                                                            const float* __restrict__ x_scale, int use_h_scale,
                                                            float* __restrict__ scales, int inv_offset,
                                                            uint8_t* __restrict__ out) {
    __shared__ float s_max[4];
    const int n = blockIdx.x;
    const float* row = w + static_cast<size_t>(n) * cols;
    float mx = 0.0F;
    for (int k = threadIdx.x; k < cols; k += blockDim.x) {
        const float v = x_scale != nullptr ? row[k] / x_scale[k] : row[k];
        mx = fmaxf(mx, fabsf(v));
    }
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) {
        s_max[threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    const float row_max = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
    const float r = row_max > 0.0F ? kFp8Max / row_max : 1.0F;
    for (int k = threadIdx.x; k < cols; k += blockDim.x) {
        const float v = x_scale != nullptr ? row[k] / x_scale[k] : row[k];
        out[static_cast<size_t>(n) * cols + k] = to_fp8(v * r);
    }
    if (threadIdx.x == 0) {
        const float extra = use_h_scale != 0 ? scales[kPropScaleH] : 1.0F;
        scales[inv_offset + n] = 1.0F / (r * extra);
    }
}

// h_scale = 224 / max relu(z1) over the sample (one block).
__global__ __launch_bounds__(256) void hidden_scale_kernel(const float* __restrict__ z1, size_t count,
                                                           float* __restrict__ scales) {
    __shared__ float s_max[4];
    float mx = 0.0F;
    for (size_t i = threadIdx.x; i < count; i += blockDim.x) {
        mx = fmaxf(mx, z1[i]);
    }
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) {
        s_max[threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const float m = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
        scales[kPropScaleH] = m > 0.0F ? 0.5F * kFp8Max / m : 1.0F;
    }
}

unsigned blocks_for(size_t count, int threads) {
    return static_cast<unsigned>((count + threads - 1) / threads);
}

// Splits of a contraction over `rows`: at least 256 rows (8 k steps) each,
// at most 32 (512 workgroups for the 256 x 256 result, two per compute
// unit; more only adds partial results to sum).
constexpr int kMaxSplits = 32;
int weight_splits(int rows) {
    return std::clamp(rows / 256, 1, kMaxSplits);
}

template <bool kAK, bool kBK, class TA, class TB>
hipError_t gemm(int M, int N, int K, int splits, const TA* a, int lda, const TB* b, int ldb, const float* bias,
                const float* mask, float* c32, __bf16* c16, int ldc, hipStream_t stream) {
    if ((kAK || kBK) && K % kGemmK != 0) {
        return hipErrorInvalidValue;
    }
    if ((!kAK && M % kGemmTile != 0) || (!kBK && N % kGemmTile != 0)) {
        return hipErrorInvalidValue;
    }
    const int steps = (K + kGemmK - 1) / kGemmK;
    const int per_split = (steps + splits - 1) / splits * kGemmK;
    const dim3 grid(static_cast<unsigned>((N + kGemmTile - 1) / kGemmTile),
                    static_cast<unsigned>((M + kGemmTile - 1) / kGemmTile), static_cast<unsigned>(splits));
    hipLaunchKernelGGL((gemm_kernel<kAK, kBK, TA, TB>), grid, dim3(256), 0, stream, M, N, K, per_split, a, lda, b,
                       ldb, bias, mask, c32, c16, ldc);
    return hipGetLastError();
}

}  // namespace

size_t proposer_workspace_floats(int rows) {
    // z1, z2, dz2, dz1 (fp32 [rows][256]); h1 (bf16 [rows][256], as floats);
    // s, ds; column partials; split partials of dW2 and dW1.
    return static_cast<size_t>(rows) * kPropHidden * 4 + static_cast<size_t>(rows) * kPropHidden / 2 +
           static_cast<size_t>(rows) * 2 + static_cast<size_t>(3) * kColMaxChunks * kPropHidden +
           static_cast<size_t>(weight_splits(rows)) * kPropHidden * (kPropHidden + kPropIn) + 64;
}

hipError_t launch_proposer_init(float* params, uint64_t seed, hipStream_t stream) {
    hipLaunchKernelGGL(init_kernel, dim3(blocks_for(kPropParams, 256)), dim3(256), 0, stream, params, seed);
    return hipGetLastError();
}

hipError_t launch_proposer_refresh(const float* params, __bf16* w1, __bf16* w2, hipStream_t stream) {
    hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(kPropHidden * kPropIn, 256)), dim3(256), 0, stream,
                       params + kOffW1, w1, kPropHidden * kPropIn);
    hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(kPropHidden * kPropHidden, 256)), dim3(256), 0, stream,
                       params + kOffW2, w2, kPropHidden * kPropHidden);
    return hipGetLastError();
}

hipError_t launch_proposer_features(const float* clip, int width, int height, int channels, int patch_time,
                                    const uint32_t* anchors, const uint32_t* candidates, int rows, __bf16* out,
                                    hipStream_t stream) {
    if (rows <= 0) {
        return hipSuccess;
    }
    hipLaunchKernelGGL(features_kernel, dim3(blocks_for(rows, 64)), dim3(64), 0, stream, clip, width, height,
                       channels, patch_time, anchors, candidates, rows, out);
    return hipGetLastError();
}

hipError_t launch_proposer_scores(const __bf16* x, int rows, const ProposerWeights& wt, int precision,
                                  float* scores, hipStream_t stream) {
    if (rows <= 0) {
        return hipSuccess;
    }
    if (precision == 1) {
        if (wt.fp8.w1 == nullptr || wt.fp8.w2 == nullptr || wt.fp8.scales == nullptr) {
            return hipErrorInvalidValue;
        }
        hipLaunchKernelGGL(scores_kernel<true>, dim3(blocks_for(rows, kPropTile)), dim3(256), 0, stream, x, rows, wt,
                           scores);
    } else {
        hipLaunchKernelGGL(scores_kernel<false>, dim3(blocks_for(rows, kPropTile)), dim3(256), 0, stream, x, rows, wt,
                           scores);
    }
    return hipGetLastError();
}

hipError_t launch_proposer_calibrate(const float* params, const __bf16* w1, const __bf16* x, int rows,
                                     float* workspace, uint8_t* w1_fp8, uint8_t* w2_fp8, float* scales,
                                     hipStream_t stream) {
    if (rows <= 0) {
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(input_scale_kernel, dim3(blocks_for(kPropIn, 64)), dim3(64), 0, stream, x, rows, scales);
    hipLaunchKernelGGL(quantize_rows_kernel, dim3(kPropHidden), dim3(256), 0, stream, params + kOffW1, kPropIn,
                       scales + kPropScaleX, 0, scales, kPropScaleW1, w1_fp8);
    // Hidden activations of the sample with the bf16 weights.
    hipError_t e = gemm<true, true>(rows, kPropHidden, kPropIn, 1, x, kPropIn, w1, kPropIn, params + kOffB1,
                                    nullptr, workspace, nullptr, kPropHidden, stream);
    if (e != hipSuccess) {
        return e;
    }
    hipLaunchKernelGGL(hidden_scale_kernel, dim3(1), dim3(256), 0, stream, workspace,
                       static_cast<size_t>(rows) * kPropHidden, scales);
    hipLaunchKernelGGL(quantize_rows_kernel, dim3(kPropHidden), dim3(256), 0, stream, params + kOffW2, kPropHidden,
                       static_cast<const float*>(nullptr), 1, scales, kPropScaleW2, w2_fp8);
    return hipGetLastError();
}

// Forward, loss and gradients of one batch: grads (flat, kPropParams) and
// loss_groups[g] (per group).  w1, w2: the bf16 copies of params.
hipError_t launch_proposer_gradients(const float* params, const __bf16* w1, const __bf16* w2, const __bf16* x,
                                     const float* targets, int rows, int group, float* workspace, float* grads,
                                     float* loss_groups, hipStream_t stream) {
    const size_t wide = static_cast<size_t>(rows) * kPropHidden;
    float* z1 = workspace;
    float* z2 = z1 + wide;
    float* dz2 = z2 + wide;
    float* dz1 = dz2 + wide;
    __bf16* h1 = reinterpret_cast<__bf16*>(dz1 + wide);
    float* s = dz1 + wide + wide / 2;
    float* ds = s + rows;
    const int chunk_rows = column_chunk_rows(rows);
    const int chunks = (rows + chunk_rows - 1) / chunk_rows;
    float* part_columns = ds + rows;  // dw3, db2, db1: [chunks][256] each
    float* part_weights = part_columns + static_cast<size_t>(3) * kColMaxChunks * kPropHidden;
    const int splits = weight_splits(rows);
    float* part_w1 = part_weights + static_cast<size_t>(splits) * kPropHidden * kPropHidden;
    const size_t columns = static_cast<size_t>(chunks) * kPropHidden;
    const int groups = rows / group;
    hipError_t e;
    // Forward.
    if ((e = gemm<true, true>(rows, kPropHidden, kPropIn, 1, x, kPropIn, w1, kPropIn, params + kOffB1, nullptr, z1,
                              h1, kPropHidden, stream)) != hipSuccess) {
        return e;
    }
    if ((e = gemm<true, true>(rows, kPropHidden, kPropHidden, 1, h1, kPropHidden, w2, kPropHidden, params + kOffB2,
                              nullptr, z2, nullptr, kPropHidden, stream)) != hipSuccess) {
        return e;
    }
    hipLaunchKernelGGL(output_kernel, dim3(blocks_for(rows, 4)), dim3(256), 0, stream, z2, params, rows, s);
    hipLaunchKernelGGL(loss_kernel, dim3(blocks_for(groups, 4)), dim3(256), 0, stream, s, targets, groups, group,
                       ds, loss_groups);
    // Output layer: dz2 and the partial sums of dw3 and db2.
    hipLaunchKernelGGL(output_grad_kernel, dim3(static_cast<unsigned>(chunks)), dim3(kPropHidden), 0, stream, z2, ds,
                       params, rows, dz2, part_columns, part_columns + columns);
    // Layer 2: dW2 = dz2^T h1, dz1 = (dz2 W2) where z1 > 0.
    if ((e = gemm<false, false>(kPropHidden, kPropHidden, rows, splits, dz2, kPropHidden, h1, kPropHidden, nullptr,
                                nullptr, part_weights, nullptr, kPropHidden, stream)) != hipSuccess) {
        return e;
    }
    if ((e = gemm<true, false>(rows, kPropHidden, kPropHidden, 1, dz2, kPropHidden, w2, kPropHidden, nullptr, z1,
                               dz1, nullptr, kPropHidden, stream)) != hipSuccess) {
        return e;
    }
    // Layer 1: db1 = column sums of dz1, dW1 = dz1^T x.
    hipLaunchKernelGGL(column_partial_kernel, dim3(static_cast<unsigned>(chunks)), dim3(kPropHidden), 0, stream, dz1,
                       rows, part_columns + 2 * columns);
    if ((e = gemm<false, false>(kPropHidden, kPropIn, rows, splits, dz1, kPropHidden, x, kPropIn, nullptr, nullptr,
                                part_w1, nullptr, kPropIn, stream)) != hipSuccess) {
        return e;
    }
    hipLaunchKernelGGL(reduce_kernel, dim3(kReduceWeightBlocks + kReduceColumnBlocks + 1), dim3(256), 0, stream,
                       part_weights, splits, part_columns, chunks, ds, rows, grads);
    return hipGetLastError();
}

hipError_t launch_proposer_adam(float* params, const float* grads, float* m, float* v, float lr, int step,
                                hipStream_t stream) {
    const float beta1 = 0.9F;
    const float beta2 = 0.999F;
    const float c1 = 1.0F - powf(beta1, static_cast<float>(step));
    const float c2 = 1.0F - powf(beta2, static_cast<float>(step));
    hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(kPropParams, 256)), dim3(256), 0, stream, params, grads, m, v,
                       kPropParams, lr, beta1, beta2, 1e-8F, c1, c2);
    return hipGetLastError();
}

}  // namespace vnlbhip
