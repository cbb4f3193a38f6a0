// The MoE block for float32 checkpoints (a model whose tensors are all f32, as the reference's
// Hugging Face fixture: gen_tiny.py:235-274 writes it in f32 because MLX runs the dense gather_mm
// only in f32). The reference then computes every op of SparseMoe::forward (moe.rs:149-174) in
// f32: nothing is rounded to bf16, and the SwiGLU's casts (activations.rs:64-66) are identities.
//
// Every output element is one wave's dot product over float4 loads, with a fixed reduction order, so
// a row's result does not depend on the batch. Widths of up to 2048, with a shared expert as wide as
// the routed ones or none, run f32_group_kernel: a wave keeps ND weight rows in registers (64 of them
// at most) and takes the rows of a tile that meets them, one after the other, so an expert's weights
// are read once per tile of 8 to 64 of its rows, not once per pair (bound by streaming them: the
// Qwen3.6-like block in f32 holds 12.6 MB per expert). Tiles, because a wave takes about 0.6 us per
// row: with all of an expert's rows in one wave, 16 experts of width 256 x 128 took 590 us at T = 2048
// (537 as single dot products, 134 in tiles of 8). Other blocks run f32_rows_kernel, one dot product
// per wave, whose bits are the same.
#include "common.hpp"
#include "kernels.hpp"

namespace mrun {

namespace {

// f32 sum over the wave by a fixed butterfly (every lane ends with the same value).
__device__ __forceinline__ float wave_sum_f32(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// lane's part of a . w over K (float4 chunks lane, lane + 64, ...; K a multiple of 4)
__device__ __forceinline__ float dot_part(const float *__restrict__ a, const float *__restrict__ w,
                                          int K, int lane) {
    float acc = 0.f;
    for (int c = lane; c < K / 4; c += 64) {
        const float4 x = ((const float4 *)a)[c], y = ((const float4 *)w)[c];
        acc = __builtin_fmaf(x.x, y.x, acc);
        acc = __builtin_fmaf(x.y, y.y, acc);
        acc = __builtin_fmaf(x.z, y.z, acc);
        acc = __builtin_fmaf(x.w, y.w, acc);
    }
    return acc;
}

__device__ __forceinline__ float sigmoid_f32(float z) { return 1.0f / (1.0f + expf(-z)); }

// out[r][n] = A[r / a_div] . W[e_r][n] (e_r = ids ? ids[r] : 0), or under GLU
// silu(A . W0[e_r][n]) * (A . W1[e_r][n]). One wave per (r, n): 4 columns per workgroup, rows
// strided over grid.y.
template <bool GLU>
__global__ __launch_bounds__(256) void f32_rows_kernel(F32Rows j) {
    const int lane = threadIdx.x & 63;
    const int n = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (n >= j.N) return;
    for (int r = blockIdx.y; r < j.R; r += gridDim.y) {
        const int e = j.ids ? (int)j.ids[r] : 0;
        const float *a = j.A + (size_t)(r / j.a_div) * j.K;
        const size_t wr = ((size_t)e * j.N + n) * j.K;
        const float g = wave_sum_f32(dot_part(a, j.W0 + wr, j.K, lane));
        float v = g;
        if (GLU) {
            const float u = wave_sum_f32(dot_part(a, j.W1 + wr, j.K, lane));
            v = (g * sigmoid_f32(g)) * u;
        }
        if (lane == 0) j.out[(size_t)r * j.N + n] = v;
    }
}

// The sums over the wave of ND values per lane (ND = 2, 4 or 8), each by the butterfly of
// wave_sum_f32 (lanes 32, 16, 8, 4, 2, 1 apart: the same additions, so the same bits). The first
// log2(ND) steps halve the values instead of keeping every sum in every lane: the lane ends with
// value  bit 5 + 2 bit 4 + 4 bit 3  of its number (the low log2(ND) of these bits).
template <int ND>
__device__ __forceinline__ float wave_sums(const float (&v)[ND], int lane) {
    float w[ND / 2];
#pragma unroll
    for (int i = 0; i < ND / 2; ++i) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[2 * i]),
                                                        __float_as_uint(v[2 * i + 1]), false, false);
        w[i] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
    }
    float x[ND > 2 ? ND / 4 : 1];
#pragma unroll
    for (int i = 0; i < (ND > 2 ? ND / 4 : 1); ++i) {
        const uint32_t a = __float_as_uint(w[ND > 2 ? 2 * i : 0]), b = __float_as_uint(w[ND > 2 ? 2 * i + 1 : 0]);
        const auto s = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        x[i] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
    }
    float y;
    if constexpr (ND == 8) {
        const bool b3 = (lane & 8) != 0;
        const float keep = b3 ? x[1] : x[0], send = b3 ? x[0] : x[1];
        y = keep + __uint_as_float(dpp_u32<0x128>(__float_as_uint(send)));
    } else {
        y = x[0] + __uint_as_float(dpp_u32<0x128>(__float_as_uint(x[0])));
    }
    // 4 apart: banks 0 and 2 read lane + 4, banks 1 and 3 lane - 4
    int m = __builtin_amdgcn_update_dpp(0, __float_as_int(y), 0x104, 0xF, 0x5, false);
    m = __builtin_amdgcn_update_dpp(m, __float_as_int(y), 0x114, 0xF, 0xA, false);
    y += __int_as_float(m);
    y += __uint_as_float(dpp_u32<0x4E>(__float_as_uint(y)));
    y += __uint_as_float(dpp_u32<0xB1>(__float_as_uint(y)));
    return y;
}

// The products of F32Group (kernels.hpp). Slot blockIdx.y: first the plain rows in pieces of
// j.piece, then the experts' tiles (or single pairs). A wave owns NW = ND (glu: ND / 2) output columns.
template <bool GLU, int NC, int ND>
__global__ __launch_bounds__(256) void f32_group_kernel(F32Group j) {
    constexpr int NW = GLU ? ND / 2 : ND;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n0 = (blockIdx.x * 4 + wave) * NW, K = j.K;
    const int cols = j.N + (j.xW ? 1 : 0);
    if (n0 >= cols) return;
    int s = blockIdx.y, p0, rows;
    const float *A, *W0, *W1;
    float *out;
    const uint32_t *map = nullptr;
    int a_div = 1;
    if (s < j.plain_slots) {
        p0 = s * j.piece, rows = min(j.piece, j.plain_rows - p0);
        A = j.pA, W0 = j.pW0, W1 = j.pW1, out = j.pout;
    } else {
        s -= j.plain_slots;
        int e;
        if (j.tiles) {
            if (s >= (int)*j.n_tiles) return;
            e = (int)j.tiles[3 * s], p0 = (int)j.tiles[3 * s + 1], rows = (int)j.tiles[3 * s + 2];
            map = j.order;
        } else {
            e = (int)j.ids[s], p0 = s, rows = 1;
        }
        A = j.A, out = j.out, a_div = j.a_div;
        const size_t w = (size_t)e * j.N * K;
        W0 = j.W0 + w, W1 = GLU ? j.W1 + w : nullptr;
    }
    // this lane's part of the weight rows (value i: under glu column i / 2's gate and up rows)
    float4 w[ND][NC];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const int n = n0 + (GLU ? i / 2 : i);
        const float *row = (GLU && (i & 1) ? W1 : W0) + (size_t)min(n, j.N - 1) * K;
        if (!GLU && j.xW && n == j.N) row = j.xW;
#pragma unroll
        for (int c = 0; c < NC; ++c)
            w[i][c] = lane + 64 * c < K / 4 ? ((const float4 *)row)[lane + 64 * c] : float4{};
    }
    const int fi = (lane >> 5) | (ND > 2 ? (lane >> 3) & 2 : 0) | (ND > 4 ? (lane >> 1) & 4 : 0);
    for (int r0 = 0; r0 < rows; r0 += 64) {
        const int nr = min(64, rows - r0);
        int pos = p0 + r0 + min(lane, nr - 1);  // lane l: row r0 + l
        if (map) pos = (int)map[pos];
        const int arow = pos / a_div;
        for (int r = 0; r < nr; ++r) {
            const float4 *x = (const float4 *)(A + (size_t)__builtin_amdgcn_readlane(arow, r) * K);
            float v[ND];
#pragma unroll
            for (int i = 0; i < ND; ++i) v[i] = 0.f;
            float4 xv[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) xv[c] = lane + 64 * c < K / 4 ? x[lane + 64 * c] : float4{};
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int i = 0; i < ND; ++i) {
                    v[i] = __builtin_fmaf(xv[c].x, w[i][c].x, v[i]);
                    v[i] = __builtin_fmaf(xv[c].y, w[i][c].y, v[i]);
                    v[i] = __builtin_fmaf(xv[c].z, w[i][c].z, v[i]);
                    v[i] = __builtin_fmaf(xv[c].w, w[i][c].w, v[i]);
                }
            float y = wave_sums<ND>(v, lane);
            const size_t orow = (size_t)__builtin_amdgcn_readlane(pos, r);
            if (GLU) {  // gates in lanes 0-31, ups in lanes 32-63
                const float u = __shfl_xor(y, 32, 64);
                y = (y * sigmoid_f32(y)) * u;
            }
            const int n = n0 + (GLU ? fi >> 1 : fi);
            // one lane per value: those whose other bits are zero
            const int own = ND == 2 ? 31 : ND == 4 ? 15 : 7;
            if ((lane & own) == 0 && !(GLU && lane >= 32)) {
                if (n < j.N) out[orow * j.N + n] = y;
                else if (!GLU && n < cols) j.xout[orow] = y;
            }
        }
    }
}

// Softmax and top-k of one token per wave: gates = exp(l - max) / sum; the k largest gates, equal
// gates by lower id, in rank order; scores = gates, or gates / (their sum in rank order) with norm.
__global__ __launch_bounds__(64) void f32_topk_kernel(const float *__restrict__ logits, int T,
                                                      int E, int k, int norm,
                                                      uint32_t *__restrict__ ids,
                                                      float *__restrict__ scores) {
    constexpr int NPER = 8;  // E <= 512
    const int t = blockIdx.x, lane = threadIdx.x;
    if (t >= T) return;
    const float *l = logits + (size_t)t * E;
    float v[NPER];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < NPER; ++i) {
        const int e = lane + 64 * i;
        v[i] = e < E ? l[e] : -INFINITY;
        m = fmaxf(m, v[i]);
    }
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) m = fmaxf(m, __shfl_xor(m, s, 64));
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < NPER; ++i) {
        v[i] = lane + 64 * i < E ? expf(v[i] - m) : 0.f;
        sum += v[i];
    }
    sum = wave_sum_f32(sum);
    // keys: gate bits (non-negative floats order as integers) over 0xffffffff - id
    uint64_t key[NPER];
#pragma unroll
    for (int i = 0; i < NPER; ++i) {
        const int e = lane + 64 * i;
        const float g = v[i] / sum;
        key[i] = e < E ? ((uint64_t)__float_as_uint(g) << 32) | (uint64_t)(0xffffffffu - (uint32_t)e)
                       : 0ull;
    }
    float tot = 0.f;
    uint64_t mine = 0;
    for (int j = 0; j < k; ++j) {
        uint64_t b = key[0];
#pragma unroll
        for (int i = 1; i < NPER; ++i) b = key[i] > b ? key[i] : b;
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) {
            const uint64_t o = __shfl_xor(b, s, 64);
            b = o > b ? o : b;
        }
#pragma unroll
        for (int i = 0; i < NPER; ++i) key[i] = key[i] == b ? 0ull : key[i];
        tot += __uint_as_float((uint32_t)(b >> 32));  // in rank order
        if (lane == j) mine = b;
    }
    if (lane < k) {
        const float g = __uint_as_float((uint32_t)(mine >> 32));
        ids[(size_t)t * k + lane] = 0xffffffffu - (uint32_t)(mine & 0xffffffffu);
        scores[(size_t)t * k + lane] = norm ? g / tot : g;
    }
}

// out[t][d] = sum_j y[t k + j][d] * scores[t k + j] (j ascending), plus, with a shared expert,
// sigmoid(glogit[t]) * shared[t][d].
__global__ __launch_bounds__(256) void f32_combine_kernel(const float *__restrict__ y,
                                                          const float *__restrict__ scores, int T,
                                                          int k, int D,
                                                          const float *__restrict__ glogit,
                                                          const float *__restrict__ shared,
                                                          float *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)T * D) return;
    const size_t t = i / D, d = i % D;
    float acc = 0.f;
    for (int j = 0; j < k; ++j) acc += y[(t * k + j) * D + d] * scores[t * k + j];
    if (shared) acc += sigmoid_f32(glogit[t]) * shared[i];
    out[i] = acc;
}

}  // namespace

hipError_t launch_f32_rows(const F32Rows &j, bool glu, hipStream_t stream) {
    if (j.R <= 0 || j.N <= 0) return hipSuccess;
    if (j.K % 4 != 0 || j.a_div < 1) return hipErrorInvalidValue;
    dim3 grid((j.N + 3) / 4, j.R < 65535 ? j.R : 65535);
    if (glu) f32_rows_kernel<true><<<grid, 256, 0, stream>>>(j);
    else f32_rows_kernel<false><<<grid, 256, 0, stream>>>(j);
    return hipGetLastError();
}

// Weight rows per wave by input width, so that a wave holds at most 64 registers of weights.
static int group_nd(int K) { return K > 1024 ? 2 : K > 512 ? 4 : 8; }

int f32_group_blocks(int K, int N, bool glu) {
    const int cols = 4 * (glu ? group_nd(K) / 2 : group_nd(K));
    return (N + cols - 1) / cols;
}

template <bool GLU>
static void run_group(const F32Group &j, int slots, hipStream_t s) {
    const dim3 grid(f32_group_blocks(j.K, j.N + (j.xW ? 1 : 0), GLU), slots);
    if (j.K > 1024) f32_group_kernel<GLU, 8, 2><<<grid, 256, 0, s>>>(j);
    else if (j.K > 512) f32_group_kernel<GLU, 4, 4><<<grid, 256, 0, s>>>(j);
    else f32_group_kernel<GLU, 2, 8><<<grid, 256, 0, s>>>(j);
}

bool f32_group_supported(int K) { return K % 4 == 0 && K <= 2048; }

hipError_t launch_f32_group(const F32Group &j0, int max_slots, bool glu, hipStream_t stream) {
    F32Group j = j0;
    j.plain_slots = j.plain_rows > 0 ? (j.plain_rows + j.piece - 1) / j.piece : 0;
    const int slots = j.plain_slots + max_slots;
    if (slots == 0 || j.N <= 0) return hipSuccess;
    if (!f32_group_supported(j.K) || slots > kF32GroupMaxSlots || (glu && j.xW)) return hipErrorInvalidValue;
    if (glu) run_group<true>(j, slots, stream);
    else run_group<false>(j, slots, stream);
    return hipGetLastError();
}

hipError_t launch_f32_topk(const float *logits, int T, int E, int k, bool norm, uint32_t *ids,
                           float *scores, hipStream_t stream) {
    if (T <= 0) return hipSuccess;
    if (E > 512 || k > E || k < 1) return hipErrorInvalidValue;
    f32_topk_kernel<<<T, 64, 0, stream>>>(logits, T, E, k, norm ? 1 : 0, ids, scores);
    return hipGetLastError();
}

hipError_t launch_f32_combine(const float *y, const float *scores, int T, int k, int D,
                              const float *glogit, const float *shared, float *out,
                              hipStream_t stream) {
    const size_t n = (size_t)T * D;
    if (n == 0) return hipSuccess;
    f32_combine_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(y, scores, T, k, D, glogit,
                                                                       shared, out);
    return hipGetLastError();
}

}  // namespace mrun
