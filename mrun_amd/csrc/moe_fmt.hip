// The prefill forward's expert products (SwitchGlu's gate/up with SwiGLU, and down: moe.rs:79-83,
// nuvec.rs:670-697) for the checkpoint formats other than 4-bit group 64 (moe_gemm.hip): 4-bit
// experts in groups of 32 or 128, 8-bit experts in groups of 32, 64 or 128, and dense bf16 experts.
// The shared expert's products are extra tiles of the same launches.
//
// These batches are bound by streaming the experts' weights: at 300 to 1000 tokens of the
// Qwen3.6-like block an expert holds 10 to 30 rows, so a launch reads 0.3 to 1 GB for a few tens
// of GFLOP. The schedule is that of moe_gemm.hip (persistent workgroups of 4 waves, two per CU,
// over (row tile x 256 B rows) items cut into eight per-XCD segments; A and weights go from global
// memory straight into an LDS ring, the next stage in flight while one is computed; the affine
// dequant folded around v_mfma_f32_32x32x16_bf16, no weight rounded), with these differences:
//  - A stage holds 64 or 128 bytes of each weight row: two K steps (of 64) of 4-bit codes, one of
//    8-bit codes, or one of bf16 weights (whole 128-byte lines). Where a stage is at
//    most 24 KB (8-bit codes, and 4-bit ones in 32-row tiles) the ring has three: the scales then
//    go to registers, a chunk ahead, which frees their LDS (block forward, 8-bit T = 1000 and group
//    32 T = 700: 3 % faster than with two). With two stages they stay in LDS (in registers, group 128
//    T = 1200 took 3 % longer).
//  - 8-bit codes become exact bf16 integers (no offset); each dword holds codes i and i + 4 of a
//    block, as the packed A has them. bf16 weights are re-paired the same way and go to the MFMAs
//    without scales, straight into the accumulators.
//  - Groups of 32: the MFMA slots of a K step are assigned so that its first two sub-steps cover
//    the first group and the last two the second (block 2 s + h instead of 4 h + s at sub-step s,
//    lane half h), each with its own partial product; the X sums are per 32 inputs.
//  - Groups of 128: the two K steps of a group apply the same scale; the X sums stay per 64.
//  - The LDS reads of a K step and their wait are one asm statement.
// Measured on the Qwen3.6-like block, whole forwards, against the register-staged GEMM of qgemm.hip
// (64 x 64 tiles, the shared expert in two launches of its own), both in turn: 8-bit experts T = 1000
// 465 -> 262 us, 4-bit group 32 T = 700 540 -> 220, bf16 T = 300 677 -> 328 (1.6 GB of weights:
// 4.9 TB/s, the rate of a large copy).
#include <type_traits>

#include "apack.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "moe_gemm_dev.hpp"

namespace mrun {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Sizes of one instantiation: NMI row fragments of 32 rows per tile, BITS per weight, GROUP inputs
// per scale (64 for bf16 weights, which have none).
template <int NMI, int BITS, int GROUP>
struct FmtCfg {
    static constexpr bool QUANT = BITS != 16;
    static constexpr int KS = BITS == 4 ? 2 : 1;         // K steps of 64 per stage
    static constexpr int A_STEP = NMI * 32 * 128, A_BYTES = KS * A_STEP;
    static constexpr int C_ROW = BITS * 8 * KS;          // bytes of a weight row per stage
    static constexpr int C_BYTES = 256 * C_ROW;
    static constexpr int STAGE = A_BYTES + C_BYTES;
    static constexpr int NSTG = STAGE <= 24576 ? 3 : 2;  // what two workgroups per CU leave room for
    static constexpr int A_PARTS = KS * NMI, C_PARTS = C_BYTES / 4096, PARTS = A_PARTS + C_PARTS;
    static constexpr int C_RPP = 256 / C_PARTS;          // weight rows per copy part
    static constexpr int CH = GROUP == 32 ? 4 : 8;       // K steps per chunk of scales and biases
    static constexpr int XG = GROUP == 32 ? 32 : 64;     // inputs per X sum
    // with three stages a chunk's scales wait in registers, else in LDS: 8 (group 128: 4) per row
    static constexpr bool SREG = NSTG == 3;
    static constexpr int B_BYTES = QUANT ? 4096 : 0, S_BYTES = SREG ? 0 : B_BYTES;
    static constexpr int X_BYTES = QUANT ? 3 * 64 * 16 : 0;
    static constexpr int OFF_S = NSTG * STAGE, OFF_R = OFF_S + 2 * S_BYTES;
    static constexpr int OFF_T = OFF_R + 512, OFF_X = OFF_T + 512, OFF_B = OFF_X + X_BYTES;
    static constexpr int LDS_BYTES = OFF_B + B_BYTES;
    static_assert(LDS_BYTES <= 81920, "two workgroups per CU");
};

// the LDS reads of a K step: A fragments of the four sub-steps (row fragments 4096 bytes apart)
#define FMT_A1                                                                                   \
    "ds_read_b128 %[a00], %[p0]\n\tds_read_b128 %[a01], %[p1]\n\tds_read_b128 %[a02], %[p2]\n\t" \
    "ds_read_b128 %[a03], %[p3]\n\t"
#define FMT_A2                                                                                    \
    FMT_A1                                                                                        \
    "ds_read_b128 %[a10], %[p0] offset:4096\n\tds_read_b128 %[a11], %[p1] offset:4096\n\t"        \
    "ds_read_b128 %[a12], %[p2] offset:4096\n\tds_read_b128 %[a13], %[p3] offset:4096\n\t"
#define FMT_A1_OUT [a00] "=&v"(a[0][0]), [a01] "=&v"(a[0][1]), [a02] "=&v"(a[0][2]), [a03] "=&v"(a[0][3])
#define FMT_A2_OUT                                                                        \
    FMT_A1_OUT, [a10] "=&v"(a[NMI - 1][0]), [a11] "=&v"(a[NMI - 1][1]),                   \
        [a12] "=&v"(a[NMI - 1][2]), [a13] "=&v"(a[NMI - 1][3])
#define FMT_A_IN [p0] "v"(pa[0]), [p1] "v"(pa[1]), [p2] "v"(pa[2]), [p3] "v"(pa[3])
#define FMT_COMMA ,
#define FMT_READ(TEXT, OUTS, ...)                                                              \
    if constexpr (NMI == 2)                                                                    \
        asm volatile(TEXT FMT_A2 "s_waitcnt lgkmcnt(0)" : OUTS, FMT_A2_OUT : FMT_A_IN, __VA_ARGS__); \
    else                                                                                       \
        asm volatile(TEXT FMT_A1 "s_waitcnt lgkmcnt(0)" : OUTS, FMT_A1_OUT : FMT_A_IN, __VA_ARGS__)

// four 8-bit codes of each of two words -> bf16 pairs (code i of w0, code i of w1): integers below
// 256 are exact in bf16, so the top half of their f32 conversion is their bf16
__device__ __forceinline__ u32x4 fmt_expand8(uint32_t w0, uint32_t w1) {
    auto pair = [](float lo, float hi) {
        return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
    };
    u32x4 e;
    e.x = pair((float)(w0 & 0xffu), (float)(w1 & 0xffu));
    e.y = pair((float)((w0 >> 8) & 0xffu), (float)((w1 >> 8) & 0xffu));
    e.z = pair((float)((w0 >> 16) & 0xffu), (float)((w1 >> 16) & 0xffu));
    e.w = pair((float)(w0 >> 24), (float)(w1 >> 24));
    return e;
}

// eight bf16 of a weight row in natural order -> pairs (i, i + 4)
__device__ __forceinline__ u32x4 fmt_pair8(u32x4 v) {
    u32x4 e;
    e.x = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);
    e.y = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);
    e.z = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);
    e.w = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);
    return e;
}

// four group-128 values (two words) as eight group-64 ones
__device__ __forceinline__ u32x4 fmt_dup(uint32_t a, uint32_t b) {
    return u32x4{__builtin_amdgcn_perm(a, a, 0x01000100u), __builtin_amdgcn_perm(a, a, 0x03020302u),
                 __builtin_amdgcn_perm(b, b, 0x01000100u), __builtin_amdgcn_perm(b, b, 0x03020302u)};
}

template <bool GLU, int NMI, int BITS, int GROUP>
__global__ __launch_bounds__(256, 2) void fmt_gemm_kernel(MoeGemmJob j) {
    using C = FmtCfg<NMI, BITS, GROUP>;
    __shared__ __align__(16) char smem[C::LDS_BYTES];
    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int fr = lane & 31, fh = lane >> 5;
    const uint32_t lds0 = lds_offset(smem);

    constexpr int NCOLS = GLU ? 128 : 256, TM = 32 * NMI;
    const int NB = j.N / NCOLS;
    const int s_tiles = j.has_shared ? (j.sh.M + TM - 1) / TM : 0;
    const int r_tiles =
        j.has_routing ? min((int)*j.routing.n_tiles, j.max_tiles) : (j.M + TM - 1) / TM;
    const int total = (s_tiles + r_tiles) * NB;
    const int G0 = (int)(gridDim.x >> 3), xcd = (int)(blockIdx.x & 7), wg = (int)(blockIdx.x >> 3);
    const int seg_lo = (int)((long long)total * xcd / 8);
    const int seg_hi = (int)((long long)total * (xcd + 1) / 8);
    // Up to three items per workgroup: as many workgroups as share the XCD's items evenly (136 items
    // on 64 workgroups: 46 with three each, not 8 with three and 56 with two), for the gate/up
    // products of bf16 weights and of groups of 32. Each workgroup streams whole lines of 256 weight
    // rows (and, for groups of 32, of their scales and biases, 16 bytes of a line at a time), so
    // fewer of them keep those lines in the XCD's L2. Block forwards, us, every workgroup against the
    // even split: Qwen3.6-like, bf16 T = 256 345 -> 325, 768 353 -> 345, group 32 T = 256 209 -> 193,
    // 768 220 -> 209; 128 experts of 2048 x 1024, bf16 T = 128 396 -> 356, group 32 T = 256 217 -> 206;
    // 64 experts of 4096 x 1536, group 32 T = 256 327 -> 299 (but T = 341 343 -> 360, the worst of
    // eight shapes); blocks with an item or less per workgroup the same. The
    // other formats need the loads in flight (8-bit T = 700 236 -> 247 us, group 128 157 -> 163), the
    // down products measured the same, and with more items the last round is a small part (group 32
    // T = 3000 423 -> 435, bf16 T = 2000 490 -> 492).
    constexpr bool EVEN = GLU && (!C::QUANT || GROUP == 32) && BITS != 8;
    const int rounds = (seg_hi - seg_lo + G0 - 1) / G0;
    const int G8 = uni(EVEN && rounds > 1 && rounds <= 3 ? (seg_hi - seg_lo + rounds - 1) / rounds : G0);
    if (EVEN && wg >= G8) return;
    const int n_items = uni(seg_hi - seg_lo > wg ? (seg_hi - seg_lo - wg + G8 - 1) / G8 : 0);
    if (n_items == 0) return;
    const int K = j.K, nks = K / 64, G = K / GROUP, axe = K / C::XG;
    const int total_steps = n_items * nks;  // a multiple of 8
    const uint32_t row_bytes = (uint32_t)(K / 8 * BITS);

    // items, tile records and token rows as in moe_gemm.hip (records one item ahead, slot n % 2)
    struct Item {
        int e, row0, mrows, n0, tile;  // tile: routed tile index (rows from the table), or -1
        bool sh;
    };
    auto item_pos = [&](int n, int &rt, int &cb) __attribute__((always_inline)) {
        const int i = seg_lo + wg + G8 * n;
        rt = uni(i / NB), cb = i - rt * NB;
    };
    auto item_of = [&](int n) __attribute__((always_inline)) {
        int rt, cb;
        item_pos(n, rt, cb);
        Item it;
        it.n0 = cb * NCOLS;
        if (rt < s_tiles) {
            it.sh = true, it.e = 0, it.row0 = rt * TM, it.mrows = min(TM, j.sh.M - it.row0);
            it.tile = -1;
        } else {
            it.sh = false;
            const int r = rt - s_tiles;
            if (j.has_routing) {
                const uint32_t rec = lds0 + C::OFF_T + (uint32_t)(n & 1) * 256;
                uint32_t e, row0, mrows;
                ds_read3_now(rec, rec + 4, rec + 8, e, row0, mrows);
                it.e = uni((int)e), it.row0 = uni((int)row0), it.mrows = uni((int)mrows);
                it.tile = j.tile_rows ? r : -1;
            } else {
                it.e = 0, it.row0 = r * TM, it.mrows = min(TM, j.M - it.row0), it.tile = -1;
            }
        }
        return it;
    };
    auto fetch_rows = [&](int n) __attribute__((always_inline)) {
        if (n >= n_items || wave != 0 || !j.has_routing) return;
        int rt, cb;
        item_pos(n, rt, cb);
        if (rt < s_tiles) return;
        const int r = rt - s_tiles;
        dma4(rsrc_of(j.routing.tiles, 12u * (uint32_t)j.max_tiles), 4u * (uint32_t)lane,
             12u * (uint32_t)r, smem + C::OFF_T + (n & 1) * 256);
        if (j.tile_rows)
            dma4(rsrc_of(j.tile_rows, 4u * (uint32_t)j.max_tiles * (uint32_t)TM),
                 4u * (uint32_t)lane, 4u * (uint32_t)(r * TM), smem + C::OFF_R + (n & 1) * 256);
    };

    // ---- load role: A row ra (and ra + 32), weight row rb of each copy part
    const int ra = wave * 8 + (lane >> 3);
    const uint32_t ua16 = 16u * (uint32_t)((lane & 7) ^ swz_a(ra));
    constexpr int UPR = C::C_ROW / 16;  // 16-byte units of a weight row per stage: 4 or 8
    const int rb = wave * (64 / UPR) + lane / UPR;
    const uint32_t uc16 = 16u * (uint32_t)((lane % UPR) ^ (UPR == 8 ? swz_a(rb) : swz_c(rb)));
    rsrc_t r_a, r_c0, r_c1, r_s0, r_s1;
    uint32_t la0 = 0, la1 = 0, lc = 0, ls0 = 0, ls1 = 0;
    int l_item = 0, l_ks = 0, l_chunk = 0, l_slot = 0;
    u32x4 sn0 = {0u, 0u, 0u, 0u}, sn1 = sn0;  // SREG: this lane's two rows' scales of the load cursor's chunk
    Item li{};   // the load cursor's item, taken over by the compute cursor at its switch
    int lx = 0;  // the load cursor's A row of tile row `lane` (the bias term's X splits)

    auto setup_load = [&](int n) __attribute__((always_inline)) {
        const Item it = item_of(n);
        int r0 = min(ra, it.mrows - 1), r1 = min(ra + 32, it.mrows - 1), r2 = min(lane, it.mrows - 1);
        if (it.tile >= 0) {
            const uint32_t t = lds0 + C::OFF_R + (uint32_t)(n & 1) * 256;
            uint32_t u0, u1, u2;
            ds_read3_now(t + 4 * r0, t + 4 * r1, t + 4 * r2, u0, u1, u2);
            r0 = (int)u0, r1 = (int)u1, r2 = (int)u2;
        } else {
            r0 += it.row0, r1 += it.row0, r2 += it.row0;
        }
        li = it, lx = r2;
        const int lda = it.sh ? j.sh.lda : j.lda;
        r_a = rsrc_of(it.sh ? j.sh.A : j.A);
        la0 = (uint32_t)r0 * (uint32_t)lda * 2u + ua16;
        la1 = (uint32_t)r1 * (uint32_t)lda * 2u + ua16;
        r_c0 = rsrc_of(it.sh ? j.sh.w0.codes : j.w0.codes);
        r_c1 = GLU ? rsrc_of(it.sh ? j.sh.w1.codes : j.w1.codes) : r_c0;
        const uint32_t wrow = (uint32_t)it.e * (uint32_t)j.N + (uint32_t)it.n0;
        lc = (wrow + (uint32_t)rb) * row_bytes + uc16;
        if (C::QUANT && !C::SREG) {  // weight row tid: gate rows then up rows under glu
            const bool up = GLU && wave >= 2;
            r_s0 = rsrc_of(up ? (it.sh ? j.sh.w1.scales : j.w1.scales)
                              : (it.sh ? j.sh.w0.scales : j.w0.scales));
            ls0 = (wrow + (uint32_t)(GLU ? (tid & 127) : tid)) * (uint32_t)G * 2u;
        } else if (C::QUANT) {  // weight rows bro0 + fr and bro1 + fr of the compute role
            r_s0 = rsrc_of(it.sh ? j.sh.w0.scales : j.w0.scales);
            r_s1 = GLU ? rsrc_of(it.sh ? j.sh.w1.scales : j.w1.scales) : r_s0;
            ls0 = (wrow + (uint32_t)((GLU ? 32 : 64) * wave + fr)) * (uint32_t)G * 2u;
            ls1 = GLU ? ls0 : ls0 + 64u * (uint32_t)G;
        }
        fetch_rows(n + 1);
    };
    // copy part p of the load cursor's stage into its ring slot: A (K step p / NMI, row fragment
    // p % NMI), then the weight rows (under glu the gate's half of the parts, then the up's)
    auto issue_part = [&](int p) __attribute__((always_inline)) {
        char *sa = smem + l_slot * C::STAGE, *sc = sa + C::A_BYTES;
        if (p < C::A_PARTS) {
            const int kk = p / NMI, mi = p % NMI;
            dma16(r_a, mi ? la1 : la0, 128u * (uint32_t)(l_ks + kk),
                  sa + kk * C::A_STEP + mi * 4096 + wave * 1024);
        } else {
            const int i = p - C::A_PARTS;
            constexpr int HP = GLU ? C::C_PARTS / 2 : C::C_PARTS;
            dma16(i >= HP ? r_c1 : r_c0, lc,
                  (uint32_t)((i % HP) * C::C_RPP) * row_bytes + (uint32_t)(8 * BITS) * (uint32_t)l_ks,
                  sc + i * 4096 + wave * 1024);
        }
    };
    // a chunk's values of each weight row into LDS: 8 (16 bytes), or for groups of 128 the chunk's
    // 4 as two words 1 KB apart
    auto copy_chunk = [&](rsrc_t r, uint32_t row, int chunk, char *lds) __attribute__((always_inline)) {
        if constexpr (GROUP == 128) {
            dma4(r, row, 8u * (uint32_t)chunk, lds + wave * 256);
            dma4(r, row, 8u * (uint32_t)chunk + 4u, lds + 1024 + wave * 256);
        } else {
            dma16(r, row, 16u * (uint32_t)chunk, lds + wave * 1024);
        }
    };
    auto begin_stage = [&]() __attribute__((always_inline)) {  // before a stage's copies
        if (C::QUANT && l_ks % C::CH == 0) {
            const uint32_t c = (uint32_t)(l_ks / C::CH);
            if constexpr (!C::SREG) {
                copy_chunk(r_s0, ls0, (int)c, smem + C::OFF_S + (l_chunk & 1) * C::S_BYTES);
                ++l_chunk;
            } else if constexpr (GROUP == 128) {
                const u32x2 v0 = __builtin_amdgcn_raw_buffer_load_b64(r_s0, ls0, 8u * c, 0);
                const u32x2 v1 = __builtin_amdgcn_raw_buffer_load_b64(r_s1, ls1, 8u * c, 0);
                sn0.x = v0.x, sn0.y = v0.y, sn1.x = v1.x, sn1.y = v1.y;
            } else {
                sn0 = __builtin_amdgcn_raw_buffer_load_b128(r_s0, ls0, 16u * c, 0);
                sn1 = __builtin_amdgcn_raw_buffer_load_b128(r_s1, ls1, 16u * c, 0);
            }
        }
    };
    // the load cursor's next stage (and item; past the last it stays on that item, in bounds)
    auto advance = [&]() __attribute__((always_inline)) {
        l_slot = l_slot + 1 == C::NSTG ? 0 : l_slot + 1;
        l_ks += C::KS;
        if (l_ks == nks) {
            l_ks = 0;
            if (++l_item < n_items) setup_load(l_item);
        }
    };

    // ---- compute role: rows mi * 32 + fr, weight rows bro0 + fr and bro1 + fr. Sub-step s of lane
    // half h takes k block 4h + s (groups of 32: 2s + h) of a K step; block b sits at position
    // 2 (b % 4) + b / 4 of the packed A row.
    constexpr bool G32 = GROUP == 32;
    uint32_t a_off[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int b = G32 ? 2 * s + fh : 4 * fh + s;
        a_off[s] = lds0 + (uint32_t)(fr * 128 + 16 * ((2 * (b & 3) + (b >> 2)) ^ swz_a(fr)));
    }
    const int bro0 = GLU ? wave * 32 : wave * 64;
    constexpr int DB = (GLU ? 128 : 32);  // bro1 - bro0
    const int bro1 = bro0 + DB;
    // 16-byte unit u of this lane's weight row (same for bro1: the swizzles repeat every 32 rows)
    auto c_unit = [&](int u) __attribute__((always_inline)) {
        return lds0 + (uint32_t)C::A_BYTES + (uint32_t)((bro0 + fr) * C::C_ROW) +
               16u * (uint32_t)(u ^ (UPR == 8 ? swz_a(fr) : swz_c(fr)));
    };
    constexpr int NCA = BITS == 16 || (BITS == 8 && G32) ? 4 : (BITS == 4 && !G32 ? 1 : 2);
    uint32_t c_off[NCA], c_step = 0;
    if constexpr (BITS == 16) {
#pragma unroll
        for (int s = 0; s < 4; ++s) c_off[s] = c_unit(4 * fh + s);
    } else if constexpr (BITS == 8 && G32) {
#pragma unroll
        for (int s = 0; s < 4; ++s) c_off[s] = c_unit(s) + 8u * (uint32_t)fh;
    } else if constexpr (BITS == 8) {
        c_off[0] = c_unit(2 * fh), c_off[1] = c_unit(2 * fh + 1);
    } else if constexpr (G32) {
        c_off[0] = c_unit(0), c_off[1] = c_unit(1);
        c_step = c_unit(2) - c_off[0];  // the second K step's units 2, 3 (u ^ 2 moves by +-32)
    } else {
        c_off[0] = c_unit(fh);
        c_step = c_unit(2 + fh) - c_off[0];
    }
    uint32_t cm = 0x000F000Fu, cx = 0x43004300u;  // in VGPRs, so that and-or fuses
    asm volatile("" : "+v"(cm), "+v"(cx));

    mg_f32x16 acc[NMI][2], part[2][NMI];
#pragma unroll
    for (int mi = 0; mi < NMI; ++mi)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[mi][b][i] = part[b][mi][i] = 0.f;

    // ---- prologue: rows of item 0, then the first NSTG - 1 stages
    fetch_rows(0);
    vm_wait_barrier<0>();
    setup_load(0);
#pragma unroll
    for (int st = 0; st < C::NSTG - 1; ++st) {
        begin_stage();
#pragma unroll
        for (int p = 0; p < C::PARTS; ++p) issue_part(p);
        if (C::KS > 1 || st + 1 < C::NSTG - 1) advance();  // (one K step per stage: at its first step)
    }

    Item ci{};     // the compute cursor's item
    int xrow = 0;  // A row of tile row `lane`
    bool no_bias = false;
    int ks = -1, c_slot = C::NSTG - 1, c_chunk = -1;
    u32x4 sch0 = {0u, 0u, 0u, 0u}, sch1 = sch0;  // scales of the current chunk
    float sc_pend = 0.f;                         // scale still to apply to part[1]

    // hand-over of act's 64-wide group sums between the two waves that cover a group (as in
    // moe_gemm.hip): written after the next stage's barrier, read two K steps later
    int x_state = 0;
    float x_pend = 0.f;
    bf16_t *x_dst = nullptr;
    const int x_oxe = j.ox_g ? j.N / j.ox_g : 0;
    const uint32_t x_slot = lds0 + C::OFF_X + 256u * (uint32_t)(wave >> 1) + 4u * (uint32_t)lane;
    auto x_store = [&](float v) __attribute__((always_inline)) {
        if (x_dst) {
            uint32_t hi, mid, lo;
            split3(v, hi, mid, lo);
            x_dst[0] = (bf16_t)hi;
            x_dst[x_oxe] = (bf16_t)mid;
            x_dst[2 * x_oxe] = (bf16_t)lo;
        }
    };
    auto x_write = [&]() __attribute__((always_inline)) {
        if (wave & 1)
            asm volatile("ds_write_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" ::"v"(x_slot), "v"(x_pend)
                         : "memory");
        x_state = 2;
    };
    auto x_read_store = [&]() __attribute__((always_inline)) {
        if (!(wave & 1)) {
            uint32_t o;
            asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(o) : "v"(x_slot));
            x_store(x_pend + __uint_as_float(o));
        }
        x_state = 0;
    };
    constexpr bool HANDOVER = GLU && C::QUANT && !G32;

    auto step = [&](auto st_c) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_c)::value;
        constexpr bool SS = ST % C::KS == 0;  // a stage starts
        if (++ks == nks) ks = 0;
        if constexpr (SS) {
            // this stage's copies have landed (with three stages the newest one's may be in
            // flight: they are the last PARTS issued), and every wave is done with the stage
            // before it, whose slot the copies issued below fill
            vm_wait_barrier<C::NSTG == 3 ? C::PARTS : 0>();
            c_slot = c_slot + 1 == C::NSTG ? 0 : c_slot + 1;
            if constexpr (HANDOVER) {
                if (ST == 0 && x_state == 1) x_write();
                else if (ST == 2 && x_state == 2) x_read_store();
            }
        }
        if (ST == 0 && ks == 0) {  // the load cursor is on this item (at least 8 K steps long)
            ci = li, xrow = lx;
            if (C::QUANT) no_bias = ci.sh ? j.sh.w0.biases == nullptr : j.w0.biases == nullptr;
        }
        // the bias term's operands of the current chunk, three K steps ahead of their use
        if (C::QUANT && ST == 0 && (ks + 4) % C::CH == 0) {
            const int c = (ks + 4) / C::CH - 1;
            if (wave < 3)
                dma16(rsrc_of(ci.sh ? j.sh.AX : j.AX), 2u * (uint32_t)((xrow * 3 + wave) * axe),
                      16u * (uint32_t)c, smem + C::OFF_X + wave * 1024);
            if (!no_bias) {
                const uint32_t wrow = (uint32_t)ci.e * (uint32_t)j.N + (uint32_t)(ci.n0 + (GLU ? (tid & 127) : tid));
                const bf16_t *bg = ci.sh ? j.sh.w0.biases : j.w0.biases;
                const bf16_t *bu = GLU ? (ci.sh ? j.sh.w1.biases : j.w1.biases) : bg;
                copy_chunk(rsrc_of(GLU && wave >= 2 ? bu : bg), 2u * wrow * (uint32_t)G, c,
                           smem + C::OFF_B);
            }
        }
        if (C::QUANT && C::SREG && ST == 0 && ks % C::CH == 0) {  // the chunk's scales, before the next are loaded
            if constexpr (GROUP == 128) sch0 = fmt_dup(sn0.x, sn0.y), sch1 = fmt_dup(sn1.x, sn1.y);
            else sch0 = sn0, sch1 = sn1;
        }
        // the load cursor moves on after the stage it last issued
        if constexpr (!SS || C::KS == 1) advance();
        if constexpr (SS) begin_stage();

        // ---- the K step's operands
        const uint32_t sbase = (uint32_t)(c_slot * C::STAGE);
        uint32_t pa[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) pa[s] = a_off[s] + sbase + (uint32_t)((ST % C::KS) * C::A_STEP);
        uint32_t pc[NCA];
#pragma unroll
        for (int s = 0; s < NCA; ++s)
            pc[s] = c_off[s] + sbase + (BITS == 4 && ST % C::KS ? c_step : 0u);
        u32x4 a[NMI][4];
        u32x4 cw[2][BITS == 16 ? 4 : 2];
        u32x2 cd[2][4];
        if constexpr (BITS == 4 && !G32) {
            FMT_READ("ds_read_b128 %[b0], %[q0]\n\tds_read_b128 %[b1], %[q0] offset:%[db]\n\t",
                     [b0] "=&v"(cw[0][0]) FMT_COMMA [b1] "=&v"(cw[1][0]), [q0] "v"(pc[0]),
                     [db] "i"(DB * C::C_ROW));
        } else if constexpr (BITS == 4 || (BITS == 8 && !G32)) {
            FMT_READ("ds_read_b128 %[b0], %[q0]\n\tds_read_b128 %[b1], %[q1]\n\t"
                     "ds_read_b128 %[b2], %[q0] offset:%[db]\n\tds_read_b128 %[b3], %[q1] offset:%[db]\n\t",
                     [b0] "=&v"(cw[0][0]) FMT_COMMA [b1] "=&v"(cw[0][1]) FMT_COMMA [b2] "=&v"(cw[1][0])
                         FMT_COMMA [b3] "=&v"(cw[1][1]),
                     [q0] "v"(pc[0]), [q1] "v"(pc[NCA > 1 ? 1 : 0]), [db] "i"(DB * C::C_ROW));
        } else if constexpr (BITS == 8) {
            FMT_READ("ds_read_b64 %[b0], %[q0]\n\tds_read_b64 %[b1], %[q1]\n\t"
                     "ds_read_b64 %[b2], %[q2]\n\tds_read_b64 %[b3], %[q3]\n\t"
                     "ds_read_b64 %[b4], %[q0] offset:%[db]\n\tds_read_b64 %[b5], %[q1] offset:%[db]\n\t"
                     "ds_read_b64 %[b6], %[q2] offset:%[db]\n\tds_read_b64 %[b7], %[q3] offset:%[db]\n\t",
                     [b0] "=&v"(cd[0][0]) FMT_COMMA [b1] "=&v"(cd[0][1]) FMT_COMMA [b2] "=&v"(cd[0][2])
                         FMT_COMMA [b3] "=&v"(cd[0][3]) FMT_COMMA [b4] "=&v"(cd[1][0])
                         FMT_COMMA [b5] "=&v"(cd[1][1]) FMT_COMMA [b6] "=&v"(cd[1][2])
                         FMT_COMMA [b7] "=&v"(cd[1][3]),
                     [q0] "v"(pc[0]), [q1] "v"(pc[NCA > 1 ? 1 : 0]), [q2] "v"(pc[NCA > 2 ? 2 : 0]),
                     [q3] "v"(pc[NCA > 3 ? 3 : 0]), [db] "i"(DB * C::C_ROW));
        } else {
            FMT_READ("ds_read_b128 %[b0], %[q0]\n\tds_read_b128 %[b1], %[q1]\n\t"
                     "ds_read_b128 %[b2], %[q2]\n\tds_read_b128 %[b3], %[q3]\n\t"
                     "ds_read_b128 %[b4], %[q0] offset:%[db]\n\tds_read_b128 %[b5], %[q1] offset:%[db]\n\t"
                     "ds_read_b128 %[b6], %[q2] offset:%[db]\n\tds_read_b128 %[b7], %[q3] offset:%[db]\n\t",
                     [b0] "=&v"(cw[0][0]) FMT_COMMA [b1] "=&v"(cw[0][1]) FMT_COMMA [b2] "=&v"(cw[0][BITS == 16 ? 2 : 0])
                         FMT_COMMA [b3] "=&v"(cw[0][BITS == 16 ? 3 : 0]) FMT_COMMA [b4] "=&v"(cw[1][0])
                         FMT_COMMA [b5] "=&v"(cw[1][1]) FMT_COMMA [b6] "=&v"(cw[1][BITS == 16 ? 2 : 0])
                         FMT_COMMA [b7] "=&v"(cw[1][BITS == 16 ? 3 : 0]),
                     [q0] "v"(pc[0]), [q1] "v"(pc[NCA > 1 ? 1 : 0]), [q2] "v"(pc[NCA > 2 ? 2 : 0]),
                     [q3] "v"(pc[NCA > 3 ? 3 : 0]), [db] "i"(DB * C::C_ROW));
        }
        if (C::QUANT && !C::SREG && ST == 0 && ks % C::CH == 0) {  // the chunk's scales
            ++c_chunk;
            const uint32_t sp = lds0 + C::OFF_S + (uint32_t)((c_chunk & 1) * C::S_BYTES);
            if constexpr (GROUP == 128) {
                uint32_t w0, w1, w2, w3;
                asm volatile("ds_read_b32 %0, %4\n\tds_read_b32 %1, %4 offset:1024\n\t"
                             "ds_read_b32 %2, %5\n\tds_read_b32 %3, %5 offset:1024\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(w0), "=&v"(w1), "=&v"(w2), "=&v"(w3)
                             : "v"(sp + 4u * (uint32_t)(bro0 + fr)), "v"(sp + 4u * (uint32_t)(bro1 + fr)));
                sch0 = fmt_dup(w0, w1), sch1 = fmt_dup(w2, w3);
            } else {
                asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(sch0), "=&v"(sch1)
                             : "v"(sp + 16u * (uint32_t)(bro0 + fr)), "v"(sp + 16u * (uint32_t)(bro1 + fr)));
            }
        }
        // the scale of group half hg (groups of 32) or of the whole K step
        auto scale_of = [&](const u32x4 &sw, int hg) __attribute__((always_inline)) {
            if constexpr (G32) {
                const uint32_t w = sw[ST];
                return hg ? bf_hi(w) : bf_lo(w);
            } else {
                const uint32_t w = (ks & 4) ? sw[2 + (ST >> 1)] : sw[ST >> 1];
                return (ST & 1) ? bf_hi(w) : bf_lo(w);
            }
        };
        // operand p = 4 ni + s: fragment ni's codes of sub-step s
        auto expand = [&](int p) __attribute__((always_inline)) {
            const int ni = p >> 2, s = p & 3;
            if constexpr (BITS == 16) {
                return fmt_pair8(cw[ni][s]);
            } else if constexpr (BITS == 8) {
                if constexpr (G32) return fmt_expand8(cd[ni][s][0], cd[ni][s][1]);
                else return fmt_expand8(cw[ni][s >> 1][2 * (s & 1)], cw[ni][s >> 1][2 * (s & 1) + 1]);
            } else {
                uint32_t w;
                if constexpr (G32) {  // block 2s + h: word 2 (s & 1) + h of unit s / 2
                    const u32x4 &u = cw[ni][s >> 1];
                    w = fh ? u[2 * (s & 1) + 1] : u[2 * (s & 1)];
                } else {
                    w = cw[ni][0][s];
                }
                u32x4 e;
                mg_expand_lo(e, w, cm, cx);
                mg_expand_hi(e, w, cm, cx);
                return e;
            }
        };
        // units: the chains of fragment ni (groups of 32: of its group half hg), SPU sub-steps of NMI
        // MFMAs; under a unit's MFMAs run the scale FMAs of the unit before and the expansion of the
        // next operand
        constexpr int NU = G32 ? 4 : 2, SPU = 8 / NU, NSLOT = 8 * NMI;
        constexpr int FPS = 16 / SPU;  // FMAs per slot
        __builtin_amdgcn_s_setprio(1);
        u32x4 e = expand(0), en = e;
#pragma unroll
        for (int q = 0; q < NSLOT; ++q) {
            const int p = q / NMI, mi = q % NMI;  // operand, row fragment
            const int u = p / SPU, s_in = p % SPU, ni = p >> 2, s = p & 3;
            const mg_f32x16 z = {};
            if constexpr (C::QUANT) {
                part[u & 1][mi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(mg_bf16x8, a[mi][s]), __builtin_bit_cast(mg_bf16x8, e),
                    s_in ? part[u & 1][mi] : z, 0, 0, 0);
            } else {
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(mg_bf16x8, a[mi][s]), __builtin_bit_cast(mg_bf16x8, e),
                    acc[mi][ni], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (SS) {
#pragma unroll
                for (int cp = 0; cp < C::PARTS; ++cp)
                    if (cp * NSLOT / C::PARTS == q) issue_part(cp);
            }
            if constexpr (C::QUANT) {
                const int pu = u ? u - 1 : NU - 1, pni = pu / (NU / 2);
                const float sc = u ? scale_of(pni ? sch1 : sch0, pu % (NU / 2)) : sc_pend;
                const int qu = q - u * SPU * NMI;  // slot in the unit
#pragma unroll
                for (int f = qu * FPS; f < (qu + 1) * FPS; ++f)
                    acc[f >> 4][pni][f & 15] += sc * part[pu & 1][f >> 4][f & 15];
            }
            if (p < 7 && mi == NMI - 1) {
                en = expand(p + 1);
                e = en;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (C::QUANT) sc_pend = scale_of(sch1, 1);
        __builtin_amdgcn_s_setprio(0);
        // the step's FMAs end here: sunk past the branches below they would keep the partial
        // products of several units alive
#pragma unroll
        for (int mi = 0; mi < NMI; ++mi) asm volatile("" : "+v"(acc[mi][0]), "+v"(acc[mi][1]));

        if (C::QUANT && ST == 3 && (ks + 1) % C::CH == 0) {
            // bias term of the chunk: X splits against b (lane half 0) and, with the 4-bit codes'
            // offset, -128 s (lane half 1)
            const uint32_t xo = lds0 + C::OFF_X + 16u * (uint32_t)fr;
            u32x4 xa[NMI][3], bv[2];
            if constexpr (NMI == 2) {
                asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:1024\n\t"
                             "ds_read_b128 %2, %6 offset:2048\n\tds_read_b128 %3, %6 offset:512\n\t"
                             "ds_read_b128 %4, %6 offset:1536\n\tds_read_b128 %5, %6 offset:2560\n\t"
                             "s_waitcnt lgkmcnt(0)"
                             : "=&v"(xa[0][0]), "=&v"(xa[0][1]), "=&v"(xa[0][2]), "=&v"(xa[NMI - 1][0]),
                               "=&v"(xa[NMI - 1][1]), "=&v"(xa[NMI - 1][2])
                             : "v"(xo));
            } else {
                asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %3 offset:1024\n\t"
                             "ds_read_b128 %2, %3 offset:2048\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(xa[0][0]), "=&v"(xa[0][1]), "=&v"(xa[0][2])
                             : "v"(xo));
            }
            const uint32_t bo = lds0 + C::OFF_B;
            if constexpr (GROUP == 128) {
                uint32_t w0, w1, w2, w3;
                asm volatile("ds_read_b32 %0, %4\n\tds_read_b32 %1, %4 offset:1024\n\t"
                             "ds_read_b32 %2, %5\n\tds_read_b32 %3, %5 offset:1024\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(w0), "=&v"(w1), "=&v"(w2), "=&v"(w3)
                             : "v"(bo + 4u * (uint32_t)(bro0 + fr)), "v"(bo + 4u * (uint32_t)(bro1 + fr)));
                bv[0] = fmt_dup(w0, w1), bv[1] = fmt_dup(w2, w3);
            } else {
                asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(bv[0]), "=&v"(bv[1])
                             : "v"(bo + 16u * (uint32_t)(bro0 + fr)), "v"(bo + 16u * (uint32_t)(bro1 + fr)));
            }
#pragma unroll
            for (int ni = 0; ni < 2; ++ni) {
                const u32x4 zero = {0u, 0u, 0u, 0u};
                u32x4 v = no_bias ? zero : bv[ni];
                if constexpr (BITS == 4) {
                    const u32x4 &sc = ni ? sch1 : sch0;
                    if (fh) v = u32x4{mg_neg128(sc.x), mg_neg128(sc.y), mg_neg128(sc.z), mg_neg128(sc.w)};
                } else if (fh) {
                    v = zero;
                }
#pragma unroll
                for (int mi = 0; mi < NMI; ++mi)
#pragma unroll
                    for (int tt = 0; tt < 3; ++tt)
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(mg_bf16x8, xa[mi][tt]),
                            __builtin_bit_cast(mg_bf16x8, v), acc[mi][ni], 0, 0, 0);
            }
        }
        if (ST != 3 || ks != nks - 1) return;
        if constexpr (C::QUANT) {  // the item's last scale
            // the products are cleared with the scale: the next item's first step adds 0 times them,
            // which an infinity or NaN of one of this item's rows would turn into NaN there
#pragma unroll
            for (int mi = 0; mi < NMI; ++mi)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    acc[mi][1][i] += sc_pend * part[1][mi][i];
                    part[1][mi][i] = 0.f;
                }
            sc_pend = 0.f;
        }

        // ---- epilogue of item ci, through a buffer resource over the tile's own rows (stores of
        // the rows past mrows fall outside it and are dropped)
        bf16_t *out = ci.sh ? j.sh.out : j.out;
        const int ldo = ci.sh ? j.sh.ldo : j.ldo;
        const rsrc_t r_out = rsrc_of(out + (size_t)ci.row0 * ldo, (uint32_t)ci.mrows * (uint32_t)ldo * 2u);
        if constexpr (GLU) {
            x_pend = store_act<NMI>(acc, r_out, ldo, ci.n0 + wave * 32 + fr, lane);
            if (C::QUANT && j.ox_g) {  // act's X sums: per wave, or per pair of waves (hand-over)
                bf16_t *OX = ci.sh ? j.sh.OX : j.OX;
                const int xr = xrow_of(lane), col = ci.n0 + 32 * wave;
                x_dst = xr < ci.mrows ? OX + (size_t)(ci.row0 + xr) * 3 * x_oxe + col / j.ox_g : nullptr;
                if (!HANDOVER || j.ox_g == 32) x_store(x_pend);
                else x_state = 1;
            }
        } else {
            store_rows<NMI>(acc, r_out, ldo, ci.n0 + bro0, ci.n0 + bro1, lane);
        }
#pragma unroll
        for (int mi = 0; mi < NMI; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[mi][ni][i] = 0.f;
    };
    for (int gs = 0; gs < total_steps; gs += 4) {
        step(std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
        step(std::integral_constant<int, 1>{});
        __builtin_amdgcn_sched_barrier(0);
        step(std::integral_constant<int, 2>{});
        __builtin_amdgcn_sched_barrier(0);
        step(std::integral_constant<int, 3>{});
        __builtin_amdgcn_sched_barrier(0);
    }
    if (HANDOVER && x_state == 1) {  // the last item's group sums
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        x_write();
        asm volatile("s_barrier" ::: "memory");
        x_read_store();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the trailing copies
}

bool fmt_gemm_supported(const MoeGemmJob &j) {
    const QW &w0 = j.w0;
    const bool quant = w0.bits != 16;
    auto ok = [&](const QW &w) {
        if (!w.codes || ((uintptr_t)w.codes & 15) || w.bits != w0.bits || w.out != j.N) return false;
        // byte offsets from the tensors' bases are 32-bit
        if ((size_t)w.experts * (size_t)w.out * (size_t)j.K * (size_t)w.bits / 8 >= ((size_t)1 << 32))
            return false;
        if (!quant) return true;
        return w.group == w0.group && w.scales && ((uintptr_t)w.scales & 15) == 0 &&
               ((uintptr_t)w.biases & 15) == 0;
    };
    auto pair_ok = [&](const QW &a, const QW &b) {  // one no-bias rule for both weights of a pair
        return ok(a) && (!j.glu || (ok(b) && (!a.biases) == (!b.biases)));
    };
    if (w0.bits != 4 && w0.bits != 8 && w0.bits != 16) return false;
    if (quant && w0.group != 32 && w0.group != 64 && w0.group != 128) return false;
    if (j.K % 512 != 0 || !pair_ok(w0, j.w1) || (j.has_shared && !pair_ok(j.sh.w0, j.sh.w1))) return false;
    if (!quant && j.tile_m != 32) return false;  // bf16 weights: 32-row tiles only (0 is 64)
    const int xg = w0.group == 32 ? 32 : 64;     // X sums of the A rows
    if (quant && (j.ax_g != xg || j.ax_e != j.K / xg)) return false;
    if (j.glu) {  // X sums of act for the down product
        if (j.ox_g != 0 && j.ox_g != 32 && j.ox_g != 64) return false;
        if (j.ox_g && (!quant || !j.OX || (j.has_shared && !j.sh.OX))) return false;
        if (j.ox_g == 64 && w0.group == 32) return false;
    }
    return true;
}

template <int NMI, int BITS, int GROUP>
static void run_fmt(const MoeGemmJob &j, unsigned grid, hipStream_t s) {
    if (j.glu) fmt_gemm_kernel<true, NMI, BITS, GROUP><<<grid, 256, 0, s>>>(j);
    else fmt_gemm_kernel<false, NMI, BITS, GROUP><<<grid, 256, 0, s>>>(j);
}

hipError_t launch_fmt_gemm(const MoeGemmJob &j, unsigned grid, hipStream_t s) {
    const int b = j.w0.bits, g = j.w0.group;
    const bool half = j.tile_m == 32;
    if (b == 16) {
        if (!half) return hipErrorInvalidValue;
        run_fmt<1, 16, 64>(j, grid, s);
    } else if (b == 8) {
        if (g == 32) half ? run_fmt<1, 8, 32>(j, grid, s) : run_fmt<2, 8, 32>(j, grid, s);
        else if (g == 64) half ? run_fmt<1, 8, 64>(j, grid, s) : run_fmt<2, 8, 64>(j, grid, s);
        else half ? run_fmt<1, 8, 128>(j, grid, s) : run_fmt<2, 8, 128>(j, grid, s);
    } else {
        if (g == 32) half ? run_fmt<1, 4, 32>(j, grid, s) : run_fmt<2, 4, 32>(j, grid, s);
        else if (g == 128) half ? run_fmt<1, 4, 128>(j, grid, s) : run_fmt<2, 4, 128>(j, grid, s);
        else return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace mrun
