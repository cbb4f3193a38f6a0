// Device helpers of the prefill grouped GEMMs (moe_gemm.hip, moe_fmt.hip): copies from global memory
// straight into LDS, LDS reads with explicit waits, the LDS swizzles and the code expansion.
#pragma once

#include "common.hpp"

namespace mrun {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 mg_bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float mg_f32x16;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ uint32_t lds_offset(const void *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)p;
}
// An LDS read whose wait comes later (an lgkmcnt asm taking the destination as "+v"). The compiler
// takes the destination as written at issue, so any copy or spill of it before the wait would read
// a register the load has not yet filled: the kernels that use it must build without VGPR spills
// (tests/test_isa.py checks the built code for both).
template <int OFF>
__device__ __forceinline__ u32x4 ds_read16(uint32_t a) {
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "i"(OFF));
    return v;
}
// Reads whose results become addresses or counts: the reads and their wait are one statement, so
// that no copy or spill of a destination register can come between a read and its arrival.
__device__ __forceinline__ void ds_read3_now(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t &v0,
                                             uint32_t &v1, uint32_t &v2) {
    asm volatile("ds_read_b32 %0, %3\n\tds_read_b32 %1, %4\n\tds_read_b32 %2, %5\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(v0), "=&v"(v1), "=&v"(v2)
                 : "v"(a0), "v"(a1), "v"(a2));
}
// Global memory goes to LDS through buffer loads (buffer_load ... lds): a raw resource per
// tensor (base address in scalar registers), a per-lane 32-bit byte offset and a scalar one, so
// that no per-lane 64-bit address arithmetic is needed. 16 (or 4) bytes per lane land at
// lds + 16 * lane (4 * lane); the LDS address is the same for the whole wave.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t rsrc_of(const void *p, uint32_t bytes = 0xFFFFFFFFu) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void dma16(rsrc_t r, uint32_t voff, uint32_t soff, char *lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t *)lds, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void dma4(rsrc_t r, uint32_t voff, uint32_t soff, char *lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t *)lds, 4, voff, soff, 0, 0);
}
// Wait until at most N of this wave's global loads are outstanding, then a workgroup barrier.
template <int N>
__device__ __forceinline__ void vm_wait_barrier() {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(N) : "memory");
}

// a code word (8 codes) into the bf16 pairs (128 + q_i, 128 + q_{i+4}), in two halves
__device__ __forceinline__ void mg_expand_lo(u32x4 &r, uint32_t w, uint32_t cm, uint32_t cx) {
    r.x = (w & cm) | cx;
    r.y = ((w >> 4) & cm) | cx;
}
__device__ __forceinline__ void mg_expand_hi(u32x4 &r, uint32_t w, uint32_t cm, uint32_t cx) {
    r.z = ((w >> 8) & cm) | cx;
    r.w = ((w >> 12) & cm) | cx;
}

// -128 s for a pair of bf16 scales (exact: a power-of-two scaling)
__device__ __forceinline__ uint32_t mg_neg128(uint32_t w) {
    const uint32_t lo = __float_as_uint(-128.f * bf_lo(w)) >> 16;
    const uint32_t hi = __float_as_uint(-128.f * bf_hi(w)) & 0xFFFF0000u;
    return lo | hi;
}

// A value the whole wave holds, moved to a scalar register: integer divisions by runtime values
// run on the VALU, and without this the compiler would treat their results (and the loads and
// branches that depend on them) as per-lane.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// LDS swizzles (16-byte units). A rows are 128 B (8 units): rows r and r + 8 (same bank window
// at 256 B per cycle) and rows of one parity in 16 get distinct masks. B rows are 64 B (4 units,
// two K steps of codes): rows r, r + 4, r + 8, r + 12 (which share a position in a 256-byte window)
// get distinct masks, and so do r, r + 2, r + 4, r + 6 (a 128-byte window).
__device__ __forceinline__ int swz_a(int r) { return (r & 7) ^ ((r >> 3) & 1); }
__device__ __forceinline__ int swz_c(int r) { return ((r >> 2) ^ (r >> 1)) & 3; }

// The tile row whose act column sum lane `l` holds after the gate/up epilogue's reduce-scatter:
// with fr = l % 32, bit 4 of fr chose the row fragment (32 rows), bits 3-2 the 8-row block,
// bits 1-0 the row in a block of 4, and the lane half (l / 32) the block of 4 within 8 (the
// MFMA's C layout: value i of lane l is row 8 (i / 4) + 4 (l / 32) + i % 4 of its fragment).
__device__ __forceinline__ int xrow_of(int l) {
    const int fr = l & 31;
    return 32 * (fr >> 4) + 8 * ((fr >> 2) & 3) + 4 * (l >> 5) + (fr & 3);
}

// The gate/up epilogue of one wave's 32 NMI rows x 32 act columns (`col`: this lane's): act =
// R(silu(R(gate)) * R(up)) of the fragments acc[.][0] (gate) and acc[.][1] (up), stored packed
// through r_out (the tile's rows; stores past them are dropped). Returns the sum of the wave's 32
// columns for act row xrow_of(lane) of the tile.
template <int NMI>
__device__ __forceinline__ float store_act(const mg_f32x16 (&acc)[NMI][2], rsrc_t r_out, int ldo,
                                           int col, int lane) {
    const int fh = lane >> 5;
    const int c64 = col & 63, kb = c64 >> 3, jj = c64 & 7;
    // lanes with jj < 4 store packed pair (jj, jj + 4) of rows i (i even); lanes jj >= 4
    // the pair of row i + 1: both at the packed position of jj & 3
    const int pcol = (col & ~63) + 8 * (2 * (kb & 3) + (kb >> 2)) + 2 * (jj & 3);
    const bool hi4 = (jj & 4) != 0;
    float va[2][16];  // the act values (rounded) of rows mi * 32 + 8 (i / 4) + 4 fh + i % 4
    if (NMI == 1)
#pragma unroll
        for (int i = 0; i < 16; ++i) va[1][i] = 0.f;
#pragma unroll
    for (int mi = 0; mi < NMI; ++mi)
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            float v[2];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const uint32_t gu = f2bf2(acc[mi][0][i + d], acc[mi][1][i + d]);
                const float g = bf_lo(gu), u = bf_hi(gu);
                // silu(g) = g / (1 + exp(-g)): v_exp and v_rcp (within 2 f32 ulp)
                const float e = __builtin_amdgcn_exp2f(-1.44269504088896f * g);
                v[d] = (g * __builtin_amdgcn_rcpf(1.f + e)) * u;
            }
            const uint32_t hv = f2bf2(v[0], v[1]);  // row i in the low half, i + 1 high
            va[mi][i] = bf_lo(hv), va[mi][i + 1] = bf_hi(hv);
            // lane l (jj < 4) keeps row i of (jj, jj + 4); lane l + 4 row i + 1
            const uint32_t send = hi4 ? (hv & 0xFFFFu) : (hv >> 16);
            const uint32_t from_up = (uint32_t)__builtin_amdgcn_mov_dpp((int)send, 0x104, 0xF, 0xF, false);   // lane l + 4
            const uint32_t from_dn = (uint32_t)__builtin_amdgcn_mov_dpp((int)send, 0x114, 0xF, 0xF, false);   // lane l - 4
            const uint32_t pair = hi4 ? (from_dn | (hv & 0xFFFF0000u)) : ((hv & 0xFFFFu) | (from_up << 16));
            const int r = mi * 32 + 8 * (i >> 2) + 4 * fh + (i & 3) + (hi4 ? 1 : 0);
            __builtin_amdgcn_raw_buffer_store_b32(pair, r_out, (r * ldo + pcol) * 2, 0, 0);
        }
    // this wave's sums of the 32 act columns for each row, by a reduce-scatter over the
    // 32 lanes of each lane half (their columns): every step pairs lane l with lane l ^ d,
    // each keeps the half of its values that its bit d selects and adds the partner's
    // copy of it. After d = 16 (permlane16_swap), 8 (row_ror:8), 4 (row_shl/shr:4 by
    // banks), 2 and 1 (quad_perm) the lane holds the sum of row xrow_of(lane).
    float w16[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {  // d = 16: lanes of even rows keep mi = 0, odd rows 1
        const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(va[0][i]),
                                                        __float_as_uint(va[1][i]), false, false);
        w16[i] = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    }
    const bool b3 = (lane & 8) != 0, b2 = (lane & 4) != 0, b1 = (lane & 2) != 0, b0 = (lane & 1) != 0;
    float w8[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {  // d = 8: keep i + 8 b3
        const float keep = b3 ? w16[i + 8] : w16[i], send = b3 ? w16[i] : w16[i + 8];
        w8[i] = keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(send), 0x128, 0xF, 0xF, false));
    }
    float w4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // d = 4: keep i + 4 b2
        const float keep = b2 ? w8[i + 4] : w8[i], send = b2 ? w8[i] : w8[i + 4];
        int m = __builtin_amdgcn_update_dpp(0, __float_as_int(send), 0x104, 0xF, 0x5, false);  // banks 0, 2: lane l + 4
        m = __builtin_amdgcn_update_dpp(m, __float_as_int(send), 0x114, 0xF, 0xA, false);      // banks 1, 3: lane l - 4
        w4[i] = keep + __int_as_float(m);
    }
    float w2[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // d = 2: keep i + 2 b1
        const float keep = b1 ? w4[i + 2] : w4[i], send = b1 ? w4[i] : w4[i + 2];
        w2[i] = keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(send), 0x4E, 0xF, 0xF, false));
    }
    {  // d = 1: keep b0
        const float keep = b0 ? w2[1] : w2[0], send = b0 ? w2[0] : w2[1];
        return keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(send), 0xB1, 0xF, 0xF, false));
    }
}

// The down epilogue of one wave's 32 NMI rows x 2 fragments of 32 columns (col0, col1: each
// fragment's first column), rounded to bf16 and stored through r_out (the tile's rows; stores past
// them are dropped).
template <int NMI>
__device__ __forceinline__ void store_rows(const mg_f32x16 (&acc)[NMI][2], rsrc_t r_out, int ldo,
                                           int col0, int col1, int lane) {
    const int fr = lane & 31, fh = lane >> 5;
    // each 4 x 4 block (4 rows of a lane, 4 columns of a lane quad) is transposed within
    // the quad (every lane then holds 4 adjacent columns of one row), and lanes l, l ^ 4
    // (the two quads of 8 adjacent columns) trade halves of two such blocks, so that every
    // lane stores 8 adjacent columns of one row (16 bytes)
    const int q = fr & 3;
    const bool hq = (fr & 4) != 0;  // keeps the odd block of each pair
    typedef unsigned u32x4s __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
        const int col8 = (ni ? col1 : col0) + (fr & ~7);
#pragma unroll
        for (int mi = 0; mi < NMI; ++mi) {
            uint2 w4[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const uint32_t p02 = f2bf2(acc[mi][ni][4 * b], acc[mi][ni][4 * b + 2]);
                const uint32_t p13 = f2bf2(acc[mi][ni][4 * b + 1], acc[mi][ni][4 * b + 3]);
                // lanes q, q ^ 1: even lanes gather rows 0 and 2, odd lanes rows 1 and 3
                const uint32_t own = (q & 1) ? p13 : p02;
                const uint32_t rcv = (uint32_t)__builtin_amdgcn_mov_dpp((int)((q & 1) ? p02 : p13), 0xB1, 0xF, 0xF, false);
                const uint32_t lo_src = (q & 1) ? rcv : own, hi_src = (q & 1) ? own : rcv;
                const uint32_t A = __builtin_amdgcn_perm(hi_src, lo_src, 0x05040100u);  // row q & 1
                const uint32_t B = __builtin_amdgcn_perm(hi_src, lo_src, 0x07060302u);  // row 2 + (q & 1)
                // lanes q, q ^ 2: lanes 0, 1 complete rows 0, 1; lanes 2, 3 rows 2, 3
                const uint32_t r2 = (uint32_t)__builtin_amdgcn_mov_dpp((int)((q & 2) ? A : B), 0x4E, 0xF, 0xF, false);
                w4[b] = (q & 2) ? make_uint2(r2, B) : make_uint2(A, r2);
            }
#pragma unroll
            for (int bp = 0; bp < 2; ++bp) {
                const uint2 keep = hq ? w4[2 * bp + 1] : w4[2 * bp];
                const uint2 send = hq ? w4[2 * bp] : w4[2 * bp + 1];
                // lane ^ 4 within each row of 16 lanes: banks 0, 2 read lane + 4, banks 1, 3 lane - 4
                int rx = __builtin_amdgcn_update_dpp(0, (int)send.x, 0x104, 0xF, 0x5, false);
                rx = __builtin_amdgcn_update_dpp(rx, (int)send.x, 0x114, 0xF, 0xA, false);
                int ry = __builtin_amdgcn_update_dpp(0, (int)send.y, 0x104, 0xF, 0x5, false);
                ry = __builtin_amdgcn_update_dpp(ry, (int)send.y, 0x114, 0xF, 0xA, false);
                const u32x4s v = hq ? u32x4s{(uint32_t)rx, (uint32_t)ry, keep.x, keep.y}
                                    : u32x4s{keep.x, keep.y, (uint32_t)rx, (uint32_t)ry};
                const int r = mi * 32 + 8 * (2 * bp + (hq ? 1 : 0)) + 4 * fh + q;
                __builtin_amdgcn_raw_buffer_store_b128(v, r_out, (r * ldo + col8) * 2, 0, 0);
            }
        }
    }
}

}  // namespace mrun
