// k_pp.hip -- large bf16 and int8 MFMA tiles whose two wave groups take turns
// on the matrix cores (gfx950).
//
// Serves the many-row end of the reference's packed paths
// (src/gemm/gemm_driver_bf16.cpp:134-218, src/gemm/gemm_int8_native.cpp:189-248):
// bf16 storage with B stored K x N or N x K, and int8 with B stored N x K.
//
// What bounds it: the matrix cores.  A 256 x 256 tile copies 64 KB into LDS
// and reads 192 KB of fragments from it per 128 bytes of k for 2048 MFMA
// cycles per SIMD.  The 8 waves form two groups of four (one wave of each on
// every SIMD, the upper and lower half of the tile's rows).  A k-block is cut
// into phases of one row half times one column part; a group spends one slot
// reading a phase's fragments and issuing one part's copy, and the next slot
// on that phase's MFMAs, and the second group runs one slot behind the first,
// so the MFMAs of one group cover the LDS reads of the other.  Measured
// (MI355X, 4096 x 4096 x 4096 bf16, B stored N x K): 2421 cycles per block
// against 2048 of MFMAs alone (85%; 2214 without the copies, 1800 without the
// MFMAs; over whole launches, first copies and epilogue included, the
// MFMA-busy counter reads 69% in bf16 and 60% in int8, without a bank
// conflict), at a clock that the power limit holds near 1.8 GHz.  32 x 32
// MFMAs need fewer cycles (2275) but draw more power and ran 8% slower, and the
// order of the MFMAs within a phase makes no difference.  Against the LDS-DMA
// tiles with one barrier per block (us): bf16 4096^3 174.9 -> 102.3 (up to 113
// where the card's clock is lower), 2048 x 11008 x 4096 225.4 -> 171.2; int8
// 4096^3 156.8 -> 60.2, 1024 x 11008 x 4096 100.1 -> 48.9.  Non-temporal stores
// of C measured 0-8% slower.
#include <type_traits>

#include "device_common.h"
#include "kernels.h"

using namespace dnnopt_dev;

namespace dnnopt_hip {

namespace {

// 16-byte chunk c (0..7) of 128-byte LDS row `row`.
__device__ __forceinline__ int pp_swz(int row, int c) { return c ^ (row & 7); }

// 32-byte segment swizzle of k row `k` of a K x N part: the 8 rows k0..k0+3,
// k0+8..k0+11 that one half of a transposing read gathers from must fall in
// 8 different 32-byte bank groups; a row of W bytes starts on group
// (k * W / 32) mod 8.
template <int W>
__device__ __forceinline__ int pp_seg(int k) {
    if constexpr (W % 256 == 0) return (k & 3) | (((k >> 3) & 1) << 2);
    else return ((k >> 1) & 1) | (((k >> 3) & 1) << 1);  // 128-byte rows
}

template <int DT>
struct PPAcc {
    using type = f32x4;
};
template <>
struct PPAcc<1> {
    using type = i32x4;
};

}  // namespace

// DT 0: bf16 storage, fp32 accumulation (EPI unused); DT 1: int8, exact
// int32, EPI 0 int32 C, EPI 1 fp32 C through s8_out.  TB = 1: B stored N x K.
// The tile is 32 MT rows (each wave 8 MT of either row half) by 64 (Q0 + Q1)
// columns in one or two parts, each wave 16 Q columns of a part.
//
// LDS holds two k-blocks of 128 bytes per row, each part (row half of A,
// column part of B) an array of its own so that the compiler's wait counts
// stay exact.  k-contiguous parts are rows of 128 bytes with XOR-swizzled
// 16-byte chunks, a K x N part is 64 rows of k, read with the transposing
// LDS load.  Parts of block i + 2 are copied into the places block i has
// left: a part is free once both groups have passed the barrier after the
// slot that read it (each group drains its LDS reads before that barrier),
// which is before either group's next read slot.  The waits leave the five
// parts issued last in flight (three where B is one part) and so cover the
// next read slot's parts, in both groups, one barrier ahead of it.
//
// k past K reads zero: whole 16-byte chunks are out of range, so K must be a
// multiple of 8 (bf16) or 16 (int8) where rows are k-contiguous; rows of a
// K x N part past K are past B's end.  A, B rows on 4-byte boundaries;
// 256 ldc 4 < 2^31.
template <int DT, int TB, int MT, int Q0, int Q1, int EPI>
__device__ __forceinline__ void pp_tile(const PPArgs& p) {
    constexpr int ES = DT == 0 ? 2 : 1;
    constexpr int BK = 128 / ES;
    constexpr int MH = MT / 2;
    constexpr int BM = 32 * MT, HM = BM / 2;
    constexpr int W0 = 64 * Q0, W1 = 64 * Q1, BN = W0 + W1;
    constexpr int UA = HM / 64, UB0 = Q0, UB1 = Q1;  // wave loads per part
    constexpr int Q1N = Q1 > 0 ? Q1 : 1;
    using acc_t = typename PPAcc<DT>::type;
    __shared__ __attribute__((aligned(1024))) char sA00[HM * 128];
    __shared__ __attribute__((aligned(1024))) char sA10[HM * 128];
    __shared__ __attribute__((aligned(1024))) char sB00[W0 * 128];
    __shared__ __attribute__((aligned(1024))) char sB10[Q1 ? W1 * 128 : 16];
    __shared__ __attribute__((aligned(1024))) char sA01[HM * 128];
    __shared__ __attribute__((aligned(1024))) char sA11[HM * 128];
    __shared__ __attribute__((aligned(1024))) char sB01[W0 * 128];
    __shared__ __attribute__((aligned(1024))) char sB11[Q1 ? W1 * 128 : 16];

    const int lane = lane_id(), r = lane & 15, g = lane >> 4;
    const int w = wave_id(), wn = w & 3, wm = w >> 2;
    const TileXY tile = xcd_tile((int)blockIdx.x, p.tiles_n, p.tiles_m);
    if (!tile.ok) return;
    const int m0 = tile.m * BM, n0 = tile.n * BN;
    const int nblk = (p.K + BK - 1) / BK;
    const int b_lo = (int)(((long long)nblk * blockIdx.z) / p.splits);
    const int b_hi = (int)(((long long)nblk * (blockIdx.z + 1)) / p.splits);
    const int nb = b_hi - b_lo;

    const char* abase = static_cast<const char*>(p.A) + (size_t)m0 * p.lda * ES;
    const char* bbase = static_cast<const char*>(p.B) + (TB ? (size_t)n0 * p.ldb : (size_t)n0) * ES;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(abase, range31((((size_t)(p.M - 1 - m0) * p.lda + p.K) * ES + 3) & ~(size_t)3));
    const size_t b_last = TB ? (size_t)(p.N - 1 - n0) * p.ldb + p.K : (size_t)(p.K - 1) * p.ldb + (p.N - n0);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(bbase, range31((b_last * ES + 3) & ~(size_t)3));

    // k-contiguous parts: a wave load fills 8 rows of 128 bytes; lane l fills
    // slot l % 8 of row l / 8 with chunk ck (the same in every load).
    const int lrow = lane >> 3, ck = pp_swz(lrow, lane & 7);
    const bool ctail = (nblk - 1) * BK + ck * (16 / ES) >= p.K;
    uint32_t ga[2][UA], gb0[UB0], gb1[Q1N];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < UA; ++j) {
            const int row = h * HM + (j * 8 + w) * 8 + lrow;
            ga[h][j] = m0 + row < p.M ? (uint32_t)row * (uint32_t)p.lda * ES + 16u * ck : kOobOffset;
        }
    auto boff = [&](int col0, int W, int j) -> uint32_t {
        if constexpr (TB) {
            const int row = col0 + (j * 8 + w) * 8 + lrow;
            return n0 + row < p.N ? (uint32_t)row * (uint32_t)p.ldb * ES + 16u * ck : kOobOffset;
        } else {
            const int q = (j * 8 + w) * 1024 + 16 * lane, kr = q / (W * 2), b = q % (W * 2);
            const int seg = (b >> 5) ^ (W == 64 ? pp_seg<128>(kr) : pp_seg<256>(kr));
            return (uint32_t)kr * (uint32_t)p.ldb * 2u + (uint32_t)(col0 * 2 + (seg << 5) + (b & 31));
        }
    };
#pragma unroll
    for (int j = 0; j < UB0; ++j) gb0[j] = boff(0, W0, j);
#pragma unroll
    for (int j = 0; j < Q1; ++j) gb1[j] = boff(W0, W1, j);

    // Blocks past the split's end are issued too (every wave's count of
    // outstanding loads stays the same) but read nothing.
    auto dma_a = [&](char* dst, int h, int blk) {
        const uint32_t ko = (uint32_t)blk * 128u;
        const bool cut = blk >= b_hi || (blk == nblk - 1 && ctail);
#pragma unroll
        for (int j = 0; j < UA; ++j) lds_dma16(ra, dst + (j * 8 + w) * 1024, cut ? kOobOffset : ga[h][j] + ko);
    };
    auto dma_b = [&](char* dst, auto part, int blk) {
        constexpr int P = decltype(part)::value, U = P ? UB1 : UB0;
        const uint32_t ko = TB ? (uint32_t)blk * 128u : (uint32_t)blk * BK * (uint32_t)p.ldb * ES;
        const bool cut = blk >= b_hi || (TB && blk == nblk - 1 && ctail);
#pragma unroll
        for (int j = 0; j < U; ++j) lds_dma16(rb, dst + (j * 8 + w) * 1024, cut ? kOobOffset : (P ? gb1[j] : gb0[j]) + ko);
    };

    acc_t acc[2][MH][Q0 + Q1];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int mt = 0; mt < MH; ++mt)
#pragma unroll
            for (int nt = 0; nt < Q0 + Q1; ++nt) acc[h][mt][nt] = acc_t{0, 0, 0, 0};

    u32x4 fa[2][MH], fb0[2][Q0], fb1[2][Q1N];
    auto read_a = [&](const char* src) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int mt = 0; mt < MH; ++mt) {
                const int row = (wm * MH + mt) * 16 + r;
                fa[kk][mt] = *reinterpret_cast<const u32x4*>(src + row * 128 + pp_swz(row, kk * 4 + g) * 16);
            }
    };
    auto read_b = [&](const char* src, auto part) {
        constexpr int P = decltype(part)::value, Q = P ? Q1 : Q0, W = P ? W1 : W0;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int nt = 0; nt < Q; ++nt) {
                u32x4 v;
                if constexpr (TB) {
                    const int row = (wn * Q + nt) * 16 + r;
                    v = *reinterpret_cast<const u32x4*>(src + row * 128 + pp_swz(row, kk * 4 + g) * 16);
                } else {
                    typedef short s16x4 __attribute__((ext_vector_type(4)));
                    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
                    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                    const int cb = ((wn * Q + nt) * 16 + 4 * (r & 3)) * 2;
                    const int k1 = kk * 32 + 8 * g + (r >> 2), k2 = k1 + 4;
                    const int o1 = k1 * W * 2 + ((((cb >> 5) ^ pp_seg<W * 2>(k1)) << 5) | (cb & 31));
                    const int o2 = k2 * W * 2 + ((((cb >> 5) ^ pp_seg<W * 2>(k2)) << 5) | (cb & 31));
                    const u32x2 l2 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(src + o1)));
                    const u32x2 h2 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(src + o2)));
                    v = u32x4{l2[0], l2[1], h2[0], h2[1]};
                }
                if constexpr (P) fb1[kk][nt] = v;
                else fb0[kk][nt] = v;
            }
    };
    // Operands swapped: lane (r, g) of a sub-tile holds row r of A's tile,
    // columns 4 g .. 4 g + 3 of B's.
    auto mma = [&](int h, auto part) {
        constexpr int P = decltype(part)::value, Q = P ? Q1 : Q0;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int mt = 0; mt < MH; ++mt)
#pragma unroll
                for (int nt = 0; nt < Q; ++nt) {
                    acc_t& c = acc[h][mt][P ? Q0 + nt : nt];
                    const u32x4 b = P ? fb1[kk][P ? nt : 0] : fb0[kk][P ? 0 : nt];
                    if constexpr (DT == 0)
                        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b),
                                                                   __builtin_bit_cast(bf16x8, fa[kk][mt]), c, 0, 0, 0);
                    else
                        c = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, b),
                                                                 __builtin_bit_cast(i32x4, fa[kk][mt]), c, 0, 0, 0);
                }
        __builtin_amdgcn_s_setprio(0);
    };
    auto slot_end = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto lgkm0 = [&]() { __builtin_amdgcn_s_waitcnt(0xC07F); };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;

    auto block = [&](int blk, auto stage_tag) {
        constexpr int S = decltype(stage_tag)::value;
        char* const a0 = S ? sA01 : sA00;
        char* const a1 = S ? sA11 : sA10;
        char* const b0 = S ? sB01 : sB00;
        char* const b1 = S ? sB11 : sB10;
        char* const a1n = S ? sA10 : sA11;
        if constexpr (Q1 > 0) {
            read_b(b0, P0{});
            read_a(a0);
            dma_a(a1n, 1, blk + 1);
            lgkm0();
            wait_vmcnt<3 * UA + UB0 + UB1>();  // B1(blk) landed
            slot_end();
            mma(0, P0{});
            slot_end();
            read_b(b1, P1{});
            dma_b(b0, P0{}, blk + 2);
            lgkm0();
            wait_vmcnt<2 * UA + 2 * UB0 + UB1>();  // A1(blk) landed
            slot_end();
            mma(0, P1{});
            slot_end();
            read_a(a1);
            dma_a(a0, 0, blk + 2);
            lgkm0();
            slot_end();
            mma(1, P1{});
            slot_end();
            dma_b(b1, P1{}, blk + 2);
            wait_vmcnt<2 * UA + UB0 + 2 * UB1>();  // A0, B0 of blk + 1 landed
            slot_end();
            mma(1, P0{});
            slot_end();
        } else {
            read_b(b0, P0{});
            read_a(a0);
            dma_a(a1n, 1, blk + 1);
            lgkm0();
            wait_vmcnt<2 * UA + UB0>();  // A1(blk) landed
            slot_end();
            mma(0, P0{});
            slot_end();
            read_a(a1);
            dma_b(b0, P0{}, blk + 2);
            dma_a(a0, 0, blk + 2);
            lgkm0();
            wait_vmcnt<2 * UA + UB0>();  // A0, B0 of blk + 1 landed
            slot_end();
            mma(1, P0{});
            slot_end();
        }
    };

    // Order of issue as in the loop: B0, A0, B1 of a block, then its A1.
    dma_b(sB00, P0{}, b_lo);
    dma_a(sA00, 0, b_lo);
    if constexpr (Q1 > 0) dma_b(sB10, P1{}, b_lo);
    dma_a(sA10, 1, b_lo);
    dma_b(sB01, P0{}, b_lo + 1);
    dma_a(sA01, 0, b_lo + 1);
    if constexpr (Q1 > 0) dma_b(sB11, P1{}, b_lo + 1);
    wait_vmcnt<2 * UA + UB0 + 2 * UB1>();  // A0, B0 of the first block landed
    slot_end();
    if (wm == 1) slot_end();  // the second group runs one slot behind
    int i = 0;
    for (; i + 2 <= nb; i += 2) {
        block(b_lo + i, std::integral_constant<int, 0>{});
        block(b_lo + i + 1, std::integral_constant<int, 1>{});
    }
    if (i < nb) block(b_lo + i, std::integral_constant<int, 0>{});
    if (wm == 0) slot_end();
    wait_vmcnt<0>();  // the run-on copies have landed

    const float dq = EPI == 1 && p.amax ? dyn_dequant_scale(p.amax, p.alpha) : 0.0f;
    // C's rows start on 4-byte boundaries, which is all a buffer access needs.
    // Partial tiles ([split][tile][BM * BN], for the reduce kernel) are whole.
    const bool part = p.splits > 1;
    const int tiles = p.tiles_n * p.tiles_m, tile_id = tile.m * p.tiles_n + tile.n;
    const uint32_t ldo = part ? (uint32_t)BN : (uint32_t)p.ldc;
    char* const obase = part ? static_cast<char*>(p.part) + ((size_t)blockIdx.z * tiles + tile_id) * (BM * BN) * 4
                             : static_cast<char*>(p.C) + ((size_t)m0 * p.ldc + n0) * 4;
    const int rows = part ? BM : (p.M - m0 < BM ? p.M - m0 : BM), cols = part ? BN : (p.N - n0 < BN ? p.N - n0 : BN);
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(obase, range31(((size_t)(rows - 1) * ldo + cols) * 4));
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int mt = 0; mt < MH; ++mt) {
            const int ml = h * HM + (wm * MH + mt) * 16 + r;
            if (ml >= rows) continue;
#pragma unroll
            for (int nt = 0; nt < Q0 + Q1; ++nt) {
                const int nl = nt < Q0 ? (wn * Q0 + nt) * 16 + 4 * g : W0 + (wn * Q1 + nt - Q0) * 16 + 4 * g;
                if (nl >= cols) continue;
                const acc_t v = acc[h][mt][nt];
                const uint32_t off = ((uint32_t)ml * ldo + (uint32_t)nl) * 4u;
                u32x4 o = __builtin_bit_cast(u32x4, v);
                if (!part && (DT == 0 || EPI == 1)) {
                    // past the last column the old values read zero and the results are not stored
                    f32x4 old = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (p.beta != 0.0f) old = __builtin_bit_cast(f32x4, buf_load_x4(rc, off));
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float oe = old[e];
                        if constexpr (DT == 0) {
                            o[e] = as_u32(epilogue(v[e], p.alpha, p.beta, &oe));
                        } else {
                            const int n = n0 + (nl + e < cols ? nl + e : nl);
                            o[e] = as_u32(s8_out(v[e], n, p.scale, p.amax, dq, p.beta, &oe));
                        }
                    }
                }
                if (nl + 4 <= cols) {
                    __builtin_amdgcn_raw_buffer_store_b128(o, rc, off, 0, 0);
                } else {
#pragma unroll
                    for (int e = 0; e < 3; ++e)
                        if (nl + e < cols) buf_store_x1(rc, off + 4u * e, o[e]);
                }
            }
        }
}

template <int TB, int MT, int Q0, int Q1>
__global__ __launch_bounds__(512, 2) void dnnopt_tile_bf16_dma_pp(PPArgs p) {
    pp_tile<0, TB, MT, Q0, Q1, 0>(p);
}
template <int EPI, int MT, int Q0, int Q1>
__global__ __launch_bounds__(512, 2) void dnnopt_s8_dma_pp(PPArgs p) {
    pp_tile<1, 1, MT, Q0, Q1, EPI>(p);
}

template <int MT, int Q0, int Q1>
static void launch_pp_shape(int dt, int tb, int epi, dim3 grid, const PPArgs& a, hipStream_t s) {
    if (dt == 1 && epi) hipLaunchKernelGGL((dnnopt_s8_dma_pp<1, MT, Q0, Q1>), grid, dim3(512), 0, s, a);
    else if (dt == 1) hipLaunchKernelGGL((dnnopt_s8_dma_pp<0, MT, Q0, Q1>), grid, dim3(512), 0, s, a);
    else if (tb) hipLaunchKernelGGL((dnnopt_tile_bf16_dma_pp<1, MT, Q0, Q1>), grid, dim3(512), 0, s, a);
    else hipLaunchKernelGGL((dnnopt_tile_bf16_dma_pp<0, MT, Q0, Q1>), grid, dim3(512), 0, s, a);
}

hipError_t launch_pp(int dt, int cfg, int tb, int epi, dim3 grid, const PPArgs& a, hipStream_t s) {
    if (dt == 1 && !tb) return hipErrorInvalidValue;
    switch (cfg) {
        case 0: launch_pp_shape<8, 2, 2>(dt, tb, epi, grid, a, s); break;  // 256 x 256
        case 1: launch_pp_shape<8, 2, 1>(dt, tb, epi, grid, a, s); break;  // 256 x 192
        case 2: launch_pp_shape<8, 2, 0>(dt, tb, epi, grid, a, s); break;  // 256 x 128
        case 3: launch_pp_shape<4, 2, 0>(dt, tb, epi, grid, a, s); break;  // 128 x 128
        case 4: launch_pp_shape<4, 2, 2>(dt, tb, epi, grid, a, s); break;  // 128 x 256
        case 5: launch_pp_shape<4, 2, 1>(dt, tb, epi, grid, a, s); break;  // 128 x 192
        case 6: launch_pp_shape<8, 1, 0>(dt, tb, epi, grid, a, s); break;  // 256 x 64
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace dnnopt_hip
