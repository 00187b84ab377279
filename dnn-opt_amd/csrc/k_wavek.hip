// k_wavek.hip -- fp32 MFMA tiles whose four waves split k (gfx950).
//
// Serves mid-size GEMMs of the reference's packed path
// (src/gemm/gemm_driver_generic.cpp:27-248): A stored M x K, B stored K x N or
// N x K, optional bias.
//
// What bounds it: the fp32 matrix cores, and how evenly a few hundred tiles
// spread over the CUs.  With the output split over the waves, a tile has to be
// a multiple of the waves' shape, its fragments are read by several waves, and
// every k-block ends at a barrier.  Here each wave owns 16 k of every 64-k
// block for the whole tile: it copies its own slices into a ring of its own
// (four stages, three ahead), waits for its own copies only, and reads every
// fragment once; the waves' sums are added in wave order at the end.  So a
// tile may be any number of 16 x 16 sub-tiles -- 96 x 48 gives 384 x 3072 256
// equal tiles -- and no barrier stands in the loop.  Measured (MI355X, us, the
// best of the other tiles -> this, in a graph): 384 x 3072 x 768 23.9 -> 20.6
// (B N x K, of which 11.8 at the rate of a large fp32 product, 154 TFLOP/s) and
// 27.5 -> 21.1 (K x N), x 3072 79.4 -> 61.8 and 78.5 -> 64.0, 384 x 768 x 768
// 11.1 -> 9.0.  In a kernel trace K = 768 and 3072 take 22.7 and 61.1 (B N x K):
// 1.07 us per block of 64 k, 9.9 us of launch, first copies from HBM and
// epilogue.  The order within a step matters little (MFMAs of a step before,
// between or after its reads and copies: 20.6-22.2).
#include <type_traits>

#include "device_common.h"
#include "kernels.h"

using namespace dnnopt_dev;

namespace dnnopt_hip {

// Tile 16 MT x 16 NT.  Rows of A and B stored N x K are copied 64 bytes (16 k)
// at a time, one wave load filling exactly one MFMA operand (16 rows), read
// back without a swizzle: the 64-byte steps between lanes cost bank conflicts
// (0.55 conflict cycles per active LDS cycle with B N x K, MFMAs busy 64% of a
// launch, both over 384 x 3072 x 768 and x 3072).  A K x N B is copied as 16
// rows of k; lane r of an operand takes columns NT r .. NT r + NT - 1 of the
// tile, one LDS read per row of k, so its sub-tiles' columns interleave.
// Offsets are 32-bit from the tile's first row over all of k (f32_dma_fits).
template <int MT, int NT, int TB>
__global__ __launch_bounds__(256, 1) void dnnopt_tile_f32_dma_wavek(TileArgs p) {
    constexpr int BM = 16 * MT, BN = 16 * NT;
    constexpr int UB = TB ? NT : (NT == 2 ? 2 : 4);  // 1 KB wave loads of B per step
    constexpr int U = MT + UB;
    constexpr int WST = U * 1024;                   // bytes of a wave's stage
    static_assert(BM * BN * 4 <= 4 * WST, "a wave's partial tile fits one stage array");
    static_assert(TB || (NT >= 2 && NT <= 4), "a lane of a K x N B reads 2 to 4 columns");
    __shared__ __attribute__((aligned(1024))) char st0[4 * WST];
    __shared__ __attribute__((aligned(1024))) char st1[4 * WST];
    __shared__ __attribute__((aligned(1024))) char st2[4 * WST];
    __shared__ __attribute__((aligned(1024))) char st3[4 * WST];

    const int lane = lane_id(), r = lane & 15, g = lane >> 4;
    const int w = wave_id();
    const TileXY tile = xcd_tile((int)blockIdx.x, p.tiles_n, p.tiles_m);
    if (!tile.ok) return;
    const int m0 = tile.m * BM, n0 = tile.n * BN;
    const int nblk = (p.K + 63) / 64;
    const int b_lo = (int)(((long long)nblk * blockIdx.z) / p.splits);
    const int b_hi = (int)(((long long)nblk * (blockIdx.z + 1)) / p.splits);
    const int nb = b_hi - b_lo;

    const char* abase = static_cast<const char*>(p.A) + (size_t)m0 * p.lda * 4;
    const char* bbase = static_cast<const char*>(p.B) + (TB ? (size_t)n0 * p.ldb : (size_t)n0) * 4;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(abase, range31(((size_t)(p.M - 1 - m0) * p.lda + p.K) * 4));
    const size_t b_last = TB ? (size_t)(p.N - 1 - n0) * p.ldb + p.K : (size_t)(p.K - 1) * p.ldb + (p.N - n0);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(bbase, range31(b_last * 4));

    // k-contiguous rows: wave load u fills 16 rows of 64 bytes (16 k), lane l
    // row l / 4, chunk l % 4: exactly one MFMA operand.
    const int lrow = lane >> 2, lch = lane & 3;
    uint32_t ga[MT], gb[UB];
#pragma unroll
    for (int u = 0; u < MT; ++u) {
        const int row = 16 * u + lrow;
        ga[u] = m0 + row < p.M ? ((uint32_t)row * (uint32_t)p.lda + 4u * lch) * 4u : kOobOffset;
    }
    // K x N: 16 rows of k, 16 lanes' NT columns each in 16 bytes (NT = 3: the
    // chunks overlap by a column in memory) or, NT = 2, 8 bytes.
    constexpr int BROW = NT == 2 ? 128 : 256;  // bytes of a k row in LDS
    int bk[UB];                                // k row of this lane in load u
#pragma unroll
    for (int u = 0; u < UB; ++u) {
        if constexpr (TB) {
            const int row = 16 * u + lrow;
            bk[u] = 0;
            gb[u] = n0 + row < p.N ? ((uint32_t)row * (uint32_t)p.ldb + 4u * lch) * 4u : kOobOffset;
        } else {
            const int q = u * 1024 + 16 * lane, kr = q / BROW, ch = (q % BROW) / 16;
            bk[u] = kr;
            gb[u] = ((uint32_t)kr * (uint32_t)p.ldb + (uint32_t)((NT == 3 ? 3 : 4) * ch)) * 4u;
        }
    }
    // Chunks and rows past K, and steps past the split's end, read zero (the
    // copies are issued all the same: every step has as many).
    auto dma_a = [&](char* st, int i) {
        const int k0 = (b_lo + i) * 64 + 16 * w;
        const bool cut = i >= nb || k0 + 4 * lch >= p.K;
#pragma unroll
        for (int u = 0; u < MT; ++u)
            lds_dma16(ra, st + w * WST + u * 1024, cut ? kOobOffset : ga[u] + (uint32_t)k0 * 4u);
    };
    auto dma_b = [&](char* st, int i) {
        const int k0 = (b_lo + i) * 64 + 16 * w;
        const uint32_t kb = TB ? (uint32_t)k0 * 4u : (uint32_t)k0 * (uint32_t)p.ldb * 4u;
#pragma unroll
        for (int u = 0; u < UB; ++u) {
            const bool cut = i >= nb || k0 + (TB ? 4 * lch : bk[u]) >= p.K;
            lds_dma16(rb, st + w * WST + (MT + u) * 1024, cut ? kOobOffset : gb[u] + kb);
        }
    };

    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Fragments: A [mt] and, N x K, B [nt] hold k = 4 g + c in component c;
    // K x N, B [c] holds the lane's NT columns of k = 4 g + c.
    constexpr int FB = TB ? NT : 4;
    f32x4 fa[2][MT], fb[2][FB];
    auto read = [&](const char* st, auto slot) {
        constexpr int S = decltype(slot)::value;
        const char* base = st + w * WST;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) fa[S][mt] = *reinterpret_cast<const f32x4*>(base + mt * 1024 + r * 64 + g * 16);
        if constexpr (TB) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                fb[S][nt] = *reinterpret_cast<const f32x4*>(base + (MT + nt) * 1024 + r * 64 + g * 16);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const char* row = base + MT * 1024 + (4 * g + c) * BROW + r * (BROW / 16);
                if constexpr (NT == 2) {
                    typedef float f32x2 __attribute__((ext_vector_type(2)));
                    const f32x2 v = *reinterpret_cast<const f32x2*>(row);
                    fb[S][c] = f32x4{v[0], v[1], 0.f, 0.f};
                } else {
                    fb[S][c] = *reinterpret_cast<const f32x4*>(row);
                }
            }
        }
    };
    // Zeroes the elements past K of the last block's chunk that holds K - 1.
    auto mask = [&](int i, auto slot) {
        constexpr int S = decltype(slot)::value;
        if ((b_lo + i + 1) * 64 <= p.K || (p.K & 3) == 0) return;
        const int kv = p.K - ((b_lo + i) * 64 + 16 * w + 4 * g);  // elements of this lane's chunk before K
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) fa[S][mt][c] = c < kv ? fa[S][mt][c] : 0.f;
            if constexpr (TB) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) fb[S][nt][c] = c < kv ? fb[S][nt][c] : 0.f;
            }
        }
    };
    auto mma = [&](auto slot, int c) {
        constexpr int S = decltype(slot)::value;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(TB ? fb[S][TB ? nt : 0][c] : fb[S][TB ? 0 : c][nt],
                                                                  fa[S][mt][c], acc[mt][nt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    // Step i: a quarter of its MFMAs, then the fragments of step i + 1 (its
    // copies are the oldest in flight) are read under the second quarter and
    // step i + 3 is copied, into the stage step i - 1 left, under the others.
    // A wave reads only what it copied itself: no barrier.
    auto step = [&](int i, char* next, char* fill, auto odd) {
        constexpr int O = decltype(odd)::value;
        constexpr std::integral_constant<int, O> cur{};
        constexpr std::integral_constant<int, 1 - O> nxt{};
        mma(cur, 0);
        wait_vmcnt<U>();
        read(next, nxt);
        __builtin_amdgcn_sched_barrier(0);
        mma(cur, 1);
        dma_a(fill, i + 3);
        __builtin_amdgcn_sched_barrier(0);
        mma(cur, 2);
        dma_b(fill, i + 3);
        __builtin_amdgcn_sched_barrier(0);
        mma(cur, 3);
        mask(i + 1, nxt);
    };
    auto dma = [&](char* st, int i) {
        dma_a(st, i);
        dma_b(st, i);
    };
    dma(st0, 0);
    dma(st1, 1);
    dma(st2, 2);
    wait_vmcnt<2 * U>();
    read(st0, I0{});
    mask(0, I0{});
    int i = 0;
    for (; i + 4 <= nb; i += 4) {
        step(i, st1, st3, I0{});
        step(i + 1, st2, st0, I1{});
        step(i + 2, st3, st1, I0{});
        step(i + 3, st0, st2, I1{});
    }
    if (i < nb) step(i, st1, st3, I0{});
    if (i + 1 < nb) step(i + 1, st2, st0, I1{});
    if (i + 2 < nb) step(i + 2, st3, st1, I0{});
    wait_vmcnt<0>();
    __syncthreads();

    // The four waves' sums, each as a row-major tile in a stage array of its
    // own, added in wave order.  Lane (r, g): row r of a sub-tile, columns
    // 4 g .. 4 g + 3 (N x K) or the lane's 4 NT consecutive ones.
    auto part_of = [&](int q) { return reinterpret_cast<float*>(q == 0 ? st0 : q == 1 ? st1 : q == 2 ? st2 : st3); };
    float* mine = part_of(w);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            f32x4 v = acc[mt][nt];
            if constexpr (!TB) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = acc[mt][(4 * nt + e) % NT][(4 * nt + e) / NT];
            }
            const int col = TB ? nt * 16 + 4 * g : 4 * NT * g + 4 * nt;
            *reinterpret_cast<f32x4*>(mine + (mt * 16 + r) * BN + col) = v;
        }
    __syncthreads();
    const bool split = p.splits > 1;
    const int rows = split ? BM : (p.M - m0 < BM ? p.M - m0 : BM), cols = split ? BN : (p.N - n0 < BN ? p.N - n0 : BN);
    const uint32_t ldo = split ? (uint32_t)BN : (uint32_t)p.ldc;
    const int tiles = p.tiles_n * p.tiles_m, tile_id = tile.m * p.tiles_n + tile.n;
    float* obase = split ? p.part + ((size_t)blockIdx.z * tiles + tile_id) * (BM * BN) : p.C + (size_t)m0 * p.ldc + n0;
    const __amdgpu_buffer_rsrc_t rc = make_rsrc(obase, range31(((size_t)(rows - 1) * ldo + cols) * 4));
    constexpr int Q4 = BN / 4;
    for (int q = (int)threadIdx.x; q < BM * Q4; q += 256) {
        const int row = q / Q4, col = 4 * (q % Q4);
        f32x4 s = *reinterpret_cast<const f32x4*>(reinterpret_cast<float*>(st0) + 4 * q);
        s += *reinterpret_cast<const f32x4*>(reinterpret_cast<float*>(st1) + 4 * q);
        s += *reinterpret_cast<const f32x4*>(reinterpret_cast<float*>(st2) + 4 * q);
        s += *reinterpret_cast<const f32x4*>(reinterpret_cast<float*>(st3) + 4 * q);
        if (row >= rows || col >= cols) continue;
        const uint32_t off = ((uint32_t)row * ldo + (uint32_t)col) * 4u;
        u32x4 o = __builtin_bit_cast(u32x4, s);
        if (!split) {
            f32x4 old = f32x4{0.f, 0.f, 0.f, 0.f};
            if (p.beta != 0.0f) old = __builtin_bit_cast(f32x4, buf_load_x4(rc, off));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float oe = old[e];
                const int n = n0 + (col + e < cols ? col + e : col);
                o[e] = as_u32(add_bias(epilogue(s[e], p.alpha, p.beta, &oe), p.bias, n));
            }
        }
        if (col + 4 <= cols) {
            __builtin_amdgcn_raw_buffer_store_b128(o, rc, off, 0, 0);
        } else {
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (col + e < cols) buf_store_x1(rc, off + 4u * e, o[e]);
        }
    }
}

template <int MT, int NT>
static void launch_wavek_shape(int tb, dim3 grid, const TileArgs& a, hipStream_t s) {
    if (tb) hipLaunchKernelGGL((dnnopt_tile_f32_dma_wavek<MT, NT, 1>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((dnnopt_tile_f32_dma_wavek<MT, NT, 0>), grid, dim3(256), 0, s, a);
}

hipError_t launch_tile_f32_wavek(int cfg, int tb, dim3 grid, const TileArgs& a, hipStream_t s) {
    switch (cfg) {
        case 0: launch_wavek_shape<6, 3>(tb, grid, a, s); break;  // 96 x 48
        case 1: launch_wavek_shape<4, 4>(tb, grid, a, s); break;  // 64 x 64
        case 2: launch_wavek_shape<4, 3>(tb, grid, a, s); break;  // 64 x 48
        case 3: launch_wavek_shape<3, 3>(tb, grid, a, s); break;  // 48 x 48
        case 4: launch_wavek_shape<4, 2>(tb, grid, a, s); break;  // 64 x 32
        case 5: launch_wavek_shape<2, 3>(tb, grid, a, s); break;  // 32 x 48
        case 6: launch_wavek_shape<2, 4>(tb, grid, a, s); break;  // 32 x 64
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace dnnopt_hip
