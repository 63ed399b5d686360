// W8A8 GEMM for many rows, exact int32 sums.
#pragma once
#include "common.h"
#include "tile_grid.h"

// A workgroup of 4 waves owns 32*MT rows x 64*NT channels (see tg_plan), wave w the w-th quarter of the channels of all the rows.  A packed weight tile is
// the operand of v_mfma_i32_16x16x64_i8 as it lies, so weights go from global memory into operand registers and nowhere else; the
// activations of a 64-wide step (tile order too) are staged in LDS once for the four waves.  Loads run three steps ahead of their use
// in three register sets, the LDS stage of a step is written one step ahead, and the rows of half a step are read behind the
// matrix instructions of the half before; one barrier per step.
//
// With all operands in registers 16x16x64 does 4345 TOP/s on random data and 32x32x32 3727 (4866 and 4976 on zeros): both fill the
// matrix pipe, and the smaller one, which reads and writes half the accumulators per operation, leaves the power budget more clock.
// What bounds the kernel is the operand traffic out of L2 (24 KiB per 4.2 M operations a step, 171 op/B, about 12 TB/s) and that
// budget: 4096 x 4096 x 16384 from warm caches 248 us on 32x32x32, 219 here (2515 TOP/s), 1531 x 37888 x 3584 with cold weights
// 203 / 187, 2077 x 4096 x 7168 73 / 67, 1531 x 3584 x 18944 118 / 118 on 168 tiles, one on a compute unit (on the 228 of
// 128 x 192 that it runs on 104).  1531 x 37888 x 3584 on 256 x 192 tiles of 8 waves with both operands through an LDS ring: 232 to 275.  Row panels of 8 or 16 blocks instead of 4, or neighbouring
// tiles paired on one compute unit, change nothing.
namespace tq {

constexpr int WAVES = 4;
template <int NT>
constexpr int BN_OF = 16 * NT * WAVES;                       // channels per workgroup of NT 16-channel tiles a wave
constexpr int BN = BN_OF<4>;
constexpr int KSTEP = 64;
constexpr int D = 3;                                          // register sets

// 16-row activation tiles that each of the four waves loads and stages per step (three 32-row blocks: as for four, the last
// two tiles are not read back)
template <int MT>
constexpr int XLOADS = (MT + 1) / 2;
template <int MT>
constexpr int LDS_BYTES = 2 * 64 * XLOADS<MT> * KSTEP;

// Where the activations come from: 16-row tile 4i + wave of the workgroup is load i of a wave, lane (r, g) of it row r, columns
// 16g .. + 15 of the step.
template <int XL>
struct TiledRows {                                            // tile order: whole KiB, m_tiles of them a step
    const uint8_t* p[XL];
    int64_t step;
    __device__ __forceinline__ TiledRows(const uint8_t* xq, int m_tile0, int m_tiles, int wv) : step((int64_t)m_tiles * 1024) {
#pragma unroll
        for (int i = 0; i < XL; ++i) p[i] = xq + (int64_t)min(m_tile0 + 4 * i + wv, m_tiles - 1) * 1024;
    }
    __device__ __forceinline__ i32x4 load(int i, int s) const {
        return bitcast<i32x4>(load16_at(p[i] + s * step, (threadIdx.x & 63) * 16));
    }
};
template <int XL>
struct PlainRows {                                            // rows m0 .. of a group of `rows` rows from row0 on, of K (a multiple of 16) bytes
    const uint8_t* p;
    uint32_t row[XL];
    int c, last;                                              // columns past K are clamped: their weights are zero
    __device__ __forceinline__ PlainRows(const uint8_t* xq, const TileSources& src, int row0, int m0, int rows, int K, int wv)
        : p(src.sources ? xq : xq + (int64_t)(row0 + m0) * K) {
        c = 16 * ((threadIdx.x >> 4) & 3);
        last = K - 16;
#pragma unroll
        for (int i = 0; i < XL; ++i) {
            const int in = min(16 * (4 * i + wv) + (int)(threadIdx.x & 15), rows - 1 - m0);
            row[i] = (uint32_t)(src.sources ? src.of(row0 + m0 + in) : in) * (uint32_t)K;
        }
    }
    __device__ __forceinline__ i32x4 load(int i, int s) const {
        return bitcast<i32x4>(load16_at(p, row[i] + (uint32_t)min(s * KSTEP + c, last)));
    }
};

// tile0: first 16-channel tile of the weights, n_tiles: tiles of a step.  half (0: none): the second half of a wave's tiles are those
// `half` tiles after the first half, the up projection's beside the gate's
// STREAM: weights that nobody else reads (non-temporal loads)
template <int MT, int NT, bool STREAM, typename Rows, typename Epilogue>
__device__ __forceinline__ void tile(const Rows& x, const uint8_t* __restrict__ wp, int tile0, int n_tiles, int half, int s_begin,
                                     int s_end, uint8_t* smem, Epilogue&& epilogue) {
    constexpr int XL = XLOADS<MT>, STAGE = 64 * XL * KSTEP;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s_last = s_end - 1;
    i32x4 xreg[D][XL], wreg[D][NT];
    auto load_x = [&](auto setc, int s) {
#pragma unroll
        for (int i = 0; i < XL; ++i) xreg[decltype(setc)::value][i] = x.load(i, min(s, s_last));
    };
    auto write_x = [&](auto setc, int stage) {
#pragma unroll
        for (int i = 0; i < XL; ++i)
            *(i32x4*)(smem + stage * STAGE + (4 * i + wv) * 1024 + lane * 16) = xreg[decltype(setc)::value][i];
    };
    // weights: a packed tile is the matrix operand of 16 channels x 64 columns; the tile addresses are the same in every lane
    const uint8_t* wbase[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int pair = tile0 + NT / 2 * wv + nt % (NT / 2);
        const int t = half ? min(pair, half - 1) + (nt >= NT / 2 ? half : 0) : min(tile0 + NT * wv + nt, n_tiles - 1);
        wbase[nt] = wp + (int64_t)t * 1024;
    }
    const uint32_t lane16 = lane * 16;
    auto load_w = [&](auto setc, int s) {
        const int64_t off = (int64_t)min(s, s_last) * n_tiles * 1024;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) wreg[decltype(setc)::value][nt] = bitcast<i32x4>(load16_at<STREAM>(wbase[nt] + off, lane16));
    };
    // activations of 16-row tile t: one KiB in operand order; tiles 0 .. MT - 1 make the first half of a step, the others the second
    i32x4 xf[2][MT];
    auto read_x = [&](auto bufc, int stage) {                 // buffer = half
        constexpr int B = decltype(bufc)::value;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[B][mt] = *(const i32x4*)(smem + stage * STAGE + (B * MT + mt) * 1024 + lane16);
    };
    i32x4 acc[MT][2][NT];                                     // [32-row block][16-row tile of it][16-channel tile]
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 2 * NT; ++j) acc[mt][j / NT][j % NT] = (i32x4)(0);
    auto mul = [&](auto bufc, auto setc) {
        constexpr int B = decltype(bufc)::value, S = decltype(setc)::value;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                i32x4& a = acc[(B * MT + mt) >> 1][(B * MT + mt) & 1][nt];
                a = __builtin_amdgcn_mfma_i32_16x16x64_i8(wreg[S][nt], xf[B][mt], a, 0, 0, 0);
            }
    };
    // one matrix instruction, then what hides behind it
    auto interleave = [&](auto writesc, auto loadsc) {
        constexpr int NM = NT * MT, R = MT, W = decltype(writesc)::value, L = decltype(loadsc)::value;
        static_for<NM>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            constexpr int r = (k + 1) * R / NM - k * R / NM, w = (k + 1) * W / NM - k * W / NM, l = (k + 1) * L / NM - k * L / NM;
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);
            if constexpr (w > 0) __builtin_amdgcn_sched_group_barrier(0x200, w, 0);
            if constexpr (l > 0) __builtin_amdgcn_sched_group_barrier(0x020, l, 0);
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    // (in the order of the loop, whose waits the compiler counts for both ways into it)
    load_x(C0{}, s_begin);
    static_for<D>([&](auto dc) {
        constexpr int d = decltype(dc)::value;
        if constexpr (d == D - 1) write_x(C0{}, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_x(std::integral_constant<int, (d + 1) % D>{}, s_begin + d + 1);
        __builtin_amdgcn_sched_barrier(0);
        load_w(dc, s_begin + d);
        __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    read_x(C0{}, 0);
    __builtin_amdgcn_sched_barrier(0);

    auto step = [&](auto jc, int s) {
        constexpr int J = decltype(jc)::value, P = J & 1;     // LDS stage P, register set J % D
        using CS = std::integral_constant<int, J % D>;
        using CN = std::integral_constant<int, (J + 1) % D>;
        read_x(C1{}, P);
        write_x(CN{}, P ^ 1);                                 // its readers passed the barrier of the step before
        mul(C0{}, CS{});
        interleave(std::integral_constant<int, XL>{}, C0{});
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        read_x(C0{}, P ^ 1);
        load_x(CN{}, s + 1 + D);
        mul(C1{}, CS{});
        interleave(C0{}, std::integral_constant<int, XL>{});
        load_w(CS{}, s + D);
        __builtin_amdgcn_sched_barrier(0);
    };
    int s = s_begin;
    for (; s + 2 * D <= s_end; s += 2 * D) static_for<2 * D>([&](auto jc) { step(jc, s + decltype(jc)::value); });
    static_for<2 * D - 1>([&](auto jc) {
        if (s + decltype(jc)::value < s_end) step(jc, s + decltype(jc)::value);
    });
    // lane (r, g) holds, of row 32mt + 16j + r, channels 4g .. + 3 of each 16-channel tile
    static_for<MT>([&](auto mtc) { epilogue(mtc, acc[decltype(mtc)::value]); });
}

}  // namespace tq
