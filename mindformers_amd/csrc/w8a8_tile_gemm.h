// W8A8 GEMM for many rows, exact int32 sums.
#pragma once
#include "common.h"

// A workgroup of 4 waves owns 32*MT rows x 256 channels, wave w channels 64w .. 64w + 63 of all the rows
// (v_mfma_i32_32x32x32_i8).  A packed weight tile is the matrix operand, so weights go from global memory into operand
// registers and nowhere else; the activations of a 64-wide step (tile order too) are staged in LDS once for the four waves.
// Loads run three steps ahead of their use in three register sets, the LDS stage of a step is written one step ahead, and the
// operands of a sub-step (32 columns) are read behind the matrix instructions of the one before; one barrier per step.
//
// The 16x16x64 int8 instruction issues at half the rate of the 32x32x32 one here (2.4 against 4.4 POP/s with independent
// accumulators).  What bounds the kernel is the operand traffic out of L2 (24 KiB per 4.2 M operations a step, 171 op/B, about
// 12 TB/s) and, with it, the power budget: 2405 TOP/s at 4096 x 4096 x 16384 from warm caches, 2070 at 4137 x 28672 x 4096 with
// cold weights.  1531 x 37888 x 3584: 275 us on 256 x 192 tiles of 8 waves with both operands through an LDS ring, 250 here;
// 1531 x 3584 x 18944: 181 us on the register-streaming kernel, 120 here.  Row panels of 8 or 16 blocks instead of 4, or
// neighbouring tiles paired on one compute unit, change nothing.
namespace tq {

constexpr int WAVES = 4;
constexpr int BN = 64 * WAVES;
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
    __device__ __forceinline__ TiledRows(const uint8_t* xq, int m_tile0, int m_tiles) : step((int64_t)m_tiles * 1024) {
#pragma unroll
        for (int i = 0; i < XL; ++i)
            p[i] = xq + (int64_t)min(m_tile0 + 4 * i + (int)(threadIdx.x >> 6), m_tiles - 1) * 1024 + (threadIdx.x & 63) * 16;
    }
    __device__ __forceinline__ i32x4 load(int i, int s) const { return *(const i32x4*)(p[i] + s * step); }
};
template <int XL>
struct PlainRows {                                            // rows m0 .. of `rows` rows of K (a multiple of 16) bytes
    const uint8_t* p[XL];
    int last;                                                 // columns past K are clamped: their weights are zero
    __device__ __forceinline__ PlainRows(const uint8_t* xq, int m0, int rows, int K) {
        const int r = threadIdx.x & 15, c = 16 * ((threadIdx.x >> 4) & 3);
#pragma unroll
        for (int i = 0; i < XL; ++i)
            p[i] = xq + (int64_t)min(m0 + 16 * (4 * i + (int)(threadIdx.x >> 6)) + r, rows - 1) * K + c;
        last = K - 16 - c;
    }
    __device__ __forceinline__ i32x4 load(int i, int s) const { return *(const i32x4*)(p[i] + min(s * KSTEP, last)); }
};

// tile0: first 16-channel tile of the weights, n_tiles: tiles of a step
template <int MT, typename Rows, typename Epilogue>
__device__ __forceinline__ void tile(const Rows& x, const uint8_t* __restrict__ wp, int tile0, int n_tiles, int s_begin,
                                     int s_end, uint8_t* smem, Epilogue&& epilogue) {
    constexpr int XL = XLOADS<MT>, STAGE = 64 * XL * KSTEP;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int h = lane >> 5;
    const int s_last = s_end - 1;
    i32x4 xreg[D][XL], wreg[D][2][2];
    auto load_x = [&](auto setc, int s) {
#pragma unroll
        for (int i = 0; i < XL; ++i) xreg[decltype(setc)::value][i] = x.load(i, min(s, s_last));
    };
    auto write_x = [&](auto setc, int stage) {
#pragma unroll
        for (int i = 0; i < XL; ++i)
            *(i32x4*)(smem + stage * STAGE + (4 * i + wv) * 1024 + lane * 16) = xreg[decltype(setc)::value][i];
    };
    // lane (r, h) of a 32-row operand: row r & 15 of tile r >> 4, columns 32u + 16h .. of sub-step u
    const int lane32 = ((lane >> 4) & 1) * 1024 + h * 256 + (lane & 15) * 16;
    const uint8_t* wbase[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const int t = min(tile0 + 4 * wv + 2 * nt + ((lane >> 4) & 1), n_tiles - 1);
        wbase[nt] = wp + (int64_t)t * 1024 + h * 256 + (lane & 15) * 16;
    }
    auto load_w = [&](auto setc, int s) {
        const int64_t off = (int64_t)min(s, s_last) * n_tiles * 1024;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int u = 0; u < 2; ++u) wreg[decltype(setc)::value][nt][u] = *(const i32x4*)(wbase[nt] + off + 512 * u);
    };
    i32x4 xf[2][MT];
    auto read_x = [&](auto bufc, int stage) {                 // buffer = sub-step
        constexpr int B = decltype(bufc)::value;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[B][mt] = *(const i32x4*)(smem + stage * STAGE + mt * 2048 + 512 * B + lane32);
    };
    i32x16 acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) acc[mt][nt] = (i32x16)(0);
    auto mul = [&](auto bufc, auto setc) {
        constexpr int B = decltype(bufc)::value, S = decltype(setc)::value;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
                acc[mt][nt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wreg[S][nt][B], xf[B][mt], acc[mt][nt], 0, 0, 0);
    };
    // one matrix instruction, then what hides behind it
    auto interleave = [&](auto writesc, auto loadsc) {
        constexpr int NM = 2 * MT, R = MT, W = decltype(writesc)::value, L = decltype(loadsc)::value;
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
    static_for<D>([&](auto dc) {
        load_x(dc, s_begin + decltype(dc)::value);
        load_w(dc, s_begin + decltype(dc)::value);
    });
    write_x(C0{}, 0);
    load_x(C0{}, s_begin + D);
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
    // lane (r, h) holds, of row 32mt + r, channels 8q + 4h .. + 3 of each 32-channel block in elements 4q .. 4q + 3
    static_for<MT>([&](auto mtc) { epilogue(mtc, acc[decltype(mtc)::value]); });
}

}  // namespace tq
