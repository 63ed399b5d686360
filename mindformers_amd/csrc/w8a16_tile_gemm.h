// W8A16 GEMM for many rows (prompts, chunked prefill): the matrix cores are the bound, not the weights.
#pragma once
#include "common.h"

// A workgroup of 4 waves (one per SIMD, two workgroups per compute unit) owns 32*MT rows x 256 channels; wave w owns channels
// 64w .. 64w + 63 of all the rows, so that every weight byte of the tile is loaded and converted by exactly one wave and goes
// from global memory straight into matrix operand registers, while the activation tile of a 64-wide k-step is staged in LDS
// once and read by all four.  Both operands are fetched two steps ahead by ordinary loads (the compiler counts them), the
// activations are written to the other of two LDS stages one step ahead, and the operands of a 16-wide sub-step are read and
// converted behind the matrix instructions of the one before (one instruction group per matrix instruction, pinned by
// scheduling groups); one barrier per step, in front of the last sub-step, whose operands are in registers by then.
//
// What bounds it: the power budget.  At 4096 x 4096 x 16384 the matrix pipes are busy 72 % of the cycles and the clock stands
// at 1.6 GHz (2.4 GHz with the conversions, loads and LDS traffic taken out), 1250 TFLOP/s; the library's bf16 GEMM draws the
// clock down to 1.5 GHz at 86 % (1362).  With MT = 8 (256 rows, one workgroup per unit) half the conversions and weight loads
// fall away, but nothing overlaps the start and the end of a tile: 1167 TFLOP/s there and 848 against 1100 at K = 4096.
// 4137 x 28672 x 4096: 1447 us in passes of 64 rows, 787 us here; 4137 x 4096 x 14336: 632 / 383 us.
namespace tg {

constexpr int WAVES = 4;
constexpr int BN = 64 * WAVES;                                // channels per workgroup
constexpr int KSTEP = 64;

// physical 16-byte chunk of chunk c of a staged activation row (128 bytes): the lanes that share an LDS cycle are those
// of one half-wave with equal parity of lane bits 2-4; bits 1, 3 and 4 of the row tell the eight rows of equal bit 0
// among them apart, so the 32-row operand reads and the writes are free of bank conflicts
__device__ __forceinline__ int key(int row) { return ((row >> 1) & 1) | (((row >> 3) & 3) << 1); }

template <typename T, int MT, typename Epilogue>
__device__ __forceinline__ void tile(const uint16_t* __restrict__ x, const uint8_t* __restrict__ wp, int M, int K, int m0,
                                     int tile0, int n_tiles, int s_begin, int s_end, uint8_t* smem, Epilogue&& epilogue) {
    using vec8 = typename T::vec8;
    constexpr int STAGE = 32 * MT * 128;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int h = lane >> 5, r32 = lane & 31;
    const int s_last = s_end - 1;

    // ---- activations: load i of a thread is chunk (t & 7) of row 32i + (t >> 3)
    const int xr = threadIdx.x >> 3, xc = threadIdx.x & 7;
    const uint8_t* xbase = (const uint8_t*)(x + (int64_t)m0 * K);
    uint32_t xoff[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) xoff[i] = (uint32_t)min(32 * i + xr, M - 1 - m0) * (uint32_t)K * 2u + 16u * xc;
    const uint32_t xdst = xr * 128 + ((xc ^ key(xr)) << 4);   // + 4096 per i (the key has no bit above 4)
    u32x4 xreg[2][MT];
    auto load_x = [&](auto setc, int s) {
        const uint32_t k = (uint32_t)min(s, s_last) * (KSTEP * 2);
#pragma unroll
        for (int i = 0; i < MT; ++i) xreg[decltype(setc)::value][i] = *(const u32x4*)(xbase + (xoff[i] + k));
    };
    auto write_x = [&](auto setc, int stage) {
#pragma unroll
        for (int i = 0; i < MT; ++i) *(u32x4*)(smem + stage * STAGE + 4096 * i + xdst) = xreg[decltype(setc)::value][i];
    };
    // ---- weights: of every 32-channel block (two packed tiles) and 64-wide step lane (r, h) holds chunks h and h + 2 of
    // its channel: columns 16h .. and 32 + 16h ..
    const uint8_t* wbase[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const int t = min(tile0 + 4 * wv + 2 * nt + ((lane >> 4) & 1), n_tiles - 1);
        wbase[nt] = wp + (int64_t)t * 1024 + h * 256 + (lane & 15) * 16;
    }
    u32x4 wreg[2][2][2];
    auto load_w = [&](auto setc, int s) {
        const int64_t off = (int64_t)min(s, s_last) * n_tiles * 1024;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int j = 0; j < 2; ++j) wreg[decltype(setc)::value][nt][j] = *(const u32x4*)(wbase[nt] + off + 512 * j);
    };
    // ---- operands of sub-step i (16 columns: 16h + 32(i >> 1) + 8(i & 1) + 0..7 in lane half h)
    const int frow = r32 * 128, fkey = key(r32);
    vec8 xf[2][MT], wf[2][2];
    auto read_x = [&](auto bufc, int stage, auto ic) {
        constexpr int I = decltype(ic)::value, B = decltype(bufc)::value;
        const int at = frow + (((2 * h + 4 * (I >> 1) + (I & 1)) ^ fkey) << 4);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xf[B][mt] = bitcast<vec8>(*(const u32x4*)(smem + stage * STAGE + 4096 * mt + at));
    };
    auto cvt_w = [&](auto bufc, auto setc, auto ic) {
        constexpr int I = decltype(ic)::value, S = decltype(setc)::value, B = decltype(bufc)::value;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
            wf[B][nt] = dequant8<T>(wreg[S][nt][I >> 1][2 * (I & 1)], wreg[S][nt][I >> 1][2 * (I & 1) + 1]);
    };
    f32x16 acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) acc[mt][nt] = (f32x16)(0.f);
    auto mul = [&](auto bufc) {
        constexpr int B = decltype(bufc)::value;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) acc[mt][nt] = T::mfma32(wf[B][nt], xf[B][mt], acc[mt][nt]);
    };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    using C3 = std::integral_constant<int, 3>;
    // one matrix instruction, then what hides behind it
    auto interleave = [&](auto readsc, auto valuc, auto writesc, auto loadsc) {
        constexpr int NM = 2 * MT;
        static_for<NM>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            constexpr int R = decltype(readsc)::value, V = decltype(valuc)::value, W = decltype(writesc)::value,
                          L = decltype(loadsc)::value;
            constexpr int r = (k + 1) * R / NM - k * R / NM, v = (k + 1) * V / NM - k * V / NM,
                          w = (k + 1) * W / NM - k * W / NM, l = (k + 1) * L / NM - k * L / NM;
            if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);
            if constexpr (w > 0) __builtin_amdgcn_sched_group_barrier(0x200, w, 0);
            if constexpr (l > 0) __builtin_amdgcn_sched_group_barrier(0x020, l, 0);
            if constexpr (v > 0) __builtin_amdgcn_sched_group_barrier(0x002, v, 0);
        });
        __builtin_amdgcn_sched_barrier(0);
    };

    load_x(C0{}, s_begin);
    load_w(C0{}, s_begin);
    load_x(C1{}, s_begin + 1);
    load_w(C1{}, s_begin + 1);
    write_x(C0{}, 0);
    load_x(C0{}, s_begin + 2);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    read_x(C0{}, 0, C0{});
    cvt_w(C0{}, C0{}, C0{});
    __builtin_amdgcn_sched_barrier(0);

    using CX = std::integral_constant<int, MT>;
    using CZ = std::integral_constant<int, 0>;
    using CV = std::integral_constant<int, 24>;
    auto step = [&](auto jc, int s) {
        constexpr int P = decltype(jc)::value;
        using CP = std::integral_constant<int, P>;
        using CQ = std::integral_constant<int, P ^ 1>;
        read_x(C1{}, P, C1{});
        cvt_w(C1{}, CP{}, C1{});
        write_x(CQ{}, P ^ 1);                                 // its readers passed the barrier of the step before
        mul(C0{});
        interleave(CX{}, CV{}, CX{}, CZ{});
        read_x(C0{}, P, C2{});
        cvt_w(C0{}, CP{}, C2{});
        load_x(CQ{}, s + 3);
        mul(C1{});
        interleave(CX{}, CV{}, CZ{}, CX{});
        read_x(C1{}, P, C3{});
        cvt_w(C1{}, CP{}, C3{});
        load_w(CP{}, s + 2);
        mul(C0{});
        interleave(CX{}, CV{}, CZ{}, std::integral_constant<int, 4>{});
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        read_x(C0{}, P ^ 1, C0{});
        cvt_w(C0{}, CQ{}, C0{});
        mul(C1{});
        interleave(CX{}, CV{}, CZ{}, CZ{});
    };
    int s = s_begin;
    for (; s + 2 <= s_end; s += 2) {
        step(C0{}, s);
        step(C1{}, s + 1);
    }
    if (s < s_end) step(C0{}, s);

    // lane (r, h) holds, of row 32mt + r, channels 8q + 4h .. + 3 of each 32-channel block in elements 4q .. 4q + 3
    // (compile-time indices: an accumulator indexed by a loop that is not unrolled would live in memory)
    static_for<MT>([&](auto mtc) { epilogue(mtc, acc[decltype(mtc)::value]); });
}

}  // namespace tg
