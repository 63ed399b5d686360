// W8A16 GEMM for many rows (prompts, chunked prefill): the matrix cores are the bound, not the weights.
#pragma once
#include "common.h"
#include "tile_grid.h"

// A workgroup of 4 waves (one per SIMD, two workgroups per compute unit) owns 32*MT rows x 64*NT channels (MT and NT: 3 or 4, see
// tg_plan; fewer rows in a group's or a plan's last block); wave w owns the w-th quarter of the channels of all the rows, so that every weight byte of the tile is loaded and converted by exactly one wave and goes
// from global memory straight into matrix operand registers, while the activation tile of a 64-wide k-step is staged in LDS
// once and read by all four.  Weights are fetched two steps ahead by ordinary loads (the compiler counts them); the activations of a
// step are written to the other of two LDS stages one step ahead.  A step is 2*NT groups, (32 columns, 16 channels) each over all
// the rows: a group's 2*MT matrix instructions share one weight operand, and behind each of them goes a piece of what is needed
// next (the conversion of the next group's weights, a row tile of the next 32 columns, a load), in the order written here; one
// barrier per step, in front of the groups that begin to read the next one.
//
// v_mfma_f32_16x16x32: with all operands in registers and two waves a SIMD, 16x16x32 does 2007 TFLOP/s on random data and 2437 on
// zeros, 32x32x16 1818 and 2484: both fill the matrix pipe, and the smaller one, which reads and writes half the accumulators per
// operation, leaves the power budget more clock.  The accumulators are held in the accumulation registers by the statements that
// name them: left to the compiler 32 accumulators of four registers wander through the file and spill.
//
// What bounds it: the power budget.  4137 x 28672 x 4096: 782-797 us on 32x32x16, 714-724 here (1360 TFLOP/s); 4137 x 4096 x 14336:
// 398 / 351-359; 2025 x 7168 x 16384: 424 / 350-360.  A lone workgroup on a compute unit (few tiles) is bound by issue: one wave starts a
// vector instruction every 8 cycles, and a step of 128 x 256 has 96 beside 64 matrix instructions of 16 (0.7 to 0.9 us a step, two
// workgroups together 1.55; 96 x 256 0.60, 128 x 192 0.56, 96 x 192 0.48).
namespace tg {

constexpr int WAVES = 4;
template <int NT>
constexpr int BN_OF = 16 * NT * WAVES;                       // channels per workgroup of NT 16-channel tiles a wave
constexpr int BN = BN_OF<4>;
constexpr int KSTEP = 64;
constexpr int DW = 2;                                         // steps of weights in flight
template <int MT>
constexpr int DX = MT == 4 ? 1 : 2;                           // steps of activations in flight
// physical 16-byte chunk of chunk c of a staged activation row (128 bytes): the lanes that share an LDS cycle are those
// of one half-wave with equal parity of lane bits 2-4.  An operand read has row bits 0-3 in lane bits 0-3 and chunk bit 1 in lane
// bit 4, a write has the chunk in bits 0-2 and row bits 0-1 above; with this key the sixteen lanes of a cycle meet the sixteen
// chunks of two rows in both
__device__ __forceinline__ int key(int row) { return ((row >> 1) & 1) | (((row >> 3) & 1) << 2); }

// EARLY: 16-row tiles of a sub-step that are read behind the last but one channel tile of the one before; the others follow behind the
// last, each into the registers of a tile that has just been used (0: half and half).  STREAM: weights that nobody else reads (non-temporal loads)
// row_of(r): the row of x that is row r of the tile (the last one where the tile has no such row), within 32-bit byte offsets
template <typename T, int MT, int NT, int EARLY, bool STREAM, typename RowOf, typename Epilogue>
__device__ __forceinline__ void tile(const uint16_t* __restrict__ x, RowOf&& row_of, const uint8_t* __restrict__ wp, int K,
                                     int tile0, int n_tiles, int s_begin, int s_end, uint8_t* smem, Epilogue&& epilogue) {
    using vec8 = typename T::vec8;
    constexpr int STAGE = 32 * MT * 128;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s_last = s_end - 1;

    // ---- activations: load i of a thread is chunk (t & 7) of row 32i + (t >> 3)
    const int xr = threadIdx.x >> 3, xc = threadIdx.x & 7;
    const uint8_t* xbase = (const uint8_t*)x;
    uint32_t xoff[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) xoff[i] = (uint32_t)row_of(32 * i + xr) * (uint32_t)K * 2u + 16u * xc;
    const uint32_t xdst = xr * 128 + ((xc ^ key(xr)) << 4);   // + 4096 per i (the key has no bit above 3)
    u32x4 xreg[DX<MT>][MT];
    auto load_x = [&](auto setc, auto ic, int s) {
        constexpr int i = decltype(ic)::value;
        xreg[decltype(setc)::value][i] = load16_at(xbase + (uint32_t)min(s, s_last) * (KSTEP * 2), xoff[i]);
    };
    auto write_x = [&](auto setc, auto ic, int stage) {
        constexpr int i = decltype(ic)::value;
        *(u32x4*)(smem + stage * STAGE + 4096 * i + xdst) = xreg[decltype(setc)::value][i];
    };
    // ---- weights: lane (r, g) of a packed 16-channel tile holds columns 16g .. 16g + 15 of channel r
    const uint8_t* wbase[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wbase[nt] = wp + (int64_t)min(tile0 + NT * wv + nt, n_tiles - 1) * 1024;
    u32x4 wreg[DW][NT];
    auto load_w = [&](auto setc, auto nc, int s) {
        constexpr int nt = decltype(nc)::value;
        wreg[decltype(setc)::value][nt] = load16_at<STREAM>(wbase[nt] + (int64_t)min(s, s_last) * n_tiles * 1024, lane * 16);
    };
    // ---- operands: a sub-step u of a step is 32 columns, 16g + 8u .. + 7 in lane (r, g).  The rows of a sub-step stay in registers
    // while the wave's four channel tiles pass by, converted one ahead
    const int frow = (lane & 15) * 128, fkey = key(lane & 15);
    vec8 xf[2][2 * MT], wf;
    auto read_x = [&](auto mc, int stage, auto uc) {
        constexpr int m = decltype(mc)::value, U = decltype(uc)::value;
        const int at = frow + (((2 * (lane >> 4) + U) ^ fkey) << 4);
        xf[U][m] = bitcast<vec8>(*(const u32x4*)(smem + stage * STAGE + 2048 * m + at));
    };
    f32x4 acc[MT][2][NT];                                     // [32-row block][16-row tile of it][16-channel tile]
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 2 * NT; ++j) acc[mt][j / NT][j % NT] = (f32x4)(0.f);
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;

    // the loop runs pairs of steps; an odd one is made a pair by a step of zeros in front (a copy of a step behind the loop costs
    // more, in code that every workgroup of a compute unit fetches and in accumulators that move).  The loads go out in the order of
    // the loop, whose waits the compiler counts for both ways into it
    const int s_first = s_begin - ((s_end - s_begin) & 1);
    static_for<MT>([&](auto ic) { load_x(C0{}, ic, max(s_first, s_begin)); });
    static_for<DW>([&](auto jc) {
        constexpr int j = decltype(jc)::value, xj = j + 1 + DX<MT> - DW;
        if constexpr (xj == DX<MT>) {
            if (s_first < s_begin)
#pragma unroll
                for (int i = 0; i < MT; ++i) xreg[0][i] = (u32x4)(0);
            static_for<MT>([&](auto ic) { write_x(C0{}, ic, 0); });
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (xj > 0) static_for<MT>([&](auto ic) { load_x(std::integral_constant<int, xj % DX<MT>>{}, ic, s_first + xj); });
        __builtin_amdgcn_sched_barrier(0);
        static_for<NT>([&](auto nc) { load_w(jc, nc, max(s_first + j, s_begin)); });
        __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    static_for<2 * MT>([&](auto mc) { read_x(mc, 0, C0{}); });
    wf = dequant8<T>(wreg[0][0][0], wreg[0][0][1]);
    __builtin_amdgcn_sched_barrier(0);

    // group (u, nt): every row of sub-step u times channel tile nt, and behind each matrix instruction a piece of what the next
    // groups need
    auto group = [&](auto jsc, auto gc, int s) {
        constexpr int J = decltype(jsc)::value, P = J & 1, G = decltype(gc)::value, U = G / NT, nt = G % NT, NM = 2 * MT;
        constexpr int NS = G == 2 * NT - 1 ? (J + 1) % DW : J, NU = (G + 1) / NT & 1, NN = (G + 1) % NT;   // the tile converted here
        using CX = std::integral_constant<int, (J + 1) % DX<MT>>;                               // the next step's activations
        if constexpr (G == 2 * NT - 2) {                            // the other stage is written, this one has been read
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
        }
        uint32_t w[4];
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 1");                              // the vector unit's last writes reach the matrix unit
        static_for<NM>([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            T::mfma16_acc(acc[m >> 1][m & 1][nt], wf, xf[U][m]);
            __builtin_amdgcn_sched_barrier(0);
            static_for<4>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                if constexpr (j * NM / 4 == m) w[j] = i8x2_to<T>(wreg[NS][NN][2 * NU + (j >> 1)], 16 * (j & 1));
            });
            // the next sub-step's rows: two halves behind every other instruction, or EARLY of them first and then one by one
            constexpr int L = nt - (NT - 2);                  // the last two channel tiles
            constexpr int R = EARLY == 0 ? (m & 1 ? MT * L + m / 2 : NM) : L == 0 ? (m < NM - EARLY ? NM : m - NM + EARLY) : EARLY + m;
            if constexpr (L >= 0 && R < NM)
                read_x(std::integral_constant<int, R>{}, U == 0 ? P : P ^ 1, std::integral_constant<int, U ^ 1>{});
            if constexpr (G == 0 && (m & 1) == 0) write_x(CX{}, std::integral_constant<int, m / 2>{}, P ^ 1);   // read before the last barrier
            if constexpr (G == 0 && (m & 1) == 1) load_x(CX{}, std::integral_constant<int, m / 2>{}, s + 1 + DX<MT>);
            if constexpr (U == 1 && m == 0) load_w(jsc, std::integral_constant<int, nt>{}, s + DW);    // converted in the group before
            __builtin_amdgcn_sched_barrier(0);
        });
        wf = bitcast<vec8>((u32x4){w[0], w[1], w[2], w[3]});
    };
    auto step = [&](auto jsc, int s) {                        // step J of a round over the weights' register sets, LDS stage J & 1
        static_for<2 * NT>([&](auto gc) { group(jsc, gc, s); });
    };
    for (int s = s_first; s < s_end; s += DW) static_for<DW>([&](auto jc) { step(jc, s + decltype(jc)::value); });
    asm volatile("s_nop 15" : "+a"(acc[MT - 1][1][NT - 1]));      // the last matrix instructions' results
    static_for<2 * NT * MT>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        f32x4& a = acc[j / (2 * NT)][j / NT & 1][j % NT];
        asm volatile("" : "+a"(a));
    });
    static_for<MT>([&](auto mtc) { epilogue(mtc, acc[decltype(mtc)::value]); });
}

}  // namespace tg
