// Work distribution of the many-row GEMMs (W8A16 and W8A8): output tiles in whole rounds of the device, the rest cut along K.
#pragma once
#include "common.h"

// Workgroup id -> (row block, channel block, part of K).  Ids below `full` are whole tiles: ids go to the XCDs in turn, so
// XCD j is given the tiles [j * full / 8, (j + 1) * full / 8) and the workgroups that run on it at one time share row and
// channel blocks in its L2.  Then come the `tail` tiles of a short last row block, side by side along the channels, and the tiles left
// over, cut into `split` parts of K each.
struct TileGrid {
    int m_blocks, n_blocks, full, split, steps_per_split;
    int mt, nt;                                               // rows of a block / 32, channels of a block / 64
    int tail;                                                 // tiles of a last row block with fewer 32-row pieces (not in m_blocks)
};
constexpr int TG_PANEL = 4;                                   // row blocks walked together along the channels
__device__ __forceinline__ void tg_locate(const TileGrid& g, int id, int& mb, int& nb, int& part, int& slot) {
    int t;
    part = slot = 0;
    if (id < g.full) {
        t = (id & 7) * (g.full >> 3) + (id >> 3);
    } else if (id < g.full + g.tail) {
        nb = id - g.full;
        mb = g.m_blocks;
        return;
    } else {
        slot = id - g.full - g.tail;
        t = g.full + slot / g.split;
        part = slot % g.split;
    }
    const int panel = t / (TG_PANEL * g.n_blocks), in = t - panel * TG_PANEL * g.n_blocks;
    const int rows = min(TG_PANEL, g.m_blocks - panel * TG_PANEL);
    nb = in / rows;
    mb = panel * TG_PANEL + in - nb * rows;
}
inline int tg_workgroups(const TileGrid& g) { return g.full + g.tail + (g.m_blocks * g.n_blocks - g.full) * g.split; }

// Measured times (us): a k-step of a tile on a compute unit of its own, of a pair of tiles on one compute unit (the clock
// follows the power draw), what a launch and a tile's start and end take, the reduce launch, and one part's share of
// writing and summing the parts.
struct TileCost {
    float alone, pair, fixed, reduce, part;
    float tail;                                               // a k-step of a tile of up to 64 rows
    // other shapes of tile (32*mt rows, 64*nt channels), each on a compute unit of its own: a launch, a k-step
    struct { int mt, nt; float fixed, step; } once[4];
};
// Whole tiles fill whole multiples of the 256 compute units; what is left over would hold a few of them for a whole tile's
// time, so it is cut along K where the shorter tail pays for its parts.
inline TileGrid tg_plan_rounds(int m, int n, int steps, const TileCost& c, float* us) {
    TileGrid g;
    const int m_blocks = (m + 127) / 128, n_blocks = (n + 255) / 256;
    g.mt = g.nt = 4;
    g.m_blocks = m_blocks;
    g.n_blocks = n_blocks;
    g.tail = 0;
    const int tiles = m_blocks * n_blocks, rounds = tiles / 256, rem = tiles % 256;
    float best = 0.f;
    g.split = 1;
    for (int s = 1; s <= 16; s *= 2) {
        if (s > 1 && (rem == 0 || steps / s < 4)) break;
        const int part = (steps + s - 1) / s;
        float t = (rounds / 2) * steps * c.pair;
        if (s == 1) {
            const int tail = (rounds & 1) * 256 + rem;
            t += tail == 0 ? 0.f : steps * (tail <= 256 ? c.alone : c.pair);
        } else {
            const int left = rem * s;
            if (rounds & 1) t += steps * c.alone + (left + 255) / 256 * part * (c.pair - c.alone);
            else t += left <= 256 ? part * c.alone : (left + 511) / 512 * part * c.pair;
            t += c.reduce + left * c.part;
        }
        if (s == 1 || t < best) {
            best = t;
            g.split = s;
        }
    }
    g.steps_per_split = (steps + g.split - 1) / g.split;
    g.split = (steps + g.steps_per_split - 1) / g.steps_per_split;
    g.full = g.split > 1 ? tiles - rem : tiles / 8 * 8;       // a multiple of 8 (see tg_locate)
    *us = best + c.fixed;
    return g;
}

// A last row block of up to 64 rows behind two rounds and more of whole tiles: tiles of just its 32-row pieces, dealt last and one after
// the other over the XCDs.  Beside whole tiles, in places that would be empty, they cost what they compute; where they overflow the
// last round they add their own length.  They replace matrix instructions on rows that are not there, which cost the power of those
// that are.  us on whole tiles | with a tail: W8A16 1048 x 28672 x 4096 230 | 224, 2080 x 28672 x 4096 393 | 381, 1057 x 37888 x 3584 254 |
// 246, 1300 x 24576 x 1536 97 | 89, W8A8 1048 x 37888 x 3584 164 | 159, 1340 x 37888 x 3584 186 | 182, 1300 x 24576 x 1536 67 | 62;
// overflowing 4137 x 4096 x 14336 366 | 425.  Pieces of 65 to 96 rows gain nothing (1632 x 28672 x 4096 311 | 314), nor do tiles of 96 rows
// throughout (1048 x 28672 x 4096 231 | 234, 2080 rows 398 | 420), and the few tiles of a narrow output are shorter cut along K
// (4137 x 6144 x 4096 168 | 171).
inline bool tg_plan_tail(int m, int n, int steps, const TileCost& c, float* us, TileGrid& g) {
    const int rows = m % 128, n_blocks = (n + 255) / 256, tiles = m / 128 * n_blocks, last = tiles % 512;
    if (rows == 0 || rows > 64 || tiles < 512 || n_blocks < 48) return false;
    const float whole = tiles / 512 * c.pair + (last == 0 ? 0.f : last <= 256 ? c.alone : c.pair);
    const float tail = last > 0 && last + n_blocks <= 512 ? c.tail * n_blocks / 256 : c.tail;
    const bool room = last > 256 && last + n_blocks <= 512;   // the round that the whole tiles would have them in takes as long
    const float t = c.fixed + steps * (whole + (room ? 0.f : tail));
    if (t > *us) return false;
    *us = t;
    g = {m / 128, n_blocks, tiles / 8 * 8, 1, steps, 4, 4, n_blocks};
    return true;
}

// Tiles of 128 x 256, or of another shape where those are all resident at once, each on a compute unit of its own, and the shape is
// the shortest: more units then share the work, or fewer rows and channels are padding.  A tile of fewer channels pays more for its
// activations a matrix instruction, a wider one needs all the registers of a compute unit, so neither gains where the device is full for
// several rounds.  us on 128 x 256 or 96 x 256 | with the other shapes: W8A16 1048 x 4096 x 4096 45.5 | 39.2 (96 x 192), 1048 x 4096 x
// 14336 135 | 122, 2500 x 2112 x 7168 76.0 | 70.4 (128 x 192); W8A8 1531 x 3584 x 18944 114 | 104 (128 x 192), 1048 x 4096 x 7168 47.1 |
// 40.6 (96 x 192), 700 x 5120 x 5120 33.6 | 29.8, 2025 x 5120 x 5120 62.0 | 53.8 (128 x 320).  On 10 shapes each of 130 to 3000 rows the
// prices find the fastest one within 1 % on average.
// A single row block does not change, nor one of fewer than 16 k-steps (24 for the shapes that are not 256 channels wide, which were
// measured from there on and have to be 6 % shorter, about what the prices err by).  Nor does a plan all of whose tiles are cut along K: its parts are all resident too, and the model prices
// parts that run at once too high (0.015 us each there, not c.part); against other kernels it counts a tenth less than 96 x 256 tiles would.
// 96 x 256 | 128 x 256 in two parts: W8A16 777 x 4096 x 4096 44.0 | 37.6, 513 x 6144 x 4096 44.5 | 38.5, W8A8 448 x 5120 x 5120 29.8 |
// 27.4.  Where only what is left over by whole rounds is cut, another shape has to be a fifth shorter.  96 x 256 | 96 x 192 on shapes that
// fill less than a round with either: W8A16 2025 x 2112 x 7168 75.3 | 64.0, 1042 x 4416 x 1600 23.2 | 20.7, 1216 x 3648 x 14336 138 |
// 123, W8A8 2025 x 2112 x 7168 45.0 | 40.0, 3322 x 1312 x 1600 14.8 | 13.4 (102 of 102 shapes of 1040 to 4416 channels, by 6 to 24 %).
inline TileGrid tg_plan(int m, int n, int steps, const TileCost& c, float* us) {
    const TileGrid g = tg_plan_rounds(m, n, steps, c, us);
    TileGrid t;
    if (tg_plan_tail(m, n, steps, c, us, t)) return t;
    if (m <= 128 || steps < 16) return g;
    const bool all_cut = g.split > 1 && g.full == 0;
    const auto tiles_of = [&](int mt, int nt) { return (int64_t)((m + 32 * mt - 1) / (32 * mt)) * ((n + 64 * nt - 1) / (64 * nt)); };
    TileGrid best = g;
    float least = (g.split == 1 ? 1.f : all_cut ? 0.85f : 0.8f) * *us;
    for (const auto& s : c.once) {
        const int64_t tiles = s.mt ? tiles_of(s.mt, s.nt) : 257;
        const float t = (all_cut ? 0.9f : 1.f) * (steps * s.step + s.fixed);
        if (tiles > 256 || t >= (s.nt == 4 ? least : 0.94f * least)) continue;
        if (s.nt != 4 && (steps < 24 || all_cut)) continue;
        least = *us = t;
        if (!all_cut) best = {(m + 32 * s.mt - 1) / (32 * s.mt), (n + 64 * s.nt - 1) / (64 * s.nt), (int)tiles / 8 * 8, 1, steps, s.mt, s.nt, 0};
    }
    return best;
}

// Grouped rows (experts): rows a group must average for tiles of 256 channels to replace 64-channel workgroups.  `least` is where
// the two meet when there are tiles enough.  With fewer tiles than compute units and a long K the units without one cost more than
// the better tiles save, until the 64-channel workgroups need a second pass over the weights.  8 experts of 4096 x 14336 (128
// tiles), W8A16 us without | with tiles: 16 rows a group 78 | 112, 33: 91 | 123, 48: 101 | 125, 65: 183 | 138; W8A8 20 rows 79 | 98,
// 48: 101 | 110.  16 experts of 2048 x 1024 (128 tiles too): 16 rows 13.2 | 11.9.
inline int tg_group_min_rows(int n_experts, int n_blocks, int k, int least) {
    return k > 2048 && (int64_t)n_experts * n_blocks < 256 ? 64 : least;
}

// Output of a kernel that streams the weights of many experts: written past the caches.  Lines that wait in L2 leave it one by one
// between the loads of the stream, and each costs the stream more than its own time; behind a short stream they stay in the caches for
// the next kernel.  256 experts of 65 rows on average (11.3 GB), W8A8, us without stores | past the caches | cached: 4096 x 7168 1098 |
// 1252 | 1320 (136 MB written), 7168 x 2048 565 | 762 | 800 (238 MB).  Both projections with what lies between them, past the
// caches | cached: W8A8 24 rows an expert 1768 | 1819, 48: 1910 | 2056, 65: 2036 | 2088, W8A16 24: 1751 | 1803, 48: 1920 | 2070, 65: 2116 |
// 2152; 8 experts of 28672 x 4096 (0.94 GB), 65 rows 309 | 306, W8A16 367 | 364; 64 of 2816 x 2048 (0.37 GB), 33 rows 114 | 110, W8A16
// 114 | 107.  The cost lies in the switches of the memory between reads and writes more than in the bytes: with a quarter of the rows
// written 1213 and 725.
inline bool tg_group_stream(int n_experts, int64_t expert_bytes) { return n_experts * expert_bytes > (1LL << 30); }

// Grouped rows (experts): the row blocks of all experts, in order, times the channel blocks.  Their number is known on the
// device only (offsets [n_experts + 1]), so the launch covers what the total allows and each workgroup finds its own by a
// scan of the offsets.  Ids go to the XCDs in turn; XCD j is given the j-th eighth of the row blocks, all channel blocks of
// one side by side, so that an expert's activations are read into one L2 and the weights of an expert with several row blocks
// are met there by all of them.  False: nothing to do.
constexpr int TG_GROUP_ROWS = 128;
inline unsigned tg_group_workgroups(int total_rows, int n_experts, int n_blocks) {
    const int64_t m_blocks = (int64_t)total_rows / TG_GROUP_ROWS + min(n_experts, total_rows);
    return (unsigned)((m_blocks + 7) / 8 * 8 * n_blocks);
}
__device__ __forceinline__ bool tg_group_locate(const int32_t* __restrict__ offsets, int n_experts, int total_rows,
                                                int n_blocks, int& expert, int& m0, int& row0, int& rows, int& nb) {
    const int lane = threadIdx.x & 63;
    auto span = [&](int e, int& r0) {
        if (e >= n_experts) return 0;
        r0 = max(0, min(offsets[e], total_rows));
        return max(r0, min(offsets[e + 1], total_rows)) - r0;
    };
    int total = 0, r0 = 0;
    for (int e = lane; e < n_experts; e += 64) total += (span(e, r0) + TG_GROUP_ROWS - 1) / TG_GROUP_ROWS;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) total += __shfl_xor(total, o, 64);
    total = __builtin_amdgcn_readfirstlane(total);
    const int id = blockIdx.x, per_xcd = (total + 7) / 8, at = (id >> 3) / n_blocks;
    nb = (id >> 3) - at * n_blocks;
    int want = (id & 7) * per_xcd + at;
    if (at >= per_xcd || want >= total) return false;
    for (int base = 0; base < n_experts; base += 64) {
        const int n = span(base + lane, r0), blocks = (n + TG_GROUP_ROWS - 1) / TG_GROUP_ROWS;
        int upto = blocks;                                    // blocks of the experts up to this lane's
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(upto, o, 64);
            if (lane >= o) upto += up;
        }
        const uint64_t past = __ballot(upto > want);
        if (past) {
            const int l = __ffsll((unsigned long long)past) - 1;
            expert = __builtin_amdgcn_readfirstlane(base + l);
            row0 = __builtin_amdgcn_readfirstlane(__shfl(r0, l, 64));
            rows = __builtin_amdgcn_readfirstlane(__shfl(n, l, 64));
            m0 = __builtin_amdgcn_readfirstlane(TG_GROUP_ROWS * (want - __shfl(upto - blocks, l, 64)));
            return true;
        }
        want -= __builtin_amdgcn_readfirstlane(__shfl(upto, 63, 64));
    }
    return false;
}

// Where the rows of a group come from: side by side at the group's place (sources null), or through an index, row i of all groups
// being row sources[i] of n_sources rows (entries out of range are clamped).
// A token's copies for its k experts are neither written nor read back that way, and the tokens stay in the caches: a layer of 256
// experts on 2077 tokens, 8 experts each, W8A8 2464 us with the copies made (35 of them the copying), 2421 through the index.  The kernels for
// fewer rows take copies: 1024 rows are copied in 5 us of 1780.
struct TileSources {
    const int32_t* sources;
    int n_sources;
    __device__ __forceinline__ int of(int i) const { return max(0, min(sources[i], n_sources - 1)); }
};

// 16 bytes at an address that is the same in every lane plus the lane's 32-bit offset: the address stays in scalar registers
template <bool NT = false>
__device__ __forceinline__ u32x4 load16_at(const uint8_t* base, uint32_t offset) {
    typedef const __attribute__((address_space(1))) uint8_t* gptr;
    gptr p = (gptr)base;
    asm("" : "+s"(p), "+v"(offset));
    const auto at = (const __attribute__((address_space(1))) u32x4*)(p + offset);
    if constexpr (NT) return __builtin_nontemporal_load(at);
    else return *at;
}

// the lanes of a wave exchange values through LDS: its own instructions stay in order
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// 32 staged rows of up to 16 * NT channels (16 bytes more a row: 16-byte slots spread over the banks) to memory as whole 16-byte pieces
// of rows, by `threads` threads of which this is number t; the residual, read the same way, is added to the rounded values.
// cols = row length of y, c0 = first channel, per = 16-byte pieces of a staged row.
// STREAM: stores past the caches, see tg_group_stream.
template <int NT>
constexpr int TG_STAGE_ROW = 32 * NT + 16;
template <typename T, int NT, bool STREAM = false>
__device__ __forceinline__ void tg_flush(uint16_t* y, const uint16_t* residual, const uint8_t* stage, int m0, int M, int c0,
                                         int cols, int per, bool aligned, int t, int threads) {
    const int row = t / per, c = c0 + 8 * (t - row * per), step = threads / per;
    if (row >= step) return;                                  // threads past the last whole row
    for (int j = row; j < 32; j += step) {
        const int m = m0 + j;
        if (m >= M || c >= cols) continue;
        u32x4 v = *(const u32x4*)(stage + j * TG_STAGE_ROW<NT> + 2 * (c - c0));
        const int64_t at = (int64_t)m * cols + c;
        if (residual) {
            float f[8], g[8];
            u32x4 rr;
            if (aligned) rr = *(const u32x4*)(residual + at);
            else
                for (int i = 0; i < 4; ++i) rr[i] = residual[at + 2 * i] | (uint32_t)residual[at + 2 * i + 1] << 16;
            unpack8<T>(v, f);
            unpack8<T>(rr, g);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = pack2<T>(__fadd_rn(f[2 * i], g[2 * i]), __fadd_rn(f[2 * i + 1], g[2 * i + 1]));
        }
        if (aligned) {
            if constexpr (STREAM) __builtin_nontemporal_store(v, (u32x4*)(y + at));
            else *(u32x4*)(y + at) = v;
        } else
            for (int i = 0; i < 8; ++i) y[at + i] = (uint16_t)(v[i >> 1] >> (16 * (i & 1)));
    }
}
