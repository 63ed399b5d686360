// Mixture-of-experts routing kernels: group-limited sigmoid top-k router, counting-sort permute,
// weighted unpermute.  Index work is exact; the heavy parts (row gather / weighted row sum) are plain
// HBM-bound copies with 16-byte lane accesses.
#include "common.h"

namespace {

constexpr int RT_MAX_E = 1024;
constexpr int RT_MAX_K = 32;

// One wavefront per token.
template <typename T>
__global__ __launch_bounds__(64) void moe_route_kernel(uint16_t* __restrict__ weights_out,
                                                      int32_t* __restrict__ index_out,
                                                      const float* __restrict__ logits,
                                                      const float* __restrict__ bias, int E, int k, int n_group,
                                                      int topk_group, float scale, int renorm,
                                                      int biased_weights) {
    __shared__ float s_plain[RT_MAX_E];     // sigmoid(logit)
    __shared__ float s_biased[RT_MAX_E];    // sigmoid(logit) + bias, later masked
    __shared__ float s_gscore[64];
    __shared__ float s_thr;
    const int t = blockIdx.x;
    const int lane = threadIdx.x;
    const float* lg = logits + (int64_t)t * E;

    for (int e = lane; e < E; e += 64) {
        const float s = 1.0f / (1.0f + __expf(-lg[e]));
        s_plain[e] = s;
        s_biased[e] = s + (bias ? bias[e] : 0.f);
    }
    __syncthreads();

    if (n_group > 1 && topk_group < n_group) {
        const int gs = E / n_group;
        float score = -INFINITY;
        if ((n_group & (n_group - 1)) == 0) {
            // 64 / n_group lanes share a group: each scans a strided part, the pairs of largest values merge by
            // shuffles (values only, so the order of the merge does not matter)
            const int lpg = 64 / n_group;
            const int grp = lane / lpg, sub = lane - grp * lpg;
            float a = -INFINITY, b = -INFINITY;               // two largest of the group
            for (int i = sub; i < gs; i += lpg) {
                const float v = s_biased[grp * gs + i];
                if (v > a) { b = a; a = v; } else if (v > b) { b = v; }
            }
            for (int o = 1; o < lpg; o <<= 1) {
                const float oa = __shfl_xor(a, o, 64), ob = __shfl_xor(b, o, 64);
                const float hi = fmaxf(a, oa);
                b = a >= oa ? fmaxf(b, oa) : fmaxf(ob, a);
                a = hi;
            }
            score = gs >= 2 ? a + b : a;
            if (sub == 0) s_gscore[grp] = score;
            __syncthreads();
            score = lane < n_group ? s_gscore[lane] : -INFINITY;
        } else {
            if (lane < n_group) {
                float a = -INFINITY, b = -INFINITY;
                for (int i = 0; i < gs; ++i) {
                    const float v = s_biased[lane * gs + i];
                    if (v > a) { b = a; a = v; } else if (v > b) { b = v; }
                }
                score = gs >= 2 ? a + b : a;
                s_gscore[lane] = score;
            }
            __syncthreads();
        }
        if (lane < n_group) {
            int rank = 0;                                     // groups strictly ahead (ties: lower index first)
            for (int j = 0; j < n_group; ++j) {
                const float o = s_gscore[j];
                rank += (o > score) || (o == score && j < lane);
            }
            if (rank == topk_group - 1) s_thr = score;        // the topk_group-th largest group score
        }
        __syncthreads();
        const float thr = s_thr;
        // keep groups with score >= threshold; experts of dropped groups score 0.0 (masked_fill)
        for (int e = lane; e < E; e += 64)
            if (!(s_gscore[e / gs] >= thr)) s_biased[e] = 0.0f;
        __syncthreads();
    }

    // top-k by repeated wave-wide argmax (larger value first, ties to the lower index); the candidates live in
    // registers, expert e = lane + 64 i in slot i
    __shared__ float s_wsel[RT_MAX_K];
    __shared__ int s_isel[RT_MAX_K];
    constexpr int SLOTS = RT_MAX_E / 64;
    float cand[SLOTS];
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) cand[i] = lane + 64 * i < E ? s_biased[lane + 64 * i] : -INFINITY;
    float wsum = 0.f;
    for (int j = 0; j < k; ++j) {
        float best = -INFINITY;
        int bi = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < SLOTS; ++i) {
            const bool live = lane + 64 * i < E;
            if (live && cand[i] > best) { best = cand[i]; bi = lane + 64 * i; }   // ascending e: first maximum wins
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(best, o, 64);
            const int oi = __shfl_xor(bi, o, 64);
            if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
        }
        if (bi >= E) bi = 0;                                  // all -inf/NaN rows: keep indices in range
        const float wv = biased_weights ? best : s_plain[bi];
        wsum += wv;
#pragma unroll
        for (int i = 0; i < SLOTS; ++i)
            if (bi == lane + 64 * i) cand[i] = -INFINITY;
        if (lane == 0) {
            s_wsel[j] = wv;
            s_isel[j] = bi;
        }
    }
    __syncthreads();
    if (lane == 0) {
        for (int j = 0; j < k; ++j) {
            float wv = s_wsel[j];
            if (renorm && k > 1) wv = wv / wsum;
            wv *= scale;
            weights_out[(int64_t)t * k + j] = T::from_float(wv);
            index_out[(int64_t)t * k + j] = s_isel[j];
        }
    }
}

// Stable counting sort of the pairs p = t*k + j by expert; a workgroup of 1024 threads places SORT_CHUNK pairs (one chunk only: of
// as many waves as its pairs and the experts take).  Every
// workgroup counts all the pairs itself (the indices are at most 256 KB, read from the L2), those in front of its chunk apart
// from the rest, so that no second launch, workspace or order among workgroups is needed: a pair's row is its expert's first
// row + the expert's pairs in earlier chunks + those of earlier waves of the chunk + those of lower lanes of its wave.
// What bounds it: the latency of a few dependent passes.  16616 pairs on 256 experts: 129 us in one workgroup that
// walked the pairs 64 at a time, 8 us here.  (The scan with a run of experts per lane of one wave: 1.6 us more at 1024 experts.)
constexpr int SORT_CHUNK = 1024;
struct SortRows {                                             // where the rows are not copied: token (of k pairs each) and scale of each
    int32_t* sources;
    float* scale;
    const float* x_scale;
    int k;
};
__global__ __launch_bounds__(SORT_CHUNK) void moe_sort_kernel(int32_t* __restrict__ row_map, int64_t* __restrict__ counts,
                                                              int32_t* __restrict__ offsets,
                                                              const int32_t* __restrict__ expert_index, int pairs,
                                                              int E, SortRows rows) {
    __shared__ int s_before[RT_MAX_E], s_rest[RT_MAX_E], s_cur[RT_MAX_E];
    __shared__ __attribute__((aligned(16))) uint8_t s_wave[SORT_CHUNK / 64][RT_MAX_E];   // pairs of the wave: at most 64
    __shared__ int s_total[SORT_CHUNK / 64];
    static_assert(RT_MAX_E <= SORT_CHUNK, "a thread per expert");
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int chunk0 = blockIdx.x * SORT_CHUNK;
    if (tid < E) s_before[tid] = s_rest[tid] = 0;
    for (int i = tid; i < (int)blockDim.x / 64 * RT_MAX_E / 16; i += blockDim.x) ((u32x4*)s_wave)[i] = (u32x4){0u, 0u, 0u, 0u};
    __syncthreads();
    const int p = chunk0 + tid;
    int e = p < pairs ? expert_index[p] : -1;
    if (e >= E) e = -1;
    for (int base = 0; base < pairs; base += 4 * SORT_CHUNK) {
        int v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int q = base + i * SORT_CHUNK + tid;
            v[i] = q < pairs ? expert_index[q] : -1;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (v[i] >= 0 && v[i] < E) atomicAdd(base + i * SORT_CHUNK < chunk0 ? &s_before[v[i]] : &s_rest[v[i]], 1);
    }
    // lanes holding the same expert (10 index bits + validity)
    uint64_t same = __ballot(e >= 0);
#pragma unroll
    for (int bit = 0; bit < 10; ++bit) {
        const uint64_t bm = __ballot((e >> bit) & 1);
        same &= ((e >> bit) & 1) ? bm : ~bm;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    if (e >= 0 && rank == 0) s_wave[wv][e] = (uint8_t)__popcll(same);
    __syncthreads();
    {                                                         // exclusive scan: an expert per thread
        const int before = tid < E ? s_before[tid] : 0, c = tid < E ? before + s_rest[tid] : 0;
        int run = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(run, o, 64);
            if (lane >= o) run += up;
        }
        if (lane == 63) s_total[wv] = run;
        __syncthreads();
        run -= c;
#pragma unroll
        for (int w = 0; w < SORT_CHUNK / 64; ++w) run += w < wv ? s_total[w] : 0;
        if (tid < E) {
            s_cur[tid] = run + before;
            if (blockIdx.x == 0) {
                offsets[tid] = run;
                counts[tid] = c;
                if (tid == E - 1) offsets[E] = run + c;
            }
        }
    }
    __syncthreads();
    if (p >= pairs) return;
    int dst = -1;
    if (e >= 0) {
        dst = s_cur[e] + rank;
        for (int w = 0; w < wv; ++w) dst += s_wave[w][e];
    }
    row_map[p] = dst;
    if (rows.sources && dst >= 0) {
        const int token = p / rows.k;
        rows.sources[dst] = token;
        if (rows.x_scale) rows.scale[dst] = rows.x_scale[token];
    }
}

// permuted_x[row_map[p]] = x[p / k]; one workgroup per pair.  Rows of int8 values come as `hidden` pairs of them, with their
// scales in x_scale (else null).
__global__ void moe_gather_kernel(uint16_t* __restrict__ permuted, float* __restrict__ permuted_scale,
                                  const uint16_t* __restrict__ x, const float* __restrict__ x_scale,
                                  const int32_t* __restrict__ row_map, int k, int hidden, int pairs) {
    const int p = blockIdx.x;
    const int dst = row_map[p];
    if (dst < 0 || dst >= pairs) return;
    const uint16_t* src = x + (int64_t)(p / k) * hidden;
    uint16_t* d = permuted + (int64_t)dst * hidden;
    if (x_scale && threadIdx.x == 0) permuted_scale[dst] = x_scale[p / k];
    for (int i = threadIdx.x * 8; i < hidden; i += blockDim.x * 8) *(u32x4*)(d + i) = *(const u32x4*)(src + i);
}

// out[t] = sum_j probs[t,j] * y[row_map[t*k+j]] (+ shared[t]); grid = (tokens, column chunks of 8 * blockDim.x), one
// 16-byte item per thread.  The k row indices and weights are read first, then the k rows are loaded in batches of
// UNP_BATCH independent loads and summed in choice order (the order fixes the fp32 sum).
constexpr int UNP_BATCH = 8;
template <typename T>
__global__ void moe_unpermute_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ y,
                                     const int32_t* __restrict__ row_map, const uint16_t* __restrict__ probs,
                                     const uint16_t* __restrict__ shared, int k, int hidden, int pairs) {
    const int t = blockIdx.x;
    const int i = (blockIdx.y * blockDim.x + threadIdx.x) * 8;
    if (i >= hidden) return;
    u32x4 sh = {0u, 0u, 0u, 0u};
    if (shared) sh = *(const u32x4*)(shared + (int64_t)t * hidden + i);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < k; j0 += UNP_BATCH) {
        int row[UNP_BATCH];
        float pw[UNP_BATCH];
        u32x4 v[UNP_BATCH];
#pragma unroll
        for (int j = 0; j < UNP_BATCH; ++j) {
            const int jj = j0 + j;
            row[j] = jj < k ? row_map[(int64_t)t * k + jj] : -1;
            pw[j] = jj < k ? T::to_float(probs[(int64_t)t * k + jj]) : 0.f;
        }
#pragma unroll
        for (int j = 0; j < UNP_BATCH; ++j) {
            const bool ok = row[j] >= 0 && row[j] < pairs;
            v[j] = (u32x4){0u, 0u, 0u, 0u};
            if (ok) v[j] = *(const u32x4*)(y + (int64_t)row[j] * hidden + i);
            else row[j] = -1;
        }
#pragma unroll
        for (int j = 0; j < UNP_BATCH; ++j) {
            if (row[j] < 0) continue;                         // a skipped choice adds nothing (not even +0)
            float f[8];
            unpack8<T>(v[j], f);
#pragma unroll
            for (int q = 0; q < 8; ++q) acc[q] += pw[j] * f[q];
        }
    }
    if (shared) {
        // the routed sum is materialised in the activation dtype before the shared-expert add
        float f[8];
        unpack8<T>(sh, f);
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[q] = T::to_float(T::from_float(acc[q])) + f[q];
    }
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = pack2<T>(acc[2 * q], acc[2 * q + 1]);
    *(u32x4*)(out + (int64_t)t * hidden + i) = o;
}


// ---- router gate projection -------------------------------------------------------------------------
// logits[t, e] = sum_h x[t, h] * w[e, h], products and sums in fp32 on the fp32 matrix instruction (16 x 16 x 4).
// The weight (E x H, a few MB) is read once: a workgroup owns 16 experts and one slice of H for up to 64 tokens;
// its 4 waves take the slice's 64-column chunks in turn and meet in LDS.  Lane (r = lane & 15, g = lane >> 4) loads
// columns 16 j + 4 g .. + 3 of a chunk for expert r and for token r: the instruction's k index is any bijection as
// long as both operands use the same one.  With more than one slice the workgroups write partial sums
// [slice][token][expert] and router_gate_reduce_kernel adds the slices in order (no atomics: results do not depend
// on scheduling).
struct RG_F32 {};
template <typename WT>
__device__ __forceinline__ f32x4 rg_load4(const void* w, int64_t idx) {
    if constexpr (std::is_same<WT, RG_F32>::value) {
        return *(const f32x4*)((const float*)w + idx);
    } else {
        const u32x2 v = *(const u32x2*)((const uint16_t*)w + idx);
        return (f32x4){WT::to_float((uint16_t)(v[0] & 0xffffu)), WT::to_float((uint16_t)(v[0] >> 16)),
                       WT::to_float((uint16_t)(v[1] & 0xffffu)), WT::to_float((uint16_t)(v[1] >> 16))};
    }
}

template <typename WT>
__device__ __forceinline__ float rg_round(float v) {
    // a 16-bit router computes in its own type: the projection's output is rounded to it before the cast to fp32
    if constexpr (std::is_same<WT, RG_F32>::value) return v;
    else return WT::to_float(WT::from_float(v));
}

constexpr int RG_TT = 4;                                      // token tiles of 16 per workgroup

template <typename T, typename WT>
__global__ __launch_bounds__(256) void router_gate_kernel(float* __restrict__ out, float* __restrict__ partial,
                                                          const uint16_t* __restrict__ x, const void* __restrict__ w,
                                                          int tokens, int E, int H, int k_per_split) {
    __shared__ f32x4 red[4][RG_TT][64];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    const int e0 = blockIdx.x * 16, t0 = blockIdx.z * (16 * RG_TT);
    const int k_begin = blockIdx.y * k_per_split, k_end = min(H, k_begin + k_per_split);
    const int64_t wrow = (int64_t)min(e0 + r, E - 1) * H;     // rows past the matrix re-read the last one, never stored
    int64_t xrow[RG_TT];
#pragma unroll
    for (int tt = 0; tt < RG_TT; ++tt) xrow[tt] = (int64_t)min(t0 + 16 * tt + r, tokens - 1) * H;
    f32x4 acc[RG_TT];
#pragma unroll
    for (int tt = 0; tt < RG_TT; ++tt) acc[tt] = (f32x4){0.f, 0.f, 0.f, 0.f};

    for (int k0 = k_begin + 64 * wv; k0 < k_end; k0 += 256) {
        f32x4 wa[4], xb[RG_TT][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = k0 + 16 * j + 4 * g;
            const bool in = k < k_end;                        // H and the slices are multiples of 4
            const int kc = in ? k : k_begin;
            wa[j] = rg_load4<WT>(w, wrow + kc);
#pragma unroll
            for (int tt = 0; tt < RG_TT; ++tt) xb[tt][j] = rg_load4<T>(x, xrow[tt] + kc);
            if (!in) {
                wa[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int tt = 0; tt < RG_TT; ++tt) xb[tt][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int tt = 0; tt < RG_TT; ++tt)
                    acc[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(wa[j][i], xb[tt][j][i], acc[tt], 0, 0, 0);
    }
#pragma unroll
    for (int tt = 0; tt < RG_TT; ++tt) red[wv][tt][lane] = acc[tt];
    __syncthreads();
    // thread (tt = wave, lane): the sum over the 4 waves, in order.  Lane (r, g) of the instruction's result holds
    // token r, experts 4 g .. 4 g + 3 of the tile.
    const int tt = wv;
    f32x4 v = red[0][tt][lane];
#pragma unroll
    for (int q = 1; q < 4; ++q) {
        const f32x4 u = red[q][tt][lane];
        v = (f32x4){v[0] + u[0], v[1] + u[1], v[2] + u[2], v[3] + u[3]};
    }
    const int t = t0 + 16 * tt + r, e = e0 + 4 * g;
    if (t >= tokens) return;
    float* dst = partial ? partial + ((int64_t)blockIdx.y * tokens + t) * E + e : out + (int64_t)t * E + e;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (e + i < E) dst[i] = partial ? v[i] : rg_round<WT>(v[i]);
}

// The same product for many tokens: a workgroup owns 64 tokens x 64 experts and a slice of H, a wave 32 x 32 of them on the
// 32 x 32 x 2 instruction.  64 columns of both operands at a time are staged in LDS as fp32 (whole rows of 256 bytes are
// fetched; the next 64 columns are in registers meanwhile), and lane half h takes columns 32 h .. 32 h + 31 of its row.
// What bounds it: the fp32 matrix instruction, half the rate of which is reached: at 2077 x 256 x 7168 (85 TFLOP/s of 157
// nominal) the matrix pipes are busy 70 % of the time that a compute unit has work and LDS 18 % (no bank conflicts), and a
// compute unit has work 77 % of the time (924 workgroups on 1024 places).  236 us there with operands fetched into registers 16
// rows at a time, where every 16 experts fetched the tokens anew, 89 us here.  Rounding: CHAINS fp32 chains a slice, four as in that
// kernel, or two where there are slices enough to have as many chains in all (plan_router_gate): RMS error against float64 7.6e-7 in
// the kernel above and 4.1e-7 here at 2077 x 256 x 7168 (1 and 7 slices), 7.6e-7 in both at 512 experts and 4200 tokens (one slice;
// two chains would give 10.7e-7).  Offsets of 32 bits from the tile's rows keep it at four workgroups a compute unit (with three,
// 2077 x 256 x 7168 takes 102 us).
constexpr int RGT = 64;                                       // tokens, experts and columns of a step
constexpr int RGT_ROW = RGT + 4;                              // floats of a staged row: 16-byte pieces of 8 rows meet all banks
template <typename T, typename WT, int CHAINS>
__global__ __launch_bounds__(256, 4) void router_gate_tile_kernel(float* __restrict__ out, float* __restrict__ partial,
                                                               const uint16_t* __restrict__ x, const void* __restrict__ w,
                                                               int tokens, int E, int H, int k_per_split) {
    __shared__ float sw[RGT * RGT_ROW], sx[RGT * RGT_ROW];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 31, h = lane >> 5;
    const int e0 = blockIdx.x * RGT, t0 = blockIdx.z * RGT;
    const int k_begin = blockIdx.y * k_per_split, k_end = min(H, k_begin + k_per_split);
    // load i of a thread: columns 4 c .. 4 c + 3 of row lr + 16 i; rows past the matrix re-read the last one, never stored.
    // Byte offsets from the tile's first row: 64 rows of an operand are far below 4 GB
    constexpr uint32_t WB = std::is_same<WT, RG_F32>::value ? 4 : 2;
    const uint8_t *wt = (const uint8_t*)w + (int64_t)e0 * H * WB, *xt = (const uint8_t*)(x + (int64_t)t0 * H);
    const int lr = threadIdx.x >> 4, lc = 4 * (threadIdx.x & 15);
    uint32_t wrow[4], xrow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        wrow[i] = (uint32_t)min(lr + 16 * i, E - 1 - e0) * (uint32_t)H * WB;
        xrow[i] = (uint32_t)min(lr + 16 * i, tokens - 1 - t0) * (uint32_t)H * 2u;
    }
    f32x4 wr[4], xr[4];
    auto load = [&](int k0) {
        const int k = k0 + lc;
        const bool in = k < k_end;                            // H and the slices are multiples of 4
        const uint32_t kc = in ? k : k_begin;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            wr[i] = rg_load4<WT>(wt + (wrow[i] + kc * WB), 0);
            xr[i] = rg_load4<T>(xt + (xrow[i] + kc * 2u), 0);
            if (!in) wr[i] = xr[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
    };
    f32x16 acc[CHAINS];
#pragma unroll
    for (int i = 0; i < CHAINS; ++i) acc[i] = (f32x16)(0.f);
    const float* pw = sw + (32 * (wv & 1) + r) * RGT_ROW + 32 * h;
    const float* px = sx + (32 * (wv >> 1) + r) * RGT_ROW + 32 * h;
    load(k_begin);
    for (int k0 = k_begin; k0 < k_end; k0 += RGT) {
        __syncthreads();                                      // the step before has been read
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *(f32x4*)(sw + (lr + 16 * i) * RGT_ROW + lc) = wr[i];
            *(f32x4*)(sx + (lr + 16 * i) * RGT_ROW + lc) = xr[i];
        }
        __syncthreads();
        if (k0 + RGT < k_end) load(k0 + RGT);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const f32x4 a = *(const f32x4*)(pw + 4 * j), b = *(const f32x4*)(px + 4 * j);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i % CHAINS] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[i], acc[i % CHAINS], 0, 0, 0);
        }
    }
    acc[0] += acc[1];
    if constexpr (CHAINS == 4) acc[0] = acc[0] + (acc[2] + acc[3]);
    // lane (r, h) holds token r, experts 8 q + 4 h .. + 3 in elements 4 q .. 4 q + 3
    const int t = t0 + 32 * (wv >> 1) + r;
    if (t >= tokens) return;
    float* dst = partial ? partial + ((int64_t)blockIdx.y * tokens + t) * E : out + (int64_t)t * E;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = e0 + 32 * (wv & 1) + 8 * q + 4 * h + i;
            if (e < E) dst[e] = partial ? acc[0][4 * q + i] : rg_round<WT>(acc[0][4 * q + i]);
        }
}

template <typename WT>
__global__ void router_gate_reduce_kernel(float* __restrict__ out, const float* __restrict__ partial, int64_t n,
                                          int splits) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v = partial[i];
    for (int s = 1; s < splits; ++s) v += partial[s * n + i];
    out[i] = rg_round<WT>(v);
}

struct GatePlan {
    int tile, chains, splits, k_per_split;                    // chains: of a tile's slice
};
// slices of H for workgroups of te experts x 64 tokens, `target` of them wanted
GatePlan slice_router_gate(int tokens, int E, int H, int te, int target) {
    GatePlan p = {te == RGT, 4, 1, H};
    const int wgs = ((E + te - 1) / te) * ((tokens + 16 * RG_TT - 1) / (16 * RG_TT));
    int s = target / wgs;
    const int max_s = H / 256 < 1 ? 1 : H / 256;              // at least one chunk per wave, or four steps of a tile
    s = s < 1 ? 1 : (s > max_s ? max_s : s);
    p.k_per_split = ((H + s - 1) / s + 63) / 64 * 64;
    p.splits = (H + p.k_per_split - 1) / p.k_per_split;
    return p;
}
GatePlan plan_router_gate(int tokens, int E, int H) {
    // Tiles take over where there are enough of them, each with enough of H, to pay for their start and end; experts that fill
    // less than three quarters of a tile of 64 need twice as many.  Measured on either side of the line, experts x H: tokens,
    // us without | with tiles: 64 x 2048: 1024 12.5 | 14.4, 2077 21.5 | 18.9; 128 x 2048: 512 12.5 | 14.5,
    // 1024 18.2 | 15.6; 160 x 5120: 384 22.1 | 22.8, 512 27.6 | 24.8; 256 x 7168: 256 27 | 28, 257 32.4 | 30.8, 2077 237 | 89;
    // 256 x 256: 1024 5.7 | 10.3, 2077 11.2 | 10.5; 32 x 7168: 2077 29.2 | 33.3, 4200 57.8 | 48.8; 16 x 4096: 8192 28.8 | 45.0.
    // Up to 256 tokens and with up to 16 experts the others always win: they read the weight once, at most 16 rows in vain.
    // (H: 64 rows stay within 32-bit offsets.)
    const GatePlan few = slice_router_gate(tokens, E, H, 16, 512);
    if (tokens <= 256 || E <= 16 || H >= (1 << 24) || (float)E * tokens <= (E < 48 ? 2.f : 1.f) * (48e3f + 120e6f / H)) return few;
    GatePlan p = slice_router_gate(tokens, E, H, RGT, 1024);
    p.chains = 2 * p.splits >= 4 * few.splits ? 2 : 4;        // never fewer chains in all than the kernel for fewer tokens makes
    return p;
}

int sort_pairs(int32_t* row_map, int64_t* counts, int32_t* offsets, const int32_t* expert_index, int pairs, int n_experts,
               const SortRows& rows, hipStream_t stream) {
    const int chunks = pairs > SORT_CHUNK ? (pairs + SORT_CHUNK - 1) / SORT_CHUNK : 1;
    // one chunk: fewer waves meet at the barriers sooner (1 token on 8 experts: 5.4 us with the gather in 16 waves, 4.7 in one)
    const int most = pairs > n_experts ? pairs : n_experts, threads = most < SORT_CHUNK ? (most + 63) / 64 * 64 : SORT_CHUNK;
    hipLaunchKernelGGL(moe_sort_kernel, dim3(chunks), dim3(threads), 0, stream, row_map, counts, offsets, expert_index,
                       pairs, n_experts, rows);
    return MF_LAUNCH_CHECK();
}

int permute(uint16_t* permuted, float* permuted_scale, int32_t* row_map, int64_t* counts, int32_t* offsets, const uint16_t* x,
            const float* x_scale, const int32_t* expert_index, int tokens, int k, int n_experts, int hidden,
            hipStream_t stream) {
    const int pairs = tokens * k;
    int rc = sort_pairs(row_map, counts, offsets, expert_index, pairs, n_experts, {nullptr, nullptr, nullptr, k}, stream);
    if (rc || pairs == 0) return rc;
    hipLaunchKernelGGL(moe_gather_kernel, dim3(pairs), dim3(256), 0, stream, permuted, permuted_scale, x, x_scale, row_map, k,
                       hidden, pairs);
    return MF_LAUNCH_CHECK();
}

}  // namespace

extern "C" int mf_moe_route(void* weights_out, int32_t* index_out, const float* logits, const float* bias,
                            int tokens, int n_experts, int k, int n_group, int topk_group, float scale, int renorm,
                            int biased_weights, int dtype, void* stream) {
    MF_REQUIRE(dtype == MF_BF16 || dtype == MF_FP16, "moe_route: dtype must be bf16 or fp16");
    if (tokens <= 0) return 0;
    MF_REQUIRE(weights_out && index_out && logits, "moe_route: null argument");
    MF_REQUIRE(n_experts > 0 && n_experts <= RT_MAX_E, "moe_route: n_experts (%d) must be in 1..%d", n_experts, RT_MAX_E);
    MF_REQUIRE(k > 0 && k <= RT_MAX_K && k <= n_experts, "moe_route: k (%d) must be in 1..min(%d, n_experts)", k, RT_MAX_K);
    if (n_group > 1 && topk_group < n_group) {
        MF_REQUIRE(n_group <= 64 && n_experts % n_group == 0 && topk_group >= 1,
                   "moe_route: n_group (%d) must divide n_experts, be <= 64, with 1 <= topk_group (%d)", n_group,
                   topk_group);
    }
    if (tokens <= 0) return 0;
    if (dtype == MF_BF16)
        hipLaunchKernelGGL(moe_route_kernel<BF16>, dim3(tokens), dim3(64), 0, (hipStream_t)stream, (uint16_t*)weights_out,
                           index_out, logits, bias, n_experts, k, n_group, topk_group, scale, renorm, biased_weights);
    else
        hipLaunchKernelGGL(moe_route_kernel<FP16>, dim3(tokens), dim3(64), 0, (hipStream_t)stream, (uint16_t*)weights_out,
                           index_out, logits, bias, n_experts, k, n_group, topk_group, scale, renorm, biased_weights);
    return MF_LAUNCH_CHECK();
}

extern "C" size_t mf_router_gate_workspace_bytes(int tokens, int n_experts, int hidden) {
    if (tokens <= 0 || n_experts <= 0 || hidden <= 0) return 0;
    const GatePlan p = plan_router_gate(tokens, n_experts, hidden);
    return p.splits > 1 ? (size_t)p.splits * tokens * n_experts * sizeof(float) : 0;
}

extern "C" int mf_router_gate_gemm(float* logits, const void* x, const void* w, int tokens, int n_experts, int hidden,
                                   int dtype, int w_dtype, void* workspace, size_t workspace_bytes, void* stream) {
    MF_REQUIRE(dtype == MF_BF16 || dtype == MF_FP16, "router_gate_gemm: dtype must be bf16 or fp16");
    MF_REQUIRE(w_dtype == MF_FP32 || w_dtype == dtype, "router_gate_gemm: the weight is fp32 or of the activation type");
    if (tokens <= 0) return 0;
    MF_REQUIRE(logits && x && w, "router_gate_gemm: null argument");
    MF_REQUIRE(n_experts > 0 && hidden > 0 && hidden % 4 == 0, "router_gate_gemm: hidden (%d) must be a multiple of 4", hidden);
    MF_REQUIRE(((uintptr_t)x & 7) == 0 && ((uintptr_t)w & (w_dtype == MF_FP32 ? 15 : 7)) == 0,
               "router_gate_gemm: x must be 8-byte aligned, w 16-byte (fp32) or 8-byte aligned");
    const GatePlan p = plan_router_gate(tokens, n_experts, hidden);
    const size_t need = mf_router_gate_workspace_bytes(tokens, n_experts, hidden);
    MF_REQUIRE(need == 0 || (workspace && workspace_bytes >= need), "router_gate_gemm: workspace of %zu bytes needed, %zu given",
               need, workspace_bytes);
    float* partial = p.splits > 1 ? (float*)workspace : nullptr;
    const int te = p.tile ? RGT : 16;
    const dim3 grid((n_experts + te - 1) / te, p.splits, (tokens + 16 * RG_TT - 1) / (16 * RG_TT));
    const int64_t n = (int64_t)tokens * n_experts;
    const dim3 rgrid((unsigned)((n + 255) / 256));
#define RG_LAUNCH(TT_, WT_)                                                                                      \
    {                                                                                                            \
        auto kern = !p.tile ? router_gate_kernel<TT_, WT_>                                                       \
                    : p.chains == 2 ? router_gate_tile_kernel<TT_, WT_, 2> : router_gate_tile_kernel<TT_, WT_, 4>; \
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, (hipStream_t)stream, logits, partial, (const uint16_t*)x, w, tokens, \
                           n_experts, hidden, p.k_per_split);                                                    \
        if (partial) {                                                                                           \
            int rc = MF_LAUNCH_CHECK();                                                                          \
            if (rc) return rc;                                                                                   \
            hipLaunchKernelGGL((router_gate_reduce_kernel<WT_>), rgrid, dim3(256), 0, (hipStream_t)stream, logits, \
                               partial, n, p.splits);                                                            \
        }                                                                                                        \
    }
    if (dtype == MF_BF16) {
        if (w_dtype == MF_FP32) RG_LAUNCH(BF16, RG_F32) else RG_LAUNCH(BF16, BF16)
    } else {
        if (w_dtype == MF_FP32) RG_LAUNCH(FP16, RG_F32) else RG_LAUNCH(FP16, FP16)
    }
#undef RG_LAUNCH
    return MF_LAUNCH_CHECK();
}

extern "C" int mf_moe_permute(void* permuted_x, int32_t* row_map, int64_t* counts, int32_t* offsets, const void* x,
                              const int32_t* expert_index, int tokens, int k, int n_experts, int hidden, int dtype,
                              void* stream) {
    MF_REQUIRE(dtype == MF_BF16 || dtype == MF_FP16, "moe_permute: dtype must be bf16 or fp16");
    MF_REQUIRE(permuted_x && row_map && counts && offsets && x && expert_index, "moe_permute: null argument");
    MF_REQUIRE(n_experts > 0 && n_experts <= RT_MAX_E, "moe_permute: n_experts (%d) must be in 1..%d", n_experts, RT_MAX_E);
    MF_REQUIRE(tokens >= 0 && k > 0 && (int64_t)tokens * k <= 65536, "moe_permute: tokens*k must be <= 65536");
    MF_REQUIRE(hidden > 0 && hidden % 8 == 0, "moe_permute: hidden (%d) must be a multiple of 8", hidden);
    MF_REQUIRE((((uintptr_t)permuted_x | (uintptr_t)x) & 15) == 0, "moe_permute: rows must be 16-byte aligned");
    return permute((uint16_t*)permuted_x, nullptr, row_map, counts, offsets, (const uint16_t*)x, nullptr, expert_index, tokens,
                   k, n_experts, hidden, (hipStream_t)stream);
}

extern "C" int mf_moe_sort(int32_t* row_map, int32_t* sources, float* permuted_scale, int64_t* counts, int32_t* offsets,
                           const float* x_scale, const int32_t* expert_index, int tokens, int k, int n_experts, void* stream) {
    MF_REQUIRE(row_map && sources && counts && offsets && expert_index && !permuted_scale == !x_scale, "moe_sort: null argument");
    MF_REQUIRE(n_experts > 0 && n_experts <= RT_MAX_E, "moe_sort: n_experts (%d) must be in 1..%d", n_experts, RT_MAX_E);
    MF_REQUIRE(tokens >= 0 && k > 0 && (int64_t)tokens * k <= 65536, "moe_sort: tokens*k must be <= 65536");
    return sort_pairs(row_map, counts, offsets, expert_index, tokens * k, n_experts, {sources, permuted_scale, x_scale, k},
                      (hipStream_t)stream);
}

extern "C" int mf_moe_permute_int8(int8_t* permuted_x, float* permuted_scale, int32_t* row_map, int64_t* counts,
                                   int32_t* offsets, const int8_t* x, const float* x_scale, const int32_t* expert_index,
                                   int tokens, int k, int n_experts, int hidden, void* stream) {
    MF_REQUIRE(permuted_x && permuted_scale && row_map && counts && offsets && x && x_scale && expert_index,
               "moe_permute_int8: null argument");
    MF_REQUIRE(n_experts > 0 && n_experts <= RT_MAX_E, "moe_permute_int8: n_experts (%d) must be in 1..%d", n_experts, RT_MAX_E);
    MF_REQUIRE(tokens >= 0 && k > 0 && (int64_t)tokens * k <= 65536, "moe_permute_int8: tokens*k must be <= 65536");
    MF_REQUIRE(hidden > 0 && hidden % 16 == 0, "moe_permute_int8: hidden (%d) must be a multiple of 16", hidden);
    MF_REQUIRE((((uintptr_t)permuted_x | (uintptr_t)x) & 15) == 0, "moe_permute_int8: rows must be 16-byte aligned");
    return permute((uint16_t*)permuted_x, permuted_scale, row_map, counts, offsets, (const uint16_t*)x, x_scale, expert_index,
                   tokens, k, n_experts, hidden / 2, (hipStream_t)stream);
}

extern "C" int mf_moe_unpermute(void* out, const void* y, const int32_t* row_map, const void* probs,
                                const void* shared, int tokens, int k, int hidden, int dtype, void* stream) {
    MF_REQUIRE(dtype == MF_BF16 || dtype == MF_FP16, "moe_unpermute: dtype must be bf16 or fp16");
    if (tokens <= 0) return 0;
    MF_REQUIRE(out && y && row_map && probs, "moe_unpermute: null argument");
    MF_REQUIRE(k > 0 && hidden > 0 && hidden % 8 == 0, "moe_unpermute: hidden (%d) must be a multiple of 8", hidden);
    MF_REQUIRE((((uintptr_t)out | (uintptr_t)y | (uintptr_t)shared) & 15) == 0,
               "moe_unpermute: rows must be 16-byte aligned");
    if (tokens <= 0) return 0;
    constexpr int UNP_THREADS = 128;
    const dim3 ugrid(tokens, (hidden / 8 + UNP_THREADS - 1) / UNP_THREADS);
    if (dtype == MF_BF16)
        hipLaunchKernelGGL(moe_unpermute_kernel<BF16>, ugrid, dim3(UNP_THREADS), 0, (hipStream_t)stream, (uint16_t*)out,
                           (const uint16_t*)y, row_map, (const uint16_t*)probs, (const uint16_t*)shared, k, hidden,
                           tokens * k);
    else
        hipLaunchKernelGGL(moe_unpermute_kernel<FP16>, ugrid, dim3(UNP_THREADS), 0, (hipStream_t)stream, (uint16_t*)out,
                           (const uint16_t*)y, row_map, (const uint16_t*)probs, (const uint16_t*)shared, k, hidden,
                           tokens * k);
    return MF_LAUNCH_CHECK();
}
