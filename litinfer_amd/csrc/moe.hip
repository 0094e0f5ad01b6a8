// Routed feed-forward: the router (logits, the `top` largest, softmax over the chosen ones, and a sigmoid gate
// for a shared expert), the plan of a step (the (token, choice) pairs sorted by expert, cut into tiles of rows),
// the products of every tile's rows with its expert's matrix, and the weighted sum back into the stream.
// Nothing here returns to the host: the numbers of rows an expert gets stay on the device, and the launches are
// sized by what a step can have at most.
#include "few_rows.h"
#include "lds_loads.h"

#define MOE_TILE 32            // rows of one expert that a tile holds
#define MOE_BIG_TILE 64        // ... where experts get hundreds of rows each (a prompt's portion): the tiles of the LDS kernel,
#define MOE_HUGE_TILE 128      // and twice that where they get still more
#define MOE_NARROW_BYTES (16l << 20)   // a decoding step's tiles against matrices below this size take 64 columns a block: more blocks, filled more evenly (1.5B sizes 38 -> 32 us; 7B sizes 138 against 155 us)
#define MOE_FEW_ROWS 32        // rows of a step up to which every row may be a matrix-vector product of its own,
#define MOE_VECTOR_ROWS 4      // ... and up to which it is one also where the kernel that streams the matrices could take them
#define MOE_STREAM_ROWS 10         // rows an expert, on average, up to which that kernel is taken (see moe_streams),
#define MOE_STREAM_ROWS_LARGE 12   // ... and against matrices of MOE_NARROW_BYTES and more

// ------------------------------------------------------------------------------------------------ router
// One block a token.  logits[e] = b[e] + sum_k W[e, k] x[k] in float32 (a wave an expert, in turns); the `top`
// largest (the lower index wins a tie), weights = softmax over the chosen logits.  gate[t] = sigmoid(wg . x).
// mode 1: scores are sigmoid(logit), the choice goes by score + corr[e] inside the best groups of neighbouring
// experts, the weights are the chosen scores over their sum.  mode 2: the same with scores = softmax over ALL logits.
// Flags on top of the mode: 4: a group's score is its largest choice value (else the sum of its two largest);
// 8: the weights are the chosen scores as they are (not divided by their sum).
template <typename T> struct RouteVec;
template <> struct RouteVec<float> { static constexpr int N = 4; };
template <> struct RouteVec<bf16_t> { static constexpr int N = 8; };

// 16 bytes of a matrix row against the row in LDS, or against 16 bytes of it (the same additions in the same order)
__device__ __forceinline__ float route_dot16(const uint4 r, const uint4 x) {
    const uint32_t u[4] = {r.x, r.y, r.z, r.w}, v[4] = {x.x, x.y, x.z, x.w};
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        s = fmaf(__uint_as_float(u[i] << 16), __uint_as_float(v[i] << 16), s);
        s = fmaf(__uint_as_float(u[i] & 0xffff0000u), __uint_as_float(v[i] & 0xffff0000u), s);
    }
    return s;
}
__device__ __forceinline__ float route_dot16(const uint4 r, const float* xs, const float*) {
    return fmaf(__uint_as_float(r.x), xs[0], fmaf(__uint_as_float(r.y), xs[1], fmaf(__uint_as_float(r.z), xs[2], __uint_as_float(r.w) * xs[3])));
}
__device__ __forceinline__ float route_dot16(const uint4 r, const float* xs, const bf16_t*) {
    const uint32_t u[4] = {r.x, r.y, r.z, r.w};
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        s = fmaf(__uint_as_float(u[i] << 16), xs[2 * i], s);
        s = fmaf(__uint_as_float(u[i] & 0xffff0000u), xs[2 * i + 1], s);
    }
    return s;
}

// What a plan is made of (see moe_plan_kernel below); plan null: none.
struct MoePlanOut { int* plan; int* row_token; int* pair_row; float* row_wt; int* count; int max_tiles, tile_rows, experts; };
#define MOE_PLAN_HELD 4
#define MOE_PLACES_CHOICE 16      // router outputs a choice, up to 64 in all, up to which all places are found at once,
#define MOE_PLACES_ONE 8          // ... and for one choice
#define MOE_PLAN_EXPERTS 64       // experts up to which the router makes the plan: one a lane

// A wave's fence: what its lanes wrote to LDS is there for its other lanes
#define LI_WAVE_LDS()                                            \
    {                                                            \
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   \
        __builtin_amdgcn_wave_barrier();                         \
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");   \
    }

// The plan of a decoding step by one wave, behind the router (moe_plan_kernel in a launch of its own is 4 to 5 us, and does less
// than a microsecond's work for so few pairs).  The choices are read from memory: other blocks wrote them.
__device__ __forceinline__ void moe_plan_by_wave(const MoePlanOut& p, const int* __restrict__ idx, const float* __restrict__ wt, int pairs, int top, int* cursor) {
    const int lane = threadIdx.x & 63;
    cursor[lane] = 0;
    LI_WAVE_LDS()
    // the first 256 choices and weights wait in registers: one trip to memory
    int held[MOE_PLAN_HELD];
    float held_wt[MOE_PLAN_HELD];
#pragma unroll
    for (int q = 0; q < MOE_PLAN_HELD; ++q) {
        const int i = lane + 64 * q < pairs ? lane + 64 * q : 0;
        held[q] = __hip_atomic_load(idx + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        held_wt[q] = __hip_atomic_load(wt + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int q = 0; q < MOE_PLAN_HELD; ++q)
        if (lane + 64 * q < pairs && held[q] >= 0 && held[q] < p.experts) atomicAdd(&cursor[held[q]], 1);
    for (int i = lane + 64 * MOE_PLAN_HELD; i < pairs; i += 64) {
        const int e = __hip_atomic_load(idx + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (e >= 0 && e < p.experts) atomicAdd(&cursor[e], 1);
    }
    LI_WAVE_LDS()
    const int rows = cursor[lane], tiles = (rows + p.tile_rows - 1) / p.tile_rows;       // (lanes past the last expert: none)
    int rows_upto = rows, tiles_upto = tiles;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int a = __shfl_up(rows_upto, o, LI_WAVE), b = __shfl_up(tiles_upto, o, LI_WAVE);
        if (lane >= o) { rows_upto += a; tiles_upto += b; }
    }
    const int start = rows_upto - rows;
    for (int i = 0, nt = tiles_upto - tiles; i < tiles && nt < p.max_tiles; ++i, ++nt) {
        const int r = i * p.tile_rows;
        int* tile = p.plan + 4 + 4 * nt;
        tile[0] = lane; tile[1] = start + r; tile[2] = rows - r < p.tile_rows ? rows - r : p.tile_rows; tile[3] = 0;
    }
    if (lane == 63) { p.plan[0] = tiles_upto < p.max_tiles ? tiles_upto : p.max_tiles; p.plan[1] = rows_upto; p.plan[2] = p.plan[3] = 0; }
    cursor[lane] = start;
    LI_WAVE_LDS()
    auto place = [&](int i, int e, float weight) {
        if (e >= 0 && e < p.experts) {
            const int row = atomicAdd(&cursor[e], 1);
            p.pair_row[i] = row;
            p.row_token[row] = i / top;
            if (p.row_wt) p.row_wt[row] = weight;
        } else {
            p.pair_row[i] = -1;
        }
    };
#pragma unroll
    for (int q = 0; q < MOE_PLAN_HELD; ++q)
        if (lane + 64 * q < pairs) place(lane + 64 * q, held[q], held_wt[q]);
    for (int i = lane + 64 * MOE_PLAN_HELD; i < pairs; i += 64)
        place(i, __hip_atomic_load(idx + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), __hip_atomic_load(wt + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// Few tokens: what bounds it is a chain of trips to memory (the row, a matrix row, the pick, the plan), so a wave asks for its first
// matrix rows, where they are short enough to wait in registers, before the token's row has come; up to 64 outputs are picked at once, and
// one token's plan is made of what the wave knows (8 tokens, 16 outputs, 4 choices 12.0 -> 10.0 us).
template <typename TX, typename TW>
struct MoeRoute {
    const TX* x;
    long x_stride;
    const TW* wr;
    const float* br;
    const TW* wg;
    int* idx;
    float* wt;
    float* gate;
    int T, K, E, top, vec, mode_flags;
    const float* corr;
    int groups, keep;
    MoePlanOut po;
};

template <typename TX, typename TW, int NT>
__device__ __forceinline__ void moe_route_token(const MoeRoute<TX, TW>& a, const int t, float* sm) {
    const TX* __restrict__ x = a.x;
    const TW* __restrict__ wr = a.wr;
    const TW* __restrict__ wg = a.wg;
    const float* __restrict__ br = a.br;
    const float* __restrict__ corr = a.corr;
    int* __restrict__ idx = a.idx;
    float* __restrict__ wt = a.wt;
    float* __restrict__ gate = a.gate;
    const long x_stride = a.x_stride;
    const int K = a.K, E = a.E, top = a.top, vec = a.vec, groups = a.groups, keep = a.keep;
    const MoePlanOut& po = a.po;
    const int mode = a.mode_flags & 3;
    const bool group_max = a.mode_flags & 4, plain_weights = a.mode_flags & 8;
    // sm: [K] the row, [E] the logits, [E] the scores, [groups] the groups' scores
    float* xs = sm;
    float* lg = sm + ((K + 3) & ~3);
    float* sc = lg + E;
    float* gs = sc + E;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const TX* row = x + (size_t)t * x_stride;
    constexpr int VE = RouteVec<TW>::N;
    constexpr int HELD = 4;                            // pieces of a matrix row that a lane holds
    const int n_rows = E + (wg ? 1 : 0);
    const bool held = NT >= 512 && (vec & 1) && K / VE <= 64 * HELD;
    constexpr int FIRST = NT >= 1024 ? 2 : 3;          // matrix rows that a wave asks for at once
    uint4 piece[FIRST][HELD];
    if constexpr (NT >= 512) {
        if (held) {
#pragma unroll
            for (int q = 0; q < FIRST; ++q) {
                const int e = w + q * (NT / 64) < n_rows ? w + q * (NT / 64) : 0;       // (never conditional: a row past the last reads the first)
                const TW* wrow = e < E ? wr + (size_t)e * K : wg;
#pragma unroll
                for (int i = 0; i < HELD; ++i) {
                    const int at = lane + 64 * i < K / VE ? lane + 64 * i : 0;
                    piece[q][i] = *reinterpret_cast<const uint4*>(wrow + (size_t)at * VE);
                }
            }
        }
    }
    // Where row and matrix are bfloat16 and a wave holds all its matrix rows, every wave reads the row for itself beside them: it does not
    // pass through LDS, and nobody waits for anybody before the logits are there.
    const bool direct = sizeof(TX) == 2 && sizeof(TW) == 2 && held && (vec & 2) && n_rows <= FIRST * (NT / 64);
    [[maybe_unused]] uint4 xp[HELD];
    if (direct) {
#pragma unroll
        for (int i = 0; i < HELD; ++i) xp[i] = *reinterpret_cast<const uint4*>(row + (lane + 64 * i < K / VE ? lane + 64 * i : 0) * VE);
    } else {
        for (int k = threadIdx.x; k < K; k += NT) xs[k] = load_as_float(row + k);
        __syncthreads();
    }
    auto have = [&](int e, float s) {                  // a row's product
        if (lane == 0) {
            if (e < E) lg[e] = s + (br ? br[e] : 0.f);
            else gate[t] = 1.0f / (1.0f + expf(-s));
        }
    };
    int e = w;
    if constexpr (NT >= 512) {                         // (rows of their own: asked for in the loop below, they made every other row 0.2 us longer)
        if (held) {
            float s[FIRST];
#pragma unroll
            for (int q = 0; q < FIRST; ++q) {
                s[q] = 0.f;
#pragma unroll
                for (int i = 0; i < HELD; ++i)
                    if (lane + 64 * i < K / VE) s[q] += direct ? route_dot16(piece[q][i], xp[i]) : route_dot16(piece[q][i], xs + (lane + 64 * i) * VE, (const TW*)nullptr);
            }
#pragma unroll
            for (int q = 0; q < FIRST; ++q) s[q] = wave_sum(s[q]);
#pragma unroll
            for (int q = 0; q < FIRST; ++q, e += NT / 64)
                if (e < n_rows) have(e, s[q]);
        }
    }
    for (; e < n_rows; e += NT / 64) {
        const TW* wrow = e < E ? wr + (size_t)e * K : wg;
        float s = 0.f;
        if (vec & 1) {                                 // 16 bytes a lane and turn, several turns on their way
#pragma unroll 4
            for (int i = lane; i < K / VE; i += 64) s += route_dot16(*reinterpret_cast<const uint4*>(wrow + (size_t)i * VE), xs + i * VE, (const TW*)nullptr);
        } else {
            for (int k = lane; k < K; k += 64) s = fmaf(load_as_float(wrow + k), xs[k], s);
        }
        have(e, wave_sum(s));
    }
    __syncthreads();
    if (w != 0) return;
    if (mode != 0) {
        float smx = -INFINITY, ssum = 1.f;
        if (mode == 2) {                               // softmax over all logits: the maximum and the sum, by the wave
            for (int e = lane; e < E; e += 64) smx = fmaxf(smx, lg[e]);
            smx = wave_max(smx);
            float part = 0.f;
            for (int e = lane; e < E; e += 64) part += expf(lg[e] - smx);
            ssum = wave_sum(part);
        }
        // scores s = sigmoid(logit) (mode 2: the softmax); the choice goes by s + corr among the experts of the `keep` groups (of E / groups
        // neighbours each) whose two largest choice values have the largest sum; the weights are the chosen s, normalised
        for (int e = lane; e < E; e += 64) {
            const float s = mode == 2 ? expf(lg[e] - smx) / ssum : 1.0f / (1.0f + expf(-lg[e]));
            sc[e] = s;
            lg[e] = s + (corr ? corr[e] : 0.f);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (groups > 1 && keep < groups) {
            const int per = E / groups;
            for (int g = lane; g < groups; g += 64) {
                float a = -INFINITY, b = -INFINITY;           // the largest and the second largest of the group
                for (int e = g * per; e < (g + 1) * per; ++e) {
                    const float v = lg[e];
                    if (v > a) { b = a; a = v; } else if (v > b) b = v;
                }
                gs[g] = (per > 1 && !group_max) ? a + b : a;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // a group is kept if fewer than `keep` groups come before it (a larger score, or an equal one and a lower number)
            for (int g = lane; g < groups; g += 64) {
                const float mine_s = gs[g];
                int before = 0;
                for (int o = 0; o < groups; ++o) {
                    const float v = gs[o];
                    before += (v > mine_s || (v == mine_s && o < g)) ? 1 : 0;
                }
                if (before >= keep)
                    for (int e = g * per; e < (g + 1) * per; ++e) lg[e] = -INFINITY;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
    float chosen = 0.f, mx = 0.f, sum = 0.f;
    int mine = -1;
    unsigned long long taken = 0;                      // (up to 64 router outputs: those that were chosen)
    // All places at once is a turn an output, a round of a maximum twelve exchanges between lanes: where the choices are few for the outputs,
    // rounds (places / rounds, 3 tokens, 1 of 64 outputs of 256 columns 9.3 / 7.1 us, 2 of 64 of 2,240 12.0 / 10.3; 128 tokens, 1 of 48 7.0 / 5.4; 16
    // tokens, 1 of 32 10.0 / 9.1).
    if (E <= 64 && E <= (top == 1 ? MOE_PLACES_ONE : MOE_PLACES_CHOICE * top)) {
        // An output a lane: its place is the number of those that go before it (a larger value, or an equal one and a lower number), all
        // places at once, where rounds of a maximum took twelve exchanges between lanes a choice.  The values are compared as whole
        // numbers of the same order (both zeros the same; what is no number before all others), so every place is some output's.
        const float v = lane < E ? lg[lane] + 0.f : 0.f;
        uint32_t key = __float_as_uint(v);
        key = v != v ? 0xffffffffu : key & 0x80000000u ? ~key : key | 0x80000000u;
        int place = 0;
        for (int o = 0; o < E; ++o) {
            const uint32_t other = __builtin_amdgcn_readlane(key, o);
            place += other > key || (other == key && o < lane) ? 1 : 0;
        }
        if (lane >= E) place = 64;
        taken = __ballot(place < top);
        const float score = mode != 0 && lane < E ? sc[lane] : 0.f;
        mx = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), __ffsll((long long)__ballot(place == 0)) - 1));
        const float ex = mode != 0 ? score : expf(v - mx);
        for (int r = 0; r < top; ++r) {
            const int from = __ffsll((long long)__ballot(place == r)) - 1;
            const float one = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ex), from));
            sum += one;
            if (lane == r) { mine = from; chosen = one; }
        }
    } else
    // wave 0 picks: `top` rounds of a maximum over the logits that are left
    for (int r = 0; r < top; ++r) {
        float best = -INFINITY;
        int bi = 0x7fffffff;
        for (int e = lane; e < E; e += 64) {
            const float v = lg[e];
            if (v > best || bi == 0x7fffffff) { best = v; bi = e; }            // (ascending e a lane: the first of equals stays)
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ob = lane_xor(best, o);
            const int oi = lane_xor(bi, o);
            if (oi != 0x7fffffff && (bi == 0x7fffffff || ob > best || (ob == best && oi < bi))) { best = ob; bi = oi; }
        }
        if (r == 0) mx = best;
        const float ex = mode != 0 ? sc[bi] : expf(best - mx);
        sum += ex;
        if (lane == r) { mine = bi; chosen = ex; }
        if (E <= 64) taken |= 1ull << (bi & 63);
        if (lane == 0) lg[bi] = -INFINITY;
        // (a wave's LDS instructions are carried out in the order of their issue: the next round reads what lane 0 wrote)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if (mode != 0) sum += 1e-20f;
    const float share = plain_weights ? chosen : chosen / sum;
    if (!po.plan) {
        if (lane < top) { idx[(size_t)t * top + lane] = mine; wt[(size_t)t * top + lane] = share; }
        return;
    }
    if (a.T == 1 && E <= 64) {
        // one token's plan: a tile of one row for every expert that was chosen, from what the lanes know
        if (lane < top) { idx[lane] = mine; wt[lane] = share; }
        taken &= po.experts < 64 ? (1ull << po.experts) - 1 : ~0ull;
        const int n = __popcll(taken);
        if (lane < top) {
            const bool real = mine < po.experts;
            const int at = __popcll(taken & ((1ull << (mine & 63)) - 1));
            po.pair_row[lane] = real ? at : -1;
            if (real) {
                po.row_token[at] = 0;
                if (po.row_wt) po.row_wt[at] = share;
                int* tile = po.plan + 4 + 4 * at;
                if (at < po.max_tiles) { tile[0] = mine; tile[1] = at; tile[2] = 1; tile[3] = 0; }
            }
        }
        if (lane == 63) { po.plan[0] = n < po.max_tiles ? n : po.max_tiles; po.plan[1] = n; po.plan[2] = po.plan[3] = 0; }
        return;
    }
    // The choices go through to memory; the block counts itself there, and the one that completes the count makes the plan.
    // Nobody waits for anybody, and the count is left at zero.
    if (lane < top) {
        __hip_atomic_store(idx + (size_t)t * top + lane, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(wt + (size_t)t * top + lane, share, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (a.T > 1) {
        int before = 0;
        if (lane == 0) before = atomicAdd(po.count, 1);
        if (__builtin_amdgcn_readfirstlane(before) != a.T - 1) return;
        if (lane == 0) atomicExch(po.count, 0);
    }
    moe_plan_by_wave(po, idx, wt, a.T * top, top, reinterpret_cast<int*>(sm));
}

template <typename TX, typename TW, int NT>
__global__ __launch_bounds__(NT) void moe_route_kernel(MoeRoute<TX, TW> a) {
    extern __shared__ __align__(16) float sm[];
    moe_route_token<TX, TW, NT>(a, blockIdx.x, sm);
}

// plan (may be null) and what follows: the plan of the step as well (li_moe_plan's, over `experts` of the E router outputs), up to 128
// tokens and MOE_PLAN_EXPERTS experts; count: an int that is zero before the call and after it.
extern "C" int li_moe_route(const void* x, int x_dtype, long x_stride, const void* wr, int w_dtype, const float* br, const void* wg,
                            int* idx, float* wt, float* gate, int T, int K, int E, int top, int mode, const float* corr,
                            int groups, int keep, int* plan, int max_tiles, int* row_token, int* pair_row, int tile_rows, float* row_wt,
                            int experts, int* count, hipStream_t stream) {
    if (plan && (T > 128 || experts <= 0 || experts > MOE_PLAN_EXPERTS || experts > E || K < 64 || max_tiles <= 0 || !row_token || !pair_row || !count ||
                 (tile_rows != MOE_TILE && tile_rows != MOE_BIG_TILE && tile_rows != MOE_HUGE_TILE)))
        return LI_ERR_SIZE;
    const MoePlanOut po{plan, row_token, pair_row, row_wt, count, max_tiles, tile_rows, experts};
    if (T <= 0 || K <= 0 || E <= 0 || top <= 0 || top > E || top > 64 || x_stride < K || (wg && !gate) || mode < 0 || mode > 15 || (mode & 3) == 3 ||
        groups <= 0 || keep <= 0 || keep > groups || E % groups || (size_t)(K + 2 * E + groups + 4) * 4 > 60000)
        return LI_ERR_SIZE;
    if ((mode & 3) != 0 && (long)top > (long)keep * (E / groups)) return LI_ERR_SIZE;      // more choices than the kept groups hold
    const size_t lds = (size_t)(((K + 3) & ~3) + 2 * E + groups) * 4;
    // whole 16-byte pieces of every matrix row (the gate row included)
    const int ve = w_dtype == LI_F32 ? 4 : 8;
    const int vec = (K % ve == 0 && ((uintptr_t)wr % 16) == 0 && (!wg || ((uintptr_t)wg % 16) == 0)) | (x_dtype == LI_BF16 && x_stride % 8 == 0 && (uintptr_t)x % 16 == 0) << 1;
    // few tokens: sixteen waves share a token's experts, so that a wave has one or two rows to go through
#define MR(TX, TW)                                                                                                                \
    {                                                                                                                             \
        const MoeRoute<TX, TW> a{(const TX*)x, x_stride, (const TW*)wr, br, (const TW*)wg, idx, wt, gate, T, K, E, top, vec, mode, corr, groups, keep, po}; \
        if (T <= 128) moe_route_kernel<TX, TW, 1024><<<T, 1024, lds, stream>>>(a);                                               \
        else moe_route_kernel<TX, TW, 256><<<T, 256, lds, stream>>>(a);                                                          \
    }
    if (x_dtype == LI_F32 && w_dtype == LI_F32) MR(float, float)
    else if (x_dtype == LI_BF16 && w_dtype == LI_BF16) MR(bf16_t, bf16_t)
    else if (x_dtype == LI_BF16 && w_dtype == LI_F32) MR(bf16_t, float)
    else if (x_dtype == LI_F32 && w_dtype == LI_BF16) MR(float, bf16_t)
    else return LI_ERR_DTYPE;
#undef MR
    return li_launch_status();
}

// -------------------------------------------------------------------------------------------------- plan
// One block.  counts per expert, their running sum, every pair's row among its expert's rows (rows of an expert lie
// together), and the tiles: (expert, first row, rows).  plan = [n_tiles, 0, 0, 0 | tiles x 4 | ...]; row_token[row] is
// the token of a sorted row, pair_row[pair] the row of pair = token * top + choice; row_wt[row] (where given) the weight
// wt[pair] of the row's pair.
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int* __restrict__ idx, int pairs, int top, int E, int* __restrict__ plan,
                                                        int max_tiles, int* __restrict__ row_token, int* __restrict__ pair_row,
                                                        int tile_rows, const float* __restrict__ wt, float* __restrict__ row_wt) {
    extern __shared__ int si[];                         // [E] counts, then cursors; [E + 1] starts
    int* cnt = si;
    int* start = si + E;
    for (int e = threadIdx.x; e < E; e += 1024) cnt[e] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < pairs; i += 1024) {
        const int e = idx[i];
        if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int at = 0, nt = 0;
        for (int e = 0; e < E; ++e) {
            start[e] = at;
            for (int r = 0; r < cnt[e] && nt < max_tiles; r += tile_rows, ++nt) {
                int* tile = plan + 4 + 4 * nt;
                tile[0] = e; tile[1] = at + r; tile[2] = (cnt[e] - r < tile_rows) ? cnt[e] - r : tile_rows; tile[3] = 0;
            }
            at += cnt[e];
        }
        start[E] = at;
        plan[0] = nt; plan[1] = at; plan[2] = plan[3] = 0;
    }
    __syncthreads();
    // a pair's row: the next free one of its expert.  Which pair of an expert gets which of its rows depends on who
    // comes first; a row's result does not depend on where it lies
    for (int e = threadIdx.x; e < E; e += 1024) cnt[e] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < pairs; i += 1024) {
        const int e = idx[i];
        if (e >= 0 && e < E) {
            const int row = start[e] + atomicAdd(&cnt[e], 1);
            pair_row[i] = row;
            row_token[row] = i / top;
            if (row_wt) row_wt[row] = wt[i];
        } else {
            pair_row[i] = -1;
        }
    }
}

extern "C" int li_moe_plan(const int* idx, int T, int top, int E, int* plan, int max_tiles, int* row_token, int* pair_row,
                           int tile_rows, const float* wt, float* row_wt, hipStream_t stream) {
    if (T <= 0 || top <= 0 || E <= 0 || E > 8000 || max_tiles <= 0 || (tile_rows != MOE_TILE && tile_rows != MOE_BIG_TILE && tile_rows != MOE_HUGE_TILE) || (row_wt && !wt)) return LI_ERR_SIZE;
    moe_plan_kernel<<<1, 1024, (size_t)(2 * E + 1) * 4, stream>>>(idx, T * top, top, E, plan, max_tiles, row_token, pair_row, tile_rows, wt, row_wt);
    return li_launch_status();
}

// What follows a product: the activation (0 none, 1 max(., 0)^2, 4 gelu(.) with the error function; 2 and 3: the columns
// are (gate, up) pairs, 2 gives silu(gate) * up, 3 gives g sigmoid(1.702 g) (u + 1) with g = min(gate, limit), u =
// clamp(up, -limit, limit)), and, where the weight of a choice multiplies the expert's INPUT, the weights of the sorted
// rows (the product is linear, so the row's sums take the factor, in float32).
// The kernels have two forms: EXT with row weights and activation 4, and without (0 to 3).
struct MoeEpilogue { int act; float limit; const float* row_wt; };

__device__ __forceinline__ bool moe_is_gated(int act) { return act == 2 || act == 3; }
template <bool EXT> __device__ __forceinline__ float moe_row_factor(const MoeEpilogue& ep, int row) {
    if constexpr (EXT) return ep.row_wt ? ep.row_wt[row] : 1.0f;
    return 1.0f;
}
template <bool EXT> __device__ __forceinline__ float moe_act1(float v, int act) {
    if (EXT && act == 4) return gelu_erf(v);
    if (act == 1) { v = fmaxf(v, 0.f); v *= v; }
    return v;
}

__device__ __forceinline__ float moe_gated(float g, float u, int act, float limit) {
    if (act == 3) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
    }
    return u * (g / (1.0f + expf(-g)));
}

// Four consecutive outputs of one row, from column `col` (a multiple of 4) on; of (gate, up) pairs the two results go to
// columns col / 2 and col / 2 + 1.
template <bool EXT, typename TO>
__device__ __forceinline__ void moe_store4(TO* __restrict__ row, int col, float v0, float v1, float v2, float v3, const MoeEpilogue& ep, float factor) {
    const int act = ep.act;
    const float limit = ep.limit;
    if constexpr (EXT) { v0 *= factor; v1 *= factor; v2 *= factor; v3 *= factor; }
    if (moe_is_gated(act)) {
        const float o0 = moe_gated(v0, v1, act, limit), o1 = moe_gated(v2, v3, act, limit);
        TO* dst = row + (col >> 1);
        if constexpr (sizeof(TO) == 2) *reinterpret_cast<uint32_t*>(dst) = pack2_bf16(o0, o1);
        else *reinterpret_cast<float2*>(dst) = float2{o0, o1};
        return;
    }
    if (act) { v0 = moe_act1<EXT>(v0, act); v1 = moe_act1<EXT>(v1, act); v2 = moe_act1<EXT>(v2, act); v3 = moe_act1<EXT>(v3, act); }
    TO* dst = row + col;
    if constexpr (sizeof(TO) == 2) {
        uint32_t* d2 = reinterpret_cast<uint32_t*>(dst);
        d2[0] = pack2_bf16(v0, v1);
        d2[1] = pack2_bf16(v2, v3);
    } else {
        *reinterpret_cast<float4*>(dst) = float4{v0, v1, v2, v3};
    }
}

// ---------------------------------------------------------------------------------------- products by tile
// out[row, j] = act(sum_k W[e, j, k] * a[src(row), k]) for the rows of every tile, e the tile's expert; src(row) =
// row_token[row] where the rows are gathered from tokens, else the row itself.  act: 0 none, 1 max(., 0)^2, 2 the
// matrix rows come in pairs (2 j: gate, 2 j + 1: up) and out[row, j] = silu(gate) * up: half as many columns.
// General form: a block takes a tile and 64 outputs; rows and matrix rows go through LDS in float32, K in steps
// of 32; a thread owns 2 rows x 4 outputs.  Sums are float32 in the order of k.
template <bool EXT, typename TA, typename TW, typename TO>
__global__ __launch_bounds__(256) void moe_linear_kernel(const TA* __restrict__ a, long a_stride, const int* __restrict__ row_token,
                                                         const TW* __restrict__ w, const int* __restrict__ plan,
                                                         TO* __restrict__ out, long out_stride, int n_out, int K, MoeEpilogue ep) {
    const int tile = blockIdx.x;
    if (tile >= plan[0]) return;
    const int e = plan[4 + 4 * tile], r0 = plan[5 + 4 * tile], nr = plan[6 + 4 * tile];
    const int j0 = blockIdx.y * 64;
    __shared__ float As[MOE_TILE][33];
    __shared__ float Ws[64][33];
    __shared__ int src[MOE_TILE];
    if (threadIdx.x < MOE_TILE) {
        const int r = r0 + (threadIdx.x < nr ? threadIdx.x : 0);
        src[threadIdx.x] = row_token ? row_token[r] : r;
    }
    const int tr = threadIdx.x / 16, tc = threadIdx.x % 16;          // rows 2 tr, 2 tr + 1; outputs 2 tc + (i & 1) + 32 (i >> 1)
    float acc[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    const TW* we = w + (size_t)e * n_out * K;
    for (int k0 = 0; k0 < K; k0 += 32) {
        __syncthreads();
        for (int i = threadIdx.x; i < MOE_TILE * 32; i += 256) {
            const int r = i / 32, k = k0 + i % 32;
            As[r][i % 32] = (r < nr && k < K) ? load_as_float(a + (size_t)src[r] * a_stride + k) : 0.f;
        }
        for (int i = threadIdx.x; i < 64 * 32; i += 256) {
            const int j = j0 + i / 32, k = k0 + i % 32;
            Ws[i / 32][i % 32] = (j < n_out && k < K) ? load_as_float(we + (size_t)j * K + k) : 0.f;
        }
        __syncthreads();
#pragma unroll 8
        for (int k = 0; k < 32; ++k) {
            const float a0 = As[2 * tr][k], a1 = As[2 * tr + 1][k];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float wv = Ws[2 * tc + (i & 1) + 32 * (i >> 1)][k];
                acc[0][i] = fmaf(a0, wv, acc[0][i]);
                acc[1][i] = fmaf(a1, wv, acc[1][i]);
            }
        }
    }
#pragma unroll
    for (int rr = 0; rr < 2; ++rr) {
        const int r = 2 * tr + rr;
        if (r >= nr) continue;
        const float factor = moe_row_factor<EXT>(ep, r0 + r);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = j0 + 2 * tc + (i & 1) + 32 * (i >> 1);
            if (j >= n_out) continue;
            const float v = acc[rr][i] * factor;
            if (moe_is_gated(ep.act)) {                // (gate, up) pairs: i even holds the gate, i + 1 the up value
                if (i & 1) continue;
                store_from_float(out + (size_t)(r0 + r) * out_stride + (j >> 1), moe_gated(v, acc[rr][i + 1] * factor, ep.act, ep.limit));
                continue;
            }
            store_from_float(out + (size_t)(r0 + r) * out_stride + j, moe_act1<EXT>(v, ep.act));
        }
    }
}

// The same on the matrix cores, for bfloat16 matrices with K a multiple of 16 and n_out a multiple of 32: a wave takes
// the tile's 32 rows and 32 outputs and works on the transposed tile (outputs x rows), so that both operands are
// 16-byte pieces of rows as they lie in memory and a lane ends with four consecutive outputs of its row.
typedef __bf16 moe_bf16x8 __attribute__((ext_vector_type(8)));
typedef float moe_f32x16 __attribute__((ext_vector_type(16)));
typedef float moe_f32x4 __attribute__((ext_vector_type(4)));
union moe_frag8 { uint4 raw; uint32_t w[4]; moe_bf16x8 v; };

template <bool EXT, typename TA, typename TO>
__global__ __launch_bounds__(256) void moe_linear_mfma_kernel(const TA* __restrict__ a, long a_stride, const int* __restrict__ row_token,
                                                              const bf16_t* __restrict__ w, const int* __restrict__ plan,
                                                              TO* __restrict__ out, long out_stride, int n_out, int K, MoeEpilogue ep) {
    const int tile = blockIdx.x;
    if (tile >= plan[0]) return;
    const int e = plan[4 + 4 * tile], r0 = plan[5 + 4 * tile], nr = plan[6 + 4 * tile];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, ql = lane & 31, h2 = lane >> 5;
    const int j0 = (blockIdx.y * 4 + wv) * 32;
    if (j0 >= n_out) return;
    const int r = r0 + (ql < nr ? ql : 0);
    const int srow = row_token ? row_token[r] : r;
    const TA* arow = a + (size_t)srow * a_stride + 8 * h2;
    const bf16_t* mrow = w + ((size_t)e * n_out + j0 + ql) * K + 8 * h2;
    moe_f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    for (int k = 0; k < K; k += 16) {
        moe_frag8 fa, fb;
        fa.raw = *reinterpret_cast<const uint4*>(mrow + k);
        if constexpr (sizeof(TA) == 2) {
            fb.raw = *reinterpret_cast<const uint4*>(arow + k);
        } else {
            const float4 u = *reinterpret_cast<const float4*>(arow + k);
            const float4 v = *reinterpret_cast<const float4*>(arow + k + 4);
            fb.w[0] = pack2_bf16(u.x, u.y); fb.w[1] = pack2_bf16(u.z, u.w);
            fb.w[2] = pack2_bf16(v.x, v.y); fb.w[3] = pack2_bf16(v.z, v.w);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa.v, fb.v, acc, 0, 0, 0);
    }
    if (ql >= nr) return;
    TO* orow = out + (size_t)(r0 + ql) * out_stride;
    const float factor = moe_row_factor<EXT>(ep, r0 + ql);
#pragma unroll
    for (int rg = 0; rg < 4; ++rg)                     // registers 4 rg .. 4 rg + 3: outputs 8 rg + 4 h2 ..
        moe_store4<EXT>(orow, j0 + 8 * rg + 4 * h2, acc[4 * rg], acc[4 * rg + 1], acc[4 * rg + 2], acc[4 * rg + 3], ep, factor);
}

// The wider form, for K a multiple of 32: a wave takes the tile's 32 rows and 32 NF outputs (NF accumulators that
// share the rows' operand), K in steps of 32 with the next step's loads asked for before this step's
// matrix products.  KSPLIT = 1: the four waves of a block take 512 outputs side by side (many rows: a prompt).
// KSPLIT = 4: they take the same outputs and a quarter of K each and add up through LDS, so that the few tiles
// of a decoding step, each of which streams its expert's whole matrix, are spread over four times the waves.
template <typename TA>
__device__ __forceinline__ void moe_load_rows(moe_frag8& f, const TA* p) {
    if constexpr (sizeof(TA) == 2) {
        f.raw = *reinterpret_cast<const uint4*>(p);
    } else {
        const float4 u = *reinterpret_cast<const float4*>(p);
        const float4 v = *reinterpret_cast<const float4*>(p + 4);
        f.w[0] = pack2_bf16(u.x, u.y); f.w[1] = pack2_bf16(u.z, u.w);
        f.w[2] = pack2_bf16(v.x, v.y); f.w[3] = pack2_bf16(v.z, v.w);
    }
}

template <bool EXT, typename TA, typename TO, int KSPLIT, int NF>
__global__ __launch_bounds__(256) void moe_linear_wide_kernel(const TA* __restrict__ a, long a_stride, const int* __restrict__ row_token,
                                                              const bf16_t* __restrict__ w, const int* __restrict__ plan,
                                                              TO* __restrict__ out, long out_stride, int n_out, int K, MoeEpilogue ep,
                                                              int max_tiles) {
    int tile = blockIdx.y, cb = blockIdx.x;            // (columns first, as in the kernel of few rows)
    if (KSPLIT == 1) {
        // Many tiles: the grid is one row of blocks, which the chip deals out to its eight XCDs in turn.  Eight tiles
        // that follow each other (mostly rows of one expert) against the same columns go to ONE XCD, next to each other
        // in time, so that the expert's matrix comes into that XCD's L2 once for them and not once for each XCD.
        const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
        const int item = (((idx >> 3) << 3) + xcd) * 8 + (idx & 7);
        const int tiles = max_tiles;
        cb = item / tiles;
        tile = item % tiles;
    }
    if (tile >= plan[0]) return;
    const int e = plan[4 + 4 * tile], r0 = plan[5 + 4 * tile], nr = plan[6 + 4 * tile];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, ql = lane & 31, h2 = lane >> 5;
    const int j0 = (KSPLIT == 1 ? cb * 4 + wv : cb) * 32 * NF;
    if (KSPLIT == 1 && j0 >= n_out) return;
    int nf = (n_out - j0) / 32;                        // column fragments of 32 that exist (n_out is a multiple of 32)
    if (nf > NF) nf = NF;
    int k0 = 0, k1 = K;
    if (KSPLIT > 1) {
        const int per = ((K / 32 + KSPLIT - 1) / KSPLIT) * 32;
        k0 = wv * per;
        k1 = k0 + per < K ? k0 + per : K;
    }
    const int r = r0 + (ql < nr ? ql : 0);
    const TA* arow = a + (size_t)(row_token ? row_token[r] : r) * a_stride + 8 * h2;
    const bf16_t* mrow[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) mrow[f] = w + ((size_t)e * n_out + j0 + 32 * (f < nf ? f : 0) + ql) * K + 8 * h2;
    moe_f32x16 acc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[f][i] = 0.f;
    moe_frag8 ca[2], cw[NF][2], na[2], nw[NF][2];
    if (k0 < k1) {
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            moe_load_rows<TA>(ca[s2], arow + k0 + 16 * s2);
#pragma unroll
            for (int f = 0; f < NF; ++f) cw[f][s2].raw = *reinterpret_cast<const uint4*>(mrow[f] + k0 + 16 * s2);
        }
    }
    for (int k = k0; k < k1; k += 32) {
        const int kn = k + 32 < k1 ? k + 32 : k;       // (the last turn asks for its own step again: no branch around the loads)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            moe_load_rows<TA>(na[s2], arow + kn + 16 * s2);
#pragma unroll
            for (int f = 0; f < NF; ++f) nw[f][s2].raw = *reinterpret_cast<const uint4*>(mrow[f] + kn + 16 * s2);
        }
        // (the compiler would fold "loaded here or before the loop, used in the next turn" into one load at its use, and
        // nothing would be on its way while the wave multiplies; a load is not moved past this)
        asm volatile("" ::: "memory");
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[f] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cw[f][s2].v, ca[s2].v, acc[f], 0, 0, 0);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            ca[s2] = na[s2];
#pragma unroll
            for (int f = 0; f < NF; ++f) cw[f][s2] = nw[f][s2];
        }
    }
    int f_lo = 0, f_hi = nf;
    if (KSPLIT > 1) {
        // the four waves' sums meet in LDS; wave f then owns column fragment f
        __shared__ float red[KSPLIT][NF][16][64];
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int i = 0; i < 16; ++i) red[wv][f][i][lane] = acc[f][i];
        __syncthreads();
        if (wv >= nf) return;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float t = 0.f;
#pragma unroll
            for (int src = 0; src < KSPLIT; ++src) t += red[src][wv][i][lane];
            acc[0][i] = t;
        }
        f_lo = wv;
        f_hi = wv + 1;
    }
    if (ql >= nr) return;
    TO* orow = out + (size_t)(r0 + ql) * out_stride;
    const float factor = moe_row_factor<EXT>(ep, r0 + ql);
    for (int f = f_lo; f < f_hi; ++f) {
        const moe_f32x16 c = KSPLIT > 1 ? acc[0] : (f == 0 ? acc[0] : f == 1 ? acc[1] : f == 2 ? acc[NF > 2 ? 2 : 0] : acc[NF > 2 ? 3 : 0]);
#pragma unroll
        for (int rg = 0; rg < 4; ++rg)                 // registers 4 rg .. 4 rg + 3: outputs 32 f + 8 rg + 4 h2 ..
            moe_store4<EXT>(orow, j0 + 32 * f + 8 * rg + 4 * h2, c[4 * rg], c[4 * rg + 1], c[4 * rg + 2], c[4 * rg + 3], ep, factor);
    }
}

// A handful of rows in all (a decoding step of few requests): every tile streams its expert's matrix for one or two
// rows, so the product is a matrix-vector product a row.  A wave owns four outputs and walks their matrix rows in
// 16-byte pieces, 64 lanes side by side along K (a kilobyte of a row at a time, all four rows' pieces asked for
// together), against up to four of the tile's rows at a time; sums in float32, lanes added up at the end.
// Up to MOE_VECTOR_ROWS rows a wave owns two (twice the blocks, spread more evenly over the compute units), and a tile's one row against
// matrices of up to MR_HELD pieces a lane is one trip to memory: all of the wave's pieces are asked for before any is multiplied.
// (Two rows of 2,240 x 1,536 7.9 -> 5.9 us, of 1,536 x 2,240 8.4 -> 6.1, an empty launch being 1.6.)
#define MR_OUT 4
#define MR_OUT_FEW 2
#define MR_ROWS 4
#define MR_HELD 5

// The operands of a product by tile, bfloat16 rows and matrices
template <typename TO>
struct MoeLinear { const bf16_t* a; long a_stride; const int* row_token; const bf16_t* w; const int* plan; TO* out; long out_stride; int n_out, K; MoeEpilogue ep; };

template <bool EXT, typename TO, int OUT>
__device__ __forceinline__ void moe_linear_rows_wave(const MoeLinear<TO>& p, const int tile, const int j0) {
    const bf16_t* __restrict__ a = p.a;
    const bf16_t* __restrict__ w = p.w;
    const int* __restrict__ plan = p.plan;
    const int* __restrict__ row_token = p.row_token;
    TO* __restrict__ out = p.out;
    const long a_stride = p.a_stride, out_stride = p.out_stride;
    const int n_out = p.n_out, K = p.K;
    const MoeEpilogue& ep = p.ep;
    const int tiles = plan[0], e = plan[4 + 4 * tile], r0 = plan[5 + 4 * tile], nr = plan[6 + 4 * tile];      // (one trip: a tile past the last has its place)
    asm volatile("" ::"s"(tiles), "s"(e), "s"(r0), "s"(nr));
    const int lane = threadIdx.x & 63;
    if (tile >= tiles || j0 >= n_out) return;
    const bf16_t* wrow[OUT];
#pragma unroll
    for (int j = 0; j < OUT; ++j) wrow[j] = w + ((size_t)e * n_out + (j0 + j < n_out ? j0 + j : n_out - 1)) * K;
    // what becomes of one row's sums, in lane 0
    auto finish = [&](int row, const float (*acc)[MR_ROWS], int r) {
        TO* orow = out + (size_t)row * out_stride;
        const float factor = moe_row_factor<EXT>(ep, row);
        if (moe_is_gated(ep.act)) {                    // (gate, up) pairs: n_out is even and j0 a multiple of OUT
#pragma unroll
            for (int j = 0; j < OUT; j += 2)
                if (j0 + j < n_out) store_from_float(orow + ((j0 + j) >> 1), moe_gated(acc[j][r] * factor, acc[j + 1][r] * factor, ep.act, ep.limit));
            return;
        }
#pragma unroll
        for (int j = 0; j < OUT; ++j)
            if (j0 + j < n_out) store_from_float(orow + j0 + j, moe_act1<EXT>(acc[j][r] * factor, ep.act));
    };
    if (nr == 1 && K <= MR_HELD * 512) {               // one row: all the wave multiplies is asked for at once
        const int at = (row_token ? row_token[r0] : r0), last = K / 8 - 1;
        const bf16_t* xrow = a + (size_t)at * a_stride;
        uint4 wp[MR_HELD][OUT], xp[MR_HELD];
#pragma unroll
        for (int i = 0; i < MR_HELD; ++i) {
            if (64 * i > last) continue;               // (the wave's own question, and nothing else writes these registers: no wait at its end)
            const int c = lane + 64 * i < last ? lane + 64 * i : last;
#pragma unroll
            for (int j = 0; j < OUT; ++j) wp[i][j] = *reinterpret_cast<const uint4*>(wrow[j] + 8 * c);
            xp[i] = *reinterpret_cast<const uint4*>(xrow + 8 * c);
        }
        float acc[OUT][MR_ROWS];
#pragma unroll
        for (int j = 0; j < OUT; ++j) acc[j][0] = 0.f;
#pragma unroll
        for (int i = 0; i < MR_HELD; ++i) {
            if (64 * i > last) continue;
            const bool mine = lane + 64 * i <= last;
#pragma unroll
            for (int j = 0; j < OUT; ++j) {
                const uint32_t u[4] = {wp[i][j].x, wp[i][j].y, wp[i][j].z, wp[i][j].w}, v[4] = {xp[i].x, xp[i].y, xp[i].z, xp[i].w};
                float s = acc[j][0];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    s = fmaf(__uint_as_float(u[q] & 0xffff0000u), __uint_as_float(v[q] & 0xffff0000u), fmaf(__uint_as_float(u[q] << 16), __uint_as_float(v[q] << 16), s));
                acc[j][0] = mine ? s : acc[j][0];
            }
        }
#pragma unroll
        for (int j = 0; j < OUT; ++j) acc[j][0] = wave_sum(acc[j][0]);
        if (lane == 0) finish(r0, acc, 0);
        return;
    }
    for (int rc = 0; rc < nr; rc += MR_ROWS) {
        const bf16_t* xrow[MR_ROWS];
#pragma unroll
        for (int r = 0; r < MR_ROWS; ++r) {
            const int row = r0 + (rc + r < nr ? rc + r : nr - 1);
            xrow[r] = a + (size_t)(row_token ? row_token[row] : row) * a_stride;
        }
        float acc[OUT][MR_ROWS];
#pragma unroll
        for (int j = 0; j < OUT; ++j)
#pragma unroll
            for (int r = 0; r < MR_ROWS; ++r) acc[j][r] = 0.f;
        // the next turn's pieces of the matrix rows are on their way while this one's are multiplied (past the end: the last
        // turn's again, not used); a load is not moved past the empty statement behind it
        uint4 wp[OUT], wn[OUT];
        const int i_last = K / 8 - 1;
#pragma unroll
        for (int j = 0; j < OUT; ++j) wp[j] = *reinterpret_cast<const uint4*>(wrow[j] + 8 * (lane < i_last ? lane : i_last));
        for (int i = lane; i < K / 8; i += 64) {
            uint4 xp[MR_ROWS];
#pragma unroll
            for (int r = 0; r < MR_ROWS; ++r) xp[r] = *reinterpret_cast<const uint4*>(xrow[r] + 8 * i);
            const int in = i + 64 < i_last ? i + 64 : i_last;
#pragma unroll
            for (int j = 0; j < OUT; ++j) wn[j] = *reinterpret_cast<const uint4*>(wrow[j] + 8 * in);
            asm volatile("" ::: "memory");
            float xf[MR_ROWS][8];
#pragma unroll
            for (int r = 0; r < MR_ROWS; ++r) {
                const uint32_t u[4] = {xp[r].x, xp[r].y, xp[r].z, xp[r].w};
#pragma unroll
                for (int q = 0; q < 4; ++q) { xf[r][2 * q] = __uint_as_float(u[q] << 16); xf[r][2 * q + 1] = __uint_as_float(u[q] & 0xffff0000u); }
            }
#pragma unroll
            for (int j = 0; j < OUT; ++j) {
                const uint32_t u[4] = {wp[j].x, wp[j].y, wp[j].z, wp[j].w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float lo = __uint_as_float(u[q] << 16), hi = __uint_as_float(u[q] & 0xffff0000u);
#pragma unroll
                    for (int r = 0; r < MR_ROWS; ++r) acc[j][r] = fmaf(hi, xf[r][2 * q + 1], fmaf(lo, xf[r][2 * q], acc[j][r]));
                }
            }
#pragma unroll
            for (int j = 0; j < OUT; ++j) wp[j] = wn[j];
        }
#pragma unroll
        for (int j = 0; j < OUT; ++j)
#pragma unroll
            for (int r = 0; r < MR_ROWS; ++r)
                if (rc + r < nr) acc[j][r] = wave_sum(acc[j][r]);
        if (lane == 0) {
#pragma unroll
            for (int r = 0; r < MR_ROWS; ++r)
                if (rc + r < nr) finish(r0 + rc + r, acc, r);
        }
    }
}

template <bool EXT, typename TO, int OUT>
__global__ __launch_bounds__(256) void moe_linear_rows_kernel(MoeLinear<TO> p) {
    // (columns first: neighbouring blocks go to different XCDs, and each XCD gets a share of every expert)
    moe_linear_rows_wave<EXT, TO, OUT>(p, blockIdx.y, (blockIdx.x * 4 + (threadIdx.x >> 6)) * OUT);
}

// A decoding step of a batch: few rows an expert, and every tile streams its expert's matrix, so the product is bound by
// how many bytes of the matrices are on their way.  A block takes a tile and 16 NT outputs; its four waves take K in
// chunks of 128 in turn, each with the loads of its NEXT chunk (16 bytes a lane, 64 neighbouring bytes of a matrix row an
// instruction; whole chunks without conditions) in flight while it multiplies one, and add up through LDS.
// v_mfma_f32_16x16x32_bf16 has the matrix as the row operand and 16 of the tile's rows as the column operand, so a lane
// ends with four neighbouring outputs of one row; a tile of more than 16 rows is gone through twice (the block's share
// of the matrix is in the L2 by then).  The rows are read 256 neighbouring bytes of a row at a time and turned into the
// operand's order through a piece of LDS of the wave's own, as in the few-row product of a dense layer.
// The matrix cores lose more on the way to a long sum than the vector ALU (in one chain a wave 1.14e-7 of a result at K =
// 1,536, 2.0e-7 at 4,736, where the kernel of few rows loses 7.2e-8 and 8.7e-8), so none of their sums is longer than 32
// k-values: a chunk's four are added in pairs to one of two running sums, and so are the waves' (7.1e-8 and 8.0e-8, in the
// same time).
#define MS_CHUNK 128
template <bool EXT, typename TO, int NT>
__global__ __launch_bounds__(256) void moe_linear_stream_kernel(const bf16_t* __restrict__ a, long a_stride, const int* __restrict__ row_token,
                                                                const bf16_t* __restrict__ w, const int* __restrict__ plan,
                                                                TO* __restrict__ out, long out_stride, int n_out, int K, MoeEpilogue ep) {
    constexpr int WAVES = 4;
    const int tile = blockIdx.y;              // (columns first: see the kernel of few rows)
    const int tiles = plan[0], e = plan[4 + 4 * tile], r0 = plan[5 + 4 * tile], nr = plan[6 + 4 * tile];      // (one trip: see the kernel of few rows)
    asm volatile("" ::"s"(tiles), "s"(e), "s"(r0), "s"(nr));
    if (tile >= tiles) return;
    __shared__ moe_f32x4 red[WAVES][NT][64];
    __shared__ __attribute__((aligned(16))) uint16_t xs_all[WAVES][16 * MS_CHUNK];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, r16 = lane & 15;
    const int j0 = blockIdx.x * 16 * NT;
    uint16_t* xs = xs_all[wave];
    // (piece p of row r lies at place p ^ r: the rows that a fragment read touches fall into all banks)
    auto xslot = [](int row, int piece) { return row * MS_CHUNK + ((piece ^ row) << 3); };
    const bf16_t* wrow[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int j = j0 + 16 * nt + r16;
        wrow[nt] = w + ((size_t)e * n_out + (j < n_out ? j : n_out - 1)) * K + 8 * g;
    }
    const int nfull = K / MS_CHUNK, nchunks = (K + MS_CHUNK - 1) / MS_CHUNK;
    const moe_frag8 zero = {};
    constexpr std::integral_constant<int, 0> FIRST{};
    constexpr std::integral_constant<int, 1> SECOND{};
    for (int rc = 0; rc < nr; rc += 16) {
        const bf16_t* xrow[4];                // this lane's rows of x: g + 4 i, the last one repeated past the tile's end
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + (rc + g + 4 * i < nr ? rc + g + 4 * i : nr - 1);
            xrow[i] = a + (size_t)(row_token ? row_token[r] : r) * a_stride + 8 * r16;
        }
        moe_f32x4 acc[NT][2];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[nt][b] = moe_f32x4{0.f, 0.f, 0.f, 0.f};
        moe_frag8 wbuf[2][NT][4], xbuf[2][4];
        auto load_chunk = [&](int c, moe_frag8 (*wd)[4], moe_frag8* xd, auto tail_tag) {
            constexpr bool TAIL = decltype(tail_tag)::value;
            const int kb = c * MS_CHUNK;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (TAIL) { xd[i] = zero; if (kb + 8 * r16 < K) xd[i].raw = *reinterpret_cast<const uint4*>(xrow[i] + kb); }
                else xd[i].raw = *reinterpret_cast<const uint4*>(xrow[i] + kb);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    if constexpr (TAIL) { wd[nt][j] = zero; if (kb + 8 * g + 32 * j < K) wd[nt][j].raw = *reinterpret_cast<const uint4*>(wrow[nt] + kb + 32 * j); }
                    else wd[nt][j].raw = *reinterpret_cast<const uint4*>(wrow[nt] + kb + 32 * j);
                }
        };
        auto multiply = [&](moe_frag8 (*wa)[4], moe_frag8* xd, auto buf_tag) {
            __builtin_amdgcn_wave_barrier();  // (a wave's LDS instructions are carried out in order; keep the compiler's too)
#pragma unroll
            for (int i = 0; i < 4; ++i) *reinterpret_cast<uint4*>(&xs[xslot(g + 4 * i, r16)]) = xd[i].raw;
            __builtin_amdgcn_wave_barrier();
            moe_frag8 xa[4];
            moe_f32x4 part[NT][4];
#pragma unroll
            for (int j = 0; j < 4; ++j) xa[j].raw = *reinterpret_cast<const uint4*>(&xs[xslot(r16, g + 4 * j)]);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int j = 0; j < 4; ++j) part[nt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[nt][j].v, xa[j].v, moe_f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[nt][decltype(buf_tag)::value] += (part[nt][0] + part[nt][1]) + (part[nt][2] + part[nt][3]);
            __builtin_amdgcn_wave_barrier();
        };
        // Nothing about the loads inside the loop is conditional: it runs while both of a turn's loads exist, and the one or
        // two chunks that are left are taken behind it (where a path with loads and one without meet, the compiler waits for all).
        int c = wave;
        if (c < nfull) {
            load_chunk(c, wbuf[0], xbuf[0], std::false_type{});
            for (; c + 2 * WAVES < nfull; c += 2 * WAVES) {
                load_chunk(c + WAVES, wbuf[1], xbuf[1], std::false_type{});
                multiply(wbuf[0], xbuf[0], FIRST);
                load_chunk(c + 2 * WAVES, wbuf[0], xbuf[0], std::false_type{});
                multiply(wbuf[1], xbuf[1], SECOND);
            }
            const bool more = c + WAVES < nfull;
            if (more) load_chunk(c + WAVES, wbuf[1], xbuf[1], std::false_type{});
            multiply(wbuf[0], xbuf[0], FIRST);
            if (more) multiply(wbuf[1], xbuf[1], SECOND);
        }
        if (nfull < nchunks && wave == nfull % WAVES) {      // the chunk that K ends in
            load_chunk(nfull, wbuf[0], xbuf[0], std::true_type{});
            multiply(wbuf[0], xbuf[0], FIRST);
        }
        if (rc) __syncthreads();              // the sums of the 16 rows before have been read
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) red[wave][nt][lane] = acc[nt][0] + acc[nt][1];
        __syncthreads();
        if (wave < NT) {                      // wave nt writes the 16 outputs of column tile nt
            const moe_f32x4 s = (red[0][wave][lane] + red[1][wave][lane]) + (red[2][wave][lane] + red[3][wave][lane]);
            const int row = rc + r16, col = j0 + 16 * wave + 4 * g;
            if (row < nr && col < n_out)
                moe_store4<EXT>(out + (size_t)(r0 + row) * out_stride, col, s[0], s[1], s[2], s[3], ep, moe_row_factor<EXT>(ep, r0 + row));
        }
    }
}

// Many rows an expert (tiles of up to 64 rows): a block takes a tile and 128 outputs, K in steps of 32 through LDS, so
// that a matrix row that came from memory serves 64 rows and a token's row 128 outputs; its four waves are two by two,
// each with 32 rows x 64 outputs (two accumulators).  The block is small on purpose: five or more of them share a compute
// unit, and while one waits for its next pieces (they wait in registers while this step is multiplied) or at its
// barriers, the others multiply.  bfloat16 rows and matrices; the same transposed tiles (outputs x rows) as above.
#define MB_COLS 128
#define MB_K 32                // k-values a step (64 bytes of a row: with 128 a block's LDS doubles and half as many blocks share a compute unit: 298 against 210 us)
#define MB_DEPTH 2             // steps whose pieces wait in registers (four: no faster)
#define MB_LD (MB_K + 8)       // elements of an LDS row: 8 of padding (144 bytes: the 16-byte reads of 16 lanes spread over the banks)

template <bool EXT, typename TO, int RF>      // RF: row fragments of 32 a wave (1: tiles of 64 rows, 2: of 128)
__global__ __launch_bounds__(256) void moe_linear_lds_kernel(const bf16_t* __restrict__ a, long a_stride, const int* __restrict__ row_token,
                                                             const bf16_t* __restrict__ w, const int* __restrict__ plan,
                                                             TO* __restrict__ out, long out_stride, int n_out, int K, MoeEpilogue ep,
                                                             int max_tiles) {
    constexpr int MB_ROWS = 64 * RF;
    __shared__ __align__(16) uint16_t As[MB_ROWS * MB_LD];
    __shared__ __align__(16) uint16_t Ws[MB_COLS * MB_LD];
    __shared__ int src[MB_ROWS];
    // (eight tiles that follow each other against the same columns go to one XCD: see the wide kernel)
    const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
    const int item = (((idx >> 3) << 3) + xcd) * 8 + (idx & 7);
    const int cb = item / max_tiles, tile = item % max_tiles;
    if (tile >= plan[0] || cb * MB_COLS >= n_out) return;
    const int e = plan[4 + 4 * tile], r0 = plan[5 + 4 * tile], nr = plan[6 + 4 * tile];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, ql = lane & 31, h2 = lane >> 5;
    const int j0 = cb * MB_COLS;
    if (tid < MB_ROWS) {
        const int r = r0 + (tid < nr ? tid : nr - 1);
        src[tid] = row_token ? row_token[r] : r;
    }
    __syncthreads();
    // what a thread brings in a step: 16-byte pieces, MB_K / 8 to a row: NA of token rows, NW of matrix rows
    constexpr int PP = MB_K / 8, RP = 256 / PP, NA = MB_ROWS / RP, NW = MB_COLS / RP;
    const int prow = tid / PP, part = tid % PP;
    const bf16_t* ga[NA];
    const bf16_t* gw[NW];
    int la[NA], lw[NW];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int row = prow + RP * i;
        ga[i] = a + (size_t)src[row] * a_stride + 8 * part;
        la[i] = row * MB_LD + 8 * part;
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const int row = prow + RP * i;
        const int j = j0 + row < n_out ? j0 + row : n_out - 1;
        gw[i] = w + ((size_t)e * n_out + j) * K + 8 * part;
        lw[i] = row * MB_LD + 8 * part;
    }
    const int wr = wv >> 1, wc = wv & 1;               // the wave's 32 * RF rows and 64 outputs
    moe_f32x16 acc[RF][2];
#pragma unroll
    for (int rf = 0; rf < RF; ++rf)
#pragma unroll
        for (int cf = 0; cf < 2; ++cf)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[rf][cf][i] = 0.f;
    // the pieces of the next MB_DEPTH steps wait in registers: a step's pieces are asked for that many steps before they go to LDS
    uint4 ra[MB_DEPTH][NA], rw[MB_DEPTH][NW];
    const int last = K - MB_K;
#pragma unroll
    for (int d = 0; d < MB_DEPTH; ++d) {
        const int kd = d * MB_K < last ? d * MB_K : last;
#pragma unroll
        for (int i = 0; i < NA; ++i) ra[d][i] = *reinterpret_cast<const uint4*>(ga[i] + kd);
#pragma unroll
        for (int i = 0; i < NW; ++i) rw[d][i] = *reinterpret_cast<const uint4*>(gw[i] + kd);
    }
    for (int k = 0; k < K; k += MB_K) {
        __syncthreads();                               // the step before has been read
#pragma unroll
        for (int i = 0; i < NA; ++i) *reinterpret_cast<uint4*>(&As[la[i]]) = ra[0][i];
#pragma unroll
        for (int i = 0; i < NW; ++i) *reinterpret_cast<uint4*>(&Ws[lw[i]]) = rw[0][i];
        __syncthreads();
        const int kn = k + MB_DEPTH * MB_K < last ? k + MB_DEPTH * MB_K : last;      // (past the end: the last step again, no branch around the loads)
#pragma unroll
        for (int i = 0; i < NA; ++i) {
#pragma unroll
            for (int d = 0; d + 1 < MB_DEPTH; ++d) ra[d][i] = ra[d + 1][i];
            ra[MB_DEPTH - 1][i] = *reinterpret_cast<const uint4*>(ga[i] + kn);
        }
#pragma unroll
        for (int i = 0; i < NW; ++i) {
#pragma unroll
            for (int d = 0; d + 1 < MB_DEPTH; ++d) rw[d][i] = rw[d + 1][i];
            rw[MB_DEPTH - 1][i] = *reinterpret_cast<const uint4*>(gw[i] + kn);
        }
#pragma unroll
        for (int s2 = 0; s2 < MB_K / 16; ++s2) {
            moe_frag8 fa[RF], fw[2];
#pragma unroll
            for (int rf = 0; rf < RF; ++rf)
                fa[rf].raw = *reinterpret_cast<const uint4*>(&As[(32 * RF * wr + 32 * rf + ql) * MB_LD + 16 * s2 + 8 * h2]);
#pragma unroll
            for (int cf = 0; cf < 2; ++cf)
                fw[cf].raw = *reinterpret_cast<const uint4*>(&Ws[(64 * wc + 32 * cf + ql) * MB_LD + 16 * s2 + 8 * h2]);
#pragma unroll
            for (int rf = 0; rf < RF; ++rf)
#pragma unroll
                for (int cf = 0; cf < 2; ++cf)
                    acc[rf][cf] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[cf].v, fa[rf].v, acc[rf][cf], 0, 0, 0);
        }
    }
#pragma unroll
    for (int rf = 0; rf < RF; ++rf) {
        const int row = 32 * RF * wr + 32 * rf + ql;
        if (row >= nr) continue;
        TO* orow = out + (size_t)(r0 + row) * out_stride;
        const float factor = moe_row_factor<EXT>(ep, r0 + row);
#pragma unroll
        for (int cf = 0; cf < 2; ++cf) {
            if (j0 + 64 * wc + 32 * cf >= n_out) continue;
#pragma unroll
            for (int rg = 0; rg < 4; ++rg)             // registers 4 rg .. 4 rg + 3: outputs 32 cf + 8 rg + 4 h2 ..
                moe_store4<EXT>(orow, j0 + 64 * wc + 32 * cf + 8 * rg + 4 * h2, acc[rf][cf][4 * rg], acc[rf][cf][4 * rg + 1],
                           acc[rf][cf][4 * rg + 2], acc[rf][cf][4 * rg + 3], ep, factor);
        }
    }
}

// 1 if tiles of MOE_BIG_TILE rows have a kernel for these operands
// Many rows an expert and K a multiple of 64: the same tiles with the loads going straight into LDS, two stages of 64 k-values in turn.  A
// block takes a tile of 64 RF rows and 64 CF outputs, its four waves two by two; a lane's row of a matrix instruction is an output, its column
// a row of the tile, and the k-values come in the order of the kernel above: the sums are the same bit for bit.
// A stage holds the rows' and the matrix's pieces of 16 bytes, piece c of row r at place c ^ (r / 2 % 8) of the row's eight: the reads of 32
// lanes fall into all banks.  The loads of the step ahead are issued one by one between the matrix instructions (back to back they
// would hold the wave until the address unit has taken them); in the middle of a step's last group the wave waits for them and meets the
// others.  Two blocks share a compute unit and cover each other's waits and the trips to memory before a block's first load; with three or
// four stages and one block, or stages of 32 k-values and three blocks, the large cases took 10 to 20 % longer.
// What it was bound by is the way from memory into the XCDs' L2 (some 9 TB/s were asked for): see the order of the blocks.
// us, the kernel above / this one with its order of blocks / with the order below, random choices: 4,096 rows, 16 experts of 2,240 x 1,536 78.9 / 57.0 /
// 50.7 (42.6 with 192 outputs a block), of 1,536 x 2,240 76.1 / 64.4 / 42.4; 8,000 rows, 14 of 4,480 x 1,536 203 / 162 / 154, of 1,536 x 2,240 125 /
// 92 / 78; 4,096 rows, 8 of 9,472 x 3,584 487 / 404 / 390 (358); tiles of 64 rows: 2,048 rows, 16 of 2,240 x 1,536 54.6 / 43.0 / 31.7.
#define MD_K 64
#define MD_STAGES 2
template <bool EXT, typename TO, int RF, int CF>
__global__ __launch_bounds__(256) void moe_linear_dma_kernel(const bf16_t* __restrict__ a, long a_stride, const int* __restrict__ row_token,
                                                             const bf16_t* __restrict__ w, const int* __restrict__ plan,
                                                             TO* __restrict__ out, long out_stride, int n_out, int K, MoeEpilogue ep) {
    constexpr int BK = MD_K, NSTAGE = MD_STAGES, ROWS = 64 * RF, COLS = 64 * CF, PP = BK / 8, WRAP = 128 / BK, RPI = 64 / PP, IA = ROWS / 4 / RPI, IW = COLS / 4 / RPI, LPW = IA + IW, STAGE = (ROWS + COLS) * BK, KS = BK / 16, GM = CF * RF;
    extern __shared__ __align__(16) uint16_t stages[];
    // Blocks go to the eight XCDs in turn.  Each XCD gets an eighth of the tiles, against all columns, and goes through them columns outside: its
    // tiles' rows stay in its L2, and an expert's matrix comes into one or two of them, not into all.
    const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, tiles = plan[0];
    const int t0 = (int)((long)xcd * tiles >> 3), mine = (int)((long)(xcd + 1) * tiles >> 3) - t0;
    if (mine <= 0) return;
    const int cb = idx / mine, tile = t0 + (idx - cb * mine);
    if (cb * COLS >= n_out) return;
    const int e = plan[4 + 4 * tile], r0 = plan[5 + 4 * tile], nr = plan[6 + 4 * tile];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ql = lane & 31, h2 = lane >> 5;
    const int j0 = cb * COLS;
    // this lane's part of a step: an instruction covers eight rows, lane l row l / 8, place l % 8
    const bf16_t* ga[IA];
    const bf16_t* gw[IW];
#pragma unroll
    for (int i = 0; i < IA; ++i) {
        const int row = (ROWS / 4) * wv + RPI * i + lane / PP, c = (lane % PP) ^ ((row / WRAP) & (PP - 1));
        const int r = r0 + (row < nr ? row : nr - 1);
        ga[i] = a + (size_t)(row_token ? row_token[r] : r) * a_stride + 8 * c;
    }
#pragma unroll
    for (int i = 0; i < IW; ++i) {
        const int row = (COLS / 4) * wv + RPI * i + lane / PP, c = (lane % PP) ^ ((row / WRAP) & (PP - 1));
        gw[i] = w + ((size_t)e * n_out + (j0 + row < n_out ? j0 + row : n_out - 1)) * K + 8 * c;
    }
    // load i of the wave's LPW of a step: its rows' first, then the matrix's
    auto issue_one = [&](int kt, int i) {
        uint16_t* st = stages + (kt % NSTAGE) * STAGE;
        if (i < IA) LI_LOAD_TO_LDS_FROM(ga[i] + (size_t)kt * BK, st + ((ROWS / 4) * wv + RPI * i) * BK);
        else LI_LOAD_TO_LDS_FROM(gw[i - IA] + (size_t)kt * BK, st + ROWS * BK + ((COLS / 4) * wv + RPI * (i - IA)) * BK);
    };
    const int nk = K / BK;
    const int wr = wv >> 1, wc = wv & 1;               // the wave's 32 RF rows and 64 outputs
    moe_f32x16 acc[RF][CF];
#pragma unroll
    for (int rf = 0; rf < RF; ++rf)
#pragma unroll
        for (int cf = 0; cf < CF; ++cf)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[rf][cf][i] = 0.f;
#pragma unroll
    for (int p = 0; p < NSTAGE - 1; ++p)
        if (p < nk)
#pragma unroll
            for (int i = 0; i < LPW; ++i) issue_one(p, i);
    moe_frag8 fa[2][RF], fw[2][CF];
    auto read = [&](int kt, int ks, int buf) {
        const uint16_t* as = stages + (kt % NSTAGE) * STAGE;
        const uint16_t* ws = as + ROWS * BK;
#pragma unroll
        for (int rf = 0; rf < RF; ++rf) {
            const int row = 32 * RF * wr + 32 * rf + ql;
            fa[buf][rf].raw = *reinterpret_cast<const uint4*>(&as[row * BK + (((2 * ks + h2) ^ ((row / WRAP) & (PP - 1))) << 3)]);
        }
#pragma unroll
        for (int cf = 0; cf < CF; ++cf) {
            const int row = 32 * CF * wc + 32 * cf + ql;
            fw[buf][cf].raw = *reinterpret_cast<const uint4*>(&ws[row * BK + (((2 * ks + h2) ^ ((row / WRAP) & (PP - 1))) << 3)]);
        }
    };
    auto multiply = [&](int buf, int m) {
        acc[m / CF][m % CF] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[buf][m % CF].v, fa[buf][m / CF].v, acc[m / CF][m % CF], 0, 0, 0);
    };
    // the loads of steps that may stay in flight: `younger` of them
    auto arrived = [&](int younger) {
        if (younger >= 2) LI_VMCNT(2 * LPW); else if (younger == 1) LI_VMCNT(LPW); else LI_VMCNT(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);            // (lgkmcnt(0): this wave's reads of the stage that is given back are done)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    static_assert(NSTAGE <= 4, "at most two steps stay in flight behind the one that is waited for");
    arrived((nk < NSTAGE - 1 ? nk : NSTAGE - 1) - 1);
    read(0, 0, 0);
    // LOADS: the step NSTAGE - 1 further on exists, and its loads are issued
    auto step = [&](int kt, auto loads_tag) {
        constexpr bool LOADS = decltype(loads_tag)::value;
        static_for<KS - 1>([&](auto ks_tag) {
            constexpr int ks = decltype(ks_tag)::value;
            constexpr int l0 = LPW * ks / (KS - 1), l1 = LPW * (ks + 1) / (KS - 1);
            read(kt, ks + 1, (ks + 1) & 1);
            static_for<GM>([&](auto m_tag) {
                constexpr int m = decltype(m_tag)::value;
                multiply(ks & 1, m);
                if constexpr (LOADS) {
#pragma unroll
                    for (int l = l0 + m * (l1 - l0) / GM; l < l0 + (m + 1) * (l1 - l0) / GM; ++l) issue_one(kt + NSTAGE - 1, l);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        constexpr int BL = (KS - 1) & 1;
#pragma unroll
        for (int m = 0; m < GM / 2; ++m) multiply(BL, m);
        if (kt + 1 < nk) {
            arrived(LOADS ? NSTAGE - 2 : (nk - 2 - kt < NSTAGE - 2 ? nk - 2 - kt : NSTAGE - 2));
            read(kt + 1, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = GM / 2; m < GM; ++m) multiply(BL, m);
    };
    int kt = 0;
    for (; kt + NSTAGE - 1 < nk; ++kt) step(kt, std::true_type{});
    for (; kt < nk; ++kt) step(kt, std::false_type{});
#pragma unroll
    for (int rf = 0; rf < RF; ++rf) {
        const int row = 32 * RF * wr + 32 * rf + ql;
        if (row >= nr) continue;
        TO* orow = out + (size_t)(r0 + row) * out_stride;
        const float factor = moe_row_factor<EXT>(ep, r0 + row);
#pragma unroll
        for (int cf = 0; cf < CF; ++cf) {
            if (j0 + 32 * CF * wc + 32 * cf >= n_out) continue;
#pragma unroll
            for (int rg = 0; rg < 4; ++rg)             // registers 4 rg .. 4 rg + 3: outputs 32 cf + 8 rg + 4 h2 ..
                moe_store4<EXT>(orow, j0 + 32 * CF * wc + 32 * cf + 8 * rg + 4 * h2, acc[rf][cf][4 * rg], acc[rf][cf][4 * rg + 1],
                                acc[rf][cf][4 * rg + 2], acc[rf][cf][4 * rg + 3], ep, factor);
        }
    }
}
// The tiles of a plan, as far as the host knows the choices: half a tile an expert is not full, and no expert with fewer rows than the average has
// fewer tiles than they need.
static int moe_tiles_expected(int rows, int max_tiles, int tile_rows) {
    const int experts = max_tiles - rows / tile_rows;
    if (experts <= 0) return max_tiles;
    const int half = rows / tile_rows + experts / 2, even = experts * ((rows / experts + tile_rows - 1) / tile_rows);
    const int tiles = half > even ? half : even;
    return tiles < max_tiles ? tiles : max_tiles;
}
// Outputs a block, 128 or 192, for tiles of 128 rows: by the rounds of two blocks a compute unit that the XCD with the most tiles takes (192 outputs read
// the rows less often, a twentieth in their favour).  (Counted over the whole chip, 4,096 rows over 14 experts of 2,240 x 1,536, 42 tiles,
// fitted one round in 192 outputs and took two on the XCDs with six tiles: 87.7 us, in 128 outputs 69.8.)
static bool moe_dma_wide(int rows, int max_tiles, int n_out) {
    const int tiles = (moe_tiles_expected(rows, max_tiles, MOE_HUGE_TILE) + 7) / 8, slots = compute_units() / 4 > 0 ? compute_units() / 4 : 1;
    const int wide = (tiles * ((n_out + 191) / 192) + slots - 1) / slots, narrow = (tiles * ((n_out + 127) / 128) + slots - 1) / slots;
    return 0.95f * 3.f * wide < 2.f * narrow;
}

template <bool EXT, typename TO, int RF, int CF>
static int launch_moe_dma(hipStream_t stream, const void* a, long a_stride, const int* row_token, const void* w, const int* plan, void* out,
                          long out_stride, int n_out, int K, const MoeEpilogue& ep, int max_tiles) {
    constexpr int COLS = 64 * CF, lds = MD_STAGES * (64 * RF + COLS) * MD_K * 2;
    const dim3 grid((unsigned)((long)((max_tiles + 7) / 8) * ((n_out + COLS - 1) / COLS) * 8));
    if constexpr (lds > 65536) {
        static const hipError_t ready = hipFuncSetAttribute((const void*)moe_linear_dma_kernel<EXT, TO, RF, CF>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (ready != hipSuccess) return LI_ERR_LAUNCH;
    }
    moe_linear_dma_kernel<EXT, TO, RF, CF><<<grid, 256, lds, stream>>>((const bf16_t*)a, a_stride, row_token, (const bf16_t*)w, plan, (TO*)out, out_stride,
                                                                           n_out, K, ep);
    return li_launch_status();
}

extern "C" int li_moe_linear_big_takes(int a_dtype, int w_dtype, int n_out, int K) {
    return a_dtype == LI_BF16 && w_dtype == LI_BF16 && K % MB_K == 0 && n_out % 32 == 0;
}

// Whether a decoding step's product takes the kernel that streams the matrices (max_tiles = rows / MOE_TILE + experts, or
// fewer where there are fewer rows than that).  It goes through the matrix of a tile of more than 16 rows twice, so the line
// is drawn by the rows an expert has on average.  Us a product, other kernels (matrix-vector products up to 32 rows, tiles of 32 rows with K
// in quarters above) / this one, random choices: 16 experts of 2,240 x 1,536 4 rows 8.5 / 8.7, 8 rows 8.9 / 8.6, 32 rows
// 26.8 / 19.7, 64 rows 30.0 / 19.7 (110 MB: 5.6 TB/s), 128 rows 30.7 / 20.8; 1,536 x 2,240 at 128 rows 27.8 / 20.8, 160 rows
// 28.4 / 22.1, 192 rows 29.0 / 26.0, 256 rows 30.1 / 34.0; gate and up together (4,480 x 1,536) at 32 rows 40.6 / 35.0; 1,024 x
// 1,024 at 128 rows 9.2 / 8.2, 160 rows 9.4 / 9.3, 192 rows 9.6 / 10.6; 64 experts of 768 x 1,536 at 640 rows 34.4 / 31.4;
// 8 experts of 4,736 x 3,584 at 8 rows 29.9 / 28.0, 64 rows 84 / 43, 96 rows 86 / 46; of 3,584 x 4,736 at 10 rows 39.3 /
// 40.1, 32 rows 58 / 42, 96 rows 57 / 49, 128 rows 59 / 69.
// Where no more rows than experts bring 15 to 45 MB of rather long matrix rows, most tiles have one row, and the products
// of few rows are the faster by a little (means of five draws: 128 experts of 768 x 2,048, 6 / 8 / 10 / 12 / 16 rows 6.6 /
// 7.7 / 8.4 / 9.3 / 11.5 against 7.5 / 8.1 / 8.3 / 10.4 / 11.1 here; 64 of 768 x 1,536 5 / 8 / 12 / 20 rows 6.0 / 6.4 / 7.5 / 10.4 against 4.6 /
// 6.3 / 7.8 / 9.5; 16 of 2,240 x 1,536 5 / 8 rows 7.9 / 12.1 against 8.3 / 10.8; 64 of 1,536 x 768 12 rows 8.6 against 7.9).
static bool moe_streams(int rows, int max_tiles, int n_out, int K) {
    const long experts = max_tiles - rows / MOE_TILE, bytes = 2l * n_out * K, reads = rows * bytes;
    if (rows <= MOE_VECTOR_ROWS || (rows <= max_tiles && K >= 1280 && reads >= 15000000 && reads <= 45000000)) return false;
    return rows <= (bytes < MOE_NARROW_BYTES ? MOE_STREAM_ROWS : MOE_STREAM_ROWS_LARGE) * experts;
}
extern "C" int li_moe_linear_streams(int rows, int max_tiles, int n_out, int K) { return moe_streams(rows, max_tiles, n_out, K); }

template <bool EXT>
static int moe_linear_launch(const void* a, int a_dtype, long a_stride, const int* row_token, const void* w, int w_dtype,
                             const int* plan, int max_tiles, void* out, int out_dtype, long out_stride, int n_out, int K, MoeEpilogue ep,
                             int tile_rows, int rows, hipStream_t stream) {
    if (tile_rows == MOE_BIG_TILE || tile_rows == MOE_HUGE_TILE) {
        if (!li_moe_linear_big_takes(a_dtype, w_dtype, n_out, K) || a_stride % 8 || out_stride % 4 ||
            ((uintptr_t)a | (uintptr_t)w | (uintptr_t)out) % 16)
            return LI_ERR_SIZE;
        const dim3 line((unsigned)((((long)max_tiles * ((n_out + MB_COLS - 1) / MB_COLS) + 63) / 64) * 64));
#define ML(TO, RF) moe_linear_lds_kernel<EXT, TO, RF><<<line, 256, 0, stream>>>((const bf16_t*)a, a_stride, row_token, (const bf16_t*)w, plan, (TO*)out, out_stride, n_out, K, ep, max_tiles)
        const bool huge = tile_rows == MOE_HUGE_TILE;
        if (K % MD_K == 0 && (out_dtype == LI_BF16 || out_dtype == LI_F32)) {
#define MD(TO, RF, CF) return launch_moe_dma<EXT, TO, RF, CF>(stream, a, a_stride, row_token, w, plan, out, out_stride, n_out, K, ep, max_tiles)
            const bool wide = huge && moe_dma_wide(rows, max_tiles, n_out);
            if (out_dtype == LI_BF16) { if (!huge) MD(bf16_t, 1, 2); if (wide) MD(bf16_t, 2, 3); MD(bf16_t, 2, 2); }
            if (!huge) MD(float, 1, 2);
            if (wide) MD(float, 2, 3);
            MD(float, 2, 2);
#undef MD
        }
        if (out_dtype == LI_BF16) { if (huge) ML(bf16_t, 2); else ML(bf16_t, 1); }
        else if (out_dtype == LI_F32) { if (huge) ML(float, 2); else ML(float, 1); }
        else return LI_ERR_DTYPE;
#undef ML
        return li_launch_status();
    }
    if (tile_rows != MOE_TILE) return LI_ERR_SIZE;
    const bool pieces = a_dtype == LI_BF16 && w_dtype == LI_BF16 && K % 8 == 0 && a_stride % 8 == 0 &&
                        ((uintptr_t)a | (uintptr_t)w) % 16 == 0 && (out_dtype == LI_BF16 || out_dtype == LI_F32);
    const int gate2 = ep.act == 2 || ep.act == 3 ? 2 : 1;        // (a store takes four sums: two outputs where they are pairs)
    if (pieces && moe_streams(rows, max_tiles, n_out, K) && n_out % 4 == 0 &&
        out_stride % (4 / gate2) == 0 && (uintptr_t)out % (4 / gate2 * (out_dtype == LI_BF16 ? 2 : 4)) == 0 && max_tiles <= 65535) {
        const bool two = rows >= 4l * max_tiles;         // two column tiles a block, half the reads of x: 128 rows over 16 experts 25.4 -> 24.7 us, 8 rows 13.2 -> 14.3
        const dim3 grid((n_out + (two ? 31 : 15)) / (two ? 32 : 16), max_tiles);
#define MS(TO, NT) moe_linear_stream_kernel<EXT, TO, NT><<<grid, 256, 0, stream>>>((const bf16_t*)a, a_stride, row_token, (const bf16_t*)w, plan, (TO*)out, out_stride, n_out, K, ep)
        if (out_dtype == LI_BF16) { if (two) MS(bf16_t, 2); else MS(bf16_t, 1); }
        else { if (two) MS(float, 2); else MS(float, 1); }
#undef MS
        return li_launch_status();
    }
    // a handful of rows in all: a matrix-vector product a row
    if (rows <= MOE_FEW_ROWS && pieces) {
        // (two outputs a wave against rows too long to be held are a loop over pieces, in which four keep more loads on their way: one token, 4 of 14
        // experts of 2,048 x 4,096, 15.0 / 13.8 us)
        const int wave_out = rows <= MOE_VECTOR_ROWS && K <= MR_HELD * 512 ? MR_OUT_FEW : MR_OUT;
        const dim3 grid((n_out + 4 * wave_out - 1) / (4 * wave_out), max_tiles);
#define MF(TO, OUT) moe_linear_rows_kernel<EXT, TO, OUT><<<grid, 256, 0, stream>>>(MoeLinear<TO>{(const bf16_t*)a, a_stride, row_token, (const bf16_t*)w, plan, (TO*)out, out_stride, n_out, K, ep})
        if (out_dtype == LI_BF16) { if (wave_out == MR_OUT) MF(bf16_t, MR_OUT); else MF(bf16_t, MR_OUT_FEW); }
        else { if (wave_out == MR_OUT) MF(float, MR_OUT); else MF(float, MR_OUT_FEW); }
#undef MF
        return li_launch_status();
    }
    if (w_dtype == LI_BF16 && K % 16 == 0 && n_out % 32 == 0 && a_stride % 8 == 0 && out_stride % 4 == 0 &&
        ((uintptr_t)a | (uintptr_t)w | (uintptr_t)out) % 16 == 0 && (a_dtype == LI_BF16 || a_dtype == LI_F32)) {
        // few tiles (a decoding step: each streams its expert's whole matrix): K in quarters over a block's waves
        const bool wide = K % 32 == 0, split = wide && max_tiles <= 128 && K >= 256;
        const bool narrow = (long)n_out * K * 2 < MOE_NARROW_BYTES;
        const dim3 grid(max_tiles, (n_out + 127) / 128);
        const dim3 line((unsigned)((((long)max_tiles * ((n_out + 511) / 512) + 63) / 64) * 64));       // whole rounds of eight tiles over eight XCDs
#define MM(TA, TO)                                                                                                                 \
    {                                                                                                                              \
        if (split && narrow) moe_linear_wide_kernel<EXT, TA, TO, 4, 2><<<dim3((n_out + 63) / 64, max_tiles), 256, 0, stream>>>((const TA*)a, a_stride, row_token, (const bf16_t*)w, plan, (TO*)out, out_stride, n_out, K, ep, max_tiles); \
        else if (split) moe_linear_wide_kernel<EXT, TA, TO, 4, 4><<<dim3((n_out + 127) / 128, max_tiles), 256, 0, stream>>>((const TA*)a, a_stride, row_token, (const bf16_t*)w, plan, (TO*)out, out_stride, n_out, K, ep, max_tiles); \
        else if (wide) moe_linear_wide_kernel<EXT, TA, TO, 1, 4><<<line, 256, 0, stream>>>((const TA*)a, a_stride, row_token, (const bf16_t*)w, plan, (TO*)out, out_stride, n_out, K, ep, max_tiles); \
        else moe_linear_mfma_kernel<EXT, TA, TO><<<grid, 256, 0, stream>>>((const TA*)a, a_stride, row_token, (const bf16_t*)w, plan, (TO*)out, out_stride, n_out, K, ep); \
    }
        if (a_dtype == LI_BF16 && out_dtype == LI_BF16) MM(bf16_t, bf16_t)
        else if (a_dtype == LI_BF16 && out_dtype == LI_F32) MM(bf16_t, float)
        else if (a_dtype == LI_F32 && out_dtype == LI_BF16) MM(float, bf16_t)
        else if (a_dtype == LI_F32 && out_dtype == LI_F32) MM(float, float)
        else return LI_ERR_DTYPE;
#undef MM
        return li_launch_status();
    }
    const dim3 grid(max_tiles, (n_out + 63) / 64);
#define ML(TA, TW, TO) moe_linear_kernel<EXT, TA, TW, TO><<<grid, 256, 0, stream>>>((const TA*)a, a_stride, row_token, (const TW*)w, plan, (TO*)out, out_stride, n_out, K, ep)
    if (a_dtype == LI_F32 && w_dtype == LI_F32 && out_dtype == LI_F32) ML(float, float, float);
    else if (a_dtype == LI_BF16 && w_dtype == LI_BF16 && out_dtype == LI_BF16) ML(bf16_t, bf16_t, bf16_t);
    else if (a_dtype == LI_BF16 && w_dtype == LI_BF16 && out_dtype == LI_F32) ML(bf16_t, bf16_t, float);
    else if (a_dtype == LI_F32 && w_dtype == LI_BF16 && out_dtype == LI_F32) ML(float, bf16_t, float);
    else if (a_dtype == LI_F32 && w_dtype == LI_BF16 && out_dtype == LI_BF16) ML(float, bf16_t, bf16_t);
    else return LI_ERR_DTYPE;
#undef ML
    return li_launch_status();
}

extern "C" int li_moe_linear(const void* a, int a_dtype, long a_stride, const int* row_token, const void* w, int w_dtype,
                             const int* plan, int max_tiles, void* out, int out_dtype, long out_stride, int n_out, int K, int act, float limit,
                             int tile_rows, int rows, const float* row_wt, hipStream_t stream) {
    const bool gated = act == 2 || act == 3;
    if (max_tiles <= 0 || n_out <= 0 || K <= 0 || a_stride < K || act < 0 || act > 4 || out_stride < (gated ? n_out / 2 : n_out) ||
        (gated && (n_out & 1)))
        return LI_ERR_SIZE;
    const MoeEpilogue ep{act, limit, row_wt};
    if (act == 4 || row_wt)
        return moe_linear_launch<true>(a, a_dtype, a_stride, row_token, w, w_dtype, plan, max_tiles, out, out_dtype, out_stride, n_out, K, ep, tile_rows, rows, stream);
    return moe_linear_launch<false>(a, a_dtype, a_stride, row_token, w, w_dtype, plan, max_tiles, out, out_dtype, out_stride, n_out, K, ep, tile_rows, rows, stream);
}

// ------------------------------------------------------------------------------- the shared expert beside the routed ones
// A decoding step's shared expert hangs on none of the router's choices, yet its two products were launches of their own behind the routed
// ones: 5 to 9 us each, in which the chip waits for a first load and a drain.  Its first product goes with the router, which is a block a token
// and leaves the chip idle, and its second with the routed experts' first: blocks of 512 threads, of which some take one and the rest the
// other.  Which form the product beside takes (see few_rows.h): up to 4 rows rows_product, up to 16 and 32 one and two tiles of rows of
// skinny_product, eight waves a block.
// Left out of a recorded step (us, 16 experts of 2,240 x 1,536, a shared one of 4,480): one token, router 8.2 and first product 4.8 apart,
// 8.0 together; routed 7.9 and shared 5.9 apart, 8.9 together; 32 tokens, router 8.8 and first product 9.2 apart, 10.9 together.  The second
// pair only for rows few enough for the kernel of few rows: in blocks of 512 threads the streaming kernel had too few of them on a
// unit (32 tokens, 23.5 and 8.2 apart, 37.1 together).
#define MOE_BESIDE_NT 512
#define MOE_BESIDE_ROWS 32
// Tokens up to which li_moe_route_beside takes a call, and rows of the routed product up to which li_moe_linear_beside does
extern "C" int li_moe_route_beside_rows() { return MOE_BESIDE_ROWS; }
extern "C" int li_moe_linear_beside_rows() { return MOE_VECTOR_ROWS; }
enum { BESIDE_ROWS = 0, BESIDE_ONE_TILE = 1, BESIDE_TWO_TILES = 2 };
template <int FORM> constexpr int beside_lds() {
    return FORM == BESIDE_ROWS ? fr_lds_bytes(2) : FORM == BESIDE_ONE_TILE ? SkinnyLds<1, 1, 8, SK_CHUNK>::BYTES : SkinnyLds<2, 1, 8, SK_CHUNK / 2>::BYTES;
}
template <int FORM, typename TO, int EPI>
__device__ __forceinline__ void beside_product(const SkinnyArgs& a, int log_rows, int block, char* lds) {
    if constexpr (FORM == BESIDE_ROWS) rows_product<TO, false, EPI, 4, true, 2>(a, log_rows, block, lds);
    else if constexpr (FORM == BESIDE_ONE_TILE) skinny_product<1, 1, 8, false, TO, false, EPI, SK_CHUNK>(a, block, lds);
    else skinny_product<2, 1, 8, false, TO, false, EPI, SK_CHUNK / 2>(a, block, lds);
}

template <int FORM>
__global__ __launch_bounds__(MOE_BESIDE_NT) void moe_route_beside_kernel(MoeRoute<bf16_t, bf16_t> r, SkinnyArgs a, int log_rows) {
    extern __shared__ __align__(16) float sm[];
    if ((int)blockIdx.x < r.T) moe_route_token<bf16_t, bf16_t, MOE_BESIDE_NT>(r, blockIdx.x, sm);
    else beside_product<FORM, bf16_t, 2>(a, log_rows, blockIdx.x - r.T, reinterpret_cast<char*>(sm));
}

template <int FORM, bool EXT>
__global__ __launch_bounds__(MOE_BESIDE_NT) void moe_linear_beside_kernel(MoeLinear<bf16_t> p, SkinnyArgs a, int log_rows, int blocks_beside, int col_blocks) {
    __shared__ __attribute__((aligned(16))) char lds[beside_lds<FORM>()];
    if ((int)blockIdx.x < blocks_beside) return beside_product<FORM, float, 0>(a, log_rows, blockIdx.x, lds);
    const int b = blockIdx.x - blocks_beside, tile = b / col_blocks, cb = b - tile * col_blocks;
    moe_linear_rows_wave<EXT, bf16_t, MR_OUT_FEW>(p, tile, (cb * (MOE_BESIDE_NT / 64) + (threadIdx.x >> 6)) * MR_OUT_FEW);
}

// The product beside: x [T, K] w [N, K]^T; the form, the columns a block takes and the blocks.  False where it takes none.
static bool beside_form(SkinnyArgs& a, const void* x, const void* w, void* out, int T, int N, int K, int& form, int& blocks, int& log_rows) {
    if (T <= 0 || T > MOE_BESIDE_ROWS || N <= 0 || K <= 0 || K % 8 || ((uintptr_t)x | (uintptr_t)w) % 16 || (uintptr_t)out % 4) return false;
    form = T <= ROWS_KERNEL_M && K % 64 == 0 ? BESIDE_ROWS : T <= 16 ? BESIDE_ONE_TILE : BESIDE_TWO_TILES;
    a = SkinnyArgs{(const bf16_t*)x, (const bf16_t*)w, nullptr, out, T, N, K, 0.f};
    a.cols = balanced_round_cols(N, 16, compute_units());
    blocks = (N + a.cols - 1) / a.cols;
    log_rows = T <= 1 ? 0 : T <= 2 ? 1 : 2;
    return true;
}

// li_moe_route for bfloat16 rows and router of up to 32 tokens, and hs[t, n] = act(sum_k x[t, k] w[n, k]) (bfloat16, act as li_linear_act's)
// in the same launch.  Returns -1, having done nothing, where it does not take the call.
extern "C" int li_moe_route_beside(const void* x, const void* wr, const float* br, const void* wg, int* idx, float* wt, float* gate, int T, int K,
                                   int E, int top, int mode, const float* corr, int groups, int keep, int* plan, int max_tiles, int* row_token,
                                   int* pair_row, int tile_rows, float* row_wt, int experts, int* count, const void* w, void* hs, int N, int act,
                                   hipStream_t stream) {
    if (plan && (T > 128 || experts <= 0 || experts > MOE_PLAN_EXPERTS || experts > E || K < 64 || max_tiles <= 0 || !row_token || !pair_row || !count ||
                 (tile_rows != MOE_TILE && tile_rows != MOE_BIG_TILE && tile_rows != MOE_HUGE_TILE)))
        return LI_ERR_SIZE;
    if (T <= 0 || K <= 0 || E <= 0 || top <= 0 || top > E || top > 64 || (wg && !gate) || mode < 0 || mode > 15 || (mode & 3) == 3 ||
        groups <= 0 || keep <= 0 || keep > groups || E % groups || (size_t)(K + 2 * E + groups + 4) * 4 > 60000)
        return LI_ERR_SIZE;
    if ((mode & 3) != 0 && (long)top > (long)keep * (E / groups)) return LI_ERR_SIZE;
    SkinnyArgs a;
    int form, blocks, log_rows;
    if (act < LI_ACT_RELU2 || act > LI_ACT_GELU_ERF || !beside_form(a, x, w, hs, T, N, K, form, blocks, log_rows)) return -1;
    a.ep = LiAct{act, 0.f, 0.f};
    const int vec = (K % 8 == 0 && ((uintptr_t)wr % 16) == 0 && (!wg || ((uintptr_t)wg % 16) == 0)) | 2;      // (K % 8 and x's alignment: beside_form)
    const MoeRoute<bf16_t, bf16_t> r{(const bf16_t*)x, K, (const bf16_t*)wr, br, (const bf16_t*)wg, idx, wt, gate, T, K, E, top, vec, mode, corr, groups, keep,
                                     MoePlanOut{plan, row_token, pair_row, row_wt, count, max_tiles, tile_rows, experts}};
    const size_t mine = (size_t)(((K + 3) & ~3) + 2 * E + groups) * 4;
#define RB(FORM)                                                                                                                  \
    {                                                                                                                             \
        const size_t his = beside_lds<FORM>(), lds = mine > his ? mine : his;                                                     \
        moe_route_beside_kernel<FORM><<<T + blocks, MOE_BESIDE_NT, lds, stream>>>(r, a, log_rows);                                \
    }
    if (form == BESIDE_ROWS) RB(BESIDE_ROWS) else if (form == BESIDE_ONE_TILE) RB(BESIDE_ONE_TILE) else RB(BESIDE_TWO_TILES)
#undef RB
    return li_launch_status();
}

// li_moe_linear for bfloat16 rows, matrices and results in tiles of MOE_TILE rows, at most MOE_VECTOR_ROWS rows, and y[t, n] = sum_k x[t, k] w2[n, k] (float32, t < T) in the
// same launch.  Returns -1, having done nothing, where it does not take the call (other forms of the routed product among it).
extern "C" int li_moe_linear_beside(const void* a, long a_stride, const int* row_token, const void* w, const int* plan, int max_tiles, void* out,
                                    long out_stride, int n_out, int K, int act, float limit, int rows, const float* row_wt, const void* x,
                                    const void* w2, float* y, int T, int N2, int K2, hipStream_t stream) {
    const bool gated = act == 2 || act == 3;
    if (max_tiles <= 0 || n_out <= 0 || K <= 0 || a_stride < K || act < 0 || act > 4 || out_stride < (gated ? n_out / 2 : n_out) || (gated && (n_out & 1)))
        return LI_ERR_SIZE;
    SkinnyArgs s;
    int form, blocks, log_rows;
    if (T > ROWS_KERNEL_M || K % 8 || a_stride % 8 || ((uintptr_t)a | (uintptr_t)w) % 16 || !beside_form(s, x, w2, y, T, N2, K2, form, blocks, log_rows)) return -1;
    if (rows > MOE_VECTOR_ROWS) return -1;
    const int block_cols = MOE_BESIDE_NT / 64 * MR_OUT_FEW, col_blocks = (n_out + block_cols - 1) / block_cols;
    const MoeLinear<bf16_t> p{(const bf16_t*)a, a_stride, row_token, (const bf16_t*)w, plan, (bf16_t*)out, out_stride, n_out, K, MoeEpilogue{act, limit, row_wt}};
    if ((long)col_blocks * max_tiles + blocks > 0x7fffffffL) return -1;
    const unsigned grid = (unsigned)(blocks + col_blocks * max_tiles);
#define LB2(FORM, EXT) moe_linear_beside_kernel<FORM, EXT><<<grid, MOE_BESIDE_NT, 0, stream>>>(p, s, log_rows, blocks, col_blocks)
#define LB(FORM) { if (act == 4 || row_wt) LB2(FORM, true); else LB2(FORM, false); }
    if (form == BESIDE_ROWS) LB(BESIDE_ROWS) else LB(BESIDE_ONE_TILE)       // (so few rows: at most 4 tokens)
#undef LB
#undef LB2
    return li_launch_status();
}

// ----------------------------------------------------------------------------------------------- the sum
// x[t, :] += factor * (the sum of what follows); with a tanh norm behind it (xn given), xn[t, :] = tanh(alpha * x[t, :]) *
// gamma + beta of the new x.  The sum: sum_c wt[t, c] (wt null: 1) * yrow[pair_row[t * top + c], :] (in the order of c) + gate[t] * shared[t, :].  A choice
// idx[t, c] >= experts (where `ident` is given) is an IDENTITY expert: its output is the token's input row ident[t, :].
template <typename TI, bool NORM>
__global__ __launch_bounds__(256) void moe_combine_kernel(float* __restrict__ x, long x_stride, const float* __restrict__ yrows,
                                                          long y_stride, const int* __restrict__ pair_row, const float* __restrict__ wt,
                                                          const float* __restrict__ gate, const float* __restrict__ shared_out,
                                                          long s_stride, int H, int top, const int* __restrict__ idx, int experts,
                                                          const TI* __restrict__ ident, long i_stride, float factor,
                                                          float alpha, const float* __restrict__ gamma, const float* __restrict__ beta,
                                                          void* __restrict__ xn, int xn_bf16) {
    const int t = blockIdx.x;
    for (int j = blockIdx.y * 256 + threadIdx.x; j < H; j += gridDim.y * 256) {
        float s = 0.f;
        for (int c = 0; c < top; ++c) {
            const int row = pair_row[(size_t)t * top + c];
            if (row >= 0) s = fmaf(wt ? wt[(size_t)t * top + c] : 1.0f, yrows[(size_t)row * y_stride + j], s);
            else if (ident && idx[(size_t)t * top + c] >= experts)
                s = fmaf(wt ? wt[(size_t)t * top + c] : 1.0f, load_as_float(ident + (size_t)t * i_stride + j), s);
        }
        if (shared_out) s = fmaf(gate ? gate[t] : 1.f, shared_out[(size_t)t * s_stride + j], s);
        const float v = fmaf(factor, s, x[(size_t)t * x_stride + j]);
        x[(size_t)t * x_stride + j] = v;
        if constexpr (NORM) {
            const float r = fmaf(tanhf(alpha * v), gamma[j], beta[j]);
            if (xn_bf16) reinterpret_cast<bf16_t*>(xn)[(size_t)t * H + j].bits = float_to_bf16(r);
            else reinterpret_cast<float*>(xn)[(size_t)t * H + j] = r;
        }
    }
}

extern "C" int li_moe_combine(float* x, long x_stride, const float* yrows, long y_stride, const int* pair_row, const float* wt,
                              const float* gate, const float* shared_out, long s_stride, int T, int H, int top,
                              const int* idx, int experts, const void* ident, int ident_dtype, long i_stride, float factor,
                              float alpha, const float* gamma, const float* beta, void* xn, int xn_dtype, hipStream_t stream) {
    if (T <= 0 || H <= 0 || top <= 0 || x_stride < H || y_stride < H || (shared_out && s_stride < H) ||
        (ident && (!idx || i_stride < H || experts < 0)) || (xn && (!gamma || !beta)))
        return LI_ERR_SIZE;
    int ys = (H + 255) / 256;
    if (ys > 64) ys = 64;
#define MC(TI, NORM)                                                                                                              \
    moe_combine_kernel<TI, NORM><<<dim3(T, ys), 256, 0, stream>>>(x, x_stride, yrows, y_stride, pair_row, wt, gate, shared_out,    \
                                                                  s_stride, H, top, idx, experts, (const TI*)ident, i_stride, factor, \
                                                                  alpha, gamma, beta, xn, xn_dtype == LI_BF16)
    if (ident && ident_dtype == LI_BF16) { if (xn) MC(bf16_t, true); else MC(bf16_t, false); }
    else if (!ident || ident_dtype == LI_F32) { if (xn) MC(float, true); else MC(float, false); }
    else return LI_ERR_DTYPE;
#undef MC
    return li_launch_status();
}

// The same for few tokens, with the RMS norms on its two sides: with w1, the sum's own norm b / sqrt(mean(b^2) + eps1) * w1 joins x; with xn,
// the row that x's next reader takes is left there: the norm of the new x with w2 and eps2 or, without w2, the new x itself.  One block a
// token, its row in registers.  Bound by trips to memory one behind the other and by launches: the choices are read a lane each and
// everything that hangs on none of them is asked for with them, so there are two trips (a trip a choice, the norms' weights behind their
// sums: 7.0 us, now 4.9).  One token of 1,536: sum and norm 3.8 + 3.3 us and the gap between them, now 4.9 in all (an answer of
// a model with such layers 11.83 -> 11.74 ms); 8 tokens with w1, the branch cleared, the sum and the norms 4.6 + 4.7 + 4.7 us, now 6.2 (an
// answer 14.33 -> 14.15).  From 256 tokens on the sum alone is spread over more blocks than one a row and the norms read their rows with
// 16 bytes a lane; the launches are then the smaller part.
#define MOE_NORM_NT 1024
#define MOE_NORM_COLUMNS 4          // of a thread: rows of up to 4,096
#define MOE_NORM_CHOICES 8          // rows asked for at a time
#define MOE_NORM_MAX_TOKENS 255

extern "C" int li_moe_combine_norm_takes(int T, int H) { return T > 0 && T <= MOE_NORM_MAX_TOKENS && H > 0 && H <= MOE_NORM_NT * MOE_NORM_COLUMNS; }

template <typename TI, typename TO>
__global__ __launch_bounds__(MOE_NORM_NT) void moe_combine_norm_kernel(
    float* x, const float* __restrict__ yrows, long y_stride, const int* __restrict__ pair_row, const float* __restrict__ wt,
    const float* __restrict__ gate, const float* __restrict__ shared_out, long s_stride, int H, int top, const int* __restrict__ idx, int experts,
    const TI* ident, long i_stride, float factor, const float* __restrict__ w1, float eps1, const float* __restrict__ w2, float eps2, TO* xn) {
    __shared__ float red[MOE_NORM_NT / LI_WAVE];
    const int t = blockIdx.x;
    float* xr = x + (size_t)t * H;                     // (x, ident and xn may be one tensor's rows: a thread has read its columns before it writes them)
    float v[MOE_NORM_COLUMNS] = {}, was[MOE_NORM_COLUMNS], sh[MOE_NORM_COLUMNS] = {}, g1[MOE_NORM_COLUMNS] = {}, g2[MOE_NORM_COLUMNS] = {}, own[MOE_NORM_COLUMNS] = {};
    const float g = shared_out && gate ? gate[t] : 1.f;
    // (a thread's columns beyond the row read its last one again, and add nothing; whole turns beyond it are left out)
#define MOE_COLUMN(i) const int j = threadIdx.x + i * MOE_NORM_NT, jj = j < H ? j : H - 1; if (i * MOE_NORM_NT >= H) continue
    const int lane = threadIdx.x & (LI_WAVE - 1);
    int my_row = -1;
    float my_f = 0.f;
    for (int c0 = 0; c0 < top; c0 += MOE_NORM_CHOICES) {
        if (c0 % LI_WAVE == 0) {                       // the next 64 choices, a lane each: one trip to memory, not one a choice
            const int c = c0 + lane < top ? c0 + lane : top - 1;
            const size_t p = (size_t)t * top + c;
            my_row = pair_row[p];
            const int choice = (ident ? idx : pair_row)[p];
            my_f = (wt ? wt : yrows)[wt ? p : 0];
            if (c0 == 0) {                             // what hangs on no choice is asked for before the first rows are waited for
#pragma unroll
                for (int i = 0; i < MOE_NORM_COLUMNS; ++i) {
                    MOE_COLUMN(i);
                    was[i] = xr[jj];
                    if (shared_out) sh[i] = shared_out[(size_t)t * s_stride + jj];
                    if (ident) own[i] = load_as_float(ident + (size_t)t * i_stride + jj);
                    if (w1) g1[i] = w1[jj];
                    if (w2) g2[i] = w2[jj];
                }
            }
            if (!wt) my_f = 1.f;
            if (my_row < 0) my_row = ident && choice >= experts ? -2 : -1;       // -2: an identity expert, the token's input row
            if (c0 + lane >= top) my_row = -1;
        }
        int row[MOE_NORM_CHOICES];
        float f[MOE_NORM_CHOICES], y[MOE_NORM_COLUMNS][MOE_NORM_CHOICES];
#pragma unroll
        for (int c = 0; c < MOE_NORM_CHOICES; ++c) {
            row[c] = __builtin_amdgcn_readlane(my_row, (c0 + c) % LI_WAVE);
            f[c] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(my_f), (c0 + c) % LI_WAVE));
        }
#pragma unroll
        for (int i = 0; i < MOE_NORM_COLUMNS; ++i) {
            MOE_COLUMN(i);
#pragma unroll
            for (int c = 0; c < MOE_NORM_CHOICES; ++c) y[i][c] = yrows[(size_t)(row[c] < 0 ? 0 : row[c]) * y_stride + jj];
        }
#pragma unroll
        for (int i = 0; i < MOE_NORM_COLUMNS; ++i) {
            if (i * MOE_NORM_NT >= H) continue;
#pragma unroll
            for (int c = 0; c < MOE_NORM_CHOICES; ++c)
                if (row[c] != -1) v[i] = fmaf(f[c], row[c] == -2 ? own[i] : y[i][c], v[i]);
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < MOE_NORM_COLUMNS; ++i) {
        MOE_COLUMN(i);
        if (shared_out) v[i] = fmaf(g, sh[i], v[i]);
        if (j < H) ss += v[i] * v[i];
    }
    float inv = 1.f;
    if (w1) inv = 1.0f / sqrtf(block_sum<MOE_NORM_NT>(ss, red) / (float)H + eps1);
    float s2 = 0.f;
#pragma unroll
    for (int i = 0; i < MOE_NORM_COLUMNS; ++i) {
        MOE_COLUMN(i);
        v[i] = w1 ? was[i] + v[i] * inv * g1[i] : fmaf(factor, v[i], was[i]);
        if (j >= H) continue;
        xr[j] = v[i];
        s2 += v[i] * v[i];
    }
    if (!xn) return;
    float inv2 = 1.f;
    if (w2) inv2 = 1.0f / sqrtf(block_sum<MOE_NORM_NT>(s2, red) / (float)H + eps2);
#pragma unroll
    for (int i = 0; i < MOE_NORM_COLUMNS; ++i) {
        MOE_COLUMN(i);
        if (j < H) store_from_float(xn + (size_t)t * H + j, w2 ? v[i] * inv2 * g2[i] : v[i]);
    }
#undef MOE_COLUMN
}

extern "C" int li_moe_combine_norm(float* x, const float* yrows, long y_stride, const int* pair_row, const float* wt, const float* gate,
                                   const float* shared_out, long s_stride, int T, int H, int top, const int* idx, int experts, const void* ident,
                                   int ident_dtype, long i_stride, float factor, const float* w1, float eps1, const float* w2, float eps2,
                                   void* xn, int xn_dtype, hipStream_t stream) {
    if (!li_moe_combine_norm_takes(T, H) || top <= 0 || y_stride < H || (shared_out && s_stride < H) ||
        (ident && (!idx || i_stride < H || experts < 0)) || (w2 && !xn) || (w1 && factor != 1.0f))
        return LI_ERR_SIZE;
#define MC(TI, TO)                                                                                                                    \
    moe_combine_norm_kernel<TI, TO><<<T, MOE_NORM_NT, 0, stream>>>(x, yrows, y_stride, pair_row, wt, gate, shared_out, s_stride, H, top, \
                                                                   idx, experts, (const TI*)ident, i_stride, factor, w1, eps1, w2, eps2, (TO*)xn)
    const bool ib = ident && ident_dtype == LI_BF16, ob = xn && xn_dtype == LI_BF16;
    if ((ident && !ib && ident_dtype != LI_F32) || (xn && !ob && xn_dtype != LI_F32)) return LI_ERR_DTYPE;
    if (ib) { if (ob) MC(bf16_t, bf16_t); else MC(bf16_t, float); }
    else { if (ob) MC(float, bf16_t); else MC(float, float); }
#undef MC
    return li_launch_status();
}
