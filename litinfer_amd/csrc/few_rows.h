// Products of few rows (a decoding step) in bfloat16, as device functions: gemm.hip launches them by themselves, other kernels take them beside
// work of their own.
#pragma once
#include "common.h"
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

template <typename TO>
__device__ __forceinline__ void epilogue_store(TO* out, size_t idx, float acc, const float* bias,
                                               int col, float accumulate) {
    if (bias) acc += bias[col];
    if (accumulate != 0.f) acc = fmaf(accumulate, acc, load_as_float(out + idx));
    store_from_float(out + idx, acc);
}

// up * gate / (1 + exp(-gate)) for a result that is rounded to bfloat16: the exponential and the reciprocal are
// the instructions' own (v_exp_f32, v_rcp_f32: an ulp each), 5 instructions where expf and the division are some
// 25; a tile of 256 x 256 makes 128 of them a thread, 7 % of the tile's time.  (A gate far below zero: the
// exponential overflows to infinity, the reciprocal is 0 and so is the result, as it should be.)  The 32-bit
// path keeps expf and the division.
__device__ __forceinline__ float swiglu_bf16(float gate, float up) {
    const float e = __builtin_amdgcn_exp2f(-1.44269504088896341f * gate);
    return up * (gate * __builtin_amdgcn_rcpf(1.0f + e));
}

// ACT: 0, or the other forms: LI_ACT_GELU_TANH, the gate through GELU in its tanh form; LI_ACT_CLAMPED with the limit a0:
// g = min(gate, a0), u = clamp(up, -a0, a0), g sigmoid(1.702 g) (u + 1); ACT_TOLD, the one of them that `ep` says.  The tiles
// have an instance each: with both forms' code in one kernel, 2,048 rows of 8,960 clamped outputs took 129.8 us instead of
// 125.7, 64 rows of 18,944 54.1 instead of 52.7.  The kernel of few rows, bound by its loads, has one for both.
#define ACT_TOLD (-1)
template <int ACT>
__device__ __forceinline__ float gated_bf16(float gate, float up, const LiAct& ep) {
    if constexpr (ACT == 0) return swiglu_bf16(gate, up);
    if constexpr (ACT == LI_ACT_GELU_TANH) return up * gelu_tanh_bf16(gate);
    if constexpr (ACT == ACT_TOLD) {
        if (ep.act == LI_ACT_GELU_TANH) return up * gelu_tanh_bf16(gate);
    }
    const float g = fminf(gate, ep.a0), u = fminf(fmaxf(up, -ep.a0), ep.a0);
    const float e = __builtin_amdgcn_exp2f(-1.702f * 1.44269504088896341f * g);
    return (u + 1.0f) * (g * __builtin_amdgcn_rcpf(1.0f + e));
}

// ------------------------------------------------- bfloat16, few rows (decode)
// With M <= 64 the product is bound by streaming W once from HBM, and the
// bandwidth reached is (bytes in flight) / (memory latency): the kernel is
// built to keep many independent 16-byte loads outstanding.  A block owns NT
// tiles of 16 rows of W (16 output columns each); its WAVES waves split K
// between them in chunks of 128 and add their partial sums through LDS in wave
// order.  The loads of a wave's next chunk are in flight while one chunk is
// multiplied.  Per chunk a lane loads four 16-byte pieces of one row of W per
// tile (the four lanes of a row together 64 contiguous bytes an instruction)
// and the matching pieces of x;
// v_mfma_f32_16x16x32_bf16 takes W as the row operand and x as the column
// operand (lane l: row/column l % 16, 8 k-values of k-group l / 16; any
// assignment of real k to (k-group, slot) is right as long as both operands
// share it).  The result's register r of lane l is row 4 * (l / 16) + r (an
// output column n), column l % 16 (an x row m).
//
// SWIGLU: W is [gate; up] with N rows each: tile 0 takes gate rows, tile 1 the
// up rows of the same columns, and out[m, n] = up * gate / (1 + exp(-gate)).
//
// ROPE (one tile of rows and of columns): W is the packed [q; k; v] projection.  A block takes,
// of one head, the 8 columns 8 i .. and their partners of the half-split rotation, dh / 2
// further on, so that lane l and lane l ^ 32 hold the two members of a pair; the epilogue adds
// the bias, rotates query and key heads by the row's angles (float32 tables), writes the
// queries to out and keys and values straight into their page slots (and to out as well).
#define SK_CHUNK 128
#define SK_MAX_PARTS 512            // blocks of a producing product whose sums one consumer adds up

struct SkinnyArgs {
    const bf16_t* x;        // [M, K]
    const bf16_t* w;        // [N, K], or [2 N, K] with SWIGLU
    const float* bias;      // [N] or null
    void* out;              // [M, N]
    int M, N, K;
    float accumulate;       // 0: out is written; else out += accumulate * (product + bias)
    // ROPE (the packed q/k/v projection of a decoding step): rotary tables [M, dh / 2], the page
    // slot of each row, the cache layer's keys and values [pages, nkv, page_size, dh]
    const float* cos;
    const float* sin;
    const int* slot_map;
    bf16_t* kc;
    bf16_t* vc;
    int nh, nkv, dh, page_size, num_pages;
    // An RMS norm between two products of up to 32 rows, without a pass of its own.  The product
    // BEFORE it (float out with accumulate: the residual sum) also writes xg[m, n] = bf16(gamma[n] *
    // out[m, n]) and, per block, the sums of squares of its columns of out to sq_parts[block * R + m],
    // R = 16 up to 16 rows and 32 above.
    const float* gamma;
    bf16_t* xg;
    float* sq_parts;
    // The product AFTER it takes such an xg as its x and scales row m's sums by
    // 1 / sqrt(sum_p row_parts[p * R + m] / K + eps): the factor of a row does not depend on k.
    const float* row_parts;
    int nparts;
    float eps;
    // Columns a block takes (with ROPE: rotation pairs a block takes); 0: as many as its tiles hold.
    // Fewer than the tiles hold where that spreads a matrix of few columns evenly over the compute units.
    int cols;
    // A tanh norm behind the sum (EPI 1 of the kernel): xg[m, n] = bf16(tanh(alpha * out[m, n]) * gamma[n] + beta[n]).  It takes
    // no statistics of a row, so it is done here and sq_parts stays as it is.
    const float* beta;
    float alpha;
    // SWIGLU with EPI 1: one of the other gated forms (see gated_bf16).  EPI 2 (bfloat16 out): out = activation(product + bias)
    LiAct ep;
    unsigned half_magic;    // with ROPE: see skinny_head
};

// The head that rotation pair p belongs to: p / (dh / 2) by a product with 2^32 / (dh / 2) rounded up (exact below 2^32 / (dh / 2) pairs)
__device__ __forceinline__ int skinny_head(const SkinnyArgs& a, int p) { return (int)__umulhi((unsigned)p, a.half_magic); }

// Rows that the shares of the sums of squares are kept for, a block and a step: 16 up to 16 rows, else 32 (the products on both sides of a
// norm see the same M, up to 32; with more rows nobody asks)
template <int MT> constexpr int SKINNY_PLACES = MT <= 1 ? 16 : 32;

// All of a kernel's arguments in one trip to memory: asked for where they are used they are two or three, one behind the other (0.1 to
// 0.5 us of a launch whose matrix takes 1 to 3).
template <bool ROPE>
__device__ __forceinline__ void skinny_arguments(const SkinnyArgs& a) {
    asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.out), "s"(a.bias), "s"(a.M), "s"(a.N), "s"(a.K), "s"(a.cols), "s"(a.row_parts), "s"(a.nparts), "s"(a.accumulate));
    if constexpr (ROPE) asm volatile("" ::"s"(a.cos), "s"(a.sin), "s"(a.slot_map), "s"(a.kc), "s"(a.vc), "s"(a.nh), "s"(a.nkv), "s"(a.dh), "s"(a.half_magic));
    else asm volatile("" ::"s"(a.gamma), "s"(a.xg), "s"(a.sq_parts));
}

// The rows' sums of squares from the shares that the blocks of the product before the norm left.  Thread t asks for four rows (a quad) of
// parts t / quads, t / quads + G, ..; the loads are conditional on the wave's own count only, into registers that nothing else writes (a
// share set to zero first made the compiler wait for the first load before it issued the second).
template <int RP, int WAVES>
struct RowShares {
    static constexpr int QUADS = RP / 4, G = WAVES * 64 / QUADS, PER = SK_MAX_PARTS / G;
    floatx4 v[PER];
    __device__ __forceinline__ void ask(const float* parts, int nparts) {
        const int q = threadIdx.x / QUADS, r = 4 * (threadIdx.x % QUADS);
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (i * G < nparts) {
                const int p = q + i * G;
                v[i] = *reinterpret_cast<const floatx4*>(parts + (size_t)(p < nparts ? p : nparts - 1) * RP + r);
            }
    }
    // each wave's sum of every row to sums[wave][row]
    __device__ __forceinline__ void add(int nparts, float (*sums)[RP]) {
        const int q = threadIdx.x / QUADS, lane = threadIdx.x & 63;
        floatx4 mine = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (q + i * G < nparts) mine += v[i];
#pragma unroll
        for (int o = QUADS; o < 64; o <<= 1)
#pragma unroll
            for (int e = 0; e < 4; ++e) mine[e] = lane_xor_add(mine[e], o);
        if (lane < QUADS) *reinterpret_cast<floatx4*>(&sums[threadIdx.x >> 6][4 * lane]) = mine;
    }
};

// What the epilogue adds to or multiplies with the sums (bias, the residual sum, a norm's weights, the rotation's cosines and sines, the
// page slot), asked for by the wave that will write the results (wave mt row tile mt: thread t of the epilogue is lane t % 64 of wave
// t / 64) before it has them to add: the epilogue waits for no memory.  Never conditional per lane: a place past the end reads the last one.
template <bool SWIGLU, int EPI> constexpr bool SKINNY_PRE = !SWIGLU && EPI != 2;
template <int NT> struct SkinnyPre { float bias[NT][4], res[NT][4], gamma[NT][4], beta[NT][4], cos[NT][4], sin[NT][4]; int slot; };

template <int NT, typename TO, bool ROPE, int EPI>
__device__ __forceinline__ void skinny_ask(const SkinnyArgs& a, SkinnyPre<NT>& pre, int n0, int nend, int mt, int lane) {
    const int m = 16 * mt + (lane & 15) < a.M ? 16 * mt + (lane & 15) : a.M - 1;
    if constexpr (ROPE) {
        const bool second = (lane >> 4) >= 2;
        const int half = a.dh / 2;
        pre.slot = a.slot_map[m];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int p = n0 + 8 * nt + 4 * ((lane >> 4) & 1) + r;
                p = p < nend ? p : nend - 1;
                const int head = skinny_head(a, p), j = p - head * half;
                pre.bias[nt][r] = a.bias ? a.bias[head * a.dh + (second ? half + j : j)] : 0.f;
                pre.cos[nt][r] = a.cos[(size_t)m * half + j];
                pre.sin[nt][r] = a.sin[(size_t)m * half + j];
            }
    } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int n = n0 + 16 * nt + 4 * (lane >> 4) + r;
                const int nc = n < nend ? n : nend - 1;
                pre.bias[nt][r] = a.bias ? a.bias[nc] : 0.f;
                pre.gamma[nt][r] = a.gamma ? a.gamma[nc] : 0.f;
                if constexpr (EPI == 1) pre.beta[nt][r] = a.beta[nc];
                if constexpr (sizeof(TO) == 4)
                    pre.res[nt][r] = a.accumulate != 0.f ? reinterpret_cast<const float*>(a.out)[(size_t)m * a.N + nc] : 0.f;
                else pre.res[nt][r] = 0.f;
            }
    }
}

// The waves' sums (red[wave][row tile, column tile][lane], as the MFMAs leave them) added in wave order, and what follows; row_squares(m):
// the sum of row m's squares where the rows are those of li_linear_residual_norm.
template <int MT, int NT, int WAVES, bool SWIGLU, typename TO, bool ROPE, int EPI, typename RowSquares>
__device__ __forceinline__ void skinny_finish(const SkinnyArgs& a, floatx4 (*red)[MT * NT][64], const SkinnyPre<NT>& pre, int n0, int nend, int block, RowSquares row_squares) {
    constexpr int RP = SKINNY_PLACES<MT>;
    const int M = a.M, N = a.N, half = a.dh / 2;
    TO* out = (TO*)a.out;
    // What skinny_ask asked for is there.  Said once: else the compiler waits for it before each result that it enters, and such a wait, by the
    // count of the wave's loads AND stores, is for the result stored just before (24 rows of 6,144 x 512 with a norm's shares 5.8 us, 5.0 without).
    if constexpr (SKINNY_PRE<SWIGLU, EPI>) __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0)
    if constexpr (EPI == 2 && !SWIGLU) {
        // one value a thread at a time, by all waves: an activation is tens of instructions a value, and by the one wave that
        // writes a row tile elsewhere its values would go through them one after the other
        for (int v = threadIdx.x; v < MT * NT * 256; v += WAVES * 64) {
            const int tile = v >> 8, l = (v >> 2) & 63, r = v & 3;
            const int m = 16 * (tile / NT) + (l & 15), n = n0 + 16 * (tile % NT) + 4 * (l >> 4) + r;
            if (m >= M || n >= nend) continue;
            float s = red[0][tile][l][r];
#pragma unroll
            for (int wv = 1; wv < WAVES; ++wv) s += red[wv][tile][l][r];
            if (a.bias) s += a.bias[n];
            store_from_float(out + (size_t)m * N + n, activation(s, a.ep));
        }
        return;
    }
    for (int t = threadIdx.x; t < MT * 64; t += WAVES * 64) {
        const int mt = t >> 6, l = t & 63;
        const int m = 16 * mt + (l & 15);
        if (m >= M) continue;                       // (with ROPE lanes l and l ^ 32 share m: both stay or both go)
        floatx4 s[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            s[nt] = red[0][mt * NT + nt][l];
#pragma unroll
            for (int wv = 1; wv < WAVES; ++wv) {
                const floatx4 o = red[wv][mt * NT + nt][l];
                s[nt][0] += o[0]; s[nt][1] += o[1]; s[nt][2] += o[2]; s[nt][3] += o[3];
            }
        }
        if ((SWIGLU || ROPE) && a.row_parts) {
            const float inv = 1.0f / sqrtf(row_squares(m) / (float)a.K + a.eps);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) { s[nt][0] *= inv; s[nt][1] *= inv; s[nt][2] *= inv; s[nt][3] *= inv; }
        }
        if constexpr (ROPE) {
            const int dh = a.dh;
            const bool second = (l >> 4) >= 2;                       // this lane holds the pairs' second members
            const int slot = pre.slot;                               // (thread t is lane l of wave mt, which asked for these: skinny_ask)
            const int page = slot / a.page_size, in_page = slot - page * a.page_size;
            const bool page_ok = page >= 0 && page < a.num_pages;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int p = n0 + 8 * nt + 4 * ((l >> 4) & 1) + r;  // the pair's number among all heads' pairs
                    float own = s[nt][r] + pre.bias[nt][r];
                    const float other = __shfl_xor(own, 32, 64);
                    if (p >= nend) continue;                         // (lanes l and l ^ 32 share p: the exchange above is done by both)
                    const int head = skinny_head(a, p), j = p - head * half;
                    const int d = second ? half + j : j;
                    const int col = head * dh + d;
                    float v = own;
                    if (head < a.nh + a.nkv) {
                        const float c = pre.cos[nt][r], sn = pre.sin[nt][r];
                        v = second ? own * c + other * sn : own * c - other * sn;
                    }
                    const uint16_t bits = float_to_bf16(v);
                    reinterpret_cast<bf16_t*>(out)[(size_t)m * N + col].bits = bits;
                    if (head >= a.nh && page_ok) {
                        const bool is_k = head < a.nh + a.nkv;
                        const int kvh = is_k ? head - a.nh : head - a.nh - a.nkv;
                        bf16_t* dst = (is_k ? a.kc : a.vc) + (((size_t)page * a.nkv + kvh) * a.page_size + in_page) * dh + d;
                        dst->bits = bits;
                    }
                }
        } else if constexpr (SWIGLU) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int n = n0 + 4 * (l >> 4) + r;
                if (n < nend) {
                    const float gv = s[0][r], uv = s[NT - 1][r];
                    store_from_float(out + (size_t)m * N + n, gated_bf16<EPI == 1 ? ACT_TOLD : 0>(gv, uv, a.ep));
                }
            }
        } else {
            [[maybe_unused]] const float factor = a.accumulate != 0.f ? a.accumulate : 1.0f;
            if constexpr (sizeof(TO) == 4) {
                if (a.xg) {                          // the sum goes out three ways (see SkinnyArgs)
                    float sq = 0.f;
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int n = n0 + 16 * nt + 4 * (l >> 4) + r;
                            if (n < nend) {
                                const size_t idx = (size_t)m * N + n;
                                const float v = fmaf(factor, s[nt][r] + pre.bias[nt][r], pre.res[nt][r]);
                                reinterpret_cast<float*>(out)[idx] = v;
                                a.xg[idx].bits = float_to_bf16(EPI == 1 ? fmaf(tanhf(a.alpha * v), pre.gamma[nt][r], pre.beta[nt][r])
                                                                        : pre.gamma[nt][r] * v);
                                sq += v * v;
                            }
                        }
                    if constexpr (EPI == 1) continue;      // (nobody asks for sums of squares)
                    // the four lanes of a row (l, l ^ 16, l ^ 32, l ^ 48: all of them are here, or none)
                    sq += __shfl_xor(sq, 16, 64);
                    sq += __shfl_xor(sq, 32, 64);
                    if ((l >> 4) == 0) a.sq_parts[(size_t)block * RP + m] = sq;
                    continue;
                }
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = n0 + 16 * nt + 4 * (l >> 4) + r;
                    if (n >= nend) continue;
                    if constexpr (SKINNY_PRE<SWIGLU, EPI>) store_from_float(out + (size_t)m * N + n, fmaf(factor, s[nt][r] + pre.bias[nt][r], pre.res[nt][r]));
                    else epilogue_store(out, (size_t)m * N + n, s[nt][r], a.bias, n, a.accumulate);
                }
        }
    }
}

// EPI 1: with SWIGLU the other gated activations, else (float out) the tanh norm of the new sum beside it (SkinnyArgs: beta).
// EPI 2: an activation of the sums (SkinnyArgs: ep).
// CH: k-values a chunk; with three or four tiles of rows half as many, so that two chunks of x still fit the registers.
template <int MT, int NT, int WAVES, int CH>
struct SkinnyLds {
    // x by wave, and the waves' sums, which with half chunks take the same place behind the loop; the rows' shares of squares
    static constexpr int XS = MT * 16 * CH, XS_BYTES = WAVES * XS * 2, RED_BYTES = WAVES * MT * NT * 64 * 16;
    static constexpr bool SAME_PLACE = CH < SK_CHUNK;
    static constexpr int XS_AT = SAME_PLACE ? 0 : RED_BYTES;
    static constexpr int SUMS_AT = SAME_PLACE ? (XS_BYTES > RED_BYTES ? XS_BYTES : RED_BYTES) : RED_BYTES + XS_BYTES;
    static constexpr int BYTES = SUMS_AT + WAVES * 64 * 4;
};

template <int MT, int NT, int WAVES, bool SWIGLU, typename TO, bool ROPE, int EPI, int CH>
__device__ __forceinline__ void skinny_product(const SkinnyArgs& a, const int block, char* lds) {
    static_assert(!(ROPE && SWIGLU) && MT <= 4, "up to four tiles of rows");
    static_assert(MT <= WAVES, "wave mt writes the results of row tile mt");
    using L = SkinnyLds<MT, NT, WAVES, CH>;
    constexpr int XS = L::XS;
    constexpr bool SAME_PLACE = L::SAME_PLACE;
    floatx4 (*red)[MT * NT][64] = reinterpret_cast<floatx4 (*)[MT * NT][64]>(lds);
    float* part_sums = reinterpret_cast<float*>(lds + L::SUMS_AT);       // [group of threads][row]: the rows' sums of squares, a share a group
    constexpr int RP = SKINNY_PLACES<MT>;
    skinny_arguments<ROPE>(a);
    const int M = a.M, N = a.N, K = a.K;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // (the same for a wave's lanes: its branches are scalar)
    const int g = lane >> 4, r16 = lane & 15;
    const int per_block = a.cols > 0 ? a.cols : (ROPE ? 8 : 16) * (SWIGLU ? 1 : NT);
    const int n0 = block * per_block;                  // first column (with ROPE: first pair) of this block
    const int half = a.dh / 2;
    const int total = ROPE ? (a.nh + 2 * a.nkv) * half : N;
    const int nend = n0 + per_block < total ? n0 + per_block : total;     // one past its last
    const bf16_t* wrow[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        int row;
        if (SWIGLU) row = ((n0 + r16 < nend) ? n0 + r16 : nend - 1) + nt * N;      // gate row, up row
        else if (ROPE) {                                    // rows 0..7 of a tile: first members of 8 pairs, 8..15: their partners
            int p = n0 + 8 * nt + (r16 & 7);
            p = p < nend ? p : nend - 1;
            const int head = skinny_head(a, p);
            row = head * a.dh + p - head * half + (r16 < 8 ? 0 : half);
        } else row = (n0 + 16 * nt + r16 < nend) ? n0 + 16 * nt + r16 : nend - 1;    // rows past the end repeat the last
        wrow[nt] = a.w + (size_t)row * K;
    }
    // x is read with whole rows of a chunk contiguous over 16 (8) lanes (lane l: row l / 16 + 4 i,
    // piece l % 16), which costs the load path a quarter of what reading it in the MFMA's
    // operand order would, and is turned into that order through a piece of LDS of the wave's own.
    constexpr int XP = CH / 8, XROWS = 64 / XP;     // 16-byte pieces of a row's chunk; rows a load of the wave covers
    constexpr int XR = MT * 16 / XROWS;             // 16-byte pieces of x per lane and chunk
    constexpr int WJ = CH / 32;                     // ... and of a tile of w
    uint16_t* xs = reinterpret_cast<uint16_t*>(lds + L::XS_AT) + wave * XS;
    const int xl_row = lane / XP, xl_piece = lane % XP;
    // piece p of row r lies at position p ^ (r % 16) (r % 8): the 16 rows a fragment read touches fall
    // into different positions, so into all banks
    auto xslot = [](int row, int piece) { return row * CH + ((piece ^ (row & (XP - 1))) << 3); };
    floatx4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = floatx4{0.f, 0.f, 0.f, 0.f};
    const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    const int nchunks = (K + CH - 1) / CH;
    const int nfull = K / CH;                          // whole chunks

    SkinnyPre<NT> pre;
    if (SKINNY_PRE<SWIGLU, EPI> && wave < MT) skinny_ask<NT, TO, ROPE, EPI>(a, pre, n0, nend, wave, lane);

    // The memory counter of a wave retires loads in the order they were issued, so waiting for
    // a chunk's x pieces also waits for every load issued before them.  All loads of a chunk (W
    // and x) are therefore issued together, one chunk ahead of their use: when chunk c is
    // multiplied, exactly the loads of chunk c + WAVES are still in flight.
    bf16x8 wbuf[2][NT][WJ], xbuf[2][XR];
    // No load of a whole chunk is conditional, and none is replaced by zeros: a load under a branch makes the
    // compiler wait for every load in flight at the next use of any (found in this kernel's code: s_waitcnt
    // vmcnt(0) before each multiplication, right behind the loads of the chunk after it, so that nothing was in
    // flight while a wave multiplied), and a value chosen between what was loaded and zero is waited for at once.
    // A row of x past the last is read from the last row (its sums are not written).  Only the last chunk of a K
    // that is no multiple of the chunk has k-values to leave out: it is taken by itself, behind the loop (TAIL).
    auto load_chunk = [&](int c, bf16x8 (*wd)[WJ], bf16x8* xd, auto tail_tag) {
        constexpr bool TAIL = decltype(tail_tag)::value;
        const int kb = c * CH;
#pragma unroll
        for (int i = 0; i < XR; ++i) {
            const int m = xl_row + XROWS * i, kk = kb + 8 * xl_piece;
            const bf16_t* row = a.x + (size_t)(m < M ? m : M - 1) * K;
            if constexpr (TAIL) xd[i] = kk < K ? *reinterpret_cast<const bf16x8*>(row + kk) : zero;
            else xd[i] = *reinterpret_cast<const bf16x8*>(row + kk);
        }
#pragma unroll
        for (int j = 0; j < WJ; ++j) {
            const int kk = kb + 8 * g + 32 * j;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if constexpr (TAIL) wd[nt][j] = kk < K ? *reinterpret_cast<const bf16x8*>(wrow[nt] + kk) : zero;
                else wd[nt][j] = *reinterpret_cast<const bf16x8*>(wrow[nt] + kk);
            }
        }
    };
    auto multiply = [&](bf16x8 (*wa)[WJ], bf16x8* xd) {
        __builtin_amdgcn_wave_barrier();            // a wave's LDS operations run in order; keep the compiler's too
#pragma unroll
        for (int i = 0; i < XR; ++i)
            *reinterpret_cast<bf16x8*>(&xs[xslot(xl_row + XROWS * i, xl_piece)]) = xd[i];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            bf16x8 xa[WJ];
#pragma unroll
            for (int j = 0; j < WJ; ++j) xa[j] = *reinterpret_cast<const bf16x8*>(&xs[xslot(16 * mt + r16, g + 4 * j)]);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int j = 0; j < WJ; ++j)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[nt][j], xa[j], acc[mt][nt], 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();
    };
    if (wave < nfull) load_chunk(wave, wbuf[0], xbuf[0], std::false_type{});
    // the rows' sums of squares: thread t adds the parts t / RP, t / RP + G, ... of row t % RP in that order; the epilogue adds the G sums in
    // theirs.  The loads are issued together, behind those of the first chunk, only as many rounds as there are parts, and never conditional
    // within a round (a part past the end reads the last one).  A part set to zero first makes the compiler wait for the first load before it
    // issues the second: the packed projection, one round of blocks, is the faster without (8 rows of 4,608 x 3,584 10.4 -> 9.9 us), the gated
    // product, whose blocks come several to a unit, with it (8 rows of 37,888 x 3,584 50.9 / 50.4).  They are added up behind the loads of the second chunk: the wait for them is the wait the first multiplication has
    // anyway.  (Exchanges between lanes in place of the G sums: 13.1 -> 13.7 us for 17,920 x 1,536, whose blocks come three to a unit.)
    constexpr int G = WAVES * 64 / RP, PER = SK_MAX_PARTS / G;
    [[maybe_unused]] float part[PER];
    [[maybe_unused]] const int part_m = threadIdx.x % RP, part_q = threadIdx.x / RP;
    if constexpr (SWIGLU || ROPE)
        if (a.row_parts) {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                if constexpr (SWIGLU) part[i] = 0.f;
                if (i * G < a.nparts) {
                    const int p = part_q + i * G;
                    part[i] = a.row_parts[(size_t)(p < a.nparts ? p : a.nparts - 1) * RP + part_m];
                }
            }
        }
    if (wave + WAVES < nfull) load_chunk(wave + WAVES, wbuf[1], xbuf[1], std::false_type{});
    if constexpr (SWIGLU || ROPE)
        if (a.row_parts) {
            float mine = 0.f;
#pragma unroll
            for (int i = 0; i < PER; ++i) mine += (part_q + i * G < a.nparts) ? part[i] : 0.f;
            part_sums[part_q * RP + part_m] = mine;
        }
    // (the first turn is written out: its loads of the second chunk stand above, before the parts are added up)
    if (wave < nfull) multiply(wbuf[0], xbuf[0]);
    if (wave + WAVES < nfull) {
        if (wave + 2 * WAVES < nfull) load_chunk(wave + 2 * WAVES, wbuf[0], xbuf[0], std::false_type{});
        multiply(wbuf[1], xbuf[1]);
        // Two chunks a turn (buffer numbers are constants).  Inside the loop nothing about the loads is
        // conditional: where a path with loads and one without meet, the compiler's count of the loads in
        // flight is the smaller one, and the next wait is for all of them.  So the loop runs while both of
        // a turn's loads exist, and the one or two chunks that are left are taken behind it.
        int c = wave + 2 * WAVES;
        for (; c + 2 * WAVES < nfull; c += 2 * WAVES) {
            load_chunk(c + WAVES, wbuf[1], xbuf[1], std::false_type{});
            multiply(wbuf[0], xbuf[0]);
            load_chunk(c + 2 * WAVES, wbuf[0], xbuf[0], std::false_type{});
            multiply(wbuf[1], xbuf[1]);
        }
        if (c < nfull) {
            const bool more = c + WAVES < nfull;
            if (more) load_chunk(c + WAVES, wbuf[1], xbuf[1], std::false_type{});
            multiply(wbuf[0], xbuf[0]);
            if (more) multiply(wbuf[1], xbuf[1]);
        }
    }
    if (nfull < nchunks && wave == nfull % WAVES) {     // the chunk that K ends in
        load_chunk(nfull, wbuf[0], xbuf[0], std::true_type{});
        multiply(wbuf[0], xbuf[0]);
    }
    if constexpr (SAME_PLACE) __syncthreads();
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) red[wave][mt * NT + nt][lane] = acc[mt][nt];
    __syncthreads();
    skinny_finish<MT, NT, WAVES, SWIGLU, TO, ROPE, EPI>(a, red, pre, n0, nend, block, [&](int m) {
        float sq = part_sums[m];
#pragma unroll
        for (int q = 1; q < WAVES * 64 / RP; ++q) sq += part_sums[q * RP + m];
        return sq;
    });
}

template <int MT, int NT, int WAVES, bool SWIGLU, typename TO, bool ROPE = false, int EPI = 0>
__global__ __launch_bounds__(WAVES * 64) void gemm_bf16_skinny_kernel(SkinnyArgs a) {
    constexpr int CH = MT <= 2 ? SK_CHUNK : SK_CHUNK / 2;
    __shared__ __attribute__((aligned(16))) char lds[SkinnyLds<MT, NT, WAVES, CH>::BYTES];
    skinny_product<MT, NT, WAVES, SWIGLU, TO, ROPE, EPI, CH>(a, blockIdx.x, lds);
}

// Up to 4 rows and K a multiple of 64: the same product where launch, first load and drain are as long as the matrix itself (1 to 30 MB).
// A block's eight waves take K in runs that follow each other (units of 64 k-values), and a wave asks for all it multiplies before it waits
// for anything: the shares of the rows' sums of squares, its part of x (the rows that there are, not sixteen), its part of w, then the
// epilogue's operands.  No load waits behind another one's answer and none is repeated to fill a tile of rows; a branch of the wave's own
// (which units there are) is around loads whose registers nobody else writes, so the compiler puts no wait at its end.  D units at a time: 4
// or 10 at once (K up to 2,048 or 5,120), or, LOOP, rounds of 4 whose loads are on their way while the round before is multiplied.
// In a chain of recorded launches over different matrices, the kernel above against this one (us, one row; an empty launch is 1.6): 896 x 896
// 3.3 -> 3.0, 896 x 4,864 6.8 -> 5.5, 1,536 x 1,536 4.0 -> 3.6, 1,536 x 4,480 6.7 -> 5.8, 1,536 x 8,960 10.5 -> 8.3, 2,048 x 11,008 13.6 -> 11.6,
// 8,240 x 1,536 9.3 -> 7.0; q/k/v with rotation and page write 896 5.0 -> 4.5, 1,536 5.8 -> 5.1.
#define FR_WAVES 8
constexpr int fr_lds_bytes(int xi) { return FR_WAVES * (xi * 1024 + 64 * 16 + 16 * 4); }      // x, sums and shares of squares by wave
template <typename TO, bool ROPE, int EPI, int D, bool LOOP, int XI>
__device__ __forceinline__ void rows_product(const SkinnyArgs& a, const int log_rows, const int block, char* lds) {
    // x of a round by wave: [unit][row][8 pieces of 16 bytes], rows a power of two (1 << log_rows; rows past the last repeat it), XI loads of
    // 64 pieces
    skinny_arguments<ROPE>(a);
    asm volatile("" ::"s"(log_rows));
    floatx4 (*red)[1][64] = reinterpret_cast<floatx4 (*)[1][64]>(lds + FR_WAVES * XI * 1024);
    float (*part_sums)[16] = reinterpret_cast<float (*)[16]>(lds + FR_WAVES * (XI * 1024 + 64 * 16));
    const int M = a.M, N = a.N, K = a.K;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, r16 = lane & 15;
    const int n0 = block * a.cols, half = a.dh / 2, total = ROPE ? (a.nh + 2 * a.nkv) * half : N;
    const int nend = n0 + a.cols < total ? n0 + a.cols : total;
    const int units = K / 64, base = units / FR_WAVES, extra = units % FR_WAVES;
    const int u0 = wave * base + (wave < extra ? wave : extra), n = base + (wave < extra ? 1 : 0);
    [[maybe_unused]] RowShares<16, FR_WAVES> shares;
    if constexpr (ROPE)
        if (a.row_parts) shares.ask(a.row_parts, a.nparts);
    uint16_t* xs = reinterpret_cast<uint16_t*>(lds) + wave * XI * 512;
    bf16x8 xb[XI];
    auto ask_x = [&](int first) {
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int f = (lane + 64 * i) >> 3, row = f & ((1 << log_rows) - 1);
            int u = first + (f >> log_rows);
            u = u < n ? u : n - 1;
            xb[i] = *reinterpret_cast<const bf16x8*>(a.x + (size_t)(row < M ? row : M - 1) * K + 64 * (u0 + u) + 8 * (lane & 7));
        }
    };
    auto put_x = [&]() {
        __builtin_amdgcn_wave_barrier();            // a wave's LDS operations run in order; keep the compiler's too
#pragma unroll
        for (int i = 0; i < XI; ++i)
            *reinterpret_cast<bf16x8*>(xs + (lane + 64 * i) * 8) = xb[i];
        __builtin_amdgcn_wave_barrier();
    };
    int row;
    if (ROPE) {                                     // rows 0..7 of a tile: first members of 8 pairs, 8..15: their partners
        int p = n0 + (r16 & 7);
        p = p < nend ? p : nend - 1;
        const int head = skinny_head(a, p);
        row = head * a.dh + p - head * half + (r16 < 8 ? 0 : half);
    } else row = (n0 + r16 < nend) ? n0 + r16 : nend - 1;
    const bf16_t* wrow = a.w + (size_t)row * K + 64 * u0 + 8 * g;
    bf16x8 wb[D][2];
    auto ask_w = [&](int u, int d) {
#pragma unroll
        for (int j = 0; j < 2; ++j) wb[d][j] = *reinterpret_cast<const bf16x8*>(wrow + 64 * u + 32 * j);
    };
    if (n > 0) {
        ask_x(0);
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (d < n) ask_w(d, d);
    }
    SkinnyPre<1> pre;
    if (SKINNY_PRE<false, EPI> && wave == 0) skinny_ask<1, TO, ROPE, EPI>(a, pre, n0, nend, 0, lane);
    if constexpr (ROPE)                   // added up while w is on its way
        if (a.row_parts) shares.add(a.nparts, part_sums);
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    const int xrow = r16 & ((1 << log_rows) - 1);
    auto multiply = [&](int d) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const bf16x8 xa = *reinterpret_cast<const bf16x8*>(xs + ((((d << log_rows) + xrow) << 3) + g + 4 * j) * 8);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[d][j], xa, acc, 0, 0, 0);
        }
    };
    if (n > 0) {
        int i = 0;
        if constexpr (LOOP) {
            for (; i + D < n; i += D) {             // (a unit past the last asks for the last again: at most three a wave)
                put_x();
                ask_x(i + D);
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    multiply(d);
                    ask_w(i + D + d < n ? i + D + d : n - 1, d);
                }
            }
        }
        put_x();
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (i + d < n) multiply(d);
    }
    red[wave][0][lane] = acc;
    __syncthreads();
    skinny_finish<1, 1, FR_WAVES, false, TO, ROPE, EPI>(a, red, pre, n0, nend, block, [&](int m) {
        float sq = part_sums[0][m];
#pragma unroll
        for (int q = 1; q < FR_WAVES; ++q) sq += part_sums[q][m];
        return sq;
    });
}

template <typename TO, bool ROPE, int EPI, int D, bool LOOP, int XI>
__global__ __launch_bounds__(FR_WAVES * 64) void gemm_bf16_rows_kernel(SkinnyArgs a, int log_rows) {
    __shared__ __attribute__((aligned(16))) char lds[fr_lds_bytes(XI)];
    rows_product<TO, ROPE, EPI, D, LOOP, XI>(a, log_rows, blockIdx.x, lds);
}

#define ROWS_KERNEL_M 4          // rows up to which gemm_bf16_rows_kernel is taken (rows_kernel_takes)

// Compute units of the current device (256 where it cannot be asked).
static int compute_units() {
    static int units[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) { (void)hipGetLastError(); return 256; }
    if (!units[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) { (void)hipGetLastError(); n = 256; }
        units[dev] = n;
    }
    return units[dev];
}

// Many columns in tiles of `unit`: the blocks of a product go round the compute units several times, and
// the units with one block more than the others set the time when the matrix is small.  The columns a
// block takes are therefore cut down until the last round is as full as the others: as many rounds as
// whole tiles would need, and equal shares of the columns within them (at least half a tile's).
static int balanced_round_cols(int total, int unit, long cu) {
    const long rounds = (total + unit * cu - 1) / (unit * cu);
    long per = (total + rounds * cu - 1) / (rounds * cu);
    per = per < unit / 2 ? unit / 2 : per;
    return (int)(per > unit ? unit : per);
}
