// Choosing the next token from float32 logits: argmax (lowest index on ties)
// and temperature / top-k / top-p sampling by inverse CDF with a uniform
// number from the request's own counter-based stream, which the host derives or,
// for requests whose sampling state lies in the per-slot table on the device
// (li_sample_prepare), the device itself.
#include "common.h"
#include "li_noalloc.h"
#include <math.h>
#include <mutex>
#include <stdio.h>

#define SMP_NT 1024

// (value, index) maximum with the lower index winning ties
__device__ __forceinline__ void argmax_combine(float& v, int& i, float ov, int oi) {
    if (ov > v || (ov == v && oi < i)) { v = ov; i = oi; }
}

__device__ __forceinline__ void block_argmax(float& v, int& i, float* sv, int* si) {
#pragma unroll
    for (int o = LI_WAVE / 2; o > 0; o >>= 1) {
        const float ov = __shfl_xor(v, o, LI_WAVE);
        const int oi = __shfl_xor(i, o, LI_WAVE);
        argmax_combine(v, i, ov, oi);
    }
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
    __syncthreads();
    if (lane == 0) { sv[w] = v; si[w] = i; }
    __syncthreads();
    v = sv[0]; i = si[0];
    for (int k = 1; k < SMP_NT / LI_WAVE; ++k) argmax_combine(v, i, sv[k], si[k]);
}

// Two stages, so that a few rows still use many compute units: stage 1 finds the
// (maximum, lowest index) of each of ARGMAX_CHUNKS contiguous chunks of a row, stage 2
// combines a row's chunks.  Ties go to the lower index in both.
#define ARGMAX_CHUNKS 32

__global__ __launch_bounds__(SMP_NT) void argmax_partial_kernel(const float* __restrict__ logits,
                                                                float* __restrict__ pv, int* __restrict__ pi,
                                                                int V, int chunk) {
    __shared__ float sv[SMP_NT / LI_WAVE];
    __shared__ int si[SMP_NT / LI_WAVE];
    const float* row = logits + (size_t)blockIdx.x * V;
    const int c0 = blockIdx.y * chunk, c1 = (c0 + chunk < V) ? c0 + chunk : V;
    float v = -INFINITY;
    int i = 0x7fffffff;
    for (int j = c0 + threadIdx.x; j < c1; j += SMP_NT) {
        const float x = row[j];
        if (x > v || i == 0x7fffffff) { v = x; i = j; }   // strictly greater: the first maximum stays
    }
    block_argmax(v, i, sv, si);
    if (threadIdx.x == 0) { pv[blockIdx.x * gridDim.y + blockIdx.y] = v; pi[blockIdx.x * gridDim.y + blockIdx.y] = i; }
}

__global__ __launch_bounds__(64) void argmax_final_kernel(const float* __restrict__ pv, const int* __restrict__ pi,
                                                          int* __restrict__ out, int nchunks) {
    float v = -INFINITY;
    int i = 0x7fffffff;
    for (int c = threadIdx.x; c < nchunks; c += 64) argmax_combine(v, i, pv[blockIdx.x * nchunks + c], pi[blockIdx.x * nchunks + c]);
#pragma unroll
    for (int o = LI_WAVE / 2; o > 0; o >>= 1) {
        const float ov = __shfl_xor(v, o, LI_WAVE);
        const int oi = __shfl_xor(i, o, LI_WAVE);
        argmax_combine(v, i, ov, oi);
    }
    if (threadIdx.x == 0) out[blockIdx.x] = i;
}

// scratch_v, scratch_i: n * ARGMAX_CHUNKS floats / ints
extern "C" int li_argmax_rows(const float* logits, int* out, float* scratch_v, int* scratch_i, int n, int V,
                              hipStream_t stream) {
    if (n <= 0 || V <= 0) return LI_ERR_SIZE;
    int nchunks = (V + 4095) / 4096;
    if (nchunks > ARGMAX_CHUNKS) nchunks = ARGMAX_CHUNKS;
    const int chunk = (V + nchunks - 1) / nchunks;
    argmax_partial_kernel<<<dim3(n, nchunks), SMP_NT, 0, stream>>>(logits, scratch_v, scratch_i, V, chunk);
    argmax_final_kernel<<<n, 64, 0, stream>>>(scratch_v, scratch_i, out, nchunks);
    return li_launch_status();
}

// ------------------------------------------------- argmax that allocates nothing
// The same two kernels with their partial results in a file-scope device array instead of
// buffers that the caller brings: for callers that cannot allocate (li_noalloc.h).  Every
// GPU holds its own copy of the array at its own address; host code must use the address
// that hipGetSymbolAddress gives for the current device, never the array's name.
static __device__ __align__(256) unsigned char scratch[LI_ARGMAX_NOALLOC_MAX_ROWS * ARGMAX_CHUNKS * 8];

#define LI_NOALLOC_MAX_DEVICES 64
static void* g_scratch_ptr[LI_NOALLOC_MAX_DEVICES];       // the array's address on each device, once asked for
static std::mutex g_scratch_mutex;
static thread_local char g_noalloc_error[200];

static int noalloc_fail(int code, const char* what, hipError_t e) {
    if (e != hipSuccess) snprintf(g_noalloc_error, sizeof g_noalloc_error, "%s: %s", what, hipGetErrorString(e));
    else snprintf(g_noalloc_error, sizeof g_noalloc_error, "%s", what);
    return code;
}

// The scratch array's address on the current device (asked for once per device).
static int noalloc_scratch(void** ptr) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return noalloc_fail(LI_ERR_LAUNCH, "li_argmax_rows_noalloc: hipGetDevice", e);
    if (dev < 0 || dev >= LI_NOALLOC_MAX_DEVICES)
        return noalloc_fail(LI_ERR_SIZE, "li_argmax_rows_noalloc: device number beyond the table of scratch addresses", hipSuccess);
    std::lock_guard<std::mutex> hold(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return noalloc_fail(LI_ERR_LAUNCH, "li_argmax_rows_noalloc: hipGetSymbolAddress(scratch)", e);
        g_scratch_ptr[dev] = p;
    }
    *ptr = g_scratch_ptr[dev];
    return LI_OK;
}

extern "C" int li_argmax_rows_noalloc_init(void) {
    void* p;
    return noalloc_scratch(&p);
}

extern "C" int li_argmax_rows_noalloc_max_rows(void) { return LI_ARGMAX_NOALLOC_MAX_ROWS; }

extern "C" const char* li_argmax_rows_noalloc_error(void) { return g_noalloc_error; }

extern "C" int li_argmax_rows_noalloc(const float* logits, int* out, int n, int V, hipStream_t stream) {
    g_noalloc_error[0] = 0;
    if (n <= 0 || V <= 0) return noalloc_fail(LI_ERR_SIZE, "li_argmax_rows_noalloc: rows and vocabulary must be positive", hipSuccess);
    if (n > LI_ARGMAX_NOALLOC_MAX_ROWS) {
        snprintf(g_noalloc_error, sizeof g_noalloc_error,
                 "li_argmax_rows_noalloc: %d rows are more than the %d that the scratch array holds; "
                 "use li_argmax_rows with buffers of the caller", n, LI_ARGMAX_NOALLOC_MAX_ROWS);
        return LI_ERR_SIZE;
    }
    void* base = nullptr;
    const int rc = noalloc_scratch(&base);
    if (rc != LI_OK) return rc;
    // partial maxima first, their indices behind them; stage 1 writes every place that stage 2
    // reads, so nothing of an earlier call's contents has to be cleared
    float* pv = reinterpret_cast<float*>(base);
    int* pi = reinterpret_cast<int*>(static_cast<unsigned char*>(base) + (size_t)LI_ARGMAX_NOALLOC_MAX_ROWS * ARGMAX_CHUNKS * 4);
    int nchunks = (V + 4095) / 4096;
    if (nchunks > ARGMAX_CHUNKS) nchunks = ARGMAX_CHUNKS;
    const int chunk = (V + nchunks - 1) / nchunks;
    argmax_partial_kernel<<<dim3(n, nchunks), SMP_NT, 0, stream>>>(logits, pv, pi, V, chunk);
    argmax_final_kernel<<<n, 64, 0, stream>>>(pv, pi, out, nchunks);
    if (li_launch_status() != LI_OK) return noalloc_fail(LI_ERR_LAUNCH, "li_argmax_rows_noalloc: launch failed", hipSuccess);
    return LI_OK;
}

// ---------------------------------------------------------------- sampling
// The candidates are ordered by (value descending, index ascending); top-k keeps the first k, top-p
// then the shortest prefix whose softmax mass (among the top-k survivors) reaches p; the survivors'
// softmax is sampled by inverse CDF over ASCENDING ids with the given uniform number.
// Two kernels.  The first has a block for every tile of SMP_TILE ids of every row, so that a few
// rows still use many compute units: a tile's maximum, and for rows without top-k and top-p its
// softmax sum, for greedy rows its argmax.  The second has one block per row.  It reads the row in
// the same tiles (thread t the 8 consecutive ids t * 8 ... of a tile: whole lines), in as few
// passes as it can: the thresholds of top-k and top-p are found four bits a pass over the
// order-preserving integer image of the floats (16 counts or 16 masses a thread and pass).  Every
// count and every mass is added in a fixed order, so the same inputs always give the same token.
constexpr int SMP_TILE = SMP_NT * 8;
constexpr int SMP_WAVES = SMP_NT / LI_WAVE;

__device__ __forceinline__ uint32_t sort_key(float z) {
    const uint32_t b = __float_as_uint(z);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
__device__ __forceinline__ bool sample_unfiltered(int k, float p, int V) { return !(k > 0 && k < V) && !(p > 0.f && p < 1.f); }

__device__ __forceinline__ int block_sum_int(int v, int* smem) {
#pragma unroll
    for (int o = LI_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, LI_WAVE);
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
    __syncthreads();
    if (lane == 0) smem[w] = v;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int i = 0; i < SMP_WAVES; ++i) t += smem[i];
    return t;
}

__device__ __forceinline__ float block_max_f(float v, float* smem) {
    v = wave_max(v);
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
    __syncthreads();
    if (lane == 0) smem[w] = v;
    __syncthreads();
    float t = smem[0];
#pragma unroll
    for (int i = 1; i < SMP_WAVES; ++i) t = fmaxf(t, smem[i]);
    return t;
}

__device__ __forceinline__ int block_min_int(int v, int* smem) {
#pragma unroll
    for (int o = LI_WAVE / 2; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, LI_WAVE));
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
    __syncthreads();
    if (lane == 0) smem[w] = v;
    __syncthreads();
    int t = smem[0];
#pragma unroll
    for (int i = 1; i < SMP_WAVES; ++i) t = min(t, smem[i]);
    return t;
}

// The 16 sums of a pass over the whole block, left in tot[0..15] for every thread to read.  Within a
// wave the lanes halve what they hold step by step (a lane keeps one half of its sums and gets the
// other lane's part of that half: 8 + 4 + 2 + 1 exchanges), until each lane holds one sum of its 16
// lanes, then the four groups of 16 lanes are added: 17 exchanges instead of 96; then the waves in
// their order.  The order of the additions is fixed.  work: WAVES * 16 values.
template <int WAVES, typename T>
__device__ __forceinline__ void block_sum16(T (&c)[16], T* work, T* tot) {
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
#define LI_HALVE(H, MASK)                                                         \
    {                                                                             \
        const bool upper = (lane & (MASK)) != 0;                                  \
        _Pragma("unroll") for (int i = 0; i < (H); ++i) {                         \
            const T give = upper ? c[i] : c[i + (H)];                             \
            const T keep = upper ? c[i + (H)] : c[i];                             \
            c[i] = keep + __shfl_xor(give, (MASK), LI_WAVE);                      \
        }                                                                         \
    }
    LI_HALVE(8, 1)
    LI_HALVE(4, 2)
    LI_HALVE(2, 4)
    LI_HALVE(1, 8)
#undef LI_HALVE
    c[0] += __shfl_xor(c[0], 16, LI_WAVE);
    c[0] += __shfl_xor(c[0], 32, LI_WAVE);
    // lane l < 16 now holds the wave's sum number 8 (l & 1) + 4 (l >> 1 & 1) + 2 (l >> 2 & 1) + (l >> 3 & 1)
    __syncthreads();                                 // (the last pass's totals have been read)
    if (lane < 16) work[w * 16 + 8 * (lane & 1) + 4 * ((lane >> 1) & 1) + 2 * ((lane >> 2) & 1) + ((lane >> 3) & 1)] = c[0];
    __syncthreads();
    if (threadIdx.x < 16) {
        T t = 0;
        for (int i = 0; i < WAVES; ++i) t += work[i * 16 + threadIdx.x];
        tot[threadIdx.x] = t;
    }
    __syncthreads();
}

// Sum of v over the threads before this one, in thread order.  work: WAVES values.
template <int WAVES = SMP_WAVES, typename T>
__device__ __forceinline__ T block_sum_before(T v, T* work) {
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
    T inc = v;
#pragma unroll
    for (int o = 1; o < LI_WAVE; o <<= 1) {
        const T t = __shfl_up(inc, o, LI_WAVE);
        if (lane >= o) inc += t;
    }
    T before = __shfl_up(inc, 1, LI_WAVE);
    if (lane == 0) before = 0;
    __syncthreads();
    if (lane == LI_WAVE - 1) work[w] = inc;
    __syncthreads();
    T base = 0;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) base += i < w ? work[i] : T(0);      // (all reads at once; adding a zero changes nothing)
    return base + before;
}

// A thread's 8 ids of a tile (whole 16-byte loads where the row allows them): the logits; and z = logit / T
__device__ __forceinline__ void load_ids8(const float* __restrict__ row, int j0, int V, bool vec, float (&x)[8]) {
    if (vec && j0 + 8 <= V) {
        const float4 a = *reinterpret_cast<const float4*>(row + j0), b = *reinterpret_cast<const float4*>(row + j0 + 4);
        x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
        x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (j0 + e < V) ? row[j0 + e] : -INFINITY;
    }
}
__device__ __forceinline__ void load_ids8(const float* __restrict__ row, int j0, int V, float T, bool vec, float (&z)[8]) {
    load_ids8(row, j0, V, vec, z);
#pragma unroll
    for (int e = 0; e < 8; ++e) z[e] /= T;
}

// f(z, id) for this thread's ids of all tiles, ascending
template <typename F>
__device__ __forceinline__ void each_id(const float* __restrict__ row, int V, float T, bool vec, int ntiles, F&& f) {
    for (int tile = 0; tile < ntiles; ++tile) {
        const int j0 = tile * SMP_TILE + (int)threadIdx.x * 8;
        if (j0 >= V) break;
        float z[8];
        load_ids8(row, j0, V, T, vec, z);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (j0 + e < V) f(z[e], j0 + e);
    }
}

// tau = the kk-th largest key among the z that `each` hands out (to all threads of the block together),
// need (>= 1) = how many of the keys equal to tau are among the kk largest.  Four bits a pass: counts of
// the 16 values of the next digit among the keys that agree with the digits found so far.
template <int WAVES = SMP_WAVES, typename Each>
__device__ __forceinline__ void radix_kth(Each&& each, int kk, uint32_t& tau, int& need, int* work_i, int* tot_i) {
    tau = 0u;
    for (int shift = 28; shift >= 0; shift -= 4) {
        int cnt[16];
#pragma unroll
        for (int b = 0; b < 16; ++b) cnt[b] = 0;
        each([&](float z) {
            const uint32_t key = sort_key(z);
            if (shift == 28 || (key >> (shift + 4)) == (tau >> (shift + 4))) {
                const int d = (key >> shift) & 15;
#pragma unroll
                for (int b = 0; b < 16; ++b) cnt[b] += (d == b);
            }
        });
        block_sum16<WAVES>(cnt, work_i, tot_i);
        int above = 0, d = 15;
        for (; d > 0; --d) {
            if (above + tot_i[d] >= kk) break;
            above += tot_i[d];
        }
        kk -= above;
        tau |= (uint32_t)d << shift;
    }
    need = kk;
}

// The same tau and need for keys that lie in registers, up to 8 a thread (0: none), in the first `waves` waves and, where the
// last one is cut short, the one behind them.  Eight passes of sixteen counts are long for one block; this takes a bound
// first.  Each of the `waves` whole waves finds the ceil(kk / waves)-th largest of its threads' largest keys: at least kk keys
// are no smaller than the least of these, and in earnest not many more (kk = 50 of 8,192 normal logits: some 150; a wave cut
// short sets no bound: its share of kk would lie far down among its few keys, or it would not have as many; 16 rows of 32,000
// ids, top-k 200 with top-p 0.9: 73.5 us with its bound, 49.5).  They go into a list in LDS, and each is held against all
// others: the one with fewer than kk keys above it and at least kk no smaller is tau.  False, with nothing done, where the
// bound leaves fewer than kk keys (a wave without enough of them sets none) or more than SMP_LIST (many equal logits):
// radix_kth then.
// 64 rows of 151,936 ids, top-k 50: tiles kernel 58 -> 45 us (one row 26 -> 13), rows kernel 22 -> 14.  Both are shorter since a tile hands
// over all that it listed (below; top-k with top-p 44 + 25 -> 24 + 19), and by tile_bound and rows_by_list (11 + 10).  What is left for this function is rows
// whose tiles hand over exactly kc ids, and those that rows_by_list leaves.
constexpr int SMP_LIST = 1024;
// the bound, as above (0: none): at least kk of the block's keys are no smaller
__device__ __forceinline__ uint32_t bound_of_kth(const uint32_t (&key)[8], int kk, int waves, int* work_i) {
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
    uint32_t cur = key[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) cur = max(cur, key[e]);
    const int rounds = (kk + waves - 1) / waves;
    if (rounds > LI_WAVE) return 0u;
    // the rounds-th largest of the wave's keys, bit by bit, down to the sixteenth (a bound; 0: the wave has fewer)
    uint32_t largest = 0u;
#pragma unroll
    for (int b = 31; b >= 16; --b) {
        const uint32_t trial = largest | (1u << b);
        if (__popcll((unsigned long long)__ballot(cur >= trial)) >= rounds) largest = trial;
    }
    __syncthreads();
    if (lane == 0) work_i[w] = (int)largest;
    __syncthreads();
    uint32_t bound = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < SMP_WAVES; ++i) bound = i < waves ? min(bound, (uint32_t)work_i[i] - 1u) : bound;      // (0, no bound, becomes the largest)
    return bound + 1u;
}
// put(place, e) for the keys no smaller than the bound, in the order of threads and keys; how many they are is left in res[0] (and is
// there for all threads behind the next barrier)
template <typename Put>
__device__ __forceinline__ void put_from(const uint32_t (&key)[8], uint32_t bound, int* work_i, int* res, Put&& put) {
    int mine = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) mine += key[e] >= bound;
    int pos = block_sum_before(mine, work_i);
    if (threadIdx.x == SMP_NT - 1) res[0] = pos + mine;
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (key[e] >= bound) put(pos++, e);
}
// n keys in the list (n at least kk): tau and need
template <int NT = SMP_NT>
__device__ __forceinline__ void kth_of_list(uint32_t* list, int n, int kk, uint32_t& tau, int& need, int* res) {
    const int tid = threadIdx.x;
    if (tid < 4 && n + tid < SMP_LIST) list[n + tid] = 0u;      // (whole pieces of four below)
    __syncthreads();
    for (int i = tid; i < n; i += NT) {
        const uint32_t own = list[i];
        int above = 0, from = 0;
#pragma unroll 8
        for (int j = 0; j < n; j += 4) {
            const uint4 v = *reinterpret_cast<const uint4*>(list + j);
            above += (v.x > own) + (v.y > own) + (v.z > own) + (v.w > own);
            from += (v.x >= own) + (v.y >= own) + (v.z >= own) + (v.w >= own);
        }
        if (above < kk && from >= kk) { res[1] = (int)own; res[2] = kk - above; }      // (all threads with this key write the same)
    }
    __syncthreads();
    tau = (uint32_t)res[1];
    need = res[2];
}
// `tag` gives each key's own number (its id), which goes beside it into list_id; n: the keys in the list
template <typename Tag>
__device__ __forceinline__ bool select_kth(const uint32_t (&key)[8], int kk, int waves, uint32_t& tau, int& need, uint32_t* list, int* list_id,
                                           int& n, int* work_i, int* res, Tag&& tag) {
    const uint32_t bound = bound_of_kth(key, kk, waves, work_i);
    if (bound == 0u) return false;
    put_from(key, bound, work_i, res, [&](int at, int e) {
        if (at < SMP_LIST) { list[at] = key[e]; list_id[at] = tag(e); }
    });
    __syncthreads();
    n = res[0];
    if (n < kk || n > SMP_LIST) return false;
    kth_of_list(list, n, kk, tau, need, res);
    return true;
}

// Top-p among the survivors of top-k where these lie in the list: the same tp as radix_mass and what is left of `remaining` =
// p x (their mass), which is worked out here.  Each key of the list is held against all others: its own mass and that above it
// (sums of four, in the list's order: they grow with every key that counts, so one key alone has the prefix's end), the
// one whose mass above is short of `remaining` and whose own reaches it is tp; below them all the keys equal to tau.
// False, with nothing done, where rounding or masses of zero leave none (radix_mass then).  64 rows of 151,936 ids, top-k 50 with
// top-p 0.9: rows kernel 25 us with radix passes (up to eight, three barriers each).
__device__ __forceinline__ bool mass_of_list(const uint32_t* list, int n, uint32_t tau, int ties, float m, float p,
                                             float& remaining, uint32_t& tp, float* mass, float* res_f, int* res) {
    const int tid = threadIdx.x;
    if (tid < ((n + 3) & ~3)) mass[tid] = tid < n && list[tid] > tau ? expf(key_value(list[tid]) - m) : 0.f;
    if (tid == 0) res[0] = 0;
    __syncthreads();
    const float e_ties = (float)ties * expf(key_value(tau) - m);
    if (tid < n) {
        const uint32_t own = list[tid];
        float above[4] = {0.f, 0.f, 0.f, 0.f}, from[4] = {0.f, 0.f, 0.f, 0.f}, all[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int j = 0; j < n; j += 4) {                // (the list is filled up to whole pieces)
            const uint4 v = *reinterpret_cast<const uint4*>(list + j);
            const float4 e = *reinterpret_cast<const float4*>(mass + j);
            const uint32_t k4[4] = {v.x, v.y, v.z, v.w};
            const float e4[4] = {e.x, e.y, e.z, e.w};
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                above[u] += k4[u] > own ? e4[u] : 0.f;
                from[u] += k4[u] >= own ? e4[u] : 0.f;
                all[u] += e4[u];
            }
        }
        const float g = (above[0] + above[1]) + (above[2] + above[3]), h = (from[0] + from[1]) + (from[2] + from[3]);
        const float z = (all[0] + all[1]) + (all[2] + all[3]), want = p * (z + e_ties);
        if (own > tau ? g < want && h >= want : own == tau && z < want && z + e_ties >= want) {
            res[0] = 1;                                  // (all threads with this key write the same)
            res[1] = (int)own;
            res_f[0] = want - (own > tau ? g : z);
        }
    }
    __syncthreads();
    if (!res[0]) return false;
    tp = (uint32_t)res[1];
    remaining = res_f[0];
    return true;
}

// Top-p among the survivors of top-k (cut: the keys above tau, and `ties` keys equal to tau with
// e_ties = their mass together; not cut: all keys): tp = the largest key c with mass(keys >= c) >=
// `remaining`, four bits a pass (masses by the next digit); on return `remaining` is what the keys
// equal to tp have to bring.  m: the maximum that masses are taken against.
// Where cut, digits in which tau, which no survivor is below, and the maximum agree are taken as they are; and with LOOK,
// once all keys that agree with the digits found are one key (alone, or several ids of one value), it is tp: a digit of which
// all mass is left changes neither `remaining` nor the choice.  64 rows, top-k 50 with top-p 0.9: rows kernel 40 -> 25 us.
// A look takes two barriers, so it is taken where the mass that is left is no more than one key's (two keys so close bring
// twice the least of them), and once behind the digits of a bfloat16 value, several ids of which there mostly are.  It is
// for keys in registers: over the row itself a pass takes as long as the one it may spare (64 rows, top-k 300 with top-p
// 0.95, logits of bfloat16's values: 762 us with it, 635 without).
template <bool LOOK, typename Each>
__device__ __forceinline__ void radix_mass(Each&& each, bool cut, uint32_t tau, int ties, float e_ties, float m,
                                           float& remaining, uint32_t& tp, float* work_f, float* tot_f, int* res) {
    tp = 0u;
    int first = 28;
    if (cut) {
        const uint32_t top = sort_key(m);
        while (first > 0 && (tau >> first) == (top >> first)) first -= 4;
        tp = first < 28 ? (top >> (first + 4)) << (first + 4) : 0u;
    }
    for (int shift = first; shift >= 0; shift -= 4) {
        float mass[16];
#pragma unroll
        for (int b = 0; b < 16; ++b) mass[b] = 0.f;
        each([&](float z) {
            const uint32_t key = sort_key(z);
            if ((!cut || key > tau) && (shift == 28 || (key >> (shift + 4)) == (tp >> (shift + 4)))) {
                const int d = (key >> shift) & 15;
                const float e = expf(z - m);
#pragma unroll
                for (int b = 0; b < 16; ++b) mass[b] += (d == b) ? e : 0.f;
            }
        });
        block_sum16<SMP_WAVES>(mass, work_f, tot_f);
        const bool ties_here = cut && ties > 0 && (shift == 28 || (tau >> (shift + 4)) == (tp >> (shift + 4)));
        const int d_ties = (tau >> shift) & 15;
        float above = 0.f;
        int d = 15, lowest = -1;
        bool reached = false;
        for (; d >= 0; --d) {
            const float t = tot_f[d] + ((ties_here && d == d_ties) ? e_ties : 0.f);
            if (t > 0.f) lowest = d;
            if (t > 0.f && above + t >= remaining) { reached = true; break; }
            above += t;
        }
        if (!reached) {                       // rounding left the target just above the sum: the lowest digit with mass
            d = lowest < 0 ? 0 : lowest;
            above = 0.f;
            for (int b = 15; b > d; --b) above += tot_f[b] + ((ties_here && b == d_ties) ? e_ties : 0.f);
        }
        remaining -= above;
        tp |= (uint32_t)d << shift;
        if (LOOK && shift > 0 && cut && !(ties > 0 && (tau >> shift) == (tp >> shift))) {
            const float least = key_value(tp), most = key_value(tp | ((1u << shift) - 1u));
            if (!(shift == 16 || (most - least < 0.69f && tot_f[d] <= 1.0001f * expf(most - m)))) continue;
            uint32_t one = 0u;                   // one of the thread's keys that are left (0: it has none; a key above tau is not 0)
            bool differ = false;
            each([&](float z) {
                const uint32_t key = sort_key(z);
                if (key > tau && (key >> shift) == (tp >> shift)) { differ |= one != 0u && key != one; one = key; }
            });
            if (one) res[0] = (int)one;          // (any of the threads' keys: the others are held against it)
            if (__syncthreads_or(one != 0u)) {
                const uint32_t all = (uint32_t)res[0];
                if (!__syncthreads_or(differ || (one && one != all))) { tp = all; return; }
            }
        }
    }
}

// how many of the keys equal to tp count, from what they have to bring
__device__ __forceinline__ int ties_needed(float remaining, uint32_t tp, float m) {
    const float e_tp = expf(key_value(tp) - m);
    if (!(e_tp > 0.f)) return 0x7fffffff;     // ties without mass: all of them
    const float q = ceilf(remaining / e_tp);
    return q < 1.f ? 1 : (q > 2.0e9f ? 0x7fffffff : (int)q);
}

// Rows with top-k or top-p: the first kernel hands the second one, per tile, the tile's SMP_KC
// or fewer largest ids (in the order (value descending, id ascending)), so that the second kernel
// searches among ntiles * kc candidates in registers instead of reading the row pass after pass.
// With top-k <= SMP_KC the candidates hold all survivors (kc = k).  With top-p alone kc = SMP_KC_P
// and the second kernel checks that the prefix ends above the kc-th largest id of the row, whose
// betters are all among the candidates; otherwise it reads the row.  0: no candidates.
constexpr int SMP_KC = 256, SMP_KC_P = 128, SMP_CAND_PER_THREAD = 8, SMP_WIDE_TILES = 512;        // (SMP_KC <= 16 * LI_WAVE and 8 keys a thread: select_kth)
__device__ __forceinline__ int sample_candidates(int k, float p, int V, int ntiles) {
    if (sample_unfiltered(k, p, V)) return 0;
    const int kc = (k > 0 && k < V) ? k : SMP_KC_P;
    return (kc <= SMP_KC && (long)kc * ntiles <= (long)SMP_NT * SMP_CAND_PER_THREAD) ? kc : 0;
}

// Do SMP_KC candidates of every tile fit the second kernel's registers?  Then a tile may hand over more than kc of them: all that
// are no smaller than a bound (tile_i: how many).  With top-p alone the second kernel goes through all candidates pass after pass, and
// twice as many cost more than the tiles save unless these are many (p 0.9, exactly kc / all from the bound: one row of 151,936 ids 52 / 57.5
// us, 16 62 / 68, 64 92 / 87, 256 219 / 177; 64 of 32,000 51 / 53, 256 78 / 77).
__device__ __forceinline__ bool sample_wide(int k, int V, int rows, int ntiles) {
    return ntiles * SMP_KC <= SMP_NT * SMP_CAND_PER_THREAD && ((k > 0 && k < V) || rows * ntiles > SMP_WIDE_TILES);
}

// ---- the first kernel.  A wave takes STEPS stretches of 512 ids that follow each other, a lane 8 neighbouring ids of each (two 16-byte
// loads): a block of 1,024 threads with one stretch a wave for few tiles, where the time is one block's, and of 256 threads with four where
// the tiles are many (TILE_MANY): 64 rows of 151,936 ids are 9.7 million values, 6.3 us at 6 TB/s, and four instructions a value are a
// microsecond of the vector ALU's, so what is done once a thread (reductions over the block, barriers, scans) is spread over 32
// values there.  What is done a value is little: quotients are only worked out where the tile's mass is asked for, by five
// instructions; the largest ids are found among the logits themselves, whose order division by T keeps.
// 64 rows of 151,936 ids, us, with blocks of 1,024 threads and every value divided first, and now: greedy 11.6 / 7.2, at a temperature 12.9 / 11.0,
// top-k 50 with top-p 0.9 22.2 / 10.9, a third each 18.4 / 10.4.  One stretch a wave below 768 tiles: at a temperature alone a thread's 32
// exponentials one behind the other are the longer time there (32 rows, 608 tiles, both kernels: 15.7 against 17.8, before 17.5; 48 rows 18.1 / 18.8, before
// 19.9), while the other rows gain at any number (16 rows with top-k 19.0 / 17.1, before 25.4).
constexpr int TILE_STRETCH = 8 * LI_WAVE;
constexpr size_t TILE_MANY = 768;           // (rows x tiles)
template <int STEPS> constexpr int TILE_NT = SMP_NT / STEPS;
template <int STEPS> constexpr int TILE_WAVES = SMP_WAVES / STEPS;

// x / T, correctly rounded (the same bits as the division) for T and x between 2^-40 and 2^40 in size, y = 1 / T rounded: the first
// quotient is off by less than two units of its last place, the second by hardly more than half of one, so that its remainder is
// exact, and by Markstein's theorem the third is the rounded quotient.  Five instructions; the division, which also serves
// the ends of the range, is twelve.
__device__ __forceinline__ float quotient(float x, float T, float y) {
    const float q0 = x * y, q1 = fmaf(fmaf(-q0, T, x), y, q0);
    return fmaf(fmaf(-q1, T, x), y, q1);
}

// The sums over the wave of a value each stretch, to smem[stretch] (numbered over the block), in the lanes' order of wave_sum.  Four at once:
// with two values in a swap's operands one half of its result is the one's sums over the lanes l and l ^ 32, the other half the
// other's, and so on, so that each row of 16 lanes is left with one value (the same sums, the same bits).
__device__ __forceinline__ void tile_sums(const float (&v)[1], float* smem) {
    const float s = wave_sum(v[0]);
    if ((threadIdx.x & (LI_WAVE - 1)) == 0) smem[threadIdx.x / LI_WAVE] = s;
}
__device__ __forceinline__ void tile_sums(const float (&v)[4], float* smem) {
    auto two = [](float a, float b, auto swap) {
        const auto r = swap(__float_as_uint(a), __float_as_uint(b));
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    };
    auto halves = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_permlane32_swap(a, b, false, false); };
    auto rows = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_permlane16_swap(a, b, false, false); };
    // lanes 0..31 of the first hold v[0], 32..63 v[1]; of the second v[2] and v[3]; then rows 0, 1, 2, 3 of lanes: v[0], v[2], v[1], v[3]
    float s = two(two(v[0], v[1], halves), two(v[2], v[3], halves), rows);
    s += __int_as_float(dpp_mov<0x128>(__float_as_int(s)));
    s += __int_as_float(dpp_mov<0x124>(__float_as_int(s)));
    s += __int_as_float(dpp_mov<0x122>(__float_as_int(s)));
    s += __int_as_float(dpp_mov<0x121>(__float_as_int(s)));
    const int lane = threadIdx.x & (LI_WAVE - 1), row = lane >> 4;
    if ((lane & 15) == 0) smem[4 * (threadIdx.x / LI_WAVE) + 2 * (row & 1) + (row >> 1)] = s;
}

// In the order of ids (wave, stretch, lane): how many of the block's n[c] lie before each of this thread's stretches; the block's number.
// work: a value a wave.
template <int STEPS>
__device__ __forceinline__ int tile_places(const int (&n)[STEPS], int (&place)[STEPS], int* work) {
    static_assert(STEPS == 1 || STEPS == 4, "one count, or two in each of two words (512 at most a stretch and wave)");
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
    uint32_t a = (uint32_t)n[0], b = 0u;
    if constexpr (STEPS == 4) { a |= (uint32_t)n[1] << 16; b = (uint32_t)n[2] | (uint32_t)n[3] << 16; }
    const uint32_t a0 = a, b0 = b;
#pragma unroll
    for (int o = 1; o < LI_WAVE; o <<= 1) {
        const uint32_t ta = __shfl_up(a, o, LI_WAVE), tb = STEPS == 4 ? __shfl_up(b, o, LI_WAVE) : 0u;
        if (lane >= o) { a += ta; b += tb; }
    }
    const uint32_t wa = __shfl(a, LI_WAVE - 1, LI_WAVE), wb = STEPS == 4 ? __shfl(b, LI_WAVE - 1, LI_WAVE) : 0u;
    __syncthreads();
    if (lane == 0) work[w] = (int)((wa & 0xffff) + (wa >> 16) + (wb & 0xffff) + (wb >> 16));
    __syncthreads();
    int base = 0, total = 0;
#pragma unroll
    for (int i = 0; i < TILE_WAVES<STEPS>; ++i) { const int t = work[i]; base += i < w ? t : 0; total += t; }
    a -= a0;
    b -= b0;
    place[0] = base + (int)(a & 0xffff);
    if constexpr (STEPS == 4) {
        base += wa & 0xffff;
        place[1] = base + (int)(a >> 16);
        base += wa >> 16;
        place[2] = base + (int)(b & 0xffff);
        base += wb & 0xffff;
        place[3] = base + (int)(b >> 16);
    }
    return total;
}

// the rounds-th largest of the wave's keys, bit by bit from the highest down to bit LAST (a bound; 0: the wave has fewer)
template <int LAST>
__device__ __forceinline__ uint32_t wave_bound(uint32_t key, int rounds) {
    uint32_t largest = 0u;
#pragma unroll
    for (int b = 31; b >= LAST; --b) {
        const uint32_t trial = largest | (1u << b);
        if (__popcll((unsigned long long)__ballot(key >= trial)) >= rounds) largest = trial;
    }
    return largest;
}
// A key (sort_key) that at least kk of the tile's values are no smaller than (0: none found): as bound_of_kth, from the largest values of
// the lanes' stretches; where a wave has four and few are asked of it, from the lanes' largest of all four (8,192 normal logits, kk = 50: some 75 values
// from that bound on; from those of the stretches 150).  Only whole stretches (waves) count.  top[c]: the lane's largest value of stretch c.
template <int STEPS>
__device__ __forceinline__ uint32_t tile_bound(const float (&top)[STEPS], int kk, int in_tile, int* work) {
    const int lane = threadIdx.x & (LI_WAVE - 1), w = threadIdx.x / LI_WAVE;
    __syncthreads();                                 // (work has been read)
    const int waves = in_tile / (STEPS * TILE_STRETCH);
    const bool by_wave = STEPS > 1 && waves > 0 && (kk + waves - 1) / waves <= 24;
    int parts = max(in_tile / TILE_STRETCH, 1);
    if (by_wave) {
        float all = top[0];
#pragma unroll
        for (int c = 1; c < STEPS; ++c) all = fmaxf(all, top[c]);
        const uint32_t largest = wave_bound<14>(sort_key(all), (kk + waves - 1) / waves);
        if (lane == 0) work[w] = (int)largest;
        parts = waves;
    } else {
        const int rounds = (kk + parts - 1) / parts;
        if (rounds > LI_WAVE) return 0u;
#pragma unroll
        for (int c = 0; c < STEPS; ++c) {
            const uint32_t largest = wave_bound<16>(sort_key(top[c]), rounds);
            if (lane == 0) work[STEPS * w + c] = (int)largest;
        }
    }
    __syncthreads();
    uint32_t bound = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < SMP_WAVES; ++i) bound = i < parts ? min(bound, (uint32_t)work[i] - 1u) : bound;      // (0, no bound, becomes the largest)
    return bound + 1u;
}

// A step's options, a row each: arrays on the device, or, up to N rows, in the launch's own arguments (which takes a copy to the device, its
// kernel and its event out of a step: SampleCall below).
struct SampleArrays {
    const float *temperature, *top_p, *uniform;
    const int* top_k;
};
template <int N>
struct SampleValues {
    float temperature[N], top_p[N], uniform[N];
    int top_k[N];
};

template <int STEPS, typename Options>
__global__ __launch_bounds__(TILE_NT<STEPS>, STEPS == 1 ? 8 : 5) void sample_tiles_kernel(
    const float* __restrict__ logits, const Options o, float* __restrict__ tile_m, float* __restrict__ tile_s,
    int* __restrict__ tile_i, float* __restrict__ cand_z, int* __restrict__ cand_id, int V) {
    constexpr int NT = TILE_NT<STEPS>, WAVES = TILE_WAVES<STEPS>, ITEMS = SMP_LIST / NT;
    __shared__ float sf[SMP_WAVES];
    __shared__ int si[SMP_WAVES];
    __shared__ int work_i[WAVES * 16], tot_i[16];
    __shared__ __align__(16) uint32_t list[SMP_LIST];
    __shared__ int list_id[SMP_LIST];
    const int tile = blockIdx.x, ntiles = gridDim.x, r = blockIdx.y, tid = threadIdx.x;
    const int lane = tid & (LI_WAVE - 1), w = tid / LI_WAVE;
    const float* row = logits + (size_t)r * V;
    const int j0 = tile * SMP_TILE + w * STEPS * TILE_STRETCH + lane * 8;
    const size_t slot = (size_t)r * ntiles + tile;
    const float T = o.temperature[r], p = o.top_p[r];
    const int k = o.top_k[r];
    float x[STEPS][8];                                         // the logits; past the end -inf
    const bool vec = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
#pragma unroll
    for (int c = 0; c < STEPS; ++c) load_ids8(row, j0 + c * TILE_STRETCH, V, vec, x[c]);
    if (!(T > 0.f)) {                                          // greedy: the tile's (maximum, lowest index)
        float v = -INFINITY;
        int i = 0x7fffffff;
#pragma unroll
        for (int c = 0; c < STEPS; ++c) {
            const int j = j0 + c * TILE_STRETCH;
            float vc = -INFINITY;
            int ic = 0x7fffffff;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (j + e < V && (x[c][e] > vc || ic == 0x7fffffff)) { vc = x[c][e]; ic = j + e; }
            argmax_combine(v, i, vc, ic);
        }
#pragma unroll
        for (int o = LI_WAVE / 2; o > 0; o >>= 1) argmax_combine(v, i, lane_xor(v, o), lane_xor(i, o));
        if (lane == 0) { sf[w] = v; si[w] = i; }
        __syncthreads();
        if (tid == 0) {
#pragma unroll
            for (int q = 1; q < WAVES; ++q) argmax_combine(v, i, sf[q], si[q]);
            tile_m[slot] = v;
            tile_i[slot] = i;
        }
        return;
    }
    float top[STEPS], m;                                       // (the largest quotient is the largest logit's)
#pragma unroll
    for (int c = 0; c < STEPS; ++c) {
        top[c] = x[c][0];
#pragma unroll
        for (int e = 1; e < 8; ++e) top[c] = fmaxf(top[c], x[c][e]);
    }
    m = top[0];
#pragma unroll
    for (int c = 1; c < STEPS; ++c) m = fmaxf(m, top[c]);
    m = wave_max(m);
    if (lane == 0) sf[w] = m;
    __syncthreads();
    m = sf[0];
#pragma unroll
    for (int i = 1; i < WAVES; ++i) m = fmaxf(m, sf[i]);
    m /= T;
    if (tid == 0) tile_m[slot] = m;
    const int kc = sample_candidates(k, p, V, ntiles);
    if (kc == 0 || !(k > 0 && k < V)) {                        // (behind top-k nothing is taken of the whole row's mass)
        // between 2^-40 and 2^40 in size, all of them: the bits without the sign, doubled, minus the bound's
        constexpr uint32_t LO = 2u * 0x2b800000u, HI = 2u * 0x53800000u;
        uint32_t off = (2u * __float_as_uint(T)) - LO;
#pragma unroll
        for (int c = 0; c < STEPS; ++c)
            if (j0 + c * TILE_STRETCH < V)
#pragma unroll
                for (int e = 0; e < 8; ++e) off = max(off, 2u * __float_as_uint(x[c][e]) - LO);
        const bool plain = __all(off <= HI - LO);
        const float y = 1.0f / T;
        float sum[STEPS];
        if (!(m > -INFINITY)) {                                // (a tile of -inf alone has no mass)
#pragma unroll
            for (int c = 0; c < STEPS; ++c) sum[c] = 0.f;
        } else if (plain) {                                    // (where ids end within a thread's eight, one of these is -inf: not plain)
#pragma unroll
            for (int c = 0; c < STEPS; ++c) {
                float e_of[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) e_of[e] = expf(quotient(x[c][e], T, y) - m);
                sum[c] = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) sum[c] += e_of[e];
                if (j0 + c * TILE_STRETCH >= V) sum[c] = 0.f;
            }
        } else {
            // (Masked logits come here.  64 rows of 151,936 ids, half of them -inf, at a temperature, both kernels: 22.6; as a loop that picks its value
            // from the registers 25.9, every stretch read once more 24.7; one row 11.7 / 12.6.)
#pragma unroll
            for (int c = 0; c < STEPS; ++c) {
                const int j = j0 + c * TILE_STRETCH;
                float z[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) z[e] = expf(x[c][e] / T - m);
                sum[c] = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) sum[c] += j + e < V ? z[e] : 0.f;
            }
        }
        __syncthreads();                                       // (sf has been read)
        tile_sums(sum, sf);
        __syncthreads();
        if (tid == 0) {
            float t = 0.f;
#pragma unroll
            for (int i = 0; i < SMP_WAVES; ++i) t += sf[i];
            tile_s[slot] = t;
        }
    }
    if (kc == 0) return;
    // The tile's kc largest ids, written in id order; or, where the second kernel has room for them, all from the bound on: these
    // hold the kc largest too, and finding exactly those takes as long again.  The bound is found among the logits.  Neighbouring
    // logits may have one quotient, three at most where it is no smaller than 2^-126, and ids of one quotient count by their number: so
    // all ids from a bound four places lower are taken.
    const int in_tile = min(SMP_TILE, V - tile * SMP_TILE);
    const size_t base = slot * SMP_KC;
    const bool all = in_tile <= kc;
    uint32_t tau = 0u;
    int need = 0x7fffffff, n[STEPS], place[STEPS];
    if (!all) {
        const bool wide = sample_wide(k, V, gridDim.y, ntiles);
        const uint32_t bound = tile_bound(top, kc, in_tile, si);
        const float from = bound > 4u ? key_value(bound - 4u) : -INFINITY;
        if (from > -INFINITY && fabsf(from / T) > 0x1p-120f) {
            // (by value, not by key: a zero more of the other sign does no harm.  A NaN counts as large)
            uint32_t mask = 0u;                                // bit 8 c + e
#pragma unroll
            for (int c = STEPS - 1; c >= 0; --c)
#pragma unroll
                for (int e = 7; e >= 0; --e) mask = (mask << 1) | (!(x[c][e] < from) ? 1u : 0u);
#pragma unroll
            for (int c = 0; c < STEPS; ++c) n[c] = __popc((mask >> (8 * c)) & 255u);
            const int total = tile_places(n, place, work_i);
            const bool direct = wide && total >= kc && total <= SMP_KC;
            if (direct || (total >= kc && total <= SMP_LIST)) {
                for (uint32_t left = mask; left; left &= left - 1u) {
                    const int i = __ffs((int)left) - 1, c = i >> 3, id = j0 + c * TILE_STRETCH + (i & 7);
                    const float z = row[id] / T;               // (once more from memory: a register cannot be chosen by number)
                    int at = place[0];
#pragma unroll
                    for (int q = 1; q < STEPS; ++q) at = c == q ? place[q] : at;
                    at += __popc(mask & ((1u << i) - 1u) & (255u << (8 * c)));
                    if (direct) { cand_z[base + at] = z; cand_id[base + at] = id; }
                    else { list[at] = sort_key(z); list_id[at] = id; }
                }
                if (direct) {
                    if (tid == 0) tile_i[slot] = total;
                    return;
                }
                kth_of_list<NT>(list, total, kc, tau, need, tot_i);
                // of the list, in its order: the keys above tau and the first `need` equal to it; a thread has the next ITEMS
                uint32_t key[ITEMS];
                int eq = 0, mine = 0;
#pragma unroll
                for (int e = 0; e < ITEMS; ++e) {
                    key[e] = tid * ITEMS + e < total ? list[tid * ITEMS + e] : 0u;      // (no key of a number)
                    eq += key[e] == tau;
                }
                const int rank0 = block_sum_before<WAVES>(eq, work_i);
                int rank = rank0;
#pragma unroll
                for (int e = 0; e < ITEMS; ++e) mine += key[e] > tau || (key[e] == tau && rank++ < need);
                int pos = block_sum_before<WAVES>(mine, work_i);
                if (tid == NT - 1) tile_i[slot] = pos + mine;
                rank = rank0;
#pragma unroll
                for (int e = 0; e < ITEMS; ++e)
                    if (key[e] > tau || (key[e] == tau && rank++ < need)) {
                        cand_z[base + pos] = key_value(key[e]);
                        cand_id[base + pos] = list_id[tid * ITEMS + e];
                        ++pos;
                    }
                return;
            }
        }
        __syncthreads();                                       // (work_i has been read)
    }
    // in general: among the quotients
#pragma unroll
    for (int c = 0; c < STEPS; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[c][e] /= T;
    if (!all) {
        // Of masked logits a tile may have fewer than kc above its lowest, which then is the kc-th; and where masked ids follow each other, the bound of
        // tile_bound comes from those stretches in which every lane has a value above the lowest.  (Four bits a pass over 32 values a thread are
        // the longest way: 64 rows of top-k with top-p, the first kernel, all but one id in a thousand masked 142 -> 63, the upper half masked 103 -> 67.)
        uint32_t lowest = 0xffffffffu;
#pragma unroll
        for (int c = 0; c < STEPS; ++c)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (j0 + c * TILE_STRETCH + e < V) lowest = min(lowest, sort_key(x[c][e]));
#pragma unroll
        for (int o = LI_WAVE / 2; o > 0; o >>= 1) lowest = min(lowest, (uint32_t)__shfl_xor((int)lowest, o, LI_WAVE));
        if (lane == 0) work_i[w] = (int)lowest;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < WAVES; ++i) lowest = min(lowest, (uint32_t)work_i[i]);
#pragma unroll
        for (int c = 0; c < STEPS; ++c) {
            n[c] = 0;
#pragma unroll
            for (int e = 0; e < 8; ++e) n[c] += (j0 + c * TILE_STRETCH + e < V) && sort_key(x[c][e]) > lowest;
        }
        const int above = tile_places(n, place, si);
        bool found = above < kc;
        if (found) {
            tau = lowest;
            need = kc - above;
        } else {
            uint32_t key[STEPS];
            int whole = 0;
#pragma unroll
            for (int c = 0; c < STEPS; ++c) {
                key[c] = 0u;
#pragma unroll
                for (int e = 0; e < 8; ++e) key[c] = max(key[c], sort_key(x[c][e]));
                const bool takes = __all(j0 + c * TILE_STRETCH + 8 <= V && key[c] > lowest);
                key[c] = takes ? key[c] : 0xffffffffu;
                whole += takes;
            }
            if (lane == 0) work_i[w] = whole;
            __syncthreads();
            whole = 0;
#pragma unroll
            for (int i = 0; i < WAVES; ++i) whole += work_i[i];
            const int rounds = whole ? (kc + whole - 1) / whole : LI_WAVE + 1;
            if (rounds <= LI_WAVE) {
                uint32_t bound = 0xffffffffu;
#pragma unroll
                for (int c = 0; c < STEPS; ++c) bound = min(bound, wave_bound<16>(key[c], rounds));
                __syncthreads();                               // (work_i has been read)
                if (lane == 0) work_i[w] = (int)bound;
                __syncthreads();
#pragma unroll
                for (int i = 0; i < WAVES; ++i) bound = min(bound, (uint32_t)work_i[i]);
#pragma unroll
                for (int c = 0; c < STEPS; ++c) {
                    n[c] = 0;
#pragma unroll
                    for (int e = 0; e < 8; ++e) n[c] += (j0 + c * TILE_STRETCH + e < V) && sort_key(x[c][e]) >= bound;
                }
                const int total = tile_places(n, place, si);
                found = total <= SMP_LIST;
                if (found) {
#pragma unroll
                    for (int c = 0; c < STEPS; ++c)
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            if ((j0 + c * TILE_STRETCH + e < V) && sort_key(x[c][e]) >= bound) list[place[c]++] = sort_key(x[c][e]);
                    kth_of_list<NT>(list, total, kc, tau, need, tot_i);
                }
            }
        }
        if (!found)
            radix_kth<WAVES>([&](auto f) {
#pragma unroll
                for (int c = 0; c < STEPS; ++c)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (j0 + c * TILE_STRETCH + e < V) f(x[c][e]);
            }, kc, tau, need, work_i, tot_i);
    }
    int rank[STEPS];
#pragma unroll
    for (int c = 0; c < STEPS; ++c) {
        n[c] = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) n[c] += (j0 + c * TILE_STRETCH + e < V) && sort_key(x[c][e]) == tau;
        rank[c] = 0;
    }
    if (!all) tile_places(n, rank, si);
    auto in = [&](int c, int e, int& place_at_tau) {
        const uint32_t key = sort_key(x[c][e]);
        return (j0 + c * TILE_STRETCH + e < V) && (all || key > tau || (key == tau && place_at_tau++ < need));
    };
#pragma unroll
    for (int c = 0; c < STEPS; ++c) {
        n[c] = 0;
        int at = rank[c];
#pragma unroll
        for (int e = 0; e < 8; ++e) n[c] += in(c, e, at);
    }
    const int total = tile_places(n, place, si);
    if (tid == 0) tile_i[slot] = total;
#pragma unroll
    for (int c = 0; c < STEPS; ++c) {
        int at = rank[c];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (in(c, e, at)) {
                cand_z[base + place[c]] = x[c][e];
                cand_id[base + place[c]] = j0 + c * TILE_STRETCH + e;
                ++place[c];
            }
    }
}

// Inverse CDF over the survivors in a list (keys above tau and the first `need` equal to it), in id order: the first wave alone, a lane the
// `per` next ones.
template <typename Choose>
__device__ __forceinline__ void pick_of_list(const uint32_t* list, const int* list_id, int n, uint32_t tau, int need, float m, float u, Choose&& choose) {
    if (threadIdx.x >= LI_WAVE) return;
    const int lane = threadIdx.x;
    const int per = (n + LI_WAVE - 1) / LI_WAVE, from = lane * per, to = min(from + per, n);
    int eq = 0;
    for (int j = from; j < to; ++j) eq += list[j] == tau;
    int rank0 = eq;
#pragma unroll
    for (int o = 1; o < LI_WAVE; o <<= 1) {
        const int t = __shfl_up(rank0, o, LI_WAVE);
        if (lane >= o) rank0 += t;
    }
    rank0 -= eq;                            // keys at tau before this lane's
    auto in = [&](int j, int& rank) { return list[j] > tau || (list[j] == tau && rank++ < need); };
    float mine = 0.f;
    bool any = false;
    for (int j = from, rank = rank0; j < to; ++j)
        if (in(j, rank)) { mine += expf(key_value(list[j]) - m); any = true; }
    float upto = mine;
#pragma unroll
    for (int o = 1; o < LI_WAVE; o <<= 1) {
        const float t = __shfl_up(upto, o, LI_WAVE);
        if (lane >= o) upto += t;
    }
    float run = __shfl_up(upto, 1, LI_WAVE);
    if (lane == 0) run = 0.f;
    const float target = u * __shfl(upto, LI_WAVE - 1, LI_WAVE);
    const unsigned long long reach = __ballot(any && run + mine >= target), some = __ballot(any);
    const int chosen = reach ? __ffsll((long long)reach) - 1 : 63 - __clzll((long long)some);      // (else the last one with a survivor)
    if (lane == chosen) {
        int pick = -1;
        for (int j = from, rank = rank0; j < to; ++j) {
            if (!in(j, rank)) continue;
            pick = list_id[j];
            run += expf(key_value(list[j]) - m);
            if (run >= target) break;
        }
        choose(pick);
    }
}

// A row with top-k (and top-p) whose tiles handed over up to SMP_KC ids each (sample_wide), from the candidates to the token; false, with nothing
// done, where the general way has to be taken.  The same as select_kth, mass_of_list and pick_of_list one after the other, in fewer and
// shorter steps: a wave takes the candidates of one tile or two (asked for with the tiles' counts, before these are known), so that places in the
// list come from ballots; and the list is held against itself once, by four threads a key (each the entries whose number is its
// own modulo four), for the number and the mass above it and from it on together: the masses above tau need no tau.
// Top-k 50 with top-p 0.9, the rows kernel: 64 rows of 151,936 ids 18.2 -> 10.4 us, one row 13.9 -> 9.2.
template <typename Choose>
__device__ __forceinline__ bool rows_by_list(const float* cand_z, const int* cand_id, const int* tile_i, int ntiles, int k, float p, int V, float m, float u, Choose&& choose,
                                             uint32_t* list, float* list_e, int* list_id, int* work_i, int* counts, float* res_f, int* res) {
    constexpr int HOLD = SMP_KC / LI_WAVE, TILES = 2;            // (up to 32 tiles: sample_wide)
    const int tid = threadIdx.x, lane = tid & (LI_WAVE - 1), w = __builtin_amdgcn_readfirstlane(tid / LI_WAVE);
    const int full = V - (ntiles - 1) * SMP_TILE >= k ? ntiles : ntiles - 1;       // tiles with at least k candidates
    const int parts = min(full, SMP_WAVES), rounds = parts > 0 ? (k + parts - 1) / parts : 0;
    if (parts == 0 || rounds > LI_WAVE) return false;
    float z[TILES][HOLD];
    int id[TILES][HOLD], held[TILES];
    uint32_t key[TILES][HOLD];
#pragma unroll
    for (int h = 0; h < TILES; ++h) {
        const int t = w + h * SMP_WAVES;
        held[h] = 0;
        if (t < ntiles) {
            held[h] = tile_i[t];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                z[h][c] = cand_z[t * SMP_KC + c * LI_WAVE + lane];
                id[h][c] = cand_id[t * SMP_KC + c * LI_WAVE + lane];
            }
        }
    }
    uint32_t most = 0u;
#pragma unroll
    for (int h = 0; h < TILES; ++h) {
        const int t = w + h * SMP_WAVES;
        if (held[h] > 2 * LI_WAVE)
#pragma unroll
            for (int c = 2; c < HOLD; ++c) {
                z[h][c] = cand_z[t * SMP_KC + c * LI_WAVE + lane];
                id[h][c] = cand_id[t * SMP_KC + c * LI_WAVE + lane];
            }
#pragma unroll
        for (int c = 0; c < HOLD; ++c) {
            key[h][c] = c * LI_WAVE + lane < held[h] ? sort_key(z[h][c]) : 0u;
            most = max(most, key[h][c]);
        }
    }
    const uint32_t largest = wave_bound<16>(most, rounds);
    if (lane == 0) work_i[w] = (int)largest;
    if (tid == 0) res[0] = 0;
    __syncthreads();
    uint32_t bound = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < SMP_WAVES; ++i) bound = i < parts ? min(bound, (uint32_t)work_i[i] - 1u) : bound;
    bound += 1u;                                                // (0, no bound, became the largest)
    if (bound == 0u) return false;
    unsigned long long in[TILES][HOLD];
#pragma unroll
    for (int h = 0; h < TILES; ++h) {
        int n = 0;
#pragma unroll
        for (int c = 0; c < HOLD; ++c) { in[h][c] = __ballot(key[h][c] >= bound); n += __popcll(in[h][c]); }
        if (lane == 0) counts[w + h * SMP_WAVES] = n;
    }
    __syncthreads();
    const int own = lane < TILES * SMP_WAVES ? counts[lane] : 0;
    auto sum = [](int v) {
#pragma unroll
        for (int o = 1; o < LI_WAVE; o <<= 1) v += lane_xor(v, o);
        return __builtin_amdgcn_readfirstlane(v);
    };
    const int n = sum(own);
    if (n > SMP_LIST) return false;
#pragma unroll
    for (int h = 0; h < TILES; ++h) {
        if (w + h * SMP_WAVES >= ntiles) continue;
        int at = sum(lane < w + h * SMP_WAVES ? own : 0);
#pragma unroll
        for (int c = 0; c < HOLD; ++c) {
            if (!in[h][c]) continue;
            if (key[h][c] >= bound) {
                const int place = at + __builtin_amdgcn_mbcnt_hi((uint32_t)(in[h][c] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)in[h][c], 0));
                list[place] = key[h][c];
                list_id[place] = id[h][c];
                list_e[place] = expf(z[h][c] - m);
            }
            at += __popcll(in[h][c]);
        }
    }
    __syncthreads();
    constexpr int TURNS = 4 * SMP_LIST / SMP_NT;
    uint32_t mykey[TURNS];
    float above_e[TURNS], from_e[TURNS];
#pragma unroll
    for (int q = 0; q < TURNS; ++q) {
        const int i = (tid >> 2) + q * (SMP_NT / 4);
        mykey[q] = 0u;
        if (q * (SMP_NT / 4) >= n) continue;                    // (the same for all threads)
        mykey[q] = i < n ? list[i] : 0u;
        int above = 0, from = 0;
        float ga = 0.f, gf = 0.f;
#pragma unroll 8
        for (int j = tid & 3; j < n; j += 4) {
            const uint32_t v = list[j];
            const float e = list_e[j];
            above += v > mykey[q];
            from += v >= mykey[q];
            ga += v > mykey[q] ? e : 0.f;
            gf += v >= mykey[q] ? e : 0.f;
        }
        above += lane_xor(above, 1); above += lane_xor(above, 2);
        from += lane_xor(from, 1); from += lane_xor(from, 2);
        above_e[q] = lane_xor_add(lane_xor_add(ga, 1), 2);
        from_e[q] = lane_xor_add(lane_xor_add(gf, 1), 2);
        if (i < n && above < k && from >= k) {                  // (all threads with this key write the same)
            res[1] = (int)mykey[q];
            res[2] = k - above;
            res_f[0] = above_e[q];
        }
    }
    __syncthreads();
    uint32_t tau = (uint32_t)res[1];
    int need = res[2];
    if (p > 0.f && p < 1.f) {
        const float mass = res_f[0], e_ties = (float)need * expf(key_value(tau) - m), want = p * (mass + e_ties);
#pragma unroll
        for (int q = 0; q < TURNS; ++q) {
            if (mykey[q] < tau || mykey[q] == 0u) continue;
            if (mykey[q] > tau ? above_e[q] < want && from_e[q] >= want : mass < want && mass + e_ties >= want) {
                res[0] = 1;
                res[3] = (int)mykey[q];
                res_f[1] = want - (mykey[q] > tau ? above_e[q] : mass);
            }
        }
        __syncthreads();
        if (!res[0]) return false;                              // (rounding, or masses of zero)
        const uint32_t tp = (uint32_t)res[3];
        const int need_p = ties_needed(res_f[1], tp, m);
        need = tp == tau ? min(need, need_p) : need_p;
        tau = tp;
    }
    pick_of_list(list, list_id, n, tau, need, m, u, choose);
    return true;
}

// tile_m, tile_s, tile_i, cand_z, cand_id: what sample_tiles_kernel left for the row's ntiles tiles (ntiles <= SMP_NT)
// out: [rows] on the device; host (may be null): the same ids once more, in memory of the host that the device can write
template <typename Options>
__global__ __launch_bounds__(SMP_NT) void sample_rows_kernel(
    const float* __restrict__ logits, const Options o, int* __restrict__ out, int* __restrict__ host, int V,
    const float* __restrict__ tile_m, const float* __restrict__ tile_s, const int* __restrict__ tile_i,
    const float* __restrict__ cand_z, const int* __restrict__ cand_id, int ntiles) {
    __shared__ float sf[SMP_WAVES];
    __shared__ int si[SMP_WAVES];
    __shared__ float tile_sum[SMP_NT];               // the survivors' mass of every tile
    __shared__ int ties_before[SMP_NT];              // ids at the threshold before every tile
    __shared__ float work_f[SMP_WAVES * 16], tot_f[16];
    __shared__ int work_i[SMP_WAVES * 16], tot_i[16];
    __shared__ __align__(16) uint32_t list[SMP_LIST];
    __shared__ __align__(16) float list_e[SMP_LIST];
    __shared__ int list_id[SMP_LIST];
    __shared__ float pick_f[3];
    __shared__ int pick_i[1];
    const int r = blockIdx.x, tid = threadIdx.x;
    const float* row = logits + (size_t)r * V;
    const float T = o.temperature[r], p = o.top_p[r], u = o.uniform[r];      // (together: one trip to memory)
    const int k = o.top_k[r];
    auto choose = [&](int id) {
        out[r] = id;
        if (host) host[r] = id;
    };
    tile_m += (size_t)r * ntiles;
    tile_s += (size_t)r * ntiles;
    tile_i += (size_t)r * ntiles;
    if (!(T > 0.f)) {                                          // greedy: the tiles' maxima, ties to the lower id
        if (tid >= LI_WAVE) return;
        float v = -INFINITY;
        int i = 0x7fffffff;
        for (int t = tid; t < ntiles; t += LI_WAVE) argmax_combine(v, i, tile_m[t], tile_i[t]);
#pragma unroll
        for (int o = LI_WAVE / 2; o > 0; o >>= 1) argmax_combine(v, i, lane_xor(v, o), lane_xor(i, o));
        if (tid == 0) choose(i);
        return;
    }
    const bool vec = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
    const bool filtered = !sample_unfiltered(k, p, V);
    const bool by_k = k > 0 && k < V, by_p = p > 0.f && p < 1.f;

    // The survivors are the ids with key > tau and the first `need` (in id order) of those with key == tau.
    bool cut = false;
    uint32_t tau = 0u;
    int need = 0x7fffffff;
    float m = -INFINITY;                              // the maximum that masses are taken against
    if (filtered) {
        for (int t = tid & (LI_WAVE - 1); t < ntiles; t += LI_WAVE) m = fmaxf(m, tile_m[t]);
        m = wave_max(m);
    }

    const int kc = sample_candidates(k, p, V, ntiles);
    if (kc > 0 && by_k && sample_wide(k, V, gridDim.x, ntiles)) {
        const size_t at = (size_t)r * ntiles * SMP_KC;
        if (rows_by_list(cand_z + at, cand_id + at, tile_i, ntiles, k, p, V, m, u, choose, list, list_e, list_id, work_i, ties_before, pick_f, tot_i)) return;
        __syncthreads();
    }
    if (kc > 0) {
        // ---- among the candidates, in ascending ids: thread t has the C of them from t * C on
        float cz[SMP_CAND_PER_THREAD];
        int cid[SMP_CAND_PER_THREAD];
        bool have[SMP_CAND_PER_THREAD];
        const int lane = tid & (LI_WAVE - 1);
        int total, first = 0;                       // candidates in all; those of the tiles before tile `lane` (where the tiles hold different numbers)
        const bool wide = sample_wide(k, V, gridDim.x, ntiles);
        if (wide) {                                 // (up to 32 tiles: a lane each)
            const int count = lane < ntiles ? tile_i[lane] : 0;
            int upto = count;
#pragma unroll
            for (int o = 1; o < LI_WAVE; o <<= 1) {
                const int t = __shfl_up(upto, o, LI_WAVE);
                if (lane >= o) upto += t;
            }
            first = upto - count;
            total = __shfl(upto, LI_WAVE - 1, LI_WAVE);
        } else {
            total = (ntiles - 1) * kc + min(kc, V - (ntiles - 1) * SMP_TILE);      // (kc < SMP_TILE)
        }
        const int C = (total + SMP_NT - 1) / SMP_NT;
#pragma unroll
        for (int c = 0; c < SMP_CAND_PER_THREAD; ++c) {
            const int s = tid * C + c;
            have[c] = c < C && s < total;
            int t = 0, i = s;
            if (wide) {
                if (c < C) {                        // (the same for all threads) the last tile that begins at s or before it
                    for (int step = 16; step > 0; step >>= 1)
                        if (__shfl(first, t + step, LI_WAVE) <= s && t + step < ntiles) t += step;
                    i = s - __shfl(first, t, LI_WAVE);
                }
            } else {
                t = min(s / kc, ntiles - 1);
                i = s - t * kc;
            }
            cz[c] = -INFINITY;
            cid[c] = 0;
            if (have[c]) {
                const size_t at = ((size_t)r * ntiles + t) * SMP_KC + i;
                cz[c] = cand_z[at];
                cid[c] = cand_id[at];
            }
        }
        auto each = [&](auto f) {
#pragma unroll
            for (int c = 0; c < SMP_CAND_PER_THREAD; ++c)
                if (have[c]) f(cz[c]);
        };
        // the k-th largest (top-k), or the kc-th: above it the candidates are all there is
        uint32_t tau_c;
        int need_c;
        uint32_t key[SMP_CAND_PER_THREAD];
#pragma unroll
        for (int c = 0; c < SMP_CAND_PER_THREAD; ++c) key[c] = have[c] ? sort_key(cz[c]) : 0u;
        const int kk = min(by_k ? k : kc, total);
        const int threads = (total + C - 1) / C;
        int n = 0;
        const bool listed = select_kth(key, kk, max(threads / LI_WAVE, 1), tau_c, need_c, list, list_id, n, work_i, tot_i, [&](int e) { return cid[e]; });
        if (!listed) radix_kth(each, kk, tau_c, need_c, work_i, tot_i);
        bool exact = true, done = false;
        if (by_k) { cut = true; tau = tau_c; need = need_c; }
        if (by_p && by_k && listed) {
            // (of the candidates equal to tau, which the list holds all, `need` count)
            float remaining;
            uint32_t tp;
            if (mass_of_list(list, n, tau, need, m, p, remaining, tp, list_e, pick_f, tot_i)) {
                const int need_p = ties_needed(remaining, tp, m);
                need = tp == tau ? min(need, need_p) : need_p;
                tau = tp;
                done = true;
            }
        }
        if (by_k && listed && (done || !by_p)) {
            pick_of_list(list, list_id, n, tau, need, m, u, choose);
            return;
        }
        if (by_p && !done) {
            float zk = 0.f;
            int eq = 0;
            each([&](float z) {
                const uint32_t key = sort_key(z);
                if (!cut || key > tau) zk += expf(z - m);
                else if (key == tau) ++eq;
            });
            zk = block_sum<SMP_NT>(zk, sf);
            const int ties = cut ? min(need, block_sum_int(eq, si)) : 0;
            const float e_ties = cut ? (float)ties * expf(key_value(tau) - m) : 0.f;
            if (!cut && total < V) {                  // the mass of all ids, from the tiles' sums
                zk = 0.f;
                for (int t = 0; t < ntiles; ++t) zk += tile_s[t] * expf(tile_m[t] - m);
            }
            float remaining = p * (zk + e_ties);
            uint32_t tp;
            radix_mass<true>(each, cut, tau, ties, e_ties, m, remaining, tp, work_f, tot_f, tot_i);
            if (!by_k && total < V && !(tp > tau_c)) exact = false;       // the prefix may go on beyond the candidates
            const int need_p = ties_needed(remaining, tp, m);
            need = (cut && tp == tau) ? min(need, need_p) : need_p;
            tau = tp;
            cut = true;
        }
        if (exact) {
            // inverse CDF over the surviving candidates in id order
            int eq = 0;
            each([&](float z) { eq += sort_key(z) == tau; });
            const bool ranked = block_sum_int(eq, si) > need;
            const int rank0 = ranked ? block_sum_before(eq, work_i) : 0;
            float mine = 0.f;
            bool any = false;
            {
                int rank = rank0;
#pragma unroll
                for (int c = 0; c < SMP_CAND_PER_THREAD; ++c) {
                    if (!have[c]) continue;
                    const uint32_t key = sort_key(cz[c]);
                    if (key > tau || (key == tau && (!ranked || rank++ < need))) { mine += expf(cz[c] - m); any = true; }
                }
            }
            const float run0 = block_sum_before(mine, work_f);
            if (tid == SMP_NT - 1) pick_f[0] = u * (run0 + mine);
            __syncthreads();
            const float target = pick_f[0];
            int chosen = block_min_int((any && run0 + mine >= target) ? tid : 0x7fffffff, si);
            if (chosen == 0x7fffffff) chosen = -block_min_int(any ? -tid : 1, si);
            if (tid == chosen) {
                float run = run0;
                int rank = rank0, pick = cid[0];
#pragma unroll
                for (int c = 0; c < SMP_CAND_PER_THREAD; ++c) {
                    if (!have[c]) continue;
                    const uint32_t key = sort_key(cz[c]);
                    if (!(key > tau || (key == tau && (!ranked || rank++ < need)))) continue;
                    pick = cid[c];
                    run += expf(cz[c] - m);
                    if (run >= target) break;
                }
                choose(pick);
            }
            return;
        }
        cut = false;                                  // from the row itself, then
        tau = 0u;
        need = 0x7fffffff;
    }

    int tile = 0;                                     // the tile that holds the target,
    float before = 0.f, target = 0.f;                 // the mass before it and the target, in units of exp(z - m)
    auto each_of_row = [&](auto f) { each_id(row, V, T, vec, ntiles, [&](float z, int) { f(z); }); };
    if (filtered) {
        if (by_k) {
            cut = true;
            radix_kth(each_of_row, k, tau, need, work_i, tot_i);
        }
        if (by_p) {
            // mass of the top-k survivors, and how many ids sit at tau
            float zk = 0.f;
            int eq = 0;
            each_of_row([&](float z) {
                const uint32_t key = sort_key(z);
                if (!cut || key > tau) zk += expf(z - m);
                else if (key == tau) ++eq;
            });
            zk = block_sum<SMP_NT>(zk, sf);
            const int ties = cut ? min(need, block_sum_int(eq, si)) : 0;
            const float e_ties = cut ? (float)ties * expf(key_value(tau) - m) : 0.f;
            float remaining = p * (zk + e_ties);      // mass that the prefix has to reach
            uint32_t tp;
            radix_mass<false>(each_of_row, cut, tau, ties, e_ties, m, remaining, tp, work_f, tot_f, tot_i);
            const int need_p = ties_needed(remaining, tp, m);
            need = (cut && tp == tau) ? min(need, need_p) : need_p;
            tau = tp;
            cut = true;
        }
    }

    // ---- inverse CDF over ascending ids among the survivors
    // Are there more ids at tau than count?  Then an id's place among them decides (ties_before).
    bool ranked = false;
    if (cut) {
        int eq = 0;
        each_of_row([&](float z) { eq += sort_key(z) == tau; });
        ranked = block_sum_int(eq, si) > need;
        if (ranked) {
            int running = 0;
            for (int t = 0; t < ntiles; ++t) {
                const int j0 = t * SMP_TILE + tid * 8;
                float z[8];
                int c = 0;
                if (j0 < V) {
                    load_ids8(row, j0, V, T, vec, z);
#pragma unroll
                    for (int e = 0; e < 8; ++e) c += (j0 + e < V) && sort_key(z[e]) == tau;
                }
                c = block_sum_int(c, si);
                if (tid == 0) ties_before[t] = running;
                running += c;
            }
            __syncthreads();
        }
    }
    // this thread's ids of a tile: their mass (sum in id order), whether any survives, and the place
    // among the ids at tau of its first one
    auto mine_of = [&](int t, bool& any, int& rank0, float (&z)[8]) {
        const int j0 = t * SMP_TILE + tid * 8;
        any = false;
        rank0 = 0;
        if (j0 < V) load_ids8(row, j0, V, T, vec, z);
        if (ranked) {
            int c = 0;
            if (j0 < V) {
#pragma unroll
                for (int e = 0; e < 8; ++e) c += (j0 + e < V) && sort_key(z[e]) == tau;
            }
            rank0 = ties_before[t] + block_sum_before(c, work_i);
        }
        float sum = 0.f;
        if (j0 < V) {
            int rank = rank0;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (j0 + e >= V) continue;
                const uint32_t key = sort_key(z[e]);
                const bool in = !cut || key > tau || (key == tau && (!ranked || rank++ < need));
                if (in) { sum += expf(z[e] - m); any = true; }
            }
        }
        return sum;
    };
    if (!filtered) {
        // The tiles' sums are there, each against its tile's own maximum: brought to the row's maximum
        // they give the tile that holds the target; within it the search goes on in the tile's own scale.
        auto look = [&](auto sum_of, float top) {
            float total = 0.f;
            for (int t = 0; t < ntiles; ++t) total += sum_of(t);
            const float want = u * total;
            float run = 0.f;
            int pick = -1, last = 0;                 // (a tile far below the maximum has no mass at all in float32)
            for (int t = 0; t < ntiles; ++t) {
                const float w = sum_of(t);
                if (w > 0.f) last = t;
                if (w > 0.f && run + w >= want) { pick = t; break; }
                run += w;
            }
            const bool past = pick < 0;              // rounding left the target just above the total:
            tile = past ? last : pick;               // the last id with mass (no sum reaches infinity below)
            m = tile_m[tile];
            target = past ? INFINITY : (want - run) / expf(m - top);
        };
        if (ntiles <= LI_WAVE) {                     // every wave by itself, a lane a tile: no barrier
            const int lane = tid & (LI_WAVE - 1), t = lane < ntiles ? lane : 0;
            const float own = tile_m[t], own_s = tile_s[t], top = wave_max(own);
            const int sum = __float_as_int(lane < ntiles ? own_s * expf(own - top) : 0.f);
            look([&](int i) { return __int_as_float(__builtin_amdgcn_readlane(sum, i)); }, top);
        } else {
            float top = -INFINITY;
            for (int t = tid & (LI_WAVE - 1); t < ntiles; t += LI_WAVE) top = fmaxf(top, tile_m[t]);
            top = wave_max(top);
            for (int t = tid; t < ntiles; t += SMP_NT) tile_sum[t] = tile_s[t] * expf(tile_m[t] - top);
            __syncthreads();
            look([&](int i) { return tile_sum[i]; }, top);
        }
    } else {
        for (int t = 0; t < ntiles; ++t) {
            bool any;
            int rank0;
            float z[8];
            const float ts = block_sum<SMP_NT>(mine_of(t, any, rank0, z), sf);
            if (tid == 0) tile_sum[t] = ts;
        }
        __syncthreads();
        if (tid == 0) {
            float total = 0.f;
            for (int t = 0; t < ntiles; ++t) total += tile_sum[t];
            const float want = u * total;
            float run = 0.f;
            int pick = -1, last = 0;
            for (int t = 0; t < ntiles; ++t) {
                if (tile_sum[t] > 0.f) last = t;
                if (tile_sum[t] > 0.f && run + tile_sum[t] >= want) { pick = t; break; }
                run += tile_sum[t];
            }
            const bool past = pick < 0;
            if (past) pick = last;
            pick_i[0] = pick;
            pick_f[0] = past ? 0.f : run;
            pick_f[1] = past ? INFINITY : want;
        }
        __syncthreads();
        tile = pick_i[0];
        before = pick_f[0];
        target = pick_f[1];
    }
    // within the tile: the first thread whose ids bring the running sum to the target, else the last one with a survivor
    bool any;
    int rank0;
    float z[8];
    const float mine = mine_of(tile, any, rank0, z);
    const float run0 = before + block_sum_before(mine, work_f);
    int chosen = block_min_int((any && run0 + mine >= target) ? tid : 0x7fffffff, si);
    if (chosen == 0x7fffffff) chosen = -block_min_int(any ? -tid : 1, si);     // (the tile has a survivor: its sum is above zero)
    if (tid == chosen) {
        const int j0 = tile * SMP_TILE + tid * 8;
        float run = run0;
        int rank = rank0, pick = j0;
        bool done = false;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t key = sort_key(z[e]);
            const bool in = !done && j0 + e < V && (!cut || key > tau || (key == tau && (!ranked || rank++ < need)));
            if (!in) continue;
            pick = j0 + e;
            run += expf(z[e] - m);
            done = run >= target;
        }
        choose(pick);
    }
}

// ------------------------------------------------- sampling state of the live requests, on the device
// One row of eight 32-bit words for every state slot of the cache: {temperature, top_p (float bits), top_k,
// seed low, seed high, draws so far, 0, 0}.  The host writes a row when a request is bound to its slot and
// never again; the device counts the draws.  (The reference keeps the same per sequence on the host:
// src/llaisys/models/qwen2.hpp:100-110.)
//
// li_sample_prepare turns the rows of a step, given as slot | flags << 24 (flag 1: this row is greedy
// whatever its slot says, e.g. a request's first token), into the per-row arrays that li_sample_rows takes:
// temperature, top_k, top_p and the uniform number of the slot's next draw, the draws-th number of the
// stream `seed`: a splitmix64 hash of both, its upper 24 bits as a value in [0, 1).  A row that samples
// (temperature > 0) advances its slot's count.  A slot outside the table gives a greedy row.
#define SAMPLE_SLOT_WORDS 8
__host__ __device__ __forceinline__ float stream_uniform(unsigned long long seed, unsigned long long counter) {
    unsigned long long z = seed * 0x9E3779B97F4A7C15ull + (counter + 1ull) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (float)(z >> 40) * (1.0f / 16777216.0f);
}

__global__ void sample_prepare_kernel(const int* __restrict__ rows, int n, int* __restrict__ table, int nslots,
                                      float* __restrict__ temperature, int* __restrict__ top_k,
                                      float* __restrict__ top_p, float* __restrict__ uniform) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int slot = rows[i] & 0xffffff, flags = (rows[i] >> 24) & 0x7f;
    float T = 0.f, P = 1.f, U = 0.f;
    int K = 0;
    if (slot < nslots && !(flags & 1)) {
        int* row = table + (size_t)slot * SAMPLE_SLOT_WORDS;
        T = __int_as_float(row[0]);
        P = __int_as_float(row[1]);
        K = row[2];
        if (T > 0.f) {
            const unsigned long long seed = (unsigned long long)(unsigned)row[3] | ((unsigned long long)(unsigned)row[4] << 32);
            const int draws = row[5];
            U = stream_uniform(seed, (unsigned long long)(unsigned)draws);
            row[5] = draws + 1;                      // (a slot stands once in a step's rows: no two threads write it)
        } else {
            T = 0.f;
        }
    }
    temperature[i] = T; top_k[i] = K; top_p[i] = P; uniform[i] = U;
}

extern "C" int li_sample_prepare(const int* rows, int n, int* table, int nslots, float* temperature, int* top_k,
                                 float* top_p, float* uniform, hipStream_t stream) {
    if (n <= 0 || nslots <= 0 || !rows || !table) return LI_ERR_SIZE;
    sample_prepare_kernel<<<(n + 255) / 256, 256, 0, stream>>>(rows, n, table, nslots, temperature, top_k, top_p, uniform);
    return li_launch_status();
}

// Floats of scratch memory that li_sample_rows needs for n rows of V logits.
extern "C" long li_sample_rows_scratch_floats(int n, int V) {
    if (n <= 0 || V <= 0) return 0;
    const long ntiles = (V + SMP_TILE - 1) / SMP_TILE;
    return (3 + 2 * (long)SMP_KC) * n * ntiles;
}

// tiles: scratch of li_sample_rows_scratch_floats(n, V) floats, in which the first kernel leaves every tile's part.
template <typename Options>
static int launch_sample(const float* logits, const Options& o, int* out, int* host, int n, int V, float* tiles, long tiles_floats, hipStream_t stream) {
    if (n <= 0 || n > 65535 || V <= 0) return LI_ERR_SIZE;
    const int ntiles = (V + SMP_TILE - 1) / SMP_TILE;
    if (ntiles > SMP_NT || !tiles || tiles_floats < li_sample_rows_scratch_floats(n, V)) return LI_ERR_SIZE;
    const size_t per = (size_t)n * ntiles;
    float* tm = tiles;
    float* ts = tiles + per;
    int* ti = reinterpret_cast<int*>(tiles + 2 * per);
    float* cz = tiles + 3 * per;
    int* ci = reinterpret_cast<int*>(tiles + (3 + (size_t)SMP_KC) * per);
    const dim3 grid(ntiles, n);
    if (per >= TILE_MANY) sample_tiles_kernel<4, Options><<<grid, TILE_NT<4>, 0, stream>>>(logits, o, tm, ts, ti, cz, ci, V);
    else sample_tiles_kernel<1, Options><<<grid, TILE_NT<1>, 0, stream>>>(logits, o, tm, ts, ti, cz, ci, V);
    sample_rows_kernel<Options><<<n, SMP_NT, 0, stream>>>(logits, o, out, host, V, tm, ts, ti, cz, ci, ntiles);
    return li_launch_status();
}

extern "C" int li_sample_rows(const float* logits, const float* temperature, const int* top_k,
                              const float* top_p, const float* uniform, int* out, int n, int V,
                              float* tiles, long tiles_floats, hipStream_t stream) {
    return launch_sample(logits, SampleArrays{temperature, top_p, uniform, top_k}, out, nullptr, n, V, tiles, tiles_floats, stream);
}

// The same from the host's own records of the rows' options (SamplingParams keeps one, so that a step only strings them together) and their
// streams' counters: nothing is sent to the device but the launches, and the ids go to the host's pinned memory by the kernel that chooses them.
// Up to SAMPLE_CALL_ROWS rows (2 KB of the 4 KB that a launch's arguments may take).  A step of 64 rows of 151,936 ids from call to call: the host's
// 52 us (packing 18, sending the arrays 14, launches 11, copying the ids back and its event 9) are 23, the step 60 -> 28 us, alone 105 -> 48.
struct SampleRecord {
    float temperature, top_p;
    unsigned long long seed;
    int top_k, unused;
};
static_assert(sizeof(SampleRecord) == 24, "as the host packs it");
#define SAMPLE_CALL_ROWS 128
template <int N>
static int sample_call(const float* logits, const SampleRecord* rec, const unsigned long long* counters, int* out, int* host, int n, int V, float* tiles,
                       long tiles_floats, hipStream_t stream) {
    SampleValues<N> v;
    for (int i = 0; i < n; ++i) {
        v.temperature[i] = rec[i].temperature > 0.f ? rec[i].temperature : 0.f;
        v.top_p[i] = rec[i].top_p;
        v.uniform[i] = stream_uniform(rec[i].seed, counters[i]);
        v.top_k[i] = rec[i].top_k;
    }
    return launch_sample(logits, v, out, host, n, V, tiles, tiles_floats, stream);
}
extern "C" int li_sample_call(const float* logits, const void* records, const unsigned long long* counters, int* out, int* host, int n, int V,
                              float* tiles, long tiles_floats, hipStream_t stream) {
    if (n <= 0 || n > SAMPLE_CALL_ROWS || !records || !counters || !out) return LI_ERR_SIZE;
    const SampleRecord* rec = reinterpret_cast<const SampleRecord*>(records);
    if (n <= 16) return sample_call<16>(logits, rec, counters, out, host, n, V, tiles, tiles_floats, stream);
    if (n <= 64) return sample_call<64>(logits, rec, counters, out, host, n, V, tiles, tiles_floats, stream);
    return sample_call<SAMPLE_CALL_ROWS>(logits, rec, counters, out, host, n, V, tiles, tiles_floats, stream);
}
