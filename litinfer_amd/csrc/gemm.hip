// out[M, N] = x[M, K] w[N, K]^T (+ bias[N]), or out += accumulate * (x w^T + bias) where the number `accumulate`
// is not 0 (1 for a plain sum), float32 accumulation.
//
// float32 operands: float32 MFMA tiles, and an LDS-tiled FMA kernel where K is no multiple of 4 (true 32-bit, no
// reduced-precision matrix mode).  bfloat16 operands: MFMA tiles for 64-wide waves.  Within a kernel the sum over K
// runs in an order that depends on K and the number of parts K is cut into, not on the element's place; which kernel
// and how many parts follow from M, N and K, so the rows of one call are all summed alike.
#include "few_rows.h"
#include "lds_loads.h"
#include <algorithm>
#include <type_traits>
#include <utility>

// ------------------------------------------------------------ float32 tiles
// 64 x 64 tile per block of 256 threads, 4 x 4 outputs per thread, K in steps of 16.
#define F32_BM 64
#define F32_BN 64
#define F32_BK 16

__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ x,
                                                        const float* __restrict__ w,
                                                        const float* __restrict__ bias,
                                                        float* __restrict__ out, int M, int N, int K,
                                                        float accumulate) {
    __shared__ float As[F32_BK][F32_BM + 4];
    __shared__ float Bs[F32_BK][F32_BN + 4];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.y * F32_BM, n0 = blockIdx.x * F32_BN;
    const int ty = tid / 16, tx = tid % 16;
    const int lrow = tid / 4, lk = (tid % 4) * 4;            // this thread's 4 consecutive k of one row
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += F32_BK) {
        float a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = k0 + lk + i;
            a[i] = (m0 + lrow < M && k < K) ? x[(size_t)(m0 + lrow) * K + k] : 0.f;
            b[i] = (n0 + lrow < N && k < K) ? w[(size_t)(n0 + lrow) * K + k] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) { As[lk + i][lrow] = a[i]; Bs[lk + i][lrow] = b[i]; }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < F32_BK; ++k) {
            float av[4], bv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) { av[i] = As[k][ty * 4 + i]; bv[i] = Bs[k][tx * 4 + i]; }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], bv[j], acc[i][j]);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = m0 + ty * 4 + i;
        if (row >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = n0 + tx * 4 + j;
            if (col < N) epilogue_store(out, (size_t)row * N + col, acc[i][j], bias, col, accumulate);
        }
    }
}

// The same product in tiles of 128 x 128 with 8 x 8 outputs a thread, for many rows and columns:
// a step reads 16 floats from LDS for 64 multiply-adds (the small tile reads 8 for 16), so the
// FMA units and not LDS bound it.  Every output element still adds its products up in ascending
// k, one fused multiply-add after the other: the results are those of the small tile bit for bit.
#define F32B_BM 128
#define F32B_BN 128
#define F32B_BK 8

__global__ __launch_bounds__(256) void gemm_f32_big_kernel(const float* __restrict__ x,
                                                            const float* __restrict__ w,
                                                            const float* __restrict__ bias,
                                                            float* __restrict__ out, int M, int N, int K,
                                                            float accumulate) {
    __shared__ __attribute__((aligned(16))) float As[2][F32B_BK][F32B_BM + 4];
    __shared__ __attribute__((aligned(16))) float Bs[2][F32B_BK][F32B_BN + 4];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.y * F32B_BM, n0 = blockIdx.x * F32B_BN;
    const int ty = tid / 16, tx = tid % 16;                  // outputs rows 4 ty .. +3 and 64 + 4 ty .., columns likewise
    const int lrow = tid / 2, lk = (tid % 2) * 4;            // this thread's 4 consecutive k of one row of each operand
    const bool vec = (K % 4) == 0;
    const float* arow = x + (size_t)(m0 + lrow < M ? m0 + lrow : M - 1) * K;
    const float* brow = w + (size_t)(n0 + lrow < N ? n0 + lrow : N - 1) * K;
    float acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = 0.f;
    float a[4], b[4];
    auto fetch = [&](int k0) {
        if (vec && k0 + lk + 4 <= K) {
            const floatx4 av = *reinterpret_cast<const floatx4*>(arow + k0 + lk);
            const floatx4 bv = *reinterpret_cast<const floatx4*>(brow + k0 + lk);
#pragma unroll
            for (int i = 0; i < 4; ++i) { a[i] = av[i]; b[i] = bv[i]; }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = k0 + lk + i;
                a[i] = k < K ? arow[k] : 0.f;
                b[i] = k < K ? brow[k] : 0.f;
            }
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) { As[buf][lk + i][lrow] = a[i]; Bs[buf][lk + i][lrow] = b[i]; }
    };
    fetch(0);
    stash(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += F32B_BK) {
        const bool more = k0 + F32B_BK < K;
        if (more) fetch(k0 + F32B_BK);                       // on its way while this step is multiplied
#pragma unroll
        for (int k = 0; k < F32B_BK; ++k) {
            const floatx4 a0 = *reinterpret_cast<const floatx4*>(&As[buf][k][4 * ty]);
            const floatx4 a1 = *reinterpret_cast<const floatx4*>(&As[buf][k][64 + 4 * ty]);
            const floatx4 b0 = *reinterpret_cast<const floatx4*>(&Bs[buf][k][4 * tx]);
            const floatx4 b1 = *reinterpret_cast<const floatx4*>(&Bs[buf][k][64 + 4 * tx]);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float av = i < 4 ? a0[i] : a1[i - 4];
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[i][j] = fmaf(av, j < 4 ? b0[j] : b1[j - 4], acc[i][j]);
            }
        }
        if (more) {
            stash(buf ^ 1);
            __syncthreads();
            buf ^= 1;
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = m0 + (i < 4 ? 4 * ty + i : 64 + 4 * ty + i - 4);
        if (row >= M) continue;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int col = n0 + (j < 4 ? 4 * tx + j : 64 + 4 * tx + j - 4);
            if (col < N) epilogue_store(out, (size_t)row * N + col, acc[i][j], bias, col, accumulate);
        }
    }
}

// ------------------------------------------------------ float32 on the matrix cores
// v_mfma_f32_32x32x2_f32 multiplies and adds in float32 (no operand is rounded to a shorter format: this
// is not one of the reduced-precision matrix modes), at twice the rate of the vector ALU's FMA and without
// the operands' way through registers that an 8 x 8 tile a lane needs.  Block tile 128 x 128, four waves
// two by two, each 64 x 64 = 2 x 2 MFMA tiles; K in steps of 16 (eight MFMAs of two k-values a tile).
// A stage holds the rows of x and w as they lie in memory, 16 k-values (four 16-byte pieces) a row; piece p of row r
// lies at place p ^ (r / 4 % 4), so that neither the writes (four rows' pieces side by side) nor the reads (a piece
// each of sixteen rows) meet a bank twice.  Lane (row, k) of an MFMA reads a whole piece, the k-th of a pair, and the
// MFMA e of a pair multiplies the e-th values of both: k-values e and 4 + e of eight (within a step the order of a
// sum is the same for every row and column).  Bound by the matrix cores: a wave's 32 MFMAs of a step take 2,048 cycles
// of its SIMD, so what a wave needs next has to be there when it is done.  The pieces of a half step are read while the
// other half is multiplied, and global loads are on their way for a whole step: a step 1.06 us where a unit has one block,
// against 1.21 with transposed stages read word by word as the MFMAs need them (0.87 if a step were its MFMAs alone);
// 1,024 x 17,920 x 1,536 520 -> 500 us, 2,048 rows 925 -> 890, 128 x 1,536 x 1,536 in one part 128 -> 113.  Steps of 32
// k-values were no faster (the same time a k-value), and loads straight into LDS were where the blocks fill whole rounds
// over the chip (1,024 x 3,584 x 18,944 in one part 1,267 -> 1,165) and up to 15 % slower where they do not
// (2,048 x 1,536 x 8,960 460 -> 540): blocks in lockstep end together, and the next ones pile up on the first unit.
// K a multiple of 4; rows and columns past the end repeat the last and are not stored.
// gridDim.z > 1: K is cut into that many parts of `part_steps` steps (the last one shorter), and part z's sums go to
// the z-th [M, N] matrix behind `out`, without bias (splitk_reduce_kernel adds them up in order; see f32_split_parts).
#define F32M_BM 128
#define F32M_BN 128
#define F32M_BK 16
__global__ __launch_bounds__(256) void gemm_f32_mfma_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             const float* __restrict__ bias, float* __restrict__ out,
                                                             int M, int N, int row_len, float accumulate, int part_steps) {
    __shared__ __align__(16) float As[2][F32M_BM * F32M_BK];
    __shared__ __align__(16) float Bs[2][F32M_BN * F32M_BK];
    // this block's k-values: [k_first, k_first + K) of rows of row_len
    const int k_first = blockIdx.z * part_steps * F32M_BK;
    const int K = gridDim.z == 1 || blockIdx.z + 1 == gridDim.z ? row_len - k_first : part_steps * F32M_BK;
    out += (size_t)blockIdx.z * M * N;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * F32M_BM, n0 = blockIdx.x * F32M_BN;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    // global loads: thread t takes the piece t % 4 of rows t / 4 and t / 4 + 64 of both tiles
    const int lrow = tid >> 2, lkq = tid & 3;
    const int put = lrow * F32M_BK + 4 * (lkq ^ ((lrow >> 2) & 3));          // (row + 64: 64 rows further on)
    const float* xa[2];
    const float* wb[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int ra = m0 + lrow + 64 * h, rb = n0 + lrow + 64 * h;
        xa[h] = x + (size_t)(ra < M ? ra : M - 1) * row_len + k_first + 4 * lkq;
        wb[h] = w + (size_t)(rb < N ? rb : N - 1) * row_len + k_first + 4 * lkq;
    }
    floatx4 ga[2], gb[2];
    // WHOLE: the step's 16 k-values lie inside K; nothing is then chosen or replaced (a value chosen between what
    // was loaded and zero is waited for at once: the loads of the next step then did not run under this step's MFMAs)
    auto fetch = [&](int k0, auto whole_tag) {
        constexpr bool WHOLE = decltype(whole_tag)::value;
        const bool ok = WHOLE || k0 + 4 * lkq < K;         // (K % 4 == 0: a 16-byte piece is inside the row or past its end)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            // (a piece past the row's end is replaced by the row's first one, which is always there: with K < 16 the
            // thread's own k-quarter may lie past the end of the LAST row, that is, of the tensor)
            ga[h] = *reinterpret_cast<const floatx4*>(xa[h] + (ok ? k0 : -4 * lkq));
            gb[h] = *reinterpret_cast<const floatx4*>(wb[h] + (ok ? k0 : -4 * lkq));
            if constexpr (!WHOLE) { if (!ok) { ga[h] = floatx4{0.f, 0.f, 0.f, 0.f}; gb[h] = floatx4{0.f, 0.f, 0.f, 0.f}; } }
        }
    };
    auto fetch_any = [&](int k0) { if (k0 + F32M_BK <= K) fetch(k0, std::true_type{}); else fetch(k0, std::false_type{}); };
    auto stash = [&](int st) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            *reinterpret_cast<floatx4*>(&As[st][put + 64 * h * F32M_BK]) = ga[h];
            *reinterpret_cast<floatx4*>(&Bs[st][put + 64 * h * F32M_BK]) = gb[h];
        }
    };
    floatx16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    const int frow = lane & 31, fk = lane >> 5;
    floatx4 fa[2][2], fb[2][2];                            // [half of the step][MFMA tile]
    auto read = [&](int st, auto half_tag) {
        constexpr int H = decltype(half_tag)::value;
        const int piece = 4 * ((2 * H + fk) ^ ((frow >> 2) & 3));
#pragma unroll
        for (int i = 0; i < 2; ++i) fa[H][i] = *reinterpret_cast<const floatx4*>(&As[st][(wm + 32 * i + frow) * F32M_BK + piece]);
#pragma unroll
        for (int j = 0; j < 2; ++j) fb[H][j] = *reinterpret_cast<const floatx4*>(&Bs[st][(wn + 32 * j + frow) * F32M_BK + piece]);
    };
    auto multiply = [&](auto half_tag) {
        constexpr int H = decltype(half_tag)::value;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[H][i][e], fb[H][j][e], acc[i][j], 0, 0, 0);
    };
    constexpr std::integral_constant<int, 0> FIRST{};
    constexpr std::integral_constant<int, 1> SECOND{};
    fetch_any(0);
    stash(0);
    if (F32M_BK < K) fetch_any(F32M_BK);
    __syncthreads();
    read(0, FIRST);
    int st = 0, k0 = 0;
    // A step: its second half's pieces are asked for, the first half is multiplied, the next step's values go to the other
    // stage (whose readers have passed the barrier of the step before), the loads of the step after it start, and behind
    // the barrier the next step's first half is asked for while the second half is multiplied.
    // While the step two further on is whole, its loads are neither conditional nor chosen from ...
    for (; k0 + 3 * F32M_BK <= K; k0 += F32M_BK) {
        read(st, SECOND);
        __builtin_amdgcn_sched_barrier(0);                 // (left to itself the compiler moves reads and loads down to where their values are used)
        multiply(FIRST);
        stash(st ^ 1);
        fetch(k0 + 2 * F32M_BK, std::true_type{});
        __syncthreads();
        st ^= 1;
        read(st, FIRST);
        __builtin_amdgcn_sched_barrier(0);
        multiply(SECOND);
    }
    // ... then the steps that are left
    for (; k0 < K; k0 += F32M_BK) {
        const bool more = k0 + F32M_BK < K;
        read(st, SECOND);
        multiply(FIRST);
        if (more) {
            stash(st ^ 1);
            if (k0 + 2 * F32M_BK < K) fetch_any(k0 + 2 * F32M_BK);
        }
        __syncthreads();
        st ^= 1;
        if (more) read(st, FIRST);
        multiply(SECOND);
    }
    // register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of a 32 x 32 tile
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int col = n0 + wn + 32 * j + frow;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = m0 + wm + 32 * i + 8 * (r >> 2) + 4 * fk + (r & 3);
                if (row < M && col < N) epilogue_store(out, (size_t)row * N + col, acc[i][j][r], bias, col, accumulate);
            }
        }
}

// ------------------------------------------------------ float32, few rows (decode)
// The product streams w once, on the matrix cores in float32 (v_mfma_f32_16x16x4_f32: operands, products and sums
// are float32, nothing is rounded to a shorter format).  A block owns up to 16 columns a tile and 16 rows a tile;
// its eight waves split K in pieces of 32 k-values (a row's whole 128-byte line), wave v taking the pieces
// v, v + 8, ...  Lane (c, q) = (lane % 16, lane / 16) loads the four values k0 + 4 q .. + 3 of column c of w
// and of row c of x with one 16-byte load each; the MFMA e of a piece multiplies the e-th of them, i.e. its
// four k-slots are the k-values k0 + e, k0 + 4 + e, k0 + 8 + e, k0 + 12 + e (the order within a piece does
// not matter for a sum; it is the same for every row and column).  No vector arithmetic and few registers,
// so a wave keeps many loads in flight: the FMA form held 8 x 8 sums a lane and one piece in flight, and
// streamed w at 3.2 TB/s.  The eight waves' sums are added in wave order.  The order of a sum is the same for every row and
// column of a call; it depends on K and on whether the halves of a piece are summed by themselves (PACK: at most 8 rows, and
// at most 8 columns a block, which follow from N).
#define F32RM_WAVES 8
template <int AHEAD, int TILES, int RT, bool SWIGLU, bool PACK = false>
__global__ __launch_bounds__(F32RM_WAVES * 64) void gemm_f32_rows_mfma_kernel(const float* __restrict__ x,
                                                                              const float* __restrict__ w,
                                                                              const float* __restrict__ bias,
                                                                              float* __restrict__ out, int M, int N, int K,
                                                                              float accumulate, int cols, LiAct gated) {
    // TILES: MFMA tiles of 16 columns side by side in a block (`cols` <= 16 TILES): they share the block's
    // loads of x, which come through the same path as w (a matrix of many columns has blocks enough).
    // RT: tiles of 16 rows one above the other (M <= 16 RT): they share the block's loads of w, which is
    // read from memory once whatever the rows.
    // SWIGLU: w is [gate; up] of N rows each, the tiles come in pairs (the gate columns n0 + 16 p .. and the
    // up columns of the same outputs), `cols` <= 8 TILES outputs a block, and out [M, N] gets
    // up * gate / (1 + exp(-gate)) from the float32 sums: the 2 N columns never go to memory.
    // PACK: at most 8 rows and 8 columns a block: an MFMA takes both halves of a piece, k-values 0 .. 15 in its rows and
    // columns 0 .. 7 and 16 .. 31 in 8 .. 15, so that no lane loads a row or a column that another one has; the two
    // quarters of the result that pair a half with itself are the sums, the other two are left.  (A matrix of few columns
    // has few of them a block, six of 1,536 on 256 units: of sixteen lanes' loads ten brought what others had.  3 rows
    // x 1,536 x 8,960, 55 MB, 22.9 -> 14.8 us.)
    static_assert(!SWIGLU || TILES % 2 == 0, "gate and up tiles in pairs");
    static_assert(!PACK || (!SWIGLU && TILES == 1 && RT == 1), "one tile");
    constexpr int UN = PACK ? 1 : 2;                          // loads a piece
    __shared__ float part[F32RM_WAVES][RT * TILES * 256];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // (the same for a wave's lanes: its branches are scalar)
    const int c = lane & 15, q = lane >> 4;
    const int cr = PACK ? c & 7 : c, kq = PACK ? 16 * (c >> 3) + 4 * q : 4 * q;      // a lane's row or column of a tile, its first k-value of a piece
    const int n0 = blockIdx.x * cols;
    const int nend = n0 + cols < N ? n0 + cols : N;
    const float* wrow[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const int col = SWIGLU ? n0 + 16 * (t / 2) + c : n0 + 16 * t + cr;
        wrow[t] = w + ((size_t)(col < nend ? col : nend - 1) + (SWIGLU && (t & 1) ? (size_t)N : 0)) * K + kq;
    }
    const float* xrow[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) xrow[i] = x + (size_t)(16 * i + cr < M ? 16 * i + cr : M - 1) * K + kq;
    floatx4 acc[RT][TILES][2];                                // two chains of MFMAs a tile (each waits for its own last result only)
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < TILES; ++t) acc[i][t][0] = acc[i][t][1] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int last = K - 4;                                   // (K is a multiple of 4: the last whole 16-byte piece of a row)
    // A trip is AHEAD pieces of 32 k-values a wave: all their loads at once, never conditional (a piece past
    // the end reads the row's last 16 bytes and multiplies by zero); the next trip's loads are issued before
    // this trip is multiplied, into the other set of registers.  (Loads that pass the caches by, `nontemporal`,
    // were 10 % slower here, as for the bfloat16 products.)
    floatx4 wv[2][AHEAD][UN][TILES], xv[2][AHEAD][UN][RT];
    constexpr int PIECE = 32 * F32RM_WAVES, TRIP = PIECE * AHEAD;
    // WHOLE: every piece of the trip lies inside K; nothing is then chosen or replaced (a value chosen between what
    // was loaded and zero is waited for at once, and so is the next use of any load behind a conditional one).
    auto fetch = [&](int buf, int k0, auto whole_tag) {
        constexpr bool WHOLE = decltype(whole_tag)::value;
#pragma unroll
        for (int a = 0; a < AHEAD; ++a)
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int k = k0 + PIECE * a + 16 * u;                    // + kq is in the row pointers
                const bool ok = WHOLE || k + kq < K;
                const int at = ok ? k : last - kq;
#pragma unroll
                for (int t = 0; t < TILES; ++t) wv[buf][a][u][t] = *reinterpret_cast<const floatx4*>(wrow[t] + at);
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    xv[buf][a][u][i] = *reinterpret_cast<const floatx4*>(xrow[i] + at);
                    if constexpr (!WHOLE) { if (!ok) xv[buf][a][u][i] = floatx4{0.f, 0.f, 0.f, 0.f}; }
                }
            }
    };
    auto whole = [&](int k0) { return k0 + PIECE * (AHEAD - 1) + 32 <= K; };    // (the same for a wave's lanes)
    auto fetch_any = [&](int buf, int k0) {
        if (whole(k0)) fetch(buf, k0, std::true_type{}); else fetch(buf, k0, std::false_type{});
    };
    auto multiply = [&](int buf) {
#pragma unroll
        for (int a = 0; a < AHEAD; ++a)
#pragma unroll
            for (int u = 0; u < UN; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < RT; ++i)
#pragma unroll
                        for (int t = 0; t < TILES; ++t)
                            acc[i][t][e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[buf][a][u][i][e], wv[buf][a][u][t][e],
                                                                                    acc[i][t][e & 1], 0, 0, 0);
    };
    int k0 = 32 * wave;
    if (k0 < K) fetch_any(0, k0);
    // while the two trips after this one are whole, nothing about the loads is conditional (where a path with
    // loads and one without meet, the compiler's count of the loads in flight is the smaller one, and the
    // next wait is for all of them) ...
    for (; whole(k0 + 2 * TRIP); k0 += 2 * TRIP) {
        fetch(1, k0 + TRIP, std::true_type{});
        multiply(0);
        fetch(0, k0 + 2 * TRIP, std::true_type{});
        multiply(1);
    }
    // ... and the trips that are left
    for (; k0 < K; k0 += 2 * TRIP) {
        if (k0 + TRIP < K) fetch_any(1, k0 + TRIP);
        multiply(0);
        if (k0 + TRIP >= K) break;
        if (k0 + 2 * TRIP < K) fetch_any(0, k0 + 2 * TRIP);
        multiply(1);
    }
    // acc[i][t][.][r] = the sum for row 16 i + 4 q + r, column c of tile t, of this wave's share of K (its even and
    // its odd k-values)
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wave][256 * (TILES * i + t) + (4 * q + r) * 16 + c] = acc[i][t][0][r] + acc[i][t][1][r];
    __syncthreads();
    constexpr int OT = SWIGLU ? TILES / 2 : TILES;            // tiles of outputs
    for (int e = threadIdx.x; e < RT * OT * 256; e += F32RM_WAVES * 64) {
        const int i = e / (OT * 256), t = (e >> 8) % OT, row = 16 * i + ((e >> 4) & 15), j = 16 * t + (e & 15);
        if (row >= M || n0 + j >= nend) continue;
        const int at = 256 * (TILES * i + (SWIGLU ? 2 * t : t)) + (e & 255);
        float v = part[0][at];
#pragma unroll
        for (int v2 = 1; v2 < F32RM_WAVES; ++v2) v += part[v2][at];
        if constexpr (PACK) {                                   // (rows and columns below 8: `row` < M and j < cols)
#pragma unroll
            for (int v2 = 0; v2 < F32RM_WAVES; ++v2) v += part[v2][at + 8 * 16 + 8];
        }
        if constexpr (SWIGLU) {
            float up = part[0][at + 256];
#pragma unroll
            for (int v2 = 1; v2 < F32RM_WAVES; ++v2) up += part[v2][at + 256];
            if (gated.act == LI_ACT_CLAMPED) {                  // (see gated_bf16)
                v = fminf(v, gated.a0);
                up = fminf(fmaxf(up, -gated.a0), gated.a0);
                out[(size_t)row * N + n0 + j] = (up + 1.0f) * (v / (1.0f + expf(-1.702f * v)));
            } else if (gated.act == LI_ACT_GELU_TANH) {
                out[(size_t)row * N + n0 + j] = up * gelu_tanh(v);
            } else {
                out[(size_t)row * N + n0 + j] = up * (v / (1.0f + expf(-v)));
            }
        } else {
            epilogue_store(out, (size_t)row * N + n0 + j, v, bias, n0 + j, accumulate);
        }
    }
}

#define F32_ROWS_MAX 64          // up to this many rows the row kernel is taken (K a multiple of 4)

static int compute_units();

// swiglu: w is [gate; up] of N rows each and out [M, N] gets the activation (no bias, no accumulation)
static int launch_f32_rows(const float* x, const float* w, const float* bias, float* out, int M, int N, int K,
                           float accumulate, hipStream_t stream, bool swiglu = false, LiAct gated = {}) {
    // as many blocks as a whole number of rounds over the compute units, each with the same share of the columns;
    // two MFMA tiles side by side where 16 columns a block would not fit one round (they share the loads of x:
    // the 7B's gate/up matrix at 8 rows 136 -> 130 us)
    const int cu = compute_units();
    const int rt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
    // (four tiles side by side were slower than two: the 7B's gate/up matrix at 8 rows 148 against 130 us)
    int tiles = N > 16 * cu ? 2 : 1;                          // tiles of 16 outputs
    if (swiglu) tiles = 1;                                    // (a pair of gate and up tiles: two tiles of w already)
    const int most = 16 * tiles;
    const int rounds = (N + cu * most - 1) / (cu * most);
    int cols = (N + cu * rounds - 1) / (cu * rounds);
    if (cols < 1) cols = 1;
    const long groups = (N + cols - 1) / cols;
    if (groups > 0x7fffffffL) return LI_ERR_SIZE;
    const unsigned grid = (unsigned)groups;
    // pieces a trip: a long K keeps four a wave in flight, a short one two (measured: 3,584 columns 136 against
    // 156 us for the 7B's gate/up matrix, 18,944 columns 68.6 against 74.0 us for its way back), a tiny one, and
    // many rows (whose registers hold the rows' pieces too), one.  At most 8 rows and 8 columns a block: both halves of a
    // piece in one load, and four pieces a trip for up to four rows over a long K or one of whole trips, else one (us with
    // the matrices in memory, halves in turn / packed with one / four: 3 rows x 1,536 x 1,536 5.7 / 5.0 / 5.5, x 1,536 x 8,960
    // 22.9 / 15.9 / 14.8, x 2,048 x 2,048 6.8 / 6.0 / 5.8, x 2,048 x 1,024 5.0 / 4.5 / 4.3; 4 rows x 1,536 x 4,096 10.7 / 8.6 /
    // 8.1; 8 rows x 1,536 x 1,536 5.9 / 5.3 / 6.4, x 1,536 x 8,960 24.7 / 17.1 / 18.3)
#define LI_F32RM(AH, TL, RTV, ...) gemm_f32_rows_mfma_kernel<AH, TL, RTV, __VA_ARGS__><<<grid, F32RM_WAVES * 64, 0, stream>>>(x, w, bias, out, M, N, K, accumulate, cols, gated)
    const int ahead = rt == 4 ? 1 : K >= 8192 && rt == 1 ? 4 : K >= 32 * F32RM_WAVES * 4 ? 2 : 1;
    if (swiglu) {
        if (rt == 1) { if (ahead == 4) LI_F32RM(4, 2, 1, true); else if (ahead == 2) LI_F32RM(2, 2, 1, true); else LI_F32RM(1, 2, 1, true); }
        else if (rt == 2) { if (ahead >= 2) LI_F32RM(2, 2, 2, true); else LI_F32RM(1, 2, 2, true); }
        else LI_F32RM(1, 2, 4, true);
        return li_launch_status();
    }
    if (rt == 1) {
        if (tiles == 2) { if (ahead == 4) LI_F32RM(4, 2, 1, false); else if (ahead == 2) LI_F32RM(2, 2, 1, false); else LI_F32RM(1, 2, 1, false); }
        else if (M <= 8 && cols <= 8) {
            if (M <= 4 && (K >= 2048 || K % 1024 == 0)) LI_F32RM(4, 1, 1, false, true); else LI_F32RM(1, 1, 1, false, true);
        } else { if (ahead == 4) LI_F32RM(4, 1, 1, false); else if (ahead == 2) LI_F32RM(2, 1, 1, false); else LI_F32RM(1, 1, 1, false); }
    } else if (rt == 2) {
        if (tiles == 2) { if (ahead >= 2) LI_F32RM(2, 2, 2, false); else LI_F32RM(1, 2, 2, false); }
        else { if (ahead >= 2) LI_F32RM(2, 1, 2, false); else LI_F32RM(1, 1, 2, false); }
    } else {
        if (tiles == 2) LI_F32RM(1, 2, 4, false); else LI_F32RM(1, 1, 4, false);
    }
#undef LI_F32RM
    return li_launch_status();
}

// ----------------------------------------------------------- bfloat16 MFMA
// Block tile 128 x 128, K in steps of 32, 4 waves in a 2 x 2 grid, each wave a
// 64 x 64 tile made of 2 x 2 MFMA 32x32x16 tiles.  Operand layout of
// v_mfma_f32_32x32x16_bf16: lane l holds 8 consecutive k of row (l % 32),
// starting at k = 8 * (l / 32), for A and for B alike; the result's register r
// of lane l is row 8 * (r / 4) + 4 * (l / 32) + r % 4, column l % 32.
#define BF_BM 128
#define BF_BN 128
#define BF_BK 32
#define BF_LDS_STRIDE (BF_BK + 8)           // in elements; the pad spreads rows over banks

struct __attribute__((aligned(16))) chunk16 { uint32_t w[4]; };

template <bool ALIGNED>
__device__ __forceinline__ chunk16 load_chunk(const bf16_t* __restrict__ base, int row, int rows,
                                              int k, int K) {
    chunk16 c = {{0u, 0u, 0u, 0u}};
    if (row >= rows || k >= K) return c;
    const bf16_t* p = base + (size_t)row * K + k;
    if (ALIGNED) {                                   // K % 8 == 0: the chunk is whole and 16-byte aligned
        c = *reinterpret_cast<const chunk16*>(p);
    } else {
        uint16_t e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = (k + i < K) ? p[i].bits : (uint16_t)0;
#pragma unroll
        for (int i = 0; i < 4; ++i) c.w[i] = (uint32_t)e[2 * i] | ((uint32_t)e[2 * i + 1] << 16);
    }
    return c;
}

template <typename TO, bool ALIGNED>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(const bf16_t* __restrict__ x,
                                                         const bf16_t* __restrict__ w,
                                                         const float* __restrict__ bias,
                                                         TO* __restrict__ out, int M, int N, int K,
                                                         float accumulate) {
    __shared__ __attribute__((aligned(16))) uint16_t As[BF_BM * BF_LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[BF_BN * BF_LDS_STRIDE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const int m0 = blockIdx.y * BF_BM, n0 = blockIdx.x * BF_BN;
    floatx16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // each thread moves two 16-byte chunks of A and two of B per K step
    const int crow0 = tid >> 2, ck = (tid & 3) * 8;
    chunk16 ra[2], rb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        ra[i] = load_chunk<ALIGNED>(x, m0 + crow0 + 64 * i, M, ck, K);
        rb[i] = load_chunk<ALIGNED>(w, n0 + crow0 + 64 * i, N, ck, K);
    }
    const int frow = lane & 31, fk = (lane >> 5) * 8;
    for (int k0 = 0; k0 < K; k0 += BF_BK) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<chunk16*>(&As[(crow0 + 64 * i) * BF_LDS_STRIDE + ck]) = ra[i];
            *reinterpret_cast<chunk16*>(&Bs[(crow0 + 64 * i) * BF_LDS_STRIDE + ck]) = rb[i];
        }
        __syncthreads();
        if (k0 + BF_BK < K) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                ra[i] = load_chunk<ALIGNED>(x, m0 + crow0 + 64 * i, M, k0 + BF_BK + ck, K);
                rb[i] = load_chunk<ALIGNED>(w, n0 + crow0 + 64 * i, N, k0 + BF_BK + ck, K);
            }
        }
#pragma unroll
        for (int ks = 0; ks < BF_BK; ks += 16) {
            bf16x8 af[2], bfr[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                af[i] = *reinterpret_cast<const bf16x8*>(&As[(wm + 32 * i + frow) * BF_LDS_STRIDE + ks + fk]);
                bfr[i] = *reinterpret_cast<const bf16x8*>(&Bs[(wn + 32 * i + frow) * BF_LDS_STRIDE + ks + fk]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
        }
    }
    const int ccol = lane & 31, crow = (lane >> 5) * 4;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int col = n0 + wn + 32 * j + ccol;
            if (col >= N) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = m0 + wm + 32 * i + 8 * (r >> 2) + crow + (r & 3);
                if (row < M) epilogue_store(out, (size_t)row * N + col, acc[i][j][r], bias, col, accumulate);
            }
        }
}

// ---------------------------------------------- bfloat16, many rows (prompts)
// With many rows the product is bound by the matrix cores and, before them, by
// how often an operand byte has to be read from LDS: a wave's tile of WM x WN
// needs (WM + WN) * BK operand elements for WM * WN * BK multiply-adds, so the
// tiles are made large.  Block tile BM x BN, 4 waves as 2 x 2, wave tile
// BM/2 x BN/2 made of MFMA 32x32x16 tiles, K in steps of 64.  Two LDS stages:
// the global loads of the next K step are in flight (in registers) while this
// step is multiplied from LDS, then written to the other stage; one barrier a
// step.  A row of a stage is 64 elements = 128 bytes = 8 chunks of 16 bytes;
// chunk c of row r lies at position c ^ ((r >> 1) & 7), which spreads the 16
// rows that one fragment read touches over all banks.
// Blocks go to the 8 XCDs in turn (block b runs on XCD b % 8), and each XCD has an L2 of its
// own.  The tiles are put in one sequence: patches of up to 8 row panels x 4 or more column panels
// (32 tiles, what an XCD runs at one time; smaller at the matrix's edges), patches along the rows
// first, then along the columns; what a patch reads from beyond its L2 is (8 + 4) panels for 32
// tiles.  Each XCD takes one eighth of the sequence in one piece: a run of neighbouring column
// panels of W, which no other XCD reads but for the two panels at its ends.  Every block has a
// tile, but for the last few of the last XCD, and no XCD has more than one tile more than another:
// blocks that return at once in the middle of the queue, and XCDs with a column panel more than
// others, made a matrix of fewer tiles than compute units take two rounds.
struct TileOrder {
    int pm, gn;                                      // row panels and column panels of a patch
    __host__ __device__ TileOrder(int mtiles) {
        pm = mtiles < 8 ? mtiles : 8;
        gn = 32 / pm;
    }
    __host__ static long blocks(long mtiles, long ntiles, long nsplit = 1) {      // grid size: the same number of blocks on each XCD
        return (mtiles * ntiles * nsplit + 7) / 8 * 8;
    }
    // With K in nsplit parts: where the tiles divide by 8 every XCD takes its eighth of them in every
    // part (the same rows of w, all of K).  Otherwise the sequence is that of the tiles nsplit times
    // over, part after part, and the XCDs share the whole of it: dealt part by part, the last XCD's
    // few tiles fewer would come nsplit times over and the other XCDs would hold more blocks than they
    // have compute units (36 tiles in 7 parts: 35 blocks on each of seven XCDs, 7 on the last).
    // (All of it in 32 bits: the launch has checked that the blocks fit.)
    __device__ bool tile(unsigned block, int mtiles, int ntiles, int nsplit, int& mt, int& nt, int& split) const {
        const unsigned tiles = (unsigned)mtiles * (unsigned)ntiles, total = tiles * (unsigned)nsplit;
        unsigned t;
        if (nsplit > 1 && (tiles & 7) == 0) {
            split = (int)(block / tiles);
            const unsigned b = block - (unsigned)split * tiles;
            t = (b & 7) * (tiles >> 3) + (b >> 3);
        } else {
            const unsigned per = (total + 7) / 8, s = (block & 7) * per + (block >> 3);
            if (s >= total) return false;
            split = (int)(s / tiles);
            t = s - (unsigned)split * tiles;
        }
        const int group = mtiles * gn;               // tiles of gn column panels
        const int cg = (int)(t / group), r = (int)(t % group);
        const int gc = ntiles - cg * gn < gn ? ntiles - cg * gn : gn;        // column panels of this group
        const int rg = r / (pm * gc), r2 = r % (pm * gc);
        const int rows_in = mtiles - rg * pm < pm ? mtiles - rg * pm : pm;  // row panels of this patch
        mt = rg * pm + r2 % rows_in;
        nt = cg * gn + r2 / rows_in;
        return true;
    }
};

template <int BM, int BN, int BK, typename TO>
__global__ __launch_bounds__(256) void gemm_bf16_big_kernel(const bf16_t* __restrict__ x,
                                                             const bf16_t* __restrict__ w,
                                                             const float* __restrict__ bias,
                                                             TO* __restrict__ out, int M, int N, int K,
                                                             float accumulate) {
    constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
    constexpr int CPR = BK / 8;                                   // 16-byte chunks in a row of a stage
    constexpr int WRAP = 128 / BK;                                // rows that fill all 64 banks once
    constexpr int CA = BM * CPR / 256, CB = BN * CPR / 256;       // chunks per thread and stage
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    uint16_t* As = lds;                                           // [2][BM][BK]
    uint16_t* Bs = lds + 2 * BM * BK;                             // [2][BN][BK]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
    const int mtiles = (M + BM - 1) / BM, ntiles = (N + BN - 1) / BN;
    int mt, nt, split;
    if (!TileOrder(mtiles).tile(blockIdx.x, mtiles, ntiles, 1, mt, nt, split)) return;
    const int m0 = mt * BM, n0 = nt * BN;
    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    auto slot = [](int row, int c) { return row * BK + ((c ^ ((row / WRAP) & (CPR - 1))) << 3); };
    // Global loads carry no branches: a row past the end is read as the last row (its products
    // land in output rows that are not stored), and only a K step that reaches past K is
    // masked, chunk by chunk.
    bf16x8 ra[CA], rb[CB];
    size_t oa[CA], ob[CB];
#pragma unroll
    for (int i = 0; i < CA; ++i) {
        const int qd = tid + 256 * i, row = qd / CPR, c = qd % CPR;
        oa[i] = (size_t)((m0 + row < M) ? m0 + row : M - 1) * K + 8 * c;
    }
#pragma unroll
    for (int i = 0; i < CB; ++i) {
        const int qd = tid + 256 * i, row = qd / CPR, c = qd % CPR;
        ob[i] = (size_t)((n0 + row < N) ? n0 + row : N - 1) * K + 8 * c;
    }
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#define LI_GLOAD(k0)                                                                                      \
    {                                                                                                     \
        const bool full_ = (k0) + BK <= K;                                                                \
        _Pragma("unroll") for (int i = 0; i < CA; ++i)                                                    \
            ra[i] = (full_ || (k0) + 8 * ((tid + 256 * i) % CPR) < K)                                     \
                        ? *reinterpret_cast<const bf16x8*>(x + oa[i] + (k0)) : zero8;                     \
        _Pragma("unroll") for (int i = 0; i < CB; ++i)                                                    \
            rb[i] = (full_ || (k0) + 8 * ((tid + 256 * i) % CPR) < K)                                     \
                        ? *reinterpret_cast<const bf16x8*>(w + ob[i] + (k0)) : zero8;                     \
    }
#define LI_LSTORE(stage)                                                                                  \
    {                                                                                                     \
        _Pragma("unroll") for (int i = 0; i < CA; ++i) {                                                  \
            const int qd = tid + 256 * i, row = qd / CPR, c = qd % CPR;                                   \
            *reinterpret_cast<bf16x8*>(&As[(stage) * BM * BK + slot(row, c)]) = ra[i];                    \
        }                                                                                                 \
        _Pragma("unroll") for (int i = 0; i < CB; ++i) {                                                  \
            const int qd = tid + 256 * i, row = qd / CPR, c = qd % CPR;                                   \
            *reinterpret_cast<bf16x8*>(&Bs[(stage) * BN * BK + slot(row, c)]) = rb[i];                    \
        }                                                                                                 \
    }
    const int frow = lane & 31, fh = lane >> 5;
    const int nk = (K + BK - 1) / BK;
    // fragments of K sub-step ks + 1 are read from LDS before the MFMAs of sub-step ks are
    // issued, so the reads' latency passes while the matrix cores work
    bf16x8 af[2][TM], bfr[2][TN];
#define LI_FREAD(stage, ks, buf)                                                                          \
    {                                                                                                     \
        const int c_ = 2 * (ks) + fh;                                                                     \
        _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                    \
            af[buf][i] = *reinterpret_cast<const bf16x8*>(&As[(stage) * BM * BK + slot(wm + 32 * i + frow, c_)]); \
        _Pragma("unroll") for (int j = 0; j < TN; ++j)                                                    \
            bfr[buf][j] = *reinterpret_cast<const bf16x8*>(&Bs[(stage) * BN * BK + slot(wn + 32 * j + frow, c_)]); \
    }
    LI_GLOAD(0)
    LI_LSTORE(0)
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int stage = kt & 1;
        if (kt + 1 < nk) LI_GLOAD((kt + 1) * BK)
        LI_FREAD(stage, 0, 0)
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
            if (ks + 1 < BK / 16) LI_FREAD(stage, ks + 1, (ks + 1) & 1)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][i], bfr[ks & 1][j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) LI_LSTORE(stage ^ 1)
        __syncthreads();
    }
#undef LI_FREAD
#undef LI_GLOAD
#undef LI_LSTORE
    // Epilogue through LDS: a wave puts a band of 32 rows of its tile into a piece of LDS of its
    // own and takes it out again row by row, 8 consecutive columns a lane, so that the stores
    // (and the loads of what is added to) are whole 16-byte pieces, 16 lanes to a row.
    __syncthreads();                               // the main loop's LDS is free now
    constexpr int ESTRIDE = WN + 4;                // floats per row of a band (pad against bank conflicts)
    float* band = reinterpret_cast<float*>(lds) + wave * 32 * ESTRIDE;
    const int ccol = lane & 31, crow = (lane >> 5) * 4;
    constexpr int LPR = WN / 8;                    // lanes that take one row of the band out (8 columns each)
    constexpr int RPP = 64 / LPR;                  // rows per pass of the wave
    const int erow = lane / LPR, ecol = (lane % LPR) * 8;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                band[(8 * (r >> 2) + crow + (r & 3)) * ESTRIDE + 32 * j + ccol] = acc[i][j][r];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int pass = 0; pass < 32 / RPP; ++pass) {
            const int row = m0 + wm + 32 * i + RPP * pass + erow;
            if (row >= M) continue;
            {
                const int col = n0 + wn + ecol;
                if (col >= N) continue;
                const float* src = &band[(RPP * pass + erow) * ESTRIDE + ecol];
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = src[e];
                const size_t idx = (size_t)row * N + col;
                if (col + 8 <= N && (N % 8) == 0) {               // whole pieces: wide loads and stores
                    if (bias) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) v[e] += bias[col + e];
                    }
                    if constexpr (sizeof(TO) == 4) {
                        float4* o = reinterpret_cast<float4*>(reinterpret_cast<float*>(out) + idx);
                        if (accumulate != 0.f) {
                            const float4 a0 = o[0], a1 = o[1];
                            v[0] = fmaf(accumulate, v[0], a0.x); v[1] = fmaf(accumulate, v[1], a0.y); v[2] = fmaf(accumulate, v[2], a0.z); v[3] = fmaf(accumulate, v[3], a0.w);
                            v[4] = fmaf(accumulate, v[4], a1.x); v[5] = fmaf(accumulate, v[5], a1.y); v[6] = fmaf(accumulate, v[6], a1.z); v[7] = fmaf(accumulate, v[7], a1.w);
                        }
                        o[0] = float4{v[0], v[1], v[2], v[3]};
                        o[1] = float4{v[4], v[5], v[6], v[7]};
                    } else {
                        chunk16 o;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o.w[e] = pack2_bf16(v[2 * e], v[2 * e + 1]);
                        *reinterpret_cast<chunk16*>(reinterpret_cast<uint16_t*>(out) + idx) = o;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (col + e < N) epilogue_store(out, idx + e, v[e], bias, col + e, accumulate);
                }
            }
        }
    }
}

// ------------------------------- bfloat16, many rows, loads straight into LDS
// The same tiling with the global loads going straight into LDS
// (global_load_lds_dwordx4: lane i's 16 bytes land at the wave's LDS base + 16 i),
// which needs no staging registers, so all stages but the one being multiplied are
// in flight: the latency of a load is long against a step.  The
// compiler does not track these loads' completion; `s_waitcnt vmcnt(n)` is
// placed by hand: a wave's loads retire in order, so allowing the loads of the
// younger steps to stay outstanding waits exactly for the oldest step, and the
// barrier after it makes that true for the loads of all four waves.
// Needs K to be a multiple of the step (a load cannot be masked to zeros).  A step is 64
// columns, so that a row of a stage is one whole 128-byte line of the caches.  Two to four stages (what fits the
// 160 KB of LDS); which tiles are this kernel's and which `gemm_bf16_tile_kernel`'s: `tiling_of`, `gated_tiling_of`.
// A wave's band of 32 rows of EW sums in LDS (ESTRIDE floats apart) goes to rows row0 .. and columns col0 .. of out: row by row,
// 8 consecutive columns a lane, so that the stores (and the loads of what is added to) are whole 16-byte pieces.
// GATED: the band holds results already; ACT otherwise: the activation of sums and bias.
template <int EW, int ESTRIDE, bool GATED, int ACT, typename TO>
__device__ __forceinline__ void band_to_memory(const float* band, int row0, int col0, int M, int NO, const float* bias, TO* out,
                                               float accumulate, const LiAct& ep) {
    constexpr int LPR = EW / 8, RPP = 64 / LPR;     // lanes that take a row; rows a pass of the wave covers
    const int lane = threadIdx.x & 63;
    const int erow = lane / LPR, ecol = (lane % LPR) * 8;      // (where 64 is no multiple of LPR the last lanes idle)
    const int col = col0 + ecol;
#pragma unroll
    for (int pass = 0; pass < (32 + RPP - 1) / RPP; ++pass) {
        const int row = row0 + RPP * pass + erow;
        if (erow >= RPP || RPP * pass + erow >= 32 || row >= M || col >= NO) continue;
        const float* src = &band[(RPP * pass + erow) * ESTRIDE + ecol];
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = src[e];
        const size_t o_idx = (size_t)row * NO + col;
        if constexpr (ACT != 0 && !GATED) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = activation(v[e] + (bias && col + e < NO ? bias[col + e] : 0.f), LiAct{ACT, ep.a0, ep.a1});
            if (col + 8 <= NO && (NO % 8) == 0) {
                chunk16 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o.w[e] = pack2_bf16(v[2 * e], v[2 * e + 1]);
                *reinterpret_cast<chunk16*>(reinterpret_cast<uint16_t*>(out) + o_idx) = o;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (col + e < NO) epilogue_store(out, o_idx + e, v[e], nullptr, col + e, 0);
            }
            continue;
        }
        if (col + 8 <= NO && (NO % 8) == 0) {
            if (bias) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] += bias[col + e];
            }
            if constexpr (sizeof(TO) == 4) {
                float4* o = reinterpret_cast<float4*>(reinterpret_cast<float*>(out) + o_idx);
                if (accumulate != 0.f) {
                    const float4 a0 = o[0], a1 = o[1];
                    v[0] = fmaf(accumulate, v[0], a0.x); v[1] = fmaf(accumulate, v[1], a0.y); v[2] = fmaf(accumulate, v[2], a0.z); v[3] = fmaf(accumulate, v[3], a0.w);
                    v[4] = fmaf(accumulate, v[4], a1.x); v[5] = fmaf(accumulate, v[5], a1.y); v[6] = fmaf(accumulate, v[6], a1.z); v[7] = fmaf(accumulate, v[7], a1.w);
                }
                o[0] = float4{v[0], v[1], v[2], v[3]};
                o[1] = float4{v[4], v[5], v[6], v[7]};
            } else {
                chunk16 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o.w[e] = pack2_bf16(v[2 * e], v[2 * e + 1]);
                *reinterpret_cast<chunk16*>(reinterpret_cast<uint16_t*>(out) + o_idx) = o;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (col + e < NO) epilogue_store(out, o_idx + e, v[e], bias, col + e, accumulate);
        }
    }
}

template <int BM, int BN, int BK, int NSTAGE, bool SWIGLU, typename TO, int ACT = 0, int WLM = 2>
__global__ __launch_bounds__(256) void gemm_bf16_dma_kernel(const bf16_t* __restrict__ x,
                                                             const bf16_t* __restrict__ w,
                                                             const float* __restrict__ bias,
                                                             TO* __restrict__ out, int M, int N, int K,
                                                             float accumulate, int nsplit,
                                                             const float* __restrict__ row_parts, int nparts, float eps,
                                                             LiAct ep) {
    // ACT: an activation, of gate and up columns (see gated_bf16) or of the sums (its number); its constants are in `ep`.
    // row_parts (SwiGLU tiles of 64 rows, up to 32 rows of x): x is the xg of li_linear_residual_norm and these
    // are its sq_parts; every row's sums are scaled by 1 / sqrt(sum of the row's parts / K + eps) before the
    // activation, which makes the result that of the RMS norm (the factor of a row does not depend on k).
    // nsplit > 1: a block multiplies one of nsplit parts of K, the y-th, and writes its sums to the y-th
    // [M, N] matrix behind `out` (float, no bias, no accumulation); splitk_reduce_kernel adds them
    // WLM: waves along the rows of the tile, 2 (two by two) or 4 (each wave 32-row bands over all columns:
    // BN may then be any multiple of 32, for matrices whose columns no other tile divides into whole rounds)
    constexpr int WLN = 4 / WLM;
    constexpr int WM = BM / WLM, WN = BN / WLN, TM = WM / 32, TN = WN / 32;
    static_assert(WM % 32 == 0 && WN % 32 == 0 && (WLM == 2 || WLM == 4), "a wave's part of the tile is made of 32 x 32 tiles");
    constexpr bool SWSPLIT = SWIGLU && (TN % 2 == 1);        // gates and ups in different waves (see the rows of w below)
    static_assert(!SWSPLIT || WLN == 2, "gates in one wave, ups in the wave beside it");
    static_assert(BM % 32 == 0 && BN % 32 == 0 && (BM / 4) % (64 / (BK / 8)) == 0 && (BN / 4) % (64 / (BK / 8)) == 0, "whole load instructions a wave");
    constexpr int CPR = BK / 8, WRAP = 128 / BK;                 // chunks in a row; rows that fill all banks once
    constexpr int RPI = 64 / CPR;                                // rows one load instruction of a wave covers
    constexpr int IA = BM / 4 / RPI, IB = BN / 4 / RPI;          // load instructions per wave and step for A and B
    constexpr int STAGE = (BM + BN) * BK;                        // elements of a stage: A rows then B rows
    constexpr int LPW = IA + IB;                                 // loads a wave issues per step
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave / WLN) * WM, wn = (wave % WLN) * WN;
    const int mtiles = (M + BM - 1) / BM, ntiles = (N + BN - 1) / BN;
    int mt, nt, split;
    if (!TileOrder(mtiles).tile(blockIdx.x, mtiles, ntiles, nsplit, mt, nt, split)) return;
    const int m0 = mt * BM, n0 = nt * BN;
    constexpr bool ROWSCALE = SWIGLU && BM == 64;
    // The shares of the rows' sums of squares are asked for now, all at once and never conditional (a share
    // past the last reads the last and is not added), before the first loads of the main loop: a wave's loads
    // retire in order, so they have arrived when the first stage has, and the waits placed by hand below
    // still count the main loop's loads only.  They are added up behind the main loop.
    constexpr int RS_PER = ROWSCALE ? 64 : 1;          // shares a thread adds: 512 at most, 16 or 8 threads a row
    [[maybe_unused]] float rs_part[RS_PER];
    [[maybe_unused]] const int rs_rows = M <= 16 ? 16 : 32;      // rows the shares are kept for (as the product before the norm wrote them)
    [[maybe_unused]] const int rs_groups = 256 / rs_rows;
    if constexpr (ROWSCALE) {
        if (row_parts) {
            const int r = threadIdx.x % rs_rows, g = threadIdx.x / rs_rows;
#pragma unroll
            for (int i = 0; i < RS_PER; ++i) {
                const int p = g + rs_groups * i;
                rs_part[i] = 0.f;
                if (rs_groups * i < nparts) rs_part[i] = row_parts[(size_t)(p < nparts ? p : nparts - 1) * rs_rows + r];      // (the same for all lanes)
            }
        }
    }
    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    // chunk c of row r lies at position c ^ ((r / WRAP) % CPR) of the row's CPR positions
    auto slot = [](int row, int c) { return row * BK + ((c ^ ((row / WRAP) & (CPR - 1))) << 3); };
    // this lane's part of a step: a wave takes BM / 4 rows of A and BN / 4 rows of B; one
    // instruction covers RPI rows, lane -> row lane / CPR, position lane % CPR
    // Addresses: a base that is the same for the whole wave (scalar registers, moved on by a step's
    // columns) plus this lane's 32-bit byte offset within the tile's rows, which never changes.
    uint32_t ga[IA], gb[IB];
    const bf16_t* abase = x + (size_t)m0 * K;
    const bf16_t* bbase = w + (size_t)(SWIGLU ? n0 / 2 : n0) * K;
#pragma unroll
    for (int i = 0; i < IA; ++i) {
        const int row = (BM / 4) * wave + RPI * i + lane / CPR, c = (lane % CPR) ^ ((row / WRAP) & (CPR - 1));
        ga[i] = (uint32_t)(((size_t)((m0 + row < M) ? row : M - 1 - m0) * K + 8 * c) * 2);       // rows past the end: the last row
    }
#pragma unroll
    for (int i = 0; i < IB; ++i) {
        const int row = (BN / 4) * wave + RPI * i + lane / CPR, c = (lane % CPR) ^ ((row / WRAP) & (CPR - 1));
        size_t rel = (n0 + row < N) ? row : N - 1 - n0;            // row of w relative to the tile's first
        if constexpr (SWIGLU && !SWSPLIT) {
            // w is [gate; up] with N / 2 rows each.  The tile's rows alternate in blocks of 32: 32
            // gate rows, the 32 up rows of the same outputs, the next 32 gate rows, ..., so that an
            // accumulator tile and its neighbour hold the two factors of one output tile.
            const int half = N / 2, blk = row / 32;
            const int o = n0 / 2 + (blk / 2) * 32 + row % 32;
            rel = (size_t)((o < half ? o : half - 1) - n0 / 2) + (size_t)(blk & 1) * half;
        } else if constexpr (SWSPLIT) {
            // (a wave's part of the tile is an odd number of blocks of 32 columns: the tile's first half
            // are gate rows, its second half the up rows of the same outputs, so that of two waves side
            // by side one holds the gates and the other the ups; they meet in the epilogue's LDS)
            const int half = N / 2;
            const int o = n0 / 2 + row % (BN / 2);
            rel = (size_t)((o < half ? o : half - 1) - n0 / 2) + (size_t)(row / (BN / 2)) * half;
        }
        gb[i] = (uint32_t)((rel * K + 8 * c) * 2);
    }
    const int uwave = __builtin_amdgcn_readfirstlane(wave);
    // load `idx` of a wave's LPW loads of step kt: first its rows of A, then its rows of B
    auto issue_one = [&](int kt, int idx) {
        uint16_t* st = lds + (kt % NSTAGE) * STAGE;
        if (idx < IA) LI_LOAD_TO_LDS_AT(abase + (size_t)kt * BK, ga[idx], st + ((BM / 4) * uwave + RPI * idx) * BK);
        else LI_LOAD_TO_LDS_AT(bbase + (size_t)kt * BK, gb[idx - IA], st + BM * BK + ((BN / 4) * uwave + RPI * (idx - IA)) * BK);
    };
    auto issue = [&](int kt) {
#pragma unroll
        for (int i = 0; i < LPW; ++i) issue_one(kt, i);
    };
    const int frow = lane & 31, fh = lane >> 5;
    // (the parts' steps: equal shares, the first parts one more where they do not divide)
    const int ksteps = K / BK, kshare = ksteps / nsplit, kmore = ksteps - kshare * nsplit;
    const int kt_first = split * kshare + (split < kmore ? split : kmore);
    const int nk = kshare + (split < kmore ? 1 : 0);
    out += (size_t)split * M * (SWIGLU ? N / 2 : N);
    abase += (size_t)kt_first * BK;
    bbase += (size_t)kt_first * BK;
    constexpr int KS = BK / 16;                    // MFMA groups of a step: 16 columns each
    constexpr int GM = TM * TN, GD = TM + TN;      // MFMAs and fragment reads of a group
    // Order of a step.  A wave issues in order and is alone on its SIMD, and the CU's address unit
    // takes a 16-byte-per-lane load of one wave every 16 cycles, i.e. one of each of the four waves
    // every 64 = two MFMAs: loads issued back to back hold the wave, and with it the SIMD's
    // MFMAs, until the unit has taken them.  So the loads of step kt + NSTAGE - 1 (into the stage
    // that the barrier of step kt - 1 freed) are issued one by one between the MFMAs of the first
    // groups of step kt, at most one per two MFMAs.  Each group's MFMAs run while the fragments
    // of the next 16 columns are read; in the middle of the LAST group the wave waits for the
    // loads of step kt + 1, meets the others at the barrier (stage kt + 1 is there for all, stage kt
    // is read by all) and reads the first fragments of step kt + 1, so that the barrier and the
    // latency of LDS fall under the remaining MFMAs.
    // With 64 rows of x a step has few MFMAs and the product waits for w from memory: there the
    // loads of step kt + NSTAGE are issued all at once, right after the barrier of step kt, so that as
    // many bytes as possible are on their way.
    constexpr bool SPREAD = BM >= 128;
    constexpr int AHEAD = SPREAD ? NSTAGE - 1 : NSTAGE;                // steps loaded before the first is multiplied
    constexpr int PER0 = GM / 2 > 0 ? GM / 2 : 1, PER1 = (LPW + KS - 2) / (KS - 1);
    constexpr int PER = PER0 > PER1 ? PER0 : PER1;                     // loads of one group
#pragma unroll
    for (int p = 0; p < AHEAD; ++p)
        if (p < nk) issue(p);
    bf16x8 af[2][TM], bfr[2][TN];
#define LI_FREAD(stage_, ks, buf)                                                                          \
    {                                                                                                     \
        const uint16_t* As_ = lds + (stage_) * STAGE;                                                     \
        const uint16_t* Bs_ = As_ + BM * BK;                                                              \
        const int c_ = 2 * (ks) + fh;                                                                     \
        _Pragma("unroll") for (int i = 0; i < TM; ++i)                                                    \
            af[buf][i] = *reinterpret_cast<const bf16x8*>(&As_[slot(wm + 32 * i + frow, c_)]);            \
        _Pragma("unroll") for (int j = 0; j < TN; ++j)                                                    \
            bfr[buf][j] = *reinterpret_cast<const bf16x8*>(&Bs_[slot(wn + 32 * j + frow, c_)]);           \
    }
#define LI_WAIT_YOUNGER(y)                                                                                 \
    { if ((y) >= 3) LI_VMCNT(3 * LPW); else if ((y) == 2) LI_VMCNT(2 * LPW); else if ((y) == 1) LI_VMCNT(LPW); else LI_VMCNT(0); }
    {
        const int inflight = nk < AHEAD ? nk : AHEAD;
        LI_WAIT_YOUNGER(inflight - 1)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        LI_FREAD(0, 0, 0)
    }
    // one step; LOADS: the loads of step kt + NSTAGE - 1 are issued between its MFMAs
    auto step = [&](int kt, auto loads_tag) {
        constexpr bool LOADS = decltype(loads_tag)::value;
        const int stage = kt % NSTAGE;
        static_for<KS - 1>([&](auto ks_tag) {
            constexpr int ks = decltype(ks_tag)::value;
            constexpr int l0 = ks * PER < LPW ? ks * PER : LPW, l1 = (ks + 1) * PER < LPW ? (ks + 1) * PER : LPW;
            constexpr int NL = LOADS && SPREAD ? l1 - l0 : 0;
            const uint16_t* As_ = lds + stage * STAGE;
            const uint16_t* Bs_ = As_ + BM * BK;
            const int c_ = 2 * (ks + 1) + fh;
            // written in the order it is to run, and kept so: before MFMA m the m-th fragment read of
            // the next 16 columns (the earlier MFMAs the more, where there are more reads than MFMAs:
            // the group's remaining MFMAs are what covers the latency of LDS), after it the loads that
            // fall to it
            static_for<GM>([&](auto m_tag) {
                constexpr int m = decltype(m_tag)::value;
                constexpr int r0 = GD > GM ? GD - ((GM - m) * GD) / GM : (m < GD ? m : GD);
                constexpr int r1 = GD > GM ? GD - ((GM - m - 1) * GD) / GM : (m < GD ? m + 1 : GD);
#pragma unroll
                for (int r = r0; r < r1; ++r) {
                    if (r < TM) af[(ks + 1) & 1][r] = *reinterpret_cast<const bf16x8*>(&As_[slot(wm + 32 * r + frow, c_)]);
                    else bfr[(ks + 1) & 1][r - TM] = *reinterpret_cast<const bf16x8*>(&Bs_[slot(wn + 32 * (r - TM) + frow, c_)]);
                }
                acc[m / TN][m % TN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks & 1][m / TN], bfr[ks & 1][m % TN], acc[m / TN][m % TN], 0, 0, 0);
#pragma unroll
                for (int l = l0 + (m * NL) / GM; l < l0 + ((m + 1) * NL) / GM; ++l) issue_one(kt + NSTAGE - 1, l);
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        constexpr int BL = (KS - 1) & 1;           // the buffer with the fragments of the last 16 columns
        constexpr int HALF = (TM / 2) * TN > 0 ? (TM / 2) * TN : GM / 2;       // MFMAs of the last group before the wait
#pragma unroll
        for (int m = 0; m < HALF; ++m)
            acc[m / TN][m % TN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[BL][m / TN], bfr[BL][m % TN], acc[m / TN][m % TN], 0, 0, 0);
        if (kt + 1 < nk) {
            // loads of later steps that may stay in flight: steps kt + 2 .. kt + NSTAGE - 1, where they exist
            const int younger = LOADS ? NSTAGE - 2 : (nk - 2 - kt < NSTAGE - 2 ? nk - 2 - kt : NSTAGE - 2);
            LI_WAIT_YOUNGER(younger)
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if constexpr (!SPREAD) {
                if (kt + NSTAGE < nk) issue(kt + NSTAGE);              // into the stage of step kt
            }
            LI_FREAD((kt + 1) % NSTAGE, 0, 0)
        }
#pragma unroll
        for (int m = HALF; m < GM; ++m)
            acc[m / TN][m % TN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[BL][m / TN], bfr[BL][m % TN], acc[m / TN][m % TN], 0, 0, 0);
    };
    int kt = 0;
    if constexpr (SPREAD)
        for (; kt + NSTAGE - 1 < nk; ++kt) step(kt, std::true_type{});
    for (; kt < nk; ++kt) step(kt, std::false_type{});
#undef LI_FREAD
#undef LI_WAIT_YOUNGER
    __syncthreads();                               // the main loop's LDS is free now
    [[maybe_unused]] float* row_inv = nullptr;
    if constexpr (ROWSCALE) {
        // the rows' factors, in the order of additions of the few-row kernel with four waves: thread t adds the
        // shares t / R, t / R + 256 / R, ... of row t % R (R = 16 rows, or 32), thread r < R the sums of row r
        __shared__ float inv_s[32], part_s[256];
        row_inv = inv_s;
        if (row_parts) {
            const int r = threadIdx.x % rs_rows, g = threadIdx.x / rs_rows;
            float mine = 0.f;
#pragma unroll
            for (int i = 0; i < RS_PER; ++i) mine += (g + rs_groups * i < nparts) ? rs_part[i] : 0.f;
            part_s[g * rs_rows + r] = mine;
            __syncthreads();
            if ((int)threadIdx.x < rs_rows) {
                float sq = part_s[threadIdx.x];
                for (int q = 1; q < rs_groups; ++q) sq += part_s[q * rs_rows + threadIdx.x];
                inv_s[threadIdx.x] = 1.0f / sqrtf(sq / (float)K + eps);
            }
            __syncthreads();
        }
    }
    if constexpr (SWSPLIT) {
        // every wave leaves its sums in its band; of two waves side by side the first then takes rows 0 .. 15
        // of the 32 and the second rows 16 .. 31: gates from the first wave's band, ups from the second's
        constexpr int ES = WN + 4;
        static_assert(4 * 32 * ES * 4 <= NSTAGE * STAGE * 2, "the waves' bands fit the main loop's LDS");
        float* bands = reinterpret_cast<float*>(lds);
        float* band = bands + wave * 32 * ES;
        const float* gband = bands + (wave & ~1) * 32 * ES;
        const float* uband = bands + (wave | 1) * 32 * ES;
        const int ccol = lane & 31, crow = (lane >> 5) * 4;
        constexpr int LPR = WN / 8, RPP = 64 / LPR;
        const int erow = lane / LPR, ecol = (lane % LPR) * 8;
        const int NO = N / 2;
        const int col = n0 / 2 + ecol;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if (i > 0) __syncthreads();              // (the bands have been read)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    band[(8 * (r >> 2) + crow + (r & 3)) * ES + 32 * j + ccol] = acc[i][j][r];
            __syncthreads();
#pragma unroll
            for (int pass = 0; pass < (16 + RPP - 1) / RPP; ++pass) {
                const int rr = RPP * pass + erow;
                const int row = m0 + wm + 32 * i + 16 * (wave & 1) + rr;
                if (erow >= RPP || rr >= 16 || row >= M || col >= NO) continue;
                const float* gs = &gband[(16 * (wave & 1) + rr) * ES + ecol];
                const float* us = &uband[(16 * (wave & 1) + rr) * ES + ecol];
                float v[8];
                float f = 1.0f;
                if constexpr (ROWSCALE) f = row_parts ? row_inv[row & 31] : 1.0f;      // (row_parts: M <= 32, so row < 32 here)
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = gated_bf16<ACT>(gs[e] * f, us[e] * f, ep);
                const size_t o_idx = (size_t)row * NO + col;
                if (col + 8 <= NO && (NO % 8) == 0) {
                    chunk16 o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) o.w[e] = pack2_bf16(v[2 * e], v[2 * e + 1]);
                    *reinterpret_cast<chunk16*>(reinterpret_cast<uint16_t*>(out) + o_idx) = o;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (col + e < NO) epilogue_store(out, o_idx + e, v[e], nullptr, col + e, 0);
                }
            }
        }
        return;
    }
    constexpr int EW = SWIGLU ? WN / 2 : WN;        // output columns of a wave
    constexpr int ESTRIDE = EW + 4;
    static_assert(4 * 32 * ESTRIDE * 4 <= NSTAGE * STAGE * 2, "the waves' bands fit the main loop's LDS");
    float* band = reinterpret_cast<float*>(lds) + wave * 32 * ESTRIDE;
    const int ccol = lane & 31, crow = (lane >> 5) * 4;
    // (band_to_memory's work, in line: as that function these kernels' tiles ended 0.35 to 0.45 us later, 641 x 768 x 448 with squared ReLU
    // 7.75 -> 8.1 us, 2,531 x 10,560 x 128 33.0 -> 35.6)
    constexpr int LPR = EW / 8, RPP = 64 / LPR;     // lanes a row of the band takes; rows a pass of the wave covers
    const int erow = lane / LPR, ecol = (lane % LPR) * 8;      // (where 64 is no multiple of LPR the last lanes idle)
    const int NO = SWIGLU ? N / 2 : N;             // columns of out
    const int col = (SWIGLU ? (n0 + wn) / 2 : n0 + wn) + ecol;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        __builtin_amdgcn_wave_barrier();
        if constexpr (SWIGLU) {
#pragma unroll
            for (int j = 0; j < TN; j += 2)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float gv = acc[i][j][r], uv = acc[i][j + 1][r];
                    if constexpr (ROWSCALE) {
                        if (row_parts) {                 // (M <= 32: only the tile's first 32 rows are written)
                            const float f = row_inv[(wm + 32 * i + 8 * (r >> 2) + crow + (r & 3)) & 31];
                            gv *= f;
                            uv *= f;
                        }
                    }
                    band[(8 * (r >> 2) + crow + (r & 3)) * ESTRIDE + 16 * j + ccol] = gated_bf16<ACT>(gv, uv, ep);
                }
        } else {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    band[(8 * (r >> 2) + crow + (r & 3)) * ESTRIDE + 32 * j + ccol] = acc[i][j][r];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int pass = 0; pass < (32 + RPP - 1) / RPP; ++pass) {
            const int row = m0 + wm + 32 * i + RPP * pass + erow;
            if (erow >= RPP || RPP * pass + erow >= 32 || row >= M || col >= NO) continue;
            const float* src = &band[(RPP * pass + erow) * ESTRIDE + ecol];
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = src[e];
            const size_t o_idx = (size_t)row * NO + col;
            if constexpr (ACT != 0 && !SWIGLU) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = activation(v[e] + (bias && col + e < NO ? bias[col + e] : 0.f), LiAct{ACT, ep.a0, ep.a1});
                if (col + 8 <= NO && (NO % 8) == 0) {
                    chunk16 o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) o.w[e] = pack2_bf16(v[2 * e], v[2 * e + 1]);
                    *reinterpret_cast<chunk16*>(reinterpret_cast<uint16_t*>(out) + o_idx) = o;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (col + e < NO) epilogue_store(out, o_idx + e, v[e], nullptr, col + e, 0);
                }
                continue;
            }
            if (col + 8 <= NO && (NO % 8) == 0) {
                if (bias) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] += bias[col + e];
                }
                if constexpr (sizeof(TO) == 4) {
                    float4* o = reinterpret_cast<float4*>(reinterpret_cast<float*>(out) + o_idx);
                    if (accumulate != 0.f) {
                        const float4 a0 = o[0], a1 = o[1];
                        v[0] = fmaf(accumulate, v[0], a0.x); v[1] = fmaf(accumulate, v[1], a0.y); v[2] = fmaf(accumulate, v[2], a0.z); v[3] = fmaf(accumulate, v[3], a0.w);
                        v[4] = fmaf(accumulate, v[4], a1.x); v[5] = fmaf(accumulate, v[5], a1.y); v[6] = fmaf(accumulate, v[6], a1.z); v[7] = fmaf(accumulate, v[7], a1.w);
                    }
                    o[0] = float4{v[0], v[1], v[2], v[3]};
                    o[1] = float4{v[4], v[5], v[6], v[7]};
                } else {
                    chunk16 o;
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        o.w[e] = pack2_bf16(v[2 * e], v[2 * e + 1]);
                    *reinterpret_cast<chunk16*>(reinterpret_cast<uint16_t*>(out) + o_idx) = o;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (col + e < NO) epilogue_store(out, o_idx + e, v[e], bias, col + e, accumulate);
            }
        }
    }
}

template <int BM, int BN, int BK, int NSTAGE, bool SWIGLU, typename TO, int ACT = 0, int WLM = 2>
static int launch_dma(const bf16_t* x, const bf16_t* w, const float* bias, TO* out, int M, int N, int K,
                      float accumulate, hipStream_t stream, int nsplit = 1, const float* row_parts = nullptr,
                      int nparts = 0, float eps = 0.f, LiAct ep = {}) {
    if (row_parts && !(SWIGLU && BM == 64 && M <= 32 && nparts > 0)) return LI_ERR_SIZE;
    const long mtiles = (M + BM - 1) / BM, ntiles = (N + BN - 1) / BN;
    if (nsplit < 1 || nsplit > 65535 || nsplit > K / BK) return LI_ERR_SIZE;
    const long blocks = TileOrder::blocks(mtiles, ntiles, nsplit);
    if (blocks > 0x7fffffffL) return LI_ERR_SIZE;
    // a lane's byte offset from its tile's first row is kept in 32 bits (the gate and up rows of a
    // SwiGLU tile lie N / 2 rows apart)
    const unsigned long long span_rows = SWIGLU ? (unsigned long long)N / 2 + BN : (unsigned long long)(BM > BN ? BM : BN);
    if (span_rows * (unsigned long long)K * 2ull >= (1ull << 32)) return LI_ERR_SIZE;
    constexpr int lds_bytes = NSTAGE * (BM + BN) * BK * 2;
    static bool configured = false;
    if (!configured) {
        if (hipFuncSetAttribute((const void*)gemm_bf16_dma_kernel<BM, BN, BK, NSTAGE, SWIGLU, TO, ACT, WLM>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
            return LI_ERR_LAUNCH;
        configured = true;
    }
    gemm_bf16_dma_kernel<BM, BN, BK, NSTAGE, SWIGLU, TO, ACT, WLM><<<(unsigned)blocks, 256, lds_bytes, stream>>>(x, w, bias, out, M, N, K, accumulate, nsplit, row_parts, nparts, eps, ep);
    return li_launch_status();
}

// ------------------------------- bfloat16, more than 64 rows: tiles of a block, two by two waves
// A block of four waves, one a SIMD, makes a tile of BM x BN; a step is 64 k-values, and NSTAGE stages lie in LDS,
// filled by loads that go straight there.  What bounds it is the time between a load's issue and its arrival (a thousand
// and more clocks under load): a wave is alone on its SIMD, so whatever it waits for, the matrix cores wait for too.  With
// whole stages handed back once a step (the form before) 8,192^3 kept the matrix cores busy 60 % of the time at 1.88 GHz.
// So a stage is handed back in pieces.  A wave's part of the tile is cut in two both ways; each of the four pieces is
// multiplied for the whole step, in an order in which one operand stays (quarter (0, X), (0, Y), (1, Y), (1, X) of rows
// and columns, X and Y the halves of the columns, which change places from step to step), and while it is multiplied the
// operand that the NEXT quarter needs anew is read from LDS, into the registers of the half that is dead by then:
//     quarter     multiplies    reads                   asks memory for, NSTAGE steps ahead
//     0           (0, X)        B half Y                A half 0
//     1           (0, Y)        A half 1                B half X         then a barrier
//     2           (1, Y)        A half 0, next step     B half Y
//     3           (1, X)        B half Y, next step     A half 1         then a barrier
// Half of the stage has been read at each barrier and its place is asked for again at once: the loads are spread evenly over the
// whole step, and no register holds an operand twice: 128 registers of operands beside the 256 of the sums.  What step kt
// asks for is step kt + NSTAGE's.  Of that, A half 0 and the B half that is multiplied first are waited for in the middle of step
// kt + NSTAGE - 1, the rest at its end.  So A half 0 and, with an even number of stages, B half X have NSTAGE - 1 steps and up to half a
// step more to arrive, B half Y the same from the middle on, A half 1 NSTAGE - 1 steps and the rest of its quarter.
// Multiplied by v_mfma_f32_16x16x32_bf16: with operands as they are in use the chip is at its power limit here, and this
// form draws less for the same product than the 32 x 32 x 16 one (a loop of nothing else 1.90 against 1.75 PFLOP/s).
// The MFMAs are assembly so that a sum stays in its registers: the instruction's result may lie elsewhere, and the compiler
// made use of that, with some 600 moves between registers a step and spills.  What it then does not see is seen to
// here: operands come from LDS reads alone, which it waits for as for any use; the same sum comes up again after four
// MFMAs at least; and before the sums are read behind the loop, two waits of 16 cycles pass.  The build looks the assembly
// of every instance through and refuses one in which a sum is moved or spilled before that.
// A half's rows of a stage: first those of the waves of the first row (column) of waves, then the others'.
// ... by the lanes that are told: all, or none (a step past the last asks for nothing, but counts as the others do)
#define LI_LOAD_TO_LDS_BY(lanes, base, voff, lptr)                                                       \
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_lo, %3\n\ts_mov_b32 exec_hi, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"   \
                 :: "s"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)(lptr)), "v"(voff), "s"(base), "s"(lanes) : "memory", "m0")

template <int BM, int BN, int NSTAGE, bool SWIGLU, typename TO, int ACT = 0>
__global__ __launch_bounds__(256) void gemm_bf16_tile_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                              const float* __restrict__ bias, TO* __restrict__ out, int M, int N, int K,
                                                              float accumulate, LiAct ep) {
    // ACT: an activation, of gate and up columns (see gated_bf16) or of the sums (its number); its constants are in `ep`
    constexpr int BK = 64;
    constexpr int TM = BM / 32, TN = BN / 32;                    // 16-row and 16-column pieces of a wave
    static_assert(BM % 64 == 0 && BN % 32 == 0 && NSTAGE >= 2, "bands of 32 rows a wave, pieces of 16 columns");
    static_assert(!SWIGLU || TN % 2 == 0, "gate and up columns in turn, 16 of each");
    constexpr int WM = 16 * TM, WN = 16 * TN;
    constexpr int STAGE = (BM + BN) * BK, LPW = TM + TN;         // elements of a stage; loads a wave issues for it
    // (a set of T pieces a wave is 32 T rows of a stage, 4 T load instructions of 8 rows, T of them a wave's)
    struct Half { int a0, a1, b0, b1; };
    constexpr Half T{(TM + 1) / 2, TM / 2, (TN + 1) / 2, TN / 2};
    constexpr int TA[2] = {T.a0, T.a1}, TB[2] = {T.b0, T.b1};
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wi = wave >> 1, wj = wave & 1;
    const int mtiles = (M + BM - 1) / BM, ntiles = (N + BN - 1) / BN;
    int mt, nt, split;
    if (!TileOrder(mtiles).tile(blockIdx.x, mtiles, ntiles, 1, mt, nt, split)) return;
    const int m0 = mt * BM, n0 = nt * BN;
    const int half_n = N / 2;                                    // (SWIGLU: w is [gate; up] of N / 2 rows each)

    // a lane's part of a load: the row of x or w, from the tile's first, as a byte offset that never changes
    uint32_t ga[TM], gb[TN];
    const bf16_t* abase = x + (size_t)m0 * K;
    const bf16_t* bbase = w + (size_t)(SWIGLU ? n0 / 2 : n0) * K;
    const int sub = lane >> 3;                                   // row of the 8 of an instruction
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int h = i < TA[0] ? 0 : 1, t = TA[h];
        const int in = (wave * t + (i - h * TA[0])) * 8 + sub;   // row within the half
        const int row = (in / (16 * t)) * WM + h * TA[0] * 16 + in % (16 * t);
        const int c = (lane & 7) ^ (in & 7);
        ga[i] = (uint32_t)(((size_t)(m0 + row < M ? row : M - 1 - m0) * K + 8 * c) * 2);       // rows past the end: the last row
    }
#pragma unroll
    for (int i = 0; i < TN; ++i) {
        const int h = i < TB[0] ? 0 : 1, t = TB[h];
        const int in = (wave * t + (i - h * TB[0])) * 8 + sub;
        const int col = (in / (16 * t)) * WN + h * TB[0] * 16 + in % (16 * t);
        const int c = (lane & 7) ^ (in & 7);
        size_t rel = n0 + col < N ? col : N - 1 - n0;
        if constexpr (SWIGLU) {                                  // 16 gate rows, the 16 up rows of the same outputs, and so on
            const int o = n0 / 2 + (col / 32) * 16 + col % 16;
            rel = (size_t)((o < half_n ? o : half_n - 1) - n0 / 2) + (size_t)((col >> 4) & 1) * half_n;
        }
        gb[i] = (uint32_t)((rel * K + 8 * c) * 2);
    }
    const int nk = K / BK;
    // a step that there is: all lanes (the loads of a step past the last count like any other, but ask for nothing)
    auto lanes_of = [&](int t) { return __builtin_amdgcn_readfirstlane((t - nk) >> 31); };

    // loads l of a step: A half 0, B half X, B half Y, A half 1 (X = par), in the order they are issued
    auto issue_one = [&](auto par_tag, auto l_tag, int stage, int kt, int lanes) {
        constexpr int X = decltype(par_tag)::value, Y = X ^ 1, l = decltype(l_tag)::value;
        constexpr bool is_a = l < TA[0] || l >= TA[0] + TB[0] + TB[1], second = l >= TA[0] + TB[X];
        constexpr int h = is_a ? (l < TA[0] ? 0 : 1) : (second ? Y : X);
        constexpr int i = is_a ? (h ? l - TA[0] - TB[0] - TB[1] : l) : l - TA[0] - (second ? TB[X] : 0);
        constexpr int t = is_a ? TA[h] : TB[h], first = is_a ? h * TA[0] : h * TB[0];
        const bf16_t* base = (is_a ? abase : bbase) + (size_t)kt * BK;
        const uint32_t off = is_a ? ga[is_a ? first + i : 0] : gb[is_a ? 0 : first + i];
        uint16_t* to = lds + stage * STAGE + ((is_a ? 0 : BM) + first * 32 + (wave * t + i) * 8) * BK;
        LI_LOAD_TO_LDS_BY(lanes, base, off, to);
    };
    // (the sums start as products of zeros: like this they are in the matrix cores' registers from the first to the last)
    floatx4 acc[TM][TN];
    bf16x8 none = {0, 0, 0, 0, 0, 0, 0, 0};
    asm volatile("s_nop 4" : "+v"(none));                        // (written by the vector ALU: a few cycles before the MFMAs may read it)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %1, 0" : "=a"(acc[i][j]) : "v"(none));
    bf16x8 af[TM][2], bf[TN][2];                                 // a step's operands: [piece][first or second 32 k-values]
    // a lane's place in a piece of 16 rows: row lane % 16, the 8 k-values of group lane / 16 (of 4 in 32)
    const int place0 = (lane & 15) * BK + (((lane >> 4) ^ (lane & 7)) << 3), place1 = place0 ^ 32;
    auto read_a = [&](int i, int kk, int stage) {
        const int h = i < TA[0] ? 0 : 1;
        af[i][kk] = *reinterpret_cast<const bf16x8*>(&lds[stage * STAGE + (h * TA[0] * 32 + wi * TA[h] * 16 + (i - h * TA[0]) * 16) * BK + (kk ? place1 : place0)]);
    };
    auto read_b = [&](int j, int kk, int stage) {
        const int h = j < TB[0] ? 0 : 1;
        bf[j][kk] = *reinterpret_cast<const bf16x8*>(&lds[stage * STAGE + (BM + h * TB[0] * 32 + wj * TB[h] * 16 + (j - h * TB[0]) * 16) * BK + (kk ? place1 : place0)]);
    };
    // (a wave's loads retire in order: allowing the younger ones waits exactly for the oldest; the reads of LDS are done too)
#define LI_ARRIVED(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | 0x0070)
#define LI_MEET()                                                                                          \
    { asm volatile("" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); }
    static_assert((NSTAGE - 1) * LPW <= 63, "vmcnt counts to 63");
    static_for<NSTAGE>([&](auto t_tag) {                         // (as if issued NSTAGE steps earlier)
        constexpr int t = decltype(t_tag)::value;
        const int lanes = lanes_of(t);
        static_for<LPW>([&](auto l_tag) { issue_one(std::integral_constant<int, (t + NSTAGE) & 1>{}, l_tag, t, t, lanes); });
    });
    // Steps are taken two by two: behind an odd number of them comes one of zeros
    auto zeros = [&](int stage) {
        for (int i = tid; i < STAGE / 8; i += 256) *reinterpret_cast<uint4*>(&lds[stage * STAGE + 8 * i]) = uint4{0u, 0u, 0u, 0u};
    };
    if (nk & 1 && nk < NSTAGE) zeros(nk);
    LI_ARRIVED((NSTAGE - 1) * LPW);
    LI_MEET()
#pragma unroll
    for (int i = 0; i < TA[0]; ++i) { read_a(i, 0, 0); read_a(i, 1, 0); }
#pragma unroll
    for (int j = 0; j < TB[0]; ++j) { read_b(j, 0, 0); read_b(j, 1, 0); }
    __builtin_amdgcn_s_waitcnt(0xC07F);                          // lgkmcnt(0)
    LI_MEET()
    // step kt, X = par (the last one reads a next stage that is not multiplied)
    auto step = [&](auto par_tag, int kt, int stage, int next) {
        constexpr int X = decltype(par_tag)::value, Y = X ^ 1;
        const int lanes = lanes_of(kt + NSTAGE);
        constexpr int H1 = TA[0] + TB[X], H2 = TB[Y] + TA[1];
        // quarter q of rows ah and columns bh; reads: half rh of A (or B) from stage rs; loads l0 .. l1 of the step
        auto quarter = [&](auto ah_t, auto bh_t, auto isa_t, auto rh_t, int rs, auto l0_t, auto l1_t) {
            constexpr int ah = decltype(ah_t)::value, bh = decltype(bh_t)::value, rh = decltype(rh_t)::value;
            constexpr bool isa = decltype(isa_t)::value;
            constexpr int l0 = decltype(l0_t)::value, NL = decltype(l1_t)::value - l0;
            constexpr int P = TA[ah] * TB[bh], G = 2 * P;        // MFMAs: all pieces for the first 32 k-values, then for the others
            constexpr int R = 2 * (isa ? TA[rh] : TB[rh]);
            constexpr int GR = G * 5 / 8 > 0 ? G * 5 / 8 : 1;    // the reads go out before the first five eighths of them
            static_for<G>([&](auto m_tag) {
                constexpr int m = decltype(m_tag)::value;
                constexpr int r0 = m < GR ? (m * R + GR - 1) / GR : R, r1 = m + 1 < GR ? ((m + 1) * R + GR - 1) / GR : R;
                static_for<r1 - r0>([&](auto r_tag) {
                    // (the first 32 k-values of all pieces first, as they are multiplied)
                    constexpr int r = r0 + decltype(r_tag)::value, n = R / 2, p = r % (n > 0 ? n : 1), kk = r / (n > 0 ? n : 1);
                    if constexpr (isa) read_a(rh * TA[0] + p, kk, rs); else read_b(rh * TB[0] + p, kk, rs);
                });
                constexpr int kk = m / P, i = ah * TA[0] + (m % P) / TB[bh], j = bh * TB[0] + (m % P) % TB[bh];
                asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(af[i][kk]), "v"(bf[j][kk]));
                constexpr int a = l0 + (m * NL) / G, b = l0 + ((m + 1) * NL) / G;
                static_for<b - a>([&](auto l_tag) { issue_one(par_tag, std::integral_constant<int, a + decltype(l_tag)::value>{}, stage, kt + NSTAGE, lanes); });
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        constexpr std::integral_constant<int, 0> c0{};
        constexpr std::integral_constant<int, 1> c1{};
        constexpr std::integral_constant<int, X> cx{};
        constexpr std::integral_constant<int, Y> cy{};
        quarter(c0, cx, std::false_type{}, cy, stage, c0, std::integral_constant<int, H1 / 2>{});
        quarter(c0, cy, std::true_type{}, c1, stage, std::integral_constant<int, H1 / 2>{}, std::integral_constant<int, H1>{});
        // A half 0 and B half Y (the next step's X) of the next step: behind them its other loads, whole steps, this step's
        // first half.  (With an odd number of stages that B half came second among its step's B halves.)
        LI_ARRIVED((NSTAGE % 2 ? TA[1] : TB[X] + TA[1]) + (NSTAGE - 2) * LPW + H1);
        LI_MEET()
        quarter(c1, cy, std::true_type{}, c0, next, std::integral_constant<int, H1>{}, std::integral_constant<int, H1 + H2 / 2>{});
        quarter(c1, cx, std::false_type{}, cy, next, std::integral_constant<int, H1 + H2 / 2>{}, std::integral_constant<int, LPW>{});
        if (nk & 1 && kt + NSTAGE == nk) zeros(stage);
        LI_ARRIVED((NSTAGE - 1) * LPW);
        LI_MEET()
    };
    auto after = [](int s) { return s + 1 == NSTAGE ? 0 : s + 1; };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    int kt = 0, s = 0;
    do {
        const int s1 = after(s), s2 = after(s1);
        step(even, kt, s, s1);
        step(odd, kt + 1, s1, s2);
        s = s2;
        kt += 2;
    } while (kt < nk);
#undef LI_ARRIVED
#undef LI_MEET
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();                               // the main loop's LDS is free now
    constexpr int EW = SWIGLU ? WN / 2 : WN;       // output columns of a wave
    constexpr int ESTRIDE = EW + 4;                // floats of a band's row: the four groups of rows of a piece on different banks
    static_assert(4 * 32 * ESTRIDE * 4 <= NSTAGE * STAGE * 2, "the waves' bands fit the main loop's LDS");
    float* band = reinterpret_cast<float*>(lds) + wave * 32 * ESTRIDE;
    const int ccol = lane & 15, crow = (lane >> 4) * 4;
#pragma unroll
    for (int i = 0; i < TM; i += 2) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int j = 0; j < TN; j += SWIGLU ? 2 : 1)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = acc[i + u][j][r];
                    if constexpr (SWIGLU) v = gated_bf16<ACT>(v, acc[i + u][j + 1][r], ep);
                    band[(16 * u + crow + r) * ESTRIDE + (SWIGLU ? 8 : 16) * j + ccol] = v;
                }
        __builtin_amdgcn_wave_barrier();
        band_to_memory<EW, ESTRIDE, SWIGLU, ACT, TO>(band, m0 + wi * WM + 16 * i, (SWIGLU ? n0 / 2 : n0) + wj * EW, M,
                                                     SWIGLU ? N / 2 : N, SWIGLU ? nullptr : bias, out, SWIGLU ? 0.f : accumulate, ep);
    }
}

template <int BM, int BN, int NSTAGE, bool SWIGLU, typename TO, int ACT = 0>
static int launch_tile(const bf16_t* x, const bf16_t* w, const float* bias, TO* out, int M, int N, int K,
                       float accumulate, hipStream_t stream, LiAct ep = {}) {
    const long mtiles = (M + BM - 1) / BM, ntiles = (N + BN - 1) / BN;
    if (K % 64) return LI_ERR_SIZE;
    const long blocks = TileOrder::blocks(mtiles, ntiles);
    if (blocks > 0x7fffffffL) return LI_ERR_SIZE;
    // a lane's byte offset from its tile's first row is kept in 32 bits (the gate and up rows of a
    // SwiGLU tile lie N / 2 rows apart)
    const unsigned long long span_rows = SWIGLU ? (unsigned long long)N / 2 + BN : (unsigned long long)(BM > BN ? BM : BN);
    if (span_rows * (unsigned long long)K * 2ull >= (1ull << 32)) return LI_ERR_SIZE;
    constexpr int lds_bytes = NSTAGE * (BM + BN) * 64 * 2;
    static bool configured = false;
    if (!configured) {
        if (hipFuncSetAttribute((const void*)gemm_bf16_tile_kernel<BM, BN, NSTAGE, SWIGLU, TO, ACT>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
            return LI_ERR_LAUNCH;
        configured = true;
    }
    gemm_bf16_tile_kernel<BM, BN, NSTAGE, SWIGLU, TO, ACT><<<(unsigned)blocks, 256, lds_bytes, stream>>>(x, w, bias, out, M, N, K, accumulate, ep);
    return li_launch_status();
}

// The sum of up to PARTS_HELD parts, or with MORE up to MID_PARTS, in their order.  All loads at once (a part past the last reads the first and
// is not added): the kernels that add up have few blocks and must not wait for memory part after part.  MORE goes by the number of parts, not
// by the rows: the question inside the kernel made a step of 1,027 tokens 4 % longer, and one of 33 to 64 rows with 8 parts and fewer 2 to 3 %.
#define PARTS_HELD 8
#define MID_PARTS 16
template <bool MORE>
struct Parts {
    float a[PARTS_HELD], b[MORE ? PARTS_HELD : 1];
    // (asked for before what else a kernel needs, whose addresses take a division: a tanh norm of 33 to 64 rows 2 to 4 % longer the other way)
    __device__ __forceinline__ void ask(const float* __restrict__ part, int nsplit, size_t mn, size_t at) {
#pragma unroll
        for (int sp = 0; sp < PARTS_HELD; ++sp) a[sp] = part[(size_t)(sp < nsplit ? sp : 0) * mn + at];
        if constexpr (MORE) {
#pragma unroll
            for (int sp = 0; sp < PARTS_HELD; ++sp) b[sp] = part[(size_t)(PARTS_HELD + sp < nsplit ? PARTS_HELD + sp : 0) * mn + at];
        }
    }
    __device__ __forceinline__ float sum(int nsplit) const {
        float t = a[0];
#pragma unroll
        for (int sp = 1; sp < PARTS_HELD; ++sp) t += sp < nsplit ? a[sp] : 0.f;
        if constexpr (MORE) {
#pragma unroll
            for (int sp = 0; sp < PARTS_HELD; ++sp) t += PARTS_HELD + sp < nsplit ? b[sp] : 0.f;
        }
        return t;
    }
};
static_assert(MID_PARTS == 2 * PARTS_HELD, "every part that a product is cut into is added up");

// out (+)= sum over the parts, in the order of the parts, + bias: of few rows (all parts at once; one after another they were a chain of trips to
// memory: 33 to 64 rows of 2,048 x 11,008, 16 parts, product included, 18.4 -> 15.9 us, of 896 x 4,864, 8 parts, 11.1 -> 9.9), and of many
template <typename TO, bool MORE>
__global__ __launch_bounds__(256) void splitk_reduce_few_kernel(const float* __restrict__ part, int nsplit, size_t mn, int N,
                                                                const float* __restrict__ bias, TO* __restrict__ out, float accumulate) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= mn) return;
    Parts<MORE> parts;
    parts.ask(part, nsplit, mn, i);
    epilogue_store(out, i, parts.sum(nsplit), bias, (int)(i % N), accumulate);
}
template <typename TO>
__global__ void splitk_reduce_kernel(const float* __restrict__ part, int nsplit, size_t mn, int N,
                                     const float* __restrict__ bias, TO* __restrict__ out, float accumulate) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= mn) return;
    float v = part[i];
    for (int s = 1; s < nsplit; ++s) v += part[(size_t)s * mn + i];
    epilogue_store(out, i, v, bias, (int)(i % N), accumulate);
}

// out = act(sum over the parts + bias), bfloat16 (see li_linear_act)
template <bool MORE>
__global__ __launch_bounds__(256) void splitk_reduce_act_kernel(const float* __restrict__ part, int nsplit, size_t mn, int N,
                                                                const float* __restrict__ bias, bf16_t* __restrict__ out, LiAct ep) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= mn) return;
    Parts<MORE> parts;
    parts.ask(part, nsplit, mn, i);
    float v = parts.sum(nsplit);
    if (bias) v += bias[(int)(i % N)];
    store_from_float(out + i, activation(v, ep));
}

// The same of one part, four values a thread (GELU, 64 x 20,000 x 1,024, product included: 16.8 us, 18.2 with the kernel above)
__global__ __launch_bounds__(256) void act_of_sums_kernel(const float* __restrict__ sums, size_t mn, int N, const float* __restrict__ bias,
                                                          bf16_t* __restrict__ out, LiAct ep) {
    const size_t i = 4 * ((size_t)blockIdx.x * 256 + threadIdx.x);
    if (i >= mn) return;
    float v[4];
    if (i + 4 <= mn) {
        const floatx4 a = *reinterpret_cast<const floatx4*>(sums + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = a[e];
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = i + e < mn ? sums[i + e] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (i + e >= mn) continue;
        store_from_float(out + i + e, activation(v[e] + (bias ? bias[(int)((i + e) % N)] : 0.f), ep));
    }
}

// The same for the residual sum, one block a row, with the RMS norm of the new sum as a second
// result: out[m, :] += factor * (sum of the parts + bias) (float32), xn[m, :] = gamma * out[m, :] /
// sqrt(mean(out[m, :]^2) + eps).  A row is kept in registers (N <= NT * PER).
// THERE: the sum is in `out` already, and its norm alone is written (nsplit does not matter).
template <typename TN, int NT, int PER, bool FEW, bool MORE, bool THERE = false>
__global__ __launch_bounds__(NT) void splitk_reduce_norm_kernel(const float* __restrict__ part, int nsplit, size_t mn, int N,
                                                                 const float* __restrict__ bias, float* __restrict__ out,
                                                                 float factor, const float* __restrict__ gamma, float eps,
                                                                 TN* __restrict__ xn) {
    __shared__ float red[NT / LI_WAVE];
    const size_t row = (size_t)blockIdx.x * N;
    float v[PER];
    [[maybe_unused]] float g[PER];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i)                       // (few rows: the norm's weights come with the parts, not behind the sum of squares)
        if (FEW && i * NT < N) g[i] = gamma[(int)threadIdx.x + i * NT < N ? threadIdx.x + i * NT : N - 1];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int n = threadIdx.x + i * NT;
        v[i] = 0.f;
        if constexpr (THERE) {
            if (n < N) v[i] = out[row + n];
        } else if (n < N) {
            Parts<MORE> parts;
            parts.ask(part, nsplit, mn, row + n);
            const float o = out[row + n];
            float t = parts.sum(nsplit);
            if (bias) t += bias[n];
            t = fmaf(factor, t, o);
            out[row + n] = t;
            v[i] = t;
        }
        ss += v[i] * v[i];
    }
    ss = block_sum<NT>(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)N + eps);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int n = threadIdx.x + i * NT;
        if (n < N) store_from_float(xn + row + n, (FEW ? g[i] : gamma[n]) * v[i] * inv);
    }
}

// The same of many rows, whose time is their bytes: a thread takes PER pieces of four columns and asks for the parts that there are (HELD: 2, 4 or
// 8 of them), a block is four waves, of which a unit holds eight.  (Blocks of 1,024 threads, of which 1,536 columns leave five waves of
// sixteen idle in the second round, one column a load and eight loads whatever the parts: 1,027 x 1,536 columns of two parts 9.4 us, now 6.6; the product
// with it, K 1,536 22.1 -> 19.1, 8,960 47.4 -> 45.8, 700 x 896 x 4,864 21.3 -> 19.9.  Below 256 rows those blocks: 100 x 1,536 x 8,960 19.3 / 19.8.)  N a
// multiple of 4, up to 1,024 PER.
#define REDUCE_ROWS_NT 256
#define REDUCE_ROWS_FROM 256
// Not where a unit has one row (256 rows) and this is long, nor, below 600 rows, where a quarter of the threads has one piece of many parts less than
// the others: us, the product with those blocks / with these, 256 x 2,048 x 4,864 (8 parts) 20.3 / 20.7, 256 x 3,584 x 4,864 (4) 25.1 / 25.5, 280 x 1,536 x
// 8,960 (7) 23.1 / 23.9, 450 (5) 28.1 / 28.7, 700 (3) 35.1 / 34.2, 280 x 2,048 x 4,864 (5) 23.7 / 23.4.
static bool reduce_by_rows(int M, int N, int nsplit) {
    if (nsplit > 4 && N > 1024 && N < 2048) return M >= 600;
    return M > REDUCE_ROWS_FROM || (M == REDUCE_ROWS_FROM && N * nsplit <= 6144);
}
template <int HELD, int PER>
__global__ __launch_bounds__(REDUCE_ROWS_NT) void splitk_reduce_norm_rows_kernel(const float* __restrict__ part, int nsplit, size_t mn, int N,
                                                                                  const float* __restrict__ bias, float* __restrict__ out,
                                                                                  float factor, const float* __restrict__ gamma, float eps,
                                                                                  bf16_t* __restrict__ xn) {
    __shared__ float red[REDUCE_ROWS_NT / LI_WAVE];
    const size_t row = (size_t)blockIdx.x * N;
    floatx4 v[PER], a[PER][HELD], o[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int n = 4 * (threadIdx.x + i * REDUCE_ROWS_NT), at = n < N ? n : 0;      // (never conditional: a piece past the end reads the first)
#pragma unroll
        for (int sp = 0; sp < HELD; ++sp) a[i][sp] = *reinterpret_cast<const floatx4*>(part + (size_t)(sp < nsplit ? sp : 0) * mn + row + at);
        o[i] = *reinterpret_cast<const floatx4*>(out + row + at);
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int n = 4 * (threadIdx.x + i * REDUCE_ROWS_NT);
        v[i] = a[i][0];
#pragma unroll
        for (int sp = 1; sp < HELD; ++sp)
            if (sp < nsplit) v[i] += a[i][sp];
        if (n < N) {
            if (bias) v[i] += *reinterpret_cast<const floatx4*>(bias + n);
#pragma unroll
            for (int e = 0; e < 4; ++e) { v[i][e] = fmaf(factor, v[i][e], o[i][e]); ss = fmaf(v[i][e], v[i][e], ss); }
            *reinterpret_cast<floatx4*>(out + row + n) = v[i];
        }
    }
    ss = block_sum<REDUCE_ROWS_NT>(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)N + eps);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int n = 4 * (threadIdx.x + i * REDUCE_ROWS_NT);
        if (n >= N) continue;
        const floatx4 g = *reinterpret_cast<const floatx4*>(gamma + n);
        floatx4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = g[e] * v[i][e] * inv;
        *reinterpret_cast<uint2*>(xn + row + n) = uint2{pack2_bf16(y[0], y[1]), pack2_bf16(y[2], y[3])};
    }
}
template <int HELD>
static void launch_reduce_norm_rows(const float* part, int nsplit, int M, int N, const float* bias, float* out, float factor, const float* gamma, float eps, bf16_t* xn,
                                    hipStream_t stream) {
    const size_t mn = (size_t)M * N;
    if (N <= 1024) splitk_reduce_norm_rows_kernel<HELD, 1><<<M, REDUCE_ROWS_NT, 0, stream>>>(part, nsplit, mn, N, bias, out, factor, gamma, eps, xn);
    else if (N <= 2048) splitk_reduce_norm_rows_kernel<HELD, 2><<<M, REDUCE_ROWS_NT, 0, stream>>>(part, nsplit, mn, N, bias, out, factor, gamma, eps, xn);
    else if (N <= 4096) splitk_reduce_norm_rows_kernel<HELD, 4><<<M, REDUCE_ROWS_NT, 0, stream>>>(part, nsplit, mn, N, bias, out, factor, gamma, eps, xn);
    else splitk_reduce_norm_rows_kernel<HELD, 8><<<M, REDUCE_ROWS_NT, 0, stream>>>(part, nsplit, mn, N, bias, out, factor, gamma, eps, xn);
}

// The same with a tanh norm, which takes no statistics of a row: out += factor * (sum of the parts + bias) (float32),
// xn = tanh(alpha * out) * gamma + beta, element by element.
template <typename TN, bool MORE>
__global__ __launch_bounds__(256) void splitk_reduce_tanh_kernel(const float* __restrict__ part, int nsplit, size_t mn, int N,
                                                                 const float* __restrict__ bias, float* __restrict__ out,
                                                                 float factor, float alpha, const float* __restrict__ gamma,
                                                                 const float* __restrict__ beta, TN* __restrict__ xn) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= mn) return;
    Parts<MORE> parts;
    parts.ask(part, nsplit, mn, i);
    const int n = (int)(i % N);
    const float o = out[i], g = gamma[n], b = beta[n];
    float t = parts.sum(nsplit);
    if (bias) t += bias[n];
    t = fmaf(factor, t, o);
    out[i] = t;
    store_from_float(xn + i, fmaf(tanhf(alpha * t), g, b));
}
#define REDUCE_NORM_NT 1024
#define REDUCE_NORM_PER 8

template <int BM, int BN, int BK, typename TO>
static int launch_big(const bf16_t* x, const bf16_t* w, const float* bias, TO* out, int M, int N, int K,
                      float accumulate, hipStream_t stream) {
    const long mtiles = (M + BM - 1) / BM, ntiles = (N + BN - 1) / BN;
    const long per_xcd = TileOrder::blocks(mtiles, ntiles) / 8;
    if (per_xcd * 8 > 0x7fffffffL) return LI_ERR_SIZE;
    dim3 grid((unsigned)(per_xcd * 8));
    constexpr int lds_bytes = 2 * (BM + BN) * BK * 2;
    static bool configured = false;
    if (!configured) {
        if (hipFuncSetAttribute((const void*)gemm_bf16_big_kernel<BM, BN, BK, TO>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
            return LI_ERR_LAUNCH;
        configured = true;
    }
    gemm_bf16_big_kernel<BM, BN, BK, TO><<<grid, 256, lds_bytes, stream>>>(x, w, bias, out, M, N, K, accumulate);
    return li_launch_status();
}

// ------------------------------------------------- bfloat16, few rows (decode): few_rows.h
// Up to 16 rows against a matrix of few columns (or rotation pairs: `unit` is 16 columns or 8 pairs a
// tile): a compute unit takes in what its blocks ask for at a rate of its own, far below its share of
// the memory's rate times the number of units, so the time of such a product is that of the unit with the
// most blocks.  Every unit therefore gets one block and every block the same number of columns (at
// most two tiles' worth, at least a quarter of a tile's), not whole tiles.  (At least a quarter, where a half was: 896 x 4,864 at one row
// 6.05 -> 5.53 us with twice the blocks.)
static int balanced_per_block(int total, int unit, int cu) {
    int per = (total + cu - 1) / cu;
    per = per < unit / 4 ? unit / 4 : per;
    return per > 2 * unit ? 0 : per;
}

// Whether a product of few rows goes to gemm_bf16_rows_kernel (columns: the matrix's rows).  Not from five rows on, where all blocks' reading of
// x bounds both and gemm_bf16_skinny_kernel, whose loads of x are whole rows of a chunk, is as fast or faster (us, 5 rows: 896 x 896 3.5 / 3.6, 8 rows:
// 2,048 x 11,008 13.7 / 14.9); nor against a wide matrix of long rows, where its chunks, which the eight waves take in turns, read w in longer
// pieces (one row: 3,584 x 3,584 7.1 / 8.0, 5,120 x 5,120 12.1 / 13.9).  The gated product stays with it too: its blocks come two and more to a
// compute unit, where this kernel's registers leave room for fewer (17,920 x 1,536 13.1 / 14.5).
static bool rows_kernel_takes(int M, long columns, int K) {
    return M <= ROWS_KERNEL_M && K % 64 == 0 && (K <= 2048 || columns <= 2048);
}
// Columns a block of it takes on cu compute units, 1 to 16: a block has one tile of 16.  One block a unit where that is enough for them, else
// whole rounds of blocks.  0: the product is gemm_bf16_skinny_kernel's, which has blocks of two tiles.  into_sum: out is added to; such a sum comes
// out of one kernel whether or not its shares of the rows' squares are asked for, whose number goes with the columns alone (li_residual_norm_parts)
static int rows_kernel_cols(int M, int N, int K, bool into_sum, int cu) {
    if (!rows_kernel_takes(M, N, K)) return 0;
    if (N <= 16l * cu) return balanced_per_block(N, 16, cu);
    return into_sum ? 0 : balanced_round_cols(N, 16, cu);
}

template <typename TO, bool ROPE, int EPI>
static int launch_rows(const SkinnyArgs& a, int total, hipStream_t stream) {
    if (a.cols < 1 || a.cols > (ROPE ? 8 : 16)) return LI_ERR_SIZE;      // (a block writes one tile)
    const int blocks = (total + a.cols - 1) / a.cols;
    const int log_rows = a.M <= 1 ? 0 : a.M <= 2 ? 1 : 2;
    const int n = (a.K / 64 + FR_WAVES - 1) / FR_WAVES;              // a wave's units
#define LI_FR(D, LOOP, X2, X4)                                                                                                          \
    {                                                                                                                                   \
        if (log_rows <= 1) gemm_bf16_rows_kernel<TO, ROPE, EPI, D, LOOP, X2><<<blocks, FR_WAVES * 64, 0, stream>>>(a, log_rows);        \
        else gemm_bf16_rows_kernel<TO, ROPE, EPI, D, LOOP, X4><<<blocks, FR_WAVES * 64, 0, stream>>>(a, log_rows);                      \
    }
    if (n <= 4) LI_FR(4, false, 1, 2)
    else if constexpr (!ROPE) {
        if (n <= 10) LI_FR(10, false, 3, 5)
        else LI_FR(4, true, 1, 2)
    } else return LI_ERR_SIZE;
#undef LI_FR
    return li_launch_status();
}

template <bool SWIGLU, typename TO, int EPI = 0>
static int launch_skinny(SkinnyArgs a, hipStream_t stream) {
    const int M = a.M, N = a.N, cu = compute_units();
    if constexpr (!SWIGLU) {
        a.cols = rows_kernel_cols(M, N, a.K, a.accumulate != 0.f, cu);
        if (a.cols > 0) return launch_rows<TO, false, EPI>(a, N, stream);
    }
#define LI_SK(MT, NT, WV) gemm_bf16_skinny_kernel<MT, NT, WV, SWIGLU, TO, false, EPI><<<(N + 16 * (SWIGLU ? 1 : NT) - 1) / (16 * (SWIGLU ? 1 : NT)), WV * 64, 0, stream>>>(a)
    if constexpr (SWIGLU) {
        a.cols = balanced_round_cols(N, 16, cu);
        const int blocks = (N + a.cols - 1) / a.cols;
        if (M <= 16) gemm_bf16_skinny_kernel<1, 2, 4, true, TO, false, EPI><<<blocks, 4 * 64, 0, stream>>>(a);
        else if (M <= 32) gemm_bf16_skinny_kernel<2, 2, 4, true, TO, false, EPI><<<blocks, 4 * 64, 0, stream>>>(a);
        else gemm_bf16_skinny_kernel<4, 2, 8, true, TO, false, EPI><<<blocks, 8 * 64, 0, stream>>>(a);
    } else if (N >= 8192) {                                 // many columns: many blocks, two tiles share each piece of x
        if (M <= 16) LI_SK(1, 2, 4); else if (M <= 32) LI_SK(2, 2, 4); else LI_SK(4, 2, 8);
    } else if (M <= 16) {                                   // few columns: a block a compute unit, eight waves split K
        a.cols = balanced_per_block(N, 16, cu);
        const int per = a.cols ? a.cols : 16, blocks = (N + per - 1) / per;
        if (per > 16) gemm_bf16_skinny_kernel<1, 2, 8, false, TO, false, EPI><<<blocks, 8 * 64, 0, stream>>>(a);
        else gemm_bf16_skinny_kernel<1, 1, 8, false, TO, false, EPI><<<blocks, 8 * 64, 0, stream>>>(a);
    } else if (M <= 32) {
        a.cols = balanced_per_block(N, 16, cu);
        const int per = a.cols ? a.cols : 16, blocks = (N + per - 1) / per;
        if (per > 16) gemm_bf16_skinny_kernel<2, 2, 4, false, TO, false, EPI><<<blocks, 4 * 64, 0, stream>>>(a);
        else gemm_bf16_skinny_kernel<2, 1, 4, false, TO, false, EPI><<<blocks, 4 * 64, 0, stream>>>(a);
    } else {                                                // 33 to 64 rows: rows up to 48 are three tiles
        a.cols = balanced_per_block(N, 16, cu);
        const int per = a.cols ? a.cols : 16, blocks = (N + per - 1) / per;
        if (per > 16) gemm_bf16_skinny_kernel<4, 2, 8, false, TO, false, EPI><<<blocks, 8 * 64, 0, stream>>>(a);
        else if (M <= 48) gemm_bf16_skinny_kernel<3, 1, 8, false, TO, false, EPI><<<blocks, 8 * 64, 0, stream>>>(a);
        else gemm_bf16_skinny_kernel<4, 1, 8, false, TO, false, EPI><<<blocks, 8 * 64, 0, stream>>>(a);
    }
#undef LI_SK
    return li_launch_status();
}

// Few rows (M <= 64), bfloat16, K a multiple of 8.  swiglu: w has 2 N rows ([gate; up]).
extern "C" int li_linear_skinny(const void* x, const void* w, const float* bias, void* out, int M, int N,
                                int K, int out_dtype, float accumulate, int swiglu, hipStream_t stream) {
    if (M <= 0 || M > 64 || N <= 0 || K <= 0 || (K % 8)) return LI_ERR_SIZE;
    if (accumulate && out_dtype != LI_F32) return LI_ERR_DTYPE;
    if (swiglu && (bias || accumulate || out_dtype != LI_BF16)) return LI_ERR_DTYPE;
    SkinnyArgs a{(const bf16_t*)x, (const bf16_t*)w, bias, out, M, N, K, accumulate,
                 nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 0, 0, nullptr, nullptr, nullptr, nullptr, 0, 0.f};
    if (swiglu) return launch_skinny<true, bf16_t>(a, stream);
    if (out_dtype == LI_BF16) return launch_skinny<false, bf16_t>(a, stream);
    if (out_dtype == LI_F32) return launch_skinny<false, float>(a, stream);
    return LI_ERR_DTYPE;
}

// The packed projection of up to 64 rows, rotated and written into its pages (SkinnyArgs: ROPE).
static int launch_skinny_rope(SkinnyArgs a, hipStream_t stream) {
    const int M = a.M, pairs = a.N / 2, half = a.dh / 2, cu = compute_units();
    if ((unsigned long long)pairs * half >= (1ull << 32)) return LI_ERR_SIZE;
    a.half_magic = (unsigned)(((1ull << 32) + half - 1) / half);
    if (rows_kernel_takes(M, a.N, a.K) && a.K <= 2048 && pairs <= 8l * cu) {
        const int even = (pairs + cu - 1) / cu;
        a.cols = even < 3 ? 3 : even;                   // (576 pairs of 896: 3 a block 4.47 us, 4 4.66, 2 4.90)
        return launch_rows<bf16_t, true, 0>(a, pairs, stream);
    }
    a.cols = balanced_per_block(pairs, 8, cu);
    const int per = a.cols ? a.cols : 8, blocks = (pairs + per - 1) / per;
    if (M <= 16) {
        if (per > 8) gemm_bf16_skinny_kernel<1, 2, 8, false, bf16_t, true><<<blocks, 8 * 64, 0, stream>>>(a);
        else gemm_bf16_skinny_kernel<1, 1, 8, false, bf16_t, true><<<blocks, 8 * 64, 0, stream>>>(a);
    } else if (M > 32) {
        if (per > 8) gemm_bf16_skinny_kernel<4, 2, 8, false, bf16_t, true><<<blocks, 8 * 64, 0, stream>>>(a);
        else if (M <= 48) gemm_bf16_skinny_kernel<3, 1, 8, false, bf16_t, true><<<blocks, 8 * 64, 0, stream>>>(a);
        else gemm_bf16_skinny_kernel<4, 1, 8, false, bf16_t, true><<<blocks, 8 * 64, 0, stream>>>(a);
    } else {                                            // (two tiles of rows: four waves, as for the plain product)
        if (per > 8) gemm_bf16_skinny_kernel<2, 2, 4, false, bf16_t, true><<<blocks, 4 * 64, 0, stream>>>(a);
        else gemm_bf16_skinny_kernel<2, 1, 4, false, bf16_t, true><<<blocks, 4 * 64, 0, stream>>>(a);
    }
    return li_launch_status();
}

// The product before an RMS norm that is fused into its neighbours (see SkinnyArgs): out += factor * (x w^T + bias)
// in float32, xg = bf16(gamma * out), sq_parts[block * R + m] = the block's share of row m's sum of
// squares (R = 16 up to 16 rows, 32 above).  Up to 32 rows.  li_residual_norm_parts(N) is the number of
// blocks, i.e. of parts.
extern "C" int li_residual_norm_parts(int N) {
    int per = 32;                                      // as launch_skinny tiles the columns of few rows
    if (N < 8192) { per = balanced_per_block(N, 16, compute_units()); per = per ? per : 16; }
    return (N + per - 1) / per;
}
// Columns a block of the kernel of one to four rows takes on a device of cu compute units, 0 where it does not take the product
extern "C" int li_rows_kernel_cols(int M, int N, int K, int into_sum, int cu) {
    return M > 0 && N > 0 && K > 0 && cu > 0 ? rows_kernel_cols(M, N, K, into_sum != 0, cu) : 0;
}

extern "C" int li_linear_residual_norm(const void* x, const void* w, const float* bias, float* out, int M, int N,
                                       int K, float factor, const float* gamma, void* xg, float* sq_parts, hipStream_t stream) {
    if (M <= 0 || M > 32 || N <= 0 || K <= 0 || (K % 8) || factor == 0.f || !gamma || !xg || !sq_parts) return LI_ERR_SIZE;
    if (li_residual_norm_parts(N) > SK_MAX_PARTS) return LI_ERR_SIZE;
    SkinnyArgs a{(const bf16_t*)x, (const bf16_t*)w, bias, out, M, N, K, factor,
                 nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 0, 0, gamma, (bf16_t*)xg, sq_parts, nullptr, 0, 0.f};
    return launch_skinny<false, float>(a, stream);
}

// Between 13 and 64 rows (a large decoding batch) the product is still bound by streaming W, but
// x is too large to be read again by every block of a few columns (every block of the few-row
// kernel reads all of x, and what a compute unit can take in then bounds the product): tiles of
// 64 rows with the loads straight into LDS, and, where the matrix has too few such tiles to fill
// the chip, K cut into parts whose sums go to `work` and are added up in a fixed order, by kernels
// that also do what follows the product (the norm of the new residual sum, the rotary encoding
// and the page write), which the few-row kernel does in its epilogue.
// Measured on the 7B layer sizes, a decode step of 17 / 24 / 32 requests: 4.57 / 4.95 / 5.33 ms
// against 4.90 / 5.33 / 5.84 ms with the few-row kernel up to 32 rows.  Returns -1 when it does
// not take the call.
// The few-row kernel with its epilogues (a norm between two products up to 32 rows, the rotation and the page write up to 64) against those tiles.
// Up to 12 rows, one tile of rows, it is the faster one for
// every product but the largest gate/up matrices (li_linear_swiglu); at 13 to 16 rows the tiles with K in
// parts are faster where the matrix is large (at 13 rows the 7B's way back from the feed-forward, 136 MB:
// 29.8 us with its adding-up kernel against 33.5 us; its q/k/v, 33 MB: 11.8 against 9.2 us; the whole step
// of 16 requests at the 7B sizes 4.28 against 4.43 ms, at the 1.5B sizes 2.22 against 1.94 ms).
#define FEW_ROWS_FUSED 12
#define FEW_ROWS_LARGE_BYTES (100l << 20)
// 17 to 32 rows (two tiles of rows a block, the fused epilogues as with one): every block reads all of x, 32
// rows of it now, so the few-row kernel wins only against small matrices, and of those with long rows only
// against the smallest.  Alone, tiles with their adding-up kernel against the few-row kernel at 24 rows: the
// 7B's q/k/v (33 MB) 12.4 / 8.7 us and o 12.3 / 8.5; the 1.5B's q/k/v 11.6 / 6.4, o 11.8 / 6.6, gate/up (55 MB)
// 16.8 / 15.7, down (27 MB, rows of 8,960) 14.2 / 12.9; the 3B's down (45 MB, rows of 11,008) 17.6 / 19.0; the
// 14B's q/k/v (73 MB) 19.7 / 19.5 and o (52 MB, rows of 5,120) 16.9 / 17.6.
#define FEW_ROWS_TWO_TILES 32
#define FEW_ROWS_TWO_TILES_BYTES (56l << 20)
#define FEW_ROWS_TWO_TILES_LONG_K 4096
#define FEW_ROWS_TWO_TILES_LONG_K_BYTES (32l << 20)
#define SWIGLU_TILES_BYTES (160l << 20)      // (see li_linear_swiglu)
extern "C" int li_few_rows_preferred(int M, long N, long K) {
    if (M <= FEW_ROWS_FUSED || (M <= 16 && N * K * 2 < FEW_ROWS_LARGE_BYTES)) return 1;
    if (M > FEW_ROWS_TWO_TILES || K % 8) return 0;
    const long bytes = N * K * 2;
    return bytes <= FEW_ROWS_TWO_TILES_BYTES && (K <= FEW_ROWS_TWO_TILES_LONG_K || bytes <= FEW_ROWS_TWO_TILES_LONG_K_BYTES);
}

// 33 to 64 rows against a small matrix of short rows: three or four tiles of rows a block of the few-row kernel, K whole, rather than the
// 64-row tiles with K in parts, whose sums go to memory and to a kernel that adds them up.  Every block reads all of x, so the line lies at the
// length of a row.  Us, in parts / whole, with the norm behind it, and with the rotation and the page write: 48 rows of 1,536 x 1,536 10.2 / 8.8
// and 9.5 / 6.2, 64 of 2,048 x 1,536 11.1 / 9.8 and 10.4 / 8.1, 48 of 2,048 x 2,048 10.8 / 9.3 and 10.8 / 8.1; 64 of 2,048 x 2,048 with the norm
// 11.8 / 12.4, of 3,584 x 3,584 15.8 / 18.  64 of 896 x 896, too short for parts: in one and the norm's own kernel 11.6 / 7.8, and 11.0 / 6.0.
#define FOUR_TILES_K 2048         // up to 48 rows,
#define FOUR_TILES_LAST_K 1536    // above
extern "C" int li_four_tiles_preferred(int M, long N, long K) {
    return M > FEW_ROWS_TWO_TILES && M <= 64 && K % 8 == 0 && K <= (M <= 48 ? FOUR_TILES_K : FOUR_TILES_LAST_K) && N <= 16l * compute_units();
}

// Parts of K for up to 64 rows and fewer than 128 tiles of 128 columns: blocks for every compute unit, at least 8 steps a part.  (Up to MID_PARTS,
// where 8 were: 64 x 1,536 x 8,960, 12 tiles, with the norm 17.5 -> 15.2 us.  Nine to eleven are a few units more for another part's sums through
// memory: 3,584 x 18,944, 28 tiles, 33 to 64 rows with a tanh norm 30.9 us in eight, 31.7 in nine; 896 x 4,864, seven tiles, 9.8 and 9.7.)
static int mid_parts(int N, int K) {
    int nsplit = 256 / ((N + 127) / 128);
    if (nsplit > MID_PARTS) nsplit = MID_PARTS;
    if (nsplit > K / 64 / 8) nsplit = K / 64 / 8;
    return nsplit > PARTS_HELD && nsplit < 12 ? PARTS_HELD : nsplit;
}

static bool mid_rows_take(int M, int N, int K) {
    return !li_few_rows_preferred(M, N, K) && M <= 64;
}

static int linear_mid_rows(const bf16_t* x, const bf16_t* w, const float* bias, void* out, int M, int N,
                           int K, int out_dtype, float accumulate, void* work, long work_bytes,
                           hipStream_t stream) {
    if (!mid_rows_take(M, N, K) || li_four_tiles_preferred(M, N, K) || K % 64 || (out_dtype != LI_F32 && out_dtype != LI_BF16)) return -1;
#define LI_MID(BN, NS, TO, dst, b, acc, split) launch_dma<64, BN, 64, NS, false, TO>(x, w, b, (TO*)(dst), M, N, K, acc, stream, split)
    if ((N + 255) / 256 >= 128)
        return out_dtype == LI_F32 ? LI_MID(256, 3, float, out, bias, accumulate, 1) : LI_MID(256, 3, bf16_t, out, bias, accumulate, 1);
    const int tiles = (N + 127) / 128;
    if (tiles >= 128)
        return out_dtype == LI_F32 ? LI_MID(128, 4, float, out, bias, accumulate, 1) : LI_MID(128, 4, bf16_t, out, bias, accumulate, 1);
    const int nsplit = mid_parts(N, K);
    const size_t mn = (size_t)M * N;
    if (nsplit < 2 || !work || (size_t)work_bytes < (size_t)nsplit * mn * sizeof(float)) return -1;
    const int rc = LI_MID(128, 4, float, work, nullptr, 0, nsplit);
    if (rc != LI_OK) return rc;
#undef LI_MID
    const unsigned blocks = (unsigned)((mn + 255) / 256);
#define LI_RS(TO, MORE) splitk_reduce_few_kernel<TO, MORE><<<blocks, 256, 0, stream>>>((const float*)work, nsplit, mn, N, bias, (TO*)out, accumulate)
    if (out_dtype == LI_F32) { if (nsplit > PARTS_HELD) LI_RS(float, true); else LI_RS(float, false); }
    else { if (nsplit > PARTS_HELD) LI_RS(bf16_t, true); else LI_RS(bf16_t, false); }
#undef LI_RS
    return li_launch_status();
}

extern "C" long li_linear_work_bytes(int M, int N, int K, int in_dtype);

// The packed q/k/v projection of 17 rows and more where it is cut along K (up to some hundred rows): the kernel that adds the parts up also adds
// the bias, rotates query and key heads (half-split pairs over the whole head, float32 tables
// [M, dh / 2]) and writes keys and values into their page slots, so that the rotation needs no
// kernel of its own.  Thread (row, head, pair): consecutive threads read consecutive sums.
template <int HELD>
__global__ __launch_bounds__(256) void splitk_reduce_rope_store_kernel(
    const float* __restrict__ part, int nsplit, size_t mn, int N, const float* __restrict__ bias, bf16_t* __restrict__ out,
    const float* __restrict__ cosv, const float* __restrict__ sinv, const int* __restrict__ slot_map,
    bf16_t* __restrict__ kc, bf16_t* __restrict__ vc, int nh, int nkv, int dh, int page_size, int num_pages, long total) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int half = dh / 2, heads = nh + 2 * nkv;
    const int j = (int)(i % half), head = (int)((i / half) % heads), m = (int)(i / ((long)half * heads));
    const size_t i0 = (size_t)m * N + (size_t)head * dh + j, i1 = i0 + half;
    float a, b;
    if constexpr (HELD > 0) {
        Parts<(HELD > PARTS_HELD)> pa, pb;
        pa.ask(part, nsplit, mn, i0);
        pb.ask(part, nsplit, mn, i1);
        a = pa.sum(nsplit);
        b = pb.sum(nsplit);
    } else {
        a = part[i0];
        b = part[i1];
        for (int sp = 1; sp < nsplit; ++sp) { a += part[(size_t)sp * mn + i0]; b += part[(size_t)sp * mn + i1]; }
    }
    if (bias) { a += bias[head * dh + j]; b += bias[head * dh + j + half]; }
    if (head < nh + nkv) {
        const float c = cosv[(size_t)m * half + j], sn = sinv[(size_t)m * half + j];
        const float ra = __builtin_fmaf(a, c, -__fmul_rn(b, sn)), rb = __builtin_fmaf(b, c, __fmul_rn(a, sn));
        a = ra; b = rb;
    }
    const uint16_t ba = float_to_bf16(a), bb = float_to_bf16(b);
    out[i0].bits = ba;
    out[i1].bits = bb;
    if (head >= nh) {
        const int slot = slot_map[m];
        if (slot < 0 || slot >= num_pages * page_size) return;               // never write outside the pool
        const bool is_k = head < nh + nkv;
        const int kvh = is_k ? head - nh : head - nh - nkv;
        const int page = slot / page_size, in_page = slot - page * page_size;
        bf16_t* dst = (is_k ? kc : vc) + (((size_t)page * nkv + kvh) * page_size + in_page) * dh;
        dst[j].bits = ba;
        dst[j + half].bits = bb;
    }
}

// Up to 64 rows of some products take the few-row kernel with its epilogue (li_four_tiles_preferred), without parts and without `work`.
// Returns -1, having done nothing, where neither that is the case nor li_linear would cut this product along K.
extern "C" int li_linear_rope_store_parts(const void* x, const void* w, const float* bias, void* out, int M, int K,
                                          const float* cos, const float* sin, const int* slot_map, void* kc, void* vc,
                                          int nh, int nkv, int dh, int page_size, int num_pages,
                                          void* work, long work_bytes, hipStream_t stream) {
    if (M <= 0 || K <= 0 || nh <= 0 || nkv <= 0 || dh <= 0 || dh % 2 || page_size <= 0 || num_pages <= 0 ||
        (long)(nh + 2 * nkv) * dh > 0x7fffffffL)
        return LI_ERR_SIZE;
    const int N = (nh + 2 * nkv) * dh;
    if (dh % 16 == 0 && li_four_tiles_preferred(M, N, K))                // (K whole: nothing to add up)
        return launch_skinny_rope(SkinnyArgs{(const bf16_t*)x, (const bf16_t*)w, bias, out, M, N, K, 0, cos, sin, slot_map,
                                             (bf16_t*)kc, (bf16_t*)vc, nh, nkv, dh, page_size, num_pages,
                                             nullptr, nullptr, nullptr, nullptr, 0, 0.f}, stream);
    if (li_few_rows_preferred(M, N, K) || K % 64) return -1;
    const long need = li_linear_work_bytes(M, N, K, LI_BF16);            // (0 where li_linear would not cut this product)
    if (need <= 0 || !work || work_bytes < need) return -1;
    const size_t mn = (size_t)M * N;
    const int nsplit = (int)(need / (long)(mn * sizeof(float)));
    const int rc = M <= 64
        ? launch_dma<64, 128, 64, 4, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work, M, N, K, 0, stream, nsplit)
        : launch_dma<128, 128, 64, 4, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work, M, N, K, 0, stream, nsplit);
    if (rc != LI_OK) return rc;
    const long total = (long)M * (nh + 2 * nkv) * (dh / 2);
#define LI_RR(HELD) splitk_reduce_rope_store_kernel<HELD><<<(unsigned)((total + 255) / 256), 256, 0, stream>>>( \
        (const float*)work, nsplit, mn, N, bias, (bf16_t*)out, cos, sin, slot_map, (bf16_t*)kc, (bf16_t*)vc, nh, nkv, dh, page_size, num_pages, total)
    // (few rows: all parts at once, as in the other kernels that add them up; read part after part, sixteen were slower than eight had been: 33 rows of
    // 2,048 x 8,960 15.3 -> 16.5 us)
    if (nsplit > PARTS_HELD) LI_RR(MID_PARTS);
    else if (M <= 64) LI_RR(PARTS_HELD);
    else LI_RR(0);
#undef LI_RR
    return li_launch_status();
}

// Estimated time, in microseconds, of x w^T in tiles of bm x bn with K in steps of 64: rounds of tiles
// over the compute units x (steps x the longer of a step's MFMAs and a step's loads + a tile's start
// and end).  A compute unit multiplies at about 4 TFLOP/s under the chip's power limit, `speed` of
// that in this tiling (small tiles spend more of their time between steps; with four waves one
// above the other the LDS reads take nearly as long as the MFMAs), and takes in about 50 GB/s, rows
// of x that other units read too included: with few rows of x a tile waits for its part of w, and
// wide tiles read x less often.  A last round that does not fill the chip counts for less than a
// whole one: the units that run clock higher.  Chooses among the widths of the gated product's 64-row tiles alone; tiles of more
// rows go by `tiling_of`, whose steps are measured ones.
static double tile_cost(int bm, int bn, double speed, int M, int N, int K) {
    const long tiles = (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    const int cu = compute_units();
    const double filled = (double)tiles / cu, whole = (double)((tiles + cu - 1) / cu);
    const double rounds = filled + 0.4 * (whole - filled);
    const double mfma_us = (double)bm * bn * 64 * 2 / (4.0e6 * speed), load_us = (double)(bm + bn) * 128 / 50.0e3;
    return rounds * ((K / 64) * (mfma_us > load_us ? mfma_us : load_us) + 2.0);
}

// Tiles of more than 64 rows: the one with the least estimated time is taken, in microseconds: rounds of tiles over the compute
// units (a last round that does not fill the chip counts for less than a whole one: the units that run clock higher and have the memory
// to themselves) x (steps of 64 k-values x `step_us`, and the tile's start and end: `ends_us` and `byte_us` for each byte of its results
// that goes to memory or comes from there).  `pieces`: gemm_bf16_tile_kernel's, whose steps go two by two; the others are
// gemm_bf16_dma_kernel's.  Where a step has few MFMAs, whole stages and one barrier a step are the faster form (128 x 128 x 3,584: 60 us
// against 64 for 2,048 x 3,584 results; 128 x 192 of 4 waves one above the other 12 % before the same tile in pieces, gated, on average), and
// so they are where K is a few steps (3,330 rows against 12,288 gated columns of 64: 26 us against 43); with more MFMAs and
// steps the stage handed back in pieces (256 x 256, 8,192^3: 827 -> 726 us; 2,048 x 37,888 x 3,584 gated 483 -> 406).
// All tiles up to 128 x 288 and 192 x 192 that were timed take in 55 GB/s a compute unit whatever they multiply (what 256 lines of a unit's
// cache, all on their way, bring at the latency of the lines that come from beyond the L2: the loads straight into LDS alone take 130 GB/s
// where all of it lies there); the larger ones are bound by the MFMAs at the chip's power limit.
// The numbers are fitted to 804 products and 880 gated ones, 65 to 6,000 rows x 512 to 28,000 columns x 64 to 19,200, half of them layers'
// matrices, each timed in every tile: what is taken is within 0.4 % of the best tile on average, and 1 % of them are more than 3 % behind
// the best that any rule took before (at worst 20 %: 162 x 14,752 x 3,392, 2,501 x 2,176 x 384 gated).
struct Tiling { int bm, bn; bool pieces; double step_us, ends_us; };
struct Fit { double byte_us, rest; };        // rest: what a last round's idle units count for
static double tile_us(const Tiling& t, const Fit& f, int bytes, int M, int N, int K) {
    const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const int cu = compute_units();
    const double filled = (double)tiles / cu, whole = (double)((tiles + cu - 1) / cu);
    const int steps = t.pieces ? (K / 64 + 1) / 2 * 2 : K / 64;
    return (filled + f.rest * (whole - filled)) * (steps * t.step_us + t.ends_us + (double)t.bm * t.bn * f.byte_us * bytes);
}
template <int COUNT>
static int least_us(const Tiling (&shape)[COUNT], const Fit& f, int bytes, int M, int N, int K) {
    int pick = 0;
    double best = 0.0;
    for (int i = 0; i < COUNT; ++i) {
        const double c = tile_us(shape[i], f, bytes, M, N, K);
        if (i == 0 || c < best) { best = c; pick = i; }
    }
    return pick;
}
static const Tiling plain_tiles[9] = {{128, 128, false, 0.523, 1.48}, {192, 128, false, 0.630, 2.22}, {256, 128, false, 0.787, 2.61},
                                      {128, 224, false, 0.801, 2.45}, {256, 256, false, 1.434, 3.58}, {192, 224, true, 0.993, 3.47},
                                      {192, 256, true, 1.106, 3.40}, {256, 224, true, 1.223, 5.43}, {256, 256, true, 1.393, 4.33}};
static int tiling_of(int M, int N, int K, int bytes) { return least_us(plain_tiles, Fit{2.884e-5, 0.617}, bytes, M, N, K); }
// (a tile's columns are gate and up columns in turn.  Wide ones of 128 rows for steps of a few hundred rows or a few more than a multiple
// of 256: 1,027 rows against the 1.5B's 17,920 columns are 504 tiles of 128 x 320, two rounds: 69 -> 58 us)
static const Tiling gated_tiles[10] = {{128, 128, false, 0.584, 1.98}, {128, 256, false, 0.869, 2.32}, {128, 192, false, 0.648, 2.62},
                                       {256, 128, false, 0.832, 3.80}, {256, 256, false, 1.478, 3.70}, {128, 320, true, 0.988, 3.12},
                                       {192, 256, true, 1.096, 3.10}, {192, 320, true, 1.289, 4.67}, {256, 192, true, 1.075, 3.82},
                                       {256, 256, true, 1.377, 4.09}};
static int gated_tiling_of(int M, int N, int K) { return least_us(gated_tiles, Fit{2.051e-5, 0.748}, 1, M, N, K); }

// The tile of a product of more than 64 rows, K a multiple of 64, that is not cut along K: rows x 65,536 + columns, negative in pieces.
// `bytes` of a result that move (float32 8 where it is added to, else 4; bfloat16 2); gated: N is both halves' columns, bytes does not matter.
extern "C" int li_linear_tile(int gated, int M, int N, int K, int bytes) {
    const Tiling& t = gated ? gated_tiles[gated_tiling_of(M, N, K)] : plain_tiles[tiling_of(M, N, K, bytes)];
    return (t.pieces ? -1 : 1) * (t.bm * 65536 + t.bn);
}

// More than 64 rows but so few 128 x 128 tiles that half of the compute units would idle (a narrow
// matrix with a long K, like the feed-forward's way back at 128 to 512 rows): K is cut into parts
// here too.  Returns the number of parts, 1 for none.
static int split_parts_many_rows(int M, int N, int K) {
    if (M <= 64 || K % 64) return 1;
    const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
    if (tiles >= 128) return 1;
    int nsplit = (int)(256 / tiles);
    if (nsplit > PARTS_HELD) nsplit = PARTS_HELD;
    if (nsplit > K / 64 / 8) nsplit = K / 64 / 8;              // at least 8 steps a part
    return nsplit < 2 ? 1 : nsplit;
}

static void launch_f32_mfma(const float* x, const float* w, const float* bias, float* out, int M, int N, int K,
                            float accumulate, int parts, hipStream_t stream) {
    const int steps = (K + F32M_BK - 1) / F32M_BK;
    const dim3 tiles((N + F32M_BN - 1) / F32M_BN, (M + F32M_BM - 1) / F32M_BM, parts);
    gemm_f32_mfma_kernel<<<tiles, 256, 0, stream>>>(x, w, bias, out, M, N, K, accumulate, (steps + parts - 1) / parts);
}

// Into how many parts K is cut for the float32 tiles of 128 x 128 (more than 64 rows): a narrow matrix has fewer tiles
// than the chip has compute units (810 rows against 1,536 columns: 84), and a tile's time is the length of K whatever the
// others do.  The least estimated time, in microseconds: a step of 16 k-values counts as 1.2 us of a unit (1.06 measured
// where blocks do not share units, up to 1.25 where they do), a block 6 for its start and end, and the parts' sums are
// written and read again at 5 TB/s by a kernel of its own (4 us).  Measured, one part against the parts taken here: 65 to
// 128 rows x 1,536 x 8,960 597 -> 54 us (16 parts), 300 rows 597 -> 100 (6), 810 rows 598 -> 206 (6), x 1,536 x 1,536
// 125 -> 51, 810 x 2,048 x 1,536 122 -> 67 (2), 1,024 x 3,584 x 18,944 1,276 -> 1,074 (8), 2,048 x 3,584 x 3,584
// 463 -> 430 (4); from some thousand tiles on (810 x 17,920: 980) parts cost what they give, and K stays whole.  The rule
// is within 7 % of the best number of parts measured at 65 to 2,048 rows against seven matrices.  At most 256 MB of parts.
#define F32_MAX_PARTS 16
#define F32_PARTS_MAX_BYTES (256l << 20)
#define F32_PART_MIN_STEPS 6
static int f32_split_parts(int M, int N, int K) {
    if (M <= F32_ROWS_MAX || K % 4) return 1;
    const long tiles = (long)((M + F32M_BM - 1) / F32M_BM) * ((N + F32M_BN - 1) / F32M_BN);
    const int steps = (K + F32M_BK - 1) / F32M_BK, cu = compute_units();
    int pick = 1;
    double best = 0.0;
    for (int p = 1; p <= F32_MAX_PARTS && p * F32_PART_MIN_STEPS <= steps; ++p) {
        const int per = (steps + p - 1) / p;
        if ((long)per * (p - 1) >= steps) continue;                      // (a part would be empty)
        if (p > 1 && (long)p * M * N * (long)sizeof(float) > F32_PARTS_MAX_BYTES) break;
        const long rounds = (tiles * p + cu - 1) / cu;
        double us = rounds * (per * 1.2 * (rounds > 1 ? 0.95 : 1.0)) + 6.0;
        if (p > 1) us += 4.0 + (p + 2) * 4.0 * M * N / 5.0e6;
        if (p == 1 || us < best) { best = us; pick = p; }
    }
    return pick;
}

// Bytes of workspace with which this product is cut along K (0: it is not).  The products of li_four_tiles_preferred have a number too: li_linear
// and what it shares their epilogues with leave K whole there and need none of it, but a tanh norm into float32 and a rotation of heads that are no
// multiple of 16 columns cut them.
extern "C" long li_linear_work_bytes(int M, int N, int K, int in_dtype) {
    if (in_dtype == LI_F32) {
        const int parts = N > 0 && K > 0 ? f32_split_parts(M, N, K) : 1;
        return parts < 2 ? 0 : (long)parts * M * N * (long)sizeof(float);
    }
    if (in_dtype != LI_BF16 || N <= 0 || K <= 0 || K % 64 || li_few_rows_preferred(M, N, K)) return 0;
    int nsplit = 1;
    if (M <= 64) {
        const int tiles = (N + 127) / 128;
        if (tiles < 128) nsplit = mid_parts(N, K);
    } else {
        nsplit = split_parts_many_rows(M, N, K);
    }
    return nsplit < 2 ? 0 : (long)nsplit * M * N * (long)sizeof(float);
}

// out += factor * (x w^T + bias) (float32 out: the residual sum) and xn = the RMS norm of the new out with weights
// gamma, where li_linear would cut K into parts anyway: the kernel that adds the parts up then has
// whole rows in its hands.  Also for the products of li_four_tiles_preferred: K whole, then the norm's kernel, which reads the sum again; no
// `work`.  xn is bfloat16 (xn_dtype LI_BF16) or float32.  Returns -1, having done
// nothing, where neither is the case (the caller then multiplies and norms in two calls).
extern "C" int li_linear_then_norm(const void* x, const void* w, const float* bias, float* out, int M, int N, int K,
                                   void* work, long work_bytes, float factor, const float* gamma, float eps, void* xn,
                                   int xn_dtype, hipStream_t stream) {
    if (N <= 0 || K <= 0 || (K % 64) || li_few_rows_preferred(M, N, K) || !gamma || !xn || eps < 0.f) return -1;
    if (N > REDUCE_NORM_NT * REDUCE_NORM_PER || (xn_dtype != LI_BF16 && xn_dtype != LI_F32)) return -1;
    const size_t mn = (size_t)M * N;
    if (factor != 0.f && li_four_tiles_preferred(M, N, K)) {      // K whole: the sum, then its norm (0 is that kernel's word for writing, not adding)
        const int rc = li_linear_skinny(x, w, bias, out, M, N, K, LI_F32, factor, 0, stream);
        if (rc != LI_OK) return rc;
        if (xn_dtype == LI_BF16)
            splitk_reduce_norm_kernel<bf16_t, REDUCE_NORM_NT, REDUCE_NORM_PER, true, false, true><<<M, REDUCE_NORM_NT, 0, stream>>>(
                nullptr, 0, mn, N, nullptr, out, 0.f, gamma, eps, (bf16_t*)xn);
        else
            splitk_reduce_norm_kernel<float, REDUCE_NORM_NT, REDUCE_NORM_PER, true, false, true><<<M, REDUCE_NORM_NT, 0, stream>>>(
                nullptr, 0, mn, N, nullptr, out, 0.f, gamma, eps, (float*)xn);
        return li_launch_status();
    }
    const long need = li_linear_work_bytes(M, N, K, LI_BF16);
    if (need <= 0 || !work || work_bytes < need) return -1;
    const int nsplit = (int)(need / (long)(mn * sizeof(float)));
    if (nsplit > MID_PARTS) return -1;
    const int rc = M <= 64
        ? launch_dma<64, 128, 64, 4, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work, M, N, K, 0, stream, nsplit)
        : launch_dma<128, 128, 64, 4, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work, M, N, K, 0, stream, nsplit);
    if (rc != LI_OK) return rc;
    const uintptr_t places = (uintptr_t)work | (uintptr_t)bias | (uintptr_t)out | (uintptr_t)gamma | (uintptr_t)xn;
    if (reduce_by_rows(M, N, nsplit) && xn_dtype == LI_BF16 && N % 4 == 0 && places % 16 == 0) {
        (nsplit <= 2 ? launch_reduce_norm_rows<2> : nsplit <= 4 ? launch_reduce_norm_rows<4> : launch_reduce_norm_rows<PARTS_HELD>)(
            (const float*)work, nsplit, M, N, bias, out, factor, gamma, eps, (bf16_t*)xn, stream);
        return li_launch_status();
    }
#define LI_RN(TN, FEW, MORE) splitk_reduce_norm_kernel<TN, REDUCE_NORM_NT, REDUCE_NORM_PER, FEW, MORE><<<M, REDUCE_NORM_NT, 0, stream>>>( \
        (const float*)work, nsplit, mn, N, bias, out, factor, gamma, eps, (TN*)xn)
    if (xn_dtype == LI_BF16) { if (nsplit > PARTS_HELD) LI_RN(bf16_t, true, true); else if (M <= 64) LI_RN(bf16_t, true, false); else LI_RN(bf16_t, false, false); }
    else { if (nsplit > PARTS_HELD) LI_RN(float, true, true); else if (M <= 64) LI_RN(float, true, false); else LI_RN(float, false, false); }
#undef LI_RN
    return li_launch_status();
}

// out += factor * (x w^T + bias) (float32: the residual sum) and xn = tanh(alpha * out) * gamma + beta in one go: in the
// epilogue of the few-row kernel (up to 32 rows, or 64 against a small matrix; bfloat16 xn), or, where li_linear would cut K into parts, in the kernel
// that adds the parts up.  Returns -1, having done nothing, where neither is the case.
extern "C" int li_linear_tanh_norm(const void* x, const void* w, const float* bias, float* out, int M, int N, int K,
                                   void* work, long work_bytes, float factor, float alpha, const float* gamma,
                                   const float* beta, void* xn, int xn_dtype, hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 8 || factor == 0.f || !gamma || !beta || !xn || (xn_dtype != LI_BF16 && xn_dtype != LI_F32)) return -1;
    if ((M <= 32 && li_few_rows_preferred(M, N, K)) || (xn_dtype == LI_BF16 && li_four_tiles_preferred(M, N, K))) {
        if (xn_dtype != LI_BF16) return -1;
        SkinnyArgs a{(const bf16_t*)x, (const bf16_t*)w, bias, out, M, N, K, factor,
                     nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 0, 0, gamma, (bf16_t*)xn, nullptr, nullptr, 0, 0.f};
        a.beta = beta;
        a.alpha = alpha;
        return launch_skinny<false, float, 1>(a, stream);
    }
    const long need = li_linear_work_bytes(M, N, K, LI_BF16);
    if (need <= 0 || !work || work_bytes < need) return -1;
    const size_t mn = (size_t)M * N;
    const int nsplit = (int)(need / (long)(mn * sizeof(float)));
    if (nsplit > MID_PARTS) return -1;
    const int rc = M <= 64
        ? launch_dma<64, 128, 64, 4, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work, M, N, K, 0.f, stream, nsplit)
        : launch_dma<128, 128, 64, 4, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work, M, N, K, 0.f, stream, nsplit);
    if (rc != LI_OK) return rc;
    const unsigned blocks = (unsigned)((mn + 255) / 256);
#define LI_RT(TN, MORE) splitk_reduce_tanh_kernel<TN, MORE><<<blocks, 256, 0, stream>>>((const float*)work, nsplit, mn, N, bias, out, factor, alpha, gamma, beta, (TN*)xn)
    if (xn_dtype == LI_BF16) { if (nsplit > PARTS_HELD) LI_RT(bf16_t, true); else LI_RT(bf16_t, false); }
    else { if (nsplit > PARTS_HELD) LI_RT(float, true); else LI_RT(float, false); }
#undef LI_RT
    return li_launch_status();
}

// `work` (may be null): device memory of work_bytes for the partial sums of a product cut along K.
// Rows of the smallest tile that a product of more than 64 rows is cut into in this dtype: a
// product of a few rows more than a multiple of it pays for a whole tile more.  Whoever cuts work
// into steps (a scheduler) asks here instead of knowing the kernels' tilings.
extern "C" int li_linear_row_tile(int in_dtype) { return in_dtype == LI_F32 ? F32_BM : BF_BM; }

extern "C" int li_linear(const void* x, const void* w, const float* bias, void* out, int M, int N,
                         int K, int in_dtype, int out_dtype, float accumulate, void* work, long work_bytes,
                         hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0) return LI_ERR_SIZE;
    if (accumulate && out_dtype != LI_F32) return LI_ERR_DTYPE;
    if (in_dtype == LI_F32) {
        if (out_dtype != LI_F32) return LI_ERR_DTYPE;
        if (M <= F32_ROWS_MAX && K % 4 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0)
            return launch_f32_rows((const float*)x, (const float*)w, bias, (float*)out, M, N, K, accumulate, stream);
        if (K % 4 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0) {       // the matrix cores' float32 form
            if ((M + F32M_BM - 1) / F32M_BM > 65535) return LI_ERR_SIZE;
            const int parts = f32_split_parts(M, N, K);
            const size_t mn = (size_t)M * N;
            if (parts > 1 && work && (size_t)work_bytes >= (size_t)parts * mn * sizeof(float)) {
                launch_f32_mfma((const float*)x, (const float*)w, nullptr, (float*)work, M, N, K, 0.f, parts, stream);
                const unsigned blocks = (unsigned)((mn + 255) / 256);
                splitk_reduce_kernel<float><<<blocks, 256, 0, stream>>>((const float*)work, parts, mn, N, bias, (float*)out, accumulate);
            } else {
                launch_f32_mfma((const float*)x, (const float*)w, bias, (float*)out, M, N, K, accumulate, 1, stream);
            }
            return li_launch_status();
        }
        if (M >= 2 * F32B_BM && N >= F32B_BN) {              // enough of both for the large tile to fill the chip
            dim3 big((N + F32B_BN - 1) / F32B_BN, (M + F32B_BM - 1) / F32B_BM);
            if (big.y > 65535) return LI_ERR_SIZE;
            gemm_f32_big_kernel<<<big, 256, 0, stream>>>((const float*)x, (const float*)w, bias, (float*)out, M, N, K, accumulate);
            return li_launch_status();
        }
        dim3 grid((N + F32_BN - 1) / F32_BN, (M + F32_BM - 1) / F32_BM);
        if (grid.y > 65535) return LI_ERR_SIZE;
        gemm_f32_kernel<<<grid, 256, 0, stream>>>((const float*)x, (const float*)w, bias, (float*)out, M, N, K, accumulate);
    } else if (in_dtype == LI_BF16) {
        dim3 grid((N + BF_BN - 1) / BF_BN, (M + BF_BM - 1) / BF_BM);
        if (grid.y > 65535) return LI_ERR_SIZE;
        const bool aligned = (K % 8) == 0;
        if (aligned && M <= 64) {
            const int rc = linear_mid_rows((const bf16_t*)x, (const bf16_t*)w, bias, out, M, N, K, out_dtype,
                                           accumulate, work, work_bytes, stream);
            if (rc >= 0) return rc;
            return li_linear_skinny(x, w, bias, out, M, N, K, out_dtype, accumulate, 0, stream);
        }
        if (aligned && M > 64) {
#define LI_BIG(BM, BN, BK) (out_dtype == LI_F32 ? launch_big<BM, BN, BK, float>((const bf16_t*)x, (const bf16_t*)w, bias, (float*)out, M, N, K, accumulate, stream) \
                                            : launch_big<BM, BN, BK, bf16_t>((const bf16_t*)x, (const bf16_t*)w, bias, (bf16_t*)out, M, N, K, accumulate, stream))
            if (out_dtype != LI_F32 && out_dtype != LI_BF16) return LI_ERR_DTYPE;
#define LI_DMA(BM, BN, BK, NS) (out_dtype == LI_F32 ? launch_dma<BM, BN, BK, NS, false, float>((const bf16_t*)x, (const bf16_t*)w, bias, (float*)out, M, N, K, accumulate, stream) \
                                               : launch_dma<BM, BN, BK, NS, false, bf16_t>((const bf16_t*)x, (const bf16_t*)w, bias, (bf16_t*)out, M, N, K, accumulate, stream))
            if (K % 64 == 0) {
                const int nsplit = split_parts_many_rows(M, N, K);
                const size_t mn = (size_t)M * N;
                if (nsplit > 1 && work && (size_t)work_bytes >= (size_t)nsplit * mn * sizeof(float)) {
                    const int rc = launch_dma<128, 128, 64, 4, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work,
                                                                              M, N, K, 0, stream, nsplit);
                    if (rc != LI_OK) return rc;
                    const unsigned blocks = (unsigned)((mn + 255) / 256);
                    if (out_dtype == LI_F32) splitk_reduce_kernel<float><<<blocks, 256, 0, stream>>>((const float*)work, nsplit, mn, N, bias, (float*)out, accumulate);
                    else splitk_reduce_kernel<bf16_t><<<blocks, 256, 0, stream>>>((const float*)work, nsplit, mn, N, bias, (bf16_t*)out, accumulate);
                    return li_launch_status();
                }
#define LI_TILE(BM, BN, NS) (out_dtype == LI_F32 ? launch_tile<BM, BN, NS, false, float>((const bf16_t*)x, (const bf16_t*)w, bias, (float*)out, M, N, K, accumulate, stream) \
                                        : launch_tile<BM, BN, NS, false, bf16_t>((const bf16_t*)x, (const bf16_t*)w, bias, (bf16_t*)out, M, N, K, accumulate, stream))
#define LI_DMA4(BM, BN, NS) (out_dtype == LI_F32 ? launch_dma<BM, BN, 64, NS, false, float, 0, 4>((const bf16_t*)x, (const bf16_t*)w, bias, (float*)out, M, N, K, accumulate, stream) \
                                        : launch_dma<BM, BN, 64, NS, false, bf16_t, 0, 4>((const bf16_t*)x, (const bf16_t*)w, bias, (bf16_t*)out, M, N, K, accumulate, stream))
                switch (tiling_of(M, N, K, out_dtype == LI_BF16 ? 2 : accumulate != 0.f ? 8 : 4)) {
                case 0: return LI_DMA(128, 128, 64, 4);
                case 1: return LI_DMA(192, 128, 64, 3);
                case 2: return LI_DMA(256, 128, 64, 3);
                case 3: return LI_DMA4(128, 224, 3);
                case 4: return LI_DMA(256, 256, 64, 2);
                case 5: return LI_TILE(192, 224, 2);
                case 6: return LI_TILE(192, 256, 2);
                case 7: return LI_TILE(256, 224, 2);
                default: return LI_TILE(256, 256, 2);
                }
#undef LI_DMA4
#undef LI_TILE
            }
#undef LI_DMA
            return LI_BIG(128, 128, 64);             // K not a multiple of 64: loads staged in registers
#undef LI_BIG
        }
#define LI_GEMM(TO, AL) gemm_bf16_kernel<TO, AL><<<grid, 256, 0, stream>>>((const bf16_t*)x, (const bf16_t*)w, bias, (TO*)out, M, N, K, accumulate)
        if (out_dtype == LI_F32) { if (aligned) LI_GEMM(float, true); else LI_GEMM(float, false); }
        else if (out_dtype == LI_BF16) { if (aligned) LI_GEMM(bf16_t, true); else LI_GEMM(bf16_t, false); }
        else return LI_ERR_DTYPE;
#undef LI_GEMM
    } else return LI_ERR_DTYPE;
    return li_launch_status();
}

// Bytes of workspace that li_linear_act needs (0: none).
extern "C" long li_linear_act_work_bytes(int M, int N, int K, int act) {
    const long parts = li_linear_work_bytes(M, N, K, LI_BF16);
    if (parts > 0 || act == LI_ACT_RELU2 || M <= 0 || N <= 0 || K <= 0 || K % 64 || !mid_rows_take(M, N, K) || (N + 127) / 128 < 128) return parts;
    return (long)M * N * (long)sizeof(float);
}

// out = act(x w^T + bias), bfloat16 throughout, the sums float32 until the activation has been taken: in the epilogue of
// the kernel that li_linear would take for these sizes, or of the one that adds its parts up.  Without it the sums go to
// memory in float32 and a kernel of their own reads them again: at a few rows that kernel costs its launch, some 2 us a layer in
// a recorded step (8 x 8,960 x 1,536 12.7 -> 10.7 us, 64 rows, K in parts, 17.0 -> 14.3), and at 2,048 rows of 8,960 columns the
// reads and writes of 73 MB (squared ReLU 93 -> 70 us, of 18,944 x 3,584 327 -> 263; 300 rows of 8,960 23.9 -> 17.7).  Tiles
// whose K is not in parts take the squared ReLU only, in instances of their own: the others are tens of instructions a value, which
// a tile's four waves take one after the other when the matrix cores are done (xIELU, 2,601 rows of 8,960 columns: product and
// kernel 96 + 24 us, in the epilogue 183; GELU, 17 to 48 rows of 18,944 x 3,584 31.7 to 35.9 -> 33.1 to 36.8), and with the
// code of all four in one kernel the squared ReLU pays too (2,048 rows of 8,960 103 us, 1,000 rows of 18,944 182 -> 223).
// Up to 64 rows the others' sums go to the lent memory (li_linear_act_work_bytes) and on to act_of_sums_kernel
// (17 / 48 rows 32.4 / 36.4); above, the caller does the same.
// Returns -1, having done nothing, where it does not take the call.
extern "C" int li_linear_act(const void* x, const void* w, const float* bias, void* out, int M, int N, int K, int act, float a0,
                             float a1, void* work, long work_bytes, hipStream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0 || act < LI_ACT_RELU2 || act > LI_ACT_XIELU) return LI_ERR_SIZE;
    if (K % 8 || (M > 64 && (K % 64 || act != LI_ACT_RELU2))) return -1;
    const LiAct ep{act, a0, a1};
    if (M <= 64 && (K % 64 || !mid_rows_take(M, N, K) || li_four_tiles_preferred(M, N, K))) {
        SkinnyArgs a{(const bf16_t*)x, (const bf16_t*)w, bias, out, M, N, K, 0.f,
                     nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 0, 0, nullptr, nullptr, nullptr, nullptr, 0, 0.f};
        a.ep = ep;
        return launch_skinny<false, bf16_t, 2>(a, stream);
    }
    const long need = li_linear_act_work_bytes(M, N, K, act);
    if (need > 0) {                                  // K in parts, or in one
        const size_t mn = (size_t)M * N;
        const int nsplit = (int)(need / (long)(mn * sizeof(float)));
        if (!work || (uintptr_t)work % 16 || work_bytes < need || nsplit > MID_PARTS) return -1;
        const int rc = M <= 64 && nsplit == 1 && (N + 255) / 256 >= 128
            ? launch_dma<64, 256, 64, 3, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work, M, N, K, 0.f, stream)
            : M <= 64
            ? launch_dma<64, 128, 64, 4, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work, M, N, K, 0.f, stream, nsplit)
            : launch_dma<128, 128, 64, 4, false, float>((const bf16_t*)x, (const bf16_t*)w, nullptr, (float*)work, M, N, K, 0.f, stream, nsplit);
        if (rc != LI_OK) return rc;
        if (nsplit == 1) act_of_sums_kernel<<<(unsigned)((mn + 1023) / 1024), 256, 0, stream>>>((const float*)work, mn, N, bias, (bf16_t*)out, ep);
        else if (nsplit > PARTS_HELD) splitk_reduce_act_kernel<true><<<(unsigned)((mn + 255) / 256), 256, 0, stream>>>((const float*)work, nsplit, mn, N, bias, (bf16_t*)out, ep);
        else splitk_reduce_act_kernel<false><<<(unsigned)((mn + 255) / 256), 256, 0, stream>>>((const float*)work, nsplit, mn, N, bias, (bf16_t*)out, ep);
        return li_launch_status();
    }
#define LI_ACT(BM, BN, NS) launch_dma<BM, BN, 64, NS, false, bf16_t, LI_ACT_RELU2>((const bf16_t*)x, (const bf16_t*)w, bias, (bf16_t*)out, M, N, K, 0.f, stream, 1, nullptr, 0, 0.f, ep)
#define LI_ACT4(BM, BN, NS) launch_dma<BM, BN, 64, NS, false, bf16_t, LI_ACT_RELU2, 4>((const bf16_t*)x, (const bf16_t*)w, bias, (bf16_t*)out, M, N, K, 0.f, stream, 1, nullptr, 0, 0.f, ep)
#define LI_ACT_TILE(BM, BN, NS) launch_tile<BM, BN, NS, false, bf16_t, LI_ACT_RELU2>((const bf16_t*)x, (const bf16_t*)w, bias, (bf16_t*)out, M, N, K, 0.f, stream, ep)
    if (M <= 64) {                                   // (as linear_mid_rows takes them)
        if ((N + 255) / 256 >= 128) return LI_ACT(64, 256, 3);
        if ((N + 127) / 128 >= 128) return LI_ACT(64, 128, 4);
        return -1;
    }
    switch (tiling_of(M, N, K, 2)) {
    case 0: return LI_ACT(128, 128, 4);
    case 1: return LI_ACT(192, 128, 3);
    case 2: return LI_ACT(256, 128, 3);
    case 3: return LI_ACT4(128, 224, 3);
    case 4: return LI_ACT(256, 256, 2);
    case 5: return LI_ACT_TILE(192, 224, 2);
    case 6: return LI_ACT_TILE(192, 256, 2);
    case 7: return LI_ACT_TILE(256, 224, 2);
    default: return LI_ACT_TILE(256, 256, 2);
    }
#undef LI_ACT_TILE
#undef LI_ACT4
#undef LI_ACT
}

// The gated forms: 0 the plain one, LI_ACT_GELU_TANH, LI_ACT_CLAMPED with a positive limit.
static bool gated_form_known(int act, float limit) { return act == 0 || act == LI_ACT_GELU_TANH || (act == LI_ACT_CLAMPED && limit > 0.f); }

// The gated product below in float32 for up to 64 rows (K a multiple of 4): the few-row product on the float32 matrix cores with
// the activation in its epilogue.
extern "C" int li_linear_swiglu_f32(const float* x, const float* w, float* out, int M, int I, int K, int act, float limit, hipStream_t stream) {
    if (!gated_form_known(act, limit)) return LI_ERR_SIZE;
    if (M <= 0 || M > F32_ROWS_MAX || I <= 0 || K <= 0 || K % 4 || I > 0x3fffffff) return LI_ERR_SIZE;
    if ((((uintptr_t)x | (uintptr_t)w) & 15) != 0) return LI_ERR_SIZE;
    return launch_f32_rows(x, w, nullptr, out, M, I, K, 0.f, stream, true, LiAct{act, limit, 0.f});
}

// out[m, n] = up * gate / (1 + exp(-gate)) with [gate, up] = x w^T, w = [gate; up] of I rows each:
// the activation as the product's epilogue, so the 2 I columns never go to memory.  bfloat16;
// K a multiple of 8 for up to 64 rows, a multiple of 64 above.  act, limit: which form (see gated_form_known and gated_bf16).
// row_parts (may be null): x is the xg of li_linear_residual_norm and these are its sq_parts, nparts of
// them; every row's result is that of the RMS norm with eps (up to 32 rows).
extern "C" int li_linear_swiglu(const void* x, const void* w, void* out, int M, int I, int K,
                                const float* row_parts, int nparts, float eps, int act, float limit, hipStream_t stream) {
    if (!gated_form_known(act, limit)) return LI_ERR_SIZE;
    const LiAct ep{act, limit, 0.f};
    if (M <= 0 || I <= 0 || K <= 0 || I > 0x3fffffff) return LI_ERR_SIZE;
    const int N = 2 * I;
    if (row_parts && (M > 32 || (K % 8) || nparts <= 0 || nparts > SK_MAX_PARTS || eps < 0.f)) return LI_ERR_SIZE;
    // Up to 64 rows the product waits for w.  From 17 rows on (more than the few-row kernel's fused form takes),
    // and from 13 on where the matrix is large (li_few_rows_preferred: the 7B's at 16 rows 51.8 against 59.6 us),
    // it goes to tiles of 64 rows if the matrix has tiles enough to fill the chip: the width with the least
    // estimated time (a compute unit takes in only so much: more units, each with a narrower tile, stream
    // more, until the tiles no longer fit one round).
    // Below that the few-row kernel, but for a large matrix of rows that are not too long whose tiles fit ONE
    // round over the compute units: there the tiles' loads straight into LDS stream w at the rate of a kernel
    // that only reads (7B sizes, 272 MB: 48.8 us; the few-row kernel 49 to 54 us at 1 to 12 rows), and the
    // rows' factors of a fused RMS norm are applied in the tile kernel's epilogue.  Measured on one machine in
    // turn, whole decode steps: 7B sizes 3.34 -> 3.32 ms at 1 request, 3.72 -> 3.62 at 8, 4.06 -> 3.90 at 12;
    // 14B 6.5 -> 6.57 / 7.66 -> 7.45 / 8.49 -> 8.09; 32B (566 MB) 13.98 -> 13.05 at 1.  Not taken where it
    // loses: small matrices (3B's 90 MB, 1.5B's 55 MB: steps 4-5 % longer), rows of 8,192 (72B sizes 173
    // against 181 us; 28,672 x 8,192: 86 against 96), or no width whose tiles fit one round (73,728 x 4,096:
    // 109 against 130 us).
    const int cu = compute_units();
    const bool few = li_few_rows_preferred(M, N, K);
    // (since the few-row kernel's waves have their next chunk in flight while they multiply, it is the faster one
    // again where the rows are few: every one of its blocks reads all of x, the tiles read x once a tile.  7B sizes
    // at 1 / 8 / 12 / 16 rows: 46.4 / 47.6 / 49.5 / 52.0 us against the tiles' 49.0 / 48.6 / 49.5 / 50.2; 14B sizes
    // at 4 / 8: 48.8 / 50.9 against 50.4 / 50.1; 32B sizes at 1 / 4: 97.4 / 100.3 against 97.4 / 97.2: the tiles
    // from rows x matrix bytes of 2.2 GB on)
    const bool stream_tiles = (long)N * K * 2 >= SWIGLU_TILES_BYTES && K <= 6144 && (double)M * N * K * 2 > 2.2e9;
    if (M <= 64 && K % 64 == 0 && (!few || stream_tiles)) {
        const int widths[3] = {256, 192, 128};
        int pick = -1;
        double best = 0.0;
        for (int i = 0; i < 3; ++i) {
            const int tiles = (N + widths[i] - 1) / widths[i];
            if (tiles < 128) continue;                                   // too few tiles: the few-row kernel
            if (few && tiles > cu) continue;                             // (few rows: one round only, see above)
            const double c = tile_cost(64, widths[i], 1.0, M, N, K);
            if (pick < 0 || c < best) { best = c; pick = i; }
        }
#define LI_SW64_AS(BN, NS, ACT) launch_dma<64, BN, 64, NS, true, bf16_t, ACT>((const bf16_t*)x, (const bf16_t*)w, nullptr, (bf16_t*)out, M, N, K, 0.f, stream, 1, row_parts, nparts, eps, ep)
#define LI_SW64(BN, NS) (act == LI_ACT_CLAMPED ? LI_SW64_AS(BN, NS, LI_ACT_CLAMPED) : act ? LI_SW64_AS(BN, NS, LI_ACT_GELU_TANH) : LI_SW64_AS(BN, NS, 0))
        if (pick == 0) return LI_SW64(256, 3);
        if (pick == 1) return LI_SW64(192, 4);
        if (pick == 2) return LI_SW64(128, 4);
#undef LI_SW64
#undef LI_SW64_AS
    }
    if (row_parts || (M <= 64 && act)) {
        if (K % 8) return LI_ERR_SIZE;
        SkinnyArgs a{(const bf16_t*)x, (const bf16_t*)w, nullptr, out, M, I, K, 0.f,
                     nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 0, 0, nullptr, nullptr, nullptr, row_parts, nparts, eps};
        a.ep = ep;
        return act ? launch_skinny<true, bf16_t, 1>(a, stream) : launch_skinny<true, bf16_t>(a, stream);
    }
    if (M <= 64) return li_linear_skinny(x, w, nullptr, out, M, I, K, LI_BF16, 0, 1, stream);
    if (K % 64) return LI_ERR_SIZE;
#define LI_GATED(LAUNCH, ...) LAUNCH((const bf16_t*)x, (const bf16_t*)w, nullptr, (bf16_t*)out, M, N, K, 0.f, stream, __VA_ARGS__)
#define LI_DMA_AS(BM, BN, NS, WLM, ACT) LI_GATED((launch_dma<BM, BN, 64, NS, true, bf16_t, ACT, WLM>), 1, nullptr, 0, 0.f, ep)
#define LI_DMA(BM, BN, NS, WLM) (act == LI_ACT_CLAMPED ? LI_DMA_AS(BM, BN, NS, WLM, LI_ACT_CLAMPED) : act ? LI_DMA_AS(BM, BN, NS, WLM, LI_ACT_GELU_TANH) : LI_DMA_AS(BM, BN, NS, WLM, 0))
#define LI_TILE_AS(BM, BN, NS, ACT) LI_GATED((launch_tile<BM, BN, NS, true, bf16_t, ACT>), ep)
#define LI_TILE(BM, BN, NS) (act == LI_ACT_CLAMPED ? LI_TILE_AS(BM, BN, NS, LI_ACT_CLAMPED) : act ? LI_TILE_AS(BM, BN, NS, LI_ACT_GELU_TANH) : LI_TILE_AS(BM, BN, NS, 0))
    switch (gated_tiling_of(M, N, K)) {
    case 0: return LI_DMA(128, 128, 4, 2);
    case 1: return LI_DMA(128, 256, 3, 2);
    case 2: return LI_DMA(128, 192, 3, 4);
    case 3: return LI_DMA(256, 128, 3, 2);
    case 4: return LI_DMA(256, 256, 2, 2);
    case 5: return LI_TILE(128, 320, 2);
    case 6: return LI_TILE(192, 256, 2);
    case 7: return LI_TILE(192, 320, 2);
    case 8: return LI_TILE(256, 192, 2);
    default: return LI_TILE(256, 256, 2);
    }
#undef LI_TILE
#undef LI_TILE_AS
#undef LI_GATED
#undef LI_DMA
#undef LI_DMA_AS
}

// The packed q/k/v projection of up to 32 rows with the half-split rotary encoding of query and key
// heads and the write of keys and values into their page slots as its epilogue (see ROPE above).
// w [(nh + 2 nkv) dh, K] bfloat16, bias float32 or null, out [M, (nh + 2 nkv) dh] bfloat16 (rotated
// q, rotated k, v), cos/sin float32 [M, dh / 2], slot_map int32 [M], kc/vc the cache layer.
// row_parts, nparts, eps: as for li_linear_swiglu.
extern "C" int li_linear_rope_store(const void* x, const void* w, const float* bias, void* out, int M, int K,
                                    const float* cos, const float* sin, const int* slot_map, void* kc, void* vc,
                                    int nh, int nkv, int dh, int page_size, int num_pages,
                                    const float* row_parts, int nparts, float eps, hipStream_t stream) {
    if (M <= 0 || M > 32 || K <= 0 || K % 8 || nh <= 0 || nkv <= 0 || dh <= 0 || dh % 16 || page_size <= 0 ||
        num_pages <= 0 || (long)(nh + 2 * nkv) * dh > 0x7fffffffL)
        return LI_ERR_SIZE;
    const int N = (nh + 2 * nkv) * dh;
    SkinnyArgs a{(const bf16_t*)x, (const bf16_t*)w, bias, out, M, N, K, 0, cos, sin, slot_map,
                 (bf16_t*)kc, (bf16_t*)vc, nh, nkv, dh, page_size, num_pages,
                 nullptr, nullptr, nullptr, row_parts, row_parts ? nparts : 0, eps};
    if (row_parts && (nparts <= 0 || nparts > SK_MAX_PARTS || eps < 0.f)) return LI_ERR_SIZE;
    return launch_skinny_rope(a, stream);
}
