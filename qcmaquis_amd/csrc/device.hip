// gfx950 kernels of the contraction path.
//
//  * gemm_kernel: grouped, batched FP64 / FP32 GEMM over a host-built tile table.  32x128, 64x64,
//    96x64 or 128x64 output tiles per 256-thread workgroup (four wave64s in a 2x2 grid), wider ones
//    in stages split along K; operands staged through LDS in K-slices of 8 with the next slice
//    prefetched into registers.  Each output tile is owned by one workgroup or, when K is
//    split, by a fixed set of partial tiles summed in order by gemm_reduce_kernel: no atomics.
//  * sblock_kernel: the MPO-term sum (reference create_s / create_s_r, solver/tasks.cpp:425-494)
//    as a block-sparse product on the matrix cores: up to 64 output tiles ("lines") of equal shape
//    at a time, in groups of 16, Y_g = alpha_g * X over the union of the T tiles they read, each
//    group only over the k-steps whose tiles it reads.
//  * copy / reshape / fill kernels for panel set-up and MPS pairing changes.
//  * FP64 Davidson vector kernels with device-resident coefficients.
#include "device.hpp"

#include <type_traits>

namespace mq {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

namespace {

// The 16x16x4 matrix-core step of each compute precision.  Operands (measured on gfx950): lane l
// supplies A[l % 16][l / 16] and B[l / 16][l % 16]; accumulator register r of lane l holds
// D[row(l, r)][l % 16] with row = l / 16 + 4 r for FP64 and 4 (l / 16) + r for FP32.
template <class T> struct Mma;
template <> struct Mma<double> {
    typedef double4_t acc_t;
    static __device__ inline acc_t step(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ inline int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <> struct Mma<float> {
    typedef float4_t acc_t;
    static __device__ inline acc_t step(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ inline int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

template <class T> __device__ inline T ld_or_zero(const T* p, bool ok) { return ok ? *p : T(0); }

// Split-BF16 products (precision MQ_PREC_BF16X3): an FP32 operand x = hi + lo with hi its leading
// 16 bits (a BF16 value, cut) and lo the rest rounded to nearest BF16, so |x - hi - lo| <= 2^-16 |x|;
// a product is hi_a hi_b + hi_a lo_b + lo_a hi_b on the BF16 matrix cores with FP32 accumulation
// (lo_a lo_b, at most 2^-14 of it, is left out).  The 16x16x16 step: lane l supplies four
// consecutive k of A[l % 16][4 (l / 16) + q] and B[4 (l / 16) + q][l % 16]; the accumulator
// layout is the one of the FP32 16x16x4 step.
typedef short bf16x4_t __attribute__((ext_vector_type(4)));
__device__ inline void split_bf16(float x, short& hi, short& lo) {
    const uint32_t u = __float_as_uint(x);
    hi = short(u >> 16);
    const uint32_t r = __float_as_uint(x - __uint_as_float(u & 0xffff0000u));
    lo = short((r + 0x7fffu + ((r >> 16) & 1u)) >> 16);
}

// One BM x BN output tile (BM = 32 FM, BN = 16 FN WN) per workgroup of 2 WN waves; the waves form a
// 2 x WN grid and take every second 16-row and every WN-th 16-column step of the tile, so a tile
// cut short by the end of C leaves each of them its share.  Operands of type TI, computed in TI,
// output converted to TO.  The tile reduces over [k0, k1) and writes C, or its partial tile (type
// TI) into the workspace (split K).  K slices of KS go through two LDS buffers (one barrier per
// slice), the next slice prefetched into registers.
//
// Every thread keeps pointers to the operand elements it stages and moves them on by a fixed step
// per slice; rows and columns past the end of C read the last valid one (their products are not
// stored), so only the last, shorter slice needs checks.  Matrix-core steps outside C, and k steps
// of four outside the last slice, are skipped: sector sizes leave 0.2-0.8 of whole tiles useful, of
// 16 x 16 x 4 steps 0.6-0.95.  T-GEMMs, FP64, checks per element and whole tiles -> now: 18 orbitals,
// TwoU1, M = 509 0.51 -> 0.32 ms, M = 128 0.11 -> 0.04 ms; 20 orbitals, SU2U1, M = 2048 17.0 -> 14.8.
template <int FM, int FN, class TI, int KS, int WN>
struct GemmLds {
    // rows padded so that the stores of a slice whose k runs across lanes meet every bank once
    static constexpr int PAD = 16 / int(sizeof(TI));
    TI A[2][KS][32 * FM + PAD];
    TI B[2][KS][16 * FN * WN + PAD];
};

// the body of gemm_kernel for one orientation of its operands
template <int FM, int FN, class TI, class TO, int KS, int WN, bool BF3, bool TA, bool TB>
__device__ __forceinline__ void gemm_tile(GemmLds<FM, FN, TI, KS, WN>& lds, GemmTile const& tile, GemmDesc const& g,
                                          const GemmRow* __restrict__ rows, Bases const& bases, TI* __restrict__ ws) {
    constexpr int THREADS = 128 * WN;
    constexpr int BM = 32 * FM, BN = 16 * FN * WN;
    constexpr int NA = BM * KS / THREADS, NB = BN * KS / THREADS;  // operand elements staged per thread and K slice
    static_assert(KS % 4 == 0 && NA * THREADS == BM * KS && NB * THREADS == BN * KS && THREADS % KS == 0 && THREADS % BN == 0,
                  "K slice geometry");
    static_assert(!BF3 || (std::is_same<TI, float>::value && KS % 16 == 0), "split-BF16 products: FP32 operands, K slices of 16");
    typedef typename Mma<TI>::acc_t acc_t;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int fr = lane & 15, fk = lane >> 4;
    const int m0 = tile.tm * BM, n0 = tile.tn * BN;
    const int ml = g.M - m0 < BM ? g.M - m0 : BM, nl = g.N - n0 < BN ? g.N - n0 : BN;  // rows and columns inside C
    const bool rmap = !TA && (g.flags & GEMM_ROWMAP);
    const TI* A = static_cast<const TI*>(bases.p[g.base_a]) + (rmap ? 0 : g.a + int64_t(tile.batch) * g.sa);
    const TI* B = static_cast<const TI*>(bases.p[g.base_b]) + g.b + int64_t(tile.batch) * g.sb;

    // element i of this thread in the BM x KS slice of A: the contiguous dimension of the operand
    // runs across consecutive threads.  Rows along threads (not transposed): with BM dividing the
    // workgroup every element of a thread is of one row, k ADK apart, so one pointer walks through
    // them.  k along threads: one k, a pointer per row.  The KS x BN slice of B likewise.
    constexpr bool AWALK = !TA && THREADS % BM == 0;
    constexpr int ADK = AWALK ? THREADS / BM : 0, ADM = THREADS / KS;
    constexpr int BDK = THREADS / BN, BDN = THREADS / KS;
    auto a_m = [&](int i) { return TA ? tid / KS + ADM * i : (tid + THREADS * i) % BM; };
    auto a_k = [&](int i) { return TA ? tid % KS : (tid + THREADS * i) / BM; };
    auto b_n = [&](int i) { return TB ? tid % BN : tid / KS + BDN * i; };
    auto b_k = [&](int i) { return TB ? tid / BN + BDK * i : tid % KS; };
    const TI *pa[AWALK ? 1 : NA], *pb[TB ? 1 : NB];
    int64_t a_step, b_step;  // per element of a walk, else per slice
#pragma unroll
    for (int i = 0; i < (AWALK ? 1 : NA); ++i) {
        const int m = m0 + (a_m(i) < ml ? a_m(i) : ml - 1);
        const int64_t k = tile.k0 + a_k(i);
        if (rmap) {
            const GemmRow r = rows[g.a + m];
            pa[i] = A + r.a + k * r.ld;
            a_step = int64_t(AWALK ? ADK : KS) * r.ld;
        } else {
            pa[i] = TA ? A + int64_t(m) * g.lda + k : A + m + k * g.lda;
            a_step = TA ? KS : int64_t(AWALK ? ADK : KS) * g.lda;
        }
    }
#pragma unroll
    for (int i = 0; i < (TB ? 1 : NB); ++i) {
        const int n = n0 + (b_n(i) < nl ? b_n(i) : nl - 1);
        const int64_t k = tile.k0 + b_k(i);
        if (TB) {
            // columns in blocks of g.nb, a block every g.sb elements
            pb[i] = (g.flags & GEMM_NBLOCKS ? B + int64_t(n / g.nb) * g.sb + n % g.nb : B + n) + k * g.ldb;
        } else {
            pb[i] = B + k + int64_t(n) * g.ldb;
        }
    }
    b_step = TB ? int64_t(BDK) * g.ldb : KS;
    TI ra[NA], rb[NB];
    auto load = [&](int kn) {  // the next kn <= KS values of k
        if (kn >= KS) {
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                const TI*& p = pa[AWALK ? 0 : i];
                ra[i] = *p;
                p += a_step;
            }
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const TI*& p = pb[TB ? 0 : i];
                rb[i] = *p;
                p += b_step;
            }
        } else {
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                const TI*& p = pa[AWALK ? 0 : i];
                ra[i] = ld_or_zero(p, a_k(i) < kn);
                p += a_step;
            }
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const TI*& p = pb[TB ? 0 : i];
                rb[i] = ld_or_zero(p, b_k(i) < kn);
                p += b_step;
            }
        }
    };

    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    // matrix-core steps of this wave inside C
    const int fm = (ml - 16 * wm + 31) / 32, fn = (nl - 16 * wn + 16 * WN - 1) / (16 * WN);
    // operands swapped in every step: the instruction accumulates the transposed tile C^T = B^T A^T
    auto multiply = [&](int buf, int kn, auto all) {
        constexpr bool ALL = decltype(all)::value;
        if constexpr (BF3) {
#pragma unroll
            for (int kk = 0; kk < KS; kk += 16) {
                bf16x4_t ah[FM], al[FM], bh[FN], bl[FN];
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        short h, l;
                        split_bf16(lds.A[buf][kk + 4 * fk + q][16 * (2 * i + wm) + fr], h, l);
                        ah[i][q] = h;
                        al[i][q] = l;
                    }
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        short h, l;
                        split_bf16(lds.B[buf][kk + 4 * fk + q][16 * (WN * j + wn) + fr], h, l);
                        bh[j][q] = h;
                        bl[j][q] = l;
                    }
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        if (ALL || (i < fm && j < fn)) {
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bh[j], ah[i], acc[i][j], 0, 0, 0);
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bh[j], al[i], acc[i][j], 0, 0, 0);
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bl[j], ah[i], acc[i][j], 0, 0, 0);
                        }
            }
        } else {
#pragma unroll
            for (int kk = 0; kk < KS; kk += 4) {
                if (kk < kn) {
                    TI af[FM], bf[FN];
#pragma unroll
                    for (int i = 0; i < FM; ++i) af[i] = lds.A[buf][kk + fk][16 * (2 * i + wm) + fr];
#pragma unroll
                    for (int j = 0; j < FN; ++j) bf[j] = lds.B[buf][kk + fk][16 * (WN * j + wn) + fr];
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j)
                            if (ALL || (i < fm && j < fn)) acc[i][j] = Mma<TI>::step(bf[j], af[i], acc[i][j]);
                }
            }
        }
    };
    auto reduce = [&](auto all) {
        int left = tile.k1 - tile.k0;
        if (left > 0) load(left);
        for (int buf = 0; left > 0; buf ^= 1, left -= KS) {
#pragma unroll
            for (int i = 0; i < NA; ++i) lds.A[buf][a_k(i)][a_m(i)] = ra[i];
#pragma unroll
            for (int i = 0; i < NB; ++i) lds.B[buf][b_k(i)][b_n(i)] = rb[i];
            __syncthreads();
            if (left > KS) load(left - KS);
            multiply(buf, left, all);
        }
    };
    if (ml == BM && nl == BN) reduce(std::true_type());
    else reduce(std::false_type());

    // D = C^T: register r of lane l holds C[l % 16][row(l, r)] of its 16 x 16 tile, so
    // consecutive lanes store consecutive rows of a column
    TO* C = static_cast<TO*>(bases.p[g.base_c]) + (rmap ? 0 : g.c + int64_t(tile.batch) * g.sc);
    const bool split = tile.ws >= 0;  // never for stacked problems
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int mm = 16 * (2 * i + wm) + fr, m = m0 + mm;
        if (mm >= ml) continue;
        // column n of this row at c_row + n * c_ld
        TO* c_row = C + m;
        int64_t c_ld = g.ldc;
        if (rmap) {
            const GemmRow r = rows[g.a + m];
            c_row = C + r.c + int64_t(tile.batch) * g.sc * r.ld;
            c_ld = r.ld;
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int nn = 16 * (WN * j + wn) + Mma<TI>::row(lane, r);
                if (nn >= nl) continue;
                if (split) ws[tile.ws + mm + int64_t(nn) * BM] = acc[i][j][r];
                else c_row[int64_t(n0 + nn) * c_ld] = TO(acc[i][j][r]);
            }
        }
    }
}

template <int FM, int FN, class TI, class TO, int KS, int MINB = 1, int WN = 2, bool BF3 = false>
__global__ __launch_bounds__(128 * WN, MINB) void gemm_kernel(const GemmDesc* __restrict__ probs,
                                                              const GemmRow* __restrict__ rows,
                                                              const GemmTile* __restrict__ tiles, Bases bases,
                                                              TI* __restrict__ ws) {
    __shared__ GemmLds<FM, FN, TI, KS, WN> lds;
    const GemmTile tile = tiles[blockIdx.x];
    const GemmDesc g = probs[tile.prob];
    const bool tb = g.flags & GEMM_TRANS_B;
    if (g.flags & GEMM_TRANS_A) {
        if (tb) gemm_tile<FM, FN, TI, TO, KS, WN, BF3, true, true>(lds, tile, g, rows, bases, ws);
        else gemm_tile<FM, FN, TI, TO, KS, WN, BF3, true, false>(lds, tile, g, rows, bases, ws);
    } else {
        if (tb) gemm_tile<FM, FN, TI, TO, KS, WN, BF3, false, true>(lds, tile, g, rows, bases, ws);
        else gemm_tile<FM, FN, TI, TO, KS, WN, BF3, false, false>(lds, tile, g, rows, bases, ws);
    }
}

// C tile = sum of its split partials, added in split order; blockIdx.y selects 256 elements of
// the tile, so one output tile is reduced by up to 64 workgroups
constexpr int REDUCE_CHUNKS = 64;  // 16384 (largest tile) / 256
constexpr bool reduce_covers(int sh) { return sh == GEMM_N_SHAPES || (gemm_bm(sh) * gemm_bn(sh) <= REDUCE_CHUNKS * 256 && reduce_covers(sh + 1)); }
static_assert(reduce_covers(0), "reduce grid covers every tile shape");
template <class TW, class TO>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const GemmDesc* __restrict__ probs,
                                                          const GemmReduce* __restrict__ jobs, Bases bases,
                                                          const TW* __restrict__ ws) {
    const GemmReduce job = jobs[blockIdx.x];
    const GemmDesc g = probs[job.prob];
    const int bm = gemm_bm(job.shape), bn = gemm_bn(job.shape);
    const int m0 = job.tm * bm, n0 = job.tn * bn;
    TO* C = static_cast<TO*>(bases.p[g.base_c]) + g.c + int64_t(job.batch) * g.sc;
    const int64_t tile_elems = int64_t(bm) * bn;
    const int idx = int(blockIdx.y) * 256 + int(threadIdx.x);
    if (idx < bm * bn) {
        const int mm = idx % bm, nn = idx / bm;
        const int m = m0 + mm, n = n0 + nn;
        if (m < g.M && n < g.N) {
            TW sum = 0;
            for (int s = 0; s < job.nsplit; ++s) sum += ws[job.ws + s * tile_elems + idx];
            C[m + int64_t(n) * g.ldc] = TO(sum);
        }
    }
}

// Block-form MPO-term sum on the matrix cores.  Per k-step (4 union tiles) every group of 16 lines
// that reads one of its tiles computes Y_g(16 lines x 16 elements) += alpha_g(16 x 4) * X(4 tiles x
// 16 elements): lane l supplies element l % 16 of tile l / 16 and alpha of line l % 16 for tile
// l / 16.  A wave owns 32 tile elements: lane l loads the consecutive elements 2 (l % 16) and
// 2 (l % 16) + 1 of its tile in one access, column tile j of the matrix-core steps takes the
// elements of parity j, and the lane's results are consecutive elements of S again.  Coefficients and
// tile offsets go to LDS without passing through registers.  The waves of a workgroup work by the
// block's tile size (SWorkCounts): one block on all of them (SBLOCK_ELEMS elements, tables staged
// once per workgroup), a block of 33 to 64 elements on two, or one block per wave; in the last two
// every wave stages its own block's tables and runs without barriers.
//
// Bound: L2-miss traffic (every block reads the union of its T tiles, T 2.1-2.5 times in all, and
// writes S) where tiles are large, waiting on the chain tables -> tiles -> matrix cores where they
// are small.  Staging a whole block's tables at once (most blocks fit one pass) in place of eight
// k-steps at a time behind two barriers each, one 16-byte load per k-step instead of two of 8, and
// line tables read once through LDS cut the vector-memory instructions to a third.  FP64, before ->
// now: 18 orbitals, TwoU1, M = 509 1.64 -> 0.81 ms; 20 orbitals, SU2U1, M = 700 2.82 -> 1.80 ms,
// M = 2048 19.2 -> 14.1 ms (75 GB read and written); FP32 there 10.97 -> 8.02 ms.  Without barriers
// at all (every wave its own loads into registers) the first took 1.36 ms; four column tiles per
// wave 1.02 ms; two or four k-steps of loads in flight 0.93 and 0.95 where three took 0.92.
constexpr int SB_XCDS = 8;                              // XCDs of an MI355X
constexpr int SB_SUB = 64;                              // coefficient sub-blocks staged per workgroup
constexpr int SB_KS = 64;                               // k-steps staged per workgroup
constexpr int SB_NC = 2;                                // column tiles per wave
constexpr int SB_U = 3;                                 // k-steps whose tile loads are issued together
constexpr int SB_THREADS = 64 * SB_WAVES;
constexpr int SB_SUB1 = SB_SUB / SB_WAVES, SB_KS1 = SB_KS / SB_WAVES;  // one wave's share of the staging
static_assert(SBLOCK_GROUP == 16 && 16 * SB_NC == 32 && SB_WAVES * 16 * SB_NC == SBLOCK_ELEMS && SB_WAVES % 2 == 0 && SB_SUB1 >= SBLOCK_GROUPS && SB_KS <= 64,
              "S block geometry");

// n bytes (a multiple of 16) from src to LDS at dst (both 16-byte aligned) by `lanes` lanes of whole
// waves, this one being number `lane`; in flight until the wave's next wait for vector memory
__device__ inline void lds_fetch(const void* src, void* dst, int n, int lane, int lanes) {
    const char* s = static_cast<const char*>(src);
    char* d = static_cast<char*>(dst);
    for (int o = __builtin_amdgcn_readfirstlane(lane & ~63) * 16; o < n; o += lanes * 16)
        if (o + 16 * (lane & 63) < n)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(s + o + 16 * (lane & 63)),
                                             (__attribute__((address_space(3))) void*)(d + o), 16, 0, 0);
}

// two consecutive elements at any element alignment
template <class T> struct PairOf { typedef T type __attribute__((ext_vector_type(2), aligned(sizeof(T)))); };

template <class T>
__global__ __launch_bounds__(SB_THREADS) __attribute__((amdgpu_waves_per_eu(4))) void sblock_kernel(
    const SBlock* __restrict__ blocks, const SWork* __restrict__ launch, const SWork* __restrict__ work, SWorkCounts n,
    const int64_t* __restrict__ utile, const uint32_t* __restrict__ kstep, const T* __restrict__ ualpha,
    const int64_t* __restrict__ lsoff, const int32_t* __restrict__ llds, const T* __restrict__ X, T* __restrict__ S,
    int xcd_contiguous) {
    typedef typename Mma<T>::acc_t acc_t;
    typedef typename PairOf<T>::type pair_t;
    __shared__ __attribute__((aligned(16))) T s_alpha[SB_SUB * 64];
    __shared__ __attribute__((aligned(16))) int64_t s_off[SB_KS * 4];
    __shared__ __attribute__((aligned(16))) int64_t s_lsoff[SB_WAVES * SBLOCK_LINES];
    __shared__ __attribute__((aligned(16))) int32_t s_llds[SB_WAVES * SBLOCK_LINES];
    // Workgroups are dispatched to the XCDs in turn (workgroup i on XCD i mod 8); with
    // xcd_contiguous each XCD takes a contiguous range of the work list instead, so consecutive
    // work items (neighbouring blocks' slices of shared T tiles) meet in one XCD's L2.  The map is
    // a bijection of [0, gridDim.x).
    int wg = int(blockIdx.x);
    if (xcd_contiguous) {
        const int nw = int(gridDim.x), q = nw / SB_XCDS, r = nw % SB_XCDS;
        const int x = wg % SB_XCDS, k = wg / SB_XCDS;
        wg = x < r ? x * (q + 1) + k : r * (q + 1) + (x - r) * q + k;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    SWork w = launch[wg];
    const bool team = w.blk >= 0;
    int sub = wave;  // this wave's slice of its work item
    if (!team) {     // -w.blk waves per item, from work[w.n0]
        const int lw = -w.blk - 1, wi = w.n0 + (wave >> lw);
        sub = wave & lw;
        if (wi >= (lw ? n.team + n.pair : n.team + n.pair + n.solo)) return;
        w = work[wi];
    }
    const SBlock b = blocks[w.blk];
    const int n0 = w.n0 + 16 * SB_NC * sub;
    // a wave past the tile end loads and stores no tile but takes part in its team's barriers
    const bool active = n0 < b.E;
    if (!team && !active) return;
    const int li = lane & 15, lk = lane >> 4;
    T* al = s_alpha + (team ? 0 : wave * SB_SUB1 * 64);
    int64_t* of = s_off + (team ? 0 : wave * SB_KS1 * 4);
    int64_t* so = s_lsoff + (team ? 0 : wave * SBLOCK_LINES);
    int32_t* ld = s_llds + (team ? 0 : wave * SBLOCK_LINES);
    const int cap_sub = team ? SB_SUB : SB_SUB1, cap_k = team ? SB_KS : SB_KS1;
    const int st_lane = team ? int(threadIdx.x) : lane, st_lanes = team ? SB_THREADS : 64;
    const uint32_t* kw = kstep + b.k_off;
    // this lane's elements e0, e0 + 1; past the tile's end it reads what follows the tile in
    // the T buffer (SB_T_SPARE elements after the last one) and stores none of it
    const int e0 = n0 + 2 * li;
    const int ec = e0 < b.E ? e0 : b.E - 1;
    acc_t acc[SBLOCK_GROUPS][SB_NC];
#pragma unroll
    for (int g = 0; g < SBLOCK_GROUPS; ++g)
#pragma unroll
        for (int j = 0; j < SB_NC; ++j) acc[g][j] = acc_t{0, 0, 0, 0};

    lds_fetch(lsoff + b.line0, so, SBLOCK_LINES * 8, st_lane, st_lanes);
    lds_fetch(llds + b.line0, ld, SBLOCK_LINES * 4, st_lane, st_lanes);
    for (int c0 = 0; c0 < b.nk;) {
        // the next k-steps whose tables fit: lane l looks at k-step c0 + l
        const int kl = c0 + lane;
        const uint32_t word = kl < b.nk ? kw[kl] : 0;
        const int a0 = __builtin_amdgcn_readfirstlane(int(word >> 8));
        const int end = kl + 1 < b.nk ? int(kw[kl + 1] >> 8) : b.na;
        const int cn = __builtin_popcountll(__ballot(kl < b.nk && lane < cap_k && end - a0 <= cap_sub));
        const int an = __builtin_amdgcn_readlane(end, cn - 1) - a0;
        if (team && c0 > 0) __syncthreads();  // the previous k-steps' tables are consumed
        asm volatile("" ::: "memory");
        lds_fetch(utile + 4 * (int64_t(b.k_off) + c0), of, 32 * cn, st_lane, st_lanes);
        lds_fetch(ualpha + 64 * (b.a_off + a0), al, 64 * int(sizeof(T)) * an, st_lane, st_lanes);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (team) __syncthreads();
        if (active) {
            // the tile elements of the k-steps [k, k + SB_U)
            auto load_x = [&](pair_t (&x)[SB_U], int k) {
#pragma unroll
                for (int u = 0; u < SB_U; ++u) {
                    const int64_t o = k + u < cn ? of[4 * (k + u) + lk] : -1;
                    const pair_t v = *reinterpret_cast<const pair_t*>(X + (o < 0 ? 0 : o) + ec);
#pragma unroll
                    for (int j = 0; j < SB_NC; ++j) x[u][j] = o < 0 ? T(0) : v[j];  // empty slot (last k-step): a zero tile
                }
            };
            auto mma = [&](pair_t (&x)[SB_U], int k) {
#pragma unroll
                for (int u = 0; u < SB_U; ++u) {
                    if (k + u >= cn) break;
                    const uint32_t wd = __builtin_amdgcn_readlane(word, k + u);
                    const T* pa = al + 64 * (int(wd >> 8) - a0) + lane;
#pragma unroll
                    for (int g = 0; g < SBLOCK_GROUPS; ++g)
                        if ((wd >> g) & 1u) {
                            const T a = *pa;
                            pa += 64;
#pragma unroll
                            for (int j = 0; j < SB_NC; ++j) acc[g][j] = Mma<T>::step(a, x[u][j], acc[g][j]);
                        }
                }
            };
            pair_t xa[SB_U], xb[SB_U];
            load_x(xa, 0);
            for (int k = 0; k < cn; k += 2 * SB_U) {
                load_x(xb, k + SB_U);
                mma(xa, k);
                load_x(xa, k + 2 * SB_U);
                mma(xb, k + SB_U);
            }
        }
        c0 += cn;
    }
    if (b.nk == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (team) __syncthreads();
    }
    if (!active || e0 >= b.E) return;
    // register r of lane l holds Y_g[line row(l, r)][element]: the lane's elements are stored at once
    // unless a tile column ends among them
    const int r_ = e0 % b.rows, c_ = e0 / b.rows;
    const bool whole = r_ + 1 < b.rows;
#pragma unroll
    for (int g = 0; g < SBLOCK_GROUPS; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = SBLOCK_GROUP * g + Mma<T>::row(lane, r);
            if (i >= b.nlines) continue;
            T* p = S + so[i] + r_ + int64_t(c_) * ld[i];
            if (whole) {
                pair_t v;
                v.x = acc[g][0][r];
                v.y = acc[g][1][r];
                *reinterpret_cast<pair_t*>(p) = v;
            } else {
                *p = acc[g][0][r];
                if (e0 + 1 < b.E) p[int64_t(ld[i]) - r_] = acc[g][1][r];
            }
        }
}

// Small-tile MPO-term sum: a work item is up to 256 >> lg lines of 2^lg lanes each (tile elements
// <= 2^lg); lane e of a line sums alpha_k * T[t_off_k + e] over the line's terms in term order,
// four terms' loads ahead of their multiply-adds, and writes element e of the line's S tile.  The
// lanes of a line read the same term entries; no LDS and no barrier, so lanes past their line's
// tile simply return.
template <class T>
__global__ __launch_bounds__(SMALL_LINE_LANES) void small_lines_kernel(const SSmallWork* __restrict__ work,
                                                                       const SLine* __restrict__ lines,
                                                                       const STerm* __restrict__ terms,
                                                                       const T* __restrict__ X, T* __restrict__ S) {
    const SSmallWork w = work[blockIdx.x];
    const int li = int(threadIdx.x) >> w.lg, e = int(threadIdx.x) & ((1 << w.lg) - 1);
    if (li >= w.n) return;
    const SLine l = lines[w.line0 + li];
    if (e >= l.rows * l.cols) return;
    T acc = T(0);
    int k = l.t0;
    for (; k + 4 <= l.t1; k += 4) {
        const STerm a = terms[k], b = terms[k + 1], c = terms[k + 2], d = terms[k + 3];
        const T xa = X[a.t_off + e], xb = X[b.t_off + e], xc = X[c.t_off + e], xd = X[d.t_off + e];
        acc += T(a.alpha) * xa;
        acc += T(b.alpha) * xb;
        acc += T(c.alpha) * xc;
        acc += T(d.alpha) * xd;
    }
    for (; k < l.t1; ++k) acc += T(terms[k].alpha) * X[terms[k].t_off + e];
    S[l.s_off + e % l.rows + int64_t(e / l.rows) * l.lds] = acc;
}

// One S line (rows x cols tile at s_off, leading dimension lds) per workgroup; element e of the
// tile is the sum over the line's terms of alpha * T[t_off + e], in term order (reference:
// compute_s_stackedv, gpu_dgemm_ddot.cu:282-359, one gather per term).  Lines without terms
// write zeros.
__global__ __launch_bounds__(256) void sline_kernel(const SLine* __restrict__ lines, const STerm* __restrict__ terms,
                                                    const double* __restrict__ T, double* __restrict__ S) {
    const SLine l = lines[blockIdx.x];
    const int E = l.rows * l.cols;
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        double acc = 0.0;
        for (int k = l.t0; k < l.t1; ++k) acc += terms[k].alpha * T[terms[k].t_off + e];
        S[l.s_off + e % l.rows + int64_t(e / l.rows) * l.lds] = acc;
    }
}

// MPO-term adjoint of the term sum.  E = <psi|H psi> = sum over terms k of alpha_k <Y_line(k),
// T_k> with Y = L_panel^T psi laid out like S, so dE/d(scale of MPO term m) is the sum over the
// terms k from m of beta_k <Y_line(k), T_k> (beta_k = d alpha_k / d scale_m).  A workgroup takes
// a run of one line's terms; each group of 2^lg lanes forms one term's dot product over the tile
// elements and reduces it with cross-lane exchanges inside the group.
__global__ __launch_bounds__(TERM_GRAD_THREADS) void term_grad_kernel(
    const TermGradWork* __restrict__ work, const SLine* __restrict__ lines, const STerm* __restrict__ terms,
    const uint32_t* __restrict__ src, const double* __restrict__ beta, const double* __restrict__ Y,
    const double* __restrict__ X, double* __restrict__ grad) {
    const TermGradWork w = work[blockIdx.x];
    const SLine l = lines[w.line];
    const int E = l.rows * l.cols;
    const int G = 1 << w.lg;
    const int grp = int(threadIdx.x) >> w.lg, e0 = int(threadIdx.x) & (G - 1);
    const int ngroups = TERM_GRAD_THREADS >> w.lg;
    for (int k = w.t0 + grp; k < w.t1; k += ngroups) {
        const int64_t toff = terms[k].t_off;
        double acc = 0.0;
        for (int e = e0; e < E; e += G) acc += Y[l.s_off + e % l.rows + int64_t(e / l.rows) * l.lds] * X[toff + e];
        // the lanes of one group share k, so a group is active or idle as a whole
        for (int off = G >> 1; off > 0; off >>= 1) acc += __shfl_xor(acc, off, G);
        if (e0 == 0) atomicAdd(grad + src[k], beta[k] * acc);
    }
}

template <class TI, class TO>
__global__ void convert_kernel(const TI* __restrict__ src, TO* __restrict__ dst, uint64_t n) {
    for (uint64_t i = blockIdx.x * uint64_t(blockDim.x) + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
        dst[i] = TO(src[i]);
}

__global__ void fill_kernel(double* p, uint64_t n, double v) {
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}

// grid: x = job, y = chunk of the job's elements
__global__ void copy_jobs_kernel(const CopyJob* __restrict__ jobs, const double* __restrict__ src,
                                 double* __restrict__ dst) {
    const CopyJob j = jobs[blockIdx.x];
    const int64_t per = int64_t(j.rows) * j.cols;
    const int64_t total = per * j.nblocks;
    for (int64_t i = int64_t(blockIdx.y) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.y) * blockDim.x) {
        int64_t b = i / per, e = i % per;
        int r = int(e % j.rows), c = int(e / j.rows);
        // destination block rows x cols; transposed source block is cols x rows
        double v = j.trans ? src[j.src + b * per + c + int64_t(r) * j.cols] : src[j.src + b * per + e];
        dst[j.dst + b * per + e] = v;
    }
}

// element (ss, rr, ll) of a segment: rp[ll + (ss*rs + rr)*ls]  <->  lp[ss*ls + ll + rr*lp_ld]
__global__ void reshape_kernel(const ReshapeSeg* __restrict__ segs, const double* __restrict__ src,
                               double* __restrict__ dst, int to_left) {
    const ReshapeSeg s = segs[blockIdx.x];
    const int64_t total = int64_t(s.ls) * s.rs * s.d;
    for (int64_t i = int64_t(blockIdx.y) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.y) * blockDim.x) {
        int ll = int(i % s.ls);
        int64_t q = i / s.ls;  // = ss*rs + rr
        int rr = int(q % s.rs), ss = int(q / s.rs);
        int64_t rp = s.rp + ll + q * s.ls;
        int64_t lp = s.lp + int64_t(ss) * s.ls + ll + int64_t(rr) * s.lp_ld;
        if (to_left) dst[lp] = src[rp];
        else dst[rp] = src[lp];
    }
}

constexpr int DOT_THREADS = 256;

__device__ inline double block_sum(double v) {
    __shared__ double red[DOT_THREADS / 64];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) red[w] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < DOT_THREADS / 64; ++i) r += red[i];
    return r;
}

__global__ __launch_bounds__(DOT_THREADS) void dot_partial_kernel(const double* __restrict__ x,
                                                                  const double* __restrict__ y, uint64_t n,
                                                                  double* __restrict__ work) {
    double s = 0.0;
    for (uint64_t i = uint64_t(blockIdx.x) * DOT_THREADS + threadIdx.x; i < n; i += uint64_t(gridDim.x) * DOT_THREADS)
        s += x[i] * y[i];
    double r = block_sum(s);
    if (threadIdx.x == 0) work[blockIdx.x] = r;
}

__global__ __launch_bounds__(DOT_THREADS) void dot_final_kernel(const double* __restrict__ work, int nparts,
                                                                double* __restrict__ out) {
    double s = 0.0;
    for (int i = threadIdx.x; i < nparts; i += DOT_THREADS) s += work[i];
    double r = block_sum(s);
    if (threadIdx.x == 0) out[0] = r;
}

__global__ void axpy_dev_kernel(double* __restrict__ y, const double* __restrict__ x, uint64_t n,
                                const double* __restrict__ num, const double* __restrict__ den, double sign) {
    const double coef = sign * num[0] / (den ? den[0] : 1.0);
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
        y[i] += coef * x[i];
}

// Segmented forms for a batch of independent vectors concatenated in one buffer (segment s is
// elements off[s] .. off[s+1]-1; blockIdx.y = segment).  Dot: SEG_CHUNKS partial sums per
// segment, then one thread per segment adds them in chunk order (deterministic).
__global__ __launch_bounds__(DOT_THREADS) void seg_dot_partial_kernel(const double* __restrict__ x,
                                                                      const double* __restrict__ y,
                                                                      const int64_t* __restrict__ off,
                                                                      double* __restrict__ part) {
    const int seg = blockIdx.y;
    const int64_t a = off[seg], b = off[seg + 1];
    double s = 0.0;
    for (int64_t i = a + int64_t(blockIdx.x) * DOT_THREADS + threadIdx.x; i < b; i += int64_t(SEG_CHUNKS) * DOT_THREADS)
        s += x[i] * y[i];
    double r = block_sum(s);
    if (threadIdx.x == 0) part[int64_t(seg) * SEG_CHUNKS + blockIdx.x] = r;
}

__global__ void seg_dot_final_kernel(const double* __restrict__ part, int nseg, double* __restrict__ out) {
    const int seg = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (seg >= nseg) return;
    double s = 0.0;
    for (int c = 0; c < SEG_CHUNKS; ++c) s += part[int64_t(seg) * SEG_CHUNKS + c];
    out[seg] = s;
}

// segment s: y = a[s]*y + b[s]*x (y not read where a[s] == 0)
__global__ void seg_axpby_kernel(double* __restrict__ y, const double* __restrict__ x, const int64_t* __restrict__ off,
                                 const double* __restrict__ ca, const double* __restrict__ cb) {
    const int seg = blockIdx.y;
    const int64_t i0 = off[seg], i1 = off[seg + 1];
    const double a = ca[seg], b = cb[seg];
    for (int64_t i = i0 + int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < i1; i += int64_t(gridDim.x) * blockDim.x)
        y[i] = a == 0.0 ? b * x[i] : a * y[i] + b * x[i];
}

// y = a*y + b*x; with a == 0 y is not read (it may hold anything, NaN included: BLAS beta = 0)
__global__ void axpby_kernel(double* __restrict__ y, const double* __restrict__ x, uint64_t n, double a, double b) {
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
        y[i] = a == 0.0 ? b * x[i] : a * y[i] + b * x[i];
}

__global__ void scale_rsqrt_kernel(double* __restrict__ x, uint64_t n, const double* __restrict__ nrm2) {
    const double s = 1.0 / sqrt(nrm2[0]);
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
        x[i] *= s;
}

inline unsigned grid_for(uint64_t n, int threads, unsigned cap = 8192) {
    uint64_t g = (n + threads - 1) / threads;
    if (g < 1) g = 1;
    return unsigned(g > cap ? cap : g);
}

}  // namespace

namespace {

// K slices of 8 with at most 128 VGPRs (two workgroups per SIMD): measured fastest for every tile
// shape on the H*psi stages of a 24-orbital, M = 512 site problem (short and long reductions alike)
constexpr int GEMM_KS = 8, GEMM_MINB = 4;

template <class TI, class TO, bool BF3 = false>
void launch_gemm_t(const GemmDesc* probs, const GemmRow* rows, const GemmTile* const* tiles, const int64_t* n_tiles,
                   const GemmReduce* reduces, int64_t n_reduces, void* ws, Bases bases, hipStream_t stream) {
    TI* w = static_cast<TI*>(ws);
    constexpr int KSL = BF3 ? 16 : GEMM_KS;  // split-BF16 steps take 16 k at a time
    for (int sh = 0; sh < GEMM_N_SHAPES; ++sh) {
        for (int64_t off = 0; off < n_tiles[sh]; off += 0x7fffffff) {
            int64_t cnt = n_tiles[sh] - off < 0x7fffffff ? n_tiles[sh] - off : 0x7fffffff;
            if (sh == GEMM_32x128)
                hipLaunchKernelGGL((gemm_kernel<1, 4, TI, TO, KSL, GEMM_MINB, 2, BF3>), dim3(unsigned(cnt)), dim3(256), 0, stream, probs,
                                   rows, tiles[sh] + off, bases, w);
            else if (sh == GEMM_64x64)
                hipLaunchKernelGGL((gemm_kernel<2, 2, TI, TO, KSL, GEMM_MINB, 2, BF3>), dim3(unsigned(cnt)), dim3(256), 0, stream, probs,
                                   rows, tiles[sh] + off, bases, w);
            else if (sh == GEMM_96x64)
                hipLaunchKernelGGL((gemm_kernel<3, 2, TI, TO, KSL, GEMM_MINB, 2, BF3>), dim3(unsigned(cnt)), dim3(256), 0, stream, probs,
                                   rows, tiles[sh] + off, bases, w);
            else if (sh == GEMM_64x128)
                hipLaunchKernelGGL((gemm_kernel<2, 4, TI, TO, KSL, GEMM_MINB, 2, BF3>), dim3(unsigned(cnt)), dim3(256), 0, stream, probs,
                                   rows, tiles[sh] + off, bases, w);
            else if (sh == GEMM_128x128)
                hipLaunchKernelGGL((gemm_kernel<4, 2, TI, TO, KSL, GEMM_MINB / 2, 4, BF3>), dim3(unsigned(cnt)), dim3(512), 0,
                                   stream, probs, rows, tiles[sh] + off, bases, w);
            else
                hipLaunchKernelGGL((gemm_kernel<4, 2, TI, TO, KSL, GEMM_MINB, 2, BF3>), dim3(unsigned(cnt)), dim3(256), 0, stream, probs,
                                   rows, tiles[sh] + off, bases, w);
        }
    }
    for (int64_t off = 0; off < n_reduces; off += 0x7fffffff) {
        int64_t cnt = n_reduces - off < 0x7fffffff ? n_reduces - off : 0x7fffffff;
        hipLaunchKernelGGL((gemm_reduce_kernel<TI, TO>), dim3(unsigned(cnt), REDUCE_CHUNKS), dim3(256), 0, stream,
                           probs, reduces + off, bases, w);
    }
}

}  // namespace

hipError_t launch_gemm(GemmPrec prec, const GemmDesc* probs, const GemmRow* rows, const GemmTile* const* tiles,
                       const int64_t* n_tiles, const GemmReduce* reduces, int64_t n_reduces, void* ws, Bases bases,
                       hipStream_t stream) {
    switch (prec) {
        case GEMM_F64:
            launch_gemm_t<double, double>(probs, rows, tiles, n_tiles, reduces, n_reduces, ws, bases, stream);
            break;
        case GEMM_F32:
            launch_gemm_t<float, float>(probs, rows, tiles, n_tiles, reduces, n_reduces, ws, bases, stream);
            break;
        case GEMM_F32_OUT_F64:
            launch_gemm_t<float, double>(probs, rows, tiles, n_tiles, reduces, n_reduces, ws, bases, stream);
            break;
        case GEMM_BF3:
            launch_gemm_t<float, float, true>(probs, rows, tiles, n_tiles, reduces, n_reduces, ws, bases, stream);
            break;
        case GEMM_BF3_OUT_F64:
            launch_gemm_t<float, double, true>(probs, rows, tiles, n_tiles, reduces, n_reduces, ws, bases, stream);
            break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_slines(const SLine* lines, int64_t n_lines, const STerm* terms, const double* T, double* S,
                         hipStream_t stream) {
    for (int64_t off = 0; off < n_lines; off += 0x7fffffff) {
        int64_t cnt = n_lines - off < 0x7fffffff ? n_lines - off : 0x7fffffff;
        hipLaunchKernelGGL(sline_kernel, dim3(unsigned(cnt)), dim3(256), 0, stream, lines + off, terms, T, S);
    }
    return hipGetLastError();
}

template <class T>
hipError_t launch_sblocks(const SBlock* blocks, const SWork* launch, int64_t n_launch, const SWork* work, SWorkCounts n,
                          const int64_t* utile, const uint32_t* kstep, const T* ualpha, const int64_t* lsoff,
                          const int32_t* llds, const T* X, T* S, bool xcd_contiguous, hipStream_t stream) {
    if (n_launch > 0x7fffffff) return hipErrorInvalidValue;
    if (n_launch > 0)
        hipLaunchKernelGGL(sblock_kernel<T>, dim3(unsigned(n_launch)), dim3(SB_THREADS), 0, stream, blocks, launch, work, n,
                           utile, kstep, ualpha, lsoff, llds, X, S, int(xcd_contiguous));
    return hipGetLastError();
}
template hipError_t launch_sblocks<double>(const SBlock*, const SWork*, int64_t, const SWork*, SWorkCounts,
                                           const int64_t*, const uint32_t*, const double*, const int64_t*,
                                           const int32_t*, const double*, double*, bool, hipStream_t);
template hipError_t launch_sblocks<float>(const SBlock*, const SWork*, int64_t, const SWork*, SWorkCounts,
                                          const int64_t*, const uint32_t*, const float*, const int64_t*, const int32_t*,
                                          const float*, float*, bool, hipStream_t);

template <class T>
hipError_t launch_small_lines(const SSmallWork* work, int64_t n_work, const SLine* lines, const STerm* terms,
                              const T* X, T* S, hipStream_t stream) {
    for (int64_t off = 0; off < n_work; off += 0x7fffffff) {
        int64_t cnt = n_work - off < 0x7fffffff ? n_work - off : 0x7fffffff;
        hipLaunchKernelGGL(small_lines_kernel<T>, dim3(unsigned(cnt)), dim3(SMALL_LINE_LANES), 0, stream, work + off,
                           lines, terms, X, S);
    }
    return hipGetLastError();
}
template hipError_t launch_small_lines<double>(const SSmallWork*, int64_t, const SLine*, const STerm*, const double*,
                                               double*, hipStream_t);
template hipError_t launch_small_lines<float>(const SSmallWork*, int64_t, const SLine*, const STerm*, const float*,
                                              float*, hipStream_t);

hipError_t launch_term_grad(const TermGradWork* work, int64_t n_work, const SLine* lines, const STerm* terms,
                            const uint32_t* src, const double* beta, const double* Y, const double* T, double* grad,
                            hipStream_t stream) {
    for (int64_t off = 0; off < n_work; off += 0x7fffffff) {
        const int64_t cnt = n_work - off < 0x7fffffff ? n_work - off : 0x7fffffff;
        hipLaunchKernelGGL(term_grad_kernel, dim3(unsigned(cnt)), dim3(TERM_GRAD_THREADS), 0, stream, work + off, lines,
                           terms, src, beta, Y, T, grad);
    }
    return hipGetLastError();
}

hipError_t launch_convert(const double* src, float* dst, uint64_t n, hipStream_t stream) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL((convert_kernel<double, float>), dim3(grid_for(n, 256)), dim3(256), 0, stream, src, dst, n);
    return hipGetLastError();
}

hipError_t launch_fill(double* p, uint64_t n, double v, hipStream_t stream) {
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(fill_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream, p, n, v);
    return hipGetLastError();
}

hipError_t launch_copy_jobs(const CopyJob* jobs, int32_t n_jobs, const double* src, double* dst, hipStream_t stream) {
    if (n_jobs <= 0) return hipSuccess;
    hipLaunchKernelGGL(copy_jobs_kernel, dim3(unsigned(n_jobs), 16), dim3(256), 0, stream, jobs, src, dst);
    return hipGetLastError();
}

hipError_t launch_reshape(const ReshapeSeg* segs, int32_t n_segs, const double* src, double* dst, int to_left,
                          hipStream_t stream) {
    if (n_segs <= 0) return hipSuccess;
    hipLaunchKernelGGL(reshape_kernel, dim3(unsigned(n_segs), 8), dim3(256), 0, stream, segs, src, dst, to_left);
    return hipGetLastError();
}

hipError_t launch_dot(const double* x, const double* y, uint64_t n, double* work, double* out, hipStream_t stream) {
    hipLaunchKernelGGL(dot_partial_kernel, dim3(DOT_BLOCKS), dim3(DOT_THREADS), 0, stream, x, y, n, work);
    hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(DOT_THREADS), 0, stream, work, DOT_BLOCKS, out);
    return hipGetLastError();
}

hipError_t launch_axpy_dev(double* y, const double* x, uint64_t n, const double* num, const double* den, double sign,
                           hipStream_t stream) {
    hipLaunchKernelGGL(axpy_dev_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream, y, x, n, num, den, sign);
    return hipGetLastError();
}

hipError_t launch_seg_dot(const double* x, const double* y, const int64_t* off, int nseg, double* part, double* out,
                          hipStream_t stream) {
    if (nseg <= 0) return hipSuccess;
    hipLaunchKernelGGL(seg_dot_partial_kernel, dim3(SEG_CHUNKS, unsigned(nseg)), dim3(DOT_THREADS), 0, stream, x, y,
                       off, part);
    hipLaunchKernelGGL(seg_dot_final_kernel, dim3(unsigned((nseg + 255) / 256)), dim3(256), 0, stream, part, nseg, out);
    return hipGetLastError();
}

hipError_t launch_seg_axpby(double* y, const double* x, const int64_t* off, int nseg, const double* a, const double* b,
                            hipStream_t stream) {
    if (nseg <= 0) return hipSuccess;
    hipLaunchKernelGGL(seg_axpby_kernel, dim3(SEG_CHUNKS, unsigned(nseg)), dim3(256), 0, stream, y, x, off, a, b);
    return hipGetLastError();
}

// Search space of mq_davidson_noalloc: one copy per GPU, allocated with the code object and held
// until the process ends.  Host code passes its device address (noalloc_scratch_address), never
// the symbol itself.
static __device__ __align__(256) double noalloc_scratch[MQ_NOALLOC_SCRATCH_ELEMS];

hipError_t noalloc_scratch_address(void** ptr) { return hipGetSymbolAddress(ptr, HIP_SYMBOL(noalloc_scratch)); }

hipError_t launch_axpby(double* y, const double* x, uint64_t n, double a, double b, hipStream_t stream) {
    hipLaunchKernelGGL(axpby_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream, y, x, n, a, b);
    return hipGetLastError();
}

hipError_t launch_scale_rsqrt(double* x, uint64_t n, const double* nrm2, hipStream_t stream) {
    hipLaunchKernelGGL(scale_rsqrt_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream, x, n, nrm2);
    return hipGetLastError();
}

}  // namespace mq
