// gfx950 kernels of the contraction path.
//
//  * gemm_kernel: grouped, batched FP64 / FP32 GEMM over a host-built list of work items of up to
//    128 rows and 128 columns, stages with few of them split along K; eight wave64s of 16 columns
//    each, operands staged through LDS in K slices of 16 with the next slice prefetched into
//    registers.  Each output tile is owned by one workgroup or, when K is split, by a fixed set of
//    partial tiles summed in order by gemm_reduce_kernel: no atomics.
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

// Grouped GEMM.  A workgroup of eight waves computes one work item: up to 128 rows and 128 columns of a
// problem's C, operands of type TI, computed in TI, output converted to TO, reduced over [k0, k1) and
// written to C or, as a partial tile (type TI), into the workspace (split K).  A wave owns 16 columns
// and all rows of the item, in 16-row steps, so the waves share the work evenly however many rows
// there are; steps of rows outside the item, and k steps of four outside the last slice, are
// skipped.  K slices of 16 go through two LDS buffers (one barrier per slice), the next slice
// prefetched into registers.
//
// Every thread keeps pointers to the operand elements it stages and moves them on by a fixed step
// per slice; rows and columns past the end of C read the last valid one (their products are not
// stored), so only the last, shorter slice needs checks.
//
// Bound: the FP64 matrix cores in stages of large sectors (L*S of 20 orbitals and M = 2048: 48 TFLOP/s of
// useful work, of 71 in a dense product of 8192), the stores of T rows and the latency of an item's
// few K slices elsewhere.  Against 256 threads on 32x128, 64x64, 96x64 and 128x64 tiles, one launch
// per tile shape: B is staged for 128 columns of up to 128 rows instead of 64, waves of an item
// no longer wait for the one with the most row steps, and the items of all heights share one launch
// and one tail.  T / L*S stages in us before -> now: 8 orbitals, M = 40 8 / 23 -> 8 / 20;
// 18, M = 509 323 / 412 -> 307 / 377; 20 with spins, M = 700 997 / 958 -> 912 / 880, M = 2048
// 14.8 / 18.9 -> 13.8 / 15.1 ms.
constexpr int GEMM_TILE = 128, GEMM_KS = 16, GEMM_THREADS = 512;
template <class TI>
struct GemmLds {
    // rows padded so that the stores of a slice whose k runs across lanes meet every bank once
    static constexpr int PAD = 8 / int(sizeof(TI));
    TI A[2][GEMM_KS][GEMM_TILE + PAD];
    TI B[2][GEMM_KS][GEMM_TILE + PAD];
    int64_t row_c[GEMM_TILE];  // stacked problems: C offset and leading dimension of every row
    int32_t row_ld[GEMM_TILE];
};

// the body of gemm_kernel for one orientation of its operands
template <class TI, class TO, bool BF3, bool TA, bool TB>
__device__ __forceinline__ void gemm_tile(GemmLds<TI>& lds, GemmItem const& tile, GemmDesc const& g,
                                          const GemmRow* __restrict__ rows, Bases const& bases, TI* __restrict__ ws) {
    constexpr int KS = GEMM_KS, THREADS = GEMM_THREADS, BT = GEMM_TILE, F = BT / 16;
    constexpr int NE = BT * KS / THREADS;  // elements of each operand staged per thread and K slice
    static_assert(NE * THREADS == BT * KS && THREADS % BT == 0 && THREADS % KS == 0 && THREADS == 64 * F, "K slice geometry");
    static_assert(!BF3 || std::is_same<TI, float>::value, "split-BF16 products: FP32 operands");
    typedef typename Mma<TI>::acc_t acc_t;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fk = lane >> 4;
    const int m0 = tile.m0, n0 = tile.n0;
    const int ml = tile.ml, nl = g.N - n0 < BT ? g.N - n0 : BT;  // rows and columns of the item
    const bool rmap = !TA && (g.flags & GEMM_ROWMAP);
    const TI* A = static_cast<const TI*>(bases.p[g.base_a]) + (rmap ? 0 : g.a + int64_t(tile.batch) * g.sa);
    const TI* B = static_cast<const TI*>(bases.p[g.base_b]) + g.b + int64_t(tile.batch) * g.sb;

    // element i of this thread in a slice: the contiguous dimension of the operand runs across
    // consecutive threads.  Rows (columns) along threads: all of one row, DK apart in k, so one
    // pointer walks through them.  k along threads: all of one k, a pointer per row, DM apart.
    constexpr int DK = THREADS / BT, DM = THREADS / KS;
    auto a_m = [&](int i) { return TA ? tid / KS + DM * i : tid % BT; };
    auto a_k = [&](int i) { return TA ? tid % KS : tid / BT + DK * i; };
    auto b_n = [&](int i) { return TB ? tid % BT : tid / KS + DM * i; };
    auto b_k = [&](int i) { return TB ? tid / BT + DK * i : tid % KS; };
    const TI *pa[TA ? NE : 1], *pb[TB ? 1 : NE];
    int64_t a_step = 0, b_step;  // per element of a walk, else per slice
#pragma unroll
    for (int i = 0; i < (TA ? NE : 1); ++i) {
        const int m = m0 + (a_m(i) < ml ? a_m(i) : ml - 1);
        const int64_t k = tile.k0 + a_k(i);
        if (rmap) {
            const GemmRow r = rows[g.a + m];
            pa[i] = A + r.a + k * r.ld;
            a_step = int64_t(DK) * r.ld;
            if (tid < BT) {
                lds.row_c[tid] = r.c;
                lds.row_ld[tid] = r.ld;
            }
        } else {
            pa[i] = TA ? A + int64_t(m) * g.lda + k : A + m + k * g.lda;
            a_step = TA ? KS : int64_t(DK) * g.lda;
        }
    }
#pragma unroll
    for (int i = 0; i < (TB ? 1 : NE); ++i) {
        const int n = n0 + (b_n(i) < nl ? b_n(i) : nl - 1);
        const int64_t k = tile.k0 + b_k(i);
        if (TB)  // columns in blocks of g.nb, a block every g.sb elements
            pb[i] = (g.flags & GEMM_NBLOCKS ? B + int64_t(n / g.nb) * g.sb + n % g.nb : B + n) + k * g.ldb;
        else
            pb[i] = B + k + int64_t(n) * g.ldb;
    }
    b_step = TB ? int64_t(DK) * g.ldb : KS;
    TI ra[NE], rb[NE];
    auto load = [&](int kn) {  // the next kn <= KS values of k
        const bool whole = kn >= KS;
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const TI*& p = pa[TA ? i : 0];
            ra[i] = whole ? *p : ld_or_zero(p, a_k(i) < kn);
            p += a_step;
        }
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const TI*& p = pb[TB ? 0 : i];
            rb[i] = whole ? *p : ld_or_zero(p, b_k(i) < kn);
            p += b_step;
        }
    };

    acc_t acc[F];
#pragma unroll
    for (int i = 0; i < F; ++i) acc[i] = acc_t{0, 0, 0, 0};
    const int fm = (ml + 15) / 16;  // row steps of the item
    const int wc = 16 * wave;       // first column of this wave
    // one slice: S row steps, of which the first fm count unless ALL do.  Operands swapped in every
    // step: the instruction accumulates the transposed tile C^T = B^T A^T
    auto multiply = [&](int buf, int kn, auto steps, auto all) {
        constexpr int S = decltype(steps)::value;
        constexpr bool ALL = decltype(all)::value;
        if constexpr (BF3) {
            bf16x4_t bh, bl;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                short h, l;
                split_bf16(lds.B[buf][4 * fk + q][wc + fr], h, l);
                bh[q] = h;
                bl[q] = l;
            }
#pragma unroll
            for (int i = 0; i < S; ++i) {
                if (!ALL && i >= fm) break;
                bf16x4_t ah, al;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    short h, l;
                    split_bf16(lds.A[buf][4 * fk + q][16 * i + fr], h, l);
                    ah[q] = h;
                    al[q] = l;
                }
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bh, ah, acc[i], 0, 0, 0);
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bh, al, acc[i], 0, 0, 0);
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bl, ah, acc[i], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int kk = 0; kk < KS; kk += 4) {
                if (kk < kn) {
                    TI af[S], bf = lds.B[buf][kk + fk][wc + fr];
#pragma unroll
                    for (int i = 0; i < S; ++i) af[i] = lds.A[buf][kk + fk][16 * i + fr];
#pragma unroll
                    for (int i = 0; i < S; ++i)
                        if (ALL || i < fm) acc[i] = Mma<TI>::step(bf, af[i], acc[i]);
                }
            }
        }
    };
    auto reduce = [&](auto steps, auto all) {
        int left = tile.k1 - tile.k0;
        if (left > 0) load(left);
        for (int buf = 0; left > 0; buf ^= 1, left -= KS) {
#pragma unroll
            for (int i = 0; i < NE; ++i) lds.A[buf][a_k(i)][a_m(i)] = ra[i];
#pragma unroll
            for (int i = 0; i < NE; ++i) lds.B[buf][b_k(i)][b_n(i)] = rb[i];
            __syncthreads();
            if (left > KS) load(left - KS);
            if (wc < nl) multiply(buf, left, steps, all);
        }
    };
    if (tile.k1 <= tile.k0) __syncthreads();  // no slice: the row table still has to reach the other waves
    if (fm == F) reduce(std::integral_constant<int, F>(), std::true_type());
    else if (fm > 4) reduce(std::integral_constant<int, F>(), std::false_type());
    else if (fm > 2) reduce(std::integral_constant<int, 4>(), std::false_type());
    else reduce(std::integral_constant<int, 2>(), std::false_type());

    // D = C^T: register r of lane l holds C[l % 16][row(l, r)] of its 16 x 16 tile, so
    // consecutive lanes store consecutive rows of a column
    if (wc >= nl) return;
    TO* C = static_cast<TO*>(bases.p[g.base_c]) + (rmap ? 0 : g.c + int64_t(tile.batch) * g.sc);
    const bool split = tile.ws >= 0;  // never for stacked problems
#pragma unroll
    for (int i = 0; i < F; ++i) {
        const int mm = 16 * i + fr, m = m0 + mm;
        if (mm >= ml) continue;
        // column n of this row at c_row + n * c_ld
        TO* c_row = C + m;
        int64_t c_ld = g.ldc;
        if (rmap) {
            c_ld = lds.row_ld[mm];
            c_row = C + lds.row_c[mm] + int64_t(tile.batch) * g.sc * c_ld;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int nn = wc + Mma<TI>::row(lane, r);
            if (nn >= nl) continue;
            if (split) ws[tile.ws + mm + int64_t(nn) * tile.bm] = acc[i][r];
            else c_row[int64_t(n0 + nn) * c_ld] = TO(acc[i][r]);
        }
    }
}

// A is transposed in FP64 only (boundary growth, the MPO-term adjoint), and never both operands
template <class TI, class TO, bool BF3 = false>
__global__ __launch_bounds__(GEMM_THREADS, 4) void gemm_kernel(const GemmDesc* __restrict__ probs,
                                                               const GemmRow* __restrict__ rows,
                                                               const GemmItem* __restrict__ items, Bases bases,
                                                               TI* __restrict__ ws) {
    __shared__ GemmLds<TI> lds;
    const GemmItem tile = items[blockIdx.x];
    const GemmDesc g = probs[tile.prob];
    constexpr bool F64 = std::is_same<TI, double>::value;
    if (g.flags & GEMM_TRANS_B) gemm_tile<TI, TO, BF3, false, true>(lds, tile, g, rows, bases, ws);
    else if (F64 && (g.flags & GEMM_TRANS_A)) gemm_tile<TI, TO, BF3, F64, false>(lds, tile, g, rows, bases, ws);
    else gemm_tile<TI, TO, BF3, false, false>(lds, tile, g, rows, bases, ws);
}

// C tile = sum of its split partials, added in split order; blockIdx.y selects 256 elements of the tile.
// Bound: the latency of the partials' loads, so REDUCE_U of them are in flight ahead of their sums.  L*S
// stages in us with 1 / 4 / 8 / 16: 14 orbitals, M = 256 96 / 85 / 85 / 87, 18 and M = 509 401 / 384 / 377 /
// 379, 18 and M = 128 56 / 49 / 48 / 51
constexpr int REDUCE_U = 8;
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
            const TW* p = ws + job.ws + idx;
            int s = 0;
            for (; s + REDUCE_U <= job.nsplit; s += REDUCE_U) {
                TW v[REDUCE_U];
#pragma unroll
                for (int u = 0; u < REDUCE_U; ++u) v[u] = p[(s + u) * tile_elems];
#pragma unroll
                for (int u = 0; u < REDUCE_U; ++u) sum += v[u];
            }
            for (; s < job.nsplit; ++s) sum += p[s * tile_elems];
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
// every wave stages its own block's tables and runs without barriers.  A block of at most 64 elements
// with many k-steps (SB_SHARE) has them shared out over the workgroup, the sums meeting in LDS.
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

// element e of every second line of a block from line i0 on, summed over the tiles that the line reads
template <class T>
__device__ inline void sum_read_tiles(SBlock const& b, int e, int i0, const int64_t* utile, const uint32_t* kw,
                                      const T* ualpha, const int64_t* so, const int32_t* ld, const T* X, T* S) {
    if (e >= b.E) return;
    for (int i = i0; i < b.nlines; i += 2) {
        const int g = i / SBLOCK_GROUP;
        T sum = T(0);
        for (int k = 0; k < b.nk; ++k) {
            const uint32_t word = kw[k];
            if (!((word >> g) & 1u)) continue;
            const T* a = ualpha + 64 * int64_t((word >> 8) + uint32_t(__popc(word & ((1u << g) - 1)))) + i % SBLOCK_GROUP;
            for (int t = 0; t < 4; ++t) {
                const int64_t o = utile[4 * k + t];
                const T at = a[SBLOCK_GROUP * t];
                if (o >= 0 && at != T(0)) sum += at * X[o + e];
            }
        }
        S[so[i] + e % b.rows + int64_t(e / b.rows) * ld[i]] = sum;
    }
}

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
    int sub = wave;              // this wave's slice of its work item
    int part = 0, parts = 1;     // its share of the k-steps
    if (!team) {                 // item work[w.n0] and, unless its k-steps are shared, the next ones
        const bool shared = w.blk < -2;
        const int lw = (-w.blk - 1) & 1, wi = w.n0 + (shared ? 0 : wave >> lw);
        sub = wave & lw;
        if (shared) {
            part = wave >> lw;
            parts = SB_WAVES >> lw;
        }
        if (wi >= (lw ? n.team + n.pair : n.team + n.pair + n.solo)) return;
        w = work[wi];
    }
    const SBlock b = blocks[w.blk];
    const int k0 = b.nk * part / parts, k1 = b.nk * (part + 1) / parts;
    const int n0 = w.n0 + 16 * SB_NC * sub;
    // a wave past the tile end loads and stores no tile but takes part in its team's barriers
    const bool active = n0 < b.E;
    if (!team && !active) return;  // never where k-steps are shared: those tiles fill their waves
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
    for (int c0 = k0; c0 < k1;) {
        // the next k-steps whose tables fit: lane l looks at k-step c0 + l
        const int kl = c0 + lane;
        const uint32_t word = kl < k1 ? kw[kl] : 0;
        const int a0 = __builtin_amdgcn_readfirstlane(int(word >> 8));
        const int end = kl + 1 < b.nk ? int(kw[kl + 1] >> 8) : b.na;
        const int cn = __builtin_popcountll(__ballot(kl < k1 && lane < cap_k && end - a0 <= cap_sub));
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
    if (k0 == k1) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (team) __syncthreads();
    }
    // shared k-steps: the upper half of the parts hands its sums to the lower half until one is left
    for (int h = parts / 2; h > 0; h /= 2) {
        constexpr int NV = SBLOCK_GROUPS * SB_NC * 4;
        static_assert(SB_WAVES / 2 * NV <= SB_SUB, "the sums of half the waves fit the coefficient buffer");
        T* p = s_alpha + 64 * NV * ((part % h) * (SB_WAVES / parts) + sub) + lane;
        __syncthreads();
        if (part >= h && part < 2 * h)
#pragma unroll
            for (int g = 0; g < SBLOCK_GROUPS; ++g)
                if (SBLOCK_GROUP * g < b.nlines)
#pragma unroll
                    for (int v = 0; v < SB_NC * 4; ++v) p[64 * (SB_NC * 4 * g + v)] = acc[g][v / 4][v % 4];
        __syncthreads();
        if (part < h)
#pragma unroll
            for (int g = 0; g < SBLOCK_GROUPS; ++g)
                if (SBLOCK_GROUP * g < b.nlines)
#pragma unroll
                    for (int v = 0; v < SB_NC * 4; ++v) acc[g][v / 4][v % 4] += p[64 * (SB_NC * 4 * g + v)];
    }
    if (part > 0) return;
    // Non-finite elements of T: a zero coefficient times one is NaN in every line of its group, also in those
    // that do not read the tile.  Where a sum came out non-finite in the tiles that the term-by-term
    // sum may take instead (at most 64 elements), the lines are summed again over the tiles they read.  A
    // non-finite element shows in every row of its group, so the first row is looked at: at 18 orbitals and
    // M = 128, where all blocks are of such tiles, H*psi takes 324 us with the look and 322 without.
    if (!team) {
        bool odd = false;
#pragma unroll
        for (int g = 0; g < SBLOCK_GROUPS; ++g)
            odd |= (e0 < b.E && !isfinite(acc[g][0][0])) | (e0 + 1 < b.E && !isfinite(acc[g][1][0]));
        if (__any(odd)) {
            sum_read_tiles(b, n0 + (lane & 31), lane >> 5, utile + 4 * int64_t(b.k_off), kw, ualpha + 64 * b.a_off, so, ld, X, S);
            return;
        }
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

// Small-tile MPO-term sum: a work item is up to 256 >> (lg + ts) lines of 2^ts shares of 2^lg lanes
// (tile elements <= 2^lg); lane e of share s sums alpha_k * T[t_off_k + e] over the line's terms
// k = s, s + 2^ts, ..., four at a time, the shares are added by lane exchanges (between waves: through
// LDS), and element e of the line's S tile is written once.  Past its last term a lane of a share reads
// that term again and leaves it out; a line of one share has few terms or a tile of many elements, and
// its last terms are read one by one.
//
// Bound: the chain terms -> tile elements in the few, small problems that come here (most lines have
// one or two terms, the longest hundreds).  One lane per element for all of a line's terms, as
// before, took 24 us for 8 orbitals and M = 40; with a line's terms shared out 10.2.  Where a caller
// sends large problems here the fetches of tiles bound it, and what a lane reads in vain counts: 18
// orbitals and M = 300, tiles up to 256 elements, 1.17 ms; lines in neighbours' order and every line's last
// terms read again 1.26, in the order of their term count 1.19, the last terms one by one 1.16.
template <class T>
__global__ __launch_bounds__(SMALL_LINE_LANES) void small_lines_kernel(const SSmallWork* __restrict__ work,
                                                                       const SLine* __restrict__ lines,
                                                                       const STerm* __restrict__ terms,
                                                                       const T* __restrict__ X, T* __restrict__ S) {
    __shared__ T part[SMALL_LINE_LANES];
    const SSmallWork w = work[blockIdx.x];
    const int W = 1 << (w.lg + w.ts), G = 1 << w.lg;  // lanes of a line, of a share
    const int tid = int(threadIdx.x), li = tid >> (w.lg + w.ts), q = tid & (W - 1), e = q & (G - 1);
    const SLine l = lines[w.line0 + (li < w.n ? li : 0)];
    const bool in = li < w.n && e < l.rows * l.cols;
    T acc = T(0);
    if (in) {
        constexpr int U = SMALL_LINE_DEPTH;
        const int last = l.t1 - 1;
        if (w.ts == 0) {
            int k = l.t0;
            for (; k + U <= l.t1; k += U) {
                STerm t[U];
#pragma unroll
                for (int u = 0; u < U; ++u) t[u] = terms[k + u];
                T x[U];
#pragma unroll
                for (int u = 0; u < U; ++u) x[u] = X[t[u].t_off + e];
#pragma unroll
                for (int u = 0; u < U; ++u) acc += T(t[u].alpha) * x[u];
            }
            for (; k < l.t1; ++k) acc += T(terms[k].alpha) * X[terms[k].t_off + e];
        } else {
            for (int k = l.t0 + (q >> w.lg); k < l.t1; k += U << w.ts) {
                STerm t[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int ku = k + (u << w.ts);
                    t[u] = terms[ku < last ? ku : last];
                }
                T x[U];
#pragma unroll
                for (int u = 0; u < U; ++u) x[u] = X[t[u].t_off + e];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool ok = k + (u << w.ts) <= last;
                    acc += ok ? T(t[u].alpha) * x[u] : T(0);
                }
            }
        }
    }
    for (int off = G; off < (W < 64 ? W : 64); off *= 2) acc += __shfl_xor(acc, off);
    if (W > 64) {
        part[tid] = acc;
        __syncthreads();
        const int step = G > 64 ? G : 64;
        if (q < G)
            for (int off = step; off < W; off += step) acc += part[tid + off];
    }
    if (in && q < G) S[l.s_off + e % l.rows + int64_t(e / l.rows) * l.lds] = acc;
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
    __syncthreads();  // an earlier sum has been read
    if (lane == 0) red[w] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < DOT_THREADS / 64; ++i) r += red[i];
    return r;
}

__device__ inline double dot_share(const double* __restrict__ x, const double* __restrict__ y, uint64_t n) {
    double s = 0.0;
    for (uint64_t i = uint64_t(blockIdx.x) * DOT_THREADS + threadIdx.x; i < n; i += uint64_t(gridDim.x) * DOT_THREADS)
        s += x[i] * y[i];
    return block_sum(s);
}

// the sum of a product's partials (thread 0)
__device__ inline double dot_total(const double* __restrict__ work) {
    double s = 0.0;
    for (int i = threadIdx.x; i < DOT_BLOCKS; i += DOT_THREADS) s += work[i];
    return block_sum(s);
}

__global__ __launch_bounds__(DOT_THREADS) void dot_partial_kernel(const double* __restrict__ x,
                                                                  const double* __restrict__ y, uint64_t n,
                                                                  double* __restrict__ work) {
    const double r = dot_share(x, y, n);
    if (threadIdx.x == 0) work[blockIdx.x] = r;
}

// The solvers' vectors are short (1e4 to 1e6 elements), so their kernels cost their launches: one by one,
// some 340 of 2 to 3 us, and the gaps between them, in eight Jacobi-Davidson iterations of 14 orbitals
// and M = 256.  Products that do not depend on each other share a launch (blockIdx.y: which), a
// Gram-Schmidt step is one kernel, linear combinations are formed in one pass, and results for the host
// go to pinned memory without a copy: the call takes 3.5 ms instead of 4.9 (H*psi 2.7 of them).
__global__ __launch_bounds__(DOT_THREADS) void dots_partial_kernel(VecPairs v, uint64_t n, double* __restrict__ work) {
    const double r = dot_share(v.x[blockIdx.y], v.y[blockIdx.y], n);
    if (threadIdx.x == 0) work[blockIdx.y * DOT_BLOCKS + blockIdx.x] = r;
}

// out[b] = the sum of the partials from work[b * stride]
__global__ __launch_bounds__(DOT_THREADS) void dots_final_kernel(const double* __restrict__ work, int stride,
                                                                 double* __restrict__ out) {
    const double r = dot_total(work + int64_t(blockIdx.x) * stride);
    if (threadIdx.x == 0) out[blockIdx.x] = r;
}

// t -= (v . t) v with the product's partials in `have`, then the partials of next . t into `want` (next
// may be t); every workgroup adds the partials up for itself
__global__ __launch_bounds__(DOT_THREADS) void gram_schmidt_kernel(double* t, const double* __restrict__ v, const double* next,
                                                                   uint64_t n, const double* __restrict__ have,
                                                                   double* __restrict__ want) {
    __shared__ double coef;
    const double total = dot_total(have);
    if (threadIdx.x == 0) coef = -total;
    __syncthreads();
    const double c = coef;
    double s = 0.0;
    for (uint64_t i = uint64_t(blockIdx.x) * DOT_THREADS + threadIdx.x; i < n; i += uint64_t(gridDim.x) * DOT_THREADS) {
        const double x = t[i] + c * v[i];
        t[i] = x;
        s += x * (next == t ? x : next[i]);
    }
    const double r = block_sum(s);
    if (threadIdx.x == 0) want[blockIdx.x] = r;
}

struct VecList {
    const double* p[VEC_MAX];
    double c[VEC_MAX];
};
__global__ void lincomb_kernel(double* out, VecList v, int count, uint64_t n) {
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x) {
        double s = v.c[0] * v.p[0][i];
        for (int j = 1; j < count; ++j) s += v.c[j] * v.p[j][i];
        out[i] = s;
    }
}

__global__ void axpy_dev_kernel(double* __restrict__ y, const double* __restrict__ x, uint64_t n,
                                const double* __restrict__ num, const double* __restrict__ den, double sign) {
    const double coef = sign * num[0] / (den ? den[0] : 1.0);
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
        y[i] += coef * x[i];
}

// Segmented forms for a batch of independent vectors concatenated in one buffer (segment s is
// elements off[s] .. off[s+1]-1; blockIdx.y = segment).  Dots (blockIdx.z = which): SEG_CHUNKS partial
// sums per segment, then one thread per segment adds them in chunk order (deterministic).
__global__ __launch_bounds__(DOT_THREADS) void seg_dots_partial_kernel(VecPairs v, const int64_t* __restrict__ off,
                                                                       double* __restrict__ part) {
    const int seg = blockIdx.y;
    const int64_t a = off[seg], b = off[seg + 1];
    const double *x = v.x[blockIdx.z], *y = v.y[blockIdx.z];
    double s = 0.0;
    for (int64_t i = a + int64_t(blockIdx.x) * DOT_THREADS + threadIdx.x; i < b; i += int64_t(SEG_CHUNKS) * DOT_THREADS)
        s += x[i] * y[i];
    double r = block_sum(s);
    if (threadIdx.x == 0) part[(int64_t(blockIdx.z) * gridDim.y + seg) * SEG_CHUNKS + blockIdx.x] = r;
}

__global__ void seg_dots_final_kernel(const double* __restrict__ part, int n, double* __restrict__ out) {
    const int q = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (q >= n) return;
    double s = 0.0;
    for (int c = 0; c < SEG_CHUNKS; ++c) s += part[int64_t(q) * SEG_CHUNKS + c];
    out[q] = s;
}

// the coefficients of SEG_COEFS consecutive segments travel with the launch
constexpr int SEG_COEFS = 32;
struct SegCoefs {
    double a[SEG_COEFS], b[SEG_COEFS];
};
// segment s: y = a[s]*y + b[s]*x (y not read where a[s] == 0)
__global__ void seg_axpby_kernel(double* y, const double* x, const int64_t* __restrict__ off, SegCoefs k) {
    const int seg = blockIdx.y;
    const int64_t i0 = off[seg], i1 = off[seg + 1];
    const double a = k.a[seg], b = k.b[seg];
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

// launches a list of n workgroups of `threads` threads in pieces: run(first, count).  A launch takes
// fewer than 2^32 threads along x, so the piece depends on the workgroup's size: 8.4 million of 512
// threads, 16.8 million of 256.
template <class F>
void in_pieces(int64_t n, int threads, F&& run) {
    const int64_t most = int64_t(0xffffffffu) / threads;
    for (int64_t off = 0; off < n; off += most) run(off, unsigned(n - off < most ? n - off : most));
}

template <class TI, class TO, bool BF3 = false>
void launch_gemm_t(const GemmDesc* probs, const GemmRow* rows, const GemmItem* items, int64_t n_items,
                   const GemmReduce* reduces, int64_t n_reduces, int32_t reduce_elems, void* ws, Bases bases,
                   hipStream_t stream) {
    TI* w = static_cast<TI*>(ws);
    in_pieces(n_items, GEMM_THREADS, [&](int64_t off, unsigned cnt) {
        hipLaunchKernelGGL((gemm_kernel<TI, TO, BF3>), dim3(cnt), dim3(GEMM_THREADS), 0, stream, probs, rows, items + off,
                           bases, w);
    });
    in_pieces(n_reduces, 256, [&](int64_t off, unsigned cnt) {
        hipLaunchKernelGGL((gemm_reduce_kernel<TI, TO>), dim3(cnt, unsigned((reduce_elems + 255) / 256)), dim3(256), 0,
                           stream, probs, reduces + off, bases, w);
    });
}

}  // namespace

hipError_t launch_gemm(GemmPrec prec, const GemmDesc* probs, const GemmRow* rows, const GemmItem* items, int64_t n_items,
                       const GemmReduce* reduces, int64_t n_reduces, int32_t reduce_elems, void* ws, Bases bases,
                       hipStream_t stream) {
    auto run = [&](auto launch) { launch(probs, rows, items, n_items, reduces, n_reduces, reduce_elems, ws, bases, stream); };
    switch (prec) {
        case GEMM_F64: run(launch_gemm_t<double, double>); break;
        case GEMM_F32: run(launch_gemm_t<float, float>); break;
        case GEMM_F32_OUT_F64: run(launch_gemm_t<float, double>); break;
        case GEMM_BF3: run(launch_gemm_t<float, float, true>); break;
        case GEMM_BF3_OUT_F64: run(launch_gemm_t<float, double, true>); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_slines(const SLine* lines, int64_t n_lines, const STerm* terms, const double* T, double* S,
                         hipStream_t stream) {
    in_pieces(n_lines, 256, [&](int64_t off, unsigned cnt) {
        hipLaunchKernelGGL(sline_kernel, dim3(cnt), dim3(256), 0, stream, lines + off, terms, T, S);
    });
    return hipGetLastError();
}

template <class T>
hipError_t launch_sblocks(const SBlock* blocks, const SWork* launch, int64_t n_launch, const SWork* work, SWorkCounts n,
                          const int64_t* utile, const uint32_t* kstep, const T* ualpha, const int64_t* lsoff,
                          const int32_t* llds, const T* X, T* S, bool xcd_contiguous, hipStream_t stream) {
    in_pieces(n_launch, SB_THREADS, [&](int64_t off, unsigned cnt) {
        hipLaunchKernelGGL(sblock_kernel<T>, dim3(cnt), dim3(SB_THREADS), 0, stream, blocks, launch + off, work, n, utile,
                           kstep, ualpha, lsoff, llds, X, S, int(xcd_contiguous));
    });
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
    in_pieces(n_work, SMALL_LINE_LANES, [&](int64_t off, unsigned cnt) {
        hipLaunchKernelGGL(small_lines_kernel<T>, dim3(cnt), dim3(SMALL_LINE_LANES), 0, stream, work + off, lines, terms, X, S);
    });
    return hipGetLastError();
}
template hipError_t launch_small_lines<double>(const SSmallWork*, int64_t, const SLine*, const STerm*, const double*,
                                               double*, hipStream_t);
template hipError_t launch_small_lines<float>(const SSmallWork*, int64_t, const SLine*, const STerm*, const float*,
                                              float*, hipStream_t);

hipError_t launch_term_grad(const TermGradWork* work, int64_t n_work, const SLine* lines, const STerm* terms,
                            const uint32_t* src, const double* beta, const double* Y, const double* T, double* grad,
                            hipStream_t stream) {
    in_pieces(n_work, TERM_GRAD_THREADS, [&](int64_t off, unsigned cnt) {
        hipLaunchKernelGGL(term_grad_kernel, dim3(cnt), dim3(TERM_GRAD_THREADS), 0, stream, work + off, lines, terms, src,
                           beta, Y, T, grad);
    });
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
    hipLaunchKernelGGL(dots_final_kernel, dim3(1), dim3(DOT_THREADS), 0, stream, work, DOT_BLOCKS, out);
    return hipGetLastError();
}

hipError_t launch_dots(VecPairs const& v, int count, uint64_t n, double* work, double* out, hipStream_t stream) {
    if (count <= 0) return hipSuccess;
    if (count > VEC_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(dots_partial_kernel, dim3(DOT_BLOCKS, unsigned(count)), dim3(DOT_THREADS), 0, stream, v, n, work);
    hipLaunchKernelGGL(dots_final_kernel, dim3(unsigned(count)), dim3(DOT_THREADS), 0, stream, work, DOT_BLOCKS, out);
    return hipGetLastError();
}

hipError_t launch_gram_schmidt(double* t, const double* const* v, int count, uint64_t n, double* work, double* out,
                               hipStream_t stream) {
    if (count <= 0) return hipErrorInvalidValue;
    // partials: t . t before in part 0, the steps' products in 1 and 2 by turns, t . t after in 3
    auto part = [&](int i) { return work + int64_t(i) * DOT_BLOCKS; };
    VecPairs first{};
    first.x[0] = first.y[0] = first.y[1] = t;
    first.x[1] = v[0];
    hipLaunchKernelGGL(dots_partial_kernel, dim3(DOT_BLOCKS, 2), dim3(DOT_THREADS), 0, stream, first, n, work);
    for (int i = 0; i < count; ++i) {
        const bool last = i + 1 == count;
        hipLaunchKernelGGL(gram_schmidt_kernel, dim3(DOT_BLOCKS), dim3(DOT_THREADS), 0, stream, t, v[i],
                           last ? t : v[i + 1], n, part(1 + i % 2), part(last ? 3 : 1 + (i + 1) % 2));
    }
    hipLaunchKernelGGL(dots_final_kernel, dim3(2), dim3(DOT_THREADS), 0, stream, work, 3 * DOT_BLOCKS, out);
    return hipGetLastError();
}

hipError_t launch_lincomb(double* out, const double* const* p, const double* c, int count, uint64_t n, hipStream_t stream) {
    if (count <= 0) return hipErrorInvalidValue;
    for (int j = 0; j < count;) {
        VecList v{};
        int m = 0;
        if (j > 0) {  // the sum so far
            v.p[m] = out;
            v.c[m++] = 1.0;
        }
        for (; j < count && m < VEC_MAX; ++j, ++m) {
            v.p[m] = p[j];
            v.c[m] = c[j];
        }
        hipLaunchKernelGGL(lincomb_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream, out, v, m, n);
    }
    return hipGetLastError();
}

hipError_t launch_axpy_dev(double* y, const double* x, uint64_t n, const double* num, const double* den, double sign,
                           hipStream_t stream) {
    hipLaunchKernelGGL(axpy_dev_kernel, dim3(grid_for(n, 256)), dim3(256), 0, stream, y, x, n, num, den, sign);
    return hipGetLastError();
}

hipError_t launch_seg_dots(VecPairs const& v, int count, const int64_t* off, int nseg, double* part, double* out,
                           hipStream_t stream) {
    if (nseg <= 0 || count <= 0) return hipSuccess;
    if (count > VEC_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(seg_dots_partial_kernel, dim3(SEG_CHUNKS, unsigned(nseg), unsigned(count)), dim3(DOT_THREADS), 0,
                       stream, v, off, part);
    hipLaunchKernelGGL(seg_dots_final_kernel, dim3(unsigned((count * nseg + 255) / 256)), dim3(256), 0, stream, part,
                       count * nseg, out);
    return hipGetLastError();
}

hipError_t launch_seg_axpby(double* y, const double* x, const int64_t* off, int nseg, const double* a, const double* b,
                            hipStream_t stream) {
    for (int s0 = 0; s0 < nseg; s0 += SEG_COEFS) {
        const int m = nseg - s0 < SEG_COEFS ? nseg - s0 : SEG_COEFS;
        SegCoefs k{};
        for (int i = 0; i < m; ++i) {
            k.a[i] = a[s0 + i];
            k.b[i] = b[s0 + i];
        }
        hipLaunchKernelGGL(seg_axpby_kernel, dim3(SEG_CHUNKS, unsigned(m)), dim3(256), 0, stream, y, x, off + s0, k);
    }
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
