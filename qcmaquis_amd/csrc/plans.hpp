// Host-built work lists of the three contraction kernels (H*psi, left growth, right growth).
//
// Each contraction has the reference's three stages (solver/tasks.cpp):
//   1. T-GEMMs:   T = psi_slice * R_cohort  (H*psi, right step)   or  L_b * psi_slice (left step)
//   2. S-assembly: S(tile) = sum_k alpha_k * T(tile_k)   -- the MPO-term sum
//   3. output GEMMs: psi' = L_panel * S  |  L' = A_bra^T * S  |  R'_b = S_b * B_bra^T
// Here all three stages are flattened into device tables: a list of GEMM problems per stage and a
// list of S "lines" (one output tile each) with their (alpha, T offset) terms.  The loops that
// generate alpha follow the reference's schedule builders term by term, so the S tiles are summed
// in the reference's order.
#pragma once

#include <cstdint>
#include <memory>
#include <type_traits>
#include <utility>
#include <vector>

#include "core.hpp"

namespace mq {

// Host table whose resize leaves new elements uninitialised: the big tables are written in full
// right after they are sized, in parallel, so no serial zero-fill (and no first touch by one
// thread) is paid.
template <class T>
struct DefaultInitAlloc : std::allocator<T> {
    template <class U>
    struct rebind {
        using other = DefaultInitAlloc<U>;
    };
    DefaultInitAlloc() = default;
    template <class U>
    DefaultInitAlloc(DefaultInitAlloc<U> const&) noexcept {}
    template <class U>
    void construct(U* p) noexcept(std::is_nothrow_default_constructible<U>::value) {
        ::new (static_cast<void*>(p)) U;
    }
    template <class U, class... A>
    void construct(U* p, A&&... a) {
        ::new (static_cast<void*>(p)) U(std::forward<A>(a)...);
    }
};
template <class T>
using HostTable = std::vector<T, DefaultInitAlloc<T>>;


// One GEMM problem: C = op(A) * op(B), column-major, optionally batched with element strides.
// Address fields hold an element offset into the role's base pointer given at launch.
enum : int32_t {
    GEMM_TRANS_A = 1,
    GEMM_TRANS_B = 2,
    GEMM_ROWMAP = 4,  // stacked problem: rows from a row table (A not transposed, never split along K)
    GEMM_NBLOCKS = 8, // columns in blocks of nb (B transposed): column n of B at (n / nb) sb + n % nb
};
enum : int32_t {  // operand base selectors
    BASE_PSI_IN = 0, BASE_PSI_OUT, BASE_T, BASE_S, BASE_LPANEL, BASE_BOUNDARY, BASE_BRA, BASE_KET,
    BASE_NEW, BASE_COUNT
};
struct GemmDesc {
    int64_t a, b, c;        // element offsets
    int64_t sa, sb, sc;     // batch strides (elements)
    int32_t M, N, K, batch;
    int32_t lda, ldb, ldc;
    int32_t flags;          // GEMM_TRANS_*
    int32_t base_a, base_b, base_c;
    int32_t nb;             // GEMM_NBLOCKS: columns of a block
};
static_assert(sizeof(GemmDesc) == 96, "GemmDesc layout");

// The stacked problems of a stage with their batch folded into the columns, for the device: T tasks
// that read a right boundary transposed are one product per block of the cohort (nb of them, N
// columns each, N often far below a tile's width), whose C columns follow each other; folded, a
// tile takes columns of as many blocks as it holds (GEMM_NBLOCKS).  Other problems are returned as
// they are.
std::vector<GemmDesc> fold_batches(std::vector<GemmDesc> const& v);

// Row of a stacked problem (GEMM_ROWMAP).  Several products that share their B operand (T-GEMMs
// reading one right-boundary cohort) run as one problem whose M rows are the rows of their A
// operands.  Row m of problem g is entry g.a + m of the row table: it reads A at element
// a + k * ld of base_a and writes C at element c + (n + batch * g.sc) * ld of base_c (g.sc counts
// columns for these problems; g.lda, g.ldc and g.sa are unused).
struct GemmRow {
    int64_t a, c;
    int32_t ld, pad;
};
static_assert(sizeof(GemmRow) == 24, "GemmRow layout");

// S-assembly output tile (rows x cols at s_off with leading dimension lds) and its term range;
// flags: SLINE_SMALL = summed by the small-tile term sum, not in a 16-line block.
constexpr int32_t SLINE_SMALL = 1;
struct SLine {
    int64_t s_off;
    int32_t lds, rows, cols, t0;
    int32_t t1, flags;
};
static_assert(sizeof(SLine) == 32, "SLine layout");
struct STerm {
    double alpha;
    int64_t t_off;  // element offset of a contiguous rows x cols tile in the T buffer
};

// Block form of the MPO-term sum for the matrix cores.  Lines of equal tile shape are grouped in
// blocks of up to SBLOCK_LINES, SBLOCK_GROUPS groups of 16.  A block stores the union of the T
// tiles its lines read, ordered by the set of groups that read each tile (then by T offset) and cut
// into k-steps of 4 tile slots (the last padded with empty slots, offset -1); utile holds the 4
// slots of k-step k of the block at 4 (k_off + k).  For every k-step, each group that reads one
// of its tiles has a 16 x 4 coefficient sub-block (64 values, [slot t][line i] at 16 t + i: alpha of
// line i for that tile, zero where the line does not read it, summed where it reads it twice);
// the sub-blocks of a block are stored in k-step order, groups ascending, from ualpha[64 a_off].
// kstep word of k-step k: bits 0..7 = the groups with a sub-block, bits 8..31 = its first sub-block
// relative to a_off.  Group g of the block's S tiles is then Y_g = sum over k-steps of
// alpha_g,k * X_k with X_k the 4 x E matrix of the step's tile elements: a group does matrix-core
// work only on the k-steps whose tiles it reads, while the tiles are read once per block.
constexpr int SBLOCK_GROUP = 16;
constexpr int SBLOCK_GROUPS = 4;
constexpr int SBLOCK_LINES = SBLOCK_GROUP * SBLOCK_GROUPS;
static_assert(SBLOCK_GROUPS <= 8, "k-step group masks are 8 bits");
struct SBlock {
    int64_t a_off;            // first coefficient sub-block (64 values each)
    int32_t k_off, nk, na;    // first k-step (kstep index; utile from 4 k_off), k-steps, sub-blocks
    int32_t E, rows;          // tile elements (rows x cols), tile rows
    int32_t nlines, line0;    // lines in the block, first entry of lsoff / llds
    int32_t pad;
};
static_assert(sizeof(SBlock) == 40, "SBlock layout");
struct SWork {
    int32_t blk, n0;          // block and first tile element of one work item
};
// Work items by the waves that share one: tiles of more than 64 elements on the four waves of a
// workgroup, of 33 to 64 on two, of at most 32 on one; the work list holds them in this order.  The
// launch list has one entry per workgroup: a team's work item itself, or for workgroups of smaller
// items (blk < 0) the first of its items (work[n0]) with -blk = 1 (one wave each) or 2, or 3 or 4
// where it runs this item alone, of one wave or of two, its k-steps shared out (SB_SHARE).
struct SWorkCounts {
    int32_t team = 0, pair = 0, solo = 0;
};
constexpr int SB_WAVES = 4;  // waves of a term-sum workgroup
// An item of one or two waves with at least this many k-steps has a workgroup to itself, its k-steps in
// equal shares for four waves or two pairs (launch entry -2 - waves): the longest lists, several
// hundred k-steps, are otherwise the last to end.  18 orbitals and M = 128, all tiles in blocks, term
// sum in us from 9999 / 64 / 32 / 16 k-steps: 299 / 252 / 255 / 303; 12 and M = 96 91 / 65 / 67 / 71;
// 18 and M = 509, where other work hides the long lists, 819 / 818 / 834 / 857
constexpr int SB_SHARE = 64;
// Lines marked SLINE_SMALL (tiles of at most SMALL_LINE_LANES elements) are summed term by term:
// each line gets a power-of-two group of lanes, one lane per tile element, and as many such groups,
// each with a share of the terms, as leave a lane SMALL_LINE_DEPTH terms (up to a workgroup's lanes).
// A work item is the consecutive lines of one kind that a workgroup of 256 lanes holds.
struct SSmallWork {
    int32_t line0, n;         // first line (small line table) and number of lines
    int32_t lg, ts;           // log2 of the lanes per tile (one an element) and of the shares of its terms
};
struct SBlockTable {
    std::vector<SBlock> blocks;
    std::vector<SWork> work;
    SWorkCounts n_work;           // the work items by team size
    std::vector<SWork> launch;    // one entry per workgroup
    HostTable<int64_t> utile;     // T element offset of each union tile slot (-1: empty slot)
    HostTable<uint32_t> kstep;    // k-step words
    HostTable<double> ualpha;     // coefficient sub-blocks
    std::vector<int64_t> lsoff;   // S offset of each line (SBLOCK_LINES entries per block)
    std::vector<int32_t> llds;    // its leading dimension
    uint64_t gathered = 0;        // sum over blocks of union tiles * E (T elements read)
    uint64_t max_union = 0;       // largest union of one block (tiles)
    uint64_t mac = 0;             // matrix-core multiply-adds: 64 * E per sub-block
    // small-tile lines: their own line and term tables (t0 / t1 index small_terms)
    std::vector<SLine> small_lines;
    HostTable<STerm> small_terms;
    std::vector<SSmallWork> small_work;
    uint64_t small_gathered = 0;  // sum over small lines of terms * tile elements
};
// Work item of the MPO-term adjoint: the terms [t0, t1) of one S line, 2^lg lanes per term (one
// dot product of the line's tile of Y = L_panel^T psi with the term's T tile each)
struct TermGradWork {
    int32_t line, t0, t1, lg;
};
constexpr int TERM_GRAD_THREADS = 256;
constexpr int32_t TERM_GRAD_RUN = 256;  // terms per work item at most
// the GEMMs Y = L_panel^T psi of the L*S products psi' = L_panel S (Y written where S is read)
std::vector<GemmDesc> adjoint_y_gemms(std::vector<GemmDesc> const& c_gemms);
// work items of the lines [l0, l1): runs of at most TERM_GRAD_RUN terms, 2^lg >= tile elements
// lanes per term (at most 64)
std::vector<TermGradWork> term_grad_work(HostTable<SLine> const& lines, size_t l0, size_t l1);
// lanes of a workgroup of the small-tile term sum; tiles up to this many elements can go there
constexpr int SMALL_LINE_LANES = 256;
constexpr int SMALL_LINE_DEPTH = 4;  // terms a lane sums before a line gets twice the lanes
// work items cover SBLOCK_ELEMS consecutive tile elements of one block
constexpr int SBLOCK_ELEMS = 128;
// the block term sum loads one element past a tile of odd size: T buffers are that much longer
constexpr int SB_T_SPARE = 2;

// Execution schedule of a grouped GEMM stage.  Output tiles are 128 columns wide and 32, 64, 96 or 128
// rows tall: a problem's rows are cut into the fewest tiles of at most 128 rows, of about equal
// height.  When the stage has too few tiles to fill the device, long reductions are split along K:
// each split tile writes its partial BM x BN tile (column-major, ld BM) into a workspace and a
// reduce job adds the partials in split order into C, so the result does not depend on scheduling.
enum GemmShape { GEMM_32 = 0, GEMM_64, GEMM_96, GEMM_128, GEMM_N_SHAPES };
constexpr int gemm_bm(int shape) { return 32 * (shape + 1); }
constexpr int gemm_bn(int) { return 128; }
struct GemmTile {
    int32_t prob, batch, tm, tn;
    int32_t k0, k1;   // reduction range of this tile
    int64_t ws;       // < 0: the tile writes C; else element offset of its partial in the workspace
};
static_assert(sizeof(GemmTile) == 32, "GemmTile layout");
struct GemmReduce {
    int32_t prob, batch, tm, tn;
    int32_t nsplit, shape;
    int64_t ws;       // first partial; partial s at ws + s * BM * BN
};
static_assert(sizeof(GemmReduce) == 32, "GemmReduce layout");
struct GemmSchedule {
    std::vector<GemmTile> tiles[GEMM_N_SHAPES];
    std::vector<GemmReduce> reduces;
    uint64_t ws_elems = 0;
    uint64_t n_tiles() const {
        uint64_t n = 0;
        for (auto const& t : tiles) n += t.size();
        return n;
    }
};
// The choices of a grouped GEMM schedule that the tile autotuner varies.  target_items: workgroups
// a stage should provide before K is split; min_chunk: shortest K range of a split tile (a multiple
// of the K step 16).  L*S stages in us at targets
// of 2048 / 4096: 18 orbitals and M = 509 376 / 400, 20 with spins and M = 700 865 / 901 (with a slower split sum), M = 2048
// 15.5 / 15.1 ms (17.1 at 1024); the shorter ranges of 4096 keep the FP32 rounding down (18 orbitals,
// M = 512: 4.3e-7 at 2048, 3.5e-7 at 4096)
struct GemmPolicy {
    int64_t target_items = 4096;
    int32_t min_chunk = 256;
};
constexpr int GEMM_N_POLICIES = 7;
// candidate i of the autotuner (0: the default rule)
GemmPolicy gemm_policy(int i);
GemmSchedule build_gemm_schedule(std::vector<GemmDesc> const& probs, GemmPolicy const& pol);
inline GemmSchedule build_gemm_schedule(std::vector<GemmDesc> const& probs, int64_t target_items = 4096,
                                        int32_t min_chunk = 256) {
    GemmPolicy p;
    p.target_items = target_items;
    p.min_chunk = min_chunk;
    return build_gemm_schedule(probs, p);
}
// the policies whose schedules of a stage differ from each other, the default rule (0) first: stacked
// problems are never split along K, so a stage of them has that one only
struct GemmCandidate {
    int policy;
    GemmSchedule schedule;
};
std::vector<GemmCandidate> gemm_candidates(std::vector<GemmDesc> const& probs);
// Work item of the device's GEMM kernel: rows [m0, m0 + ml), ml <= 128, and up to 128 columns from n0 of
// a problem's C (of batch entry `batch`), reduced over [k0, k1); ws < 0: written to C, else the
// partial tile at element ws of the workspace with leading dimension bm.
struct GemmItem {
    int32_t prob, batch;
    int32_t m0, ml, n0;
    int32_t k0, k1;
    int32_t bm;
    int64_t ws;
};
static_assert(sizeof(GemmItem) == 40, "GemmItem layout");
// the work items of a schedule, all shapes in one list, the most work first
std::vector<GemmItem> gemm_items(std::vector<GemmDesc> const& probs, GemmSchedule const& sch);
// Key of a stage's (m, n, k) histogram for the autotuner: the flop-weighted means of log2 M,
// log2 N and log2 K (in quarters), the share of flops in problems of at most 32, 64 and 96 rows
// (in eighths), log2 of the output tiles at the default rule, and whether rows come from a row
// table; stages of neighbouring site problems usually share it
uint64_t gemm_stage_key(std::vector<GemmDesc> const& probs);


// block table of a list of S lines (lines without terms become zero tiles)
// lines marked SLINE_SMALL go to the small-tile tables, the others into 16-line blocks
// panel > 0: work items ordered element range by element range over panels of up to that many
// consecutive blocks of one tile shape (0: block by block)
SBlockTable build_sblocks(HostTable<SLine> const& lines, HostTable<STerm> const& terms, int32_t panel = 0);
// small-tile limit of the lines [l0, l1) of one site problem under the automatic rule: 64 when
// their mean tile has at most 16 elements and the plan at most SMALL_TERMS_MAX terms (n_terms; 0:
// those of the lines count), else 0.  Term by term every term fetches its tile; a block reads it once
// for 64 lines, but each has its chain of tables, tiles and matrix cores, some 30 us with few blocks.
// FP64 term sum in us, term by term / in blocks: 8 orbitals and M = 40 (0.2 million terms) 10.5 / 29, 9
// and 60 (0.35) 23 / 40, 12 and 96 (2.2) 97 / 59, 18 and 128 (21) 482 / 253.  The line is on the safe
// side for the blocks: between 0.4 and 5 million terms those win where some tiles have more than 64
// elements and go to blocks anyway (10 and M = 70, 0.76 million, 68 / 45; 11 and 80, 1.2, 94 / 66), and
// the terms where none has (10 and M = 45 23 / 39; 12 and 60, 2.2, 34 / 46; 14 and 50, 5.3, 38 / 54).
// n_terms are those of all problems of a batch, so one of them may be summed in the other form, and
// rounded otherwise, than in a plan of its own
constexpr uint64_t SMALL_TERMS_MAX = 1u << 19;
int32_t auto_small_tile_max(HostTable<SLine> const& lines, size_t l0, size_t l1, uint64_t n_terms = 0);
// marks the lines [l0, l1) whose tiles have 1 .. limit elements SLINE_SMALL (limit <= 256)
void mark_small_lines(HostTable<SLine>& lines, size_t l0, size_t l1, int32_t limit);
void check_sblocks(SBlockTable const& B, uint64_t t_size, uint64_t s_size);

struct FlopStats {
    uint64_t flops_total = 0, flops_gemm = 0, flops_gemm_exec = 0, n_terms = 0;
};

// One block copy job for building L panels: dst(rows x cols) <- src block, optionally transposed.
struct CopyJob {
    int64_t src, dst;       // element offsets (src in boundary arena, dst in panel buffer)
    int32_t rows, cols;     // of the destination block
    int32_t nblocks, trans; // trans: src block is cols x rows
};

// One chunk of an H*psi plan: the output columns of a set of right sectors of the two-site MPS.
// Its T-GEMMs, S lines and L*S GEMMs touch only the T intermediates and S panels of these
// columns, which it addresses from offset 0: the chunks run one after the other on one T and one S
// buffer of the largest chunk's size.  Ranges index the plan's tables.
struct HpsiChunk {
    size_t t_gemm0 = 0, t_gemm1 = 0;   // t_gemms
    size_t t_row0 = 0, t_row1 = 0;     // t_rows
    size_t line0 = 0, line1 = 0;       // lines
    size_t c_gemm0 = 0, c_gemm1 = 0;   // c_gemms
    size_t t_task0 = 0, t_task1 = 0;   // t_gemms_task
    size_t c_coh0 = 0, c_coh1 = 0;     // c_gemms_cohort
    uint64_t t_elems = 0, s_elems = 0;
};

struct HpsiPlanHost {
    MPSLayout mps;
    std::vector<HpsiChunk> chunks;  // empty: one chunk over all tables
    std::vector<GemmDesc> t_gemms, c_gemms;
    std::vector<GemmRow> t_rows;  // row table of the stacked T-GEMMs
    std::vector<GemmDesc> t_gemms_task;  // the same T-GEMMs, one problem per task (reference layout)
    // the L*S products per cohort (per cohort and run of the chunk's columns when the plan has
    // several chunks), to be summed into psi'
    std::vector<GemmDesc> c_gemms_cohort;
    HostTable<SLine> lines;
    HostTable<STerm> terms;
    // with term sources: per S term, the MPO term it comes from and d alpha / d(that term's scale)
    HostTable<uint32_t> term_src;
    HostTable<double> term_beta;
    std::vector<CopyJob> lpanel_jobs;
    uint64_t t_elems = 0, s_elems = 0, lpanel_elems = 0;  // T and S: sums over the chunks
    uint64_t t_buf = 0, s_buf = 0;                          // T and S buffers: the largest chunk's
    uint64_t n_cohorts = 0, n_t_tasks = 0;
    uint64_t bytes_compulsory = 0;
    FlopStats flops;
};

// Boundary-growth plan: new boundary index + device tables
struct GrowPlanHost {
    BoundaryIndex out;      // index of the new boundary (with data_off layout)
    uint64_t out_elems = 0;
    std::vector<GemmDesc> t_gemms, c_gemms;
    std::vector<GemmRow> t_rows;  // row table of stacked T-GEMMs (right step)
    HostTable<SLine> lines;
    HostTable<STerm> terms;
    uint64_t t_elems = 0, s_elems = 0;
    FlopStats flops;
};

// chunk_elems: largest T + S (elements) of one chunk; the right sectors are gathered in index
// order into chunks up to that size (a sector larger than it is a chunk of its own); 0 = one chunk.
// term_sources: also fill term_src / term_beta (the MPO-term adjoint)
HpsiPlanHost build_hpsi_plan(Sym sym, MPO const& mpo, BoundaryIndex const& L, BoundaryIndex const& R,
                             Index const& left_i, Index const& phys_i, Index const& right_i,
                             uint64_t chunk_elems = 0, bool term_sources = false);

GrowPlanHost build_lstep_plan(Sym sym, MPO const& mpo, BoundaryIndex const& L, MPSLayout const& bra,
                              MPSLayout const& ket, bool symmetric);

// Host-side bounds validation of device tables: every operand span of every GEMM problem (and
// every row of a stacked one), S line and T term must lie inside its buffer (sizes indexed by
// BASE_*); throws mq::Error otherwise.
void check_gemms(std::vector<GemmDesc> const& v, const uint64_t* sizes,
                 std::vector<GemmRow> const& rows = std::vector<GemmRow>());
void check_lines(HostTable<SLine> const& lines, HostTable<STerm> const& terms, uint64_t t_size, uint64_t s_size);

GrowPlanHost build_rstep_plan(Sym sym, MPO const& mpo, BoundaryIndex const& R, MPSLayout const& bra,
                              MPSLayout const& ket, bool symmetric);

}  // namespace mq
