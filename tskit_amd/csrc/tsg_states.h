// The state plan: the count states of a tree sequence and the places where
// statistics read them (built once per tree sequence, query-independent).
//
// A *state* is the set of samples below one node over one run of trees.  A
// query's counts of a state are the sums of the counts of at most
// TSG_STATE_IN earlier states, so all states of the whole sequence are
// counted level by level, every state of a level in parallel: the depth is
// that of a few merged tree levels, not the length of the genome.
//   state 0       no samples
//   state 1 + s   sample s alone
//   the others    in levels, each level's inputs in earlier ones
// A branch statistic is a sum over *events*: at an event's position the sum
// over branches of length x summary changes by ev_b x F(counts of ev_state)
// (a branch appearing, disappearing, changing its samples or its length;
// the first tree's branches appear at 0).  A site statistic is a sum over
// *rows*, one allele (or a biallelic site's two) each.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

struct tsg_treeseq;

// inputs per state, padded with state 0 (32 bytes a state: two 16-byte loads)
#define TSG_STATE_IN 8
// events / rows per workgroup of the evaluation kernels
#define TSG_BRANCH_TILE 512
#define TSG_SITE_TILE 256

// Columns up to which a tile holds counts as FP64 (48 KB of LDS at 8 columns:
// three workgroups a CU, which is what their registers allow too): the
// conversion is paid once an event instead of once an output.
#define TSG_STATE_F64_COLUMNS 16

// outputs and threads per workgroup of k_state_finish
#define TSG_FINISH_OUTPUTS 8
#define TSG_FINISH_THREADS 1024

// pieces of a node one thread adds up
#define TSG_NODE_RUN 16

// kinds of a site row
#define TSG_ROW_PAIR 0     // a biallelic site of one mutation: both alleles
#define TSG_ROW_DERIVED 1  // one derived allele of another site
#define TSG_ROW_ANCESTRAL 2

// A branch's contribution to the allele frequency spectrum: the state of a
// node of time tu under a parent of time tp (edge inserted at ins) over
// [from, to).
struct TsgBranchPiece {
    double tu, tp, ins, from, to;
    int32_t state, pad;
};

// Node `node` is in `state` from `from` to its next piece (or the end).
struct TsgNodePiece {
    int32_t node, state;
    double from;
};
// The node pieces by node, and runs of at most TSG_NODE_RUN pieces of one
// node: run r has the pieces piece0[r] .. piece0[r + 1].
struct TsgNodeRuns {
    std::vector<int32_t> node, piece0, state;
    std::vector<double> from;
};

struct TsgStateDevice {
    int device = -1;
    // allocations: the plan, and what node statistics, the allele frequency
    // spectrum and genotypes add on first use
    void *block = nullptr, *nodes_block = nullptr, *afs_block = nullptr, *bits_block = nullptr;
    int32_t *order = nullptr;      // [states] by level (null: the states are numbered so)
    int32_t *in = nullptr;         // [(states - 1 - n) x TSG_STATE_IN], of state 1 + n on
    int32_t *ev_state = nullptr;   // [events]
    double *ev_b = nullptr;
    double *ev_pos = nullptr;
    int32_t *row_ref = nullptr;    // [rows]: state of a pair row, or -1 - list of the others
    double *row_pos = nullptr;
    int32_t *list_off = nullptr;   // [lists + 1] into list_ent
    int32_t *list_kind = nullptr;  // [lists]
    int32_t *list_ent = nullptr;   // state * 2 + (1: subtracted)
    double *btile_pos = nullptr;   // [branch tiles] position of each tile's first event
    double *stile_pos = nullptr;   // [site tiles]
    // node statistics (uploaded on first use)
    int32_t *run_node = nullptr, *run_piece0 = nullptr, *run_state = nullptr;
    double *run_from = nullptr;
    int32_t runs = 0;
    // allele frequency spectrum (uploaded on first use)
    int32_t *row_all = nullptr;
    TsgBranchPiece *pieces = nullptr;
    // genotypes
    int32_t *mut_state = nullptr;
    size_t bytes = 0;
};

struct tsg_stateplan {
    bool usable = false;
    int32_t num_states = 0, num_lists = 0;
    std::vector<int32_t> level0;   // [levels + 1] into order; level 0: states 0 .. n
    std::vector<int32_t> order;    // (empty: the states are numbered by level)
    std::vector<int32_t> in;
    std::vector<int32_t> ev_state;
    std::vector<double> ev_b, ev_pos;
    std::vector<int32_t> row_ref;
    std::vector<double> row_pos;
    std::vector<int32_t> list_off, list_kind, list_ent;
    std::vector<double> btile_pos, stile_pos;
    int32_t btiles = 1, stiles = 1;
    // Node statistics: every node's states along the genome (tsg_node_runs).
    std::vector<TsgNodePiece> node_pieces;
    // Allele frequency spectrum: samples below each row's allele, and the
    // branch pieces as the reference's updates cut them (trees.c:3650-3690, 3738-3770: a node is updated as a node on the
    // path of an edge in or out, and as the child of an edge out; the state
    // and parent are those at the update).  Pieces that cover no sample or
    // all of them count nothing and are left out.
    std::vector<int32_t> row_all;
    std::vector<TsgBranchPiece> pieces;
    // Genotypes: the state of each mutation's node at its site.
    std::vector<int32_t> mut_state;
    TsgStateDevice dev;
};

// --- device side ------------------------------------------------------------
// One output: a summary of the columns c[0..3] (set sizes or, for weights,
// column totals n[]).  Read by scalar loads (one 104-byte record a wave).
struct TsgStateOut {
    int32_t stat;            // tsg_stat_id
    int32_t polarised;
    int32_t c[4];
    int32_t par;             // weighted summaries: offset of their parameters in opar
    int32_t cbase, ccount;   // trait regression: its covariates
    int32_t samples;         // ... and the number of samples
    int32_t run;             // outputs from this one on of the same summary
    int32_t pad;
    double n[4];
    double scale;            // 1 / denominator, twice that where one(x) = one(n - x)
    double coef[2];          // centred relatedness: 1 / n; weighted: its parameters
};

// One query of a run on the state plan.  Its windows' sums come per segment:
// tile t and window w share segment t + w when the tile's events reach into
// the window (a tile's windows run from its first event's to the next tile's
// first event's, so that no segment between them is left out).
struct TsgStateQuery {
    int32_t W, M, mbase;
    uint32_t flags;          // TSG_F_SPAN_NORMALISE
    int32_t branch;          // 1 branch, 0 site
    int32_t new_windows;     // 0: the previous query's, of the same mode
    int32_t tw;              // of its tiles' windows, then its windows' tiles, in tile_w
    int32_t rel_c0, rel_cn;  // columns of the centred relatedness mean (rel_cn 0: none)
    int32_t wbase, bbase;    // workgroups before it: k_state_windows, k_state_finish
    int64_t win_off;         // of its windows
    int64_t pbase, cbase;    // of its segment / window sums
    int64_t obase;           // of its outputs in raw (to_out 0) or out (1)
    int32_t to_out;
    int32_t by_window;       // 1: its segments are added up by k_state_windows first
    int32_t pad;
};

struct TsgStateArgs {
    // plan
    const int32_t *order, *in;
    const int32_t *ev_state;
    const double *ev_b, *ev_pos, *btile_pos;
    const int32_t *row_ref;
    const double *row_pos, *stile_pos;
    const int32_t *list_off, *list_kind, *list_ent;
    int32_t num_states, num_samples, nev, nrow, btiles, stiles;
    // columns: rows of RW 32-bit words a state (16-bit or 32-bit counts, or
    // FP64 sums of weights)
    int32_t K, RW;
    uint32_t *x;
    int32_t npairs;
    const int32_t *pair_sample, *pair_col;
    const double *pair_w;
    const int32_t *col_total;
    const double *col_total_w, *opar;
    // queries, branch mode first: [0, QB) and [QB, Q)
    int32_t QB, Q;
    const TsgStateOut *outs;
    const TsgStateQuery *queries;
    const double *windows;
    // per set of windows: each tile's first event's window (tiles + 1
    // entries), then each window's first tile (W + 1 entries)
    int32_t *tile_w;
    int32_t ntile_w;
    double *partial;         // segment sums
    double *wsum;            // window sums of the by_window queries
    double *raw, *out;
    // host arrays to bring over first (pinned memory; 16-byte words)
    const uint4 *stage_src;
    uint4 *stage_dst;
    int64_t stage_words;
    // composites (TsgFinal), after the sums
    const void *fin;
    int32_t nfin;
    const int32_t *ipar;
    const double *dpar;
    int64_t fincount;
};

// how a run's rows hold a column
#define TSG_ROW_U16 0
#define TSG_ROW_I32 1
#define TSG_ROW_F64 2

// 32-bit words of a row of K columns: 1, 2 or a multiple of 4, so that a row
// is read in whole 4-, 8- or 16-byte loads
inline int tsg_state_row_words(int K, int type) {
    const int w = type == TSG_ROW_U16 ? (K + 1) / 2 : type == TSG_ROW_I32 ? K : 2 * K;
    return w <= 2 ? w : (w + 3) / 4 * 4;
}
// LDS bytes of the evaluation kernels; whether their tiles hold K columns as
// FP64 (TSG_STATE_F64_COLUMNS) or as the rows' counts
size_t tsg_state_shmem(int K, int type, bool branch);

struct TsgStateLaunch {
    TsgStateArgs a;
    int type = 0;
    const int32_t *level0 = nullptr;  // host
    int levels = 0;                   // level 0 included
    int wgroups = 0, fgroups = 0;     // workgroups of k_state_windows, k_state_finish
};

// Node statistics of query 0 on the counts of a run.
struct TsgNodeArgs {
    const int32_t *run_node, *run_piece0, *run_state;
    const double *run_from;
    int32_t runs;
    int64_t num_nodes;
    double length;
    double *res;             // [W x nodes x M], zero
};
// The allele frequency spectrum on the counts of a run (columns: the sets).
#define TSG_SPECTRUM_SETS 16
struct TsgSpectrumArgs {
    const int32_t *row_all;
    const TsgBranchPiece *pieces;
    int32_t npieces, polarised, W, TW;
    const double *windows, *time_windows;
    const int64_t *dims;     // set sizes + 1
    int64_t size;            // product of dims
    unsigned long long *hist_u;  // site: [W x size] half-units, zero
    double *hist_d;              // branch: [W x TW x size], zero
};
// The counts alone (begin: recorded after the host arrays are over).
hipError_t tsg_launch_state_counts(const TsgStateLaunch &r, hipEvent_t begin, hipStream_t s);
// The levels from 1 on, of rows whose level 0 is there (16- or 32-bit words).
hipError_t tsg_launch_state_levels(const TsgStateLaunch &r, hipStream_t s);
hipError_t tsg_launch_state_nodes(const TsgStateLaunch &r, const TsgNodeArgs &g, int M,
                                  hipStream_t s);
hipError_t tsg_launch_spectrum(const TsgStateLaunch &r, const TsgSpectrumArgs &g, bool branch,
                               hipStream_t s);

// One run: counts, then (begin / mid / end: recorded around the branch and
// site evaluations where not null) evaluation, window sums, composites.
hipError_t tsg_launch_states(const TsgStateLaunch &r, hipEvent_t begin, hipEvent_t mid,
                             hipEvent_t end, hipStream_t s);
// Many runs of one row type, all of up to TSG_STATE_F64_COLUMNS columns or all
// of more, one launch per phase: their arguments in device
// memory, in the order of `runs`, and the block prefixes of the phases
// (tsg_state_prefixes; -1: too many for one launch) on the host and in device
// memory.
int tsg_state_prefixes(const TsgStateLaunch *runs, int nrun, std::vector<int32_t> &pre);
hipError_t tsg_launch_states_multi(const TsgStateLaunch *runs, const TsgStateArgs *args, int nrun,
                                   const std::vector<int32_t> &pre_h, const int32_t *pre,
                                   hipStream_t s);

// Builds ts->states (tsg_states.cpp); not usable where it would be out of
// proportion to the edges (see there).
int tsg_build_states(tsg_treeseq *ts);
void tsg_node_runs(const tsg_treeseq *ts, TsgNodeRuns &r);
void tsg_state_device_free(TsgStateDevice *d);
