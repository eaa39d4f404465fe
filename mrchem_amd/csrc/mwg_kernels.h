// Kernel launchers and the device-side tables they consume.
#pragma once

#include <hip/hip_runtime.h>

#include "mwg_core.h"
#include "mwg_dev.h"

// CALL with KK = K as a constant, for the orders the library is built for
#define MWG_DISPATCH_K(K, CALL)                                       \
    switch (K) {                                                      \
        case 4: { constexpr int KK = 4; CALL; } break;                \
        case 5: { constexpr int KK = 5; CALL; } break;                \
        case 6: { constexpr int KK = 6; CALL; } break;                \
        case 7: { constexpr int KK = 7; CALL; } break;                \
        case 8: { constexpr int KK = 8; CALL; } break;                \
        case 9: { constexpr int KK = 9; CALL; } break;                \
        case 10: { constexpr int KK = 10; CALL; } break;              \
        default: return hipErrorInvalidValue;                         \
    }

namespace mwg {

constexpr double GAUSS_CUT_D = GAUSS_CUT;

struct DevBasis {
    int K;
    const double *U;     // K x K
    const double *qx;    // K
    const double *qw;    // K
    const double *phiq;  // K x K, [q][i]
    const double *W;     // 2K x 2K
    // products: components -> values at the quadrature points of the children, and values ->
    // components with the quadrature weights (2K x 2K, row-major)
    const double *E, *C;
};

struct ProjGeom {
    double lo[3];
    double sfac;
    int n0;
};

struct WorkItem {
    int job;
    int node;    // index in the job's output tree
    int l[3];    // translation relative to the root corner
    int parent;  // the node's parent in the output tree (-1 on the roots)
};

struct JobTab {
    DHash inHash;
    DHash genHash;
    const double *inCoef;
    const double *inNorm;
    const double *operBlocks;  // this depth's block array of the job's operator
    // split-FP16 copies (mixed precision): each K x K operator block and each K^3 input
    // component as rows of f16 hi and lo parts (layouts at split16_block_uint4), a
    // power-of-two exponent per block
    const uint4 *operBlocks16;
    const int *operExp16;
    const uint4 *inCoef16;
    const int *inExp16;
    const double *operNorms;   // this depth's norm array
    double *outCoef;
    double *outNorm;
    double thr;
    double route;  // mixed mode: slices with a bound above this run in FP64
    const int *pre;   // [ntab + 1] candidate prefix over terms (union boxes ub), device-built
    int tab0, ntab;
    int lmax[3];
    int depth;
    int ubox[3];  // union of ub over the table's terms (device-built)
    // refinement-predictor features of the nodes' children (see k_child_features)
    double feat_tnorm;   // output norm estimate at the start of the iteration
    double feat_innorm;  // input tree norm
    double prec;
    float feat_mu;       // log10(mu + 1e-3)
    float feat_cell;     // log10 of the children's cell width
    int n0;              // root scale
};

// Device-built contraction schedule of one refinement iteration (sizes the host reads
// back with the output norms; overflow set when a buffer capacity was too small or the
// generated-node pool did not hold every generated node, and then no kernel of the
// schedule runs).
struct TaskSummary {
    long long nslices64, nslices;  // FP64 and MFMA slices
    int ntasks, nstasks;           // their tasks (one slot of 8 K^3 doubles each)
    int overflow;  // bit 0: a capacity below, bit 1: generated-node pool
    int gen_count, gen_overflow;  // generated-node counter and table-overflow flag, for the host
    int chunk, schunk;            // slices per FP64 and MFMA task used by the schedule
};
struct TaskCaps {
    long long slices64, slices;
    int tasks, stasks;
};
// an output node's slices and tasks: FP64 (64) and split-FP16 MFMA (16); a task's slot has its
// index
struct NodeSched {
    long long start64, start16;
    int count64, count16;
    int task64, task16;  // first tasks
};

// one Gaussian term of one operator level, as the screening-box kernel reads it
struct LevTerm {
    double w;        // weight (unit coordinates)
    long long blk;   // block offset (doubles) in the level block array
    long long nrm;   // norm offset (doubles) in the level norm array
    long long env;   // offset of the term's 4 x (band + 1) norm envelopes in the level envelope array
    double maxn[4];  // largest block norm per type over the band
    int band;
    int active;
};

// screening-box request for one (job, depth) table
struct BoxJob {
    const LevTerm *terms;
    const double *env;
    double thr;   // tuple threshold of the job at this depth (0 on the roots)
    double F[8];  // largest input component norm per component at this depth
    int nterms;
    int depth;
    int tab0;     // first TermTab of this table
    int jt;       // index of the JobTab that receives the routing bound
    int pre_off;  // first entry of this table's prefix arrays (tab0 + jt)
};

// the candidate walk of an output node is split over up to ENUM_MAX_PARTS workgroups so
// that a work list of nw nodes launches about ENUM_BLOCKS of them (host and device agree)
constexpr int ENUM_BLOCKS = 512, ENUM_MAX_PARTS = 16;
__host__ __device__ inline int enum_parts(int nw) {
    if (nw <= 0) return 1;
    const int p = (ENUM_BLOCKS + nw - 1) / nw;
    return p < 1 ? 1 : (p > ENUM_MAX_PARTS ? ENUM_MAX_PARTS : p);
}

struct GenState {
    uint64_t *keys;
    int *job;
    int *count;
    int cap;
    int *overflow;
    double *pool;  // pcap x K^3
    double *norm;  // pcap
    int pcap;      // entries allocated in pool and norm (<= cap)
    long long *tabcnt;  // per job table: [4 t + 3] counts the generated nodes it inserted
};

hipError_t launch_tblock_mom(hipStream_t s, int n, const int *item_term, const long long *item_delta, const double *b,
                             const double *pre, int K, const double *ccoef, const double *gx, const double *gw,
                             double *out);
// where a group of NS block rows goes (blocks and norms may be null) and its first row
struct NSOut {
    double *blocks, *norms, *nrm;
    long long first;
};
// per row: translation, child-scale rows (the first one's index, their range), group
struct NSItems {
    const long long *delta;
    const int *row0, *tlo, *thi, *grp;
    const NSOut *outs;
};
hipError_t launch_nsblocks(hipStream_t s, long long first, long long n, const NSItems &items, const double *t1,
                           const double *W, int K);
hipError_t launch_norms(hipStream_t s, int n, const double *coef, double *norm, int K3);
// two nodes' coefficients (skip0: without their scaling parts)
struct DotPair {
    const double *a, *b;
    long long skip0;
};
hipError_t launch_dot(hipStream_t s, int n, const DotPair *pairs, int K3, double *part);
// sum over node pairs of a . b (part: nblocks doubles of block sums, res: the total)
hipError_t launch_dot_pairs(hipStream_t s, int n, const unsigned long long *pairs, const double *A,
                            const double *B, int K3, int nblocks, double *part, double *res);
hipError_t launch_scale(hipStream_t s, size_t n, double *x, double c);
// the device loop's start of an iteration, done by the screening-box kernels (LoopJob etc.
// are declared below): thresholds from the jobs' running norms instead of the tables'
// (table jb = job jb), table counts cleared, work counters and contraction stamps reset,
// generated-node range started
struct LoopJob;
struct LoopCtl;
struct LoopInit {
    const LoopJob *lj;  // null: the host loop (thresholds from the tables)
    long long *tabcnt;
    LoopCtl *ctl;
    unsigned long long *ts;
    const int *gen_count;
};
// TermTab[tab0 + t] for every (table, term): per-combination screening boxes from the
// monotone norm envelopes, union boxes, and the table's FP64 routing bound
hipError_t launch_job_boxes(hipStream_t s, int nbj, int max_terms, const BoxJob *bj, TermTab *tabs, double *tbmax,
                            JobTab *jobs, int *pre, int *gen_overflow, const LoopInit &li = LoopInit{});
// Device work counts: the work-list kernels below take an optional nwp, the work list's
// node count on the device (written by an earlier kernel of the stream); nw is then only
// an upper bound for the launch, and the kernels loop over the nodes on a grid of at most
// DEVCOUNT_GRID workgroups, taking them from the zeroed counter *queue when one is given.
constexpr int DEVCOUNT_GRID = 2048;
hipError_t launch_gen_mark(hipStream_t s, int nw, const WorkItem *work, const JobTab *jobs, const TermTab *tabs,
                           const GenState &gs, const int *nwp = nullptr, int *queue = nullptr);
// generated nodes first .. min(device count, cap) - 1 (cap = entries allocated in the pool;
// firstp: first read on the device)
hipError_t launch_gen_compute(hipStream_t s, int first, int cap, const JobTab *jobs, const GenState &gs,
                              const double *W, int K, const int *firstp = nullptr);
// A task: a run of slices of one output node (one workgroup, one slot of 8 K^3 doubles)
struct SliceTask {
    long long start;
    int count;
    int g;     // work index
    int slot;
};
// nparts workgroups share each output node's candidates (counts and offsets per
// (node, segment, part)); mode 0 counts (and adds the jobs' statistics), mode 1 writes the
// slices and tasks.  Plain method: one segment, the FP64 slices.
hipError_t launch_enum(hipStream_t s, int mode, int K, int nw, int nparts, const WorkItem *work, const JobTab *jobs,
                       const TermTab *tabs, const GenState &gs, int *seg_total, const long long *seg_ofs, Slice *out,
                       const TaskSummary *sum, const NodeSched *nodes, SliceTask *tasks, const int *nwp = nullptr,
                       int *queue = nullptr);
// FP64 slice contraction (mwg_fp64.hip).  With sum: the task count is read on the device; grid
// (tasks) covers the capacity.  infinite: an input has an infinite norm.  With ts: an extra first
// workgroup stamps the start.
hipError_t launch_contract_slices64(hipStream_t s, int K, bool infinite, int ntask, const TaskSummary *sum, int grid,
                                    const SliceTask *tasks, const WorkItem *work, const JobTab *jobs,
                                    const Slice *slices, const double *genPool, double *slots,
                                    unsigned long long *ts = nullptr);
// the device clock into *t (one thread; marks the end of the kernels before it on the stream)
hipError_t launch_stamp(hipStream_t s, unsigned long long *t);
struct TransformItem {
    double *coef;
    double *norm;  // component norms of the tree
    int parent;
    int first_child;
};
// (compact: the parents' norms in item order, mode 0)
hipError_t launch_transform(hipStream_t s, int mode, int n, const TransformItem *items, const double *M, int K,
                            double *compact = nullptr);
hipError_t launch_enum_mixed(hipStream_t s, int mode, int K, int nw, int nparts, const WorkItem *work,
                             const JobTab *jobs, const TermTab *tabs, const GenState &gs, int *thread_off,
                             int *seg_total, const long long *seg_ofs, Slice *out64, Slice *out16,
                             const TaskSummary *sum, const NodeSched *nodes, SliceTask *tasks, SliceTask *stasks,
                             const int *nwp = nullptr, int *queue = nullptr);
// Split-FP16 copies of FP64 blocks (mwg_mfma.hip): block b (values src[b bvals ..]) as rows
// of K values, scaled by 2^exp[b] so that the block's largest magnitude lies in [0.5, 1)
// (exp 0 for a zero block); x 2^e = hi + lo up to about 2^-23 of it.  K = 8: each row
// [hi 8 | lo 8] (two uint4).  K = 10, role 0 (operator blocks, A operands): each row
// [hi 10 | hi 10 | lo 10 | 0 0] (four uint4); role 1 (input nodes, B operands): each row
// [hi 10 | lo 10] (40 bytes).  With count, only blocks first .. min(*count, first + n) - 1;
// with firstp, first is read on the device and the blocks are first .. min(*count, n) - 1.
// the same for the blocks of several arrays (e.g. the input trees of a batch) in one launch:
// item i's blocks are first[i] .. first[i + 1] - 1 of the concatenation (first[nitems] = total)
struct Split16Item {
    const double *src;
    uint4 *dst;
    int *exp;
};
hipError_t launch_split16_multi(hipStream_t s, int nitems, const Split16Item *items, const long long *first,
                                long long total, int bvals, int K, int role);
hipError_t launch_split16(hipStream_t s, int n, int first, const int *count, int bvals, int K, const double *src,
                          uint4 *dst, int *exp, int role = 0, const int *firstp = nullptr);
// uint4 per block of bvals values of a split-FP16 copy
inline size_t split16_block_uint4(int K, int role, int bvals) {
    return K == 8 ? (size_t)bvals / 4 : role == 0 ? (size_t)bvals / 10 * 4 : (size_t)bvals / 10 * 40 / 16;
}
// FP32 / split-FP16 MFMA slice contraction (K = 8 or 10; mwg_mfma.hip).  A task is a run of
// slices of one output node; mfma_tasks_per_block(K) tasks share a 256-thread block.  Each
// task adds the surviving tuples of its slices to tabcnt[4 t + 2] of its job table t.
// genPool16 / genExp16: the generated nodes' split-FP16 copies.
int mfma_tasks_per_block(int K);
hipError_t launch_contract_mfma(hipStream_t s, int K, int ntask, const TaskSummary *sum, int grid,
                                const SliceTask *tasks, const WorkItem *work, const JobTab *jobs,
                                const TermTab *tabs, const Slice *slices, const double *genPool, double *nodeslots,
                                long long *tabcnt, const uint4 *genPool16, const int *genExp16);
// a tree's node table and where its nodes' keys lie
struct HashItem {
    DHash h;
    long long first;
    int n;
};
hipError_t launch_hash_build(hipStream_t s, int n, const HashItem *items, const unsigned long long *keys);
// n doubles from p to dst + first
struct GatherItem {
    const double *p;
    long long first;
    int n;
};
hipError_t launch_gather(hipStream_t s, int n, const GatherItem *items, double *dst);
// an output node of a product, sum or projection, with the inputs that represent it
struct MulItem {
    int node;
    int depth;
    int l[3];
    int asrc, asteps;  // input a: node (steps = 0) or leaf ancestor and levels to refine
    int bsrc, bsteps;
    int job;
};
// product (coef a b)
struct MulJobDev {
    const double *a, *b;
    double *out, *norm;
    double coef;
};
// an output node of a linear combination: its coefficients and norms, its terms
struct SumItem {
    double *out, *norm;
    int lx, ly, lz;
    int src0, nsrc;
};
// a term: the node (steps = 0) or leaf ancestor that represents the input, levels to refine
struct SumSrc {
    const double *p;
    double coef;
    long long steps;
};
// each writes the nodes' coefficients, their norms into the tree and into compact[8 item]
hipError_t launch_multiply(hipStream_t s, int n, const MulItem *items, const MulJobDev *jobs, const ProjGeom &geo,
                           const DevBasis &B, double *compact);
hipError_t launch_sum(hipStream_t s, int n, const SumItem *items, const SumSrc *srcs, const DevBasis &B,
                      double *compact);
hipError_t launch_project_gauss(hipStream_t s, int nw, const MulItem *items, const ProjGeom &geo, const DevBasis &B,
                                int nterm, const double *coef, const double *alpha, const double *center,
                                const double *poly, double *out, double *norm, double *compact);
hipError_t launch_project_hyd(hipStream_t s, int nw, const MulItem *items, const ProjGeom &geo, const DevBasis &B,
                              int nterm, const double *coef, const int *q, double Z, const double *origin, double *out,
                              double *norm, double *compact);
// from the per-(node, segment, part) counts (nseg = 1: plain FP64, 2: mixed): part offsets,
// task sizes, every node's first slices and tasks.  wchunk: slices per MFMA task, or (<= 0)
// about -wchunk tasks over the iteration's slices.
hipError_t launch_build_tasks(hipStream_t s, int nw, int nseg, int nparts, int chunk, int wchunk, const int *tot,
                              TaskCaps caps, const int *gen_count, int gen_pcap, long long *ofs, NodeSched *nodes,
                              TaskSummary *sum, const int *gen_overflow, const int *nwp = nullptr);
// ---- device-resident refinement (mwg_kernels.hip)
// The plain method's refinement loop without a host round trip: every job of the batch has
// one job table per iteration (table index = job index, all work nodes of iteration d at
// depth d); after the contraction and the output norms, k_loop_split takes the split test
// and appends the children to the output trees, k_loop_emit writes the next work list.
constexpr int LOOP_MAX_DEPTH = 32, LOOP_MAX_JOBS = 4096;
struct LoopJob {
    int *depth, *parent, *child, *lr;  // output tree topology on the device (lr: 3 per node), cap nodes
    int n, cap;                        // nodes so far, capacity
    int w0, nwk;                       // this iteration's work nodes [w0, w0 + nwk) of the work list
    int splits, pad;                   // nodes split by this iteration
    double sNorm, wNorm, gsq;          // running output norm (gsq < 0: none yet)
    double prec;
    long long tuples, tuples_fp64, slices, gen;  // statistics (as mwg_apply_stats)
};
// what the host reads back after each iteration
struct LoopIter {
    int nw_next;   // work nodes of the next iteration (0: done, or stopped by an overflow)
    int overflow;  // sticky: bit 0 schedule capacity, 1 generated-node pool, 2 node capacity,
                   // 3 work-list capacity, 4 generated-node table, 5 transform-item capacity
};
struct LoopCtl {
    int nw[2];     // work list sizes: iteration d reads nw[d & 1], writes nw[(d + 1) & 1]
    int queue[4];  // work counters of the iteration's k_gen_mark, k_enum count and fill (zeroed)
    int genFirst;  // generated-node counter at the start of the iteration
    int overflow;  // sticky (LoopIter bits)
    double splitfac[LOOP_MAX_DEPTH];  // 2^(-(n0 + d + 1) / 2) of the split test at depth d
    LoopIter iter[LOOP_MAX_DEPTH];
    int tofs[LOOP_MAX_DEPTH + 1];     // first transform item of the split nodes of depth d
    unsigned long long ts[LOOP_MAX_DEPTH][2];  // contraction start and end, device clock
};
// the roots (nr per job, translations rootlr, the same for every job) in the topology and
// the first work list
hipError_t launch_loop_init(hipStream_t s, int njobs, int nr, const LoopJob *lj, const int *rootlr, WorkItem *work);
// per job (one workgroup): running norm, split test of its work nodes, children appended
// (cidx[i]: first child of work node i, -1 if not split)
hipError_t launch_loop_split(hipStream_t s, int njobs, LoopJob *lj, const WorkItem *work, const double *wnorm,
                             int max_depth, LoopCtl *ctl, int *cidx, const long long *tabcnt,
                             unsigned long long *ts_end = nullptr);
// the next work list (and its size in *nw_next and in ctl->iter[d] and host_iter[d], pinned
// host memory the host reads once the iteration is done), and the split nodes as transform
// items of depth d (from ctl->tofs[d], capacity tcap)
hipError_t launch_loop_emit(hipStream_t s, int njobs, LoopJob *lj, const WorkItem *work, const int *nwp,
                            const int *cidx, WorkItem *next, int *nw_next, int wcap, const TaskSummary *sum,
                            LoopCtl *ctl, int d, const JobTab *jt, TransformItem *titems, int tcap,
                            LoopIter *host_iter);

// refinement-predictor features of the 8 children of every work node (row i*8 + a, a the
// child index), from the work nodes' norms just computed, their parents' norms and the
// input tree around each child
hipError_t launch_child_features(hipStream_t s, int nw, const WorkItem *work, const JobTab *jobs,
                                 const double *wnorms, float *feat);
hipError_t launch_move_groups(hipStream_t s, int npairs, const int *from_to, double *coef, double *norm, int nb);
// output components (and their norms, also to wnorm) from the task slots
hipError_t launch_reduce_slots(hipStream_t s, int nw, const int *nwp, const TaskSummary *sum, const NodeSched *nodes,
                               const WorkItem *work, const JobTab *jobs, const double *slots64, const double *slots16,
                               int K3, double *wnorm);

}  // namespace mwg
