// FP64 slice contraction of the apply (gfx950, wave64).
//
// A slice (g, f, ft, term) holds every surviving output component gt of node g from input
// component ft of node f (mask: bit gt): out_gt[c][b][a] += w sum Z[c][l] Y[b][j] X[a][i] f[l][j][i]
// with X = X_{gt_x, ft_x}(dx) etc.  A task is a run of slices of one node; the work list orders
// the slices of a term by (dz, ft_z), then (dy, ft_y), then (dx, ft_x), so that runs share their
// Z and Y blocks and the three passes are not paid per combination:
//   pass x  T1 = X f             once per slice and gt_x; added to U[gt] for every gt of the mask
//   pass y  V[gt] += Y U[gt]     once per run of equal (dy, ft_y) and gt
//   pass z  W[gt] += (w Z) V[gt] once per run of equal (dz, ft_z) and gt
// (the sums are linear, so exactly the surviving combinations enter; only the order of the
// FP64 additions differs from one combination at a time).  A list in any other order gives
// the same result with shorter runs: the FP64 slices of a mixed apply come in the order of the
// candidates, each thread's after another's, and pay all three passes nearly every time.  INF: the batch has an input of infinite norm; the products with
// zero that otherwise mask components and row ends would carry it into components that it does not
// contribute to (they are selects then, which takes 5 to 11 % longer).
//
// Every pass runs on v_mfma_f64_4x4x4_4b_f64: four blocks of (4 rows) x (4 columns), 4 products
// long, in 16 cycles, the full FP64 rate of the chip.  Lane L = 16 kq + 4 blk + r supplies
// A[row r][k = kq] and B[k = kq][column r] of block blk and holds D[row kq][column r].  So a
// result can be the next product's operand as it is: its row index becomes the contraction
// index, its column and block indices stay.  An index of length K is spread over four lane
// positions p and G = ceil(K / 4) registers g: value m(p, g) = min(G p, K - G) + g (positions whose
// range is cut repeat values; their products are zeroed in one operand, their results unused).
// A wave holds four of the 2 K stacked output rows a' (gt_x, a) and all of j, l:
//   x  T1[j][a'; l]: rows j, columns a', blocks l.  A = f, B = X'
//   y  V[b][a'; l]:  rows b, columns a', blocks l.  A = Y, B = U (k = j: the rows of T1)
//   z  W[c][a'; b]:  rows c, columns a', blocks b.  A = Z, B = V with rows b and blocks l
//      exchanged (k = l): the one shuffle, a lane permutation through the wave's LDS
// with no exchange between waves.  G^3 instructions per pass.
//
// What bounds it: the FP64 pipe, which the products share with the other vector instructions
// (a v_fma_f64 and a product do not overlap).  Per slice and wave at K = 8 about 18 products
// (290 cycles) and 78 other vector instructions (310 cycles), the staging and the schedule among
// them; the counters show the pipe busy 52 % of the time, the rest are LDS latencies and the
// barriers with at most three waves per SIMD (2.3 on average, 35 % of their cycles waiting).
// One combination at a time on v_fma_f64, each with its three passes through LDS, took
// 4.29 ms on the contractions of five k = 7 Helmholtz applies at prec 1e-6 (5.55 M combinations
// in 1.05 M slices, 32 TFLOP/s of 6 K^4 flops each); this takes 2.06 ms (66).  Loading the operands
// straight from global memory in their lane layout (a line per lane) took 3.8 ms, four staged
// slices per buffer (two workgroups per CU instead of three) 2.5.
#include <hip/hip_ext.h>

#include "mwg_kernels.h"

namespace mwg {

namespace {

typedef const double __attribute__((address_space(1))) gdbl;

__device__ inline int wave_index() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline double mfma4(double a, double b, double c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

template <int K>
struct F64 {
    static constexpr int G = (K + 3) / 4;
    static constexpr int NA = (2 * K + 3) / 4;  // waves of a task: groups of four stacked rows a'
    static constexpr bool EVEN = K % 4 == 0;    // no repeated values, gt_x uniform in a wave
};

// A workgroup (the NA waves of a task) stages the operands of NS slices at a time in LDS, two
// buffers in turn: the global loads of the next batch are issued before a batch is contracted
// and written to LDS after it, in whole lines (an operand's own lane layout would touch a
// line per lane), one barrier per batch.
template <int K>
struct Stg {
    static constexpr int NS = 2;
    static constexpr int NT = F64<K>::NA * 64;
    static constexpr int K2 = K * K, K3 = K2 * K;
    // values of a slice: f | X, Y, Z block pairs, moved in pieces of P values
    static constexpr int P = K % 2 == 0 ? 2 : 1;
    static constexpr int FN = K3, PN = 2 * K2, SLOT = FN + 3 * PN;
    static constexpr int FC = (FN / P + NT - 1) / NT, PC = (3 * PN / P + NT - 1) / NT;  // pieces per thread
};

// place of the piece q of an input block in LDS (K = 8: in the order of the operand
// registers, turned so that neither the writes nor the reads meet in a bank)
template <int K>
__device__ inline int f_place(int q) {
    if constexpr (K == 8) {
        const int kq = q & 3, row = q >> 2, j = row & 7, l = row >> 3;
        return (((l & 1) * 2 + (j & 1)) * 64 + 16 * kq + ((4 * (l >> 1) + (j >> 1)) ^ (4 * kq) ^ (2 * (j & 1)))) * 2;
    } else {
        return Stg<K>::P * q;
    }
}

}  // namespace

template <int K, bool INF>
__global__ void __launch_bounds__(F64<K>::NA * 64) __attribute__((amdgpu_waves_per_eu(3)))
k_contract_slices64(int ntask_arg, const TaskSummary *sum, const SliceTask *tasks, const WorkItem *work,
                    const JobTab *jobs, const Slice *slices, const double *genPool, double *slots,
                    unsigned long long *ts) {
    using D = Stg<K>;
    constexpr int G = F64<K>::G, NA = F64<K>::NA, K2 = K * K, K3 = K2 * K, NS = D::NS, NT = D::NT;
    constexpr int RB = 64;  // records in LDS
    __shared__ __align__(16) double stage[2][NS][(D::SLOT + 1) & ~1];
    __shared__ __align__(16) double xch[NA][G * G][80];  // pass z: 64 lanes + a gap of 4 after every 16
    __shared__ __align__(16) Slice recs[RB + NS + 1];
    // (with ts, block 0, dispatched first, only stamps the contraction's start)
    if (ts && blockIdx.x == 0) {
        if (threadIdx.x == 0) *ts = (unsigned long long)wall_clock64();
        return;
    }
    const int ntask = sum ? (sum->overflow ? 0 : sum->ntasks) : ntask_arg;
    const int ti = (int)blockIdx.x - (ts ? 1 : 0);
    if (ti >= ntask) return;
    const SliceTask task = tasks[ti];
    const int wv = wave_index(), tid = threadIdx.x;
    const int lane = tid & 63, kq = lane >> 4, blk = (lane >> 2) & 3, r4 = lane & 3;
    const JobTab &J = jobs[work[task.g].job];
    const gdbl *oper = (const gdbl *)J.operBlocks, *in = (const gdbl *)J.inCoef, *gen = (const gdbl *)genPool;
    // index m(p, 0) for this lane's p = kq, blk, r4
    const int mk = min(G * kq, K - G), mb = min(G * blk, K - G), mr = min(G * r4, K - G);
    const int ap = 4 * wv + r4, gxl = ap >= K ? 1 : 0, al = min(ap - gxl * K, K - 1);  // this lane's column a'
    bool ok[G];  // the entries m(kq, s) that are not repeated
#pragma unroll
    for (int g = 0; g < G; g++) ok[g] = F64<K>::EVEN || mk + g >= G * kq;
    double U[4][G][G], V[4][G][G], W[4][G][G];  // [gt_y + 2 gt_z]: U[jg][lg], V[bg][lg], W[cg][bg]
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int r = 0; r < G; r++)
#pragma unroll
            for (int t = 0; t < G; t++) U[p][r][t] = V[p][r][t] = W[p][r][t] = 0.0;
    const Slice *srec = slices + task.start;
    const int count = task.count;
    // records r0 .. r0 + RB + NS (clamped to the task) into LDS
    auto load_recs = [&](int r0) {
        const int n = 2 * min(RB + NS + 1, count - r0);
        // (K = 7 has no register to spare for these addresses)
        for (int q = K == 7 ? (int)thread_here() : tid; q < n; q += NT) ((uint4 *)recs)[q] = ((const uint4 *)(srec + r0))[q];
    };
    auto u = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    typedef double piece __attribute__((ext_vector_type(D::P)));
    typedef const piece __attribute__((address_space(1))) gpiece;
    piece lf[NS][D::FC], lp[NS][D::PC];
    // the pieces of the slices b .. b + NS - 1 that this thread stages (r0: first record in LDS)
    auto load_batch = [&](int b, int r0) {
#pragma unroll
        for (int i = 0; i < NS; i++) {
            const Slice &sl = recs[min(b + i, count - 1) - r0];
            const int f = u(sl.f), ft = u((int)sl.ft), xo = u(sl.xo), yo = u(sl.yo), zo = u(sl.zo);
            const gdbl *fp = f >= 0 ? in + ((size_t)f * 8 + ft) * K3 : gen + (size_t)(-f - 1) * K3;
#pragma unroll
            for (int c = 0; c < D::FC; c++) {
                const int q = min(tid + c * NT, K3 / D::P - 1);
                lf[i][c] = *(gpiece *)(fp + D::P * (unsigned)q);
            }
#pragma unroll
            for (int c = 0; c < D::PC; c++) {
                // pieces of the block pairs X | Y | Z (gt_d = 0, 1: blocks o and o + 2)
                const int q = min(tid + c * NT, 3 * D::PN / D::P - 1), e = D::P * q, pr = e / D::PN, r = e - pr * D::PN;
                const int o = pr == 0 ? xo : pr == 1 ? yo : zo;
                lp[i][c] = *(gpiece *)(oper + (size_t)(unsigned)o * K2 + (unsigned)(r + (r >= K2 ? K2 : 0)));
            }
        }
    };
    auto store_batch = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NS; i++) {
            double *st = stage[buf][i];
#pragma unroll
            for (int c = 0; c < D::FC; c++) {
                const int q = tid + c * NT;
                if (K == 8 || q < K3 / D::P) *(piece *)(st + f_place<K>(q)) = lf[i][c];
            }
#pragma unroll
            for (int c = 0; c < D::PC; c++) {
                const int q = tid + c * NT;
                if (q < 3 * D::PN / D::P) *(piece *)(st + D::FN + D::P * q) = lp[i][c];
            }
        }
    };
    // the A entries of the operators of both gt_d from a staged block pair
    auto pair_a = [&](const double *pr, double (&a)[2][G][G]) {
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int r = 0; r < G; r++)
#pragma unroll
                for (int s = 0; s < G; s++) {
                    const double v = pr[q * K2 + (mr + r) * K + mk + s];
                    a[q][r][s] = ok[s] ? v : 0.0;
                }
    };
    // the wave's gt_x: one, or (a wave across the two) both
    const bool both = !F64<K>::EVEN && 4 * wv < K && 4 * wv + 3 >= K;
    const int gxw = 4 * wv >= K ? 1 : 0;
    // components (bit 2 p) of the run in U and in V, and whether (bit 2 gt_y) the two gt_z of a
    // gt_y got different slices in the run: else U is the same for both and pass y runs once
    int umask = 0, udiff = 0, vmask = 0;
    auto slice_step = [&](const double *st, int mask, bool endy, bool endz, double w) {
        int mw = mask >> gxw, dw = mw ^ (mw >> 4);
        if (both) {
            dw = mask ^ (mask >> 4);
            mw = mask | (mask >> 1);
            dw |= dw >> 1;
        }
        mw &= 0x55;
        if (mw) {  // pass x
            double f[G][G][G], x[G], t1[G][G];
#pragma unroll
            for (int l = 0; l < G; l++)
#pragma unroll
                for (int j = 0; j < G; j++)
#pragma unroll
                    for (int s = 0; s < G; s++) {
                        if constexpr (K == 8)
                            f[l][j][s] = st[((l * 2 + j) * 64 + 16 * kq + ((4 * blk + r4) ^ (4 * kq) ^ (2 * j))) * 2 + s];
                        else
                            f[l][j][s] = st[((mb + l) * K + mr + j) * K + mk + s];
                    }
#pragma unroll
            for (int s = 0; s < G; s++) {
                const double v = st[D::FN + gxl * K2 + al * K + mk + s];
                x[s] = ok[s] ? v : 0.0;
            }
#pragma unroll
            for (int j = 0; j < G; j++)
#pragma unroll
                for (int l = 0; l < G; l++) t1[j][l] = mfma4(f[l][j][0], x[0], 0.0);
#pragma unroll
            for (int s = 1; s < G; s++)
#pragma unroll
                for (int j = 0; j < G; j++)
#pragma unroll
                    for (int l = 0; l < G; l++) t1[j][l] = mfma4(f[l][j][s], x[s], t1[j][l]);
            // added to the components of the mask: a product with 1 or 0 (exact for finite values, no
            // branches), a select where there may be others
            const int m = F64<K>::EVEN ? mask >> gxw : mask >> gxl;
            if constexpr (INF) {
#pragma unroll
                for (int p = 0; p < 4; p++)
#pragma unroll
                    for (int j = 0; j < G; j++)
#pragma unroll
                        for (int l = 0; l < G; l++) U[p][j][l] += (m >> (2 * p)) & 1 ? t1[j][l] : 0.0;
            } else {
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const double on1 = __hiloint2double((m >> (2 * p)) & 1 ? 0x3ff00000 : 0, 0);
#pragma unroll
                    for (int j = 0; j < G; j++)
#pragma unroll
                        for (int l = 0; l < G; l++) U[p][j][l] = fma(t1[j][l], on1, U[p][j][l]);
                }
            }
            umask |= mw;
            udiff |= dw;
        }
        if (!endy) return;
        if (umask) {  // pass y
            double Y[2][G][G];
            pair_a(st + D::FN + D::PN, Y);
#pragma unroll
            for (int gy = 0; gy < 2; gy++) {
                const int mm = umask >> (2 * gy);
                if ((mm & 0x11) == 0x11 && !((udiff >> (2 * gy)) & 1)) {
                    double t[G][G];
#pragma unroll
                    for (int b = 0; b < G; b++)
#pragma unroll
                        for (int l = 0; l < G; l++) t[b][l] = mfma4(Y[gy][b][0], U[gy][0][l], 0.0);
#pragma unroll
                    for (int s = 1; s < G; s++)
#pragma unroll
                        for (int b = 0; b < G; b++)
#pragma unroll
                            for (int l = 0; l < G; l++) t[b][l] = mfma4(Y[gy][b][s], U[gy][s][l], t[b][l]);
#pragma unroll
                    for (int b = 0; b < G; b++)
#pragma unroll
                        for (int l = 0; l < G; l++) {
                            V[gy][b][l] += t[b][l];
                            V[gy + 2][b][l] += t[b][l];
                        }
                } else {
#pragma unroll
                    for (int p = gy; p < 4; p += 2)
                        if ((umask >> (2 * p)) & 1) {
#pragma unroll
                            for (int s = 0; s < G; s++)
#pragma unroll
                                for (int b = 0; b < G; b++)
#pragma unroll
                                    for (int l = 0; l < G; l++)
                                        V[p][b][l] = mfma4(Y[gy][b][s], U[p][s][l], V[p][b][l]);
                        }
                }
            }
#pragma unroll
            for (int p = 0; p < 4; p++)
#pragma unroll
                for (int j = 0; j < G; j++)
#pragma unroll
                    for (int l = 0; l < G; l++) U[p][j][l] = 0.0;
            vmask |= umask;
            umask = udiff = 0;
        }
        if (!endz || !vmask) return;
        // pass z: lane 16 kq + 4 blk + r takes the values of lane 16 blk + 4 kq + r
        double Z[2][G][G];
        pair_a(st + D::FN + 2 * D::PN, Z);
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int c = 0; c < G; c++)
#pragma unroll
                for (int s = 0; s < G; s++) Z[q][c][s] *= w;
        const int from = 20 * blk + 4 * kq + r4;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            if (!((vmask >> (2 * p)) & 1)) continue;
#pragma unroll
            for (int b = 0; b < G; b++)
#pragma unroll
                for (int l = 0; l < G; l++) {
                    xch[wv][b * G + l][lane + 4 * kq] = V[p][b][l];
                    V[p][b][l] = 0.0;
                }
            wave_sync();
            double v[G][G];
#pragma unroll
            for (int b = 0; b < G; b++)
#pragma unroll
                for (int l = 0; l < G; l++) v[b][l] = xch[wv][b * G + l][from];
            wave_sync();
#pragma unroll
            for (int s = 0; s < G; s++)
#pragma unroll
                for (int c = 0; c < G; c++)
#pragma unroll
                    for (int b = 0; b < G; b++) W[p][c][b] = mfma4(Z[p >> 1][c][s], v[b][s], W[p][c][b]);
        }
        vmask = 0;
    };
    load_recs(0);
    __syncthreads();
    load_batch(0, 0);
    store_batch(0);
    __syncthreads();
    int r0 = 0, buf = 0;
    for (int b = 0; b < count; b += NS) {
        if (b - r0 == RB) {  // (every wave is past the last use of the records)
            r0 = b;
            load_recs(r0);
            __syncthreads();
        }
        const int n = min(NS, count - b);
        load_batch(b + NS, r0);
        for (int i = 0; i < n; i++) {
            const Slice &cur = recs[b + i - r0], &nxt = recs[min(b + i + 1, count - 1) - r0];
            const bool end = b + i == count - 1;
            const bool endz = end || u(cur.zo) != u(nxt.zo), endy = endz || u(cur.yo) != u(nxt.yo);
            const double w = cur.w;
            slice_step(stage[buf][i], u((int)cur.mask), endy, endz,
                       __hiloint2double(u(__double2hiint(w)), u(__double2loint(w))));
        }
        buf ^= 1;
        store_batch(buf);
        __syncthreads();
    }
    double *dst = slots + (size_t)task.slot * 8 * K3 + gxl * K3 + al;
    const bool aok = ap < 2 * K;
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int c = 0; c < G; c++)
#pragma unroll
            for (int b = 0; b < G; b++)
                if (F64<K>::EVEN || (aok && ok[c] && mb + b >= G * blk))
                    dst[2 * p * K3 + (mk + c) * K2 + (mb + b) * K] = W[p][c][b];
}

// ------------------------------------------------------------------ k = 8 and 9 (K = 9, 10)
//
// With G = 3 the accumulators of a wave's four rows a' fill the registers and a third of the
// products are repeats, so the planes l are split over the waves instead: wave w holds l = S w ..
// S w + S - 1 as dense columns, (l, j) in pass x, (a, l) in pass y, T tiles of 16 (column = lane %
// 16; the four blocks of an instruction get the same A rows), a workgroup one gt_x.  Passes x
// and y exchange through the wave's own LDS rows, pass z over the workgroup.  Eight k = 9
// Helmholtz applies at prec 1e-6 (6.6 M combinations in 1.2 M slices): contractions 14.7 ms one
// combination at a time, 11.2 with the split over rows a' above (one wave per SIMD), 10.1 here with a
// select per entry of A and a branch per exchanged value, 9.6 with neither: the staged rows end in
// zeros, and what has no place goes to a row's padding.  Now the FP64 pipe is busy 47 % of the
// time and LDS 47 %, with the two waves per SIMD that the accumulators leave room for.
template <int K>
struct Wide {
    static constexpr int RG = (K + 3) / 4, KS = RG;  // row groups; products per lane group
    static constexpr int WV = K == 9 ? 3 : 4, S = (K + WV - 1) / WV, T = (S * K + 15) / 16, NT = WV * 64;
    static constexpr int K2 = K * K, K3 = K2 * K, ROW = (K + 1) | 1;  // ROW: an LDS row, odd
    // rows of the staged operator blocks: a lane group's KS entries are there for all four, zeros
    // beyond K (a select per entry of A otherwise)
    static constexpr int AR = 4 * KS, A2 = K * AR;
    static constexpr int U_WAVE = 4 * S * K * ROW, V_ALL = 4 * K2 * ROW;
    static constexpr int XCH = WV * U_WAVE > V_ALL ? WV * U_WAVE : V_ALL;
    // staged values of a slice: f | X | Y, Z block pairs
    static constexpr int P = K % 2 == 0 ? 2 : 1, SLOT = K3 + AR - K + 5 * A2, A0 = K3 + AR - K;
    static constexpr int FC = (K3 / P + NT - 1) / NT, PC = (5 * K2 / P + NT - 1) / NT;
};

template <int K, bool INF>
__global__ void __launch_bounds__(Wide<K>::NT) __attribute__((amdgpu_waves_per_eu(2)))
k_contract_slices64w(int ntask_arg, const TaskSummary *sum, const SliceTask *tasks, const WorkItem *work,
                     const JobTab *jobs, const Slice *slices, const double *genPool, double *slots,
                     unsigned long long *ts) {
    using D = Wide<K>;
    constexpr int RG = D::RG, KS = D::KS, T = D::T, S = D::S, K2 = D::K2, K3 = D::K3, NT = D::NT, ROW = D::ROW;
    constexpr int RB = 64;  // records in LDS
    __shared__ __align__(16) double stage[2][(D::SLOT + 1) & ~1];
    __shared__ __align__(16) double xch[D::XCH + D::AR];  // rows of U per wave; rows of V of the workgroup
    __shared__ __align__(16) Slice recs[RB + 2];
    if (ts && blockIdx.x == 0) {
        if (threadIdx.x == 0) *ts = (unsigned long long)wall_clock64();
        return;
    }
    const int ntask = sum ? (sum->overflow ? 0 : sum->ntasks) : ntask_arg;
    // the two gt_x of a task follow each other on one XCD (blocks go to the 8 XCDs in turn)
    const int bid = (int)blockIdx.x - (ts ? 1 : 0), gx = (bid >> 3) & 1, ti = (bid >> 4) * 8 + (bid & 7);
    if (ti >= ntask) return;
    const SliceTask task = tasks[ti];
    const int wave = wave_index(), tid = threadIdx.x, lane = tid & 63, col = lane & 15, kq = lane >> 4, r4 = lane & 3;
    const JobTab &J = jobs[work[task.g].job];
    const gdbl *oper = (const gdbl *)J.operBlocks, *in = (const gdbl *)J.inCoef, *gen = (const gdbl *)genPool;
    double *Ul = xch + wave * D::U_WAVE, *Vl = xch;
    const int ib = KS * kq;  // entries ib + s of a row (beyond K: the next row's, times a zero of A)
    int ar[RG];
#pragma unroll
    for (int r = 0; r < RG; r++) ar[r] = min(4 * r + r4, K - 1) * D::AR + ib;
    bool zok[T];  // this lane's column of pass x (l, j), pass y (a, l), pass z (b, a) exists
    // (positions: rows and columns that do not exist go to entry K of some row, which counts for nothing)
    int xb[T], xu[RG][T], yv[RG][T], yr[T], zc[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
        const int n = t * 16 + col, nc = min(n, S * K - 1), l = nc / K, j = nc % K, a = nc / S, m = nc % S;
        const bool xok = n < S * K && wave * S + l < K, yok = n < S * K && wave * S + m < K;
        xb[t] = (min(wave * S + l, K - 1) * K + j) * K + ib;  // f
        yr[t] = nc * ROW + ib;                                // row nc of U
#pragma unroll
        for (int r = 0; r < RG; r++) {
            const int q = 4 * r + kq;
            xu[r][t] = xok && q < K ? (q * S + l) * ROW + j : col * ROW + K;            // row (a, l), entry j of U
            yv[r][t] = yok && q < K ? (q * K + a) * ROW + wave * S + m : lane * ROW + K;  // row (b, a), entry l of V
        }
        const int z = (wave * T + t) * 16 + col;
        zok[t] = z < K2;
        zc[t] = min(z, K2 - 1);
    }
    double U[4][RG][T], V[4][RG][T], W[4][RG][T];
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int r = 0; r < RG; r++)
#pragma unroll
            for (int t = 0; t < T; t++) U[p][r][t] = V[p][r][t] = W[p][r][t] = 0.0;
    const Slice *srec = slices + task.start;
    const int count = task.count;
    auto load_recs = [&](int r0) {
        const int n = 2 * min(RB + 2, count - r0);
        for (int q = tid; q < n; q += NT) ((uint4 *)recs)[q] = ((const uint4 *)(srec + r0))[q];
    };
    auto u = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    typedef double piece __attribute__((ext_vector_type(D::P)));
    typedef const piece __attribute__((address_space(1))) gpiece;
    piece lf[D::FC], lp[D::PC];
    auto load = [&](int b, int r0) {  // slice b's operands: this thread's pieces
        const Slice &sl = recs[min(b, count - 1) - r0];
        const int f = u(sl.f), ft = u((int)sl.ft), xo = u(sl.xo) + 2 * gx, yo = u(sl.yo), zo = u(sl.zo);
        const gdbl *fp = f >= 0 ? in + ((size_t)f * 8 + ft) * K3 : gen + (size_t)(-f - 1) * K3;
#pragma unroll
        for (int c = 0; c < D::FC; c++) lf[c] = *(gpiece *)(fp + D::P * (unsigned)min(tid + c * NT, K3 / D::P - 1));
#pragma unroll
        for (int c = 0; c < D::PC; c++) {
            const int e = D::P * min(tid + c * NT, 5 * K2 / D::P - 1), pr = e / K2, r = e - pr * K2;  // X Y0 Y1 Z0 Z1
            const int o = pr == 0 ? xo : pr < 3 ? yo + 2 * (pr - 1) : zo + 2 * (pr - 3);
            lp[c] = *(gpiece *)(oper + (size_t)(unsigned)o * K2 + (unsigned)r);
        }
    };
    auto store = [&](double *st) {
#pragma unroll
        for (int c = 0; c < D::FC; c++)
            if (tid + c * NT < K3 / D::P) *(piece *)(st + D::P * (tid + c * NT)) = lf[c];
#pragma unroll
        for (int c = 0; c < D::PC; c++)
            if (tid + c * NT < 5 * K2 / D::P) {
                const int e = D::P * (tid + c * NT), row = e / K;
                *(piece *)(st + D::A0 + row * D::AR + (e - row * K)) = lp[c];
            }
    };
    auto load_a = [&](const double *blk, double (&a)[RG][KS]) {
#pragma unroll
        for (int r = 0; r < RG; r++)
#pragma unroll
            for (int s = 0; s < KS; s++) a[r][s] = blk[ar[r] + s];
    };
    // entries of a row beyond K, times a zero of A: what another component left there may be infinite
    auto row_end = [&](double (&v)[T][KS]) {
        if constexpr (INF) {
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int s = 0; s < KS; s++) v[t][s] = ib + s < K ? v[t][s] : 0.0;
        }
    };
    // zeros behind the rows of f and of the blocks; finite values wherever a row's end is read
    for (int q = tid; q < 2 * ((D::SLOT + 1) & ~1); q += NT) (&stage[0][0])[q] = 0.0;
    for (int q = tid; q < D::XCH + D::AR; q += NT) xch[q] = 0.0;
    load_recs(0);
    __syncthreads();
    load(0, 0);
    store(stage[0]);
    __syncthreads();
    int r0 = 0, umask = 0, vmask = 0;
    for (int b = 0; b < count; b++) {
        if (b - r0 == RB) {  // (every wave is past the last use of the records)
            r0 = b;
            load_recs(r0);
            __syncthreads();
        }
        load(b + 1, r0);
        const double *st = stage[b & 1];
        const Slice &cur = recs[b - r0], &nxt = recs[min(b + 1, count - 1) - r0];
        const int mask = (u((int)cur.mask) >> gx) & 0x55;
        const bool end = b == count - 1;
        const bool endz = end || u(cur.zo) != u(nxt.zo), endy = endz || u(cur.yo) != u(nxt.yo);
        if (mask) {  // pass x
            double X[RG][KS], f[T][KS], t1[RG][T];
            load_a(st + D::A0, X);
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int s = 0; s < KS; s++) f[t][s] = st[xb[t] + s];
#pragma unroll
            for (int r = 0; r < RG; r++)
#pragma unroll
                for (int t = 0; t < T; t++) t1[r][t] = mfma4(X[r][0], f[t][0], 0.0);
#pragma unroll
            for (int s = 1; s < KS; s++)
#pragma unroll
                for (int r = 0; r < RG; r++)
#pragma unroll
                    for (int t = 0; t < T; t++) t1[r][t] = mfma4(X[r][s], f[t][s], t1[r][t]);
            if constexpr (INF) {  // (as above)
#pragma unroll
                for (int p = 0; p < 4; p++)
#pragma unroll
                    for (int r = 0; r < RG; r++)
#pragma unroll
                        for (int t = 0; t < T; t++) U[p][r][t] += (mask >> (2 * p)) & 1 ? t1[r][t] : 0.0;
            } else {
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const double on1 = __hiloint2double((mask >> (2 * p)) & 1 ? 0x3ff00000 : 0, 0);
#pragma unroll
                    for (int r = 0; r < RG; r++)
#pragma unroll
                        for (int t = 0; t < T; t++) U[p][r][t] = fma(t1[r][t], on1, U[p][r][t]);
                }
            }
            umask |= mask;
        }
        if (endy && umask) {
            // pass y: U (rows a, columns (l, j)) -> LDS rows (a, l) of j -> V (rows b, columns (a, l))
            wave_sync();
#pragma unroll
            for (int p = 0; p < 4; p++)
                if ((umask >> (2 * p)) & 1) {
#pragma unroll
                    for (int r = 0; r < RG; r++)
#pragma unroll
                        for (int t = 0; t < T; t++) {
                            Ul[p * S * K * ROW + xu[r][t]] = U[p][r][t];
                            U[p][r][t] = 0.0;
                        }
                }
            wave_sync();
#pragma unroll
            for (int gy = 0; gy < 2; gy++) {
                double Y[RG][KS];
                load_a(st + D::A0 + (1 + gy) * D::A2, Y);
#pragma unroll
                for (int p = gy; p < 4; p += 2)
                    if ((umask >> (2 * p)) & 1) {
                        double v[T][KS];
#pragma unroll
                        for (int t = 0; t < T; t++)
#pragma unroll
                            for (int s = 0; s < KS; s++) v[t][s] = Ul[p * S * K * ROW + yr[t] + s];
                        row_end(v);
#pragma unroll
                        for (int s = 0; s < KS; s++)
#pragma unroll
                            for (int r = 0; r < RG; r++)
#pragma unroll
                                for (int t = 0; t < T; t++) V[p][r][t] = mfma4(Y[r][s], v[t][s], V[p][r][t]);
                    }
            }
            vmask |= umask;
            umask = 0;
        }
        if (endz && vmask) {
            // pass z: V (rows b, columns (a, l)) -> LDS rows (b, a) of l -> W (rows c, columns (b, a))
            __syncthreads();  // (the rows of U and V share their memory)
#pragma unroll
            for (int p = 0; p < 4; p++)
                if ((vmask >> (2 * p)) & 1) {
#pragma unroll
                    for (int r = 0; r < RG; r++)
#pragma unroll
                        for (int t = 0; t < T; t++) {
                            Vl[p * K2 * ROW + yv[r][t]] = V[p][r][t];
                            V[p][r][t] = 0.0;
                        }
                }
            __syncthreads();
            const double w = cur.w;
#pragma unroll
            for (int gz = 0; gz < 2; gz++) {
                double Z[RG][KS];
                load_a(st + D::A0 + (3 + gz) * D::A2, Z);
#pragma unroll
                for (int r = 0; r < RG; r++)
#pragma unroll
                    for (int s = 0; s < KS; s++) Z[r][s] *= w;
#pragma unroll
                for (int p = 2 * gz; p < 2 * gz + 2; p++)
                    if ((vmask >> (2 * p)) & 1) {
                        double v[T][KS];
#pragma unroll
                        for (int t = 0; t < T; t++)
#pragma unroll
                            for (int s = 0; s < KS; s++) v[t][s] = Vl[(p * K2 + zc[t]) * ROW + ib + s];
                        row_end(v);
#pragma unroll
                        for (int s = 0; s < KS; s++)
#pragma unroll
                            for (int r = 0; r < RG; r++)
#pragma unroll
                                for (int t = 0; t < T; t++) W[p][r][t] = mfma4(Z[r][s], v[t][s], W[p][r][t]);
                    }
            }
            vmask = 0;
        }
        store(stage[(b + 1) & 1]);
        __syncthreads();
    }
    double *dst = slots + (size_t)task.slot * 8 * K3 + gx * K3;
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int r = 0; r < RG; r++)
#pragma unroll
            for (int t = 0; t < T; t++) {
                const int c = 4 * r + kq;
                if (zok[t] && c < K) dst[2 * p * K3 + c * K2 + zc[t]] = W[p][r][t];
            }
}

template <int K>
static void launch_slices64(bool infinite, hipStream_t s, int ntask, const TaskSummary *sum, int nt,
                            const SliceTask *tasks, const WorkItem *work, const JobTab *jobs, const Slice *slices,
                            const double *genPool, double *slots, unsigned long long *ts) {
    if constexpr (F64<K>::G <= 2) {
        const auto kern = infinite ? k_contract_slices64<K, true> : k_contract_slices64<K, false>;
        hipLaunchKernelGGL(kern, dim3(nt + (ts ? 1 : 0)), dim3(F64<K>::NA * 64), 0, s, ntask, sum, tasks, work, jobs,
                           slices, genPool, slots, ts);
    } else {
        const auto kern = infinite ? k_contract_slices64w<K, true> : k_contract_slices64w<K, false>;
        hipLaunchKernelGGL(kern, dim3((nt + 7) / 8 * 16 + (ts ? 1 : 0)), dim3(Wide<K>::NT), 0, s, ntask, sum, tasks,
                           work, jobs, slices, genPool, slots, ts);
    }
}

hipError_t launch_contract_slices64(hipStream_t s, int K, bool infinite, int ntask, const TaskSummary *sum, int grid,
                                    const SliceTask *tasks, const WorkItem *work, const JobTab *jobs,
                                    const Slice *slices, const double *genPool, double *slots,
                                    unsigned long long *ts) {
    const int nt = sum ? grid : ntask;
    if (nt <= 0) return hipSuccess;
    MWG_DISPATCH_K(K, (launch_slices64<KK>(infinite, s, ntask, sum, nt, tasks, work, jobs, slices, genPool, slots, ts)));
    return hipGetLastError();
}

}  // namespace mwg
