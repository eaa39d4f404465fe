// HIP kernels of the MI355X multiwavelet apply (gfx950, wave64).
//
// Coefficient layout of a node: 8 components x K^3 FP64 (K = k+1), component bit
// 0 = x, 1 = y, 2 = z (0 = scaling), index (iz*K + iy)*K + ix inside a component.
// Two-scale transforms work on the interleaved (2K)^3 tensor whose per-dimension
// index is bit*K + i; each 1D pass multiplies every line of 2K values in place.
#include "mwg_kernels.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <climits>
#include <cmath>

namespace mwg {

// sum over the block of one value per thread, same order every call (all threads get it)
__device__ inline double block_sum_256(double v, double *wsum) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    return (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
}

// ----------------------------------------------------------------- operator blocks

// Scaling-scaling block of one unit Gaussian exp(-b (delta + u - v)^2) at cell scale m:
// t[i][j] = pre * int_{-1}^{1} exp(-b (delta+z)^2) C_ij(z) dz, C_ij(z) = int phi_i(u) phi_j(u - z) du,
// by moments: t[i][j] = pre * sum_h sum_p ccoef[h][i][j][p] M_h[p] with
// M_h[p] = int_half exp(-b (delta+z)^2) L_p(t(z)) dz on 24-point Gauss-Legendre panels of width
// <= 0.5/sqrt(b) around the peak.
// One wave per block: lanes take quadrature points independently and keep the 2 x 2K
// moments in registers; one wave reduction, then the K^2 entries.
template <int K>
__global__ void __launch_bounds__(64) k_tblock_mom(int n, const int *item_term, const long long *item_delta,
                                                   const double *bvals, const double *pres, const double *ccoef,
                                                   const double *gx, const double *gw, double *out) {
    const int it = blockIdx.x;
    if (it >= n) return;
    constexpr int P = 2 * K, K2 = K * K;
    __shared__ double Ms[2 * P];
    const double b = bvals[item_term[it]], pre = pres[item_term[it]];
    const double delta = (double)item_delta[it];
    const double zc = -delta;
    const double R = sqrt(GAUSS_CUT_D / b);
    const double pw = (b > 4.0) ? 0.5 / sqrt(b) : 0.25;
    double M[2][P];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int p = 0; p < P; p++) M[h][p] = 0.0;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const double lo = half == 0 ? -1.0 : 0.0, hi = half == 0 ? 0.0 : 1.0;
        const double a0 = fmax(lo, zc - R), a1 = fmin(hi, zc + R);
        if (a1 <= a0) continue;
        int np = (int)ceil((a1 - a0) / pw);
        if (np < 1) np = 1;
        const double ph = (a1 - a0) / np;
        for (int e = threadIdx.x; e < np * 24; e += 64) {
            const int pnl = e / 24, q = e % 24;
            const double z = a0 + pnl * ph + ph * gx[q];
            const double g = exp(-b * (delta + z) * (delta + z)) * ph * gw[q];
            const double x = 2.0 * (z - lo) - 1.0;
            double p0 = 1.0, p1 = x;
            M[half][0] += g;
            if (P > 1) M[half][1] += g * sqrt(3.0) * x;
#pragma unroll
            for (int k = 2; k < P; k++) {
                const double p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
                p0 = p1;
                p1 = p2;
                M[half][k] += g * sqrt(2.0 * k + 1.0) * p2;
            }
        }
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int p = 0; p < P; p++) {
            double v = M[h][p];
            for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
            if (threadIdx.x == 0) Ms[h * P + p] = v;
        }
    __syncthreads();
    for (int e = threadIdx.x; e < K2; e += 64) {
        double t = 0.0;
        for (int h = 0; h < 2; h++) {
            const double *c = ccoef + ((size_t)h * K2 + e) * P;
            for (int p = 0; p < P; p++) t += c[p] * Ms[h * P + p];
        }
        out[(size_t)it * K2 + e] = t * pre;
    }
}

// NS blocks from the child-scale scaling blocks: R = W M W^T with
// M = [[t(2d), t(2d-1)], [t(2d+1), t(2d)]]; type = 2*gt_bit + ft_bit.  The 4 block norms of
// each translation, and the blocks themselves, go to their group's arrays.
__global__ void k_nsblocks(long long first, NSItems items, const double *t1, const double *W, int K) {
    const long long it = first + blockIdx.x;
    const NSOut o = items.outs[items.grp[it]];
    const size_t row = (size_t)(it - o.first);
    const int N = 2 * K, K2 = K * K, tid = threadIdx.x, nt = blockDim.x;
    __shared__ double Ms[4 * MAXK * MAXK], R1[4 * MAXK * MAXK], Ws[4 * MAXK * MAXK];
    __shared__ double red[4][256];
    const long long d = items.delta[it];
    const int row0 = items.row0[it], tlo = items.tlo[it], thi = items.thi[it];
    for (int e = tid; e < N * N; e += nt) Ws[e] = W[e];
    for (int e = tid; e < N * N; e += nt) {
        const int r = e / N, c = e % N;
        const int a = r / K, i = r % K, bb = c / K, j = c % K;
        const long long dd = 2 * d + a - bb;
        double v = 0.0;
        if (dd >= tlo && dd <= thi) v = t1[(size_t)(row0 + (dd - tlo)) * K2 + i * K + j];
        Ms[e] = v;
    }
    __syncthreads();
    for (int e = tid; e < N * N; e += nt) {
        const int i = e / N, j = e % N;
        double s = 0.0;
        for (int l = 0; l < N; l++) s += Ws[i * N + l] * Ms[l * N + j];
        R1[e] = s;
    }
    __syncthreads();
    double part[4] = {0, 0, 0, 0};
    for (int e = tid; e < N * N; e += nt) {
        const int i = e / N, j = e % N;
        double s = 0.0;
        for (int l = 0; l < N; l++) s += R1[i * N + l] * Ws[j * N + l];
        const int gb = i / K, a = i % K, fb = j / K, i2 = j % K;
        const int type = 2 * gb + fb;
        if (o.blocks) o.blocks[(row * 4 + type) * K2 + a * K + i2] = s;
        part[type] += s * s;
    }
    for (int q = 0; q < 4; q++) red[q][tid] = part[q];
    __syncthreads();
    for (int s = nt / 2; s > 0; s >>= 1) {
        if (tid < s)
            for (int q = 0; q < 4; q++) red[q][tid] += red[q][tid + s];
        __syncthreads();
    }
    if (tid < 4) {
        const double v = sqrt(red[tid][0]);
        o.nrm[row * 4 + tid] = v;
        if (o.norms) o.norms[row * 4 + tid] = v;
    }
}

// component norms of a tree's nodes (a workgroup per node, a wave per two components)
__global__ void __launch_bounds__(256) k_norms(int n, const double *coef, double *norm, int K3) {
    const int node = blockIdx.x, lane = threadIdx.x & 63;
    if (node >= n) return;
    const double *p = coef + (size_t)node * 8 * K3;
    for (int c = threadIdx.x >> 6; c < 8; c += 4) {
        double s = 0.0;
        for (int e = lane; e < K3; e += 64) s += p[c * K3 + e] * p[c * K3 + e];
        for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
        if (lane == 0) norm[(size_t)node * 8 + c] = sqrt(s);
    }
}

// Node tables of trees that become an apply's inputs, HASH_BLOCKS workgroups a tree: cleared, then
// every node takes the first free slot from its hash on (the load is at most 1/2).  Built on
// the host and uploaded, a table was 24 to 48 bytes a node and two blocking copies a tree: the
// inputs of a batch of 36 pair potentials took 1.5 ms before the first launch, 0.35 now.
constexpr int HASH_BLOCKS = 8;

__global__ void __launch_bounds__(256) k_hash_clear(const HashItem *items) {
    const DHash h = items[blockIdx.x / HASH_BLOCKS].h;
    for (uint32_t i = (blockIdx.x % HASH_BLOCKS) * 256 + threadIdx.x; i <= h.mask; i += 256 * HASH_BLOCKS) h.keys[i] = 0ull;
}

__global__ void __launch_bounds__(256) k_hash_insert(const HashItem *items, const unsigned long long *keys) {
    const HashItem it = items[blockIdx.x / HASH_BLOCKS];
    for (int i = (blockIdx.x % HASH_BLOCKS) * 256 + threadIdx.x; i < it.n; i += 256 * HASH_BLOCKS) {
        const unsigned long long key = keys[it.first + i], kk = key + 1ull;
        uint32_t q = dkey_hash(key) & it.h.mask;
        for (uint32_t probe = 0; probe <= it.h.mask; probe++) {
            if (atomicCAS(&it.h.keys[q], 0ull, kk) == 0ull) {
                it.h.vals[q] = i;
                break;
            }
            q = (q + 1) & it.h.mask;
        }
    }
}

// several trees' norms into one array (one transfer to the host)
__global__ void __launch_bounds__(256) k_gather(const GatherItem *items, double *dst) {
    const GatherItem it = items[blockIdx.x / HASH_BLOCKS];
    for (int i = (blockIdx.x % HASH_BLOCKS) * 256 + threadIdx.x; i < it.n; i += 256 * HASH_BLOCKS)
        dst[it.first + i] = it.p[i];
}

// Per-pair partial dot products, one workgroup per node pair, the pairs of several tree pairs in one
// launch: the overlaps of four orbitals took ten of them, each with an upload and a wait (an SCF
// step at k = 7 without its export 4.6 ms, 4.3 now).
__global__ void __launch_bounds__(256) k_dot(const DotPair *pairs, int K3, double *part) {
    __shared__ double wsum[4];
    const DotPair p = pairs[blockIdx.x];
    double s = 0.0;
#pragma unroll 8
    for (int e = (int)p.skip0 * K3 + threadIdx.x; e < 8 * K3; e += 256) s += p.a[e] * p.b[e];
    s = block_sum_256(s, wsum);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// node-pair dot products over a fixed grid, one wave per pair (a pair word holds the a node
// in bits 0..30, a flag to skip component 0 in bit 31 and the b node in bits 32..63); every
// block writes its sum to part[blockIdx.x], so part needs no clearing
__global__ void __launch_bounds__(256) k_dot_pairs(int n, const unsigned long long *pairs, const double *A,
                                                   const double *B, int K3, double *part) {
    __shared__ double red[4];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double s = 0.0;
    for (int i = (int)blockIdx.x * 4 + wave; i < n; i += (int)gridDim.x * 4) {
        const unsigned long long p = pairs[i];
        const int ia = (int)(p & 0x7fffffffu), c0 = (int)((p >> 31) & 1u), ib = (int)(p >> 32);
        const double *a = A + (size_t)ia * 8 * K3;
        const double *b = B + (size_t)ib * 8 * K3;
        for (int e = c0 * K3 + lane; e < 8 * K3; e += 64) s += a[e] * b[e];
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// one wave: *res = sum of part[0 .. n)
__global__ void __launch_bounds__(64) k_sum_parts(int n, const double *part, double *res) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 64) s += part[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if (threadIdx.x == 0) *res = s;
}

__global__ void k_scale(size_t n, double *x, double c) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] *= c;
}

// ----------------------------------------------------------------- projection

// Gaussian sums are separable: the children's scaling tensor is a sum of outer
// products of 2K-vectors (one per dimension), and so is its compression.  CH terms at a time: their
// values at the quadrature points (one exponential per thread and round), the vectors from
// these, their compression, then the outer products along z, so that a wave writes whole lines.
// Latency bounds it: launches of the six orbitals of a projection at k = 7 (8 to 296 nodes) 26.5 us on
// average with the values formed anew for each entry of the vectors and lines along x, 24.0 now.
template <int K>
__global__ void __launch_bounds__(256) k_project_gauss(const MulItem *items, ProjGeom geo, DevBasis B, int nterm, const double *coef,
                                                       const double *alpha, const double *center,
                                                       const double *poly, double *out, double *norm,
                                                       double *compact) {
    constexpr int N = 2 * K, K3 = K * K * K;
    constexpr int LPER = (N * N + 255) / 256;  // z-lines (component bits of x and y, y, x) per thread
    constexpr int CH = 8;
    __shared__ double P[CH][3][N], WP[CH][3][N], Ws[N * N], phi[K * K], cf[CH];
    const MulItem it = items[blockIdx.x];
    const int node = it.node, d = it.depth;
    const double hc = geo.sfac * ldexp(1.0, -(geo.n0 + d + 1));
    const double pre = sqrt(hc);
    const int tid = threadIdx.x;
    for (int e = tid; e < N * N; e += 256) Ws[e] = B.W[e];
    for (int e = tid; e < K * K; e += 256) phi[e] = B.phiq[e];
    double acc[LPER][N];
#pragma unroll
    for (int r = 0; r < LPER; r++)
#pragma unroll
        for (int x = 0; x < N; x++) acc[r][x] = 0.0;
    for (int t0 = 0; t0 < nterm; t0 += CH) {
        __syncthreads();
        const int nt = min(CH, nterm - t0);
        for (int e = tid; e < nt * 3 * N; e += 256) {
            const int tt = e / (3 * N), dim = (e / N) % 3, p = e % N, t = t0 + tt;
            const int bit = p / K, q = p % K;
            const int l = dim == 0 ? it.l[0] : dim == 1 ? it.l[1] : it.l[2];
            const double x0 = geo.lo[dim] + hc * (double)(2 * l + bit);
            const double u = x0 + hc * B.qx[q] - center[3 * t + dim];
            double pv = 0.0, up = 1.0;
#pragma unroll
            for (int ee = 0; ee < 5; ee++) {
                pv += poly[15 * t + 5 * dim + ee] * up;
                up *= u;
            }
            WP[tt][dim][p] = pv * exp(-alpha[t] * u * u) * B.qw[q];
            if (e < nt) cf[e] = coef[t0 + e];
        }
        __syncthreads();
        for (int e = tid; e < nt * 3 * N; e += 256) {
            const int tt = e / (3 * N), dim = (e / N) % 3, p = e % N;
            const int bit = p / K, i = p % K;
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < K; q++) s += phi[q * K + i] * WP[tt][dim][bit * K + q];
            P[tt][dim][p] = s * pre;
        }
        __syncthreads();
        for (int e = tid; e < nt * 3 * N; e += 256) {
            const int tt = e / (3 * N), dim = (e / N) % 3, p = e % N;
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < N; q++) s += Ws[p * N + q] * P[tt][dim][q];
            WP[tt][dim][p] = s;
        }
        __syncthreads();
        // the thread's z-lines accumulate the outer products term by term
#pragma unroll 1
        for (int tt = 0; tt < nt; tt++) {
#pragma unroll
            for (int r = 0; r < LPER; r++) {
                const int line = tid + 256 * r;
                if (line < N * N) {
                    const int b = line / (K * K), px = (b & 1) * K + line % K, py = (b >> 1) * K + line / K % K;
                    const double xy = cf[tt] * WP[tt][0][px] * WP[tt][1][py];
#pragma unroll
                    for (int z = 0; z < N; z++) acc[r][z] += xy * WP[tt][2][z];
                }
            }
        }
    }
    __shared__ double wsum[4][8];
    double ss[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int r = 0; r < LPER; r++) {
        const int line = tid + 256 * r;
        if (line < N * N) {
            const int b = line / (K * K);  // neighbours in a wave hold neighbouring (x, y): whole lines are written
            double *dst = out + (size_t)node * 8 * K3 + b * K3 + line % (K * K);
            double s[2] = {0.0, 0.0};
#pragma unroll
            for (int pz = 0; pz < N; pz++) {
                dst[(pz / K) * 4 * K3 + pz % K * K * K] = acc[r][pz];
                s[pz / K] += acc[r][pz] * acc[r][pz];
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (b == q) {
                    ss[q] += s[0];
                    ss[4 + q] += s[1];
                }
        }
    }
    put_norms(ss, wsum, norm + (size_t)node * 8, compact + (size_t)blockIdx.x * 8);
}


// ----------------------------------------------------------------- apply: generated nodes

__device__ inline bool in_box(const short *b, int dx, int dy, int dz) {
    return b[0] >= 0 && abs(dx) <= b[0] && abs(dy) <= b[1] && abs(dz) <= b[2];
}

// bit c (= gt * 8 + ft) set iff the screening box of combo c holds (dx, dy, dz)
__device__ inline unsigned long long combo_mask(const TermTab &tb, int dx, int dy, int dz) {
    const int ax = abs(dx), ay = abs(dy), az = abs(dz);
    if (ax < BM && ay < BM && az < BM) return tb.bm[0][ax] & tb.bm[1][ay] & tb.bm[2][az];
    unsigned long long m = 0;
    for (int c = 0; c < 64; c++)
        if (in_box(tb.box[c], dx, dy, dz)) m |= 1ull << c;
    return m;
}
constexpr unsigned long long FT0_COMBOS = 0x0101010101010101ull;  // the combos with ft = 0

// mark the input nodes that the output nodes need at this depth but the input
// tree does not have (scaling-only "generated" nodes)
// translations cached per output node in LDS (the union box over all terms, cells)
constexpr int FCACHE = 4096;

__device__ inline void gen_insert(const JobTab &J, const GenState &gs, int job, uint64_t key) {
    const unsigned long long kk = (unsigned long long)key + 1ull;
    uint32_t i = dkey_hash(key) & J.genHash.mask;
    for (uint32_t probe = 0; probe <= J.genHash.mask; probe++) {
        unsigned long long old = atomicCAS(&J.genHash.keys[i], 0ull, kk);
        if (old == 0ull) {
            const int idx = atomicAdd(gs.count, 1);
            atomicAdd((unsigned long long *)&gs.tabcnt[4 * job + 3], 1ull);
            if (idx < gs.cap) {
                gs.keys[idx] = key;
                gs.job[idx] = job;
            } else {
                atomicOr(gs.overflow, 1);
            }
            J.genHash.vals[i] = idx;
            return;
        }
        if (old == kk) return;
        i = (i + 1) & J.genHash.mask;
        if (probe == J.genHash.mask) atomicOr(gs.overflow, 2);
    }
}

__device__ inline int wave_incl_scan(int v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    return v;
}

// marks one translation of an output node, if the box holds it and the input does not
__device__ __forceinline__ void gen_mark_one(const WorkItem &wi, const JobTab &J, const GenState &gs, int dx, int dy,
                                             int dz) {
    const int fx = wi.l[0] - dx, fy = wi.l[1] - dy, fz = wi.l[2] - dz;
    if (fx < 0 || fy < 0 || fz < 0 || fx >= J.lmax[0] || fy >= J.lmax[1] || fz >= J.lmax[2]) return;
    const uint64_t key = dnode_key(J.depth, fx, fy, fz);
    if (dhash_find(J.inHash, key) < 0) gen_insert(J, gs, wi.job, key);
}

// Walks the (term, |delta|) candidates of the ft = 0 boxes (a box is symmetric in every
// dimension): the |delta| that some term needs are first collected in an LDS bitmap over the job's
// union box, so that each input position is probed once.  A union box beyond the bitmap is
// walked candidate by candidate.  One workgroup per node; its time is a chain of reads, so the fewer
// rounds the better: over every signed delta of every term it was 9.7 us a launch for a Poisson
// apply at k = 5 and 61 for the 36 pair potentials of an exchange step, 7.4 and 53 over |delta|.
__device__ __forceinline__ void gen_mark_node(int item, const WorkItem *work, const JobTab *jobs,
                                              const TermTab *tabs, const GenState &gs) {
    const WorkItem wi = work[item];
    const JobTab &J = jobs[wi.job];
    __shared__ int start[257];
    __shared__ short4 ub0[256];
    __shared__ unsigned need[FCACHE / 32];
    const int ux = J.ubox[0], uy = J.ubox[1], uz = J.ubox[2];
    if (ux < 0) return;  // (no term has a box)
    const int nx = 2 * ux + 1, ny = 2 * uy + 1, nz = 2 * uz + 1, ax = ux + 1, ay = uy + 1;
    const bool cached = nx * ny * nz <= FCACHE;
    if (threadIdx.x < 64) {  // the terms' boxes and the prefix of their candidates
        int carry = 0;
        for (int base = 0; base < J.ntab; base += 64) {
            const int t = base + (int)threadIdx.x;
            int v = 0;
            if (t < J.ntab) {
                const TermTab &tb = tabs[J.tab0 + t];
                const short4 u = make_short4(tb.ub0[0], tb.ub0[1], tb.ub0[2], 0);
                ub0[t] = u;
                v = u.x < 0 ? 0 : (u.x + 1) * (u.y + 1) * (u.z + 1);
            }
            const int incl = wave_incl_scan(v);
            if (t < J.ntab) start[t] = carry + incl - v;
            carry += __shfl(incl, 63, 64);
        }
        if (threadIdx.x == 0) start[J.ntab] = carry;
    } else {
        for (int q = threadIdx.x - 64; q < FCACHE / 32; q += blockDim.x - 64) need[q] = 0u;
    }
    __syncthreads();
    const int total = start[J.ntab];
    for (int k = threadIdx.x; k < total; k += blockDim.x) {
        int lo = 0, hi = J.ntab - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (start[mid] <= k) lo = mid;
            else hi = mid - 1;
        }
        const short4 u = ub0[lo];
        const int c = k - start[lo], wx = u.x + 1, wy = u.y + 1;
        const int dx = c % wx, dy = (c / wx) % wy, dz = c / (wx * wy);
        if (!(combo_mask(tabs[J.tab0 + lo], dx, dy, dz) & FT0_COMBOS)) continue;
        if (cached) {
            const int cell = (dz * ay + dy) * ax + dx;
            atomicOr(&need[cell >> 5], 1u << (cell & 31));
            continue;
        }
        for (int sgn = 0; sgn < 8; sgn++) {
            if (((sgn & 1) && !dx) || ((sgn & 2) && !dy) || ((sgn & 4) && !dz)) continue;
            gen_mark_one(wi, J, gs, (sgn & 1) ? -dx : dx, (sgn & 2) ? -dy : dy, (sgn & 4) ? -dz : dz);
        }
    }
    if (!cached) return;
    __syncthreads();
    for (int cell = threadIdx.x; cell < nx * ny * nz; cell += blockDim.x) {
        const int dx = cell % nx - ux, dy = (cell / nx) % ny - uy, dz = cell / (nx * ny) - uz;
        const int c = (abs(dz) * ay + abs(dy)) * ax + abs(dx);
        if ((need[c >> 5] >> (c & 31)) & 1u) gen_mark_one(wi, J, gs, dx, dy, dz);
    }
}

// Items 0 .. total - 1 of a workgroup-per-item kernel: item blockIdx.x first, then
// grid-stride, or (queue) the items beyond the grid taken one at a time from a zeroed
// counter, so that workgroups that drew cheap items take more of them.  Workgroups without
// an item leave at once; the others leave once the counter has passed total.
template <class F>
__device__ __forceinline__ void for_items(int total, int *queue, F f) {
    if ((int)blockIdx.x >= total) return;
    f((int)blockIdx.x);
    if (total <= (int)gridDim.x) return;
    __syncthreads();  // (LDS reused by the next item)
    if (!queue) {
        for (int b = blockIdx.x + gridDim.x; b < total; b += gridDim.x) {
            f(b);
            __syncthreads();
        }
        return;
    }
    __shared__ int s_item;
    while (true) {
        if (threadIdx.x == 0) s_item = (int)gridDim.x + atomicAdd(queue, 1);
        __syncthreads();
        const int b = s_item;
        __syncthreads();
        if (b >= total) break;
        f(b);
        __syncthreads();
    }
}

// one workgroup per work node (nwp: the node count on the device)
__global__ void __launch_bounds__(256) k_gen_mark(int nw, const int *nwp, int *queue, const WorkItem *work,
                                                  const JobTab *jobs, const TermTab *tabs, GenState gs) {
    const int n = nwp ? *nwp : nw;
    for_items(n, queue, [&](int i) { gen_mark_node(i, work, jobs, tabs, gs); });
}

// Per output node, the input node (>= 0), generated node (-(g+1)) or nothing
// (INT_MIN) at every translation of the union box over all terms, cached in LDS so
// that each term's loop reads the cache instead of probing the hash tables again.
struct FCache {
    int ux, uy, uz;  // half-widths, ux < 0: no cache (box too large)
};

__device__ inline int probe_f(const JobTab &J, const GenState &gs, int fx, int fy, int fz) {
    if (fx < 0 || fy < 0 || fz < 0 || fx >= J.lmax[0] || fy >= J.lmax[1] || fz >= J.lmax[2]) return INT_MIN;
    const uint64_t key = dnode_key(J.depth, fx, fy, fz);
    const int f = dhash_find(J.inHash, key);
    if (f >= 0) return f;
    const int gi = dhash_find(J.genHash, key);
    return gi >= 0 ? -(gi + 1) : INT_MIN;
}

__device__ inline FCache fill_fcache(int *cache, const WorkItem &wi, const JobTab &J, const TermTab *tabs,
                                     const GenState &gs) {
    const int ux = J.ubox[0], uy = J.ubox[1], uz = J.ubox[2];
    FCache fc{ux, uy, uz};
    (void)tabs;
    if (ux < 0) return fc;
    const int nx = 2 * ux + 1, ny = 2 * uy + 1, nz = 2 * uz + 1;
    if (nx * ny * nz > FCACHE) {
        fc.ux = -1;
        return fc;
    }
    for (int c = threadIdx.x; c < nx * ny * nz; c += blockDim.x) {
        const int dx = c % nx - ux, dy = (c / nx) % ny - uy, dz = c / (nx * ny) - uz;
        cache[c] = probe_f(J, gs, wi.l[0] - dx, wi.l[1] - dy, wi.l[2] - dz);
    }
    __syncthreads();
    return fc;
}

__device__ inline int lookup_f(const int *cache, const FCache &fc, const WorkItem &wi, const JobTab &J,
                               const GenState &gs, int dx, int dy, int dz) {
    if (fc.ux >= 0)
        return cache[((dz + fc.uz) * (2 * fc.uy + 1) + (dy + fc.uy)) * (2 * fc.ux + 1) + (dx + fc.ux)];
    return probe_f(J, gs, wi.l[0] - dx, wi.l[1] - dy, wi.l[2] - dz);
}


// The screening of one candidate (term, delta, input node): bit gt of surv[ft] is set when
// the combination is inside its screening box (bit 8 gt + ft of cm) and its bound
// (((|w| ||X_tx||) ||Y_ty||) ||Z_tz||) ||f_ft|| exceeds thr; maxb[ft] is the largest such
// bound.  The products are formed in that order, as in the oracle's screening, so the
// decisions are the same to the bit.  Unrolled and free of branches: the lanes of a wave
// hold different candidates.
template <bool MAXB>
__device__ inline void screen_candidate(double aw, const double *nx, const double *ny, const double *nz,
                                        const double *fn, unsigned long long cm, double thr, unsigned (&surv)[8],
                                        double (&maxb)[8]) {
    double pxy[4][4];
#pragma unroll
    for (int tx = 0; tx < 4; tx++) {
        const double ax = aw * nx[tx];
#pragma unroll
        for (int ty = 0; ty < 4; ty++) pxy[tx][ty] = ax * ny[ty];
    }
#pragma unroll
    for (int ft = 0; ft < 8; ft++) {
        unsigned sv = 0u;
        double mb = 0.0;
#pragma unroll
        for (int gt = 0; gt < 8; gt++) {
            const int tx = 2 * (gt & 1) + (ft & 1);
            const int ty = 2 * ((gt >> 1) & 1) + ((ft >> 1) & 1);
            const int tz = 2 * ((gt >> 2) & 1) + ((ft >> 2) & 1);
            const double b = (pxy[tx][ty] * nz[tz]) * fn[ft];
            const bool ok = ((cm >> (8 * gt + ft)) & 1ull) && b > thr;
            sv |= (unsigned)ok << gt;
            if (MAXB) mb = ok ? fmax(mb, b) : mb;
        }
        surv[ft] = sv;
        maxb[ft] = mb;
    }
}

// Flattened candidate walk: every (term, delta) cell of the job's screened boxes is
// one candidate, spread over all threads of the block (term prefix sums in LDS).
// For each candidate with an input node the visitor gets the 12 operator norms
// (4 block types per dimension) and the input component norms.
struct CandTerms {
    int start[257];
};

__device__ inline void term_prefix(CandTerms &ct, const JobTab &J, const TermTab *tabs) {
    for (int t = threadIdx.x; t <= J.ntab; t += blockDim.x) ct.start[t] = J.pre[t];
    __syncthreads();
    (void)tabs;
}

// the candidates of part of nparts workgroups that share an output node
__device__ inline void part_range(int total, int part, int nparts, int &k0, int &k1) {
    k0 = (int)((long long)total * part / nparts);
    k1 = (int)((long long)total * (part + 1) / nparts);
}

template <class Visit>
__device__ inline void walk_candidates(const CandTerms &ct, const int *fcache, const FCache &fc, const WorkItem &wi,
                                       const JobTab &J, const TermTab *tabs, const GenState &gs, int k0, int k1,
                                       Visit &&visit) {
    for (int k = k0 + threadIdx.x; k < k1; k += blockDim.x) {
        int lo = 0, hi = J.ntab - 1;  // last t with start[t] <= k
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (ct.start[mid] <= k) lo = mid;
            else hi = mid - 1;
        }
        const int t = lo;
        const TermTab &tb = tabs[J.tab0 + t];
        const int c = k - ct.start[t];
        const int ux = tb.ub[0], uy = tb.ub[1], uz = tb.ub[2];
        const int dx = c % (2 * ux + 1) - ux;
        const int dy = (c / (2 * ux + 1)) % (2 * uy + 1) - uy;
        const int dz = c / ((2 * ux + 1) * (2 * uy + 1)) - uz;
        const int f = lookup_f(fcache, fc, wi, J, gs, dx, dy, dz);
        if (f == INT_MIN) continue;
        double fn[8];
        if (f >= 0) {
            for (int q = 0; q < 8; q++) fn[q] = J.inNorm[(size_t)f * 8 + q];
        } else {
            // an entry past the allocated pool (its count is redone after the pool grows)
            fn[0] = -f - 1 < gs.pcap ? gs.norm[-f - 1] : 0.0;
            for (int q = 1; q < 8; q++) fn[q] = 0.0;  // (no wavelet part: no bound above thr >= 0)
        }
        const double *nrm = J.operNorms + tb.nrm;
        double nx[4], ny[4], nz[4];
        for (int q = 0; q < 4; q++) {
            nx[q] = nrm[(dx + tb.band) * 4 + q];
            ny[q] = nrm[(dy + tb.band) * 4 + q];
            nz[q] = nrm[(dz + tb.band) * 4 + q];
        }
        visit(k, t, tb, dx, dy, dz, f, fn, nx, ny, nz);
    }
}

// ----------------------------------------------------------------- apply: screening boxes

// One wavefront per (table, term); lane = combination gt*8+ft.  For the bound
// |w| F_ft prod_d ||X_d|| of the combination to exceed thr somewhere, each dimension's
// translation must stay inside the largest m with env_type[m] > thr / (|w| F_ft prod of
// the other two dimensions' largest norms); env is non-increasing in m.
__device__ inline int wave_max_int(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ inline double wave_max_double(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

constexpr int ENV_LDS = 512;  // envelope entries per type staged in LDS
// the tuple threshold of a device-loop job: the host loop's expression,
// SCREEN_REL prec sqrt(||g||^2 / terms), 0 before any norm
__device__ inline double loop_thr(const LoopJob &L, int nterms) {
    const double gsq = L.gsq;
    return gsq > 0.0 ? SCREEN_REL * L.prec * sqrt(gsq / (double)nterms) : 0.0;
}

__global__ void __launch_bounds__(64) k_job_boxes(int nbj, const BoxJob *bjs, TermTab *tabs, double *tbmax,
                                                  int max_terms, LoopInit li) {
    const int jb = blockIdx.x, t = blockIdx.y;
    if (jb >= nbj) return;
    const BoxJob &B = bjs[jb];
    if (t >= B.nterms) return;
    const double thr = li.lj ? loop_thr(li.lj[jb], B.nterms) : B.thr;
    const LevTerm &lt = B.terms[t];  // (read in place: maxn is indexed by the lane's types)
    TermTab *tb = tabs + B.tab0 + t;
    const int c = threadIdx.x, gt = c >> 3, ft = c & 7;
    // the term's norm envelopes (4 types x (band + 1)) staged in LDS for the searches
    __shared__ double senv[4 * ENV_LDS];
    const int ne = 4 * (lt.band + 1);
    const bool env_lds = ne <= 4 * ENV_LDS;
    if (env_lds)
        for (int e = c; e < ne; e += 64) senv[e] = B.env[lt.env + e];
    __syncthreads();
    const double *envb = env_lds ? senv : B.env + lt.env;
    int m3[3] = {-1, -1, -1};
    double full = 0.0;
    bool ok = false;
    if (lt.active && !(B.depth > 0 && c == 0)) {
        const double F = B.F[ft];
        if (F > 0.0) {
            int ty[3];
#pragma unroll
            for (int q = 0; q < 3; q++) ty[q] = 2 * ((gt >> q) & 1) + ((ft >> q) & 1);
            const double base = fabs(lt.w) * F;
            const double f3 = base * lt.maxn[ty[0]] * lt.maxn[ty[1]] * lt.maxn[ty[2]];
            if (f3 > thr) {
                full = f3;
                ok = true;
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    double other = base;
#pragma unroll
                    for (int q2 = 0; q2 < 3; q2++)
                        if (q2 != q) other *= lt.maxn[ty[q2]];
                    const double tau = thr / other;
                    const double *env = envb + (long long)ty[q] * (lt.band + 1);
                    int m = -1;
                    if (env[0] > tau) {
                        int lo = 0, hi = lt.band;
                        while (lo < hi) {
                            const int mid = (lo + hi + 1) / 2;
                            if (env[mid] > tau) lo = mid;
                            else hi = mid - 1;
                        }
                        m = lo;
                    }
                    if (m < 0) ok = false;
                    m3[q] = m;
                }
            }
        }
    }
    int u[3], u0[3];
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const short v = ok ? (short)m3[q] : (short)-1;
        tb->box[c][q] = v;
        u[q] = wave_max_int(v);
        u0[q] = wave_max_int(ft == 0 ? v : -1);
        for (int m = 0; m < BM; m++) {
            const unsigned long long b = __ballot(ok && m3[q] >= m);
            if (c == 0) tb->bm[q][m] = b;
        }
    }
    const double bmax = wave_max_double(full);
    if (c == 0) {
        tb->w = lt.w;
        tb->blk = lt.blk;
        tb->nrm = lt.nrm;
        tb->band = lt.band;
        for (int q = 0; q < 3; q++) {
            tb->ub[q] = (short)u[q];
            tb->ub0[q] = (short)u0[q];
        }
        tbmax[(size_t)jb * max_terms + t] = bmax;
    }
}

// Per table, one wave: the FP64 routing bound (mixed mode: slices whose bound exceeds
// it run in FP64; above the roots a fixed multiple of the screening threshold, on the
// roots (no screening) a fraction of the largest bound of the table), the union box of
// the terms, and the prefix sums over terms of the candidate counts of the union boxes
// ub (the work-list kernels split their walks by these).

__global__ void __launch_bounds__(64) k_job_route(int nbj, const BoxJob *bjs, const TermTab *tabs,
                                                  const double *tbmax, int max_terms, JobTab *jobs, int *pre,
                                                  int *gen_overflow, LoopInit li) {
    const int jb = blockIdx.x;
    if (jb >= nbj) return;
    if (jb == 0 && threadIdx.x == 0) *gen_overflow = 0;  // the iteration's generated-table flag
    const BoxJob &B = bjs[jb];
    const int lane = threadIdx.x;
    const double thr = li.lj ? loop_thr(li.lj[jb], B.nterms) : B.thr;
    if (li.lj) {  // the device loop's iteration start (before any kernel that uses these)
        if (lane == 0) jobs[B.jt].thr = thr;
        if (lane < 4) li.tabcnt[4 * (size_t)jb + lane] = 0;
        if (jb == 0 && lane == 0) {
            li.ctl->genFirst = *(volatile const int *)li.gen_count;
            for (int q = 0; q < 4; q++) li.ctl->queue[q] = 0;
            li.ts[0] = li.ts[1] = 0ull;
        }
    }
    double m = 0.0;
    int ux = -1, uy = -1, uz = -1, carry = 0;
    for (int base = 0; base < B.nterms; base += 64) {
        const int t = base + lane;
        int v = 0;
        if (t < B.nterms) {
            m = fmax(m, tbmax[(size_t)jb * max_terms + t]);
            const TermTab &tb = tabs[B.tab0 + t];
            if (tb.ub[0] >= 0) {
                v = (2 * tb.ub[0] + 1) * (2 * tb.ub[1] + 1) * (2 * tb.ub[2] + 1);
                ux = max(ux, (int)tb.ub[0]);
                uy = max(uy, (int)tb.ub[1]);
                uz = max(uz, (int)tb.ub[2]);
            }
        }
        const int incl = wave_incl_scan(v);
        if (t < B.nterms) pre[B.pre_off + t] = carry + incl - v;
        carry += __shfl(incl, 63, 64);
    }
    m = wave_max_double(m);
    ux = wave_max_int(ux);
    uy = wave_max_int(uy);
    uz = wave_max_int(uz);
    if (lane == 0) {
        pre[B.pre_off + B.nterms] = carry;
        JobTab &J = jobs[B.jt];
        J.route = thr > 0.0 ? ROUTE_FP64 * thr : ROUTE_ROOT * m;
        J.ubox[0] = ux;
        J.ubox[1] = uy;
        J.ubox[2] = uz;
    }
}

// ----------------------------------------------------------------- apply: work list

// Enumerates, for one output node, every (term, delta, ft, gt) candidate inside the screened
// boxes and keeps the combinations whose bound |w| prod_d ||X_d|| ||f_ft|| exceeds the job
// threshold; the surviving gt of a (term, delta, ft) make one slice.
//   mode 0 counts the slices of the part (and the job's tuples);
//   mode 1 writes them from the node's start (from the schedule) + the part's offset, and
//          the node's tasks (part 0).
// The contraction shares its y and z passes between neighbours in the list, so the slices of
// a term go in the order (dz, ft_z, dy, ft_y, dx, ft_x).  Candidates come in the order (term, dz,
// dy, dx), every one with its 8 ft: ENUM_CHUNK of them at a time are screened into LDS (8 masks
// each), their slices counted per (candidate, ft_z, ft_y) in the order of the list, and the
// prefix of these counts gives every slice its place.  (A plane (term, dz) that a chunk or a
// part cuts is ordered within each piece: the runs are shorter there.)
constexpr int ENUM_CHUNK = 1024;

// the node's tasks: at most chunk slices each (slot = task index)
__device__ __forceinline__ void emit_tasks(int g, long long start, int count, int chunk, int task0, SliceTask *tasks) {
    const int n = (count + chunk - 1) / chunk;
    for (int h = threadIdx.x; h < n; h += blockDim.x)
        tasks[task0 + h] = SliceTask{start + (long long)h * chunk, min(chunk, count - h * chunk), g, task0 + h};
}

__device__ inline int block_sum_256i(int v, int *wsum) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    return (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
}

template <int MODE>
__device__ __forceinline__ void enum_node(int g, int part, int nparts, int K2, const WorkItem *work,
                                          const JobTab *jobs, const TermTab *tabs, const GenState &gs, int *seg_total,
                                          const long long *seg_ofs, Slice *out, const TaskSummary *sum,
                                          const NodeSched *nodes, SliceTask *tasks) {
    const WorkItem wi = work[g];
    const JobTab &J = jobs[wi.job];
    __shared__ int fcache[FCACHE];
    __shared__ CandTerms ct;
    __shared__ int wsum[4];
    __shared__ uint2 smask[MODE == 1 ? ENUM_CHUNK : 1];
    __shared__ __align__(16) unsigned short place[MODE == 1 ? 4 * ENUM_CHUNK : 1];
    const FCache fc = fill_fcache(fcache, wi, J, tabs, gs);
    term_prefix(ct, J, tabs);
    int k0, k1;
    part_range(ct.start[J.ntab], part, nparts, k0, k1);
    if (MODE == 0) {
        int ns = 0, nt = 0;
        walk_candidates(ct, fcache, fc, wi, J, tabs, gs, k0, k1,
                        [&](int k, int t, const TermTab &tb, int dx, int dy, int dz, int f, const double *fn,
                            const double *nx, const double *ny, const double *nz) {
                            unsigned surv[8];
                            double maxb[8];
                            screen_candidate<false>(fabs(tb.w), nx, ny, nz, fn, combo_mask(tb, dx, dy, dz), J.thr, surv,
                                                    maxb);
#pragma unroll
                            for (int ft = 0; ft < 8; ft++) {
                                ns += surv[ft] ? 1 : 0;
                                nt += __popc(surv[ft]);
                            }
                        });
        ns = block_sum_256i(ns, wsum);
        nt = block_sum_256i(nt, wsum);
        if (threadIdx.x == 0) {
            seg_total[(size_t)g * nparts + part] = ns;
            if (nt) atomicAdd((unsigned long long *)&gs.tabcnt[4 * wi.job], (unsigned long long)nt);
        }
        return;
    }
    const NodeSched nd = nodes[g];
    if (part == 0) emit_tasks(g, nd.start64, nd.count64, sum->chunk, nd.task64, tasks);
    long long base = nd.start64 + (nparts > 1 ? seg_ofs[(size_t)g * nparts + part] : 0);
    for (int kc = k0; kc < k1; kc += ENUM_CHUNK) {
        const int ke = min(k1, kc + ENUM_CHUNK), n = ke - kc;
        for (int q = threadIdx.x; q < n; q += 256) smask[q] = make_uint2(0u, 0u);
        for (int q = threadIdx.x; q < ENUM_CHUNK / 2; q += 256) ((uint4 *)place)[q] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        walk_candidates(ct, fcache, fc, wi, J, tabs, gs, kc, ke,
                        [&](int k, int t, const TermTab &tb, int dx, int dy, int dz, int f, const double *fn,
                            const double *nx, const double *ny, const double *nz) {
                            unsigned surv[8];
                            double maxb[8];
                            screen_candidate<false>(fabs(tb.w), nx, ny, nz, fn, combo_mask(tb, dx, dy, dz), J.thr, surv,
                                                    maxb);
                            smask[k - kc] = make_uint2(surv[0] | surv[1] << 8 | surv[2] << 16 | surv[3] << 24,
                                                       surv[4] | surv[5] << 8 | surv[6] << 16 | surv[7] << 24);
                        });
        // a candidate's places: f(ft_z, ft_y) -> index of its counter in the order of the list
        auto visit = [&](auto &&fn) {
            for (int k = kc + threadIdx.x; k < ke; k += 256) {
                const uint2 m = smask[k - kc];
                if (!(m.x | m.y)) continue;
                int lo = 0, hi = J.ntab - 1;
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (ct.start[mid] <= k) lo = mid;
                    else hi = mid - 1;
                }
                const TermTab &tb = tabs[J.tab0 + lo];
                const int nx = 2 * tb.ub[0] + 1, ny = 2 * tb.ub[1] + 1;
                const int c = k - ct.start[lo], iz = c / (nx * ny), e = c - iz * nx * ny, iy = e / nx;
                const int ps = ct.start[lo] + iz * nx * ny;  // the plane's and the row's first candidates
                const int a = max(ps, kc), b = min(ps + nx * ny, ke);
                const int ra = max(ps + iy * nx, a), rb = min(ps + (iy + 1) * nx, b);
                const int p0 = 4 * (a - kc) + 2 * (ra - a) + (k - ra);
                fn(k, m, tb, e - iy * nx - tb.ub[0], iy - tb.ub[1], iz - tb.ub[2], p0, 2 * (b - a), rb - ra);
            }
        };
        __syncthreads();
        visit([&](int k, const uint2 m, const TermTab &tb, int dx, int dy, int dz, int p0, int sz, int sy) {
#pragma unroll
            for (int c = 0; c < 4; c++) {  // c = ft_y + 2 ft_z: the bytes ft = 2 c, 2 c + 1
                const unsigned w = (c < 2 ? m.x : m.y) >> (16 * (c & 1));
                place[p0 + (c >> 1) * sz + (c & 1) * sy] = (unsigned short)(((w & 0xffu) ? 1 : 0) + ((w & 0xff00u) ? 1 : 0));
            }
        });
        __syncthreads();
        // exclusive prefix of the counters: 16 of them per thread
        constexpr int PER = 4 * ENUM_CHUNK / 256;
        unsigned short v[PER];
#pragma unroll
        for (int q = 0; q < PER; q++) v[q] = place[threadIdx.x * PER + q];
        int tsum = 0;
#pragma unroll
        for (int q = 0; q < PER; q++) tsum += v[q];
        const int incl = wave_incl_scan(tsum);
        if ((threadIdx.x & 63) == 63) wsum[threadIdx.x >> 6] = incl;
        __syncthreads();
        int run = incl - tsum, total = 0;
        for (int w = 0; w < 4; w++) {
            if (w < (int)(threadIdx.x >> 6)) run += wsum[w];
            total += wsum[w];
        }
#pragma unroll
        for (int q = 0; q < PER; q++) {
            place[threadIdx.x * PER + q] = (unsigned short)run;
            run += v[q];
        }
        __syncthreads();
        visit([&](int k, const uint2 m, const TermTab &tb, int dx, int dy, int dz, int p0, int sz, int sy) {
            const int f = lookup_f(fcache, fc, wi, J, gs, dx, dy, dz);
            const unsigned long long wb = (unsigned long long)__double_as_longlong(tb.w);
            const int blk = (int)(tb.blk / K2);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const unsigned w2 = (c < 2 ? m.x : m.y) >> (16 * (c & 1));
                if (!(w2 & 0xffffu)) continue;
                Slice *dst = out + base + place[p0 + (c >> 1) * sz + (c & 1) * sy];
#pragma unroll
                for (int fx = 0; fx < 2; fx++) {
                    const unsigned surv = (w2 >> (8 * fx)) & 0xffu;
                    if (!surv) continue;
                    const int ft = 2 * c + fx;
                    const int xo = blk + (dx + tb.band) * 4 + (ft & 1), yo = blk + (dy + tb.band) * 4 + ((ft >> 1) & 1);
                    const int zo = blk + (dz + tb.band) * 4 + (ft >> 2);
                    ((uint4 *)dst)[0] = make_uint4((unsigned)wb, (unsigned)(wb >> 32), (unsigned)f, (unsigned)xo);
                    ((uint4 *)dst)[1] = make_uint4((unsigned)yo, (unsigned)zo, (unsigned)ft | (surv << 8), 0u);
                    dst++;
                }
            }
        });
        base += total;
        __syncthreads();
    }
}

// one workgroup per (work node, part) (grid-stride; nwp: the node count on the device, the
// parts then follow from it as on the host)
template <int MODE>
__global__ void __launch_bounds__(256) k_enum(int nw, const int *nwp, int *queue, int nparts, int K2,
                                              const WorkItem *work, const JobTab *jobs, const TermTab *tabs,
                                              GenState gs, int *seg_total, const long long *seg_ofs, Slice *out,
                                              const TaskSummary *sum, const NodeSched *nodes, SliceTask *tasks) {
    if (MODE == 1 && sum->overflow) return;
    const int n = nwp ? *nwp : nw, np = nwp ? enum_parts(n) : nparts;
    for_items(n * np, queue, [&](int b) {
        enum_node<MODE>(b / np, b % np, np, K2, work, jobs, tabs, gs, seg_total, seg_ofs, out, sum, nodes, tasks);
    });
}

// ----------------------------------------------------------------- apply: predictor features

// One thread per (work node, child).  Features (norms relative to split thresholds, so
// that one network serves several precisions; thresholds use the output-norm estimate
// at the start of the iteration):
//  0 log10(||w_parent|| / split threshold of the parent)
//  1 log10(||s_parent|| / split threshold of the child)
//  2 log10(||w_parent|| / ||w_grandparent||) (0 below the roots)
//  3 log10(||w_parent|| / ||s_parent||)    4 input tree has the child's cell (0/1)
//  5 log10(||w_input(cell)|| ||g|| / ||input|| / split threshold of the child), -20 absent
//  6 the input node of the cell has children (0/1)
//  7 as 5 for the largest of the 26 neighbouring cells, -20 when none
//  8 log10(mu + 1e-3)                      9 log10(cell width of the child)
__device__ inline float feat_lg(double v) {
    return (float)fmin(20.0, fmax(-20.0, log10(fmax(v, 1e-300))));
}

__device__ inline double input_wnorm(const JobTab &J, int i) {
    double a = 0.0;
    for (int q = 1; q < 8; q++) a += J.inNorm[(size_t)i * 8 + q] * J.inNorm[(size_t)i * 8 + q];
    return sqrt(a);
}

// 32 lanes per child: lanes 0..25 look up the 26 same-level neighbours of the child
// in the input tree, lane 26 the child itself, lane 27 its first child, lane 28 the
// parent's wavelet norm; the features are then gathered with shuffles in the half-wave
__global__ void __launch_bounds__(256) k_child_features(int nw, const WorkItem *work, const JobTab *jobs,
                                                        const double *wnorms, float *feat) {
    const int tt = (int)((blockIdx.x * (size_t)blockDim.x + threadIdx.x) >> 5);
    const int l = threadIdx.x & 31;
    const bool valid = tt < nw * 8;
    const int t = valid ? tt : nw * 8 - 1;
    const int i = t >> 3, a = t & 7;
    const WorkItem wi = work[i];
    const JobTab &J = jobs[wi.job];
    const int d = J.depth + 1;
    const int cx = 2 * wi.l[0] + (a & 1), cy = 2 * wi.l[1] + ((a >> 1) & 1), cz = 2 * wi.l[2] + ((a >> 2) & 1);
    double v = 0.0;  // lanes < 26: neighbour wavelet norm; 26: own norm (-1: absent); 28: parent's
    int found = 0;   // lanes 26 and 27: node present in the input tree
    if (l < 26) {
        const int c = l < 13 ? l : l + 1;  // 27 cells without the centre
        const int x = cx + c % 3 - 1, y = cy + (c / 3) % 3 - 1, z = cz + c / 9 - 1;
        if (x >= 0 && y >= 0 && z >= 0 && x < 2 * J.lmax[0] && y < 2 * J.lmax[1] && z < 2 * J.lmax[2]) {
            const int j = dhash_find(J.inHash, dnode_key(d, x, y, z));
            if (j >= 0) v = input_wnorm(J, j);
        }
    } else if (l == 26) {
        const int i0 = dhash_find(J.inHash, dnode_key(d, cx, cy, cz));
        found = i0 >= 0;
        v = found ? input_wnorm(J, i0) : 0.0;
    } else if (l == 27) {
        found = dhash_find(J.inHash, dnode_key(d + 1, 2 * cx, 2 * cy, 2 * cz)) >= 0;
    } else if (l == 28 && wi.parent >= 0) {
        double wpp = 0.0;
        for (int q = 1; q < 8; q++) {
            const double u = J.outNorm[(size_t)wi.parent * 8 + q];
            wpp += u * u;
        }
        v = sqrt(wpp);
    }
    double nb = l < 26 ? v : 0.0;
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) nb = fmax(nb, __shfl_xor(nb, o, 32));
    const double own = __shfl(v, 26, 32), wpp = __shfl(v, 28, 32);
    const int has = __shfl(found, 26, 32), has2 = __shfl(found, 27, 32);
    if (!valid || l != 0) return;
    const double *pn = wnorms + (size_t)i * 8;
    double w2 = 0.0;
    for (int q = 1; q < 8; q++) w2 += pn[q] * pn[q];
    const double wn = sqrt(w2), sn = pn[0];
    const int np = J.n0 + J.depth;
    const double eps2 = 2.0 * 2.220446049250313e-16;
    const double thr = fmax(eps2, J.prec * J.feat_tnorm * exp2(-0.5 * (np + 1)));
    const double thr_c = fmax(eps2, J.prec * J.feat_tnorm * exp2(-0.5 * (np + 2)));
    const double in_to_out = J.feat_tnorm / fmax(J.feat_innorm, 1e-300);
    float *f = feat + (size_t)t * 10;
    f[0] = feat_lg(wn / thr);
    f[1] = feat_lg(sn / thr_c);
    f[2] = wpp > 0.0 ? feat_lg(wn / wpp) : 0.0f;
    f[3] = feat_lg(wn / fmax(fabs(sn), 1e-300));
    f[4] = has ? 1.0f : 0.0f;
    f[5] = has ? feat_lg(own * in_to_out / thr_c) : -20.0f;
    f[6] = (has && has2) ? 1.0f : 0.0f;
    f[7] = nb > 0.0 ? feat_lg(nb * in_to_out / thr_c) : -20.0f;
    f[8] = J.feat_mu;
    f[9] = J.feat_cell;
}

hipError_t launch_child_features(hipStream_t s, int nw, const WorkItem *work, const JobTab *jobs,
                                 const double *wnorms, float *feat) {
    if (nw <= 0) return hipSuccess;
    const int n = nw * 8;
    hipLaunchKernelGGL(k_child_features, dim3((n + 7) / 8), dim3(256), 0, s, nw, work, jobs, wnorms, feat);
    return hipGetLastError();
}

// ----------------------------------------------------------------- apply: contraction schedule

__device__ inline long long wave_incl_scan_ll(long long v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const long long u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    return v;
}

// exclusive prefixes of NV values at once over the 1024 threads of the block (one
// exchange through LDS for all of them); tot[k] gets the sums
template <int NV>
__device__ inline void block_excl_scan_1024_n(long long (&v)[NV], long long (*wsum)[NV], long long (&tot)[NV]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    long long incl[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) incl[k] = wave_incl_scan_ll(v[k]);
    __syncthreads();
    if (lane == 63)
#pragma unroll
        for (int k = 0; k < NV; k++) wsum[wave][k] = incl[k];
    __syncthreads();
    if (threadIdx.x < NV) {
        const int k = threadIdx.x;
        long long acc = 0;
        for (int w = 0; w < 16; w++) {
            const long long x = wsum[w][k];
            wsum[w][k] = acc;
            acc += x;
        }
        wsum[16][k] = acc;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) {
        tot[k] = wsum[16][k];
        v[k] = wsum[wave][k] + incl[k] - v[k];
    }
}


// One workgroup.  Per node the slices of its (one or two) segments over all parts, and the parts'
// offsets inside them; from the totals the task sizes; one block scan of slices and tasks gives
// every node its first slices and tasks.  The fill kernels write the tasks themselves.
// FP64 tasks an iteration aims at (task size permitting): a k = 9 Poisson apply contracts in 1.70 ms
// with 2048, 1.94 with 4096, 1.61 with 1024 and 1.66 with 512; smaller orders within 2 % of each
// other.  Of at least FP64_TASK_MIN slices: 2 to 8 are equal (the slots cost what the waves gain).
constexpr long long FP64_TASKS = 1024;
constexpr int FP64_TASK_MIN = 8;

__global__ void __launch_bounds__(1024)
    k_build_tasks(int nw, const int *nwp, int nseg, int nparts, int chunk, int wchunk, const int *__restrict__ tot,
                  TaskCaps caps, const int *__restrict__ gen_count, int gen_pcap, long long *__restrict__ ofs,
                  NodeSched *__restrict__ nodes, TaskSummary *__restrict__ sum,
                  const int *__restrict__ gen_overflow) {
    __shared__ long long wsum4[17][4];
    if (nwp) {  // the work list's size on the device (its parts as the enumeration derived them)
        nw = *nwp;
        nparts = enum_parts(nw);
    }
    const bool mixed = nseg == 2;
    const int g0 = (int)((long long)nw * threadIdx.x / 1024), g1 = (int)((long long)nw * (threadIdx.x + 1) / 1024);
    long long v2[2] = {0, 0}, t2[2];
    for (int g = g0; g < g1; g++) {
        int c[2] = {0, 0};
        for (int q = 0; q < nseg; q++) {
            const size_t sg = ((size_t)g * nseg + q) * nparts;
            if (nparts == 1) {  // (the fill kernels know that the only part's offset is 0)
                c[q] = tot[sg];
                continue;
            }
            for (int p = 0; p < nparts; p++) {
                ofs[sg + p] = c[q];
                c[q] += tot[sg + p];
            }
        }
        nodes[g].count64 = c[0];
        nodes[g].count16 = c[1];
        v2[0] += c[0];
        v2[1] += c[1];
    }
    // task sizes from the iteration's totals.  FP64 tasks: at most chunk slices, fewer (down
    // to FP64_TASK_MIN) when the iteration has fewer than FP64_TASKS x chunk of them, so that a
    // coarse iteration still spreads over the GPU.  Slices per MFMA task when automatic
    // (wchunk <= 0): about -wchunk tasks, at least 16 and at most 128 slices each (larger
    // tasks leave too few to balance the k = 9 slices over the CUs)
    {
        long long w2[2] = {v2[0], v2[1]};
        block_excl_scan_1024_n<2>(w2, (long long(*)[2])wsum4, t2);
        chunk = (int)min((long long)chunk, max((long long)FP64_TASK_MIN, (t2[0] + FP64_TASKS - 1) / FP64_TASKS));
        if (mixed && wchunk <= 0) {
            const long long want = (t2[1] + (-wchunk) - 1) / (-wchunk);
            wchunk = (int)min(128LL, max(16LL, want));
        }
        __syncthreads();
    }
    long long nt64 = 0, nt16 = 0;
    for (int g = g0; g < g1; g++) {
        nt64 += (nodes[g].count64 + chunk - 1) / chunk;
        if (mixed) nt16 += (nodes[g].count16 + wchunk - 1) / wchunk;
    }
    long long pv[4] = {v2[0], v2[1], nt64, nt16}, pt[4];
    block_excl_scan_1024_n<4>(pv, wsum4, pt);
    int overflow = 0;
    if (pt[0] > caps.slices64 || pt[1] > caps.slices || pt[2] > caps.tasks || pt[3] > caps.stasks) overflow |= 1;
    if (*(volatile const int *)gen_count > gen_pcap) overflow |= 2;
    if (threadIdx.x == 0) {
        sum->nslices64 = pt[0];
        sum->nslices = pt[1];
        sum->ntasks = (int)pt[2];
        sum->nstasks = (int)pt[3];
        sum->overflow = overflow;
        sum->gen_count = *(volatile const int *)gen_count;
        sum->gen_overflow = *(volatile const int *)gen_overflow;
        sum->chunk = chunk;
        sum->schunk = mixed ? wchunk : 1;
    }
    if (overflow) return;
    for (int g = g0; g < g1; g++) {
        const int c64 = nodes[g].count64, c16 = nodes[g].count16;
        NodeSched nd;
        nd.start64 = pv[0];
        nd.start16 = pv[1];
        nd.count64 = c64;
        nd.count16 = c16;
        nd.task64 = (int)pv[2];
        nd.task16 = (int)pv[3];
        nodes[g] = nd;
        pv[0] += c64;
        pv[1] += c16;
        pv[2] += (c64 + chunk - 1) / chunk;
        if (mixed) pv[3] += (c16 + wchunk - 1) / wchunk;
    }
}

// The sum of n slots, in order, SLOT_FLY reads in flight.  One at a time, the latency of the reads
// was the kernel's time: 18.6 us per launch of a Poisson apply at k = 5 (6.2 now), 39 of a
// Coulomb potential at k = 7 (10), 59 of eight Helmholtz applies at k = 9 (43; there the traffic
// counts too).  Workgroups of 1024 with a quarter of the slots each were no better for few nodes
// (8 and 14 us) and slower for many (75).
constexpr int SLOT_FLY = 16;

__device__ inline double sum_slots(const double *p, int n, size_t stride) {
    double s = 0.0;
    int q = 0;
    for (; q + SLOT_FLY <= n; q += SLOT_FLY) {
        double v[SLOT_FLY];
#pragma unroll
        for (int i = 0; i < SLOT_FLY; i++) v[i] = p[(q + i) * stride];
#pragma unroll
        for (int i = 0; i < SLOT_FLY; i++) s += v[i];
    }
    if (q == n) return s;
    double v[SLOT_FLY];
#pragma unroll
    for (int i = 0; i < SLOT_FLY; i++) v[i] = q + i < n ? p[(q + i) * stride] : 0.0;
#pragma unroll
    for (int i = 0; i < SLOT_FLY; i++) s += v[i];
    return s;
}

// Sums the task slots of an output component in a fixed order (FP64 tasks, then MFMA tasks)
// into the node, and its norm into the tree and the compact per-work-node array.  One
// workgroup per (work node, component).
__global__ void __launch_bounds__(256) k_reduce_slots(int nw, const int *nwp, const TaskSummary *sum,
                                                      const NodeSched *nodes, const WorkItem *work, const JobTab *jobs,
                                                      const double *slots64, const double *slots16, int K3,
                                                      double *wnorm) {
    __shared__ double wsum[4];
    if (sum->overflow) return;
    const int n = 8 * (nwp ? *nwp : nw), chunk = sum->chunk, wchunk = sum->schunk;
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        const int g = i >> 3, gt = i & 7;
        const NodeSched nd = nodes[g];
        const WorkItem wi = work[g];
        const JobTab &J = jobs[wi.job];
        const int n64 = (nd.count64 + chunk - 1) / chunk, n16 = (nd.count16 + wchunk - 1) / wchunk;
        double *dst = J.outCoef + (size_t)wi.node * 8 * K3 + gt * K3;
        const double *p64 = slots64 + ((size_t)nd.task64 * 8 + gt) * K3;
        const double *p16 = slots16 + ((size_t)nd.task16 * 8 + gt) * K3;
        double ss = 0.0;
        for (int e = threadIdx.x; e < K3; e += blockDim.x) {
            const double s = sum_slots(p64 + e, n64, (size_t)8 * K3) + sum_slots(p16 + e, n16, (size_t)8 * K3);
            dst[e] = s;
            ss += s * s;
        }
        ss = block_sum_256(ss, wsum);
        if (threadIdx.x == 0) {
            const double v = sqrt(ss);
            J.outNorm[(size_t)wi.node * 8 + gt] = v;
            wnorm[(size_t)g * 8 + gt] = v;
        }
    }
}


// ----------------------------------------------------------------- apply: mixed-precision work list

// Same candidates and bounds as k_enum.  A slice (term, delta, ft) whose surviving combinations
// all stay below the route bound is contracted on split-FP16 MFMA, the others in FP64.
// Segments per node: 0 the FP64 slices, 1 the MFMA slices; layout of thread_off and
// seg_total: [g][2][...].
template <int MODE>
__device__ __forceinline__ void enum_mixed_node(int g, int part, int nparts, int K2, const WorkItem *work,
                                                const JobTab *jobs, const TermTab *tabs, const GenState &gs,
                                                int *thread_off, int *seg_total, const long long *seg_ofs,
                                                Slice *out64, Slice *out16, const TaskSummary *sum,
                                                const NodeSched *nodes, SliceTask *tasks, SliceTask *stasks) {
    const WorkItem wi = work[g];
    const JobTab &J = jobs[wi.job];
    __shared__ int scan[2][256];
    __shared__ int fcache[FCACHE];
    __shared__ CandTerms ct;
    __shared__ int wsum[4];
    const FCache fc = fill_fcache(fcache, wi, J, tabs, gs);
    term_prefix(ct, J, tabs);
    int cnt[2] = {0, 0}, nt64 = 0;
    long long base[2] = {0, 0};
    if (MODE == 1) {
        const NodeSched nd = nodes[g];
        if (part == 0) {
            emit_tasks(g, nd.start64, nd.count64, sum->chunk, nd.task64, tasks);
            emit_tasks(g, nd.start16, nd.count16, sum->schunk, nd.task16, stasks);
        }
        for (int q = 0; q < 2; q++) {
            const size_t sp = ((size_t)g * 2 + q) * nparts + part;  // (segment, part)
            base[q] = (q ? nd.start16 : nd.start64) + (nparts > 1 ? seg_ofs[sp] : 0) +
                      thread_off[sp * 256 + threadIdx.x];
        }
    }
    int k0, k1;
    part_range(ct.start[J.ntab], part, nparts, k0, k1);
    walk_candidates(ct, fcache, fc, wi, J, tabs, gs, k0, k1,
                    [&](int k, int t, const TermTab &tb, int dx, int dy, int dz, int f, const double *fn,
                        const double *nx, const double *ny, const double *nz) {
                        const double aw = fabs(tb.w);
                        const unsigned long long cm = combo_mask(tb, dx, dy, dz);
                        unsigned survs[8];
                        double maxbs[8];
                        screen_candidate<true>(aw, nx, ny, nz, fn, cm, J.thr, survs, maxbs);
#pragma unroll
                        for (int ft = 0; ft < 8; ft++) {
                            const unsigned surv = survs[ft];
                            if (!surv) continue;
                            const bool r64 = maxbs[ft] > J.route;
                            if (MODE == 1) {
                                // the record as two 16-byte stores (layout of Slice): weight, f,
                                // block offsets of the three dimensions (MFMA: in values; FP64: in
                                // blocks), ft and the surviving components
                                const unsigned long long wb = (unsigned long long)__double_as_longlong(tb.w);
                                const int unit = r64 ? 1 : K2, blk = (int)(r64 ? tb.blk / K2 : tb.blk);
                                const int xo = blk + ((dx + tb.band) * 4 + (ft & 1)) * unit;
                                const int yo = blk + ((dy + tb.band) * 4 + ((ft >> 1) & 1)) * unit;
                                const int zo = blk + ((dz + tb.band) * 4 + ((ft >> 2) & 1)) * unit;
                                uint4 *dst = (uint4 *)(r64 ? out64 + base[0] + cnt[0] : out16 + base[1] + cnt[1]);
                                dst[0] = make_uint4((unsigned)wb, (unsigned)(wb >> 32), (unsigned)f, (unsigned)xo);
                                dst[1] = make_uint4((unsigned)yo, (unsigned)zo, (unsigned)ft | (surv << 8), 0u);
                            } else if (r64) {
                                nt64 += __popc(surv);
                            }
                            if (r64) cnt[0]++;
                            else cnt[1]++;
                        }
                    });
    if (MODE == 0) {
        nt64 = block_sum_256i(nt64, wsum);
        for (int q = 0; q < 2; q++) scan[q][threadIdx.x] = cnt[q];
        __syncthreads();
        for (int off = 1; off < 256; off <<= 1) {
            int v[2];
            for (int q = 0; q < 2; q++) v[q] = threadIdx.x >= off ? scan[q][threadIdx.x - off] : 0;
            __syncthreads();
            for (int q = 0; q < 2; q++) scan[q][threadIdx.x] += v[q];
            __syncthreads();
        }
        for (int q = 0; q < 2; q++)
            thread_off[(((size_t)g * 2 + q) * nparts + part) * 256 + threadIdx.x] = scan[q][threadIdx.x] - cnt[q];
        if (threadIdx.x == 255) {
            for (int q = 0; q < 2; q++) seg_total[((size_t)g * 2 + q) * nparts + part] = scan[q][255];
            if (nt64) atomicAdd((unsigned long long *)&gs.tabcnt[4 * wi.job], (unsigned long long)nt64);
            if (scan[1][255])
                atomicAdd((unsigned long long *)&gs.tabcnt[4 * wi.job + 1], (unsigned long long)scan[1][255]);
        }
    }
}

template <int MODE>
__global__ void __launch_bounds__(256) k_enum_mixed(int nw, const int *nwp, int *queue, int nparts, int K2,
                                                    const WorkItem *work, const JobTab *jobs, const TermTab *tabs,
                                                    GenState gs, int *thread_off, int *seg_total,
                                                    const long long *seg_ofs, Slice *out64, Slice *out16,
                                                    const TaskSummary *sum, const NodeSched *nodes, SliceTask *tasks,
                                                    SliceTask *stasks) {
    if (MODE == 1 && sum->overflow) return;
    const int n = nwp ? *nwp : nw, np = nwp ? enum_parts(n) : nparts;
    for_items(n * np, queue, [&](int b) {
        enum_mixed_node<MODE>(b / np, b % np, np, K2, work, jobs, tabs, gs, thread_off, seg_total, seg_ofs, out64,
                              out16, sum, nodes, tasks, stasks);
    });
}

// ----------------------------------------------------------------- apply: device-resident refinement

__global__ void __launch_bounds__(256) k_loop_init(int njobs, int nr, const LoopJob *lj, const int *rootlr,
                                                   WorkItem *work) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < njobs * nr; i += gridDim.x * blockDim.x) {
        const int j = i / nr, r = i % nr;
        const LoopJob &L = lj[j];
        WorkItem wi;
        wi.job = j;
        wi.node = r;
        wi.parent = -1;
        L.depth[r] = 0;
        L.parent[r] = -1;
        L.child[r] = -1;
        for (int q = 0; q < 3; q++) {
            wi.l[q] = rootlr[3 * r + q];
            L.lr[3 * r + q] = wi.l[q];
        }
        work[i] = wi;
    }
}

// One workgroup per job.  The running norm adds the squared norms of the job's work nodes
// (scaling parts on the roots, wavelet parts everywhere; per thread over a contiguous run,
// then a fixed reduction tree); the split test is the host's (split_check with the factor
// 2^(-(n0 + d + 1) / 2) the host computed); the split nodes' children follow the node count in
// work-list order, 8 each, as the host appends them.
__global__ void __launch_bounds__(256) k_loop_split(int njobs, LoopJob *lj, const WorkItem *work, const double *wn,
                                                    int max_depth, LoopCtl *ctl, int *cidx, const long long *tabcnt,
                                                    unsigned long long *ts_end) {
    const int j = blockIdx.x, tid = threadIdx.x;
    if (ts_end && j == 0 && tid == 0) *ts_end = (unsigned long long)wall_clock64();
    if (j >= njobs) return;
    LoopJob &L = lj[j];
    __shared__ double rs[256], rw[256];
    __shared__ int sc[256];
    __shared__ double s_tn;
    __shared__ int s_n;
    if (tid == 0) {
        L.tuples += tabcnt[4 * (size_t)j] + tabcnt[4 * (size_t)j + 2];
        L.tuples_fp64 += tabcnt[4 * (size_t)j];
        L.slices += tabcnt[4 * (size_t)j + 1];
        L.gen += tabcnt[4 * (size_t)j + 3];
    }
    const int w0 = L.w0, nwk = L.nwk;
    if (nwk <= 0) {
        if (tid == 0) L.splits = 0;
        return;
    }
    const int d = L.depth[work[w0].node];
    const int per = (nwk + 255) / 256, i0 = min(nwk, tid * per), i1 = min(nwk, i0 + per);
    double s = 0.0, w = 0.0;
    for (int i = i0; i < i1; i++) {
        const double *p = wn + (size_t)(w0 + i) * 8;
        if (d == 0) s += p[0] * p[0];
        for (int c = 1; c < 8; c++) w += p[c] * p[c];
    }
    rs[tid] = s;
    rw[tid] = w;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (tid < off) {
            rs[tid] += rs[tid + off];
            rw[tid] += rw[tid + off];
        }
        __syncthreads();
    }
    if (tid == 0) {
        L.sNorm += rs[0];
        L.wNorm += rw[0];
        L.gsq = L.sNorm + L.wNorm;
        s_tn = sqrt(L.gsq);
        s_n = L.n;
    }
    __syncthreads();
    const double thr = fmax(2.0 * 2.220446049250313e-16, L.prec * s_tn * ctl->splitfac[d]);
    const bool can = d < max_depth;
    auto splits_at = [&](int i) {
        const double *p = wn + (size_t)(w0 + i) * 8;
        double w2 = 0.0;
        for (int c = 1; c < 8; c++) w2 += p[c] * p[c];
        return can && sqrt(w2) > thr;
    };
    int cnt = 0;
    for (int i = i0; i < i1; i++) cnt += splits_at(i) ? 1 : 0;
    sc[tid] = cnt;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const int v = tid >= off ? sc[tid - off] : 0;
        __syncthreads();
        sc[tid] += v;
        __syncthreads();
    }
    const int S = sc[255], n0 = s_n;
    const bool fits = (long long)n0 + 8LL * S <= (long long)L.cap;
    int r = sc[tid] - cnt;
    for (int i = i0; i < i1; i++) {
        const bool sp = fits && splits_at(i);
        cidx[w0 + i] = sp ? n0 + 8 * r : -1;
        if (!sp) continue;
        const WorkItem wi = work[w0 + i];
        const int c0 = n0 + 8 * r;
        L.child[wi.node] = c0;
        for (int a = 0; a < 8; a++) {
            const size_t c = (size_t)c0 + a;
            L.depth[c] = d + 1;
            L.parent[c] = wi.node;
            L.child[c] = -1;
            L.lr[3 * c] = 2 * wi.l[0] + (a & 1);
            L.lr[3 * c + 1] = 2 * wi.l[1] + ((a >> 1) & 1);
            L.lr[3 * c + 2] = 2 * wi.l[2] + ((a >> 2) & 1);
        }
        r++;
    }
    if (tid == 0) {
        if (!fits) atomicOr(&ctl->overflow, 4);
        L.n = fits ? n0 + 8 * S : n0;
        L.splits = fits ? S : 0;
    }
}

// The next work list: job j's children start at 8 x (split nodes of the jobs before j),
// its split nodes' children in work-list order (the order of the host loop).  Every
// workgroup forms the same prefix over the jobs; workgroup 0 also records the jobs' ranges,
// the list's size and the iteration's read-back entry.
__global__ void __launch_bounds__(256) k_loop_emit(int njobs, LoopJob *lj, const WorkItem *work, const int *nwp,
                                                   const int *cidx, WorkItem *next, int *nw_next, int wcap,
                                                   const TaskSummary *sum, LoopCtl *ctl, int d, const JobTab *jt,
                                                   TransformItem *titems, int tcap, LoopIter *host_iter) {
    __shared__ int base[LOOP_MAX_JOBS];
    __shared__ int sc[256];
    const int tid = threadIdx.x;
    const int per = (njobs + 255) / 256, j0 = min(njobs, tid * per), j1 = min(njobs, j0 + per);
    int c = 0;
    for (int j = j0; j < j1; j++) c += lj[j].splits;
    sc[tid] = c;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const int v = tid >= off ? sc[tid - off] : 0;
        __syncthreads();
        sc[tid] += v;
        __syncthreads();
    }
    int b = sc[tid] - c;
    for (int j = j0; j < j1; j++) {
        base[j] = b;
        b += lj[j].splits;
    }
    const long long total = sc[255];
    __syncthreads();
    // (bits of earlier kernels; the ones added here follow from the same inputs in every workgroup)
    const int t0 = ctl->tofs[d];
    int ovf = *(volatile int *)&ctl->overflow;
    if (sum->overflow) ovf |= sum->overflow & 3;
    if (sum->gen_overflow) ovf |= 16;
    if (8 * total > (long long)wcap) ovf |= 8;
    if ((long long)t0 + total > (long long)tcap) ovf |= 32;
    if (blockIdx.x == 0) {
        for (int j = tid; j < njobs; j += 256) {
            lj[j].w0 = 8 * base[j];
            lj[j].nwk = ovf ? 0 : 8 * lj[j].splits;
        }
        if (tid == 0) {
            const int nn = ovf ? 0 : (int)(8 * total);
            ctl->overflow = ovf;
            *nw_next = nn;
            ctl->iter[d].nw_next = nn;
            ctl->iter[d].overflow = ovf;
            host_iter[d].nw_next = nn;
            host_iter[d].overflow = ovf;
            ctl->tofs[d + 1] = t0 + (ovf ? 0 : (int)total);
        }
    }
    if (ovf) return;
    const int n = *nwp;
    for (int i = blockIdx.x * 256 + tid; i < n; i += gridDim.x * 256) {
        const int c0 = cidx[i];
        if (c0 < 0) continue;
        const WorkItem wi = work[i];
        const int j = wi.job;
        const int first = lj[j].n - 8 * lj[j].splits;  // the job's node count before this iteration
        const int rank = (c0 - first) >> 3;
        const int p = 8 * (base[j] + rank);
        titems[t0 + base[j] + rank] = TransformItem{jt[j].outCoef, jt[j].outNorm, wi.node, c0};
        for (int a = 0; a < 8; a++) {
            WorkItem ch;
            ch.job = j;
            ch.node = c0 + a;
            ch.l[0] = 2 * wi.l[0] + (a & 1);
            ch.l[1] = 2 * wi.l[1] + ((a >> 1) & 1);
            ch.l[2] = 2 * wi.l[2] + ((a >> 2) & 1);
            ch.parent = wi.node;
            next[p + a] = ch;
        }
    }
}

// ----------------------------------------------------------------- tree compaction

// node groups (8 siblings) moved inside a tree: pair i copies the group at node
// from_to[2i] to node from_to[2i+1], one block per node of the group (nb coefficient
// doubles and 8 norms per node); no source of a pair is the destination of another
__global__ void __launch_bounds__(256) k_move_groups(int npairs, const int *from_to, double *coef, double *norm,
                                                     int nb) {
    const int i = blockIdx.x, a = blockIdx.y;
    if (i >= npairs) return;
    const size_t f = (size_t)from_to[2 * i] + a, t = (size_t)from_to[2 * i + 1] + a;
    for (int e = threadIdx.x; e < nb; e += blockDim.x) coef[t * nb + e] = coef[f * nb + e];
    if (threadIdx.x < 8) norm[t * 8 + threadIdx.x] = norm[f * 8 + threadIdx.x];
}

hipError_t launch_move_groups(hipStream_t s, int npairs, const int *from_to, double *coef, double *norm, int nb) {
    if (npairs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_move_groups, dim3(npairs, 8), dim3(256), 0, s, npairs, from_to, coef, norm, nb);
    return hipGetLastError();
}

// ----------------------------------------------------------------- launchers

hipError_t launch_tblock_mom(hipStream_t s, int n, const int *item_term, const long long *item_delta, const double *b,
                             const double *pre, int K, const double *ccoef, const double *gx, const double *gw,
                             double *out) {
    if (n <= 0) return hipSuccess;
    MWG_DISPATCH_K(K, hipLaunchKernelGGL(k_tblock_mom<KK>, dim3(n), dim3(64), 0, s, n, item_term, item_delta, b, pre,
                                         ccoef, gx, gw, out));
    return hipGetLastError();
}

hipError_t launch_nsblocks(hipStream_t s, long long first, long long n, const NSItems &items, const double *t1,
                           const double *W, int K) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_nsblocks, dim3((unsigned)n), dim3(256), 0, s, first, items, t1, W, K);
    return hipGetLastError();
}

hipError_t launch_norms(hipStream_t s, int n, const double *coef, double *norm, int K3) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_norms, dim3(n), dim3(256), 0, s, n, coef, norm, K3);
    return hipGetLastError();
}

hipError_t launch_dot_pairs(hipStream_t s, int n, const unsigned long long *pairs, const double *A,
                            const double *B, int K3, int nblocks, double *part, double *res) {
    if (n < 0 || nblocks < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_dot_pairs, dim3(nblocks), dim3(256), 0, s, n, pairs, A, B, K3, part);
    hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(64), 0, s, nblocks, part, res);
    return hipGetLastError();
}

hipError_t launch_dot(hipStream_t s, int n, const DotPair *pairs, int K3, double *part) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dot, dim3(n), dim3(256), 0, s, pairs, K3, part);
    return hipGetLastError();
}

hipError_t launch_hash_build(hipStream_t s, int n, const HashItem *items, const unsigned long long *keys) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_hash_clear, dim3(n * HASH_BLOCKS), dim3(256), 0, s, items);
    hipLaunchKernelGGL(k_hash_insert, dim3(n * HASH_BLOCKS), dim3(256), 0, s, items, keys);
    return hipGetLastError();
}

hipError_t launch_gather(hipStream_t s, int n, const GatherItem *items, double *dst) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather, dim3(n * HASH_BLOCKS), dim3(256), 0, s, items, dst);
    return hipGetLastError();
}

hipError_t launch_scale(hipStream_t s, size_t n, double *x, double c) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_scale, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, x, c);
    return hipGetLastError();
}

hipError_t launch_project_gauss(hipStream_t s, int nw, const MulItem *items, const ProjGeom &geo, const DevBasis &B,
                                int nterm, const double *coef, const double *alpha, const double *center,
                                const double *poly, double *out, double *norm, double *compact) {
    if (nw <= 0) return hipSuccess;
    MWG_DISPATCH_K(B.K, hipLaunchKernelGGL(k_project_gauss<KK>, dim3(nw), dim3(256), 0, s, items, geo, B, nterm, coef,
                                           alpha, center, poly, out, norm, compact));
    return hipGetLastError();
}

hipError_t launch_job_boxes(hipStream_t s, int nbj, int max_terms, const BoxJob *bj, TermTab *tabs, double *tbmax,
                            JobTab *jobs, int *pre, int *gen_overflow, const LoopInit &li) {
    if (nbj <= 0 || max_terms <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_job_boxes, dim3(nbj, max_terms), dim3(64), 0, s, nbj, bj, tabs, tbmax, max_terms, li);
    hipLaunchKernelGGL(k_job_route, dim3(nbj), dim3(64), 0, s, nbj, bj, tabs, tbmax, max_terms, jobs, pre,
                       gen_overflow, li);
    return hipGetLastError();
}

hipError_t launch_gen_mark(hipStream_t s, int nw, const WorkItem *work, const JobTab *jobs, const TermTab *tabs,
                           const GenState &gs, const int *nwp, int *queue) {
    if (nw <= 0) return hipSuccess;
    const int nb = nwp ? std::min(nw, DEVCOUNT_GRID) : nw;
    hipLaunchKernelGGL(k_gen_mark, dim3(nb), dim3(256), 0, s, nw, nwp, queue, work, jobs, tabs, gs);
    return hipGetLastError();
}

hipError_t launch_enum(hipStream_t s, int mode, int K, int nw, int nparts, const WorkItem *work, const JobTab *jobs,
                       const TermTab *tabs, const GenState &gs, int *seg_total, const long long *seg_ofs, Slice *out,
                       const TaskSummary *sum, const NodeSched *nodes, SliceTask *tasks, const int *nwp, int *queue) {
    if (nw <= 0) return hipSuccess;
    const unsigned nb = nwp ? (unsigned)DEVCOUNT_GRID : (unsigned)nw * (unsigned)nparts;
    if (mode == 0)
        hipLaunchKernelGGL(k_enum<0>, dim3(nb), dim3(256), 0, s, nw, nwp, queue, nparts, K * K, work, jobs, tabs, gs,
                           seg_total, seg_ofs, out, sum, nodes, tasks);
    else
        hipLaunchKernelGGL(k_enum<1>, dim3(nb), dim3(256), 0, s, nw, nwp, queue, nparts, K * K, work, jobs, tabs, gs,
                           seg_total, seg_ofs, out, sum, nodes, tasks);
    return hipGetLastError();
}

__global__ void k_stamp(unsigned long long *t) { *t = (unsigned long long)wall_clock64(); }

hipError_t launch_stamp(hipStream_t s, unsigned long long *t) {
    hipLaunchKernelGGL(k_stamp, dim3(1), dim3(1), 0, s, t);
    return hipGetLastError();
}

hipError_t launch_loop_init(hipStream_t s, int njobs, int nr, const LoopJob *lj, const int *rootlr, WorkItem *work) {
    const int n = njobs * nr;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_loop_init, dim3(std::min((n + 255) / 256, 1024)), dim3(256), 0, s, njobs, nr, lj, rootlr,
                       work);
    return hipGetLastError();
}

hipError_t launch_loop_split(hipStream_t s, int njobs, LoopJob *lj, const WorkItem *work, const double *wnorm,
                             int max_depth, LoopCtl *ctl, int *cidx, const long long *tabcnt,
                             unsigned long long *ts_end) {
    if (njobs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_loop_split, dim3(njobs), dim3(256), 0, s, njobs, lj, work, wnorm, max_depth, ctl, cidx,
                       tabcnt, ts_end);
    return hipGetLastError();
}

hipError_t launch_loop_emit(hipStream_t s, int njobs, LoopJob *lj, const WorkItem *work, const int *nwp,
                            const int *cidx, WorkItem *next, int *nw_next, int wcap, const TaskSummary *sum,
                            LoopCtl *ctl, int d, const JobTab *jt, TransformItem *titems, int tcap,
                            LoopIter *host_iter) {
    if (njobs <= 0 || njobs > LOOP_MAX_JOBS || d < 0 || d >= LOOP_MAX_DEPTH) return hipErrorInvalidValue;
    const int nb = std::max(1, std::min((wcap + 255) / 256, 1024));
    hipLaunchKernelGGL(k_loop_emit, dim3(nb), dim3(256), 0, s, njobs, lj, work, nwp, cidx, next, nw_next, wcap, sum,
                       ctl, d, jt, titems, tcap, host_iter);
    return hipGetLastError();
}

hipError_t launch_build_tasks(hipStream_t s, int nw, int nseg, int nparts, int chunk, int wchunk, const int *tot,
                              TaskCaps caps, const int *gen_count, int gen_pcap, long long *ofs, NodeSched *nodes,
                              TaskSummary *sum, const int *gen_overflow, const int *nwp) {
    hipLaunchKernelGGL(k_build_tasks, dim3(1), dim3(1024), 0, s, nw, nwp, nseg, nparts, chunk, wchunk, tot, caps,
                       gen_count, gen_pcap, ofs, nodes, sum, gen_overflow);
    return hipGetLastError();
}

hipError_t launch_reduce_slots(hipStream_t s, int nw, const int *nwp, const TaskSummary *sum, const NodeSched *nodes,
                               const WorkItem *work, const JobTab *jobs, const double *slots64, const double *slots16,
                               int K3, double *wnorm) {
    if (nw <= 0) return hipSuccess;
    const int nb = (int)std::min<long long>(8LL * nw, 4096);
    hipLaunchKernelGGL(k_reduce_slots, dim3(nb), dim3(256), 0, s, nw, nwp, sum, nodes, work, jobs, slots64, slots16,
                       K3, wnorm);
    return hipGetLastError();
}

hipError_t launch_enum_mixed(hipStream_t s, int mode, int K, int nw, int nparts, const WorkItem *work, const JobTab *jobs,
                             const TermTab *tabs, const GenState &gs, int *thread_off, int *seg_total,
                             const long long *seg_ofs, Slice *out64, Slice *out16, const TaskSummary *sum,
                             const NodeSched *nodes, SliceTask *tasks, SliceTask *stasks, const int *nwp, int *queue) {
    if (nw <= 0) return hipSuccess;
    const unsigned nb = nwp ? (unsigned)DEVCOUNT_GRID : (unsigned)nw * (unsigned)nparts;
    if (mode == 0)
        hipLaunchKernelGGL(k_enum_mixed<0>, dim3(nb), dim3(256), 0, s, nw, nwp, queue, nparts, K * K, work, jobs,
                           tabs, gs, thread_off, seg_total, seg_ofs, out64, out16, sum, nodes, tasks, stasks);
    else
        hipLaunchKernelGGL(k_enum_mixed<1>, dim3(nb), dim3(256), 0, s, nw, nwp, queue, nparts, K * K, work, jobs,
                           tabs, gs, thread_off, seg_total, seg_ofs, out64, out16, sum, nodes, tasks, stasks);
    return hipGetLastError();
}

}  // namespace mwg
