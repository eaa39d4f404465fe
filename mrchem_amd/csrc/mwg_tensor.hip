// Node-tensor kernels: two-scale transforms, generated nodes, products, sums and the
// projection of hydrogen functions (gfx950, wave64).
//
// A node's 8 components form the interleaved (2K)^3 tensor (index per dimension: bit * K + i);
// everything here is a matrix applied to every line of it along each dimension.  The tensor sits
// in LDS, x rows padded to 2K + 1 doubles, and a pass is done in place, 16 lines per wave at a time,
// on v_mfma_f64_4x4x4_4b_f64: the matrix rows in registers for the whole pass (A, 4 rows per
// instruction, the same for the 4 blocks), 16 lines as the columns of B, 4 products long.  One
// thread per line with the matrix read from LDS for every product was bound by those reads.
// Before and after (kernel time, norms launches not counted): the products of an eight-orbital
// exchange step at k = 7, 34.7 ms -> 6.2; k_transform
// 17.7 -> 8.7 us (k = 7, Coulomb potential of six Gaussians) and 48 -> 19 (k = 9, eight
// Helmholtz applies); k_gen_compute there 58 -> 33.  What bounds them now is the latency of one node's
// chain (read, three or nine passes with a barrier each, write), 2 to 3 workgroups per CU.
#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>

#include "mwg_kernels.h"

namespace mwg {

namespace {

__device__ inline double mfma4(double a, double b, double c) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

template <int K>
struct PadT {
    static constexpr int N = 2 * K, P = N + 1, PL = N * P, SIZE = N * PL;
};

template <int K>
__device__ inline int padded_index(int c, int e) {
    constexpr int N = 2 * K, P = N + 1;
    const int x = e % K, y = (e / K) % K, z = e / (K * K);
    const int bx = c & 1, by = (c >> 1) & 1, bz = (c >> 2) & 1;
    return ((bz * K + z) * N + (by * K + y)) * P + bx * K + x;
}

// The rows of an R x KI matrix (row-major, row stride ms) as A operands, lane 16 kq + 4 blk + r of the
// products: A[row r][k = kq], B[k = kq][column 4 blk + r], D[row kq][column].  Lane group kq takes
// the G = ceil(KI / 4) consecutive k from min(G kq, KI - G), those of the group before as zeros.
template <int R, int KI>
struct Rows {
    static constexpr int G = (KI + 3) / 4, RG = (R + 3) / 4;
    double a[RG][G];
    __device__ inline void load(const double *M, int ms) {
        const int lane = threadIdx.x & 63, kq = lane >> 4, r4 = lane & 3, kb = min(G * kq, KI - G);
#pragma unroll
        for (int r = 0; r < RG; r++)
#pragma unroll
            for (int s = 0; s < G; s++) {
                const double v = M[min(4 * r + r4, R - 1) * ms + kb + s];
                a[r][s] = KI % 4 == 0 || kb + s >= G * kq ? v : 0.0;
            }
    }
};

// In place along dim (0 = x): the first KI values of every line -> its first R values, line = M
// line.  Lines: the e1 x e2 positions (u, v) of the other two dimensions, in the order x, y, z.  A
// wave reads the lines of a tile before it writes them; no other wave touches them.
template <int N, int R, int KI>
__device__ inline void line_pass(double *T, const Rows<R, KI> &M, int dim, int e1, int e2) {
    constexpr int P = N + 1, G = Rows<R, KI>::G, RG = Rows<R, KI>::RG;
    const int lane = threadIdx.x & 63, col = lane & 15, kq = lane >> 4, kb = min(G * kq, KI - G);
    const int nl = e1 * e2, stride = dim == 0 ? 1 : dim == 1 ? P : N * P;
    for (int t = (int)(threadIdx.x >> 6) * 16; t < nl; t += (int)(blockDim.x >> 6) * 16) {
        const int line = min(t + col, nl - 1), v = line / e1, u = line - v * e1;
        double *p = T + (dim == 0 ? (v * N + u) * P : dim == 1 ? v * N * P + u : v * P + u);
        double b[G], d[RG];
#pragma unroll
        for (int s = 0; s < G; s++) b[s] = p[(kb + s) * stride];
#pragma unroll
        for (int r = 0; r < RG; r++) d[r] = mfma4(M.a[r][0], b[0], 0.0);
#pragma unroll
        for (int s = 1; s < G; s++)
#pragma unroll
            for (int r = 0; r < RG; r++) d[r] = mfma4(M.a[r][s], b[s], d[r]);
        if (t + col < nl) {
#pragma unroll
            for (int r = 0; r < RG; r++)
                if (R % 4 == 0 || 4 * r + kq < R) p[(4 * r + kq) * stride] = d[r];
        }
    }
}
// the same with the matrix read for this pass
template <int N, int R, int KI>
__device__ inline void line_pass(double *T, const double *M, int ms, int dim, int e1, int e2) {
    Rows<R, KI> m;
    m.load(M, ms);
    line_pass<N, R, KI>(T, m, dim, e1, e2);
}

// Per dimension the K x 2K matrix that takes a node's (s, d) line to the scaling line of its
// descendant `steps` levels down along the path bits of (lx, ly, lz) (bit steps - 1 first): the
// reconstruction of one child, then low-pass filters.  F: 3 x (K x 2K), S the same size
// (scratch); the result is in F.
template <int K>
__device__ inline void descent_matrices(double *F, double *S, const double *W, int lx, int ly, int lz, int steps) {
    constexpr int N = 2 * K, KN = K * N;
    double *cur = (steps & 1) ? F : S, *nxt = (steps & 1) ? S : F;  // (the last product lands in F)
    for (int e = threadIdx.x; e < 3 * KN; e += blockDim.x) {
        const int dim = e / KN, j = (e % KN) / N, p = e % N;
        const int a = ((dim == 0 ? lx : dim == 1 ? ly : lz) >> (steps - 1)) & 1;
        cur[e] = W[p * N + a * K + j];
    }
    __syncthreads();
    for (int sh = steps - 2; sh >= 0; sh--) {
        for (int e = threadIdx.x; e < 3 * KN; e += blockDim.x) {
            const int dim = e / KN, j = (e % KN) / N, p = e % N;
            const int a = ((dim == 0 ? lx : dim == 1 ? ly : lz) >> sh) & 1;
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < K; q++) s += W[q * N + a * K + j] * cur[dim * KN + q * N + p];
            nxt[e] = s;
        }
        __syncthreads();
        double *t = cur;
        cur = nxt;
        nxt = t;
    }
}

// A node tensor on its way to LDS: all of a thread's global reads in flight at once (coalesced),
// then stored interleaved.
template <int K>
struct NodeRegs {
    static constexpr int NV = 8 * K * K * K, PER = (NV + 255) / 256;
    double v[PER];
    // value e of the tensor at src(e)
    template <class F>
    __device__ inline void load(F src) {
#pragma unroll
        for (int w = 0; w < PER; w++) v[w] = *src(min(threadIdx.x + 256u * w, NV - 1u));
    }
    __device__ inline void store(double *T, unsigned t = threadIdx.x) const {
#pragma unroll
        for (int w = 0; w < PER; w++) {
            const int e = t + 256 * w;
            if (NV % 256 == 0 || e < NV) T[padded_index<K>(e / (K * K * K), e % (K * K * K))] = v[w];
        }
    }
};

}  // namespace

// ----------------------------------------------------------------- two-scale transforms

// batched two-scale transforms over (tree, parent) items:
// mode 0 compress children -> parent (and the parent's 8 component norms, also to the item's
// entry of compact if given), mode 1 add reconstruct(parent) to the children's scaling parts
// (and their norms)
template <int K>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(K <= 8 ? 3 : 2)))
k_transform(int mode, const TransformItem *items, const double *M, double *compact) {
    using L = PadT<K>;
    constexpr int N = L::N, K3 = K * K * K;
    extern __shared__ double T[];
    __shared__ double wsum[4][8];
    constexpr int PER = NodeRegs<K>::PER;
    const TransformItem it = items[blockIdx.x];
    Rows<N, N> m;
    NodeRegs<K> in, sum;
    // (coefficients of the children's scaling parts, child after child)
    auto child = [&](int e) { return it.coef + (size_t)(it.first_child + e / K3) * 8 * K3 + e % K3; };
    auto parent = [&](int e) { return it.coef + (size_t)it.parent * 8 * K3 + e; };
    if (mode == 0) {
        in.load(child);
    } else {
        in.load(parent);
        sum.load(child);
    }
    m.load(M, N);
    in.store(T);
    __syncthreads();
    for (int dim = 0; dim < 3; dim++) {
        line_pass<N, N, N>(T, m, dim, N, N);
        __syncthreads();
    }
    double ss[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int w = 0; w < PER; w++) {
        const int e = threadIdx.x + 256 * w;
        if (8 * K3 % 256 != 0 && e >= 8 * K3) break;
        const int c = e / K3;
        double v = T[padded_index<K>(c, e % K3)];
        if (mode == 0) {
            *parent(e) = v;
        } else {
            v += sum.v[w];
            *child(e) = v;
        }
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (256 * w / K3 <= q && q <= (256 * w + 255) / K3) ss[q] += c == q ? v * v : 0.0;
    }
    if (mode == 0) {
        put_norms(ss, wsum, it.norm + (size_t)it.parent * 8, compact ? compact + (size_t)blockIdx.x * 8 : nullptr);
    } else {
        const double v = sqrt(block_sum8(ss, wsum));
        if (threadIdx.x < 8) it.norm[(size_t)(it.first_child + threadIdx.x) * 8] = v;
    }
}

// ----------------------------------------------------------------- generated nodes

// scaling block of a generated node: reconstruct from the leaf ancestor (using its
// wavelets for the first step), then refine with the low-pass filters, as one K x 2K matrix
// per dimension
template <int K>
__device__ void gen_one(int g, const JobTab *jobs, const GenState &gs, double *T, double *F, const double *W) {
    using L = PadT<K>;
    constexpr int N = L::N, P = L::P, K3 = K * K * K;
    const uint64_t key = gs.keys[g];
    const JobTab &J = jobs[gs.job[g]];
    const int d = (int)(key >> 57);
    const int lx = (int)((key >> 38) & 0x7FFFF), ly = (int)((key >> 19) & 0x7FFFF), lz = (int)(key & 0x7FFFF);
    // the deepest ancestor present in the input tree: one thread per level probes it
    __shared__ int s_anc, s_ad;
    if (threadIdx.x == 0) {
        s_anc = -1;
        s_ad = -1;
    }
    __syncthreads();
    const int my_dd = d - 1 - (int)threadIdx.x;
    int my_a = -1;
    if (my_dd >= 0) {
        const int sh = d - my_dd;
        my_a = dhash_find(J.inHash, dnode_key(my_dd, lx >> sh, ly >> sh, lz >> sh));
        if (my_a >= 0) atomicMax(&s_ad, my_dd);
    }
    __syncthreads();
    if (my_a >= 0 && my_dd == s_ad) s_anc = my_a;
    __syncthreads();
    const int anc = s_anc, ad = s_ad;
    double *outp = gs.pool + (size_t)g * K3;
    if (anc < 0) {
        for (int e = threadIdx.x; e < K3; e += blockDim.x) outp[e] = 0.0;
        if (threadIdx.x == 0) gs.norm[g] = 0.0;
        __syncthreads();
        return;
    }
    NodeRegs<K> in;
    in.load([&](int e) { return J.inCoef + (size_t)anc * 8 * K3 + e; });
    descent_matrices<K>(F, T, W, lx, ly, lz, d - ad);  // (T as scratch; ends with a barrier)
    in.store(T);
    __syncthreads();
    line_pass<N, K, N>(T, F, N, 0, N, N);
    __syncthreads();
    line_pass<N, K, N>(T, F + K * N, N, 1, K, N);
    __syncthreads();
    line_pass<N, K, N>(T, F + 2 * K * N, N, 2, K, K);
    __syncthreads();
    __shared__ double wsum[4];
    double s2 = 0.0;
    for (int e = threadIdx.x; e < K3; e += blockDim.x) {
        const int x = e % K, y = (e / K) % K, z = e / (K * K);
        const double v = T[(z * N + y) * P + x];
        outp[e] = v;
        s2 += v * v;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s2 += __shfl_xor(s2, o, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = s2;
    __syncthreads();
    if (threadIdx.x == 0) gs.norm[g] = sqrt((wsum[0] + wsum[1]) + (wsum[2] + wsum[3]));
    __syncthreads();
}

// Generated nodes first .. min(count, cap) - 1, count read from the device counter
// that k_gen_mark advanced (no host round trip); grid-stride over the range.
template <int K>
__global__ void __launch_bounds__(256) k_gen_compute(int first, const int *firstp, int cap, const JobTab *jobs,
                                                     GenState gs, const double *W) {
    extern __shared__ double smem[];
    double *T = smem, *F = T + PadT<K>::SIZE;
    if (firstp) first = *firstp;
    const int end = min(*(volatile const int *)gs.count, cap);
    for (int g = first + blockIdx.x; g < end; g += gridDim.x) gen_one<K>(g, jobs, gs, T, F, W);
}

// ----------------------------------------------------------------- products

// out = coef * a * b at the listed output nodes: both inputs to values at the K^3
// quadrature points of the 8 children, product, quadrature projection, compression.
// Reconstruction and evaluation are one 2K x 2K matrix per dimension (B.E), for an input that
// ends above the node together with its descent; projection and compression are another (B.C,
// weights included).  The values of a wait in registers while b uses the tensor.  At K = 10 these, a
// node on its way to LDS and the matrix rows fill the registers: with the addresses of both places
// held as well it spilled 106 of them (a launch of 21 orbital products 1277 us, 987 now).
template <int K>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(K <= 8 ? 3 : 2)))
k_multiply(const MulItem *items, const MulJobDev *jobs, ProjGeom geo, DevBasis B, double *compact) {
    using L = PadT<K>;
    constexpr int N = L::N, P = L::P, N2 = N * N, N3 = N2 * N, K3 = K * K * K, KN = K * N;
    constexpr int PER = (N3 + 255) / 256, MP = (3 * N2 + 255) / 256;
    extern __shared__ double smem[];
    __shared__ double wsum[4][8];
    double *T = smem, *M = T + L::SIZE;  // M: 3 N x N
    const MulItem it = items[blockIdx.x];
    const MulJobDev J = jobs[it.job];
    double va[PER];
    for (int q = 0; q < 2; q++) {
        const int steps = q ? it.bsteps : it.asteps;
        const double *src = (q ? J.b : J.a) + (size_t)(q ? it.bsrc : it.asrc) * 8 * K3;
        NodeRegs<K> in;
        in.load([&](unsigned e) { return src + e; });
        if (steps > 0) {
            double *F = T, *S = T + 3 * KN;  // (the tensor is not there yet)
            descent_matrices<K>(F, S, B.W, it.l[0], it.l[1], it.l[2], steps);
            // E (its scaling columns) x descent
#pragma unroll
            for (int w = 0; w < MP; w++) {
                const int e = threadIdx.x + 256 * w;
                if (e < 3 * N2) {
                    const int dim = e / N2, r = (e % N2) / N, p = e % N;
                    double s = 0.0;
#pragma unroll
                    for (int j = 0; j < K; j++) s += B.E[r * N + j] * F[dim * KN + j * N + p];
                    M[e] = s;
                }
            }
            __syncthreads();
        }
        in.store(T, K <= 9 ? threadIdx.x : thread_here());  // (K = 10: the registers are full)
        Rows<N, N> m;
        if (steps == 0) m.load(B.E, N);
        __syncthreads();
        for (int dim = 0; dim < 3; dim++) {
            if (steps > 0) m.load(M + dim * N2, N);
            line_pass<N, N, N>(T, m, dim, N, N);
            __syncthreads();
        }
        if (q == 0) {
            const unsigned t0 = K <= 9 ? threadIdx.x : thread_here();
#pragma unroll
            for (int w = 0; w < PER; w++) {
                const int e = t0 + 256 * w;
                va[w] = N3 % 256 == 0 || e < N3 ? T[(e / N) * P + e % N] : 0.0;
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int w = 0; w < PER; w++) {
        const int e = threadIdx.x + 256 * w;
        if (N3 % 256 == 0 || e < N3) T[(e / N) * P + e % N] *= va[w];
    }
    Rows<N, N> m;
    m.load(B.C, N);
    __syncthreads();
    for (int dim = 0; dim < 3; dim++) {
        line_pass<N, N, N>(T, m, dim, N, N);
        __syncthreads();
    }
    const double h = geo.sfac * ldexp(1.0, -(geo.n0 + it.depth + 1));
    const double scale = J.coef / (h * sqrt(h));
    double ss[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        ss[c] = 0.0;
        for (int r = threadIdx.x; r < K3; r += 256) {
            const double v = T[padded_index<K>(c, r)] * scale;
            J.out[(size_t)it.node * 8 * K3 + c * K3 + r] = v;
            ss[c] += v * v;
        }
    }
    put_norms(ss, wsum, J.norm + (size_t)it.node * 8, compact + (size_t)blockIdx.x * 8);
}

// ----------------------------------------------------------------- sums

// out = sum of coef_k f_k at the listed output nodes, all terms at once.  A term that ends above
// the node contributes its descended scaling block only (the wavelet parts below a leaf are
// zero).  Bound by the reads of the terms, so two terms' are in flight.  As a chain of pairwise sums
// the 56 sums of an eight-orbital exchange step (k = 7) wrote and read every partial sum and
// cost a union grid and a round trip each: the SCF step of four orbitals 9.2 -> 7.6 ms, the density
// and Coulomb potential of six 4.1 -> 3.1, a five-orbital exchange step 20.9 -> 18.8.
template <int K>
__global__ void __launch_bounds__(256) k_sum(const SumItem *items, const SumSrc *srcs, DevBasis B, double *compact) {
    using L = PadT<K>;
    constexpr int N = L::N, P = L::P, K3 = K * K * K, KN = K * N, PER = NodeRegs<K>::PER;
    extern __shared__ double smem[];
    __shared__ double wsum[4][8];
    double *T = smem, *F = T + L::SIZE, *sc = F + 3 * KN;
    const SumItem it = items[blockIdx.x];
    const SumSrc *src = srcs + it.src0;
    bool any = false;  // sc holds the descended parts
    for (int q = 0; q < it.nsrc; q++) {
        const SumSrc t = src[q];
        if (t.steps == 0) continue;
        NodeRegs<K> in;
        in.load([&](unsigned e) { return t.p + e; });
        // (T as scratch; ends with a barrier)
        descent_matrices<K>(F, T, B.W, it.lx, it.ly, it.lz, (int)t.steps);
        in.store(T);
        __syncthreads();
        line_pass<N, K, N>(T, F, N, 0, N, N);
        __syncthreads();
        line_pass<N, K, N>(T, F + KN, N, 1, K, N);
        __syncthreads();
        line_pass<N, K, N>(T, F + 2 * KN, N, 2, K, K);
        __syncthreads();
        for (int e = threadIdx.x; e < K3; e += 256) {
            const int x = e % K, y = (e / K) % K, z = e / (K * K);
            const double v = t.coef * T[(z * N + y) * P + x];
            sc[e] = any ? sc[e] + v : v;
        }
        any = true;
        __syncthreads();
    }
    NodeRegs<K> acc;
#pragma unroll
    for (int w = 0; w < PER; w++) {
        const int e = threadIdx.x + 256 * w;
        acc.v[w] = any && e < K3 ? sc[e] : 0.0;
    }
    for (int q = 0; q < it.nsrc;) {
        // the next two terms given at the node itself
        while (q < it.nsrc && src[q].steps) q++;
        if (q == it.nsrc) break;
        const int qa = q++;
        while (q < it.nsrc && src[q].steps) q++;
        const bool two = q < it.nsrc;
        const SumSrc ta = src[qa], tb = src[two ? q : qa];
        q++;
        NodeRegs<K> va, vb;
        va.load([&](unsigned e) { return ta.p + e; });
        if (two) vb.load([&](unsigned e) { return tb.p + e; });
#pragma unroll
        for (int w = 0; w < PER; w++) {
            acc.v[w] += ta.coef * va.v[w];
            if (two) acc.v[w] += tb.coef * vb.v[w];
        }
    }
    double ss[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int w = 0; w < PER; w++) {
        const int e = threadIdx.x + 256 * w;
        if (8 * K3 % 256 != 0 && e >= 8 * K3) break;
        const int c = e / K3;
        const double v = acc.v[w];
        it.out[e] = v;
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (256 * w / K3 <= q && q <= (256 * w + 255) / K3) ss[q] += c == q ? v * v : 0.0;
    }
    put_norms(ss, wsum, it.norm, compact + (size_t)blockIdx.x * 8);
}

// ----------------------------------------------------------------- hydrogen functions

__device__ double d_hydrogen_orb(int N, int L, int M, double Z, double x, double y, double z) {
    const double r = sqrt(x * x + y * y + z * z);
    double c0;
    if (N == 1 && L == 0) c0 = 2.0;
    else if (N == 2 && L == 0) c0 = 1.0 / (2.0 * sqrt(2.0));
    else if (N == 3 && L == 0) c0 = 1.0 / (9.0 * sqrt(3.0));
    else if (N == 2 && L == 1) c0 = 1.0 / (2.0 * sqrt(6.0));
    else if (N == 3 && L == 1) c0 = 1.0 / (9.0 * sqrt(6.0));
    else if (N == 3 && L == 2) c0 = 1.0 / (9.0 * sqrt(30.0));
    else return 0.0;
    c0 *= pow(Z, 1.5);
    const double rho = 2.0 * Z / N * r;
    double poly;
    if (N == 1 && L == 0) poly = 1.0;
    else if (N == 2 && L == 0) poly = 2.0 - rho;
    else if (N == 3 && L == 0) poly = 6.0 - 6.0 * rho + rho * rho;
    else if (N == 2 && L == 1) poly = rho;
    else if (N == 3 && L == 1) poly = rho * (4.0 - rho);
    else poly = rho * rho;
    const double Rr = c0 * poly * exp(-rho / 2.0);
    double ang, ca;
    if (L == 0) {
        ca = 1.0;
        ang = 1.0;
    } else if (L == 1) {
        ca = sqrt(3.0);
        const double q = (M == 0) ? x : (M == 1) ? y : z;
        ang = (r > 0.0) ? q / r : 0.0;
    } else {
        const double r2 = r * r;
        ca = (M <= 2) ? sqrt(15.0) : (M == 3 ? sqrt(15.0 / 4.0) : sqrt(5.0 / 4.0));
        if (r2 == 0.0) ang = 0.0;
        else if (M == 0) ang = x * y / r2;
        else if (M == 1) ang = x * z / r2;
        else if (M == 2) ang = y * z / r2;
        else if (M == 3) ang = (x * x - y * y) / r2;
        else ang = (2.0 * z * z - x * x - y * y) / r2;
    }
    return Rr * ca / (2.0 * sqrt(M_PI)) * ang;
}

// hydrogen functions are not separable: values at the K^3 quadrature points of
// each child, then three 1D quadrature passes, then compression
template <int K>
__global__ void __launch_bounds__(256) k_project_hyd(const MulItem *items, ProjGeom geo, DevBasis B, int nterm, const double *coef,
                                                     const int *q, double Z, const double *origin, double *out,
                                                     double *norm, double *compact) {
    using L = PadT<K>;
    constexpr int N = L::N, P = L::P, N3 = N * N * N, K3 = K * K * K;
    extern __shared__ double smem[];
    double *T = smem;
    double *Qm = smem + L::SIZE;  // N x N block-diagonal quadrature matrix: phi_i(x_q) w_q * pre
    const MulItem it = items[blockIdx.x];
    const int node = it.node, d = it.depth;
    const double hc = geo.sfac * ldexp(1.0, -(geo.n0 + d + 1));
    const double pre = sqrt(hc);
    for (int e = threadIdx.x; e < N * N; e += blockDim.x) {
        const int p = e / N, qq = e % N;
        Qm[e] = ((p / K) == (qq / K)) ? B.phiq[(qq % K) * K + (p % K)] * B.qw[qq % K] * pre : 0.0;
    }
    for (int e = threadIdx.x; e < N3; e += blockDim.x) {
        const int px = e % N, py = (e / N) % N, pz = e / (N * N);
        const double x = geo.lo[0] + hc * ((double)(2 * it.l[0] + px / K) + B.qx[px % K]) - origin[0];
        const double y = geo.lo[1] + hc * ((double)(2 * it.l[1] + py / K) + B.qx[py % K]) - origin[1];
        const double z = geo.lo[2] + hc * ((double)(2 * it.l[2] + pz / K) + B.qx[pz % K]) - origin[2];
        double v = 0.0;
        for (int t = 0; t < nterm; t++) {
            double a = d_hydrogen_orb(q[6 * t], q[6 * t + 1], q[6 * t + 2], Z, x, y, z);
            if (q[6 * t + 3] > 0) a *= d_hydrogen_orb(q[6 * t + 3], q[6 * t + 4], q[6 * t + 5], Z, x, y, z);
            v += coef[t] * a;
        }
        T[(pz * N + py) * P + px] = v;
    }
    __syncthreads();
    for (int dim = 0; dim < 3; dim++) {
        line_pass<N, N, N>(T, Qm, N, dim, N, N);
        __syncthreads();
    }
    for (int dim = 0; dim < 3; dim++) {
        line_pass<N, N, N>(T, B.W, N, dim, N, N);
        __syncthreads();
    }
    __shared__ double wsum[4][8];
    double ss[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        ss[c] = 0.0;
        for (int r = threadIdx.x; r < K3; r += 256) {
            const double v = T[padded_index<K>(c, r)];
            out[(size_t)node * 8 * K3 + c * K3 + r] = v;
            ss[c] += v * v;
        }
    }
    put_norms(ss, wsum, norm + (size_t)node * 8, compact + (size_t)blockIdx.x * 8);
}

// ----------------------------------------------------------------- launchers

// kernels with more than 64 KiB of dynamic LDS must say so before their launch
template <class Kern>
static hipError_t allow_smem(Kern *k, size_t sm) {
    if (sm <= 65536) return hipSuccess;
    return hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
}

template <int K>
static constexpr size_t tensor_bytes(int extra) {
    return (size_t)(PadT<K>::SIZE + extra) * sizeof(double);
}

hipError_t launch_gen_compute(hipStream_t s, int first, int cap, const JobTab *jobs, const GenState &gs,
                              const double *W, int K, const int *firstp) {
    if (cap <= first) return hipSuccess;
    const int nb = std::min(cap - first, 2048);
    MWG_DISPATCH_K(K, {
        const size_t sm = tensor_bytes<KK>(6 * KK * KK);
        hipError_t e = allow_smem(k_gen_compute<KK>, sm);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_gen_compute<KK>, dim3(nb), dim3(256), sm, s, first, firstp, cap, jobs, gs, W);
    });
    return hipGetLastError();
}

hipError_t launch_transform(hipStream_t s, int mode, int n, const TransformItem *items, const double *M, int K,
                            double *compact) {
    if (n <= 0) return hipSuccess;
    MWG_DISPATCH_K(K, {
        const size_t sm = tensor_bytes<KK>(0);
        hipError_t e = allow_smem(k_transform<KK>, sm);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_transform<KK>, dim3(n), dim3(256), sm, s, mode, items, M, compact);
    });
    return hipGetLastError();
}

hipError_t launch_multiply(hipStream_t s, int n, const MulItem *items, const MulJobDev *jobs, const ProjGeom &geo,
                           const DevBasis &B, double *compact) {
    if (n <= 0) return hipSuccess;
    MWG_DISPATCH_K(B.K, {
        const size_t sm = tensor_bytes<KK>(12 * KK * KK);
        hipError_t e = allow_smem(k_multiply<KK>, sm);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_multiply<KK>, dim3(n), dim3(256), sm, s, items, jobs, geo, B, compact);
    });
    return hipGetLastError();
}

hipError_t launch_sum(hipStream_t s, int n, const SumItem *items, const SumSrc *srcs, const DevBasis &B,
                      double *compact) {
    if (n <= 0) return hipSuccess;
    MWG_DISPATCH_K(B.K, {
        const size_t sm = tensor_bytes<KK>(6 * KK * KK + KK * KK * KK);
        hipError_t e = allow_smem(k_sum<KK>, sm);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_sum<KK>, dim3(n), dim3(256), sm, s, items, srcs, B, compact);
    });
    return hipGetLastError();
}

hipError_t launch_project_hyd(hipStream_t s, int nw, const MulItem *items, const ProjGeom &geo, const DevBasis &B, int nterm, const double *coef, const int *q,
                              double Z, const double *origin, double *out, double *norm, double *compact) {
    if (nw <= 0) return hipSuccess;
    MWG_DISPATCH_K(B.K, {
        const size_t sm = tensor_bytes<KK>(4 * KK * KK);
        hipError_t e = allow_smem(k_project_hyd<KK>, sm);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_project_hyd<KK>, dim3(nw), dim3(256), sm, s, items, geo, B, nterm, coef, q, Z,
                           origin, out, norm, compact);
    });
    return hipGetLastError();
}

}  // namespace mwg
