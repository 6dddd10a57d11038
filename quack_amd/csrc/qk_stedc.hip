// Eigenvalues and eigenvectors of symmetric tridiagonal matrices (gfx950),
// batched: the middle part of the full eigensolve, between the
// tridiagonalisation and the back-transformation.
//
// Values only (tri_values): multisection with Sturm counts, as LAPACK's dstebz
// does it by bisection.  Each eigenvalue has a group of lanes that counts at
// as many interior points of its interval at once.
//
// With vectors (tri_vectors): Cuppen's divide and conquer (J. J. M. Cuppen,
// Numer. Math. 36 (1981) 177) with the deflation of LAPACK's dlaed2 and the
// re-derived z of M. Gu and S. C. Eisenstat (SIAM J. Matrix Anal. Appl. 16 (1995)
// 172), which makes the vectors orthogonal to working precision from roots
// that are accurate only to the last bits of their distance to a pole.  n is
// cut at floor(n i / 2^k) into leaves of at most 16, which Jacobi rotations solve;
// then, for the nodes of a level and all matrices together,
//   k_dc_setup    z, merge of the two sorted halves, deflation, column lists
//   k_dc_secular  one wave per root; further blocks rotate the columns of close poles
//   k_dc_zhat     one wave per pole
//   k_dc_vectors  one wave per column of the rank-one update's eigenvectors
//   k_dc_gemm     Q <- Q U on the matrix cores; further blocks copy the deflated columns
// Counts stay on the device: grids are sized for no deflation and blocks past
// the counts leave.  The two halves of Q are zero outside their own rows, so
// the columns go in the order first half, both (rotated), second half, and each
// half's rows meet only its own stretch of U (half the product).
// Bound: the chain of five launches a level for small orders, the last product for
// large ones.  RPA-like matrices: 0.33 ms at n = 225, 0.57 at 900, 1.15 at 2025, 7.2 at
// 5600, where rocSOLVER's dstedc took 36 (a thread per root) and 4.8 at 1326.
#include "qk_kernels.h"

namespace qk {
namespace {

constexpr double EPS = 1.1102230246251565e-16;  // 2^-53
constexpr int LEAF = 16;

__device__ inline double wsum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ inline double wmax(double v) {
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ inline double lane_of(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
// 1/x from the hardware reciprocal and two Newton steps
__device__ inline double rcp2(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}

// 1/sqrt(x) likewise
__device__ inline double rsq2(double x) {
    double r = __builtin_amdgcn_rsq(x);
    r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
    return fma(0.5 * r, fma(-x * r, r, 1.0), r);
}

// ---- scaling, bounds ----------------------------------------------------------
// One block per matrix: a power-of-two scale that brings max |T| to [1/2, 1), the
// Gershgorin interval, and info = 1 where an entry is not finite.  Such a matrix goes
// on as zeros (k_dc_leaf, k_dc_setup) and its values come out as NaN: the merges below
// index by the order of their values, which must be numbers.
// hd: [0] scale, [1] 1/scale, [2] lower bound, [3] upper bound, [4] 1 where not finite;
// de: 2 n scaled pairs (d_i, e_{i-1}^2) for the counts (null: not wanted).
__global__ __launch_bounds__(256) void k_tri_prep(const double* __restrict__ D, const double* __restrict__ E,
                                                  long long sd, int n, double* __restrict__ hd, double* __restrict__ de,
                                                  int* __restrict__ info) {
    __shared__ double s1[4], s2[4];
    const int z = blockIdx.x, t = threadIdx.x;
    D += z * sd;
    E += z * sd;
    hd += 8LL * z;
    double mx = 0.0;
    bool bad = false;
    for (int i = t; i < n; i += 256) {
        const double a = fabs(D[i]), b = i + 1 < n ? fabs(E[i]) : 0.0;
        bad = bad || !(a < 1e300) || !(b < 1e300);
        mx = fmax(mx, fmax(a, b));
    }
    mx = wmax(mx);
    if ((t & 63) == 0) s1[t >> 6] = mx;
    const int anybad = __syncthreads_or(bad ? 1 : 0);
    mx = fmax(fmax(s1[0], s1[1]), fmax(s1[2], s1[3]));
    int ex = 0;
    if (mx > 0.0 && !anybad) (void)frexp(mx, &ex);
    const double scale = ldexp(1.0, -ex);
    double lo = 1e300, hi = -1e300;
    for (int i = t; i < n; i += 256) {
        const double d = D[i] * scale;
        const double el = i > 0 ? fabs(E[i - 1]) * scale : 0.0, er = i + 1 < n ? fabs(E[i]) * scale : 0.0;
        lo = fmin(lo, d - el - er);
        hi = fmax(hi, d + el + er);
        if (de) {
            de[2LL * n * z + 2 * i] = d;
            de[2LL * n * z + 2 * i + 1] = fmax(el * el, EPS * EPS / 16.0);
        }
    }
    lo = -wmax(-lo);
    hi = wmax(hi);
    __syncthreads();
    if ((t & 63) == 0) {
        s1[t >> 6] = lo;
        s2[t >> 6] = hi;
    }
    __syncthreads();
    if (t == 0) {
        lo = fmin(fmin(s1[0], s1[1]), fmin(s1[2], s1[3]));
        hi = fmax(fmax(s2[0], s2[1]), fmax(s2[2], s2[3]));
        const double m = 4.0 * EPS * fmax(fabs(lo), fabs(hi)) * n + 1e-290;
        hd[0] = scale;
        hd[1] = ldexp(1.0, ex);
        hd[2] = lo - m;
        hd[3] = hi + m;
        hd[4] = anybad ? 1.0 : 0.0;
        info[z] = anybad ? 1 : 0;
    }
}

// ---- values only -------------------------------------------------------------------
// LPE lanes per eigenvalue.  The number of eigenvalues below x is the number of sign
// changes of p_i = (d_i - x) p_{i-1} - e_{i-1}^2 p_{i-2}: one dependent FMA a row
// where the pivots q_i = p_i / p_{i-1} need a reciprocal.  Rows go in eights between
// rescalings; e^2 is kept from vanishing (an eighth of an ulp of |T|), so that after a
// zero p_{i+1} has the sign opposite to p_{i-1}, whatever sign the zero carries,
// and eight rows neither overflow nor vanish.  More lanes per eigenvalue cut the
// passes (10 with 64, 14 with 16), fewer keep the waves few once n of them fill
// the device.  Intervals end at half an ulp of the largest |T|.  The pivot form,
// with its operands from global memory, took 1.1 ms at n = 900 and 8.5 at 5600.
constexpr int SR = 512;  // rows staged in LDS at a time
template <int LPE>
__global__ __launch_bounds__(256) void k_tri_values(const double* __restrict__ de, const double* __restrict__ hd, int n,
                                                    double* __restrict__ w, long long sw) {
    __shared__ double2 row[SR];
    __shared__ int more;
    const int z = blockIdx.y, t = threadIdx.x;
    const int g = (blockIdx.x * 256 + t) / LPE;
    const int k = min(g, n - 1);  // groups past the end repeat the last
    const int l = t & (LPE - 1);
    const int first = (t & 63) & ~(LPE - 1);
    const double2* __restrict__ p = reinterpret_cast<const double2*>(de) + (long long)n * z;
    const double back = hd[8LL * z + 1];
    double lo = hd[8LL * z + 2], hi = hd[8LL * z + 3];
    const double tol = EPS * 0.5 * fmax(fabs(lo), fabs(hi));
    for (int pass = 0; pass < 16; ++pass) {
        if (t == 0) more = 0;
        __syncthreads();
        if (hi - lo > tol) more = 1;
        __syncthreads();
        if (!more) break;
        const double x = lo + (hi - lo) * ((l + 1) * (1.0 / (LPE + 1)));
        int cnt = 0;
        double p1 = 1.0, p2 = 0.0;
        for (int b = 0; b < n; b += SR) {
            const int rows = min(SR, n - b);
            __syncthreads();
            for (int i = t; i < rows; i += 256) row[i] = p[b + i];
            for (int i = rows + t; i < ((rows + 7) & ~7); i += 256) row[i] = double2{1e4, 0.0};  // no change of sign
            __syncthreads();
            for (int i = 0; i < rows; i += 8) {
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const double2 r = row[i + u];
                    const double q = fma(r.x - x, p1, -(r.y * p2));
                    cnt += (unsigned)(__double2hiint(q) ^ __double2hiint(p1)) >> 31;
                    p2 = p1;
                    p1 = q;
                }
                const int e1 = p1 != 0.0 ? __builtin_amdgcn_frexp_exp(p1) : -2000;
                const int e2 = p2 != 0.0 ? __builtin_amdgcn_frexp_exp(p2) : -2000;
                const int ex = -max(e1, e2);
                p1 = ldexp(p1, ex);
                p2 = ldexp(p2, ex);
            }
        }
        const unsigned long long bal = __ballot(cnt > k) >> first;
        const unsigned long long m = LPE == 64 ? bal : bal & ((1ULL << (LPE & 63)) - 1);
        const int f = m ? __builtin_ctzll(m) : LPE;  // first point with more than k eigenvalues below it
        const double xl = __shfl(x, first + (f > 0 ? f - 1 : 0), 64), xh = __shfl(x, first + (f < LPE ? f : 0), 64);
        lo = f > 0 ? xl : lo;
        hi = f < LPE ? xh : hi;
    }
    if (l == 0 && g < n) w[z * sw + g] = hd[8LL * z + 4] == 0.0 ? 0.5 * (lo + hi) * back : __builtin_nan("");
}

// ---- leaves --------------------------------------------------------------------------
// boundary i of 2^k pieces
__host__ __device__ inline int cut(int n, int i, int k) { return (int)(((long long)n * i) >> k); }

// One wave per leaf: cyclic Jacobi in LDS, 8 disjoint rotations at a time in
// the round-robin order.  Writes the sorted eigenvalues (scaled) and the block of Q.
// Leaves of 32 by 256 threads took 0.19 ms (31 rounds a sweep, three barriers each);
// a wave needs no barrier, and the level more that leaves of 16 cost is 25 us.
__global__ __launch_bounds__(64) void k_dc_leaf(const double* __restrict__ D, const double* __restrict__ E,
                                                long long sd, const double* __restrict__ hd, int n, int k,
                                                double* __restrict__ d, long long sdd, double* __restrict__ Q,
                                                long long sQ) {
    constexpr int LD = LEAF + 1;
    __shared__ double A[LEAF * LD], V[LEAF * LD];
    __shared__ double dv[LEAF];
    const int z = blockIdx.y, t = threadIdx.x;
    D += z * sd;
    E += z * sd;
    const double scale = hd[8LL * z];
    const bool ok = hd[8LL * z + 4] == 0.0;
    const int p0 = cut(n, blockIdx.x, k), p1 = cut(n, blockIdx.x + 1, k), m = p1 - p0;
    for (int x = t; x < LEAF * LD; x += 64) {
        A[x] = 0.0;
        V[x] = 0.0;
    }
    __syncthreads();
    if (t < m) {
        double v = D[p0 + t] * scale;
        if (t == 0 && p0 > 0) v -= fabs(E[p0 - 1]) * scale;
        if (t == m - 1 && p1 < n) v -= fabs(E[p1 - 1]) * scale;
        A[t * LD + t] = ok ? v : 0.0;
        V[t * LD + t] = 1.0;
        if (t + 1 < m) A[t * LD + t + 1] = A[(t + 1) * LD + t] = ok ? E[p0 + t] * scale : 0.0;
    }
    __syncthreads();
    const int me = (m + 1) & ~1;  // players (one may sit out)
    const int pr = t >> 3, r0 = t & 7;
    for (int sweep = 0; sweep < 16; ++sweep) {
        bool turned = false;
        for (int rd = 0; rd < me - 1; ++rd) {
            // round robin: player me-1 stays, the others move round; the eight lanes of a pair
            // all work out its rotation
            int a = pr == 0 ? me - 1 : rd + pr, b = pr == 0 ? rd : rd + me - 1 - pr;
            if (pr != 0) {
                a = a >= me - 1 ? a - (me - 1) : a;
                b = b >= me - 1 ? b - (me - 1) : b;
            }
            if (a > b) {
                const int x = a;
                a = b;
                b = x;
            }
            // Rutishauser's form (H. Rutishauser, Numer. Math. 9 (1966) 1): elements change by
            // s times a correction, and the pivot's block by t a_pq, so that the small
            // rotations of the last sweeps add next to no rounding
            double s = 0.0, h = 0.0, na = 0.0, nb = 0.0;
            const bool on = pr < me / 2 && b < m;
            if (on) {
                const double apq = A[a * LD + b], app = A[a * LD + a], aqq = A[b * LD + b];
                if (fabs(apq) > EPS * 0.125) {  // |T| is about 1
                    const double th = (aqq - app) * rcp2(2.0 * apq), q = 1.0 + th * th;
                    const double tt = copysign(rcp2(fabs(th) + q * rsq2(q)), th);
                    const double c = rsq2(1.0 + tt * tt);
                    s = tt * c;
                    h = s * rcp2(1.0 + c);
                    na = app - tt * apq;
                    nb = aqq + tt * apq;
                    turned = true;
                }
            }
            __syncthreads();
            if (s != 0.0)
                for (int r = r0; r < m; r += 8) {
                    double x = A[r * LD + a], y = A[r * LD + b];
                    A[r * LD + a] = x - s * (y + h * x);
                    A[r * LD + b] = y + s * (x - h * y);
                    x = V[r * LD + a];
                    y = V[r * LD + b];
                    V[r * LD + a] = x - s * (y + h * x);
                    V[r * LD + b] = y + s * (x - h * y);
                }
            __syncthreads();
            if (s != 0.0)
                for (int r = r0; r < m; r += 8) {
                    const double x = A[a * LD + r], y = A[b * LD + r];
                    const bool pa = r == a, pb = r == b;  // the pivot's own block
                    A[a * LD + r] = pa ? na : pb ? 0.0 : x - s * (y + h * x);
                    A[b * LD + r] = pb ? nb : pa ? 0.0 : y + s * (x - h * y);
                }
            __syncthreads();
        }
        if (__ballot(turned) == 0) break;
    }
    if (t < m) dv[t] = A[t * LD + t];
    __syncthreads();
    Q += z * sQ;
    for (int x = t; x < m * m; x += 64) {
        const int r = x % m, c = x / m;
        int rank = 0;
        for (int i = 0; i < m; ++i) rank += dv[i] < dv[c] || (dv[i] == dv[c] && i < c);
        rank = min(rank, m - 1);
        Q[(p0 + r) + (long long)n * (p0 + rank)] = V[r * LD + c];
        if (r == 0) d[z * sdd + p0 + rank] = dv[c];
    }
}

// ---- one level of merges ---------------------------------------------------------------
// Work arrays of a matrix, all indexed by position 0..n-1 (a node uses its own
// stretch s..t-1), column numbers relative to the node.
struct Dc {
    int n, k, lev;  // nodes of this level: pieces 2^(lev+1) j .. 2^(lev+1) (j+1), lev = 0 first
    const double *E, *hd;
    long long sE, sm;         // strides of E and of the work arrays below
    double *d, *dn;           // values before and after, ascending in each node
    double *cd, *cz;          // survivors of the first deflation test, in order
    double *dk, *zk;          // poles and weights
    double *mu, *lam, *zh;    // roots: distance to the pole org, value; re-derived z
    double *dd;               // deflated values
    double *rc, *rs;          // rotations
    int *csrc, *cty, *cfl;    // survivors: column, type, kept
    int *col, *kp;            // columns in product order and their pole
    int *dcol, *org, *pos;    // deflated columns, root's pole, root's place
    int *ra, *rb;             // rotated column pairs
    int* nd;                  // 8 per node: K, k1 + k2, k1, rotations, deflated
    int ndstride;
    const double* Q;          // before
    double *Qn, *U;           // after; eigenvectors of the updates
    long long sQ, sU;
};
__device__ inline void node_of(const Dc& a, int j, int& s, int& m, int& t) {
    s = cut(a.n, (2 * j) << a.lev, a.k);
    m = cut(a.n, (2 * j + 1) << a.lev, a.k);
    t = cut(a.n, (2 * j + 2) << a.lev, a.k);
}

// position of this thread's flagged element among the block's flagged ones; total in tot
template <int NT>
__device__ inline int block_rank(bool f, int* sh, int& tot) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned long long b = __ballot(f);
    __syncthreads();
    if (lane == 0) sh[w] = __popcll(b);
    __syncthreads();
    int before = 0;
    tot = 0;
    for (int i = 0; i < NT / 64; ++i) {
        if (i < w) before += sh[i];
        tot += sh[i];
    }
    return before + __popcll(b & ((1ULL << lane) - 1));
}

// One block per node.
constexpr int ST = 512;
__global__ __launch_bounds__(ST) void k_dc_setup(Dc a) {
    __shared__ int sh[ST / 64];
    __shared__ double s1[ST / 64], s2[ST / 64];
    __shared__ int nrot;
    const int tid = threadIdx.x, lane = tid & 63, z = blockIdx.y;
    int s, m, t;
    node_of(a, blockIdx.x, s, m, t);
    const int N = t - s, n1 = m - s;
    const long long o = z * a.sm + s;
    const double* d = a.d + o;
    const double scale = a.hd[8LL * z];
    const double e = a.hd[8LL * z + 4] == 0.0 ? a.E[z * a.sE + m - 1] * scale : 0.0;
    const double rho = 2.0 * fabs(e), sg = (e < 0.0 ? -1.0 : 1.0) * 0.70710678118654752440;
    const double* Q = a.Q + z * a.sQ + (long long)a.n * s;
    // sorted merge of the halves into mu (values), lam (z), org (columns): free until the roots
    double *ds = a.mu + o, *zs = a.lam + o;
    int* src = a.org + o;
    // The places p are a permutation because each half's values ascend: k_dc_leaf sorts
    // them, and later ones are roots between poles that lie more than tol apart, and
    // deflated values by rank.  (Columns read back from src are held inside the node all
    // the same: a wrong one would send k_dc_gemm out of Q.)
    const auto source = [&](int i) { return (int)min((unsigned)src[i], (unsigned)(N - 1)); };
    double md = 0.0, mz = 0.0;
    for (int i = tid; i < N; i += ST) {
        const double x = d[i];
        const double zz = i < n1 ? 0.70710678118654752440 * Q[(m - 1) + (long long)a.n * i]
                                 : sg * Q[m + (long long)a.n * i];
        int lo = i < n1 ? n1 : 0, hi = i < n1 ? N : n1;
        const int base = lo;
        while (lo < hi) {  // entries of the other half before x (equal ones: the first half's go first)
            const int c = (lo + hi) >> 1;
            const bool less = i < n1 ? d[c] < x : d[c] <= x;
            if (less) lo = c + 1;
            else hi = c;
        }
        const int p = (i < n1 ? i : i - n1) + lo - base;
        ds[p] = x;
        zs[p] = zz;
        src[p] = i;
        md = fmax(md, fabs(x));
        mz = fmax(mz, fabs(zz));
    }
    md = wmax(md);
    mz = wmax(mz);
    if (lane == 0) {
        s1[tid >> 6] = md;
        s2[tid >> 6] = mz;
    }
    if (tid == 0) nrot = 0;
    __syncthreads();
    md = mz = 0.0;
    for (int i = 0; i < ST / 64; ++i) {
        md = fmax(md, s1[i]);
        mz = fmax(mz, s2[i]);
    }
    const double tol = 8.0 * EPS * fmax(md, mz);
    // small z deflate
    double *cd = a.cd + o, *cz = a.cz + o, *dd = a.dd + o;
    int *csrc = a.csrc + o, *cty = a.cty + o, *cfl = a.cfl + o, *dcol = a.dcol + o;
    int M = 0, nd = 0;
    for (int b = 0; b < N; b += ST) {
        const int i = b + tid;
        const double x = i < N ? ds[i] : 0.0, zz = i < N ? zs[i] : 0.0;
        const bool keep = i < N && rho * fabs(zz) > tol;
        int tot;
        const int r = block_rank<ST>(keep, sh, tot);
        if (keep) {
            cd[M + r] = x;
            cz[M + r] = zz;
            csrc[M + r] = source(i);
            cty[M + r] = source(i) < n1 ? 0 : 2;
            cfl[M + r] = 1;
        } else if (i < N) {
            const int q = nd + tid - r;  // dropped so far
            dd[q] = x;
            dcol[q] = source(i);
        }
        M += tot;
        nd += min(ST, N - b) - tot;
    }
    __syncthreads();
    // close poles: the first wave walks windows of 64 that overlap by one; a lane tests
    // its pair, and the pairs up to the first hit stand
    if (tid < 64) {
        double cx = 0.0, cy = 0.0;  // carried first element
        int ct = 0, nr = 0;
        for (int p = 0; p < M - 1; p += 63) {
            const int i = p + lane;
            double x = i < M ? cd[i] : 0.0, y = i < M ? cz[i] : 0.0;
            int ty = i < M ? cty[i] : 0;
            if (p > 0 && lane == 0) {
                x = cx;
                y = cy;
                ty = ct;
            }
            int from = 0;
            while (from < 63) {
                const double xn = __shfl_down(x, 1, 64), yn = __shfl_down(y, 1, 64);
                const bool hit = lane >= from && lane < 63 && i + 1 < M &&
                                 fabs((xn - x) * y * yn) <= tol * (y * y + yn * yn);
                const unsigned long long b = __ballot(hit);
                if (b == 0) break;
                const int f = __builtin_ctzll(b);
                const double d0 = lane_of(x, f), d1 = lane_of(x, f + 1), z0 = lane_of(y, f), z1 = lane_of(y, f + 1);
                const int t0 = __builtin_amdgcn_readlane(ty, f), t1 = __builtin_amdgcn_readlane(ty, f + 1);
                const double tau = sqrt(z0 * z0 + z1 * z1), c = z1 / tau, sn = -z0 / tau;
                const int tn = t0 == t1 ? t0 : 1;
                if (lane == f) {
                    x = d0 * c * c + d1 * sn * sn;
                    cd[i] = x;
                    cfl[i] = 0;
                    a.ra[o + nr] = csrc[i];
                    a.rb[o + nr] = csrc[i + 1];
                    a.rc[o + nr] = c;
                    a.rs[o + nr] = sn;
                }
                if (lane == f + 1) {
                    x = d0 * sn * sn + d1 * c * c;
                    y = tau;
                    ty = tn;
                    cd[i] = x;
                    cz[i] = y;
                    cty[i] = ty;
                }
                ++nr;
                from = f + 1;
            }
            cx = lane_of(x, 63);
            cy = lane_of(y, 63);
            ct = __builtin_amdgcn_readlane(ty, 63);
        }
        if (lane == 0) nrot = nr;
    }
    __syncthreads();
    // poles, and the other deflated columns
    int K = 0;
    int cnt[3] = {0, 0, 0};
    for (int b = 0; b < M; b += ST) {
        const int i = b + tid;
        const bool on = i < M, keep = on && cfl[i] != 0;
        int tot;
        const int r = block_rank<ST>(keep, sh, tot);
        if (keep) {
            a.dk[o + K + r] = cd[i];
            a.zk[o + K + r] = cz[i];
        } else if (on) {
            const int q = nd + tid - r;
            dd[q] = cd[i];
            dcol[q] = csrc[i];
        }
        K += tot;
        nd += min(ST, M - b) - tot;
    }
    // product order by type
    int done = 0;
    for (int ty = 0; ty < 3; ++ty) {
        int kk = 0;
        for (int b = 0; b < M; b += ST) {
            const int i = b + tid;
            const bool keep = i < M && cfl[i] != 0, f = keep && cty[i] == ty;
            int tot, tk;
            const int rk = block_rank<ST>(keep, sh, tk);
            const int r = block_rank<ST>(f, sh, tot);
            if (f) {
                a.col[o + done + cnt[ty] + r] = csrc[i];
                a.kp[o + done + cnt[ty] + r] = kk + rk;
            }
            kk += tk;
            cnt[ty] += tot;
        }
        done += cnt[ty];
    }
    if (tid == 0) {
        int* nn = a.nd + (long long)z * a.ndstride + 8 * blockIdx.x;
        nn[0] = K;
        nn[1] = cnt[0] + cnt[1];
        nn[2] = cnt[0];
        nn[3] = nrot;
        nn[4] = nd;
    }
}

// One wave per root j of 1/rho + sum_i z_i^2 / (d_i - x), x between pole j and the
// next: x = d_org + mu with the nearer pole as org, so that the distances to both
// neighbours keep full relative accuracy.  Steps solve the two-pole model that
// matches value and slope of the sums left and right of x (R.-C. Li, LAPACK Working
// Note 89); a step out of the bracket is replaced by bisection.  Blocks past the
// roots rotate the columns of close poles, a thread per row.
__global__ __launch_bounds__(256) void k_dc_secular(Dc a, int rootblocks) {
    const int z = blockIdx.z;
    int s, m, t;
    node_of(a, blockIdx.y, s, m, t);
    const int* nn = a.nd + (long long)z * a.ndstride + 8 * blockIdx.y;
    const int K = nn[0];
    const long long o = z * a.sm + s;
    if ((int)blockIdx.x >= rootblocks) {
        const int nr = nn[3], N = t - s;
        double* Q = const_cast<double*>(a.Q) + z * a.sQ + (long long)a.n * s + s;
        const int r = ((int)blockIdx.x - rootblocks) * 256 + threadIdx.x;
        if (r < N)
            for (int i = 0; i < nr; ++i) {
                double *x = Q + r + (long long)a.n * a.ra[o + i], *y = Q + r + (long long)a.n * a.rb[o + i];
                const double c = a.rc[o + i], sn = a.rs[o + i], u = *x, v = *y;
                *x = c * u + sn * v;
                *y = c * v - sn * u;
            }
        return;
    }
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (j >= K) return;
    const double *dk = a.dk + o, *zk = a.zk + o;
    const double rho = 2.0 * fabs(a.E[z * a.sE + m - 1] * a.hd[8LL * z]);
    const double rinv = 1.0 / rho;
    const bool lastr = j == K - 1;
    int org = j;
    double lo, hi, mu;
    if (lastr) {
        double s2 = 0.0;
        for (int i = lane; i < K; i += 64) s2 += zk[i] * zk[i];
        lo = 0.0;
        hi = rho * wsum(s2) * (1.0 + 8.0 * EPS);
        mu = 0.5 * hi;
    } else {
        lo = 0.0;
        hi = 0.5 * (dk[j + 1] - dk[j]);
        mu = hi;
    }
    if (K == 1) {
        if (lane == 0) {
            a.mu[o] = rho * zk[0] * zk[0];
            a.org[o] = 0;
            a.lam[o] = dk[0] + a.mu[o];
        }
        return;
    }
    // pole fixed on the left of the step model, and on the right (the last root: j-1 and j)
    const int pl = lastr ? j - 1 : j, pr = lastr ? j : j + 1;
    double dorg = dk[org];
    for (int it = 0; it < 120; ++it) {
        double psi = 0.0, phi = 0.0, dpsi = 0.0, dphi = 0.0;
        for (int i = lane; i < K; i += 64) {
            const double r = rcp2((dk[i] - dorg) - mu), zz = zk[i];
            const double u = zz * (zz * r), du = (zz * r) * (zz * r);
            if (i <= pl) {
                psi += u;
                dpsi += du;
            } else {
                phi += u;
                dphi += du;
            }
        }
        psi = wsum(psi);
        phi = wsum(phi);
        dpsi = wsum(dpsi);
        dphi = wsum(dphi);
        const double g = rinv + psi + phi;
        if (it == 0 && !lastr) {
            // the midpoint tells which pole is nearer
            if (g < 0.0) {
                org = j + 1;
                const double half = hi;
                dorg = dk[org];
                mu = -half;
                lo = -half;
                hi = 0.0;
            }
        } else if (g > 0.0) {
            hi = mu;
        } else {
            lo = mu;
        }
        if (fabs(g) <= EPS * (8.0 * (rinv + fabs(psi) + fabs(phi)) + fabs(mu) * (dpsi + dphi)) ||
            !(hi - lo > 2.0 * EPS * fmax(fabs(lo), fabs(hi))))
            break;
        const double dl = (dk[pl] - dorg) - mu, dr = (dk[pr] - dorg) - mu;
        const double c = rinv + (psi - dpsi * dl) + (phi - dphi * dr);
        const double b1 = dpsi * dl * dl, b2 = dphi * dr * dr;
        const double aa = c * (dl + dr) + b1 + b2, bb = dl * dr * g;
        const double disc = sqrt(fabs(aa * aa - 4.0 * bb * c));
        double eta;
        if (lastr) eta = aa >= 0.0 ? (aa + disc) / (2.0 * c) : 2.0 * bb / (aa - disc);
        else eta = c == 0.0 ? bb / aa : aa <= 0.0 ? (aa - disc) / (2.0 * c) : 2.0 * bb / (aa + disc);
        if (!(g * eta < 0.0)) eta = -g / (dpsi + dphi);
        double next = mu + eta;
        if (!(next > lo && next < hi)) {
            if (lo > 0.0) next = sqrt(lo) * sqrt(hi);
            else if (hi < 0.0) next = -sqrt(-lo) * sqrt(-hi);
            else next = it < 8 ? 0.5 * (lo + hi) : (lo + hi) * 0.0009765625;  // a root next to its pole
            if (!(next > lo && next < hi)) next = 0.5 * (lo + hi);
        }
        mu = next;
    }
    if (lane == 0) {
        a.mu[o + j] = mu;
        a.org[o + j] = org;
        a.lam[o + j] = dorg + mu;
    }
}

// One wave per pole: z_i^2 rho = (lam_last - d_i) prod_{j<i} (lam_j - d_i)/(d_j - d_i)
// prod_{i<=j<last} (lam_j - d_i)/(d_{j+1} - d_i), every factor below one but the first.
__global__ __launch_bounds__(256) void k_dc_zhat(Dc a) {
    const int z = blockIdx.z;
    int s, m, t;
    node_of(a, blockIdx.y, s, m, t);
    const int K = a.nd[(long long)z * a.ndstride + 8 * blockIdx.y];
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= K) return;
    const long long o = z * a.sm + s;
    const double *dk = a.dk + o, *mu = a.mu + o;
    const int* org = a.org + o;
    const double di = dk[i];
    double p = 1.0;
    for (int j = lane; j < K; j += 64) {
        const double num = (dk[org[j]] - di) + mu[j];
        if (j == K - 1) p *= num;
        else p *= num / (dk[j < i ? j : j + 1] - di);
    }
    for (int w = 32; w > 0; w >>= 1) p *= __shfl_xor(p, w, 64);
    if (lane == 0) a.zh[o + i] = copysign(sqrt(fabs(p)), a.zk[o + i]);
}

// One wave per root: its place among all the node's new values, its column of U
// (rows in product order), normalised.
__global__ __launch_bounds__(256) void k_dc_vectors(Dc a) {
    const int z = blockIdx.z;
    int s, m, t;
    node_of(a, blockIdx.y, s, m, t);
    const int* nn = a.nd + (long long)z * a.ndstride + 8 * blockIdx.y;
    const int K = nn[0], nd = nn[4];
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (j >= K) return;
    const long long o = z * a.sm + s;
    const double *dk = a.dk + o, *zh = a.zh + o, *dd = a.dd + o;
    const int* kp = a.kp + o;
    const double lam = a.lam[o + j], mu = a.mu[o + j], dorg = dk[a.org[o + j]];
    int below = 0;
    for (int i = lane; i < nd; i += 64) below += dd[i] < lam;
    for (int w = 32; w > 0; w >>= 1) below += __shfl_xor(below, w, 64);
    if (lane == 0) {
        a.pos[o + j] = j + below;
        a.dn[o + j + below] = lam;
    }
    double nrm = 0.0;
    for (int i = lane; i < K; i += 64) {
        const double u = zh[i] * rcp2((dk[i] - dorg) - mu);
        nrm += u * u;
    }
    const double inv = 1.0 / sqrt(wsum(nrm));
    double* U = a.U + z * a.sU + s + (long long)a.n * (s + j);
    for (int r = lane; r < K; r += 64) {
        const int i = kp[r];
        U[r] = zh[i] * rcp2((dk[i] - dorg) - mu) * inv;
    }
}

typedef double d4 __attribute__((ext_vector_type(4)));

// Qn(:, pos[j]) = sum_r Q(:, col[r]) U(r, j): tiles of 32 BK x 32 BK (2 x 2 waves of
// BK x BK 16x16 accumulators), the rows of the two halves in tiles of their own, each
// against its stretch of r; K in slabs of 16, the next slab in registers while one
// is used.  Blocks past the tiles copy the deflated columns, a wave each.
template <int BK>
__global__ __launch_bounds__(256, 2) void k_dc_gemm(Dc a, int tm, int tn) {
    constexpr int BM = 32 * BK, PAD = BM + 2, KT = 16, LD = BM * KT / 256;
    __shared__ double As[KT * PAD], Bs[KT * PAD];
    const int z = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int s, m, t;
    node_of(a, blockIdx.y, s, m, t);
    const int* nn = a.nd + (long long)z * a.ndstride + 8 * blockIdx.y;
    const int K = nn[0], nd = nn[4], N = t - s, n1 = m - s;
    const long long o = z * a.sm + s;
    const double* Q = a.Q + z * a.sQ + s + (long long)a.n * s;
    double* Qn = a.Qn + z * a.sQ + s + (long long)a.n * s;
    if ((int)blockIdx.x >= tm * tn) {
        const int q = ((int)blockIdx.x - tm * tn) * 4 + wave;
        if (q >= nd) return;
        const double x = a.dd[o + q];
        int lo = 0, hi = K;  // roots not above x
        while (lo < hi) {
            const int c = (lo + hi) >> 1;
            if (a.lam[o + c] <= x) lo = c + 1;
            else hi = c;
        }
        int p = 0;
        for (int i = lane; i < nd; i += 64) {
            const double y = a.dd[o + i];
            p += y < x || (y == x && i < q);
        }
        for (int w = 32; w > 0; w >>= 1) p += __shfl_xor(p, w, 64);
        p += lo;
        const double* from = Q + (long long)a.n * a.dcol[o + q];
        double* to = Qn + (long long)a.n * p;
        for (int r = lane; r < N; r += 64) to[r] = from[r];
        if (lane == 0) a.dn[o + p] = x;
        return;
    }
    const int tm1 = (n1 + BM - 1) / BM;
    const int ti = blockIdx.x % tm, j0 = (int)(blockIdx.x / tm) * BM;
    const bool second = ti >= tm1;
    const int m0 = second ? n1 + (ti - tm1) * BM : ti * BM, mend = second ? N : n1;
    if (m0 >= mend || j0 >= K) return;
    const int k0 = second ? nn[2] : 0, k1 = second ? K : nn[1];
    const int* col = a.col + o;
    const double* U = a.U + z * a.sU + s + (long long)a.n * s;
    const int wm = (wave & 1) * 16 * BK, wn = (wave >> 1) * 16 * BK, l16 = lane & 15, lk = lane >> 4;
    double ra[LD], rb[LD];
    auto fetch = [&](int kb) {
#pragma unroll
        for (int u = 0; u < LD; ++u) {
            const int x = tid + u * 256;
            const int i = x % BM, ka = kb + x / BM;
            ra[u] = m0 + i < mend && ka < k1 ? Q[m0 + i + (long long)a.n * col[ka]] : 0.0;
            const int kk = kb + x % KT, j = x / KT;
            rb[u] = kk < k1 && j0 + j < K ? U[kk + (long long)a.n * (j0 + j)] : 0.0;
        }
    };
    d4 acc[BK][BK];
#pragma unroll
    for (int x = 0; x < BK; ++x)
#pragma unroll
        for (int y = 0; y < BK; ++y) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    fetch(k0);
    for (int kb = k0; kb < k1; kb += KT) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < LD; ++u) {
            const int x = tid + u * 256;
            As[(x / BM) * PAD + x % BM] = ra[u];
            Bs[(x % KT) * PAD + x / KT] = rb[u];
        }
        __syncthreads();
        if (kb + KT < k1) fetch(kb + KT);
#pragma unroll
        for (int kk = 0; kk < KT; kk += 4) {
            double fa[BK], fb[BK];
#pragma unroll
            for (int x = 0; x < BK; ++x) {
                fa[x] = As[(kk + lk) * PAD + wm + x * 16 + l16];
                fb[x] = Bs[(kk + lk) * PAD + wn + x * 16 + l16];
            }
#pragma unroll
            for (int x = 0; x < BK; ++x)
#pragma unroll
                for (int y = 0; y < BK; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[y], fa[x], acc[x][y], 0, 0, 0);
        }
    }
    // acc[x][y][r] at this lane: row wm + 16 x + l16, column wn + 16 y + lk + 4 r
#pragma unroll
    for (int x = 0; x < BK; ++x) {
        const int i = m0 + wm + x * 16 + l16;
        if (i >= mend) continue;
#pragma unroll
        for (int y = 0; y < BK; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = j0 + wn + y * 16 + lk + 4 * r;
                if (j < K) Qn[i + (long long)a.n * a.pos[o + j]] = acc[x][y][r];
            }
    }
}

// w = d / scale (NaN for a matrix that is not finite)
__global__ void k_dc_out(const double* __restrict__ d, long long sdd, const double* __restrict__ hd, int n,
                         double* __restrict__ w, long long sw) {
    const int i = blockIdx.x * 256 + threadIdx.x, z = blockIdx.y;
    if (i < n) w[z * sw + i] = hd[8LL * z + 4] == 0.0 ? d[z * sdd + i] * hd[8LL * z + 1] : __builtin_nan("");
}

__global__ void k_dc_zero(double* __restrict__ x, long long count) {
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < count; t += (long long)gridDim.x * blockDim.x)
        x[t] = 0.0;
}

constexpr int NDBL = 12, NINT = 9;  // arrays of doubles (values twice) and of ints per matrix

int dc_levels(int n) {
    int k = 0;
    while ((n + (1 << k) - 1) >> k > LEAF) ++k;
    return k;
}

}  // namespace

size_t tri_work_doubles(int n, int batch, bool vectors) {
    const size_t b = batch, N = n;
    if (!vectors) return b * (8 + 2 * N) + 1;
    const size_t nodes = (size_t)1 << dc_levels(n);
    return b * (8 + NDBL * N + (NINT * N + 8 * nodes + 1) / 2 + 1);
}

void tri_values(hipStream_t s, int n, const double* D, const double* E, long long sd, int batch, double* w, long long sw,
                double* work, int* info) {
    double *hd = work, *de = work + 8 * (size_t)batch;
    hipLaunchKernelGGL(k_tri_prep, dim3(batch), dim3(256), 0, s, D, E, sd, n, hd, de, info);
    QK_HIP(hipGetLastError());
    // 64 lanes an eigenvalue until that is some 8 waves a CU on all 256
    if ((long long)n * batch <= 2048)
        hipLaunchKernelGGL(k_tri_values<64>, dim3((n + 3) / 4, batch), dim3(256), 0, s, de, hd, n, w, sw);
    else
        hipLaunchKernelGGL(k_tri_values<16>, dim3((n + 15) / 16, batch), dim3(256), 0, s, de, hd, n, w, sw);
    QK_HIP(hipGetLastError());
}

void tri_vectors(hipStream_t s, int n, const double* D, const double* E, long long sd, int batch, double* w, long long sw,
                 double* Z, double* Z2, long long sZ, double* U, long long sU, double* work, int* info) {
    QK_CHECK(n >= 1 && batch >= 1 && batch <= 65535 && (batch == 1 || sZ == (long long)n * n), QK_E_ARG,
             "tri_vectors: bad size");
    const int k = dc_levels(n);
    const size_t b = batch, N = n;
    double* hd = work;
    double* p = hd + 8 * b;
    const auto dbl = [&] {
        double* r = p;
        p += b * N;
        return r;
    };
    Dc a{};
    a.n = n;
    a.k = k;
    a.E = E;
    a.hd = hd;
    a.sE = sd;
    a.sm = n;
    double* dv[2] = {dbl(), dbl()};
    for (double** x : {&a.cd, &a.cz, &a.dk, &a.zk, &a.mu, &a.lam, &a.zh, &a.dd, &a.rc, &a.rs}) *x = dbl();
    int* q = reinterpret_cast<int*>(p);
    for (int** x : {&a.csrc, &a.cty, &a.cfl, &a.col, &a.kp, &a.dcol, &a.org, &a.pos, &a.ra}) {
        *x = q;
        q += b * N;
    }
    a.rb = a.pos;  // the pairs are used up before the roots' places are set
    a.nd = q;
    a.ndstride = 8 << k;
    a.U = U;
    a.sU = sU;
    a.sQ = sZ;
    hipLaunchKernelGGL(k_tri_prep, dim3(batch), dim3(256), 0, s, D, E, sd, n, hd, (double*)nullptr, info);
    QK_HIP(hipGetLastError());
    double* q2[2] = {Z, Z2};
    int cur = k & 1;  // the last level writes Z
    if (k > 0)
        for (double* x : q2) {
            const long long cnt = (long long)n * n * batch;
            hipLaunchKernelGGL(k_dc_zero, dim3((unsigned)std::min<long long>((cnt + 255) / 256, 8192)), dim3(256), 0, s, x,
                               cnt);
            QK_HIP(hipGetLastError());
        }
    hipLaunchKernelGGL(k_dc_leaf, dim3(1 << k, batch), dim3(64), 0, s, D, E, sd, hd, n, k, dv[0], (long long)n, q2[cur],
                       sZ);
    QK_HIP(hipGetLastError());
    int dc = 0;
    for (int lev = 0; lev < k; ++lev) {
        const int nodes = 1 << (k - lev - 1);
        const int big = (n + nodes - 1) / nodes, half = (big + 1) / 2 + 1;  // largest node, largest half
        a.lev = lev;
        a.d = dv[dc];
        a.dn = dv[dc ^ 1];
        a.Q = q2[cur];
        a.Qn = q2[cur ^ 1];
        const int quarters = (big + 3) / 4;
        hipLaunchKernelGGL(k_dc_setup, dim3(nodes, batch), dim3(ST), 0, s, a);
        hipLaunchKernelGGL(k_dc_secular, dim3(quarters + (big + 255) / 256, nodes, batch), dim3(256), 0, s, a, quarters);
        hipLaunchKernelGGL(k_dc_zhat, dim3(quarters, nodes, batch), dim3(256), 0, s, a);
        hipLaunchKernelGGL(k_dc_vectors, dim3(quarters, nodes, batch), dim3(256), 0, s, a);
        QK_HIP(hipGetLastError());
        // 128 x 128 tiles once they fill the device
        const long long t128 = 2LL * ((half + 127) / 128) * ((big + 127) / 128) * nodes * batch;
        if (t128 >= 256) {
            const int tm = 2 * ((half + 127) / 128), tn = (big + 127) / 128;
            hipLaunchKernelGGL(k_dc_gemm<4>, dim3(tm * tn + quarters, nodes, batch), dim3(256), 0, s, a, tm, tn);
        } else {
            const int tm = 2 * ((half + 63) / 64), tn = (big + 63) / 64;
            hipLaunchKernelGGL(k_dc_gemm<2>, dim3(tm * tn + quarters, nodes, batch), dim3(256), 0, s, a, tm, tn);
        }
        QK_HIP(hipGetLastError());
        cur ^= 1;
        dc ^= 1;
    }
    hipLaunchKernelGGL(k_dc_out, dim3((n + 255) / 256, batch), dim3(256), 0, s, dv[dc], (long long)n, hd, n, w, sw);
    QK_HIP(hipGetLastError());
}

}  // namespace qk
