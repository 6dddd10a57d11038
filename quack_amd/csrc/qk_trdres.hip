// Householder tridiagonalisation with the matrix held in registers (gfx950).
//
// Same result as sytrd_upper (qk_sytrd.hip; LAPACK dsytd2, UPLO = 'U'), for
// matrices of order n <= 3072 and for the leading block of that order
// that is left of a larger one.  The launch-per-step form pays two launches
// a column (about 16 us a column at n = 1326, whatever the work); here one
// launch runs every column and the G workgroups that share a matrix meet once
// a column.
//
// Layout.  Workgroup g owns the full rows r = g (mod G), so y = A v needs no
// sum over workgroups, and the rows that are still active stay balanced as the
// matrix shrinks.  At column c every workgroup
//   1. applies the previous column's A -= v w^T + w v^T to its rows and forms
//      y_r = A_r v in the same pass over its registers;
//   2. publishes its y_r; the owner of row c-1 publishes that row as well;
//   3. reads all of y and row c-1, and from them computes w and the next
//      column x = A(:, c-1) - v w_{c-1} - w and its reflector.  Every workgroup
//      does the same arithmetic in the same order, so all hold the same bits
//      and no second exchange is needed.
// The exchange carries its own arrival flags: each double travels as two 64-bit
// words, half of the value beside the column number, stored and loaded with
// single agent-scope atomics, so a reader that sees the column number has the
// value (one trip through the shared cache instead of store, counter, poll and
// load).  Two buffers alternate, so a reader of column c has to be done before anyone
// writes column c-2.  A writer of c-2 has read the y of column c-1 of every workgroup that
// has a row there (g < c-1), and those publish it after reading c.  The others must not
// read c: workgroup g > 0 leaves once it has published column g+1, its last rows' y, and
// the reflector goes to memory from the workgroup of row c-1, which has one in column c.
// (Workgroup 0 has row 0 in every column and stays to the end.)
//
// Two shapes of the same algorithm: k_trd_small (n <= 160) is one workgroup and
// needs no exchange; k_trd_wide (n <= 3072) spreads the columns over the 512
// or 256 threads of each of its workgroups.
//
// Bound: the latency of a column's chain (two sums over the columns, three barriers, the
// exchange), not arithmetic or memory.  What shortened it, at n = 900 from 5.6 to 3.0 ms:
// row c-1 goes out before the reflector is worked out, and only y is polled for once the
// row is there (5.1 -> 4.4 and 3.4 -> 2.9); 16 rows a workgroup instead of 32, no
// branch between the rows of a group.
// Measured per column: 1.5 us at n = 95, 1.6 at 128, 2.1 at 225, 2.4 at 324, 3.3 at 900,
// 3.7 at 1326, 4.1 at 2025, 5.2 at 2500, 7.3 at 3025; 24 matrices of 324 take 1.05 ms, one 0.77.
// About 45 % of a column is the wait for the others' y.
//
// Waits end: a reader that sees no progress for SPIN_TICKS raises *fail, which
// the other workgroups read, and all leave; the caller then runs sytrd_upper, and its
// owner's later solves do so at once (Resident).  A launch takes 25 ms at most, but its
// workgroups may come late by the length of whatever kernel another stream of the
// process has on the device (0.7 s: the densities of 600 orbitals in FP64).
// Launches whose workgroups wait for each other are kept one after another on
// the device (resident_gate), each with no more workgroups than it holds.
#include <mutex>

#include "qk_kernels.h"

namespace qk {
namespace {

typedef unsigned long long u64;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

constexpr int TT = 512;  // threads per CU: two waves per SIMD, 256 VGPRs each
constexpr long long SPIN_TICKS = 200000000LL;  // 2 s of the 100 MHz clock

__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int CTRL>
__device__ inline double row_rot(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// sum over the 16 lanes of a row, in every lane of it
__device__ inline double row_sum(double v) {
    v += row_rot<0x128>(v);
    v += row_rot<0x124>(v);
    v += row_rot<0x122>(v);
    v += row_rot<0x121>(v);
    return v;
}
// v_permlane32_swap / v_permlane16_swap of two doubles, then their sum: the upper
// half (odd rows) of a changes places with the lower half (even rows) of b
__device__ inline double swap32_add(double a, double b) {
    const u32x2 l = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const u32x2 h = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}
__device__ inline double swap16_add(double a, double b) {
    const u32x2 l = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const u32x2 h = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}
// sum over the wave, in every lane
__device__ inline double wave_sum(double v) {
    v = row_sum(v);
    v = swap16_add(v, v);
    return swap32_add(v, v);
}
// four wave sums at once: lanes of row q (16 lanes) get the sum of a[q]
__device__ inline double wave_sum4(const double* a) {
    const double s0 = swap32_add(a[0], a[2]), s1 = swap32_add(a[1], a[3]);
    return row_sum(swap16_add(s0, s1));
}
__device__ inline double lane_value(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// sum of N values st apart in LDS, N a power of two, as a tree
template <int N>
__device__ inline double tree_sum(const double* v, int st) {
    double t[N];
#pragma unroll
    for (int i = 0; i < N; ++i) t[i] = v[i * st];
#pragma unroll
    for (int m = N / 2; m > 0; m /= 2)
#pragma unroll
        for (int i = 0; i < m; ++i) t[i] += t[i + m];
    return t[0];
}

// one double with its column number beside either half
__device__ inline void publish(u64* w, double v, unsigned tag) {
    const u64 t = (u64)tag << 32;
    __hip_atomic_store(w, t | (unsigned)__double2loint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(w + 1, t | (unsigned)__double2hiint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline bool arrived(const u64* w, unsigned tag, double& v) {
    const u64 a = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const u64 b = __hip_atomic_load(w + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = __hiloint2double((int)(unsigned)b, (int)(unsigned)a);
    return (unsigned)(a >> 32) == tag && (unsigned)(b >> 32) == tag;
}
// bookkeeping of a wait; true when it has to be given up
__device__ inline bool give_up(unsigned& spins, long long& t0, int* fail) {
    if ((++spins & 255) != 0) return false;
    if (__hip_atomic_load(fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return true;
    const long long t = wall_clock64();
    if (t0 == 0) t0 = t;
    if (t - t0 < SPIN_TICKS) return false;
    __hip_atomic_store(fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

struct TrdArgs {
    const double* A;  // upper triangle read
    long long lda, sA;
    int n, G;
    double* V;  // reflectors, v_j in column j (rows < n), or null
    long long ldv, sV;
    double *D, *E, *TAU;
    long long sd;  // stride of D, E, TAU between matrices
    u64* X;        // exchange words, 8 n per matrix, zeroed
    int* fail;
};

__device__ inline double load_sym(const double* A, long long lda, int r, int col) {
    return col <= r ? A[col + lda * r] : A[r + lda * col];
}

struct Reflector {
    double beta, tau, scale;
};
__device__ inline Reflector reflector(double alpha, double xx) {
    Reflector h;
    if (xx == 0.0) {
        h.beta = alpha;
        h.tau = 0.0;
        h.scale = 0.0;
    } else {
        // beta = -sign(alpha) |x|, tau = (beta - alpha) / beta, scale = 1 / (alpha - beta), from the
        // hardware's reciprocal (square root) and Newton steps: every column waits for them
        const double s = alpha * alpha + xx, a = fabs(alpha);
        double r = __builtin_amdgcn_rsq(s);
        r = fma(0.5 * r, fma(-s * r, r, 1.0), r);
        r = fma(0.5 * r, fma(-s * r, r, 1.0), r);
        double nrm = s * r;
        nrm = fma(0.5 * r, fma(-nrm, nrm, s), nrm);
        h.beta = alpha >= 0.0 ? -nrm : nrm;
        h.tau = fma(a, r, 1.0);
        const double d = a + nrm;
        double q = __builtin_amdgcn_rcp(d);
        q = fma(q, fma(-d, q, 1.0), q);
        q = fma(q, fma(-d, q, 1.0), q);
        h.scale = alpha >= 0.0 ? q : -q;
    }
    return h;
}

// One workgroup per matrix: n <= 64 KC, n <= 8 R.  Wave q owns rows q + 8 j, j < R; lane l
// holds columns l + 64 k of them.  Every wave has all columns, so all sums stay inside
// a wave; y and row c-1 pass through LDS, one barrier a column.
template <int KC, int R>
__global__ __launch_bounds__(TT) void k_trd_small(TrdArgs p) {
    static_assert(R % 4 == 0, "rows go in fours");
    __shared__ double ys[2][64 * KC], as[2][64 * KC];
    __shared__ double2 vw[8][64 * KC];  // each wave's copy of (v, w), for its rows' entries
    const int z = blockIdx.x, n = p.n;
    const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
    const double* A = p.A + z * p.sA;
    double* V = p.V ? p.V + z * p.sV : nullptr;
    double *D = p.D + z * p.sd, *E = p.E + z * p.sd, *TAU = p.TAU + z * p.sd;
    double2* vwq = vw[q];
    double a[R][KC], v[KC], vp[KC], wp[KC], x[KC];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int r = q + 8 * j;
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int col = lane + 64 * k;
            a[j][k] = r < n && col < n ? load_sym(A, p.lda, r, col) : 0.0;
        }
    }
    int c = n - 1;
#pragma unroll
    for (int k = 0; k < KC; ++k) {
        const int col = lane + 64 * k;
        x[k] = col <= c ? A[col + p.lda * c] : 0.0;
        vp[k] = wp[k] = 0.0;
        vwq[col] = double2{0.0, 0.0};
        if (q == 0 && col == c) D[c] = x[k];
    }
    for (; c >= 1; --c) {
        const int par = c & 1;
        if (q == ((c - 1) & 7)) {  // row c-1, brought up to date
            const int jr = (c - 1) >> 3;
            const double2 f = vwq[c - 1];
#pragma unroll
            for (int j = 0; j < R; ++j)
                if (j == jr)
#pragma unroll
                    for (int k = 0; k < KC; ++k) {
                        const int col = lane + 64 * k;
                        if (col < c) as[par][col] = a[j][k] - f.x * wp[k] - f.y * vp[k];
                    }
        }
        // reflector of column c from x
        double xx = 0.0, sel = 0.0;
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int col = lane + 64 * k;
            if (k == (c - 1) >> 6) sel = x[k];
            if (col < c - 1) xx += x[k] * x[k];
        }
        const Reflector h = reflector(lane_value(sel, (c - 1) & 63), wave_sum(xx));
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int col = lane + 64 * k;
            v[k] = col < c - 1 ? x[k] * h.scale : (col == c - 1 ? 1.0 : 0.0);
        }
        // update of the previous column and y = A v, four rows at a time
#pragma unroll
        for (int j0 = 0; j0 < R; j0 += 4) {
            if (q + 8 * j0 < c) {
                double acc[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    // (rows past c are done: their v and w are zero, and nobody takes their y)
                    const double2 f = vwq[min(q + 8 * (j0 + u), n - 1)];
                    acc[u] = 0.0;
#pragma unroll
                    for (int k = 0; k < KC; ++k)
                        if (64 * k < c) {
                            const double t = a[j0 + u][k] - f.x * wp[k] - f.y * vp[k];
                            a[j0 + u][k] = t;
                            acc[u] += t * v[k];
                        }
                }
                const double y = wave_sum4(acc);
                const int r = q + 8 * (j0 + (lane >> 4));
                if ((lane & 15) == 0 && r < c) ys[par][r] = y;
            }
        }
        if (V && q == (c & 7)) {
#pragma unroll
            for (int k = 0; k < KC; ++k) {
                const int col = lane + 64 * k;
                if (col < n) V[col + p.ldv * (c - 1)] = v[k];
            }
        }
        if (threadIdx.x == 0) {
            E[c - 1] = h.beta;
            TAU[c - 1] = h.tau;
        }
        lds_barrier();
        // w = tau y - tau^2 (y . v) v / 2
        double y[KC], dot = 0.0;
        sel = 0.0;
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int col = lane + 64 * k;
            y[k] = col < c ? ys[par][col] : 0.0;
            x[k] = col < c ? as[par][col] : 0.0;
            dot += y[k] * v[k];
        }
        const double half = -0.5 * h.tau * h.tau * wave_sum(dot);
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            wp[k] = h.tau * y[k] + half * v[k];
            vp[k] = v[k];
            if (k == (c - 1) >> 6) sel = wp[k];
        }
        const double wl = lane_value(sel, (c - 1) & 63);
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int col = lane + 64 * k;
            x[k] = col < c ? x[k] - (v[k] * wl + wp[k]) : 0.0;  // v(c-1) = 1
            if (q == 0 && col == c - 1) D[c - 1] = x[k];
            vwq[col] = double2{v[k], wp[k]};
        }
    }
}

// n <= NT KC.  Workgroup g owns rows g + G j, j < R; thread t holds columns t + NT k
// of them.  Needs n <= R G.
template <int KC, int R, int NT>
__global__ __launch_bounds__(NT) void k_trd_wide(TrdArgs p) {
    static_assert(R % 4 == 0 && R <= 64, "rows go in fours");
    __shared__ double2 vw[NT * KC];  // (v, w)
    __shared__ double yp[NT / 64][R];
    __shared__ double red1[NT / 64], red2[NT / 64];
    __shared__ double ylast, xlast;
    __shared__ int quit;
    const int G = p.G, z = blockIdx.x / G, g = blockIdx.x % G, n = p.n;
    const int tid = threadIdx.x, lane = tid & 63, q = tid >> 6;
    const double* A = p.A + z * p.sA;
    double* V = p.V ? p.V + z * p.sV : nullptr;
    double *D = p.D + z * p.sd, *E = p.E + z * p.sd, *TAU = p.TAU + z * p.sd;
    u64* X = p.X + (long long)z * 8 * n;
    double a[R][KC], v[KC], vp[KC], wp[KC], x[KC];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int r = g + G * j;
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int col = tid + NT * k;
            a[j][k] = r < n && col < n ? load_sym(A, p.lda, r, col) : 0.0;
        }
    }
    int c = n - 1;
    double part = 0.0;
#pragma unroll
    for (int k = 0; k < KC; ++k) {
        const int col = tid + NT * k;
        x[k] = col <= c ? A[col + p.lda * c] : 0.0;
        vp[k] = wp[k] = 0.0;
        vw[col] = double2{0.0, 0.0};
        if (g == 0 && col == c) D[c] = x[k];
        if (col < c - 1) part += x[k] * x[k];
        if (col == c - 1) xlast = x[k];
    }
    part = wave_sum(part);
    if (lane == 0) red2[q] = part;
    if (tid == 0) quit = 0;
    lds_barrier();
    unsigned spins = 0;
    for (; c >= 1; --c) {
        const int par = c & 1;
        // row c-1, brought up to date, goes to everyone first: it is on its way while the
        // reflector and y are worked out
        if (g == (c - 1) % G) {
            const int jr = (c - 1) / G;
            const double2 f = vw[c - 1];
#pragma unroll
            for (int j = 0; j < R; ++j)
                if (j == jr)
#pragma unroll
                    for (int k = 0; k < KC; ++k) {
                        const int col = tid + NT * k;
                        const double t = a[j][k] - f.x * wp[k] - f.y * vp[k];
                        if (col < c) publish(X + 4LL * n * par + 2LL * n + 2 * col, t, c);
                    }
        }
        const Reflector h = reflector(xlast, tree_sum<NT / 64>(red2, 1));
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int col = tid + NT * k;
            v[k] = col < c - 1 ? x[k] * h.scale : (col == c - 1 ? 1.0 : 0.0);
        }
#pragma unroll
        for (int j0 = 0; j0 < R; j0 += 4) {
            if (g + G * j0 < c) {
                double acc[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (KC >= 5) __builtin_amdgcn_sched_barrier(0);  // registers for one row's loads at a time
                    // (rows past c are done: their v and w are zero, and nobody takes their y)
                    const double2 f = vw[min(g + G * (j0 + u), n - 1)];
                    acc[u] = 0.0;
#pragma unroll
                    for (int k = 0; k < KC; ++k)
                        if (NT * k < c) {
                            const double t = a[j0 + u][k] - f.x * wp[k] - f.y * vp[k];
                            a[j0 + u][k] = t;
                            acc[u] += t * v[k];
                        }
                }
                const double y = wave_sum4(acc);
                if ((lane & 15) == 0) yp[q][j0 + (lane >> 4)] = y;
            }
        }
        lds_barrier();
        if (tid < R) {
            const int r = g + G * tid;
            if (r < c) {
                publish(X + 4LL * n * par + 2 * r, tree_sum<NT / 64>(&yp[0][tid], R), c);
            }
        }
        if (V && g == (c - 1) % G) {
#pragma unroll
            for (int k = 0; k < KC; ++k) {
                const int col = tid + NT * k;
                if (col < n) V[col + p.ldv * (c - 1)] = v[k];
            }
        }
        if (g == 0 && tid == 0) {
            E[c - 1] = h.beta;
            TAU[c - 1] = h.tau;
        }
        // This workgroup's last rows are out.  It goes at the next return, after one look at
        // words that may be gone: a return here, or another bound of the loop, costs 34
        // registers (order 3072: 219 spilled instead of 54, 65 ms instead of 23).
        const bool leave = g > 0 && c <= g + 1;
        double y[KC], dot = 0.0;
        {
            long long t0 = 0;
            const u64* w = X + 4LL * n * par + 2 * tid;
            bool row = false;  // row c-1, sent early, is here
            for (;;) {
                bool all = true;
                if (!row) {
                    row = true;
#pragma unroll
                    for (int k = 0; k < KC; ++k) {
                        x[k] = 0.0;
                        if (tid + NT * k < c) row = arrived(w + 2LL * n + 2 * NT * k, c, x[k]) && row;
                    }
                }
#pragma unroll
                for (int k = 0; k < KC; ++k) {
                    y[k] = 0.0;
                    if (tid + NT * k < c) all = arrived(w + 2 * NT * k, c, y[k]) && all;
                }
                if ((all && row) || leave) break;
                if (give_up(spins, t0, p.fail)) {
                    quit = 1;
                    break;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            dot += y[k] * v[k];
            if (tid + NT * k == c - 1) ylast = y[k];
        }
        dot = wave_sum(dot);
        if (lane == 0) red1[q] = dot;
        lds_barrier();
        if (quit || leave) return;
        dot = tree_sum<NT / 64>(red1, 1);
        const double half = -0.5 * h.tau * h.tau * dot;
        const double wl = h.tau * ylast + half;  // w(c-1), v(c-1) = 1
        part = 0.0;
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int col = tid + NT * k;
            wp[k] = h.tau * y[k] + half * v[k];
            vp[k] = v[k];
            x[k] = col < c ? x[k] - (v[k] * wl + wp[k]) : 0.0;
            if (g == 0 && col == c - 1) D[c - 1] = x[k];
            vw[col] = double2{v[k], wp[k]};
            if (col < c - 2) part += x[k] * x[k];
            if (col == c - 2) xlast = x[k];
        }
        part = wave_sum(part);
        if (lane == 0) red2[q] = part;
        lds_barrier();
    }
}

__global__ void k_zero_words(u64* __restrict__ X, long long count) {
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < count; t += (long long)gridDim.x * blockDim.x)
        X[t] = 0;
}

// The kernels above wait inside a launch for the other workgroups of the same
// launch, so two such launches must not each hold a part of the device: every
// one waits for the one before it, on whatever stream that ran.
struct Gate {
    std::mutex mu;
    hipEvent_t last[64] = {};
};
Gate& gate() {
    static Gate* g = new Gate();  // lives until process exit, as the streams that wait on its events may
    return *g;
}
template <class F>
void resident_gate(hipStream_t s, F&& launch) {
    int dev = 0;
    QK_HIP(hipGetDevice(&dev));
    QK_CHECK(dev >= 0 && dev < 64, QK_E_HIP, "device number");
    Gate& g = gate();
    std::lock_guard<std::mutex> lock(g.mu);
    if (g.last[dev]) QK_HIP(hipStreamWaitEvent(s, g.last[dev], 0));
    else QK_HIP(hipEventCreateWithFlags(&g.last[dev], hipEventDisableTiming));
    launch();
    QK_HIP(hipGetLastError());
    QK_HIP(hipEventRecord(g.last[dev], s));
}

// Rows and threads of a workgroup and the kernel for them.  R KC register pairs hold a
// thread's share of A (at most 72 of the 128 pairs; the rest are the column vectors).
typedef void (*TrdKernel)(TrdArgs);
struct Shape {
    int top, rows, threads;  // largest order, rows and threads of a workgroup
    TrdKernel k;
};
#define QK_SMALL(KC, R) {64 * KC, 8 * R, TT, k_trd_small<KC, R>}
#define QK_WIDE(KC, R, NT) {NT * KC, R, NT, k_trd_wide<KC, R, NT>}
// In each range of orders the fastest shape for one matrix first, then those that take
// fewer workgroups a matrix.  Four waves instead of eight, with twice the columns a thread,
// halve the sums over a row and the barriers' skew (n = 225: 0.56 -> 0.50 ms, with 8
// rows 0.43; n = 474: 1.23 -> 1.17), up to where a thread's longer rows cost
// more (n = 1326: 4.8 -> 5.7).
const Shape SHAPES[] = {
    QK_SMALL(1, 8),      QK_SMALL(2, 16),     {160, 160, TT, k_trd_small<3, 20>},
    QK_WIDE(1, 8, 256),  QK_WIDE(1, 16, 256), QK_WIDE(1, 32, 256),
    QK_WIDE(2, 8, 256),  QK_WIDE(2, 16, 256), QK_WIDE(2, 32, 256),
    {1024, 8, 256, k_trd_wide<4, 8, 256>},    QK_WIDE(2, 16, 512), QK_WIDE(2, 32, 512),
    QK_WIDE(3, 12, 512), QK_WIDE(3, 24, 512),
    QK_WIDE(4, 8, 512),  QK_WIDE(4, 16, 512),
    QK_WIDE(5, 12, 512), QK_WIDE(6, 12, 512)};

// Matrices whose workgroups a launch holds at once: one of 512 or two of 256 threads a CU
// (what 256 registers a lane allow).
int trd_at_once(const Shape& s, int g) {
    int dev = 0, cu = 0;
    QK_HIP(hipGetDevice(&dev));
    QK_HIP(hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev));
    return cu * (TT / s.threads) / g;
}
// The first shape of n's range that takes the whole batch at once, else its last one:
// 24 matrices of order 324 take 1.53 ms with 8 rows a workgroup (four a CU), 1.05
// with 16, 1.22 with 32; 12 of order 474 2.13, 1.55 and 1.68.  Null where one
// matrix does not fit the device.
const Shape* trd_shape(int n, int batch) {
    const Shape* best = nullptr;
    for (const Shape& s : SHAPES) {
        if (n > s.top || (best && best->top != s.top)) continue;
        const int g = (n + s.rows - 1) / s.rows, most = trd_at_once(s, g);
        if (g > 1 && most < 1) continue;
        best = &s;
        if (g == 1 || batch <= most) break;
    }
    return best;
}

}  // namespace

int trd_resident_max() { return 3072; }
size_t trd_resident_words(int n, int batch) { return 8 * (size_t)n * batch + 1; }
const int* trd_resident_fail(int n, int batch, const double* words) {
    return reinterpret_cast<const int*>(words + trd_resident_words(n, batch) - 1);
}
bool trd_resident_fits(int n) { return n >= 1 && n <= trd_resident_max() && trd_shape(n, 1) != nullptr; }
bool trd_resident_waits(int n, int batch) { return n > trd_shape(n, batch)->rows; }

bool trd_resident(hipStream_t s, int n, const double* A, long long lda, long long sA, double* V, long long ldv,
                  long long sV, double* D, double* E, double* TAU, long long sd, int batch, double* words) {
    QK_CHECK(trd_resident_fits(n) && lda >= n && (!V || ldv >= n) && batch >= 1, QK_E_ARG, "trd_resident: bad size");
    const Shape& sh = *trd_shape(n, batch);
    const int G = (n + sh.rows - 1) / sh.rows;
    u64* X = reinterpret_cast<u64*>(words);  // exchange words, then the flag of a wait given up
    int* fail = reinterpret_cast<int*>(words + trd_resident_words(n, batch) - 1);
    const int per = G > 1 ? std::min(batch, trd_at_once(sh, G)) : batch;  // matrices of one launch
    if (G > 1) {
        const long long cnt = (long long)trd_resident_words(n, batch);
        hipLaunchKernelGGL(k_zero_words, dim3((unsigned)std::min<long long>((cnt + 255) / 256, 1024)), dim3(256), 0, s, X,
                           cnt);
        QK_HIP(hipGetLastError());
    }
    for (int b0 = 0; b0 < batch; b0 += per) {
        const int nb = std::min(per, batch - b0);
        TrdArgs p{A + b0 * sA, lda, sA, n, G, V ? V + b0 * sV : nullptr, ldv, sV, D + b0 * sd, E + b0 * sd,
                  TAU + b0 * sd, sd, X + 8LL * n * b0, fail};
        const dim3 grid(G * nb), blk(sh.threads);
        auto go = [&] { hipLaunchKernelGGL(sh.k, grid, blk, 0, s, p); };
        if (G > 1) resident_gate(s, go);
        else go();
        QK_HIP(hipGetLastError());
    }
    return G > 1;
}

}  // namespace qk
