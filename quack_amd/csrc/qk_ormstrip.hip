// Back-transformation Z <- Q Z of eigenvectors with the columns of Z held in
// registers (gfx950): LAPACK dormtr, SIDE = 'L', UPLO = 'U', TRANS = 'N', in blocks
// of 128 reflectors, Z(0:m, :) -= V (T (V^T Z(0:m, :))), as ormtr_apply (qk_sytrd.hip).
//
// There every block is four GEMMs whose 128-row products leave most CUs idle
// (n = 900: 8 blocks, 1.8 ms for 1.5 GFLOP; here 0.33.  n = 225: 0.44 and 0.038 ms,
// n = 2025: 3.8 and 1.16).  The columns of Z do not depend on each
// other, so here a workgroup takes 16 of them through all blocks in one launch:
// its eight waves hold the strip's 16-row tiles as matrix-core accumulators
// (row tile w + 8 u in wave w).  An f64 16x16x4 accumulator holds element (i, j) in lane
// j + 16 (i % 4), register i / 4, and the B operand of step r wants row k in lane
// group k: register r of a tile is the operand of its rows 4 r .. 4 r + 3 as it is, so
// neither product moves Z.  Only the 128 x 16 sums V^T Z cross waves, through LDS.
// V is read from the caches by every workgroup, in the layout each product reads
// 128 bytes at a time: by columns (V, rows fastest) for V W, transposed for V^T Z.
// Orders up to 2048: a thread holds n / 128 x 4 doubles of Z (64 at most).
#include "qk_kernels.h"

namespace qk {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
constexpr int OB = 128;  // reflectors per block
constexpr int NT = 512;

// V's padding (rows n .. np-1 and columns n-1 .. nbk-1) and, column by column,
// whatever of it A still holds: reflectors j >= m - 1 and, past row m, zeros.
// Then VT, its transpose (nbk fastest).  32 x 32 tiles through LDS.
__global__ __launch_bounds__(256) void k_orm_layouts(const double* __restrict__ A, long long sA, int n, int m, int np,
                                                     int nbk, double* __restrict__ V, double* __restrict__ VT,
                                                     long long sV) {
    __shared__ double t[32][33];
    A += blockIdx.z * sA;
    V += blockIdx.z * sV;
    VT += blockIdx.z * sV;
    const int r0 = blockIdx.x * 32, j0 = blockIdx.y * 32, x = threadIdx.x & 31, y = threadIdx.x >> 5;
    for (int jj = y; jj < 32; jj += 8) {
        const int r = r0 + x, j = j0 + jj;
        double v = 0.0;
        if (r < np && j < nbk) {
            if (r < m && j < m - 1) {
                v = V[r + (long long)np * j];
            } else {
                if (r < n && j < n - 1 && j >= m - 1) v = r < j ? A[r + (long long)n * (j + 1)] : (r == j ? 1.0 : 0.0);
                V[r + (long long)np * j] = v;
            }
        }
        t[jj][x] = v;
    }
    __syncthreads();
    for (int rr = y; rr < 32; rr += 8) {
        const int r = r0 + rr, j = j0 + x;
        if (r < np && j < nbk) VT[j + (long long)nbk * r] = t[x][rr];
    }
}

// G = V_b^T V_b of block b (128 x 128): a workgroup per 32 x 32 tile on or below the
// diagonal; its waves take the 16-row steps of V in turn, and their sums meet in LDS.
__global__ __launch_bounds__(NT) void k_orm_gram(const double* __restrict__ VT, long long sV, int np, int nbk,
                                                 double* __restrict__ G, long long sG) {
    __shared__ double part[8][4][4][64];
    VT += blockIdx.z * sV;
    const int b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l16 = lane & 15, q = lane >> 4;
    int ti = 0, tj = blockIdx.x;  // tile (ti, tj), ti >= tj, of 4 x 4
    while (tj > ti) tj -= ++ti;
    const int steps = min(OB * (b + 1), np) / 16;
    d4 acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    for (int st = w; st < steps; st += 8)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const double* p = VT + (long long)nbk * (16 * st + 4 * r + q) + OB * b + l16;
            double fa[2], fb[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                fa[x] = p[32 * ti + 16 * x];
                fb[x] = p[32 * tj + 16 * x];
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[x], fb[y], acc[x][y], 0, 0, 0);
        }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[w][2 * x + y][r][lane] = acc[x][y][r];
    __syncthreads();
    double* g = G + blockIdx.z * sG + (long long)b * OB * OB;
    for (int e = tid; e < 1024; e += NT) {
        const int ln = e & 63, r = (e >> 6) & 3, xy = e >> 8;
        double s = 0.0;
#pragma unroll
        for (int u = 0; u < 8; ++u) s += part[u][xy][r][ln];
        const int i = 32 * ti + 16 * (xy >> 1) + 4 * r + (ln >> 4), j = 32 * tj + 16 * (xy & 1) + (ln & 15);
        g[j + OB * i] = s;  // row by row, as k_orm_t reads it
    }
}

// T of each block, lower triangular with (V T V^T): rows i of column j solve
// T(i, j) = tau_i (delta_ij - sum_{j <= l < i} G(i, l) T(l, j)).  Eight lanes share a
// column (l = lane mod 8), a wave takes eight columns, so no barrier is needed; one
// workgroup per block and column by column it took 0.22 ms.
__global__ __launch_bounds__(256) void k_orm_t(const double* __restrict__ G, const double* __restrict__ TAU, long long sT,
                                               int n, double* __restrict__ T, long long sG) {
    const int b = blockIdx.y, lane = threadIdx.x & 63, sub = lane & 7;
    const int j = 32 * blockIdx.x + 8 * (threadIdx.x >> 6) + (lane >> 3);
    const double* g = G + blockIdx.z * sG + (long long)b * OB * OB;
    double* t = T + blockIdx.z * sG + (long long)b * OB * OB + (long long)OB * j;
    TAU += blockIdx.z * sT;
    double x[OB / 8];
#pragma unroll
    for (int u = 0; u < OB / 8; ++u) x[u] = 0.0;
#pragma unroll
    for (int v = 0; v < OB / 8; ++v)
        for (int c = 0; c < 8; ++c) {
            const int i = 8 * v + c;
            double s = 0.0;
#pragma unroll
            for (int u = 0; u <= v; ++u) {
                const int l = sub + 8 * u;
                s += (l < i ? g[l + OB * i] : 0.0) * x[u];  // x is zero before row j
            }
            s += __shfl_xor(s, 1, 64);
            s += __shfl_xor(s, 2, 64);
            s += __shfl_xor(s, 4, 64);
            const int ref = OB * b + i;
            const double tau = ref < n - 1 ? TAU[ref] : 0.0;
            const double val = i < j ? 0.0 : tau * ((i == j ? 1.0 : 0.0) - s);
            if (sub == c) {
                x[v] = val;
                t[i] = val;
            }
        }
}

template <int RT>
__global__ __launch_bounds__(NT) void k_orm_strip(const double* __restrict__ V, const double* __restrict__ VT,
                                                  long long sV, const double* __restrict__ T, long long sG, int n, int np,
                                                  int nbk, double* __restrict__ Z, long long sZ) {
    __shared__ double part[8][8][4][64];  // 128 KB: each wave's V^T Z
    __shared__ double sum[8][4][64];      // 128 x 16 in operand order
    const int z = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l16 = lane & 15, q = lane >> 4;
    V += z * sV;
    VT += z * sV;
    T += z * sG;
    const int col = blockIdx.x * 16 + l16;
    double* zc = Z + z * sZ + (long long)n * min(col, n - 1);
    d4 t[RT];
#pragma unroll
    for (int u = 0; u < RT; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * (w + 8 * u) + 4 * r + q;
            t[u][r] = row < n && col < n ? zc[row] : 0.0;
        }
    for (int b = 0; b < nbk / OB; ++b) {
        const int tiles = min(OB * (b + 1), np) / 16;
        {
            d4 acc[8];
#pragma unroll
            for (int x = 0; x < 8; ++x) acc[x] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int u = 0; u < RT; ++u)
                if (w + 8 * u < tiles) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const double* p = VT + (long long)nbk * (16 * (w + 8 * u) + 4 * r + q) + OB * b + l16;
                        double f[8];
#pragma unroll
                        for (int x = 0; x < 8; ++x) f[x] = p[16 * x];
#pragma unroll
                        for (int x = 0; x < 8; ++x)
                            acc[x] = __builtin_amdgcn_mfma_f64_16x16x4f64(f[x], t[u][r], acc[x], 0, 0, 0);
                        if (RT > 8) __builtin_amdgcn_sched_barrier(0);  // keeps the loads of one step only in registers
                    }
                }
#pragma unroll
            for (int x = 0; x < 8; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r) part[w][x][r][lane] = acc[x][r];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            double s = 0.0;
#pragma unroll
            for (int u = 0; u < 8; ++u) s += part[u][w][r][lane];
            sum[w][r][lane] = s;
        }
        __syncthreads();
        {
            // rows 16 w .. of T (V^T Z): T is lower triangular
            d4 acc = d4{0.0, 0.0, 0.0, 0.0};
            const double* tb = T + (long long)b * OB * OB + 16 * w + l16;
            for (int x = 0; x <= w; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(tb[OB * (16 * x + 4 * r + q)], sum[x][r][lane], acc, 0, 0, 0);
            __syncthreads();
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[w][r][lane] = -acc[r];
        }
        __syncthreads();
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            double f[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) f[r] = sum[x][r][lane];
#pragma unroll
            for (int u = 0; u < RT; ++u)
                if (w + 8 * u < tiles) {
                    const double* p = V + 16 * (w + 8 * u) + l16 + (long long)np * (OB * b + 16 * x + q);
                    double a[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) a[r] = p[(long long)np * 4 * r];
#pragma unroll
                    for (int r = 0; r < 4; ++r) t[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], f[r], t[u], 0, 0, 0);
                    if (RT > 8 && (u & 3) == 3) __builtin_amdgcn_sched_barrier(0);
                }
        }
        __syncthreads();  // sum is read by every wave
    }
    if (col < n)
#pragma unroll
        for (int u = 0; u < RT; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * (w + 8 * u) + 4 * r + q;
                if (row < n) zc[row] = t[u][r];
            }
}

int pad16(int n) { return (n + 15) / 16 * 16; }
int blocks_of(int n) { return (n - 1 + OB - 1) / OB; }

}  // namespace

int orm_strip_max() { return 2048; }
int orm_strip_ld(int n) { return pad16(n); }
// V, VT, G, T of one matrix
size_t orm_strip_doubles(int n) {
    const size_t nbk = (size_t)blocks_of(n) * OB;
    return 2 * nbk * pad16(n) + 2 * nbk * OB;
}

void orm_strip_prepare(hipStream_t s, int n, int batch, const double* A, long long sA, const double* TAU, long long sT,
                       double* work, int m) {
    if (n == 1) return;
    const int np = pad16(n), nb = blocks_of(n), nbk = nb * OB;
    const long long sW = orm_strip_doubles(n);
    double *VT = work + (size_t)nbk * np, *G = VT + (size_t)nbk * np, *T = G + (size_t)nbk * OB;
    hipLaunchKernelGGL(k_orm_layouts, dim3((np + 31) / 32, nbk / 32, batch), dim3(256), 0, s, A, sA, n, m, np, nbk, work, VT,
                       sW);
    hipLaunchKernelGGL(k_orm_gram, dim3(10, nb, batch), dim3(NT), 0, s, VT, sW, np, nbk, G, sW);
    hipLaunchKernelGGL(k_orm_t, dim3(OB / 32, nb, batch), dim3(256), 0, s, G, TAU, sT, n, T, sW);
    QK_HIP(hipGetLastError());
}

void orm_strip_apply(hipStream_t s, int n, int batch, double* Z, long long sZ, double* work) {
    QK_CHECK(n >= 1 && n <= orm_strip_max(), QK_E_ARG, "orm_strip: bad size");
    if (n == 1) return;
    const int np = pad16(n), nb = blocks_of(n), nbk = nb * OB;
    const long long sW = orm_strip_doubles(n);
    const double *V = work, *VT = work + (size_t)nbk * np, *T = VT + (size_t)nbk * np + (size_t)nbk * OB;
    const dim3 grid((n + 15) / 16, batch), blk(NT);
    const int rt = (np / 16 + 7) / 8;  // row tiles per wave
    auto go = [&](auto k) { hipLaunchKernelGGL(k, grid, blk, 0, s, V, VT, sW, T, sW, n, np, nbk, Z, sZ); };
    if (rt <= 2) go(k_orm_strip<2>);
    else if (rt <= 4) go(k_orm_strip<4>);
    else if (rt <= 8) go(k_orm_strip<8>);
    else if (rt <= 12) go(k_orm_strip<12>);
    else go(k_orm_strip<16>);
    QK_HIP(hipGetLastError());
}

}  // namespace qk
