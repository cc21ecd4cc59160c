// cad_mg.hip -- aggregation multigrid, the preconditioner of the mixed and
// learned forms, in FP32 (and in FP64 for measuring what FP32 buys).
//
// The mixed form solves the pressure system of VF_VPCOEF (the same FP64
// matrix AD..AUK, BB as the plain form) by FP64 iterative refinement around
// an FP32 BiCGSTAB (cad_refine.hip) whose preconditioner is one V-cycle of
// this multigrid.  It replaces the reference's MILU preconditioner
// (vf_mzdcmp.f, vf_mzminv.f), whose triangular sweeps are a serial chain:
// every multigrid pass is a data-parallel 7-point stencil bound by HBM
// bandwidth.
//
// Levels.  Level 0 is the pressure grid with the matrix rounded to FP32;
// inactive rows (INDC = -1) get AD = 1 and no couplings.  A coarse cell
// aggregates the 2x2x2 block of fine cells (fine interior index 2I-2, 2I-1 of
// coarse interior index I, 1-based with one ghost layer), and its row is the
// Galerkin product with piecewise-constant transfer over the active fine
// cells: the coarse diagonal sums the fine diagonals and the couplings
// between cells of the block, a coarse coupling sums the fine couplings that
// cross the block face.  The structure stays 7-point on every level.  A
// coarse row without active fine cells, or with a diagonal that is not
// positive, is inactive.
//
// Storage.  Each level stores the two colours of the red-black ordering
// apart: a (J,K) line of ld cells (NUMI rounded up to a multiple of eight) holds first its
// cells with I+J+K even, then those with I+J+K odd, each half in ascending
// I.  A half-sweep then reads and writes whole lines of its own colour and
// reads the other colour's x at the same positions of the neighbouring lines,
// so a thread's neighbours are its neighbour threads' cells and no line is
// fetched for half of its cells.
//
// V-cycle.  Red-black Gauss-Seidel (one sweep = the cells with I+J+K even,
// then odd) before and after the coarse correction; the residual of the fine
// cells is summed into the coarse right-hand side in one kernel (after the
// odd half-sweep only the even cells' residuals are not zero up to rounding);
// the coarse correction is added scaled by MG_SCALE (piecewise-constant
// prolongation under-corrects smooth errors), on the fly inside the even
// half-sweep that follows it; the coarsest level is smoothed MG_COARSE
// times.  Every level starts from x = 0, so the first (even) half of its
// first sweep is x = b/AD, which the kernel that sets b writes at once.  The
// coarsest levels run as one workgroup (k_mg_tail), so the small grids cost
// one launch instead of four per level.
#include "cad_common.h"

#include <algorithm>

#define RET_IF(x)              \
    do {                       \
        const int rc_ = (x);   \
        if (rc_ != CAD_OK)     \
            return rc_;        \
    } while (0)

namespace {

constexpr float MG_SCALE = 1.8f;
constexpr int MG_COARSE = 12;

// position of cell (i,j,k) (1-based, ghosts included) in a level's arrays (32
// bits: a grid of 2^31 cells has more than 500 GB of FP64 arrays)
template <typename L>
__device__ __forceinline__ int pos(const L &v, int i, int j, int k)
{
    return v.ld * ((j - 1) + v.d.nj * (k - 1)) + ((i + j + k) & 1) * (v.ld >> 1) + ((i - 1) >> 1);
}

__device__ __forceinline__ long long nat(const Dims &d, int i, int j, int k)
{
    return (long long)(i - 1) + (long long)d.ni * (j - 1) + d.nij * (k - 1);
}

// level 0 from the FP64 matrix
template <typename V>
__global__ void __launch_bounds__(256) k_mg_fine(Dims d, const double *__restrict__ ad,
                                                 const double *__restrict__ ali,
                                                 const double *__restrict__ alj,
                                                 const double *__restrict__ alk,
                                                 const double *__restrict__ aui,
                                                 const double *__restrict__ auj,
                                                 const double *__restrict__ auk,
                                                 const int *__restrict__ indc, MgLevelT<V> L,
                                                 long long n0, long long n1)
{
    const long long n = n0 + (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= n1) return;
    const int i = (int)(n % d.ni) + 1, j = (int)((n / d.ni) % d.nj) + 1, k = (int)(n / d.nij) + 1;
    const long long m = pos(L, i, j, k);
    const bool a = indc[n] != -1 && ad[n] > 0.0;
    const V r[7] = {a ? (V)ad[n] : (V)1, a ? (V)ali[n] : (V)0, a ? (V)alj[n] : (V)0, a ? (V)alk[n] : (V)0,
                    a ? (V)aui[n] : (V)0, a ? (V)auj[n] : (V)0, a ? (V)auk[n] : (V)0};
    L.act[m] = a ? 1 : 0;
    L.ad[m] = r[0];
    L.ali[m] = r[1];
    L.alj[m] = r[2];
    L.alk[m] = r[3];
    L.aui[m] = r[4];
    L.auj[m] = r[5];
    L.auk[m] = r[6];
}

// A cell's neighbours are all of the other colour: cell i of half-line position
// q is i = 2q+1+p, and its I neighbours are at positions q-1+p and q+p of its
// line's other half, its J and K neighbours at q of the other half of their
// lines.
template <typename V>
struct Cell {
    int n, o;      // position of the cell, and of position q of its line's other half
    int p;
};

template <typename V>
__device__ __forceinline__ Cell<V> cell_at(const MgLevelT<V> &L, int q, int i, int j, int k, int color)
{
    const int half = L.ld >> 1, line = L.ld * ((j - 1) + L.d.nj * (k - 1));
    return {line + color * half + q, line + (1 - color) * half + q, i - 2 * q - 1};
}

// Galerkin coarse row of coarse interior cell (I,J,K), K from k0; one thread
// per cell, its loads all in flight before the first is used: a term that does not
// count is added as 0, and the terms keep their order (with each cell's loads
// behind its activity the levels of 97x61x45 took 86 us a solve, now 44, and the
// first of 512x256x128 115, now 73).
template <typename V>
__global__ void __launch_bounds__(256) k_mg_coarsen(MgLevelT<V> F, MgLevelT<V> C, int k0)
{
    const int I = blockIdx.x * blockDim.x + threadIdx.x + 2;
    const int J = blockIdx.y * blockDim.y + threadIdx.y + 2;
    const int K = blockIdx.z + k0;
    if (I > C.d.ni - 1 || J > C.d.nj - 1 || K > C.d.nk - 1) return;
    const Dims &fd = F.d;
    V s_ad = 0, s_li = 0, s_lj = 0, s_lk = 0, s_ui = 0, s_uj = 0, s_uk = 0;
    bool any = false;
    const int lj = F.ld, lk = F.ld * fd.nj;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int oi = c & 1, oj = (c >> 1) & 1, ok = c >> 2;
        const int i0 = 2 * I - 2 + oi, j0 = 2 * J - 2 + oj, k0f = 2 * K - 2 + ok;
        const int i = min(i0, fd.ni - 1), j = min(j0, fd.nj - 1), k = min(k0f, fd.nk - 1);
        const Cell<V> e = cell_at(F, (i - 1) >> 1, i, j, k, (i + j + k) & 1);
        const V ad = F.ad[e.n], li = F.ali[e.n], ui = F.aui[e.n], vlj = F.alj[e.n], vuj = F.auj[e.n];
        const V vlk = F.alk[e.n], vuk = F.auk[e.n];
        const bool a = i == i0 && j == j0 && k == k0f && F.act[e.n] != 0;
        any = any || a;
        // a coupling counts towards an active neighbour
        auto on = [&](V v, int n) { return a && F.act[n] != 0 ? v : (V)0; };
        const V wli = on(li, e.o - 1 + e.p), wui = on(ui, e.o + e.p), wlj = on(vlj, e.o - lj), wuj = on(vuj, e.o + lj);
        const V wlk = on(vlk, e.o - lk), wuk = on(vuk, e.o + lk);
        s_ad += a ? ad : (V)0;
        // -I: inside the block when oi = 1
        if (oi) s_ad += wli; else s_li += wli;
        const bool in_i = !oi && i + 1 <= fd.ni - 1, in_j = !oj && j + 1 <= fd.nj - 1, in_k = !ok && k + 1 <= fd.nk - 1;
        s_ad += in_i ? wui : (V)0;
        s_ui += in_i ? (V)0 : wui;
        if (oj) s_ad += wlj; else s_lj += wlj;
        s_ad += in_j ? wuj : (V)0;
        s_uj += in_j ? (V)0 : wuj;
        if (ok) s_ad += wlk; else s_lk += wlk;
        s_ad += in_k ? wuk : (V)0;
        s_uk += in_k ? (V)0 : wuk;
    }
    const int m = pos(C, I, J, K);
    const bool a = any && s_ad > (V)0;
    C.act[m] = a ? 1 : 0;
    C.ad[m] = a ? s_ad : (V)1;
    C.ali[m] = a ? s_li : (V)0;
    C.alj[m] = a ? s_lj : (V)0;
    C.alk[m] = a ? s_lk : (V)0;
    C.aui[m] = a ? s_ui : (V)0;
    C.auj[m] = a ? s_uj : (V)0;
    C.auk[m] = a ? s_uk : (V)0;
}

// the off-diagonal part of the cell's row
template <typename V>
__device__ __forceinline__ V row_off(const MgLevelT<V> &L, const Cell<V> &c)
{
    const V *x = L.x;
    const int lj = L.ld, lk = L.ld * L.d.nj;
    return L.ali[c.n] * x[c.o - 1 + c.p] + L.aui[c.n] * x[c.o + c.p]
         + L.alj[c.n] * x[c.o - lj] + L.auj[c.n] * x[c.o + lj]
         + L.alk[c.n] * x[c.o - lk] + L.auk[c.n] * x[c.o + lk];
}

// The passes of a V-cycle are bound by HBM bandwidth on grids of millions of
// cells and by their loads' latency on small ones, where a pass is one round of
// loads if none waits for another's value.  So the activity is tested when the
// result is stored (an inactive row's operands are finite and in bounds), and
// only on levels of more than MG_SKIP_CELLS, whose waves without an active cell
// are worth skipping, before the loads (SKIP).  Tested first everywhere, the
// restriction took 6.6 us on 97x61x29 and 35.7 on 512x256x45 cells, the
// correction 5.7 and 41.5; now 4.6 and 31.7, 3.9 and 29.8.
constexpr long long MG_SKIP_CELLS = 1 << 20;

// one colour of a Gauss-Seidel sweep: thread x covers position q of its
// (J,K) line's half of that colour (cell I = 2q+1 or 2q+2), K from k0
template <typename V, bool SKIP>
__global__ void __launch_bounds__(256) k_mg_smooth(MgLevelT<V> L, int color, int k0)
{
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 2;
    const int k = blockIdx.z + k0;
    if (j > L.d.nj - 1 || k > L.d.nk - 1) return;
    const int q = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int i = 2 * q + 1 + ((color + 1 + j + k) & 1);
    if (i < 2 || i > L.d.ni - 1) return;
    const Cell<V> c = cell_at(L, q, i, j, k, color);
    const bool act = L.act[c.n] != 0;
    if (SKIP && !act) return;
    const V x = (L.b[c.n] - row_off(L, c)) / L.ad[c.n];
    if (act) L.x[c.n] = x;
}

// Coarse right-hand side = sum of the fine residuals of the block; coarse
// x = 0.  It follows the odd half-sweep, after which an odd cell's residual
// is zero up to rounding (its x was just solved from its row), so only the
// block's four even cells are summed, one on each of its (J,K) lines.
template <typename V, bool SKIP>
__device__ __forceinline__ V block_residual(const MgLevelT<V> &F, int I, int J, int K)
{
    Cell<V> e[4];
    bool act[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int j0 = 2 * J - 2 + (c & 1), k0 = 2 * K - 2 + (c >> 1), i0 = 2 * I - 2 + ((j0 + k0) & 1);
        const int i = min(i0, F.d.ni - 1), j = min(j0, F.d.nj - 1), k = min(k0, F.d.nk - 1);
        e[c] = cell_at(F, (i - 1) >> 1, i, j, k, 0);
        act[c] = i == i0 && j == j0 && k == k0 && F.act[e[c].n] != 0;
    }
    V s = 0;
    if (SKIP && !(act[0] || act[1] || act[2] || act[3])) return s;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const V r = F.b[e[c].n] - F.ad[e[c].n] * F.x[e[c].n] - row_off(F, e[c]);
        if (act[c]) s += r;
    }
    return s;
}

template <typename V, bool SKIP>
__global__ void __launch_bounds__(256) k_mg_restrict(MgLevelT<V> F, MgLevelT<V> C, int k0)
{
    const int I = blockIdx.x * blockDim.x + threadIdx.x + 2;
    const int J = blockIdx.y * blockDim.y + threadIdx.y + 2;
    const int K = blockIdx.z + k0;
    if (I > C.d.ni - 1 || J > C.d.nj - 1 || K > C.d.nk - 1) return;
    const long long m = pos(C, I, J, K);
    const bool act = C.act[m] != 0;
    const V ad = C.ad[m];
    const V s = block_residual<V, SKIP>(F, I, J, K);
    const V bc = act ? s : (V)0;
    C.b[m] = bc;
    // from x = 0 the even half of the first sweep is x = b/AD
    C.x[m] = act && ((I + J + K) & 1) == 0 ? bc / ad : (V)0;
}

// The coarse correction and the even half-sweep after it, in one pass.  The
// correction x += MG_SCALE * coarse x of the block matters only at the odd
// cells: the even half-sweep solves each even cell's x from its row, which
// reads the odd neighbours only.  So each even cell reads its odd
// neighbours' x plus their correction (what a separate correction pass would
// have stored), and the odd cells, which the odd half-sweep that follows
// solves from their rows in turn, are not corrected in memory.  Of the six
// neighbours one in each direction is in the cell's own block, so four coarse
// values serve them.
template <typename V, bool SKIP>
__global__ void __launch_bounds__(256) k_mg_correct_even(MgLevelT<V> F, MgLevelT<V> C, int k0)
{
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 2;
    const int k = blockIdx.z + k0;
    if (j > F.d.nj - 1 || k > F.d.nk - 1) return;
    const int q = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const int i = 2 * q + 1 + ((1 + j + k) & 1);
    if (i < 2 || i > F.d.ni - 1) return;
    const Cell<V> e = cell_at(F, q, i, j, k, 0);
    const bool act = F.act[e.n] != 0;
    if (SKIP && !act) return;
    const int I = (i + 2) >> 1, J = (j + 2) >> 1, K = (k + 2) >> 1;
    const bool oi = i & 1, oj = j & 1, ok = k & 1;   // the upper cell of its block
    const V own = C.x[pos(C, I, J, K)];
    const V xi = C.x[pos(C, oi ? I + 1 : I - 1, J, K)], xj = C.x[pos(C, I, oj ? J + 1 : J - 1, K)];
    const V xk = C.x[pos(C, I, J, ok ? K + 1 : K - 1)];
    const int lj = F.ld, lk = F.ld * F.d.nj;
    const int n6[6] = {e.o - 1 + e.p, e.o + e.p, e.o - lj, e.o + lj, e.o - lk, e.o + lk};
    const V c6[6] = {oi ? own : xi, oi ? xi : own, oj ? own : xj, oj ? xj : own, ok ? own : xk, ok ? xk : own};
    V y[6];
#pragma unroll
    for (int a = 0; a < 6; a++) {
        const V x = F.x[n6[a]];
        y[a] = F.act[n6[a]] ? x + (V)MG_SCALE * c6[a] : x;
    }
    const V off = F.ali[e.n] * y[0] + F.aui[e.n] * y[1] + F.alj[e.n] * y[2] + F.auj[e.n] * y[3]
                + F.alk[e.n] * y[4] + F.auk[e.n] * y[5];
    const V x = (F.b[e.n] - off) / F.ad[e.n];
    if (act) F.x[e.n] = x;
}

// level-0 right-hand side from a vector of the grid (natural order) on the K
// planes k0..k1 (the rows outside them are inactive: their x stays 0); from
// x = 0 the even half of the first sweep is x = b/AD
template <typename V, typename T>
__global__ void __launch_bounds__(256) k_mg_in(MgLevelT<V> L, const T *__restrict__ y, int k0)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 2;
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 2;
    const int k = blockIdx.z + k0;
    if (i > L.d.ni - 1 || j > L.d.nj - 1) return;
    const long long m = pos(L, i, j, k);
    const bool a = L.act[m] != 0;
    const V b = a ? (V)y[nat(L.d, i, j, k)] : (V)0;
    L.b[m] = b;
    L.x[m] = a && ((i + j + k) & 1) == 0 ? b / L.ad[m] : (V)0;
}

// the result from level 0 into a vector of the grid on the K planes k0..k1
// (0 on inactive rows)
template <typename V, typename T>
__global__ void __launch_bounds__(256) k_mg_out(const MgLevelT<V> L, T *__restrict__ x, int k0)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 2;
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 2;
    const int k = blockIdx.z + k0;
    if (i > L.d.ni - 1 || j > L.d.nj - 1) return;
    const long long m = pos(L, i, j, k);
    x[nat(L.d, i, j, k)] = L.act[m] ? (T)L.x[m] : (T)0;
}

// k_mg_out and, on the same rows, the level's residual b - A x in V (the
// learned preconditioner's input), with the block partials of its sum of
// squares and of the row count at part[b * stride] and part[b * stride + 1]
// (grid-stride over the K planes k0..k1, gridDim.x blocks of 256)
template <typename V, typename T>
__global__ void __launch_bounds__(256) k_mg_out_resid(const MgLevelT<V> L, T *__restrict__ x, T *__restrict__ r,
                                                      int k0, int k1, double *__restrict__ part, int stride)
{
    const int ni = L.d.ni - 2, nj = L.d.nj - 2;
    const long long total = (long long)ni * nj * (k1 - k0 + 1);
    double a = 0.0, cnt = 0.0;
    for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(e % ni) + 2;
        const long long q = e / ni;
        const int j = (int)(q % nj) + 2, k = (int)(q / nj) + k0;
        const long long m = pos(L, i, j, k), n = nat(L.d, i, j, k);
        if (!L.act[m]) {
            x[n] = (T)0;
            r[n] = (T)0;
            continue;
        }
        const V xm = L.x[m];
        const V rv = L.b[m] - L.ad[m] * xm - row_off(L, cell_at(L, (i - 1) >> 1, i, j, k, (i + j + k) & 1));
        x[n] = (T)xm;
        r[n] = (T)rv;
        a += (double)rv * (double)rv;
        cnt += 1.0;
    }
    __shared__ double sh[2][4];
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_down(a, o, 64);
        cnt += __shfl_down(cnt, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = a;
        sh[1][threadIdx.x >> 6] = cnt;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[(long long)blockIdx.x * stride] = sh[0][0] + sh[0][1] + sh[0][2] + sh[0][3];
        part[(long long)blockIdx.x * stride + 1] = sh[1][0] + sh[1][1] + sh[1][2] + sh[1][3];
    }
}

// The V-cycle below level t0 inside one workgroup (k_mg_tail): for each level
// down to the coarsest the odd half-sweep (the even half is set with b) and the
// coarse right-hand side; MG_COARSE sweeps on the coarsest; then up: the
// correction, the even half-sweep and the odd one.  Its time is the latency of
// some forty phases, so nothing in them touches memory: x is in LDS (natural
// order with a ghost layer), and each thread keeps its cells' rows and b in
// registers, loaded at once at the start.  On 32x16x8 cells and three levels
// below them this takes 17 us where phases that read the rows from memory took
// 34, on 64x4x12 and one below 13 against 25.
//
// A thread owns up to A cells of each colour on level t0 and, below it, two,
// one and one (a coarsened level has at most 27/125 of the cells).  The
// residuals of every level have their own zeroed place in LDS, so a block that
// reaches beyond the grid sums its ghost cells' zeros.
constexpr int TAIL_THREADS = 512;
constexpr int TAIL_LEVELS = 4;
constexpr int TAIL_LDS = 18432;              // values of x and residuals

template <typename V>
struct MgTail {
    MgLevelT<V> L[TAIL_LEVELS];
    float inv_h[TAIL_LEVELS], inv_j[TAIL_LEVELS];   // 1 / positions a half line, 1 / lines a plane
    int base[TAIL_LEVELS];                   // first LDS position of a level's x
    int res, nt;                             // residuals are res behind x; number of levels
};

template <typename V>
struct TailRow {
    V ad, li, ui, lj, uj, lk, uk, b;
    int o, n;                                // LDS position and position in the level; o < 0: no cell
    int up, src;                             // LDS positions of its coarse cell's x and of its block's first residual
    bool act;
};

// positions of a colour on the interior part of a half line
__device__ __host__ __forceinline__ int tail_half(int ni) { return (ni - 1) / 2; }

template <typename V>
__device__ __forceinline__ void tail_load(const MgTail<V> &T, int l, int color, int e, TailRow<V> &r)
{
    const MgLevelT<V> &L = T.L[l];
    const int ni = L.d.ni, nj = L.d.nj, nk = L.d.nk;
    // e / h: (e + 1/2) / h is at least 1/2h from a whole number, far beyond the product's rounding
    const int line = (int)(((float)e + 0.5f) * T.inv_h[l]), u = e - line * tail_half(ni);
    const int kk = (int)(((float)line + 0.5f) * T.inv_j[l]), k = kk + 2, j = line - kk * (nj - 2) + 2;
    const int i = 2 * u + 2 + ((color + j + k) & 1);
    const bool in = k <= nk - 1 && i <= ni - 1;
    r.n = in ? (int)pos(L, i, j, k) : 0;
    r.o = in ? T.base[l] + i - 1 + ni * (j - 1 + nj * (k - 1)) : -1;
    r.act = in && L.act[r.n] != 0;
    if (l + 1 < T.nt) {
        const Dims &c = T.L[l + 1].d;
        r.up = T.base[l + 1] + ((i + 2) >> 1) - 1 + c.ni * (((j + 2) >> 1) - 1 + c.nj * (((k + 2) >> 1) - 1));
    }
    if (l > 0) {
        const Dims &f = T.L[l - 1].d;
        r.src = T.res + T.base[l - 1] + 2 * i - 3 + f.ni * (2 * j - 3 + f.nj * (2 * k - 3));
    }
    r.ad = L.ad[r.n];
    r.li = L.ali[r.n];
    r.ui = L.aui[r.n];
    r.lj = L.alj[r.n];
    r.uj = L.auj[r.n];
    r.lk = L.alk[r.n];
    r.uk = L.auk[r.n];
    r.b = l == 0 ? L.b[r.n] : (V)0;
}

template <typename V>
__device__ __forceinline__ V tail_off(const TailRow<V> &r, const V *x, int ni, int nij)
{
    const int o = r.o;
    return r.li * x[o - 1] + r.ui * x[o + 1] + r.lj * x[o - ni] + r.uj * x[o + ni] + r.lk * x[o - nij]
         + r.uk * x[o + nij];
}

template <typename V, int N>
__device__ __forceinline__ void tail_sweep(const TailRow<V> (&r)[N], V *x, int ni, int nij)
{
#pragma unroll
    for (int s = 0; s < N; s++)
        if (r[s].act) x[r[s].o] = (r[s].b - tail_off(r[s], x, ni, nij)) / r[s].ad;
}

// Down from a level with N rows of each colour a thread to one with M.
template <typename V, int N, int M>
__device__ __forceinline__ void tail_down(const MgTail<V> &T, int l, const TailRow<V> (&ev)[N], const TailRow<V> (&od)[N],
                                          TailRow<V> (&cev)[M], TailRow<V> (&cod)[M], V *x)
{
    const int ni = T.L[l].d.ni, nij = ni * T.L[l].d.nj;
    tail_sweep(od, x, ni, nij);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < N; s++)
        if (ev[s].act) x[T.res + ev[s].o] = ev[s].b - ev[s].ad * x[ev[s].o] - tail_off(ev[s], x, ni, nij);
    __syncthreads();
    // the block's even cells in the order of k_mg_restrict
    auto sum = [&](const TailRow<V> &r) {
        const V *q = x + r.src;
        return q[0] + q[1 + ni] + q[1 + nij] + q[ni + nij];
    };
#pragma unroll
    for (int s = 0; s < M; s++) {
        if (cev[s].act) {
            cev[s].b = sum(cev[s]);
            x[cev[s].o] = cev[s].b / cev[s].ad;   // the even half from x = 0
        }
        if (cod[s].act) cod[s].b = sum(cod[s]);
    }
    __syncthreads();
}

// MG_COARSE sweeps of the coarsest level (the even half of the first came with
// b).  A level whose colours fit the first wave is swept by it alone.
template <typename V, int N>
__device__ __forceinline__ void tail_coarsest(const MgTail<V> &T, int l, const TailRow<V> (&ev)[N],
                                              const TailRow<V> (&od)[N], V *x)
{
    const Dims &d = T.L[l].d;
    const int ni = d.ni, nij = d.ni * d.nj;
    if (tail_half(ni) * (d.nj - 2) * (d.nk - 2) <= 64) {
        if (threadIdx.x < 64) {
            for (int s = 0; s < MG_COARSE; s++) {
                if (s) tail_sweep(ev, x, ni, nij);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
                tail_sweep(od, x, ni, nij);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            }
        }
        __syncthreads();
        return;
    }
    for (int s = 0; s < MG_COARSE; s++) {
        if (s) {
            tail_sweep(ev, x, ni, nij);
            __syncthreads();
        }
        tail_sweep(od, x, ni, nij);
        __syncthreads();
    }
}

template <typename V, int N>
__device__ __forceinline__ void tail_up(const MgTail<V> &T, int l, const TailRow<V> (&ev)[N], const TailRow<V> (&od)[N],
                                        V *x)
{
    const int ni = T.L[l].d.ni, nij = ni * T.L[l].d.nj;
#pragma unroll
    for (int s = 0; s < N; s++)
        if (od[s].act) x[od[s].o] = x[od[s].o] + (V)MG_SCALE * x[od[s].up];
    __syncthreads();
    tail_sweep(ev, x, ni, nij);
    __syncthreads();
    tail_sweep(od, x, ni, nij);
    __syncthreads();
}

template <typename V, int A>
__global__ void __launch_bounds__(TAIL_THREADS) k_mg_tail(MgTail<V> T)
{
    __shared__ V x[TAIL_LDS];
    TailRow<V> e0[A], o0[A], e1[2], o1[2], e2[1], o2[1], e3[1], o3[1];
    const int t = threadIdx.x;
#pragma unroll
    for (int s = 0; s < A; s++) {
        tail_load(T, 0, 0, t + s * TAIL_THREADS, e0[s]);
        tail_load(T, 0, 1, t + s * TAIL_THREADS, o0[s]);
    }
    if (T.nt > 1) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            tail_load(T, 1, 0, t + s * TAIL_THREADS, e1[s]);
            tail_load(T, 1, 1, t + s * TAIL_THREADS, o1[s]);
        }
    }
    if (T.nt > 2) {
        tail_load(T, 2, 0, t, e2[0]);
        tail_load(T, 2, 1, t, o2[0]);
    }
    if (T.nt > 3) {
        tail_load(T, 3, 0, t, e3[0]);
        tail_load(T, 3, 1, t, o3[0]);
    }
    for (int p = t; p < 2 * T.res; p += TAIL_THREADS) x[p] = (V)0;
    __syncthreads();
    // from x = 0 the even half of the first sweep is x = b/AD
#pragma unroll
    for (int s = 0; s < A; s++)
        if (e0[s].act) x[e0[s].o] = e0[s].b / e0[s].ad;
    __syncthreads();
    if (T.nt > 1) {
        tail_down(T, 0, e0, o0, e1, o1, x);
        if (T.nt > 2) {
            tail_down(T, 1, e1, o1, e2, o2, x);
            if (T.nt > 3) {
                tail_down(T, 2, e2, o2, e3, o3, x);
                tail_coarsest(T, 3, e3, o3, x);
                tail_up(T, 2, e2, o2, x);
            } else {
                tail_coarsest(T, 2, e2, o2, x);
            }
            tail_up(T, 1, e1, o1, x);
        } else {
            tail_coarsest(T, 1, e1, o1, x);
        }
        tail_up(T, 0, e0, o0, x);
    } else {
        tail_coarsest(T, 0, e0, o0, x);
    }
#pragma unroll
    for (int s = 0; s < A; s++) {
        if (e0[s].o >= 0) T.L[0].x[e0[s].n] = x[e0[s].o];
        if (o0[s].o >= 0) T.L[0].x[o0[s].n] = x[o0[s].o];
    }
}

// The tail from level t0 on: the rows a thread of k_mg_tail holds of each colour
// on level t0, or 0 where the levels do not fit it.
template <typename V>
int tail_rows(const MgLevelT<V> *mg, int nl, int t0, MgTail<V> *T)
{
    if (nl - t0 > TAIL_LEVELS) return 0;
    long long lds = 0, need[TAIL_LEVELS] = {0, 0, 0, 0};
    for (int l = t0; l < nl; l++) {
        const Dims &d = mg[l].d;
        const int h = tail_half(d.ni), q = l - t0;
        need[q] = ((long long)h * (d.nj - 2) * (d.nk - 2) + TAIL_THREADS - 1) / TAIL_THREADS;
        T->L[q] = mg[l];
        T->inv_h[q] = 1.0f / (float)h;
        T->inv_j[q] = 1.0f / (float)(d.nj - 2);
        T->base[q] = (int)std::min(lds, (long long)TAIL_LDS);
        lds += d.nc;
    }
    T->res = (int)std::min(lds, (long long)TAIL_LDS);
    T->nt = nl - t0;
    if (2 * lds > TAIL_LDS || need[0] > 6 || need[1] > 2 || need[2] > 1 || need[3] > 1) return 0;
    return need[0] <= 2 ? 2 : need[0] <= 4 ? 4 : 6;
}

dim3 lvl_grid(const Dims &d, int k0, int k1)
{
    return dim3((unsigned)((d.ni - 2 + 63) / 64), (unsigned)((d.nj - 2 + 3) / 4), (unsigned)(k1 - k0 + 1));
}

// threads over one colour's half lines: positions 0 .. NUMI/2
dim3 half_grid(const Dims &d, int k0, int k1)
{
    const int half = d.ni / 2 + 1;
    return dim3((unsigned)((half + 63) / 64), (unsigned)((d.nj - 2 + 3) / 4), (unsigned)(k1 - k0 + 1));
}

// half-sweep of a colour on K planes k0..k1
template <typename V>
int smooth(cad_ctx *c, const MgLevelT<V> &L, int k0, int k1, int color)
{
    const dim3 b(64, 4, 1), g = half_grid(L.d, k0, k1);
    if (L.d.nc > MG_SKIP_CELLS)
        hipLaunchKernelGGL((k_mg_smooth<V, true>), g, b, 0, c->stream, L, color, k0);
    else
        hipLaunchKernelGGL((k_mg_smooth<V, false>), g, b, 0, c->stream, L, color, k0);
    CAD_CHECK(hipGetLastError());
    return CAD_OK;
}

template <typename V>
void free_levels(MgLevelT<V> *mg, int &n)
{
    for (int l = 0; l < n; l++) {
        MgLevelT<V> &L = mg[l];
        void *p[] = {L.ad, L.ali, L.alj, L.alk, L.aui, L.auj, L.auk, L.x, L.b, L.act};
        for (void *q : p)
            if (q) (void)hipFree(q);
        L = MgLevelT<V>();
    }
    n = 0;
}

// The levels of a grid: colour-split arrays of ld x NUMJ x NUMK per level, each level counted
// before its arrays so that a failed allocation frees what was allocated.
template <typename V>
int alloc_levels(const Dims &d0, MgLevelT<V> *mg, int &nl)
{
    if (nl > 0) return CAD_OK;
    Dims d = d0;
    int n = 0;
    for (;;) {
        if (n == CAD_MG_MAX) break;
        MgLevelT<V> &L = mg[n];
        L = MgLevelT<V>();
        L.d = d;
        L.ld = (d.ni + 7) / 8 * 8;   // half lines of whole 16-byte vectors
        nl = n + 1;
        const size_t ns = (size_t)L.ld * d.nj * d.nk;
        V **f[] = {&L.ad, &L.ali, &L.alj, &L.alk, &L.aui, &L.auj, &L.auk, &L.x, &L.b};
        for (V **p : f) {
            CAD_CHECK(hipMalloc((void **)p, ns * sizeof(V)));
            CAD_CHECK(hipMemset(*p, 0, ns * sizeof(V)));
        }
        CAD_CHECK(hipMalloc((void **)&L.act, ns));
        CAD_CHECK(hipMemset(L.act, 0, ns));
        n++;
        // coarsen while every interior extent is at least 4
        const int ei = d.ni - 2, ej = d.nj - 2, ek = d.nk - 2;
        if (ei < 4 || ej < 4 || ek < 4) break;
        Dims cd;
        cd.ni = (ei + 1) / 2 + 2;
        cd.nj = (ej + 1) / 2 + 2;
        cd.nk = (ek + 1) / 2 + 2;
        cd.nij = (long long)cd.ni * cd.nj;
        cd.nc = cd.nij * cd.nk;
        cd.numb = 0;
        d = cd;
    }
    const MgLevelT<V> &top = mg[nl - 1];
    if ((long long)(top.d.ni - 2) * (top.d.nj - 2) * (top.d.nk - 2) > (1 << 20)) {
        cad_set_error("multigrid: coarsest level %d x %d x %d too large", top.d.ni - 2, top.d.nj - 2,
                      top.d.nk - 2);
        return CAD_ERR_ARG;
    }
    CAD_CHECK(hipDeviceSynchronize());
    return CAD_OK;
}

// The levels' rows from the context's matrix on level 0's K planes lo..hi
// and, level by level, the coarse planes whose rows read those (coarse plane
// K reads fine planes 2K-3 .. 2K); every other row keeps what it holds.
template <typename V>
int setup_levels(cad_ctx *c, MgLevelT<V> *mg, int nl, int lo, int hi)
{
    const Dims &d = c->d;
    const long long n0 = (long long)(lo - 1) * d.nij, n1 = (long long)hi * d.nij;
    hipLaunchKernelGGL(k_mg_fine<V>, dim3((unsigned)((n1 - n0 + 255) / 256)), dim3(256), 0, c->stream, d,
                       c->ad, c->ali, c->alj, c->alk, c->aui, c->auj, c->auk, c->f.indc, mg[0], n0, n1);
    for (int l = 1; l < nl; l++) {
        const Dims &cd = mg[l].d;
        lo = std::max(2, (lo + 1) / 2);
        hi = std::min(cd.nk - 1, (hi + 3) / 2);
        if (lo > hi) break;
        hipLaunchKernelGGL(k_mg_coarsen<V>, lvl_grid(cd, lo, hi), dim3(64, 4, 1), 0, c->stream, mg[l - 1],
                           mg[l], lo);
    }
    CAD_CHECK(hipGetLastError());
    return CAD_OK;
}

// One V-cycle's passes; level 0 holds b and the first half-sweep's x.  k0..k1
// limits level 0 to the K planes that hold active cells.
template <typename V>
int passes(cad_ctx *c, const MgLevelT<V> *mg, int nl, int k0, int k1)
{
    const dim3 b(64, 4, 1);
    // the first level from which on one workgroup holds the rest (nl: none, the
    // coarsest is too large for it)
    MgTail<V> tl;
    int t0 = 0, rows = 0;
    while (t0 < nl && !(rows = tail_rows(mg, nl, t0, &tl))) t0++;
    // Each level's passes run on the K planes that can hold its active rows:
    // level 0's k0..k1, and on a coarser level the planes of their parents
    // (fine plane k lies in coarse plane (k + 2) / 2).  Rows outside are
    // inactive, and no active row couples to them (coarsening sums only the
    // couplings between active rows), so what they hold is never used.
    int lo[CAD_MG_MAX], hi[CAD_MG_MAX];
    lo[0] = k0;
    hi[0] = k1;
    for (int l = 1; l < nl; l++) {
        lo[l] = std::max(2, (lo[l - 1] + 2) / 2);
        hi[l] = std::min(mg[l].d.nk - 1, (hi[l - 1] + 2) / 2);
    }
    // down: the odd half-sweep (the even half came with b), the coarse b
    for (int l = 0; l < std::min(t0, nl - 1); l++) {
        const MgLevelT<V> &F = mg[l], &C = mg[l + 1];
        RET_IF(smooth(c, F, lo[l], hi[l], 1));
        const dim3 g = lvl_grid(C.d, lo[l + 1], hi[l + 1]);
        if (F.d.nc > MG_SKIP_CELLS)
            hipLaunchKernelGGL((k_mg_restrict<V, true>), g, b, 0, c->stream, F, C, lo[l + 1]);
        else
            hipLaunchKernelGGL((k_mg_restrict<V, false>), g, b, 0, c->stream, F, C, lo[l + 1]);
        CAD_CHECK(hipGetLastError());
    }
    if (t0 == nl) {
        const MgLevelT<V> &B = mg[nl - 1];
        for (int h = 1; h < 2 * MG_COARSE; h++) RET_IF(smooth(c, B, lo[nl - 1], hi[nl - 1], h & 1));
    } else {
        const dim3 tb(TAIL_THREADS);
        if (rows == 2)
            hipLaunchKernelGGL((k_mg_tail<V, 2>), dim3(1), tb, 0, c->stream, tl);
        else if (rows == 4)
            hipLaunchKernelGGL((k_mg_tail<V, 4>), dim3(1), tb, 0, c->stream, tl);
        else
            hipLaunchKernelGGL((k_mg_tail<V, 6>), dim3(1), tb, 0, c->stream, tl);
        CAD_CHECK(hipGetLastError());
    }
    // up: correct, then one sweep (the correction rides on the even half)
    for (int l = std::min(t0, nl - 1) - 1; l >= 0; l--) {
        const MgLevelT<V> &F = mg[l], &C = mg[l + 1];
        const dim3 g = half_grid(F.d, lo[l], hi[l]);
        if (F.d.nc > MG_SKIP_CELLS)
            hipLaunchKernelGGL((k_mg_correct_even<V, true>), g, b, 0, c->stream, F, C, lo[l]);
        else
            hipLaunchKernelGGL((k_mg_correct_even<V, false>), g, b, 0, c->stream, F, C, lo[l]);
        CAD_CHECK(hipGetLastError());
        RET_IF(smooth(c, F, lo[l], hi[l], 1));
    }
    return CAD_OK;
}

// x = M^-1 y: one V-cycle from x = 0.  With r set, also r = y - A x on level 0's matrix
// and the partials of its sum of squares (k_mg_out_resid, REDUCE_BLOCKS blocks).
template <typename V, typename T>
int vcycle(cad_ctx *c, const MgLevelT<V> *mg, int nl, const T *y, T *x, int k0, int k1, T *r = nullptr,
           double *part = nullptr, int stride = 0)
{
    const dim3 b(64, 4, 1);
    hipLaunchKernelGGL((k_mg_in<V, T>), lvl_grid(mg[0].d, k0, k1), b, 0, c->stream, mg[0], y, k0);
    CAD_CHECK(hipGetLastError());
    RET_IF(passes(c, mg, nl, k0, k1));
    if (r)
        hipLaunchKernelGGL((k_mg_out_resid<V, T>), dim3(REDUCE_BLOCKS), dim3(256), 0, c->stream, mg[0], x, r, k0, k1,
                           part, stride);
    else
        hipLaunchKernelGGL((k_mg_out<V, T>), lvl_grid(mg[0].d, k0, k1), b, 0, c->stream, mg[0], x, k0);
    CAD_CHECK(hipGetLastError());
    return CAD_OK;
}

// Algorithmic bytes of one V-cycle with vs-byte values: per cell of a level
// below the coarsest, three half-sweeps (each cell once in one of them: 7
// coefficients, b, x written and the activity byte; x of the other colour's
// neighbours read once: 10 values + 1 byte per cell and colour pair), the
// residual-restriction of the even cells (7 coefficients, b, x, activity,
// and a share of the coarse b and x) and the coarse x that the corrected
// even half-sweep reads; on the coarsest level MG_COARSE full sweeps.  Level 0
// counts with the planes from the first to the last active cell, also where its
// passes run on more.
double vcycle_bytes(const cad_ctx *c, const Dims *dims, int nl, int vs)
{
    const double half = (10.0 * vs + 1.0) / 2.0;
    const double restr = (9.0 * vs + 1.0) / 2.0 + 2.0 * vs / 8.0;
    const double prol = vs / 8.0;
    double by = 0.0;
    for (int l = 0; l < nl; l++) {
        const Dims &d = dims[l];
        const int planes = l == 0 ? c->mg_planes : d.nk - 2;
        const double cells = (double)(d.ni - 2) * (double)(d.nj - 2) * (double)planes;
        by += l == nl - 1 ? 2.0 * half * MG_COARSE * cells : (3.0 * half + restr + prol) * cells;
    }
    return by;
}

}  // namespace

void cad_mg_free(cad_ctx *c)
{
    c->mg_set_k0 = c->mg_set_k1 = 0;
    free_levels(c->mg, c->mg_n);
    free_levels(c->mg64, c->mg64_n);
}

int cad_mg_alloc(cad_ctx *c) { return alloc_levels(c->d, c->mg, c->mg_n); }

// the hierarchy of the context's current matrix.  Outside the K planes that
// hold active cells every row is inactive (INDC = -1 there), as a freshly
// allocated level's are, so the rows are rebuilt only on the planes of this
// solve and of the last build (where rows may have been active); the rows
// are those of a build over every plane.
int cad_mg_setup(cad_ctx *c)
{
    RET_IF(cad_mg_alloc(c));
    int lo = c->mg_k0, hi = c->mg_k1;
    if (c->mg_set_k0 > 0) {
        lo = std::min(lo, c->mg_set_k0);
        hi = std::max(hi, c->mg_set_k1);
    }
    c->mg_set_k0 = c->mg_k0;
    c->mg_set_k1 = c->mg_k1;
    return setup_levels(c, c->mg, c->mg_n, lo, hi);
}

int cad_mg_apply(cad_ctx *c, const double *y, double *x, int k0, int k1)
{
    return vcycle(c, c->mg, c->mg_n, y, x, k0, k1);
}

int cad_mg_apply_resid(cad_ctx *c, const double *y, double *x, double *r, double *part, int stride, int k0, int k1)
{
    return vcycle(c, c->mg, c->mg_n, y, x, k0, k1, r, part, stride);
}

int cad_mg_cycle(cad_ctx *c, float *b, float *x)
{
    MgLevel mg[CAD_MG_MAX];
    std::copy(c->mg, c->mg + c->mg_n, mg);
    mg[0].b = b;
    mg[0].x = x;
    RET_IF(cad_kt_begin(c, CAD_KT_VCYCLE));
    RET_IF(passes(c, mg, c->mg_n, c->mg_k0, c->mg_k1));
    double by = 0.0;
    if (c->kt && c->kt->on) {
        Dims dims[CAD_MG_MAX];
        for (int l = 0; l < c->mg_n; l++) dims[l] = c->mg[l].d;
        by = vcycle_bytes(c, dims, c->mg_n, 4);
    }
    return cad_kt_end(c, CAD_KT_VCYCLE, by);
}

// One V-cycle on the hierarchy and K range of the last mixed or learned
// solve, timed with HIP events on the library's stream (right-hand side BB),
// with its algorithmic bytes (vcycle_bytes); fp64 != 0: the same V-cycle with
// every level in FP64 (a hierarchy of its own, built from the same matrix),
// for comparison.
int cad_mg_time(cad_ctx *c, int reps, int fp64, float *ms_avg, double *bytes)
{
    if (c->mg_n <= 0 || c->mg_span == 0) {
        cad_set_error("cad_time_precond: no mixed solve has run on this context");
        return CAD_ERR_STATE;
    }
    if (reps < 1) reps = 1;
    if (fp64) {
        RET_IF(alloc_levels(c->d, c->mg64, c->mg64_n));
        RET_IF(setup_levels(c, c->mg64, c->mg64_n, 1, c->d.nk));
    }
    const dim3 g = lvl_grid(c->d, c->mg_k0, c->mg_k1), tb(64, 4, 1);
    if (fp64)
        hipLaunchKernelGGL((k_mg_in<double, double>), g, tb, 0, c->stream, c->mg64[0], c->bb, c->mg_k0);
    else
        hipLaunchKernelGGL((k_mg_in<float, double>), g, tb, 0, c->stream, c->mg[0], c->bb, c->mg_k0);
    CAD_CHECK(hipGetLastError());
    hipEvent_t a, b;
    CAD_CHECK(hipEventCreate(&a));
    CAD_CHECK(hipEventCreate(&b));
    CAD_CHECK(hipEventRecord(a, c->stream));
    for (int r = 0; r < reps; r++) {
        if (fp64)
            RET_IF(passes(c, c->mg64, c->mg64_n, c->mg_k0, c->mg_k1));
        else
            RET_IF(passes(c, c->mg, c->mg_n, c->mg_k0, c->mg_k1));
    }
    CAD_CHECK(hipEventRecord(b, c->stream));
    CAD_CHECK(hipEventSynchronize(b));
    float ms = 0.0f;
    CAD_CHECK(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    *ms_avg = ms / reps;
    Dims dims[CAD_MG_MAX];
    const int nl = fp64 ? c->mg64_n : c->mg_n;
    for (int l = 0; l < nl; l++) dims[l] = fp64 ? c->mg64[l].d : c->mg[l].d;
    *bytes = vcycle_bytes(c, dims, nl, fp64 ? 8 : 4);
    return CAD_OK;
}
