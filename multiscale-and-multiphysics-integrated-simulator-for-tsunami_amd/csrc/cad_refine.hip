// cad_refine.hip -- the mixed form's pressure solve: FP64 iterative
// refinement around an FP32 Krylov solve.
//
// The system is VF_VPCOEF's (the FP64 matrix AD..AUK and BB that VF_M1BCGS
// solves, vf_m1bcgs.f:101-262).  Outer iteration, in FP64:
//   r = BB - A x,  stop when ||r|| <= CGEPSR ||BB|| + CGEPSA  (the true residual)
//   solve A d = r / ||r|| approximately in FP32
//   x = x + ||r|| d
// Inner solve, in FP32: BiCGSTAB right-preconditioned by one multigrid V-cycle
// (cad_mg.hip).  Every vector is FP32, the dot products are accumulated in
// FP64.  The vectors lie in level 0's colour-split layout, so they are the
// V-cycle's right-hand side and result themselves, and the matvec reads level
// 0's rows (the matrix rounded to FP32).  The kernel that forms a right-hand
// side b also writes the first (even) half-sweep x = b/AD.
//
// The scalars stay on the device: a kernel that needs alpha or omega forms it
// from the partials of the dot product before it, and one block at an
// iteration's end forms rho, tests the residual and writes {(r, r) or -1 to
// stop, a tag} to host memory.  An iteration's launches take no argument that changes from one
// iteration to the next, so they are captured once into a graph: a launch of its own
// costs the host 2.5-4 us, more than most of these kernels run on
// grids of 10^5 cells, and a graph's kernel 2 us with the host free.  The host
// launches an iteration before it has read the last one's record where the
// residuals' trend says that it will be needed (never a second one, so two records in
// turn hold what it has not read); one launched beyond the stop changes nothing.
// With all this 20 steps of drops on 97x61x45 cells take 52 ms instead of 70, ten of a tank
// with buildings on 512x256x128 155 instead of 176.
//
// The inner solve stops at a relative residual eta = max(1e-6, 0.1
// tol / ||r||): about what FP32 can resolve, and on the last outer step a
// tenth of what is left to the stop test, so that the answer lands below it
// with room to spare.  A solve takes two or three outer steps.  An outer step
// that does not halve the true residual, or more than the iteration cap
// (cad_krylov_cap), hands the solve to VF_M1BCGS from the current x with the
// same true-residual stop.
#include "cad_common.h"

#include <algorithm>
#include <cmath>
#include <new>

#define RET_IF(x)              \
    do {                       \
        int rc_ = (x);         \
        if (rc_) return rc_;   \
    } while (0)

namespace {

constexpr int VB = 2048;
constexpr int KV = 6;                    // vectors beside level 0's b and x
constexpr double TAG0 = 1099511627776.0; // 2^40: beyond the plain solve's tags
// slots of ksc
enum { S_RHO1 = 0, S_RHO, S_ALPHA, S_OM, S_FLAG, S_DONE, S_ETA2, S_TAG, S_REC };

// The FP32 vectors, in level 0's layout: r (also s), the V-cycles' results ph
// and sh.
struct Vecs {
    float *r, *r0, *p, *v, *t, *ph, *sh, *d;
};

__device__ __forceinline__ double wsum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// block sums of up to two products into partial[q * REDUCE_BLOCKS + block]
template <int N>
__device__ __forceinline__ void block_sums(const double (&a)[2], double *partial)
{
    __shared__ double sh[2][REDUCE_THREADS / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < N; q++) {
        const double s = wsum(a[q]);
        if (lane == 0) sh[q][w] = s;
    }
    __syncthreads();
    if (threadIdx.x < N) {
        double s = 0.0;
        for (int i = 0; i < REDUCE_THREADS / 64; i++) s += sh[threadIdx.x][i];
        partial[threadIdx.x * REDUCE_BLOCKS + blockIdx.x] = s;
    }
}

// the N products' sums over nb blocks' partials, the same in every block
template <int N>
__device__ __forceinline__ void final_sums(const double *__restrict__ partial, int nb, double (&s)[N])
{
    __shared__ double sh[N][REDUCE_THREADS / 64], out[N];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double a[N];
#pragma unroll
    for (int q = 0; q < N; q++) {
        a[q] = 0.0;
        for (int b = threadIdx.x; b < nb; b += REDUCE_THREADS) a[q] += partial[q * REDUCE_BLOCKS + b];
    }
#pragma unroll
    for (int q = 0; q < N; q++) {
        const double v = wsum(a[q]);
        if (lane == 0) sh[q][w] = v;
    }
    __syncthreads();
    if (threadIdx.x < N) {
        double v = 0.0;
        for (int i = 0; i < REDUCE_THREADS / 64; i++) v += sh[threadIdx.x][i];
        out[threadIdx.x] = v;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; q++) s[q] = out[q];
}

// the cells n0 <= n < n1 of the grid's order with their positions m in level 0
#define CELL_LOOP(L, n, m, n0, n1)                                                            \
    for (unsigned q_ = blockIdx.x * blockDim.x + threadIdx.x, nq_ = (unsigned)((n1) - (n0)); q_ < nq_; \
         q_ += gridDim.x * blockDim.x)                                                        \
        if (const long long n = (n0) + (long long)q_; true)                                   \
            if (const int m = split_pos(L, n); true)

__device__ __forceinline__ int split_pos(const MgLevel &L, long long n)
{
    const unsigned u = (unsigned)n, ni = (unsigned)L.d.ni, l = u / ni, i = u - l * ni;
    const unsigned k = l / (unsigned)L.d.nj, j = l - k * (unsigned)L.d.nj;
    // 1-based I+J+K = i+j+k+3
    return (int)(l * (unsigned)L.ld + ((i + j + k + 1) & 1) * (unsigned)(L.ld >> 1) + (i >> 1));
}

// r = r0 = (float)(r64 / rn), p = v = d = 0 (0 on inactive rows) over level
// 0's planes, and the partials of (r0, r)
__global__ void __launch_bounds__(REDUCE_THREADS) k_r_init(MgLevel L, long long n0, long long n1,
                                                           const double *__restrict__ r64, double inv, Vecs w,
                                                           double *partial)
{
    double a[2] = {0.0, 0.0};
    CELL_LOOP(L, n, m, n0, n1) {
        const float b = L.act[m] ? (float)(r64[n] * inv) : 0.0f;
        w.r[m] = b;
        w.r0[m] = b;
        w.p[m] = 0.0f;
        w.v[m] = 0.0f;
        w.d[m] = 0.0f;
        a[0] += (double)b * (double)b;
    }
    block_sums<1>(a, partial);
}

__global__ void __launch_bounds__(REDUCE_THREADS) k_r_start(const double *__restrict__ partial, int nb, double *sc,
                                                            double eta2, double tag)
{
    double s[1];
    final_sums<1>(partial, nb, s);
    if (threadIdx.x != 0) return;
    sc[S_RHO1] = s[0];
    sc[S_RHO] = 1.0;
    sc[S_ALPHA] = 1.0;
    sc[S_OM] = 1.0;
    sc[S_FLAG] = std::isfinite(s[0]) && s[0] != 0.0 ? 0.0 : 1.0;
    sc[S_DONE] = 0.0;
    sc[S_ETA2] = eta2;
    sc[S_TAG] = tag;
}

struct alignas(4) Act4 {
    unsigned char v[4];
};

// Level 0's positions e four at a time, e0 <= e < e1 (a line's halves are
// multiples of four).
#define VEC_LOOP(e, e0, e1)                                                                   \
    for (int e = (e0) + (int)(blockIdx.x * blockDim.x + threadIdx.x); e < (e1); e += (int)(gridDim.x * blockDim.x))

// the first (even) half-sweep of the V-cycle for b: x = b/AD on the even half
__device__ __forceinline__ void even_start(const MgLevel &L, int e, const Act4 &a, const float (&b)[4], float *x)
{
    const int h4 = L.ld >> 3;
    if ((e / h4) & 1) return;
    const float4 ad = reinterpret_cast<const float4 *>(L.ad)[e];
    const float q[4] = {b[0] / ad.x, b[1] / ad.y, b[2] / ad.z, b[3] / ad.w};
    reinterpret_cast<float4 *>(x)[e] =
        make_float4(a.v[0] ? q[0] : 0.0f, a.v[1] ? q[1] : 0.0f, a.v[2] ? q[2] : 0.0f, a.v[3] ? q[3] : 0.0f);
}

// p = r + beta (p - om v),  beta = (rho1 / rho) (alpha / om); starts ph
__global__ void __launch_bounds__(256) k_r_p(MgLevel L, int e0, int e1, const double *__restrict__ sc, Vecs w)
{
    if (sc[S_DONE] != 0.0) return;
    const float beta = (float)((sc[S_RHO1] / sc[S_RHO]) * (sc[S_ALPHA] / sc[S_OM]));
    const float om = (float)sc[S_OM];
    VEC_LOOP(e, e0, e1) {
        const Act4 a = reinterpret_cast<const Act4 *>(L.act)[e];
        const float4 r = reinterpret_cast<const float4 *>(w.r)[e], p = reinterpret_cast<const float4 *>(w.p)[e];
        const float4 v = reinterpret_cast<const float4 *>(w.v)[e];
        const float b[4] = {a.v[0] ? r.x + beta * (p.x - om * v.x) : 0.0f, a.v[1] ? r.y + beta * (p.y - om * v.y) : 0.0f,
                            a.v[2] ? r.z + beta * (p.z - om * v.z) : 0.0f, a.v[3] ? r.w + beta * (p.w - om * v.w) : 0.0f};
        reinterpret_cast<float4 *>(w.p)[e] = make_float4(b[0], b[1], b[2], b[3]);
        even_start(L, e, a, b, w.ph);
    }
}

// s = r - alpha v (in place of r),  alpha = rho1 / (r0, v); starts sh
__global__ void __launch_bounds__(REDUCE_THREADS) k_r_s(MgLevel L, int e0, int e1, double *__restrict__ sc,
                                                        const double *__restrict__ partial, int nb, Vecs w)
{
    if (sc[S_DONE] != 0.0) return;
    double s[1];
    final_sums<1>(partial, nb, s);
    const bool ok = std::isfinite(s[0]) && s[0] != 0.0;
    const double al = ok ? sc[S_RHO1] / s[0] : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc[S_ALPHA] = al;
        if (!ok) sc[S_FLAG] = 1.0;
    }
    const float alpha = (float)al;
    VEC_LOOP(e, e0, e1) {
        const Act4 a = reinterpret_cast<const Act4 *>(L.act)[e];
        const float4 r = reinterpret_cast<const float4 *>(w.r)[e], v = reinterpret_cast<const float4 *>(w.v)[e];
        const float b[4] = {a.v[0] ? r.x - alpha * v.x : 0.0f, a.v[1] ? r.y - alpha * v.y : 0.0f,
                            a.v[2] ? r.z - alpha * v.z : 0.0f, a.v[3] ? r.w - alpha * v.w : 0.0f};
        reinterpret_cast<float4 *>(w.r)[e] = make_float4(b[0], b[1], b[2], b[3]);
        even_start(L, e, a, b, w.sh);
    }
}

// Tiles of 64 positions of one colour by four lines over the K planes k0..k1,
// an XCD's next to each other (k_r_mv 58.6 -> 50.7 us on 512x256x45 cells, 49 of
// them at the rate of a large copy).
struct Tiles {
    int k0, qt, jt, n;
};

// y = A x (FP32 rows of level 0) with the partials of (w, y) and, N = 2, (y, y)
template <int N>
__global__ void __launch_bounds__(REDUCE_THREADS) k_r_mv(MgLevel L, Tiles T, const double *__restrict__ sc,
                                                         const float *__restrict__ x, const float *__restrict__ w,
                                                         float *__restrict__ y, double *partial)
{
    if (sc[S_DONE] != 0.0) return;
    const int lj = L.ld, lk = L.ld * L.d.nj, half = L.ld >> 1;
    double a[2] = {0.0, 0.0};
    const int b0 = gridDim.x % 8 == 0 ? xcd_block(gridDim.x) : (int)blockIdx.x;
    for (int t = b0; t < T.n; t += gridDim.x) {
        const int qt = t % T.qt, r1 = t / T.qt, color = r1 & 1, r2 = r1 >> 1, jt = r2 % T.jt, k = T.k0 + r2 / T.jt;
        const int q = qt * 64 + (int)(threadIdx.x & 63), j = jt * 4 + (int)(threadIdx.x >> 6) + 2;
        const int i = 2 * q + 1 + ((color + 1 + j + k) & 1);
        if (j > L.d.nj - 1 || i < 2 || i > L.d.ni - 1) continue;
        const int line = lj * (j - 1) + lk * (k - 1), n = line + color * half + q;
        // the neighbours are in the other half of their lines, at q, those in I at q-1+p and q+p
        const int o = line + (1 - color) * half + q, p = i - 2 * q - 1;
        if (!L.act[n]) continue;
        const float s = L.ad[n] * x[n] + L.ali[n] * x[o - 1 + p] + L.aui[n] * x[o + p] + L.alj[n] * x[o - lj]
                      + L.auj[n] * x[o + lj] + L.alk[n] * x[o - lk] + L.auk[n] * x[o + lk];
        y[n] = s;
        a[0] += (double)w[n] * (double)s;
        if (N == 2) a[1] += (double)s * (double)s;
    }
    block_sums<N>(a, partial);
}

// d += alpha ph + om sh; r = s - om t, om = (s, t) / (t, t); partials of (r, r)
// and (r0, r) behind those it reads
__global__ void __launch_bounds__(REDUCE_THREADS) k_r_xr(MgLevel L, int e0, int e1, double *__restrict__ sc, int nb,
                                                         Vecs w, double *__restrict__ partial)
{
    if (sc[S_DONE] != 0.0) return;
    double s[2];
    final_sums<2>(partial, nb, s);
    const bool ok = std::isfinite(s[1]) && s[1] > 0.0;
    const double omd = ok ? s[0] / s[1] : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc[S_OM] = omd;
        if (!ok) sc[S_FLAG] = 1.0;
    }
    const float alpha = (float)sc[S_ALPHA], om = (float)omd;
    double a[2] = {0.0, 0.0};
    VEC_LOOP(e, e0, e1) {
        const Act4 act = reinterpret_cast<const Act4 *>(L.act)[e];
        float ph[4], sh[4], sv[4], t[4], r0[4], d[4];
        auto load = [e](const float *f, float (&o)[4]) {
            const float4 q = reinterpret_cast<const float4 *>(f)[e];
            o[0] = q.x, o[1] = q.y, o[2] = q.z, o[3] = q.w;
        };
        load(w.ph, ph), load(w.sh, sh), load(w.r, sv), load(w.t, t), load(w.r0, r0), load(w.d, d);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            d[i] = act.v[i] ? d[i] + (alpha * ph[i] + om * sh[i]) : 0.0f;
            sv[i] = act.v[i] ? sv[i] - om * t[i] : 0.0f;
            a[0] += (double)sv[i] * (double)sv[i];
            a[1] += (double)r0[i] * (double)sv[i];
        }
        reinterpret_cast<float4 *>(w.d)[e] = make_float4(d[0], d[1], d[2], d[3]);
        reinterpret_cast<float4 *>(w.r)[e] = make_float4(sv[0], sv[1], sv[2], sv[3]);
    }
    block_sums<2>(a, partial + 2 * REDUCE_BLOCKS);
}

// rho for the next iteration and the stop test on (r, r), with the host's record
__global__ void __launch_bounds__(REDUCE_THREADS) k_r_end(const double *__restrict__ partial, int nb, double *sc,
                                                          double *rec)
{
    if (sc[S_DONE] != 0.0) return;
    double s[2];
    final_sums<2>(partial + 2 * REDUCE_BLOCKS, nb, s);
    if (threadIdx.x != 0) return;
    sc[S_RHO] = sc[S_RHO1];
    sc[S_RHO1] = s[1];
    const bool bad = sc[S_FLAG] != 0.0 || !(std::isfinite(s[1]) && s[1] != 0.0) || !(sc[S_OM] != 0.0);
    const bool stop = bad || !(s[0] > sc[S_ETA2]);
    const double v = stop ? -1.0 : s[0], tag = sc[S_TAG] + 1.0;
    sc[S_DONE] = stop ? 1.0 : 0.0;
    sc[S_TAG] = tag;
    sc[S_REC] = v;
    if (rec) {
        rec += 2 * ((long long)tag & 1);
        __hip_atomic_store(rec, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(rec + 1, tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// x += scale d (active rows), FP64
__global__ void __launch_bounds__(256) k_r_update(MgLevel L, long long n0, long long n1, double scale,
                                                  const float *__restrict__ d, double *__restrict__ x)
{
    CELL_LOOP(L, n, m, n0, n1) {
        if (L.act[m]) x[n] += scale * (double)d[m];
    }
}

// b = a on the active rows, FP64
__global__ void __launch_bounds__(256) k_r_copy(MgLevel L, long long n0, long long n1, const double *__restrict__ a,
                                                double *__restrict__ b)
{
    CELL_LOOP(L, n, m, n0, n1) {
        if (L.act[m]) b[n] = a[n];
    }
}

__global__ void k_r_fill32(long long n, float *a, float *b)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        a[i] = 0.0f;
        b[i] = 0.0f;
    }
}

__global__ void k_r_fill(long long n, double *a)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        a[i] = 0.0;
}

}  // namespace

// The vectors and the captured iteration of a context.
struct cad_mixed {
    float *mem;              // KV vectors
    hipGraphExec_t exec;     // one iteration on planes k0..k1 (null: none captured)
    int k0, k1;
    bool no_graph;           // a capture failed: launches of their own
    double tag;              // of the last record
};

void cad_mixed_free(cad_ctx *c)
{
    if (!c->mx) return;
    if (c->mx->exec) (void)hipGraphExecDestroy(c->mx->exec);
    if (c->mx->mem) (void)hipFree(c->mx->mem);
    delete c->mx;
    c->mx = nullptr;
}

namespace {

int mixed_alloc(cad_ctx *c)
{
    if (c->mx) return CAD_OK;
    const MgLevel &L = c->mg[0];
    cad_mixed *mx = new (std::nothrow) cad_mixed();
    if (!mx) {
        cad_set_error("mixed form: out of host memory");
        return CAD_ERR_ARG;
    }
    mx->tag = TAG0;
    const size_t bytes = (size_t)KV * L.ld * L.d.nj * L.d.nk * sizeof(float);
    if (hipMalloc((void **)&mx->mem, bytes) != hipSuccess || hipMemset(mx->mem, 0, bytes) != hipSuccess ||
        hipDeviceSynchronize() != hipSuccess) {
        cad_set_error("mixed form: %s", hipGetErrorString(hipGetLastError()));
        if (mx->mem) (void)hipFree(mx->mem);
        delete mx;
        return CAD_ERR_HIP;
    }
    c->mx = mx;
    return CAD_OK;
}

// The inner solve of a context: its vectors and launch shapes.
struct Inner {
    cad_ctx *c;
    Vecs w;
    Tiles tiles;
    int e0, e1;              // level 0's positions of the planes, four at a time
    int nb_mv, nb_vec;       // blocks of the matvec and of the vector kernels

    // one iteration's launches
    int iteration() const
    {
        hipStream_t st = c->stream;
        const MgLevel &L = c->mg[0];
        const dim3 tb(REDUCE_THREADS), vb(nb_vec), mb(nb_mv);
        double *sc = c->ksc, *part = c->red_partial;
        hipLaunchKernelGGL(k_r_p, vb, tb, 0, st, L, e0, e1, sc, w);
        RET_IF(cad_mg_cycle(c, w.p, w.ph));
        hipLaunchKernelGGL(k_r_mv<1>, mb, tb, 0, st, L, tiles, sc, w.ph, w.r0, w.v, part);
        hipLaunchKernelGGL(k_r_s, vb, tb, 0, st, L, e0, e1, sc, part, nb_mv, w);
        RET_IF(cad_mg_cycle(c, w.r, w.sh));
        hipLaunchKernelGGL(k_r_mv<2>, mb, tb, 0, st, L, tiles, sc, w.sh, w.r, w.t, part);
        hipLaunchKernelGGL(k_r_xr, vb, tb, 0, st, L, e0, e1, sc, nb_mv, w, part);
        hipLaunchKernelGGL(k_r_end, dim3(1), tb, 0, st, part, nb_vec, sc, c->host_rec);
        CAD_CHECK(hipGetLastError());
        return CAD_OK;
    }

    bool timed() const { return c->kt && c->kt->on; }

    // the iteration as a graph for these planes, or none: events are recorded
    // around its V-cycles, or the capture failed
    int capture()
    {
        cad_mixed *mx = c->mx;
        if (timed() || mx->no_graph) return CAD_OK;
        if (mx->exec && mx->k0 == c->mg_k0 && mx->k1 == c->mg_k1) return CAD_OK;
        if (mx->exec) (void)hipGraphExecDestroy(mx->exec);
        mx->exec = nullptr;
        hipGraph_t g = nullptr;
        int rc = CAD_OK;
        if (hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal) == hipSuccess) {
            rc = iteration();
            if (hipStreamEndCapture(c->stream, &g) != hipSuccess) g = nullptr;
        }
        if (rc != CAD_OK || !g || hipGraphInstantiate(&mx->exec, g, nullptr, nullptr, 0) != hipSuccess) {
            mx->exec = nullptr;
            mx->no_graph = true;
            (void)hipGetLastError();
        }
        if (g) (void)hipGraphDestroy(g);
        mx->k0 = c->mg_k0;
        mx->k1 = c->mg_k1;
        return CAD_OK;
    }

    int launch() const
    {
        if (timed() || !c->mx->exec) return iteration();
        CAD_CHECK(hipGraphLaunch(c->mx->exec, c->stream));
        return CAD_OK;
    }

    // (r, r) of the iteration with that tag, or -1 where it stopped
    int record(double tag, double *v) const
    {
        if (c->host_rec) return cad_wait_record(c, (int)((long long)tag & 1), tag, v);
        CAD_CHECK(hipMemcpyAsync(c->host_red, c->ksc + S_REC, sizeof(double), hipMemcpyDeviceToHost, c->stream));
        CAD_CHECK(hipStreamSynchronize(c->stream));
        *v = c->host_red[0];
        return CAD_OK;
    }

    // up to lim iterations, until (r, r) <= eta2 or a breakdown
    int run(int lim, double eta2, int *count)
    {
        RET_IF(capture());
        const double tag = c->mx->tag;
        c->mx->tag += lim + 1;
        hipLaunchKernelGGL(k_r_start, dim3(1), dim3(REDUCE_THREADS), 0, c->stream, c->red_partial, nb_vec, c->ksc, eta2,
                           tag);
        CAD_CHECK(hipGetLastError());
        const bool may_lead = c->host_rec && !timed();
        int launched = 0, known = 0;
        double rr = 1.0, trend = 0.01;   // (r, r) of the scaled residual; a V-cycled iteration's usual reduction
        for (;;) {
            if (launched == known) {
                RET_IF(launch());
                launched++;
            }
            if (may_lead && launched < lim && rr * trend > eta2) {
                RET_IF(launch());
                launched++;
            }
            double v = 0.0;
            RET_IF(record(tag + (double)(known + 1), &v));
            known++;
            if (v < 0.0 || known == lim) break;
            trend = std::fmin(1.0, v / rr);
            rr = v;
        }
        *count = known;
        return CAD_OK;
    }
};

}  // namespace

int cad_solve_mixed(cad_ctx *c, double *x0, double *bnorm_out, double *xnorm_out, int *iter_out)
{
    const Dims &d = c->d;
    const long long nc = d.nc;
    hipStream_t st = c->stream;
    const dim3 vb(VB), tb(256);
    double *x = c->xw, *r64 = c->rr;   // FP64: the solution, the outer residual
    hipLaunchKernelGGL(k_r_fill, vb, tb, 0, st, nc, x);
    CAD_CHECK(hipGetLastError());
    unsigned long long hr[2];
    RET_IF(cad_ext_active_range(c, hr));
    if (hr[0] >= hr[1]) {
        *bnorm_out = 0.0;
        *xnorm_out = 0.0;
        *iter_out = 0;
        return CAD_OK;
    }
    // level 0's planes: those with active cells, widened to fours so that a
    // moving surface seldom asks for another graph (the planes between hold
    // inactive rows only)
    const int ka = (int)(hr[0] / (unsigned long long)d.nij) + 1, kb = (int)((hr[1] - 1) / (unsigned long long)d.nij) + 1;
    c->mg_span = hr[1] - hr[0];
    c->mg_planes = kb - ka + 1;
    c->mg_k0 = std::max(2, ka & ~3);
    c->mg_k1 = std::min(d.nk - 1, kb | 3);
    RET_IF(cad_mg_setup(c));
    RET_IF(mixed_alloc(c));
    const MgLevel &L0 = c->mg[0];
    const long long lk = (long long)L0.ld * d.nj, ns = lk * d.nk;
    const long long n0 = (c->mg_k0 - 1) * d.nij, n1 = c->mg_k1 * d.nij;
    Inner in;
    in.c = c;
    float *f = c->mx->mem;
    in.w = {L0.b, f, f + ns, f + 2 * ns, f + 3 * ns, f + 4 * ns, L0.x, f + 5 * ns};
    in.e0 = (int)(lk * (c->mg_k0 - 1) / 4);
    in.e1 = (int)(lk * c->mg_k1 / 4);
    const int planes = c->mg_k1 - c->mg_k0 + 1;
    in.tiles = {c->mg_k0, (d.ni / 2 + 64) / 64, (d.nj - 2 + 3) / 4, 0};
    in.tiles.n = in.tiles.qt * in.tiles.jt * planes * 2;
    in.nb_mv = std::min(REDUCE_BLOCKS, in.tiles.n);
    in.nb_vec = std::min(REDUCE_BLOCKS, (in.e1 - in.e0 + 255) / 256);
    // the V-cycles' results are read one plane beyond theirs, where they stay 0
    const long long x_lo = lk * (c->mg_k0 - 2), x_n = lk * (planes + 2);
    hipLaunchKernelGGL(k_r_fill32, vb, tb, 0, st, x_n, in.w.ph + x_lo, in.w.sh + x_lo);
    // x = x0 on the active rows
    hipLaunchKernelGGL(k_r_copy, vb, tb, 0, st, L0, n0, n1, x0, x);
    CAD_CHECK(hipGetLastError());
    double bn2 = 0.0;
    RET_IF(cad_ext_dot(c, c->bb, c->bb, &bn2));
    const double bnorm = std::sqrt(bn2);
    // the reference's stop on the true residual, held to the context's true
    // relative residual when one is set
    double tol = c->prm.cgepsr * bnorm + c->prm.cgepsa;
    if (c->true_stop > 0.0) tol = std::fmin(tol, c->true_stop * bnorm);
    const int cap = cad_krylov_cap(c);
    int inner_total = 0, outer = 0;
    double rn = 0.0, prev = -1.0;
    bool fail = false;
    for (;;) {
        RET_IF(cad_ext_residual(c, x, r64));
        double rr64 = 0.0;
        RET_IF(cad_ext_dot(c, r64, r64, &rr64));
        rn = std::sqrt(rr64);
        if (!std::isfinite(rn)) {
            fail = true;
            break;
        }
        if (rn <= tol) break;
        if (inner_total >= cap || outer >= 20 || (prev > 0.0 && !(rn < 0.5 * prev))) {
            fail = true;
            break;
        }
        prev = rn;
        const double eta = std::fmax(1.0e-6, 0.1 * tol / rn);
        hipLaunchKernelGGL(k_r_init, dim3(in.nb_vec), tb, 0, st, L0, n0, n1, r64, 1.0 / rn, in.w, c->red_partial);
        CAD_CHECK(hipGetLastError());
        int count = 0;
        RET_IF(in.run(std::min(60, cap - inner_total), eta * eta, &count));
        inner_total += count;
        hipLaunchKernelGGL(k_r_update, vb, tb, 0, st, L0, n0, n1, rn, in.w.d, x);
        CAD_CHECK(hipGetLastError());
        outer++;
    }
    if (fail && std::isfinite(rn)) {
        // the refinement stalled: the reference's MILU-BiCGSTAB finishes the
        // solve from the current x, held to the same true relative residual
        hipLaunchKernelGGL(k_r_copy, vb, tb, 0, st, L0, n0, n1, x, x0);
        CAD_CHECK(hipGetLastError());
        const double keep_stop = c->true_stop;
        c->true_stop = keep_stop > 0.0 ? std::fmin(keep_stop, c->prm.cgepsr) : c->prm.cgepsr;
        double bn = 0.0, xn = 0.0;
        int fit = 0;
        const int rc = cad_solve_m1bcgs(c, x0, &bn, &xn, &fit);
        c->true_stop = keep_stop;
        RET_IF(rc);
        c->mixed_fallbacks++;
        c->mixed_fallback_iters = fit;
        *bnorm_out = bnorm;
        if (fit >= 0 && fit <= c->prm.icgmax) {
            double rel = 0.0;
            RET_IF(cad_poisson_residual_x(c, x0, &rel));
            *xnorm_out = rel;
            *iter_out = inner_total + fit;
        } else {
            *xnorm_out = bnorm > 0.0 ? rn / bnorm : rn;
            *iter_out = fit < 0 ? fit : c->prm.icgmax + 1;
        }
        return CAD_OK;
    }
    if (!fail) {
        hipLaunchKernelGGL(k_r_copy, vb, tb, 0, st, L0, n0, n1, x, x0);
        CAD_CHECK(hipGetLastError());
    }
    *bnorm_out = bnorm;
    *xnorm_out = bnorm > 0.0 ? rn / bnorm : rn;
    *iter_out = fail ? -2 : inner_total;
    return CAD_OK;
}
