// cad_wave_sweep.hip -- the MILU sweeps of M^-1 (vf_mzfrwd.f:37-48,
// vf_mzbkwd.f:37-47) on operands laid out in the order a wavefront walks them.
//
// Every cell evaluates the reference's expression on the same operands in the
// same order (cad_sweep.hip), so the results are the serial sweep's bits.  The
// recurrence is a chain: its time is (steps of the longest path through the
// grid) x (time of a step) + (handovers between workgroups) x (their latency),
// far above what its bytes cost.  So a step holds only what the recurrence
// needs, and nothing that takes long is waited for inside it.  A single wave
// issues one instruction every 4.5 cycles whatever its kind (measured), so the
// walk's time is its instruction count: everything that is not the recurrence
// is done by other waves.
//
// Tiles.  A workgroup has one or two walking waves of 16 (J) x 4 (K) lines
// along I, stacked in K, a helper wave for each, and two receivers.  Lane
// jl + 16 kl walks line (J,K) with a skew of jl + 2 kl steps: its cell of step
// (diagonal) d is I = d - jl - 2 kl.  The J neighbour is then lane jl-1's value of
// the last step, one DPP row shift (lanes jl = 0 keep the halo value that the
// shift leaves in place).  The K neighbour is lane kl-1's value of two steps
// before: every step's value goes to a ring in LDS and comes back with a read
// issued behind the write, a step before it is needed; lanes kl = 0 read
// the halo ring at the same offsets.  A backward sweep walks the same diagonals
// downwards with the roles of the first and last lanes swapped.
//
// Operands.  The matrix products and coefficients are packed once per
// factorisation as [wave][diagonal pair][lane][2] (k_wave_pack): one 16-byte
// load per lane and pair, 1 KB contiguous per wave, straight into registers 16
// steps ahead.  The intermediate X of the two sweeps has that layout too.  Y and
// the final X are in the grid's order; the helpers move them between memory and
// the rings, four lanes to the 64 bytes of a line's stage (8 steps).
//
// Handovers.  Values for the next tile go out as {value, sequence number}
// mailbox entries, written by the helpers, never waited for.  They are indexed
// by the consumer's own diagonal, so a stage of a tile's K halo is 2 KB
// contiguous and of a wave's J halo 512 bytes.  The receivers (one for the K
// halo, one for the J halos) poll them a stage at a time and put them into rings
// (a poll's latency grows with its cache lines: polls of two stages ahead
// made M^-1 9 % slower on 512x256x128, three polls in flight 14 to 25 %); a second walking wave reads the first
// one's ring.  All waves keep pace by stage counters in LDS, which a walking wave
// looks at once a stage, a stage ahead.  LDS operations of a wave execute in
// order, so a counter written after its values is seen after them.
//
// Order.  Workgroups take tiles in dependency order from an atomic ticket, so
// a tile waits only on tiles that run; every wait is bounded and sets the error
// flag that the host reports.
//
// What bounds it: a step is 65-80 ns, about 20 instructions and, with two walking
// waves on a CU, the L1's 64 bytes a cycle; a tile-to-tile handover costs 2-3 us,
// half of it the steps of the skew, the rest the way through memory.  With a skew of
// four steps between K rows (values through the ring in pairs) M^-1 took 55 us on
// 64x16x48 and 382 on 512x256x128, with two 46 and 368, with polls of one stage
// and the J halo whole in its own entries 43 and 312.  M^-1 on water
// of the workloads, against the 64-line tiles of cad_sweep.hip (whose step was 240
// ns, waiting for its mailbox accesses): buildings 512x256x128 661 -> 313 us, run-up
// 512x32x96 330 -> 157, 250x70x90 267 -> 130, dam break 64x16x48 61 -> 43.  Those
// tiles stay for the factorisation, for the fixed tile shapes, on tall columns, and
// where these arrays do not fit.
#include "cad_common.h"
#include "cad_sweep.h"

#include <algorithm>
#include <climits>
#include <new>

namespace {

typedef double v2d __attribute__((ext_vector_type(2)));

constexpr int TJ = 16, TKW = 4;                  // lines of a wave in J and K
constexpr int DK = 2;                            // steps between a wave's K rows
constexpr int SKMAX = (TJ - 1) + DK * (TKW - 1);   // largest skew in a wave
constexpr int S = 8, PQ = S / 2;                 // steps and step pairs of a stage
constexpr int KOFF = DK * (TKW - 1);             // diagonals between a wave's first and last K row
constexpr int KPAD = 16, JPAD = 24;              // mailbox diagonals before 0
constexpr int RX = 8, RY = 4;                    // stages of the LDS rings (value and halo rings; Y)
constexpr int SLOT = 1024;                       // bytes of a ring slot: a pair of steps of 64 lanes
constexpr unsigned LDS_SPINS = 1u << 22;

struct WGeom {
    int ni, nj, nk;
    int ntj, ntk, ntiles;
    int nd;                         // diagonals per wave, a multiple of S
    long long nij, nc;
};

struct WCtl {
    const int *order;               // tiles in dependency order
    const int2 *range;              // per tile: first, last active I (0-based); x > y: none
    v4u *mb;                        // K entries [tile][nd + 2 KPAD][16], then J [tile][wave][nd + 2 JPAD][4]
    unsigned mb_bytes, j_base;      // bytes in all; offset of the J entries
    unsigned long long *ticket;
    unsigned long long base;
    unsigned seq;
    int *err;
    const double *stop;             // not null and not 0: nothing to do
};

// forward: LPI, LPJ, LPK packed (LPI = MARK on cells that are not active), Y in
// the grid's order, X packed out
struct WFwd {
    static constexpr int NP = 3, DIR = 1;
    const v2d *src[NP];
    const double *nat_in;
    v2d *pk_out;
    double *nat_out;
    __device__ __forceinline__ static double step(const double *v, double y, double xi, double xj, double xk)
    {
        const double r = y - v[0] * xi - v[1] * xj - v[2] * xk;
        return is_mark(v[0]) ? 0.0 : r;
    }
};

// backward: AUI, AUJ, AUK, DD (0 on cells that are not active), X packed, X out
// in the grid's order
struct WBwd {
    static constexpr int NP = 5, DIR = -1;
    const v2d *src[NP];
    const double *nat_in;
    v2d *pk_out;
    double *nat_out;
    __device__ __forceinline__ static double step(const double *v, double, double xi, double xj, double xk)
    {
        const double r = (v[4] - v[0] * xi - v[1] * xj - v[2] * xk) * v[3];
        return v[3] != 0.0 ? r : 0.0;
    }
};

// Rings are indexed by the walking order: slot of pair q of stage ordinal m is
// (m % depth) * PQ + q, and a pair holds its first step's value first.
template <int NW>
struct __attribute__((aligned(16))) WSmem {
    char xr[NW][RX * PQ * SLOT];     // values of walking wave o (in walking order): [slot][lane][2]
    char kr[RX * PQ * SLOT];         // K halo of wave 0: [slot][jl][2] at the same pitch
    char yr[NW][RY * PQ * SLOT];     // forward: Y of wave o: [slot][lane][2]
    double jr[NW][RX * PQ][TKW][2];  // J halo of wave o: [slot][kl][2]
    // stage counters that wave o waits for: K halo (o = 0), J halo, Y, stages its
    // helper has stored; unused ones hold INT_MAX
    int in[NW][4];
    int done[NW][64];                // stages wave o has walked (in [o][0]; one lane each)
    int tile;
};

// LDS counters: plain LDS accesses that the compiler neither drops nor moves
// across order_lds()
__device__ __forceinline__ void order_lds() { __asm__ __volatile__("" ::: "memory"); }
__device__ __forceinline__ int cnt_load(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void cnt_store(int *p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int DIR>
__device__ __forceinline__ double from_j(double halo, double x)
{
    const v2u h = __builtin_bit_cast(v2u, halo), b = __builtin_bit_cast(v2u, x);
    constexpr int ctl = DIR > 0 ? 0x111 : 0x101;   // row_shr:1 / row_shl:1
    v2u r;
    r.x = (unsigned)__builtin_amdgcn_update_dpp((int)h.x, (int)b.x, ctl, 0xF, 0xF, false);
    r.y = (unsigned)__builtin_amdgcn_update_dpp((int)h.y, (int)b.y, ctl, 0xF, 0xF, false);
    return __builtin_bit_cast(double, r);
}

// physical step within a stage of walking step e
template <int DIR>
__device__ __forceinline__ int phys(int e)
{
    return DIR > 0 ? e : S - 1 - e;
}

// The K receiver: halo of walking wave 0.
template <int DIR, int NW>
__device__ void receive_k(WSmem<NW> &sm, const WGeom &g, const WCtl &c, int bj, int bk, int s0, int nst, int lane)
{
    int *flag = &sm.in[0][0];
    const int *done = &sm.done[0][0];
    const int pbk = bk - DIR;
    const int pt = pbk >= 0 && pbk < g.ntk ? bj + pbk * g.ntj : -1;
    const int2 pr = pt >= 0 ? c.range[pt] : make_int2(1, 0);
    const int jl = lane & 15, e0 = lane >> 4;
    if (pr.x > pr.y) {
        for (int n = e0; n < RX * PQ; n += 4) *reinterpret_cast<v2d *>(sm.kr + n * SLOT + jl * 16) = v2d{0.0, 0.0};
        order_lds();
        if (lane == 0) cnt_store(flag, INT_MAX);
        return;
    }
    const int lo = pr.x / S * S, hi = (pr.y + SKMAX) / S * S + S - 1;   // diagonals the producer walks
    const __amdgpu_buffer_rsrc_t r = rsrc(c.mb, c.mb_bytes);
    const unsigned base = (unsigned)(((pt * (g.nd + 2 * KPAD) + KPAD) * TJ + jl) * 16);
    bool late = false;
    unsigned spins = 0;
    for (int m = 0; m < nst;) {
        v3u e[2];
        bool need[2], ok = true;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int d1 = S * (s0 + DIR * m) + phys<DIR>(e0 + 4 * h), d = d1 + KOFF * DIR;
            need[h] = d >= lo && d <= hi;
            e[h] = mb_load(r, need[h] ? base + (unsigned)(d1 * (TJ * 16)) : OOB);
        }
#pragma unroll
        for (int h = 0; h < 2; h++) ok = ok && (!need[h] || e[h].z == c.seq);
        if (__builtin_amdgcn_ballot_w64(!ok) != 0) {
            __builtin_amdgcn_s_sleep(1);
            if ((++spins & 1023u) == 0u) {
                if (spins > SPIN_LIMIT) atomicOr(c.err, 2);
                if (__hip_atomic_load(c.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
            }
            continue;
        }
        unsigned n = 0;
        while (!late && cnt_load(done) <= m - RX) {
            __builtin_amdgcn_s_sleep(1);
            if (++n > LDS_SPINS) late = true;
        }
        order_lds();
        const int sl = (m & (RX - 1)) * PQ;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int w = e0 + 4 * h;
            *reinterpret_cast<double *>(sm.kr + (sl + (w >> 1)) * SLOT + jl * 16 + (w & 1) * 8) =
                need[h] ? __builtin_bit_cast(double, v2u{e[h].x, e[h].y}) : 0.0;
        }
        m++;
        spins = 0;
        order_lds();
        if (lane == 0) cnt_store(flag, m);
        order_lds();
    }
    order_lds();
    if (lane == 0) {
        cnt_store(flag, INT_MAX);
        if (late) atomicOr(c.err, 2);
    }
}

// The J receiver: lanes 0..31 serve walking wave 0, lanes 32..63 wave 1.  With one
// walking wave the upper lanes leave: a lane's load is its own, served at a time of
// its own, so a second lane with the same entry would store a value whose
// sequence number nobody has looked at.
template <int DIR, int NW>
__device__ void receive_j(WSmem<NW> &sm, const WGeom &g, const WCtl &c, int bj, int bk, int s0, int nst, int lane)
{
    if (lane >= 32 * NW) return;
    const int o = lane >> 5, w = DIR > 0 ? o : NW - 1 - o;
    int *flag = &sm.in[o][1];
    const int *done = &sm.done[o][0];
    const int pbj = bj - DIR;
    const int pt = pbj >= 0 && pbj < g.ntj ? pbj + bk * g.ntj : -1;
    const int2 pr = pt >= 0 ? c.range[pt] : make_int2(1, 0);
    const int kl = lane & 3, e0 = (lane & 31) >> 2;
    if (pr.x > pr.y) {
        for (int n = e0; n < RX * PQ; n += 8) *reinterpret_cast<v2d *>(&sm.jr[o][n][kl][0]) = v2d{0.0, 0.0};
        order_lds();
        if ((lane & 31) == 0) cnt_store(flag, INT_MAX);
        return;
    }
    const int lo = pr.x / S * S, hi = (pr.y + SKMAX) / S * S + S - 1;
    const __amdgpu_buffer_rsrc_t r = rsrc(c.mb, c.mb_bytes);
    const unsigned base = c.j_base + (unsigned)((((pt * NW + w) * (g.nd + 2 * JPAD) + JPAD) * TKW + kl) * 16);
    int m = 0;                       // stages ready, per half
    unsigned spins = 0;
    const unsigned long long half = o ? 0xFFFFFFFF00000000ull : 0x00000000FFFFFFFFull;
    while (__builtin_amdgcn_ballot_w64(m < nst) != 0) {
        const int d1 = S * (s0 + DIR * m) + phys<DIR>(e0), d = d1 + (TJ - 1) * DIR;
        const bool need = m < nst && d >= lo && d <= hi;
        const v3u e = mb_load(r, need ? base + (unsigned)(d1 * (TKW * 16)) : OOB);
        const int dn = cnt_load(done);
        const bool ok = m < nst && (!need || e.z == c.seq) && dn > m - RX;
        const bool got = (__builtin_amdgcn_ballot_w64(!ok) & half) == 0;
        order_lds();
        if (got) {
            sm.jr[o][(m & (RX - 1)) * PQ + (e0 >> 1)][kl][e0 & 1] =
                need ? __builtin_bit_cast(double, v2u{e.x, e.y}) : 0.0;
            m++;
        }
        order_lds();
        if (got && (lane & 31) == 0) cnt_store(flag, m);
        order_lds();
        if (__builtin_amdgcn_ballot_w64(got) == 0) {
            __builtin_amdgcn_s_sleep(1);
            if ((++spins & 1023u) == 0u) {
                if (spins > SPIN_LIMIT) atomicOr(c.err, 2);
                if (__hip_atomic_load(c.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
            }
        } else {
            spins = 0;
        }
    }
    order_lds();
    if ((lane & 31) == 0) cnt_store(flag, INT_MAX);
}

// The helper of walking wave o (physical wave w): publishes and stores the
// stages it has walked and, forward, brings Y up to RY stages ahead.
template <class Op, int NW>
__device__ void help(WSmem<NW> &sm, const WGeom &g, const WCtl &c, const Op &op, int tile, int bj, int bk, int o, int w,
                     int s0, int nst, int lane)
{
    constexpr int DIR = Op::DIR;
    constexpr bool FWD = DIR > 0;
    constexpr int JP = FWD ? TJ - 1 : 0, KP = FWD ? TKW - 1 : 0;   // publishing lanes
    const bool has_j = bj + DIR >= 0 && bj + DIR < g.ntj, has_k = bk + DIR >= 0 && bk + DIR < g.ntk;
    const bool pub_k = o == NW - 1 && has_k;
    const __amdgpu_buffer_rsrc_t rmb = rsrc(c.mb, c.mb_bytes);
    // K entries: lane = jl + 16 e0, walking steps e0 and e0 + 4; J: kl + 4 e
    const int e0 = lane >> 4, kj = lane & 3, ej = lane >> 2;
    const unsigned kbase = (unsigned)(((tile * (g.nd + 2 * KPAD) + KPAD - KOFF * DIR) * TJ + (lane & 15)) * 16);
    const bool jlane = has_j && ej < S;
    const unsigned jbase =
        c.j_base + (unsigned)((((tile * NW + w) * (g.nd + 2 * JPAD) + JPAD - (TJ - 1) * DIR) * TKW + kj) * 16);
    // grid order: lane = pair + 4 (line % 16), lines in four groups of 16; in a
    // group kl is fixed.  nat: byte offset of diagonal 0's cell (positive: j > jl,
    // k > kl)
    const __amdgpu_buffer_rsrc_t rnat = rsrc(FWD ? op.nat_in : op.nat_out, (unsigned long long)g.nc * 8);
    const int pq = lane & 3, jn = lane >> 2, pp = FWD ? pq : 3 - pq;   // walking and physical pair
    unsigned nat[TKW];
#pragma unroll
    for (int kl = 0; kl < TKW; kl++) {
        const int j = 1 + bj * TJ + jn, k = 1 + (bk * NW + w) * TKW + kl;
        nat[kl] = j <= g.nj - 2 && k <= g.nk - 2
                      ? (unsigned)(((long long)j * g.ni + (long long)k * g.nij - jn - DK * kl) * 8)
                      : OOB;
    }
    const unsigned long long pk0 = (unsigned long long)(tile * NW + w) * g.nd * 512, pkn = (unsigned long long)g.nd * 512;
    const __amdgpu_buffer_rsrc_t rpx = rsrc(reinterpret_cast<const char *>(op.pk_out) + pk0, pkn);
    const int *done = &sm.done[o][0];
    char *xr = sm.xr[o], *yr = sm.yr[o];

    // Y goes through registers YS stages before its ring slot is free
    constexpr int YS = 3;
    v2d y[YS][TKW];
    auto load_y = [&](int m, v2d (&v)[TKW]) {
        const int s = s0 + DIR * min(m, nst - 1);
#pragma unroll
        for (int kl = 0; kl < TKW; kl++)
            v[kl] = __builtin_bit_cast(v2d, __builtin_amdgcn_raw_buffer_load_b128(
                                                rnat, m < nst && nat[kl] != OOB ? nat[kl] + 16 * pp : OOB, s * 64, 0));
    };
    auto put_y = [&](int m, const v2d (&v)[TKW]) {
        char *p = yr + ((m & (RY - 1)) * PQ + pq) * SLOT + jn * 16;
#pragma unroll
        for (int kl = 0; kl < TKW; kl++) *reinterpret_cast<v2d *>(p + kl * 256) = v[kl];
    };
    // one stage of zeros past the last (an odd walk ends with it)
    const int ny = nst + 1;
    if (FWD) {
#pragma unroll
        for (int m = 0; m < YS; m++) load_y(m, y[m]);
#pragma unroll
        for (int m = 0; m < RY; m++) {
            put_y(m, y[m % YS]);
            order_lds();
            if (lane == 0) cnt_store(&sm.in[o][2], m + 1);
            order_lds();
            load_y(m + YS, y[m % YS]);
        }
    }
    bool late = false;
    for (int m0 = 0; m0 < nst; m0 += YS) {
#pragma unroll
        for (int u = 0; u < YS; u++) {
            const int m = m0 + u;
            if (m >= nst) continue;
            unsigned n = 0;
            while (!late && cnt_load(done) <= m)
                if (++n > LDS_SPINS) late = true;
            order_lds();
            const int s = s0 + DIR * m;
            const char *slot = xr + (m & (RX - 1)) * (PQ * SLOT);
            if (pub_k) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int e = e0 + 4 * h, d = S * s + phys<DIR>(e);
                    const double x = *reinterpret_cast<const double *>(slot + (e >> 1) * SLOT +
                                                                       (16 * KP + (lane & 15)) * 16 + (e & 1) * 8);
                    mb_store(rmb, kbase + (unsigned)(d * (TJ * 16)), x, c.seq);
                }
            }
            if (has_j) {
                const int d = S * s + phys<DIR>(ej & 7);
                const double x =
                    *reinterpret_cast<const double *>(slot + ((ej & 7) >> 1) * SLOT + (JP + 16 * kj) * 16 + (ej & 1) * 8);
                mb_store(rmb, jlane ? jbase + (unsigned)(d * (TKW * 16)) : OOB, x, c.seq);
            }
            if (FWD) {
                // stage m + RY: its Y was loaded YS stages ago
                put_y(m + RY, y[(u + RY) % YS]);
                order_lds();
                if (lane == 0) cnt_store(&sm.in[o][2], m + RY + 1 < ny ? m + RY + 1 : INT_MAX);
                order_lds();
                load_y(m + RY + YS, y[(u + RY) % YS]);
#pragma unroll
                for (int q = 0; q < PQ; q++)
                    __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const v4u *>(slot + q * SLOT + lane * 16),
                                                           rpx, lane * 16 + q * 1024, s * 4096, 0);
            } else {
#pragma unroll
                for (int kl = 0; kl < TKW; kl++) {
                    // cells of the line, and the ghost cells at its ends, which
                    // hold 0 and get 0
                    const v2d x = *reinterpret_cast<const v2d *>(slot + pq * SLOT + (jn + 16 * kl) * 16);
                    const int i = S * s + 2 * pp - jn - DK * kl;
                    const unsigned off =
                        nat[kl] != OOB && (unsigned)(i + 1) <= (unsigned)g.ni ? nat[kl] + 16 * pp : OOB;
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v2d{x[1], x[0]}), rnat, off, s * 64, 0);
                }
            }
            order_lds();
            if (lane == 0) cnt_store(&sm.in[o][3], m + 1);
            order_lds();
        }
    }
    if (lane == 0) {
        cnt_store(&sm.in[o][2], INT_MAX);
        cnt_store(&sm.in[o][3], INT_MAX);
    }
    if (late && lane == 0) atomicOr(c.err, 2);
}

// waves of a workgroup: walking waves, their helpers, the receivers
constexpr int waves(int nw) { return 2 * nw + 2; }

template <class Op, int NW>
__global__ void __launch_bounds__(64 * waves(NW), 1) k_wave(WGeom g, WCtl c, Op op)
{
    constexpr int DIR = Op::DIR, NP = Op::NP;
    constexpr bool FWD = DIR > 0;
    __shared__ WSmem<NW> sm;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (threadIdx.x == 0) {
        const unsigned long long tk = atomicAdd(c.ticket, 1ull);
        const long long tix = (long long)(tk - c.base);
        if (tix < 0 || tix >= g.ntiles) {
            atomicOr(c.err, 1);
            sm.tile = -1;
        } else {
            sm.tile = c.order[DIR > 0 ? tix : g.ntiles - 1 - tix];
        }
    }
    // counters; the two pairs before the first step are zero
    if (threadIdx.x < NW * 4) {
        const int q = threadIdx.x;   // [1][0] is unused; [o][2] is used forward
        sm.in[q >> 2][q & 3] = q == 4 || (!FWD && (q & 3) == 2) ? INT_MAX : 0;
    }
    if (threadIdx.x < NW * 64) {
        const int o = threadIdx.x >> 6;
        sm.done[o][lane] = 0;
#pragma unroll
        for (int q = 2; q < PQ; q++)
            *reinterpret_cast<v2d *>(sm.xr[o] + ((RX - 1) * PQ + q) * SLOT + lane * 16) = v2d{0.0, 0.0};
    }
    __syncthreads();
    const int tile = __builtin_amdgcn_readfirstlane(sm.tile);
    if (tile < 0 || (c.stop && *c.stop != 0.0)) return;
    const int2 rg = c.range[tile];
    if (rg.x > rg.y) return;
    const int bj = tile % g.ntj, bk = tile / g.ntj;
    const int sa = rg.x / S, sb = (rg.y + SKMAX) / S, nst = sb - sa + 1;
    const int s0 = FWD ? sa : sb;
    if (wid == 2 * NW) {
        receive_k<DIR, NW>(sm, g, c, bj, bk, s0, nst, lane);
        return;
    }
    if (wid > 2 * NW) {
        receive_j<DIR, NW>(sm, g, c, bj, bk, s0, nst, lane);
        return;
    }
    const int o = wid & (NW - 1), w = FWD ? o : NW - 1 - o;
    if (wid >= NW) {
        help<Op, NW>(sm, g, c, op, tile, bj, bk, o, w, s0, nst, lane);
        return;
    }

    // ------------------------------------------------------- walking waves
    const int jl = lane & 15, kl = lane >> 4;
    constexpr int KH = FWD ? 0 : TKW - 1, KP = TKW - 1 - KH;   // K row that takes the halo, and the last one
    const unsigned long long pk0 = (unsigned long long)(tile * NW + w) * g.nd * 512, pkn = (unsigned long long)g.nd * 512;
    __amdgpu_buffer_rsrc_t rp[NP];
#pragma unroll
    for (int a = 0; a < NP; a++) rp[a] = rsrc(reinterpret_cast<const char *>(op.src[a]) + pk0, pkn);

    v2d buf[2][PQ][NP];
    // operands of pair q (in walking order) of stage ordinal m; zeros past the
    // last stage
    auto fetch = [&](unsigned lo, int so, int q, v2d (&b)[NP]) {
#pragma unroll
        for (int a = 0; a < NP; a++)
            b[a] = __builtin_bit_cast(
                v2d, __builtin_amdgcn_raw_buffer_load_b128(rp[a], lo + 1024 * (FWD ? q : PQ - 1 - q), so, 0));
    };
    const unsigned lane16 = lane * 16;
    auto fetch_lo = [&](int m) { return m < nst ? lane16 : OOB - 4096; };
    auto fetch_so = [&](int m) { return (s0 + DIR * min(m, nst - 1)) * 4096; };
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int q = 0; q < PQ; q++) fetch(fetch_lo(u), fetch_so(u), q, buf[u][q]);

    // where this lane's K neighbour comes from: the own wave's ring a pair back,
    // the K halo ring, or the first wave's ring three pairs on
    char *const lds = reinterpret_cast<char *>(&sm);
    const char *kbase;
    int koff;
    if (kl != KH) {
        kbase = sm.xr[o] + (lane - 16 * DIR) * 16;
        koff = -DK / 2;
    } else if (o == 0) {
        kbase = sm.kr + jl * 16;
        koff = 0;
    } else {
        kbase = sm.xr[0] + (jl + 16 * KP) * 16;
        koff = KOFF / 2;
    }
    const int kb = (int)(kbase - lds);
    char *const xw = sm.xr[o] + lane * 16;
    const char *const yb = sm.yr[o] + lane * 16;
    const int *f = sm.in[o], *other = &sm.done[NW - 1 - o][0];
    int *const mine = &sm.done[o][lane];
    v2d kq[PQ], jq[PQ], yq[PQ];
    auto kaddr = [&](int p) { return kb + ((p + koff) & (RX * PQ - 1)) * SLOT; };
    // J halo and Y of pair q of stage m
    auto halo = [&](int m, int q) {
        jq[q] = *reinterpret_cast<const v2d *>(&sm.jr[o][(m & (RX - 1)) * PQ + q][kl][0]);
        if (FWD) yq[q] = *reinterpret_cast<const v2d *>(yb + ((m & (RY - 1)) * PQ + q) * SLOT);
    };
    bool late = false;
    // whether stage m may be read and the ring has room for it (a: in[o], b: the
    // other wave's stages).  Wave 1 reads wave 0's stage m + 1 during its own
    // stage m; wave 0 must not overtake it by the ring.
    const int ahead = NW == 1 ? INT_MIN / 2 : o == 0 ? 1 - RX : 2;
    auto allowed = [&](int4 a, int b, int m) {
        const int k = __builtin_amdgcn_readfirstlane(a.x), j = __builtin_amdgcn_readfirstlane(a.y);
        const int y = __builtin_amdgcn_readfirstlane(a.z), h = __builtin_amdgcn_readfirstlane(a.w);
        return min(min(k, j), y) > m && h >= m - (RX - 1) && __builtin_amdgcn_readfirstlane(b) >= m + ahead;
    };
    auto wait_for = [&](int m) {
        unsigned n = 0;
        for (;;) {
            order_lds();
            const int4 a = *reinterpret_cast<const int4 *>(f);
            const int b = *other;
            if (late || allowed(a, b, m)) break;
            // once a wait has given up none waits again
            if (++n > LDS_SPINS) late = true;
        }
        order_lds();
    };
    wait_for(0);
    kq[0] = *reinterpret_cast<const v2d *>(lds + kaddr(0));
    halo(0, 0);
    halo(0, 1);

    // Two stages a turn; an odd walk ends with a stage of zeros.
    double x = 0.0;
    for (int m0 = 0; m0 < nst; m0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int m = m0 + u;
            const unsigned flo = fetch_lo(m + 2);
            const int fso = fetch_so(m + 2);
            // the K neighbours' pairs PQ m + 1 .. 3 lie in one stage's slots
            const int ka1 = kaddr(PQ * m + 1), ka2 = kaddr(PQ * m + 4);
            char *const xs = xw + (m & (RX - 1)) * (PQ * SLOT);
            int4 fa;
            int fb;
#pragma unroll
            for (int q = 0; q < PQ; q++) {
                const char *const kn = lds + (q < PQ - 1 ? ka1 + q * SLOT : ka2);
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const int h = FWD ? t : 1 - t;   // physical step of the pair
                    double v[NP];
#pragma unroll
                    for (int a = 0; a < NP; a++) v[a] = buf[u][q][a][h];
                    const double xj = from_j<DIR>(jq[q][t], x);
                    x = Op::step(v, FWD ? yq[q][t] : 0.0, x, xj, kq[q][t]);
                    // and the same step's K value of the next pair
                    *reinterpret_cast<double *>(xs + q * SLOT + 8 * t) = x;
                    order_lds();
                    kq[(q + 1) & (PQ - 1)][t] = *reinterpret_cast<const double *>(kn + 8 * t);
                }
                fetch(flo, fso, q, buf[u][q]);
                // the pair after next
                order_lds();
                if (q < 2)
                    halo(m, q + 2);
                else
                    halo(m + 1, q - 2);
                if (q == 0) {
                    fa = *reinterpret_cast<const int4 *>(f);
                    fb = *other;
                }
                if (q == 1 && !allowed(fa, fb, m + 1)) wait_for(m + 1);
            }
            order_lds();
            *mine = m + 1;
            order_lds();
        }
    }
    if (o == 0) {
        // the second wave reads up to three pairs past the last stage: the lines
        // hold no active cell there
        const int mz = (nst + 1) / 2 * 2;
        wait_for(mz + 1);
        for (int p = PQ * mz; p < PQ * nst + KOFF / 2; p++)
            *reinterpret_cast<v2d *>(xw + (p & (RX * PQ - 1)) * SLOT) = v2d{0.0, 0.0};
        order_lds();
        *mine = INT_MAX;
    } else {
        *mine = INT_MAX;
    }
    if (late && lane == 0) atomicOr(c.err, 2);
}

// First and last active I of every line (0-based; x > y: none): one wave a line.
__global__ void __launch_bounds__(256) k_line_range(WGeom g, const int *__restrict__ indc, int2 *__restrict__ lr)
{
    const int lane = threadIdx.x & 63;
    const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (n >= (g.nj - 2) * (g.nk - 2)) return;
    const int j = 1 + n % (g.nj - 2), k = 1 + n / (g.nj - 2);
    const int *row = indc + (long long)j * g.ni + (long long)k * g.nij;
    int lo = INT_MAX, hi = -1;
    for (int i = 1 + lane; i <= g.ni - 2; i += 64)
        if (row[i] != -1) {
            lo = min(lo, i);
            hi = max(hi, i);
        }
    for (int off = 32; off > 0; off >>= 1) {
        lo = min(lo, __shfl_down(lo, off, 64));
        hi = max(hi, __shfl_down(hi, off, 64));
    }
    if (lane == 0) lr[n] = make_int2(lo, hi);
}

// the tiles' ranges from their lines'
template <int NW>
__global__ void __launch_bounds__(64 * NW) k_wave_range(WGeom g, const int2 *__restrict__ lr, int2 *__restrict__ range)
{
    const int tile = blockIdx.x, l = threadIdx.x;
    const int j = tile % g.ntj * TJ + l % TJ, k = tile / g.ntj * (TKW * NW) + l / TJ;
    __shared__ int slo[64 * NW], shi[64 * NW];
    const bool ok = j < g.nj - 2 && k < g.nk - 2;
    const int2 r = ok ? lr[k * (g.nj - 2) + j] : make_int2(INT_MAX, -1);
    slo[l] = r.x;
    shi[l] = r.y;
    __syncthreads();
    for (int n = 32 * NW; n > 0; n >>= 1) {
        if (l < n) {
            slo[l] = min(slo[l], slo[l + n]);
            shi[l] = max(shi[l], shi[l + n]);
        }
        __syncthreads();
    }
    if (l == 0) range[tile] = shi[0] < 0 ? make_int2(1, 0) : make_int2(slo[0], shi[0]);
}

// The operands of both sweeps in walking order, 64 diagonals of one wave and one
// operand per block: lines are read along I, turned in LDS and written a
// diagonal pair at a time (the seven operands one after the other took 62 us on
// 64x16x48, side by side 12).  LPI = ALI*DD(n-1), LPJ = ALJ*DD(n-NI), LPK = ALK*DD(n-NIJ), the products
// the reference forms before multiplying by X.
struct PackArgs {
    const double *ali, *alj, *alk, *aui, *auj, *auk, *dd;
    v2d *out[7];
};
template <int NW>
__global__ void __launch_bounds__(256) k_wave_pack(WGeom g, const int2 *__restrict__ range,
                                                   const int *__restrict__ indc, PackArgs a)
{
    __shared__ double t[64][65];
    const int wt = blockIdx.x, tile = wt / NW, w = wt % NW;
    const int2 rg = range[tile];
    const int d0 = blockIdx.y * 64;
    if (rg.x > rg.y || d0 > (rg.y + SKMAX) / S * S + S - 1 || d0 + 63 < rg.x / S * S) return;
    const int bj = tile % g.ntj, bk = tile / g.ntj;
    const int wv = threadIdx.x >> 6, ii = threadIdx.x & 63;
    const double *src[7] = {a.ali, a.alj, a.alk, a.aui, a.auj, a.auk, a.dd};
    const long long back[3] = {1, g.ni, g.nij};
    const long long np = g.nd / 2;
    {
        const int q = blockIdx.z;
        for (int L = wv; L < 64; L += 4) {
            const int jl = L & 15, kl = L >> 4;
            const int j = 1 + bj * TJ + jl, k = 1 + (bk * NW + w) * TKW + kl, i = d0 + ii - jl - DK * kl;
            double v = 0.0;
            if (q == 0) v = __builtin_bit_cast(double, MARK);
            if (j <= g.nj - 2 && k <= g.nk - 2 && i >= 1 && i <= g.ni - 2) {
                const long long n = (long long)j * g.ni + (long long)k * g.nij + i;
                if (indc[n] != -1) v = q < 3 ? src[q][n] * a.dd[n - back[q]] : src[q][n];
            }
            t[L][ii] = v;
        }
        __syncthreads();
        for (int p = wv; p < 32; p += 4)
            if (d0 / 2 + p < np)
                a.out[q][((long long)wt * np + d0 / 2 + p) * 64 + ii] = v2d{t[ii][2 * p], t[ii][2 * p + 1]};
    }
}

constexpr size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

}  // namespace

// The arrays of the packed sweeps: eight packed operands, tile order and
// ranges, mailboxes, in one allocation made on a context's first plain solve.
struct cad_wsweep {
    WGeom g;
    int nw;                 // walking waves of a workgroup
    char *mem;
    v2d *pk[8];             // LPI, LPJ, LPK, AUI, AUJ, AUK, DD, X
    int *order;
    int2 *range, *lines;
    v4u *mb;
    unsigned mb_bytes, j_base;
    size_t pk_bytes;        // of one packed operand
};

namespace {

WCtl wctl(const cad_ctx *c, const double *stop)
{
    const cad_wsweep *ws = c->ws;
    WCtl s;
    s.order = ws->order;
    s.range = ws->range;
    s.mb = ws->mb;
    s.mb_bytes = ws->mb_bytes;
    s.j_base = ws->j_base;
    s.ticket = c->sw_ticket;
    s.base = c->sw_base;
    s.seq = c->sw_seq;
    s.err = c->sw_err;
    s.stop = stop;
    return s;
}

template <class Op>
int wave_launch(cad_ctx *c, const Op &op, const double *stop)
{
    const cad_wsweep *ws = c->ws;
    if (ws->nw == 1)
        hipLaunchKernelGGL((k_wave<Op, 1>), dim3(ws->g.ntiles), dim3(64 * waves(1)), 0, c->stream, ws->g, wctl(c, stop), op);
    else
        hipLaunchKernelGGL((k_wave<Op, 2>), dim3(ws->g.ntiles), dim3(64 * waves(2)), 0, c->stream, ws->g, wctl(c, stop), op);
    CAD_CHECK(hipGetLastError());
    c->sw_base += (unsigned long long)ws->g.ntiles;
    c->sw_seq += 1;
    return CAD_OK;
}

}  // namespace

namespace {

struct WSizes {
    size_t pk, ctl, mb;   // bytes of the packed operands, of order, ranges and lines, of the mailboxes
};

// the geometry and the arrays' sizes for a grid; false where 32-bit offsets do
// not reach, and on tall columns
bool wave_geometry(const Dims &d, cad_wsweep *ws, WSizes *z)
{
    // A tall column's sweep is a chain of tiles in K with next to no walk, and the
    // 64-line tiles of cad_sweep.hip hand over in less time: M^-1 of those / of
    // this file's in us, I x J x K: 105 / 147 on 2x2x200, 204 / 226 on 4x4x300,
    // 235 / 247 on 40x8x300, 294 / 315 on 24x8x400, 554 / 600 on 6x30x800; equal on
    // 24x8x200 and 12x40x400; 126 / 129 on 8x8x160, 135 / 120 on 20x20x128, 106 / 102 on
    // 24x8x120.
    if (d.nk - 2 >= 5 * std::max(d.ni - 2, d.nj - 2) + 80) return false;
    // One walking wave a workgroup has its CU's cache bandwidth to itself, two
    // share it but hand over in LDS what one would through memory, which pays
    // where the K rows are many against the walk and the J tiles.  M^-1 of two / of
    // one in us on tanks filled to 0.7 of their height, I x J x K, inside the line:
    // 43 / 48 on 24x8x40, 34 / 37 on 16x16x32, 42 / 45 on 64x16x32, 63 / 70 on
    // 30x16x64, 72 / 77 on 32x32x64, 120 / 130 on 20x20x128, 76 / 81 on 100x12x64, 68 / 69
    // on 160x10x40, 61 / 60 on 64x16x48 (52 / 53 with water on a third of it), 89 / 90 on
    // 100x30x64, 57 / 60 on 45x25x40, 48 / 47 on 48x12x36, 124 / 121 on 128x24x96.  Outside it: fewer K rows, 28 / 25 on
    // 30x16x16, 43 / 40 on 64x16x24, 37 / 35 on 30x10x28; longer walks, 99 / 96 on
    // 300x8x48; more J tiles, 186 / 152 on 2x300x50, 76 / 73 on 20x60x48, 72 / 70 on 36x36x48,
    // 99 / 93 on 62x60x62; beyond 4096 cells of a plane 167 / 164 on 200x30x128, 89 / 82 on
    // 64x64x48, 452 / 367 on 128x128x256.
    const int ei = d.ni - 2, ej = d.nj - 2, ek = d.nk - 2;
    const int nw = ws->nw = d.ni * d.nj < 4096 && ek >= 30 && 3 * ej <= 2 * ek && ei <= 4 * ek ? 2 : 1;
    WGeom &g = ws->g;
    g.ni = d.ni;
    g.nj = d.nj;
    g.nk = d.nk;
    g.nij = d.nij;
    g.nc = d.nc;
    g.ntj = (d.nj - 2 + TJ - 1) / TJ;
    g.ntk = (d.nk - 2 + TKW * nw - 1) / (TKW * nw);
    g.nd = (d.ni + SKMAX + S - 1) / S * S;
    const unsigned long long nt = (unsigned long long)g.ntj * g.ntk;
    const unsigned long long kb = nt * (g.nd + 2 * KPAD) * TJ * 16, jb = nt * nw * (g.nd + 2 * JPAD) * TKW * 16;
    if (kb + jb > 0x7FFFFFF0ull || (unsigned long long)d.nc * 8 > 0xFFFFFFF0ull) return false;
    g.ntiles = (int)nt;
    ws->mb_bytes = (unsigned)(kb + jb);
    ws->j_base = (unsigned)kb;
    ws->pk_bytes = align256(nt * nw * (size_t)g.nd * 64 * 8);
    z->pk = 8 * ws->pk_bytes;
    z->ctl = align256(nt * sizeof(int)) + align256(nt * sizeof(int2)) +
             align256((size_t)(d.nj - 2) * (d.nk - 2) * sizeof(int2));
    z->mb = align256(ws->mb_bytes);
    return true;
}

// the arrays at their places and the tile order
int wave_place(cad_ctx *c, cad_wsweep *ws, char *pk, char *ctl, char *mb)
{
    for (v2d *&q : ws->pk) {
        q = reinterpret_cast<v2d *>(pk);
        pk += ws->pk_bytes;
    }
    const WGeom &g = ws->g;
    ws->order = reinterpret_cast<int *>(ctl);
    ctl += align256(g.ntiles * sizeof(int));
    ws->range = reinterpret_cast<int2 *>(ctl);
    ctl += align256(g.ntiles * sizeof(int2));
    ws->lines = reinterpret_cast<int2 *>(ctl);
    ws->mb = reinterpret_cast<v4u *>(mb);
    hipLaunchKernelGGL(k_tile_order, dim3((g.ntiles + 255) / 256), dim3(256), 0, c->stream, g.ntj, g.ntk, ws->order);
    CAD_CHECK(hipGetLastError());
    return CAD_OK;
}

__global__ void k_wave_clear(v4u *p, unsigned n)
{
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v4u{0, 0, 0, 0};
}

}  // namespace

// Allocates the packed sweeps' arrays; leaves c->ws null (the caller then uses
// the natural-layout sweeps) on tall columns, when their offsets exceed 31 bits or
// the memory is not there.
int cad_wave_alloc(cad_ctx *c)
{
    if (c->ws || c->ws_off) return CAD_OK;
    c->ws_off = true;
    cad_wsweep *ws = new (std::nothrow) cad_wsweep();
    if (!ws) return CAD_OK;
    WSizes z;
    if (!wave_geometry(c->d, ws, &z)) {
        delete ws;
        return CAD_OK;
    }
    if (hipMalloc((void **)&ws->mem, z.pk + z.ctl + z.mb) != hipSuccess) {
        (void)hipGetLastError();
        delete ws;
        return CAD_OK;
    }
    c->ws = ws;
    c->ws_off = false;
    // the entries start below every launch's sequence number
    char *mb = ws->mem + z.pk + z.ctl;
    hipLaunchKernelGGL(k_wave_clear, dim3(1024), dim3(256), 0, c->stream, reinterpret_cast<v4u *>(mb),
                       (unsigned)(ws->mb_bytes / 16));
    return wave_place(c, ws, ws->mem, ws->mem + z.pk, mb);
}

// The same arrays in memory that the caller owns; leaves c->ws null where they
// do not fit.  *store is the caller's, made on the first call and kept.  The
// mailboxes' memory holds nothing but mailbox entries of earlier calls, whose
// sequence numbers c->sw_seq exceeds (0 at first).
int cad_wave_bind(cad_ctx *c, cad_wsweep **store, char *pk, size_t pk_bytes, char *ctl, size_t ctl_bytes, char *mb,
                  size_t mb_bytes)
{
    if (!*store) *store = new (std::nothrow) cad_wsweep();
    WSizes z;
    if (!*store || !wave_geometry(c->d, *store, &z) || z.pk > pk_bytes || z.ctl > ctl_bytes || z.mb > mb_bytes)
        return CAD_OK;
    c->ws = *store;
    return wave_place(c, *store, pk, ctl, mb);
}

void cad_wave_sweep_free(cad_ctx *c)
{
    if (!c->ws) return;
    (void)hipFree(c->ws->mem);
    delete c->ws;
    c->ws = nullptr;
}

// The packed operands of the context's factorisation (DD, INDC, matrix).
int cad_wave_pack(cad_ctx *c)
{
    const cad_wsweep *ws = c->ws;
    const WGeom &g = ws->g;
    const int nl = (g.nj - 2) * (g.nk - 2);
    hipLaunchKernelGGL(k_line_range, dim3((nl + 3) / 4), dim3(256), 0, c->stream, g, c->f.indc, ws->lines);
    if (ws->nw == 1)
        hipLaunchKernelGGL(k_wave_range<1>, dim3(g.ntiles), dim3(64), 0, c->stream, g, ws->lines, ws->range);
    else
        hipLaunchKernelGGL(k_wave_range<2>, dim3(g.ntiles), dim3(128), 0, c->stream, g, ws->lines, ws->range);
    PackArgs a;
    a.ali = c->ali;
    a.alj = c->alj;
    a.alk = c->alk;
    a.aui = c->aui;
    a.auj = c->auj;
    a.auk = c->auk;
    a.dd = c->dd;
    for (int q = 0; q < 7; q++) a.out[q] = ws->pk[q];
    const dim3 pg(g.ntiles * ws->nw, (g.nd + 63) / 64, 7);
    if (ws->nw == 1)
        hipLaunchKernelGGL(k_wave_pack<1>, pg, dim3(256), 0, c->stream, g, ws->range, c->f.indc, a);
    else
        hipLaunchKernelGGL(k_wave_pack<2>, pg, dim3(256), 0, c->stream, g, ws->range, c->f.indc, a);
    CAD_CHECK(hipGetLastError());
    return CAD_OK;
}

// x = M^-1 y (vf_mzminv.f:38-41); x may be y.  Does nothing if stop is given and
// *stop is not 0.
int cad_wave_minv(cad_ctx *c, double *x, const double *y, const double *stop)
{
    const cad_wsweep *ws = c->ws;
    WFwd f;
    for (int q = 0; q < 3; q++) f.src[q] = ws->pk[q];
    f.nat_in = y;
    f.pk_out = ws->pk[7];
    f.nat_out = x;
    if (int rc = wave_launch(c, f, stop)) return rc;
    WBwd b;
    for (int q = 0; q < 4; q++) b.src[q] = ws->pk[3 + q];
    b.src[4] = ws->pk[7];
    b.nat_in = y;
    b.pk_out = ws->pk[7];
    b.nat_out = x;
    return wave_launch(c, b, stop);
}
