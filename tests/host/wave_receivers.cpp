// The receivers of the packed sweeps (receive_j, receive_k of
// cad_wave_sweep.hip) compiled for the host: the 64 lanes of a wave are fibers
// that meet at the ballots and LDS ordering points, and a mailbox load of one
// lane may be served before the producer's store while another lane's of the
// same poll is served after it, as the memory system is free to do.  A model of the
// walking wave takes each stage when its counter allows and compares the halo
// with what the producer stored.
//
// usage: wave_receivers j|k fwd|bwd NW seed   values under random service order
//        wave_receivers stuck fwd|bwd NW      a walking wave that never walks
// prints "ok" and returns 0, or the first difference and 1.
#include <hip/hip_runtime.h>
#include <ucontext.h>

#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

struct EmuDim {
    unsigned x, y, z;
};
static EmuDim threadIdx, blockIdx, blockDim, gridDim;

// ------------------------------------------------------------ lanes as fibers
namespace emu {
constexpr int LANES = 64;
ucontext_t main_ctx, ctx[LANES];
std::vector<char> stack[LANES];
bool alive[LANES], bits[LANES];
int cur;
void (*body)(int);

void yield() { swapcontext(&ctx[cur], &main_ctx); }
// meeting point of the lanes that have not returned
void sync() { yield(); }
unsigned long long ballot(bool p)
{
    bits[cur] = p;
    sync();
    unsigned long long b = 0;
    for (int l = 0; l < LANES; l++) b |= (unsigned long long)(alive[l] && bits[l]) << l;
    sync();
    return b;
}
void entry(int l)
{
    body(l);
    alive[l] = false;
    bits[l] = false;
    swapcontext(&ctx[l], &main_ctx);
}
// the lanes in turn between meeting points; tick() after each
template <class Tick>
void run(void (*f)(int), Tick tick)
{
    body = f;
    for (int l = 0; l < LANES; l++) {
        stack[l].resize(1 << 17);
        getcontext(&ctx[l]);
        ctx[l].uc_stack.ss_sp = stack[l].data();
        ctx[l].uc_stack.ss_size = stack[l].size();
        ctx[l].uc_link = nullptr;
        makecontext(&ctx[l], (void (*)())entry, 1, l);
        alive[l] = true;
        bits[l] = false;
    }
    for (bool any = true; any;) {
        any = false;
        for (int l = 0; l < LANES; l++)
            if (alive[l]) {
                cur = l;
                swapcontext(&main_ctx, &ctx[l]);
                any = any || alive[l];
            }
        tick();
    }
}

struct Rsrc {
    const char *p;
    unsigned n;
};
typedef unsigned v3 __attribute__((ext_vector_type(3)));
v3 mailbox_load(const Rsrc &r, unsigned off);   // below
}  // namespace emu

#define __amdgpu_buffer_rsrc_t emu::Rsrc
#define __builtin_amdgcn_make_buffer_rsrc(p, s, n, f) (emu::Rsrc{(const char *)(p), (unsigned)(n)})
#define __builtin_amdgcn_raw_buffer_load_b96(r, off, so, pol) emu::mailbox_load(r, off)
#define __builtin_amdgcn_ballot_w64(p) emu::ballot(p)
#define __builtin_amdgcn_s_sleep(n) ((void)0)
#define __builtin_amdgcn_readfirstlane(x) (x)
// of the rest of the file, which is compiled but not run here
#define __builtin_amdgcn_raw_buffer_load_b128(r, off, so, pol) (v4u{0, 0, 0, 0})
#define __builtin_amdgcn_raw_buffer_store_b128(...) ((void)0)
#define __builtin_amdgcn_raw_ptr_buffer_load_lds(...) ((void)0)
#define __builtin_amdgcn_update_dpp(old, src, ctl, rm, bm, bc) (old)
#define __HIP_MEMORY_SCOPE_WORKGROUP 0
#define __HIP_MEMORY_SCOPE_AGENT 0
#undef __hip_atomic_load
#undef __hip_atomic_store
#define __hip_atomic_load(p, o, s) (*(p))
#define __hip_atomic_store(p, v, o, s) ((void)(*(p) = (v)))
#define __launch_bounds__(...)
#define __shared__ static
#define __syncthreads() ((void)0)
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(...) ((void)0)
#define __shfl_down(v, ...) (v)
template <class T>
T atomicAdd(T *p, T v) { T o = *p; *p += v; return o; }
inline int atomicOr(int *p, int v) { int o = *p; *p |= v; return o; }
template <class T>
T min(T a, T b) { return a < b ? a : b; }
template <class T>
T max(T a, T b) { return a > b ? a : b; }
// order_lds() is a meeting point: LDS operations of a wave execute in order
#define __asm__
#define __volatile__(...) emu::sync()
#include WAVE_SOURCE
#undef __asm__
#undef __volatile__

// what the file's host code calls
extern "C" hipError_t hipMalloc(void **, size_t) { return hipErrorOutOfMemory; }
extern "C" hipError_t hipFree(void *) { return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" const char *hipGetErrorString(hipError_t) { return ""; }
void cad_set_error(const char *, ...) {}

// ------------------------------------------------------------------ the case
namespace {

std::mt19937 rng;
std::vector<v4u> box;                    // what the producer has stored, or will
std::vector<int> arrival;                // time from which an entry is stored
std::vector<v4u> old;                    // the entries of the last launch
int now;                                 // time, in meeting points
unsigned seed_, loads[64];               // loads that a lane has made

constexpr unsigned SEQ = 7;

v4u entry_of(double x, unsigned seq)
{
    const v2u b = __builtin_bit_cast(v2u, x);
    return v4u{b.x, b.y, seq, seq};
}

}  // namespace

emu::v3 emu::mailbox_load(const Rsrc &r, unsigned off)
{
    if (off + 12 > r.n || off + 12 < off) return v3{0, 0, 0};
    const size_t e = off / 16;
    // a load instruction's lanes are served in groups of sixteen, some time apart
    std::minstd_rand h(1 + seed_ + 977 * loads[cur]++ + 131071 * (unsigned)(cur >> 4));
    h.discard(4);
    const int t = now - 4 * (int)(h() % 8);
    const v4u v = t >= arrival[e] ? box[e] : old[e];
    return v3{v.x, v.y, v.z};
}

namespace {

template <int DIR, int NW>
struct Case {
    static WSmem<NW> sm;
    static WGeom g;
    static WCtl c;
    static int2 range[4];
    static int err, bj, bk, s0, nst;
    static bool for_j;

    static void lane(int l)
    {
        if (for_j)
            receive_j<DIR, NW>(sm, g, c, bj, bk, s0, nst, l);
        else
            receive_k<DIR, NW>(sm, g, c, bj, bk, s0, nst, l);
    }

    static int main(const std::string &what, unsigned seed)
    {
        rng.seed(seed);
        seed_ = 7919 * seed;
        for_j = what == "j";
        // two tiles in a row or a column; the last one walked is received for
        g.ni = 150;
        g.ntj = for_j ? 2 : 1;
        g.ntk = for_j ? 1 : 2;
        g.nj = 2 + TJ * g.ntj;
        g.nk = 2 + TKW * NW * g.ntk;
        g.nij = (long long)g.ni * g.nj;
        g.nc = g.nij * g.nk;
        g.ntiles = 2;
        g.nd = (g.ni + SKMAX + S - 1) / S * S;
        bj = for_j ? (DIR > 0 ? 1 : 0) : 0;
        bk = for_j ? 0 : (DIR > 0 ? 1 : 0);
        const int pt = DIR > 0 ? 0 : 1;
        range[pt] = make_int2(20 + (int)(rng() % 20), 100 + (int)(rng() % 40));
        range[1 - pt] = make_int2(1 + (int)(rng() % 60), 80 + (int)(rng() % 60));
        const int2 rg = range[1 - pt];
        const int sa = rg.x / S, sb = (rg.y + SKMAX) / S;
        nst = sb - sa + 1;
        s0 = DIR > 0 ? sa : sb;

        const size_t kn = (size_t)2 * (g.nd + 2 * KPAD) * TJ, jn = (size_t)2 * NW * (g.nd + 2 * JPAD) * TKW;
        box.assign(kn + jn, entry_of(-1.0, SEQ - 2));
        old.assign(kn + jn, entry_of(-2.0, SEQ - 2));
        arrival.assign(kn + jn, 0);
        c = WCtl{};
        c.range = range;
        c.mb = box.data();
        c.mb_bytes = (unsigned)((kn + jn) * 16);
        c.j_base = (unsigned)(kn * 16);
        c.seq = SEQ;
        c.err = &err;
        err = 0;

        // the producer's stores, a stage after the other, some time apart: its
        // diagonal d is the consumer's d - (TJ - 1) DIR (J), d - KOFF DIR (K)
        const int2 pr = range[pt];
        const int lo = pr.x / S * S, hi = (pr.y + SKMAX) / S * S + S - 1;
        auto value = [&](int w, int d, int line) { return 1.0 + line + 100.0 * w + 1000.0 * (d + 64); };
        int when = 1;
        for (int d = DIR > 0 ? lo : hi; d >= lo && d <= hi; d += DIR) {
            if ((d & 7) == (DIR > 0 ? 0 : 7)) when += (int)(rng() % 40);
            for (int w = 0; w < (for_j ? NW : 1); w++)
                for (int line = 0; line < (for_j ? TKW : TJ); line++) {
                    const size_t e = for_j ? kn + ((size_t)(pt * NW + w) * (g.nd + 2 * JPAD) + JPAD + d - (TJ - 1) * DIR) * TKW + line
                                           : ((size_t)pt * (g.nd + 2 * KPAD) + KPAD + d - KOFF * DIR) * TJ + line;
                    box[e] = entry_of(value(w, d, line), SEQ);
                    arrival[e] = when + (int)(rng() % 4);
                }
        }

        std::memset((void *)&sm, 0, sizeof sm);
        const bool stuck = what == "stuck";
        bool bad = false;
        int walked[2] = {0, 0};
        auto walk = [&](int o) {
            const int m = walked[o], w = DIR > 0 ? o : NW - 1 - o;
            if (stuck || m >= nst || sm.in[o][for_j ? 1 : 0] <= m || rng() % 2) return;
            for (int e = 0; e < S; e++)
                for (int line = 0; line < (for_j ? TKW : TJ); line++) {
                    const int d = S * (s0 + DIR * m) + phys<DIR>(e) + (for_j ? TJ - 1 : KOFF) * DIR;
                    const double want = d >= lo && d <= hi ? value(for_j ? w : 0, d, line) : 0.0;
                    const int slot = (m & (RX - 1)) * PQ + (e >> 1);
                    const double got = for_j ? sm.jr[o][slot][line][e & 1]
                                             : *reinterpret_cast<const double *>(sm.kr + slot * SLOT + line * 16 + (e & 1) * 8);
                    if (got != want && !bad) {
                        std::printf("wave %d stage %d step %d line %d: %g, stored %g\n", o, m, e, line, got, want);
                        bad = true;
                    }
                }
            walked[o]++;
            for (int &d : sm.done[o]) d = walked[o];
        };
        emu::run(lane, [&] {
            now++;
            for (int o = 0; o < (for_j ? NW : 1); o++) walk(o);
        });
        if (stuck) {
            if (err == 0) {
                std::printf("the wait for ring space gave up without the error flag\n");
                return 1;
            }
            std::puts("ok");
            return 0;
        }
        // the lanes have returned; what they left in the ring is taken too
        for (int n = 0; n < 64 * (nst + 1); n++)
            for (int o = 0; o < (for_j ? NW : 1); o++) walk(o);
        if (bad) return 1;
        if (err != 0 || walked[0] != nst || (for_j && NW == 2 && walked[1] != nst)) {
            std::printf("error flag %d, stages %d and %d of %d\n", err, walked[0], walked[1], nst);
            return 1;
        }
        std::puts("ok");
        return 0;
    }
};
template <int DIR, int NW> WSmem<NW> Case<DIR, NW>::sm;
template <int DIR, int NW> WGeom Case<DIR, NW>::g;
template <int DIR, int NW> WCtl Case<DIR, NW>::c;
template <int DIR, int NW> int2 Case<DIR, NW>::range[4];
template <int DIR, int NW> int Case<DIR, NW>::err;
template <int DIR, int NW> int Case<DIR, NW>::bj;
template <int DIR, int NW> int Case<DIR, NW>::bk;
template <int DIR, int NW> int Case<DIR, NW>::s0;
template <int DIR, int NW> int Case<DIR, NW>::nst;
template <int DIR, int NW> bool Case<DIR, NW>::for_j;

}  // namespace

int main(int argc, char **argv)
{
    if (argc < 4) return 2;
    const std::string what = argv[1];
    const bool fwd = std::string(argv[2]) == "fwd";
    const int nw = std::atoi(argv[3]);
    const unsigned seed = argc > 4 ? (unsigned)std::atoi(argv[4]) : 1;
    if (nw == 1) return fwd ? Case<1, 1>::main(what, seed) : Case<-1, 1>::main(what, seed);
    return fwd ? Case<1, 2>::main(what, seed) : Case<-1, 2>::main(what, seed);
}
