// resident.hip -- k_resident: the steps of casim_dyad_step with the state on
// the chip.  A site's interior x-planes are dealt to G workgroups (slabs);
// every slab keeps its planes in registers over all K steps of the call, so
// HBM moves the state once per call instead of once per two steps, and a step
// costs no launch.
//
// A slab is one workgroup on one CU: up to nine waves hold one node column
// each lane (PL planes of three fields in registers), one more wave runs the
// channels.  A step is a row of phases between barriers: first the slab's two
// edge planes, so that the neighbours get them a step ahead of their use, then
// PH planes each; a phase's old planes are staged in LDS for the y- and
// z-neighbours while the phase before it is computed.  Edge planes and mouth
// values pass between the slabs of a site by agent-scope stores (3 us from
// store to load among 256 workgroups, ordinary stores with fences 20-30 us),
// published by one flag each.  The channel wave of every slab gates the whole
// site, so that only mouth values travel: it draws, waits for the mouths and
// gates between the barriers of the same phases.  Workgroups take their slab
// from a ticket in the order in which they start, so the slabs of a site run
// together and a waiting slab's partners have started or will start when
// earlier sites end.
//
// What bounds it: phases that do one thing at a time.  At 20 planes of doubles
// a step takes 8.8 us on every CU: 2420 vector instructions per SIMD (4.0 us)
// and 2300 LDS instructions per CU (3.8 us), which two waves per SIMD between
// barriers hardly overlap.  In FP32 40 planes take 12 us, 10 us of them vector
// issue.  Fewer planes per slab finish a step sooner, more planes carry more
// sites at once.
// Measured (81x81x5, us per step in calls of 2000 steps, 200 for 1024 and 4096
// sites; shorter calls share the load and write-out of the state among fewer
// steps; k_sweep2 with the channel kernels before):
//   sites   FP64 k_sweep2   FP64 here   FP32 k_sweep2   FP32 here
//       1        98             3.5           -             2.9
//       6        99             3.5           -             2.9
//      32       106             5.6           -             4.2
//    1024         -           139             -            96
//    4096       780           554           440           379
// At 4096 sites in FP64, when a step here took 572 us: two planes at a time
// 604; waves waiting for their neighbour waves by LDS counters in place of
// barriers 919 and more; two workgroups per CU with 128 registers each 765.
// In FP32 those two workgroups took 362 us against 392; they are not built,
// because a variant of that arrangement ended in an illegal memory access whose
// cause was not shown.
// A register spilled in a divergent block must not be read after the lanes meet
// again: this compiler places the store of such a spill in front of the mask
// that brings the other lanes back, which lose the value.  The channel wave's
// shared stores are therefore made by all lanes, the file is built without the
// hoisting of constants that caused most spills, and tests/test_code_objects.py
// reads the built code for it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "dyad_internal.hpp"
#include "site_stream.hpp"

namespace casim {
namespace {

constexpr int RES_PAR = 4;   // steps that the exchange buffers between the slabs of a site hold
constexpr int RES_CH = 128;  // channels per site, nodes in y (padded)

struct ResArgs {
    int K;        // steps of the call
    int G;        // slabs (workgroups) per site
    int groups;   // sites on the chip at once
    int units;    // groups * G workgroups
    int nw;       // waves that hold nodes; one more wave runs the channels
    unsigned long long *ticket;
    unsigned *mflag, *eflag;  // [units * 32] steps of which mouths / edge planes are out
    void *edge;               // T [units][RES_PAR][2][NG][PS]
    double *mouth;            // [groups][RES_PAR][RES_CH]
    int *err;                 // host-visible: set when a wait ran into its limit
    int *stop;                // the same for later launches, which leave at once
    long long limit;          // of a wait, in ticks of 10 ns
    // channels (see Channels; one ion)
    const int *off, *perm, *snode, *type;
    int *state;
    uint32_t *rng;
    const uint32_t *jump;
    const double *jsr, *totals, *kin;  // kin: [MAXT][NPAR + 1] rate parameters, conductance
    double *stats;
    uint8_t *trace;
    int trace_every, trace_bins, M, ca;
    // jSR pool (see Pools; one ion, no cytosol pool)
    int pool, jsr_const;
    double cq, Vjsr, Velem, nCQ, KCQ, tau;
    double *jions, *jnew, *IjSR, *jnsr;
    const double *nsr;
    // cytosol box (2D sites): exchanged fields 0 .. ne - 1, its accumulator
    int ne, nlink;
    double exD[3];
    const double *link_fac;
    double *acc;
    int carry;  // the accumulator holds the effluxes of earlier launches of this box step
};

// SRPool::Update and SRPool::Run (SRPool.cpp:55-89) of one site held in
// registers, the operations of pool_update_site and pool_advance_site.
struct SitePool {
    double jions, jnew, IjSR, jnsr;
    __device__ __forceinline__ void update(const ResArgs &r, double total, double nsr) {
#pragma clang fp contract(off)
        if (r.jsr_const) return;
        IjSR = total * r.Velem;
        jnsr = nsr;
        jions = jnew;
    }
    __device__ __forceinline__ void advance(const ResArgs &r, double dt) {
#pragma clang fp contract(off)
        if (r.jsr_const) return;
        double beta = 1;
        const double c = jions;
        beta += r.nCQ * r.KCQ * r.cq / ((r.KCQ + c) * (r.KCQ + c));
        const double Iref = 1 / r.tau * (jnsr - c);
        jnew = c + dt / beta * (Iref - IjSR / r.Vjsr);
    }
};

template <typename T>
__device__ __forceinline__ void xst(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T xld(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// every store of this wave has reached the point where all workgroups see it
__device__ __forceinline__ void stores_out() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// LDS of one workgroup.
template <typename T, int NG, int PL, int PH, int PS, bool FLAT>
struct ResLds {
    static constexpr int SP = PH > 2 ? PH : 2;  // planes per staging buffer
    T stage[2][SP][NG][PS];
    double pg[2][RES_CH], jv[RES_CH], jvp[2];  // state * conductance, jSR of the mouth entries; the pool's jSR
    double jn[36];                             // jump of the streams over a step (high and low 16 bits of each word)
    unsigned char map[PL][FLAT ? PS : RES_CH];  // mouth entry + 1 of each (slot, y) on z = 0, 0: none
    // accumulated effluxes: of the links to the y-rims per slot, half, side and
    // field, of those to the x-rims per field and lane
    double yacc[FLAT ? PL * 12 : 1], xacc[FLAT ? 3 * PS : 1];
    int abort;
    unsigned ready;  // steps of which the neighbours' edge planes are out
    int unit;
    unsigned base;   // steps that the slab had published before this launch
};

// Flags that a wave's lanes watch (null: none) and their target.
__device__ __forceinline__ bool flags_out(const unsigned *watch, unsigned target) {
    return !__ballot(watch && (int)(xld(watch) - target) < 0);
}
// Wait for them; false when the limit has passed, which only a missing partner
// workgroup could cause.
__device__ __forceinline__ bool wait_flags(const unsigned *watch, unsigned target, long long limit) {
    long long t0 = 0;
    for (unsigned n = 1; !flags_out(watch, target); ++n) {
        if ((n & 255u) == 0) {
            const long long t = wall_clock64();
            if (!t0) t0 = t;
            if (t - t0 > limit) return false;
        }
    }
    return true;
}

// ---------------------------------------------------------------------------
// waves of a workgroup for planes of PS nodes, and per SIMD
constexpr int res_waves(int PS) { return (PS + 63) / 64 + 1; }
// FLAT: 2D sites with four grid fields (the coupled cleft), two slabs to a
// workgroup: lanes 0 .. ny - 1 hold the columns y of the first, ny .. 2 ny - 1
// those of the second, which takes the place of z.  The two pass their edge
// rows to each other through the staging buffer of phase 0.  Lanes past the
// nodes add up the effluxes across the y-rims from the staged rows.
template <typename T, int PL, int PH, int PS, bool FLAT>
__global__ __launch_bounds__(64 * res_waves(PS), (res_waves(PS) + 3) / 4) void k_resident(const T *__restrict__ gin,
                                                                            T *__restrict__ gout,
                                                                            const T *__restrict__ fin,
                                                                            T *__restrict__ fout, const Params p,
                                                                            const ResArgs r, double dt_) {
    constexpr int DIM = FLAT ? 2 : 3, NG = FLAT ? 4 : 3, NF = 1, LY = FLAT ? 2 : 1, H = PL / 2;
    constexpr int NPH = 1 + (PL - 2 + PH - 1) / PH;  // phases (barriers) per step
    static_assert(NPH % 2 == 0, "the staging buffers alternate over the phases of a step");
    constexpr int EB = NPH > 2 ? 2 : 1;   // barrier before which the edge planes' stores are out
    constexpr int GL = NPH > 2 ? 2 : 1;   // last phase in which the channel wave may gate
    constexpr int RNG = NPH > 2 ? 3 : 0;  // phase in which it forms the next draws
    constexpr int DM = H - 1 < PL - 2 - H ? H - 1 : PL - 2 - H, DMAX = DM < 3 ? DM : 3;
    static_assert(H - 1 - DMAX >= (H - 1) / PH * PH + 1 - PH, "slot H - 1 - d is staged one phase before slot H at most");
    using Lds = ResLds<T, NG, PL, PH, PS, FLAT>;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    Lds &S = *reinterpret_cast<Lds *>(smem);
    T *faces = reinterpret_cast<T *>(smem + sizeof(Lds));  // [2 * ny][PLF]
    constexpr int PLF = PL | 1;
    typedef __attribute__((address_space(3))) T LdsT;

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (threadIdx.x == 0) {
        // units in the order in which workgroups start, so that the slabs of a
        // site run together whatever the dispatch order
        S.unit = (int)(atomicAdd(r.ticket, 1ull) % (unsigned long long)r.units);
        S.base = xld(r.mflag + (size_t)S.unit * 32);
        S.ready = S.base;
        S.abort = xld(r.stop);  // the slabs of a site may stand at different steps
    }
    __syncthreads();
    const int unit = __builtin_amdgcn_readfirstlane(S.unit);
    unsigned E = __builtin_amdgcn_readfirstlane(S.base);
    const int grp = unit / r.G, gi = unit - grp * r.G;
    const int N = p.nx - 2;
    const int base = N / r.G, extra = N - base * r.G;
    const int np = base + (gi < extra ? 1 : 0);               // planes of this slab
    const int x0 = 1 + gi * base + min(gi, extra);            // first of them
    const int x1 = x0 + np;
    const int npa = FLAT ? (np + 1) / 2 : np;  // of the first half
    const int d = PL - np;  // slots that repeat a plane (0 .. DMAX)
    const int P = p.ny * p.nz;
    const size_t fs = (size_t)p.S * p.NS;
    const T dt = (T)dt_;
    const bool pool = r.pool != 0;
    T *edge = reinterpret_cast<T *>(r.edge);
    constexpr size_t EST = (size_t)NG * PS;  // one edge plane
    auto edge_at = [&](int u, unsigned step, int side) {
        return edge + (((size_t)u * RES_PAR + (step & (RES_PAR - 1))) * 2 + side) * EST;
    };
    auto mouth_at = [&](unsigned step) { return r.mouth + ((size_t)grp * RES_PAR + (step & (RES_PAR - 1))) * RES_CH; };
    auto aborted = [&] { return __builtin_amdgcn_readfirstlane(*(volatile int *)&S.abort) != 0; };

    // slot i of a node wave holds plane x0 + i in the lower half and, counted
    // from the other end, x1 - PL + i in the upper half, so that the slab's
    // first and last planes sit in fixed slots; with d > 0 the d planes around
    // the middle sit in two slots
    if (wave < r.nw) {
        // ---- node waves ---------------------------------------------------
        const int q = threadIdx.x;
        const bool act = q < (FLAT ? 2 * P : P);
        const int z = FLAT ? q >= P : q % p.nz, y = FLAT ? q - z * P : q / p.nz;  // FLAT: z is the half
        const int yq = FLAT ? y : q, mi = FLAT ? q : y;  // index in a plane of the state, in the mouth map
        const bool mouths = FLAT ? act : z == 0 && act;
        const bool inner = act && y >= 1 && y <= p.ny - 2;
        const int zl = z == 0 ? 1 : -1, zr = z == p.nz - 1 ? -1 : 1;
        const bool face = !FLAT && act && (z == 0 || z == p.nz - 1);
        T *const fl = faces + ((z == 0 ? 0 : p.ny) + (act ? y : 0)) * PLF;  // this node's face values, one per slot
        const int fg = (z == 0 ? 0 : p.nFP) + (act ? y : 0);
        const T ihx2 = (T)p.ihx2, ihy2 = (T)p.ihy2, ihz2 = (T)p.ihz2;
        // this lane's slab: its first plane, the plane after its last, its doubled slots
        const int lx0 = FLAT && z ? x0 + npa : x0, lx1 = FLAT && !z ? x0 + npa : x1, ld = FLAT ? PL - (lx1 - lx0) : d;
        // effluxes across the y-rims: lane al takes half al & 1, side al >> 1 & 1 and
        // field (al >> 2) % 3 of every third plane of a phase
        const int al = FLAT && r.ne ? q - 2 * P : -1, asub = al / 12, af = al < 0 ? 0 : (al >> 2) % 3;
        const bool acc_lane = FLAT && al >= 0 && al < 36 && af < r.ne;
        const int arim = (al & 1) * P + (al >> 1 & 1 ? P - 1 : 0), ain = arim + (al >> 1 & 1 ? -1 : 1);
        // ... of slots i: the place in its phase, the plane, the accumulator of its side
        const int ah0 = al & 1 ? x0 + npa : x0, ah1 = al & 1 ? x1 : x0 + npa;
        auto acc_place = [&](int i) { return i == 0 ? 0 : i == PL - 1 ? 1 : (i - 1) % PH; };
        auto acc_plane = [&](int i) { return i < H ? ah0 + i : ah1 - PL + i; };
        auto acc_y = [&](int s) { return r.acc + ((size_t)af * p.S + s) * r.nlink + 2 * (P - 2) + (al >> 1 & 1) * N; };
        const double exd = FLAT ? (af == 0 ? r.exD[0] : af == 1 ? r.exD[1] : r.exD[2]) : 0.0;
        const double facx = FLAT && r.ne ? r.link_fac[0] : 0.0, facy = FLAT && r.ne ? r.link_fac[2 * (P - 2)] : 0.0;
        auto flux = [&](double v, double D, double fac, double u, double ur) {  // k_box_efflux
#pragma clang fp contract(off)
            return v + dt_ * (D * (fac * (u - ur)));
        };
        for (int s = grp; s < p.S; s += r.groups) {
            __syncthreads();  // the last site's tables are free
            if (aborted()) return;
            const T *gs = gin + (size_t)s * p.NS;
            const T *ffs = fin + (size_t)s * 2 * p.nFP;
            T R[PL][NG];
            {
                // opaque copies: the planes' offsets are formed here and at the
                // write-out, not kept in registers over the steps and sites
                int lo = lx0, hi = lx1 - PL, qo = yq, fo = fg;
                if constexpr (FLAT) asm volatile("" : "+v"(lo), "+v"(hi), "+v"(qo));
                else asm volatile("" : "+s"(lo), "+s"(hi), "+v"(qo), "+v"(fo));
#pragma unroll
                for (int i = 0; i < PL; ++i) {
                    const int x = i + (i < H ? lo : hi);
#pragma unroll
                    for (int g = 0; g < NG; ++g)
                        R[i][g] = act ? ld_off(gs + g * fs, (unsigned)((x * P + qo) * (int)sizeof(T))) : (T)0;
                    if (face) fl[i] = ffs[fo + x * p.ny];
                    if (mouths) S.map[i][mi] = 0;
                }
            }
            // planes next to the slab: the rim planes, or the neighbours' edge
            // planes, loaded anew each step
            T hl[NG], hr[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                hl[g] = act ? ld_off(gs + g * fs, (unsigned)(((lx0 - 1) * P + yq) * (int)sizeof(T))) : (T)0;
                hr[g] = act ? ld_off(gs + g * fs, (unsigned)((lx1 * P + yq) * (int)sizeof(T))) : (T)0;
            }
            if (FLAT && r.ne && !r.carry) {
                for (int i = q; i < PL * 12; i += r.nw * 64) S.yacc[i] = 0.0;
                for (int e = 0; e < 3; ++e)
                    if (q < PS) S.xacc[e * PS + q] = 0.0;
            }
            if (FLAT && r.carry) {  // every lane what it adds to, from where it is written out below
                if (acc_lane) {
                    const double *from = acc_y(s);
#pragma unroll 1
                    for (int i = 0; i < PL; ++i)
                        if (acc_place(i) % 3 == asub) S.yacc[i * 12 + al % 12] = from[acc_plane(i) - 1];
                }
                if (inner && (z ? gi == r.G - 1 : gi == 0))
#pragma unroll
                    for (int e = 0; e < 3; ++e)
                        if (e < r.ne) S.xacc[e * PS + q] = r.acc[((size_t)e * p.S + s) * r.nlink + z * (P - 2) + y - 1];
            }
            __syncthreads();  // map cleared: the channel wave enters the mouths
            __syncthreads();
            using Mask = std::conditional_t<(PL > 32), uint64_t, uint32_t>;
            Mask mask = 0;  // slots in which this node is a mouth
            if (mouths)
#pragma unroll
                for (int i = 0; i < PL; ++i)
                    if (S.map[i][mi]) mask |= (Mask)1 << i;
            if (mask) {
                double *mo = mouth_at(E);
#pragma unroll
                for (int i = 0; i < PL; ++i)
                    if (mask >> i & 1) xst(mo + S.map[i][mi] - 1, (double)R[i][0]);
            }

            T prev[NG], last[NG];
            using Nbr = RegNbr<T, NG>;
            // this node's column of a staging buffer.  Opaque, so that every access is
            // this pointer plus a constant: otherwise each of them (the buffers span
            // more than an offset field) keeps an address register over the steps.
            auto column = [&](int b) {
                LdsT *c = (LdsT *)&S.stage[b][0][0][q];
                asm volatile("" : "+v"(c));
                return c;
            };
            struct Beside {
                LdsT *yl, *yr, *zl, *zr;
            };
            auto beside = [&](LdsT *c) { return Beside{c - p.nz, c + p.nz, c + zl, c + zr}; };
            auto nbrs = [&](const Beside &b, int i) {  // plane i of the buffer
                Nbr n;
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    const int o = (i * NG + g) * PS;
                    n.v[0][g] = b.yl[o];
                    n.v[1][g] = b.yr[o];
                    if (!FLAT) n.v[2][g] = b.zl[o];
                    if (!FLAT) n.v[3][g] = b.zr[o];
                }
                // doubles issued here: left to itself the scheduler puts each pair of reads
                // next to its sum and waits for every pair in turn (4096 sites of 81x81x5:
                // 0.61 ms per step, 0.71 without, with phases of four planes; FP32 0.40, 0.39 without)
                if (sizeof(T) == 8) __builtin_amdgcn_sched_barrier(0);
                return n;
            };
            // slot i: one step
            auto update = [&](int i, const Nbr &nb, const T(&Cm)[NG], const T(&Cp)[NG], T &F, const T J0, T(&O)[NG]) {
                const T Fv[NF] = {F};
                const T J[1] = {J0};
                T Fo[NF] = {F};
                node_update<T, DIM, 1, 3, NG, NF, LY>(p, Cm, R[i], Cp, nb, z, face, Fv, J, dt, ihx2, ihy2, ihz2, O, Fo);
                F = Fo[0];
                // one plane at a time: without this the compiler gathers every
                // plane's neighbours at the head of a phase and spills
                if constexpr (FLAT) asm volatile("" : "+v"(O[0]), "+v"(O[1]), "+v"(O[2]), "+v"(O[NG - 1])::"memory");
                else asm volatile("" : "+v"(O[0]), "+v"(O[1]), "+v"(O[2])::"memory");
            };
            // the current of a mouth node: state * conductance as gated, times jSR - mouth
            auto current = [&](int i, int par) {
                const int e = S.map[i][mi] - 1;
                const double jvv = pool ? S.jvp[par] : S.jv[e];
                return (T)(S.pg[par][e] * (jvv - (double)R[i][0]));
            };
            // phase j's planes into its staging buffer; phase 0 has the edge planes
            auto stage = [&](int j) {
                if (!act) return;
                const int i0 = 1 + (j - 1) * PH, i1 = i0 + PH < PL - 1 ? i0 + PH : PL - 1;
                LdsT *c = column(j & 1);
#pragma unroll
                for (int i = 0; i < PH; ++i) {
                    const int l = j ? i0 + i : i ? PL - 1 : 0;
                    if (j ? l < i1 : i < 2)
#pragma unroll
                        for (int g = 0; g < NG; ++g) c[(i * NG + g) * PS] = R[l][g];
                }
            };
            auto ready = [&](unsigned t) {
                return (int)(__builtin_amdgcn_readfirstlane(*(volatile unsigned *)&S.ready) - t) >= 0;
            };
            auto halos = [&](int k1) {
                if (act && gi > 0 && !(FLAT && z)) {
                    const T *e = edge_at(unit - 1, E + k1, 1);
#pragma unroll
                    for (int g = 0; g < NG; ++g) hl[g] = xld(e + g * PS + yq);
                }
                if (act && gi < r.G - 1 && !(FLAT && !z)) {
                    const T *e = edge_at(unit + 1, E + k1, 0);
#pragma unroll
                    for (int g = 0; g < NG; ++g) hr[g] = xld(e + g * PS + yq);
                }
            };
            // the y-rims' effluxes of the planes staged for phase j
            auto effluxes = [&](int j) {
                const int i0 = 1 + (j - 1) * PH, i1 = i0 + PH < PL - 1 ? i0 + PH : PL - 1;
                const T *c = &S.stage[j & 1][0][af][0];
#pragma unroll
                for (int i = 0; i < PH; ++i) {
                    const int l = j ? i0 + i : i ? PL - 1 : 0;
                    if (!(j ? l < i1 : i < 2) || i % 3 != asub) continue;
                    double &v = S.yacc[l * 12 + al % 12];
                    v = flux(v, exd, facy, (double)c[i * NG * PS + ain], (double)c[i * NG * PS + arim]);
                }
            };
            stage(0);
            bool got = false;  // the next step's neighbour planes are under way
            for (int k = 0; k < r.K; ++k) {
                const int par = k & 1;
                double *mo = mouth_at(E + k + 1);
                if (k && r.G > 1 && !got) {
                    while (!ready(E + k) && !aborted()) __builtin_amdgcn_s_sleep(1);
                    halos(k);
                }
                got = false;
                stores_out();  // this step's mouth values
                lds_barrier();
                if (aborted()) return;
                stage(1);
                // phase 0: the edge planes, first so that the neighbours get them early
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    prev[g] = R[0][g];
                    last[g] = R[PL - 1][g];
                }
                if (FLAT && acc_lane) effluxes(0);
                if (FLAT && r.ne && inner) {
                    // across the x-rims
                    if (gi == 0 && !z)
#pragma unroll
                        for (int e = 0; e < 3; ++e)
                            if (e < r.ne) S.xacc[e * PS + q] = flux(S.xacc[e * PS + q], r.exD[e], facx, (double)R[0][e], (double)hl[e]);
                    if (gi == r.G - 1 && z)
#pragma unroll
                        for (int e = 0; e < 3; ++e)
                            if (e < r.ne)
                                S.xacc[e * PS + q] = flux(S.xacc[e * PS + q], r.exD[e], facx, (double)R[PL - 1][e], (double)hr[e]);
                }
                if (inner) {
                    T J0 = (T)0, J1 = (T)0;
                    const bool hot = (mask & ((Mask)1 | (Mask)1 << (PL - 1))) != 0;
                    if (hot) {
                        if (mask & 1u) J0 = current(0, par);
                        if (mask >> (PL - 1) & 1u) J1 = current(PL - 1, par);
                    }
                    T n0[NG], n1[NG], F0 = (T)0, F1 = (T)0;
                    if (face) {
                        F0 = fl[0];
                        F1 = fl[PL - 1];
                    }
                    const Beside bs = beside(column(0));
                    const Nbr b0 = nbrs(bs, 0), b1 = nbrs(bs, 1);
                    if constexpr (FLAT) {
                        // the halves' inner edges: the second's first row, the first's last one
                        const LdsT *o = column(0) + (z ? NG * PS - P : P);
                        T ml[NG], mr[NG];
#pragma unroll
                        for (int g = 0; g < NG; ++g) {
                            const T v = o[g * PS];
                            ml[g] = z ? v : hl[g];
                            mr[g] = z ? hr[g] : v;
                        }
                        update(0, b0, ml, R[1], F0, J0, n0);
                        update(PL - 1, b1, R[PL - 2], mr, F1, J1, n1);
                    } else {
                        update(0, b0, hl, R[1], F0, J0, n0);
                        update(PL - 1, b1, R[PL - 2], hr, F1, J1, n1);
                    }
                    if (face) {
                        fl[0] = F0;
                        fl[PL - 1] = F1;
                    }
#pragma unroll
                    for (int g = 0; g < NG; ++g) {
                        R[0][g] = n0[g];
                        R[PL - 1][g] = n1[g];
                    }
                    if (r.G > 1 && k + 1 < r.K) {
                        if constexpr (FLAT) {
                            T *e = edge_at(unit, E + k + 1, z) + y;
#pragma unroll
                            for (int g = 0; g < NG; ++g) xst(e + g * PS, z ? R[PL - 1][g] : R[0][g]);
                        } else {
                            T *e0 = edge_at(unit, E + k + 1, 0) + q, *e1 = edge_at(unit, E + k + 1, 1) + q;
#pragma unroll
                            for (int g = 0; g < NG; ++g) {
                                xst(e0 + g * PS, R[0][g]);
                                xst(e1 + g * PS, R[PL - 1][g]);
                            }
                        }
                    }
                    if (hot && k + 1 < r.K) {
                        if (mask & 1u) xst(mo + S.map[0][mi] - 1, (double)R[0][0]);
                        if (mask >> (PL - 1) & 1u) xst(mo + S.map[PL - 1][mi] - 1, (double)R[PL - 1][0]);
                    }
                }
                // the planes between them
#pragma unroll
                for (int j = 1; j < NPH; ++j) {
                    const int i0 = 1 + (j - 1) * PH, i1 = i0 + PH < PL - 1 ? i0 + PH : PL - 1;
                    if (j == EB) stores_out();
                    lds_barrier();
                    // with d > 0 the lower neighbour of slot H is slot H - 1 - d, whose old
                    // values this thread has staged for this phase or the one before
                    T keep[NG];
                    if (H >= i0 && H < i1 && (FLAT ? act : d != 0)) {
                        const int l = H - 1 - ld;  // FLAT: the halves may differ, and with ld == 0 it is prev
                        LdsT *lp = l >= i0 ? column(j & 1) + (l - i0) * NG * PS
                                           : column((j & 1) ^ 1) + (l == 0 ? 0 : l - (i0 - PH)) * NG * PS;
#pragma unroll
                        for (int g = 0; g < NG; ++g) keep[g] = lp[g * PS];
                    }
                    if (j == NPH - 1 && r.G > 1 && k + 1 < r.K && ready(E + k + 1)) {
                        halos(k + 1);
                        got = true;
                    }
                    // the next phase's planes go out while this one is computed
                    if (j + 1 < NPH || k + 1 < r.K) stage(j + 1 < NPH ? j + 1 : 0);
                    if (FLAT && acc_lane) effluxes(j);
                    if (inner) {
                        T J[PH], F[PH];
#pragma unroll
                        for (int i = 0; i < PH; ++i) J[i] = F[i] = (T)0;
                        if (face)
#pragma unroll
                            for (int i = i0; i < i1; ++i) F[i - i0] = fl[i];
                        const Mask pm = (((Mask)1 << (i1 - i0)) - 1u) << i0;
                        const bool hot = (mask & pm) != 0;
                        if (hot)
#pragma unroll
                            for (int i = i0; i < i1; ++i)
                                if (mask >> i & 1u) J[i - i0] = current(i, par);
                        const Beside bs = beside(column(j & 1));
                        Nbr nb = nbrs(bs, 0);
#pragma unroll
                        for (int i = i0; i < i1; ++i) {
                            Nbr nx = nb;
                            if (i + 1 < i1) nx = nbrs(bs, i + 1 - i0);  // under way while plane i is computed
                            T lo[NG], hi[NG], n[NG];
#pragma unroll
                            for (int g = 0; g < NG; ++g) {
                                lo[g] = i == H && (FLAT || d) ? keep[g] : prev[g];
                                hi[g] = i + 1 == PL - 1 ? last[g] : R[i + 1][g];
                            }
                            if (i == H - 1) {
#pragma unroll
                                for (int e = 1; e <= DMAX; ++e)
#pragma unroll
                                    for (int g = 0; g < NG; ++g) hi[g] = ld == e ? R[H + e][g] : hi[g];
                            }
                            update(i, nb, lo, hi, F[i - i0], J[i - i0], n);
#pragma unroll
                            for (int g = 0; g < NG; ++g) {
                                prev[g] = R[i][g];
                                R[i][g] = n[g];
                            }
                            nb = nx;
                        }
                        if (face)
#pragma unroll
                            for (int i = i0; i < i1; ++i) fl[i] = F[i - i0];
                        if (hot && k + 1 < r.K)
#pragma unroll
                            for (int i = i0; i < i1; ++i)
                                if (mask >> i & 1u) xst(mo + S.map[i][mi] - 1, (double)R[i][0]);
                    }
                }
            }
            // the slab's planes, rim nodes included (each plane in one slot)
            T *os = gout + (size_t)s * p.NS;
            T *ofs = fout + (size_t)s * 2 * p.nFP;
            if (FLAT && acc_lane) {
                double *to = acc_y(s);
#pragma unroll 1
                for (int i = 0; i < PL; ++i)
                    if (acc_place(i) % 3 == asub && (i < H || i >= H + PL - (ah1 - ah0)))
                        to[acc_plane(i) - 1] = S.yacc[i * 12 + al % 12];
            }
            if (FLAT && r.ne && inner && (z ? gi == r.G - 1 : gi == 0))
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    if (e < r.ne) r.acc[((size_t)e * p.S + s) * r.nlink + z * (P - 2) + y - 1] = S.xacc[e * PS + q];
            if (act) {
                int lo = lx0, hi = lx1 - PL, qo = yq, fo = fg;
                if constexpr (FLAT) asm volatile("" : "+v"(lo), "+v"(hi), "+v"(qo));
                else asm volatile("" : "+s"(lo), "+s"(hi), "+v"(qo), "+v"(fo));
#pragma unroll
                for (int i = 0; i < PL; ++i) {
                    if (i >= H && i < H + ld) continue;
                    const int x = i + (i < H ? lo : hi);
#pragma unroll
                    for (int g = 0; g < NG; ++g) st_off(os + g * fs, (unsigned)((x * P + qo) * (int)sizeof(T)), R[i][g]);
                    if (face) ofs[fo + x * p.ny] = fl[i];
                }
            }
            E += (unsigned)r.K;
        }
        return;
    }

    // ---- channel wave: gates the whole site (every slab does the same) and
    // watches the flags -----------------------------------------------------
    unsigned *mf = r.mflag + (size_t)unit * 32, *ef = r.eflag + (size_t)unit * 32;
    const unsigned *mwatch = lane < r.G ? r.mflag + (size_t)(grp * r.G + lane) * 32 : nullptr;
    const unsigned *ewatch = nullptr;
    if (lane == 0 && gi > 0) ewatch = ef - 32;
    if (lane == 1 && gi < r.G - 1) ewatch = ef + 32;
    for (int s = grp; s < p.S; s += r.groups) {
        __syncthreads();
        if (aborted()) return;
        const int off = r.off[s], n = r.off[s + 1] - off;
        const int *sn = r.snode + off;
        // this lane's channels, i = lane + 64 c
        int st[2], ent[2], pos_e[2], typ[2];
        double gch[2];
        float w[2][4];  // kopen0, ncaopen, kclose0, ncaclose
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int i = lane + 64 * c;
            st[c] = 0;
            ent[c] = 0;
            gch[c] = 0.0;
            pos_e[c] = typ[c] = 0;
            w[c][0] = w[c][1] = w[c][2] = w[c][3] = 0.f;
            if (i < n) {
                const int e = pos_e[c] = r.perm[off + i];
                typ[c] = r.type[off + i];
                st[c] = r.state[off + i];
                const double *q = r.kin + typ[c] * (NPAR + 1);
                gch[c] = q[NPAR];
                w[c][0] = (float)q[0];
                w[c][1] = (float)q[1];
                w[c][2] = (float)q[3];
                w[c][3] = (float)q[4];
                S.pg[0][e] = S.pg[1][e] = (double)st[c] * gch[c];
                if (!pool) S.jv[e] = r.jsr[i + (size_t)r.M * s];
                int l = e;  // the last entry on the node holds its mouth value
                while (l + 1 < n && sn[l + 1] == sn[l]) ++l;
                ent[c] = l;
            }
        }
        if (lane < 18) {
            const uint32_t a = r.jump[n * 18 + lane];
            S.jn[2 * lane] = (double)(a >> 16);
            S.jn[2 * lane + 1] = (double)(a & 0xffffu);
        }
        SitePool sp{};
        double nsr = 0.0, total0 = 0.0;
        if (pool) {
            sp = {r.jions[s], r.jnew[s], r.IjSR[s], r.jnsr[s]};
            nsr = r.nsr[s];
            total0 = r.totals[s];
            S.jvp[0] = sp.jnew;
        }
        __syncthreads();
        // entries of this slab's mouths
        const int elo = first_channel_at(sn, 0, n, x0 * P), ehi = first_channel_at(sn, 0, n, x1 * P);
        for (int e = elo + lane; e < ehi; e += 64) {
            if (e + 1 < n && sn[e + 1] == sn[e]) continue;  // the last channel on a node wins
            const int x = sn[e] / P, yy = (sn[e] - x * P) / p.nz;
            const int half = FLAT && x >= x0 + npa, h0 = half ? x0 + npa : x0, h1 = FLAT && !half ? x0 + npa : x1;
            const int lo = x - h0, hi = x - h1 + PL, at = half ? P + yy : yy;  // its slots
            if (lo < H) S.map[lo][at] = (unsigned char)(e + 1);
            if (hi >= H) S.map[hi][at] = (unsigned char)(e + 1);
        }
        // stream: per channel the state one step into its draw if no channel
        // toggles before it in the step, and the draw's first value
        double L6[2][6], u[2];
        auto lane_states = [&](const uint32_t(&S6)[6]) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if (c && 64 * c >= n) break;  // the first chunk holds the stream, also of a site without channels
                uint32_t o[6];
                const uint32_t *J = r.jump + (size_t)(lane + 64 * c) * 18;
                mrg::matvec(J, S6, o, mrg::C1, mrg::M1);
                mrg::matvec(J + 9, S6 + 3, o + 3, mrg::C2, mrg::M2);
                (void)mrg::step(o);
#pragma unroll
                for (int i = 0; i < 6; ++i) L6[c][i] = (double)o[i];
            }
        };
        // the site's state at the step's start
        auto site_state = [&](uint32_t(&S6)[6]) {
            uint32_t o[6];
#pragma unroll
            for (int i = 0; i < 6; ++i)
                o[i] = __builtin_amdgcn_readfirstlane((uint32_t)mod53(L6[0][i], i < 3 ? RM1 : RM2));
            step_back(o, S6);
        };
        auto draws = [&] {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if (64 * c >= n) break;
                u[c] = first53(L6[c]);
            }
        };
        {
            uint32_t S6[6];
#pragma unroll
            for (int i = 0; i < 6; ++i) S6[i] = r.rng[s * 6 + i];
            lane_states(S6);
        }
        draws();
        const double *stp = r.stats + (size_t)s * NSTAT;
        double q_steps = stp[ST_STEPS], q_n = stp[ST_NOPEN], q_amp = stp[ST_AMP], q_ttp = stp[ST_TTP],
               q_tte = stp[ST_TTE], q_q = stp[ST_Q];
        // steps until the next time-histogram bin, and that bin
        const long long m0 = (long long)q_steps + 1;  // a step's count + 1 selects its bin
        int bin_in = r.trace ? (int)(r.trace_every - m0 % r.trace_every) : 0;
        long long bin = r.trace ? m0 / r.trace_every + 1 : 0;
        __syncthreads();  // map complete
        bool ok = r.limit != 0 || r.G == 1;  // without a limit to wait, give up right away
        int pos = n;     // draws of the last step
        int stale = 0;   // 1: the other copy of pg misses the last step's toggles
        // streams and draws of the next step
        auto next_draws = [&] {
            if (pos == n) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    if (c && 64 * c >= n) break;
                    jump53(S.jn, L6[c]);
                }
            } else {
                uint32_t S6[6], o6[6];
                site_state(S6);
                const uint32_t *J = r.jump + (size_t)pos * 18;
                mrg::matvec(J, S6, o6, mrg::C1, mrg::M1);
                mrg::matvec(J + 9, S6 + 3, o6 + 3, mrg::C2, mrg::M2);
                lane_states(o6);
            }
            draws();
        };
        // gate the site on the step's mouth values (DyadChannels::RunMC)
        auto gate = [&](int k) {
            const int par = k & 1;
            const double *mo = mouth_at(E + k);
            double ca[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) ca[c] = lane + 64 * c < n ? xld(mo + ent[c]) : 0.0;
            if (pool) {
                // site total of the currents in channel order, SRPool::Update
                double acc = total0;  // the first step keeps the last update's total
                if (k > 0) {
                    acc = 0.0;
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const double J = (double)st[c] * (gch[c] * (sp.jnew - ca[c]));
                        unsigned long long m = __ballot(lane + 64 * c < n && !(J == 0.0));
                        while (m) {  // zero terms leave the sum as it is
                            const int l = __builtin_ctzll(m);
                            m &= m - 1;
                            acc += __shfl(J, l);
                        }
                    }
                }
                sp.update(r, acc, nsr);
            }
            // a cheap bound from above decides whether any channel can toggle:
            // the rates are ~1e-5 per step, so almost every step ends here
            bool may = false;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if (64 * c >= n) break;
                const float x = (float)((r.ca >= 0 ? ca[c] : 0.0) * 1e-3);
                const float lx = __builtin_amdgcn_logf(x);  // log2; x below the normal range is never passed over
                const float rate = (st[c] ? w[c][2] : w[c][0]) * __builtin_amdgcn_exp2f((st[c] ? w[c][3] : w[c][1]) * lx);
                const float ub = 1.02f * rate * (float)(1e-3 * dt_) + 1e-30f;
                may = may || (lane + 64 * c < n && (!((float)u[c] >= ub) || u[c] > 0.9999999 || !(x > 1e-30f)));
            }
            pos = n;
            bool toggled = false;
            if (__ballot(may)) {
                uint32_t S6[6];
                site_state(S6);
                pos = 0;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const int c0 = 64 * c;
                    if (c0 >= n) break;
                    const int i = lane + c0;
                    const double thr = i < n ? channel_rate(CASIM_MODEL_SHEEP_CANNELL, r.kin + typ[c] * (NPAR + 1), st[c],
                                                            r.ca >= 0 ? ca[c] : 0.0, 0.0) * dt_
                                             : -1.0;
                    const int end = n < c0 + 64 ? n : c0 + 64;
                    int first = c0;
                    while (first < end) {
                        const bool active = i < n && i >= first;
                        const double uu = active ? draw_at(r.jump, S6, pos + (i - first)) : 2.0;
                        const unsigned long long m = __ballot(active && uu < thr);
                        if (m == 0ull) {
                            pos += end - first;
                            break;
                        }
                        const int jl = __builtin_ctzll(m);
                        if (lane == jl) st[c] ^= 1;
                        toggled = true;
                        pos += (c0 + jl - first) + 2;
                        first = c0 + jl + 1;
                    }
                }
            }
            // the next step's conductances; the copy in use now follows a step later
            if (toggled || stale) {
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    if (lane + 64 * c < n) S.pg[par ^ 1][pos_e[c]] = (double)st[c] * gch[c];
                stale = toggled;
            }
            if (pool) {
                sp.advance(r, dt_);
                S.jvp[par ^ 1] = sp.jnew;
            }
            // release statistics
            q_steps += 1.0;
            if (toggled || k == 0) {
                double nn = 0.0;
#pragma unroll
                for (int c = 0; c < 2; ++c) nn += (double)__popcll(__ballot(lane + 64 * c < n && st[c] == 1));
                const double t = q_steps * dt_;
                if (nn != q_n) q_tte = t;
                if (nn > q_amp) {
                    q_amp = nn;
                    q_ttp = t;
                }
                q_n = nn;
            }
            q_q += q_n * dt_;
            if (r.trace && --bin_in == 0) {
                if (gi == 0 && lane == 0 && bin < r.trace_bins)
                    r.trace[(size_t)bin * p.S + s] = (uint8_t)(q_n < 254.0 ? q_n : 254.0);
                ++bin;
                bin_in = r.trace_every;
            }
        };
        for (int k = 0; k < r.K; ++k) {
            bool gated = false;
            bool out = k + 1 == r.K || r.G == 1;  // the neighbours' edge planes of the next step are out
            auto look = [&] {  // every lane stores: a branch on the lane here would make the loop's control flow per lane
                if (!out && flags_out(ewatch, E + k + 1)) {
                    out = true;
                    *(volatile unsigned *)&S.ready = E + k + 1;
                }
            };
#pragma unroll 1
            for (int j = 0; j < NPH; ++j) {
                lds_barrier();
                if (j == 0 && lane == 0) xst(mf, E + k + 1);  // the step's mouth values are out
                if (j == EB && k + 1 < r.K && r.G > 1 && lane == 0) xst(ef, E + k + 1);
                if (j == RNG && (RNG || k)) next_draws();
                if (j >= 1 && !gated && ok) {
                    gated = flags_out(mwatch, E + k + 1);
                    if (j >= EB) look();
                    if (!gated && j == GL) gated = ok = wait_flags(mwatch, E + k + 1, r.limit);
                    if (gated) gate(k);
                }
                if (j >= EB && ok) {
                    look();
                    if (!out && j == NPH - 1) {
                        ok = wait_flags(ewatch, E + k + 1, r.limit);
                        look();
                    }
                }
                if (j == NPH - 1 && !ok && lane == 0) {
                    *(volatile int *)&S.abort = 1;
                    xst(r.stop, 1);
                    __hip_atomic_store(r.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                }
            }
            if (!ok) return;  // the node waves leave at their next check
        }
        if (!RNG) next_draws();
        E += (unsigned)r.K;
        if (gi == 0) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
                if (lane + 64 * c < n) r.state[off + lane + 64 * c] = st[c];
            uint32_t S6[6];
            site_state(S6);
            if (lane == 0) {
#pragma unroll
                for (int i = 0; i < 6; ++i) r.rng[s * 6 + i] = S6[i];
                double *so = r.stats + (size_t)s * NSTAT;
                so[ST_STEPS] = q_steps;
                so[ST_NOPEN] = q_n;
                so[ST_AMP] = q_amp;
                so[ST_TTP] = q_ttp;
                so[ST_TTE] = q_tte;
                so[ST_Q] = q_q;
                if (pool) {
                    r.jions[s] = sp.jions;
                    r.jnew[s] = sp.jnew;
                    r.IjSR[s] = sp.IjSR;
                    r.jnsr[s] = sp.jnsr;
                }
            }
        }
    }
}

// ---- host -------------------------------------------------------------------

constexpr int RES_CUS = 256;  // CUs, one workgroup each (registers and LDS of a CU)

struct Form {
    int PL, PH, PS, flat;
    int f64;
    double us0, us1;  // measured: a step of the sites on the chip takes us0 + us1 * PL
    size_t lds;
    void (*launch)(CasimDyad *, double, const ResArgs &, size_t);
};

template <typename T, int PL, int PH, int PS, bool FLAT>
void launch_form(CasimDyad *d, double dt, const ResArgs &r, size_t lds) {
    auto *k = k_resident<T, PL, PH, PS, FLAT>;
    HIPCK(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k, dim3(r.units), dim3((r.nw + 1) * 64), lds, d->stream, (const T *)d->g[d->cur],
                       (T *)d->g[d->cur ^ 1], (const T *)d->f[d->cur], (T *)d->f[d->cur ^ 1], d->P, r, dt);
    HIPCK(hipGetLastError());
}
template <typename T, int PL, int PH, int PS, bool FLAT = false>
Form form(double us0, double us1) {
    return {PL,  PH,  PS, FLAT, sizeof(T) == 8, us0, us1, sizeof(ResLds<T, FLAT ? 4 : 3, PL, PH, PS, FLAT>),
            launch_form<T, PL, PH, PS, FLAT>};
}
const Form FORMS[] = {
    // six planes a phase, built for up to 408 nodes (4096 sites: 572 us per step when four took 599); four up to 440,
    // though LDS would hold six there.  G slabs of 20 planes take nx - 2 from 17 G to 20 G; the widths between (61 to
    // 67, 81 to 84) fall to 10 planes, which gain little over the sweeps in large batches.
    form<double, 20, 6, 408>(2.1, 0.343), form<double, 20, 4, 440>(2.1, 0.37), form<double, 10, 3, 440>(2.1, 0.37),
    form<double, 5, 3, 440>(2.1, 0.37),
    form<float, 40, 8, 440>(2.0, 0.25),  form<float, 20, 6, 440>(2.0, 0.25),  form<float, 10, 3, 440>(2.0, 0.25),
    form<float, 5, 3, 440>(2.0, 0.25),
    // three waves per SIMD, 168 registers (81x96x6, 100 steps, ms, the sweeps before: 32 sites 15.2 -> 1.1,
    // 200 sites 17.5 -> 7.1, FP32 2500 sites 41.6 -> 30.7; FP64 2500 sites 73.5, 79.8 here, so by the sweeps)
    form<double, 10, 3, 576>(0.6, 0.94), form<double, 5, 3, 576>(0.6, 0.94), form<float, 20, 6, 576>(3.7, 0.18),
    form<float, 10, 3, 576>(3.7, 0.18),  form<float, 5, 3, 576>(3.7, 0.18),
    // two slabs of 2D columns to a workgroup (201x201, 100 steps, ms, the sweeps before: 1 site 10.8 -> 0.53,
    // 200 sites 15.0 -> 4.0, 800 sites 24.0 -> 15.8, FP32 800 sites 16.5 -> 8.7; 20 planes of doubles would spill)
    form<double, 17, 3, 412, true>(1.0, 0.39), form<double, 10, 3, 412, true>(1.0, 0.39), form<float, 20, 6, 412, true>(2.0, 0.17),
};

}  // namespace

struct Resident {
    const Form *f = nullptr;
    ResArgs a{};
    double *kin = nullptr;
    size_t lds = 0;
    bool ready = false;
};

static void clear_flags(CasimDyad *d, const ResArgs &a) {
    const size_t flags = (size_t)a.units * 32 * sizeof(unsigned);
    HIPCK(hipMemsetAsync(a.mflag, 0, flags, d->stream));
    HIPCK(hipMemsetAsync(a.eflag, 0, flags, d->stream));
    HIPCK(hipMemsetAsync(a.ticket, 0, 2 * sizeof(*a.ticket), d->stream));
}

// What the kernel keeps between launches, made before the first of them: a call
// that stays with the sweeps allocates nothing.
static void resident_buffers(CasimDyad *d, Resident &res) {
    const bool flat = res.f->flat;
    ResArgs &a = res.a;
    const size_t flags = (size_t)a.units * 32 * sizeof(unsigned);
    HIPCK(hipMalloc(&a.mflag, flags));
    HIPCK(hipMalloc(&a.eflag, flags));
    HIPCK(hipMalloc(&a.ticket, 2 * sizeof(*a.ticket)));
    a.stop = (int *)(a.ticket + 1);
    HIPCK(hipMalloc(&a.edge, (size_t)a.units * RES_PAR * 2 * (flat ? 4 : 3) * res.f->PS * d->tsize));
    HIPCK(hipMalloc(&a.mouth, (size_t)a.groups * RES_PAR * RES_CH * sizeof(double)));
    HIPCK(hipHostMalloc((void **)&a.err, sizeof(int), hipHostMallocMapped));
    *a.err = 0;
    std::vector<double> kin((size_t)MAXT * (NPAR + 1));
    for (int t = 0; t < MAXT; ++t) {
        for (int q = 0; q < NPAR; ++q) kin[t * (NPAR + 1) + q] = d->Ch.par[t * NPAR + q];
        kin[t * (NPAR + 1) + NPAR] = d->Ch.g[t * MAXI];
    }
    HIPCK(hipMalloc(&res.kin, sizeof(double) * kin.size()));
    HIPCK(hipMemcpyAsync(res.kin, kin.data(), sizeof(double) * kin.size(), hipMemcpyHostToDevice, d->stream));
    HIPCK(hipStreamSynchronize(d->stream));  // kin is a local
    clear_flags(d, a);
    res.ready = true;
}

// The call pays for the load and the write-out of the state once, K steps share
// it.  Both sides in us per call, measured over 1 to 4096 sites and 1 to 100
// steps: here 25 + PL / 2 and K (us0 + us1 PL) per round of sites on the chip,
// the sweeps K (40 + 5.9e-6 per node), FP32 3.3e-6.  4096 sites in FP64 cross
// between 8 steps (7.1 ms here, 6.5) and 16 (11.9, 12.7), 701 sites between 2
// and 3, fewer than 128 sites never.
bool resident_ok(CasimDyad *d, int K) {
    const Params &p = d->P;
    auto pays = [&] {
        const Form &f = *d->res->f;
        const double rounds = (p.S + d->res->a.groups - 1) / d->res->a.groups;
        const double here = rounds * (25.0 + 0.5 * f.PL + K * (f.us0 + f.us1 * f.PL));
        return here <= K * (40.0 + (f.f64 ? 5.9e-6 : 3.3e-6) * (double)p.S * (double)p.NS);
    };
    const bool flat = p.dim == 2;
    if (!d->chan_small || (d->Q.on && d->Q.cyto) || d->steps_per_pass < 2 || !d->use_sweep || d->M >= RES_CH) return false;
    if (flat ? layout_id(p) != 2 || !box_links(d, nullptr) : d->box || layout_id(p) != 1 || p.nz < 2 || p.ny > RES_CH)
        return false;
    // a failed allocation leaves no plan behind, and the next call makes it anew
    auto buffers = [&] {
        if (d->res->ready) return true;
        try {
            resident_buffers(d, *d->res);
        } catch (...) {
            resident_free(d);
            d->res_tried = false;
            throw;
        }
        return true;
    };
    if (d->res_tried) return d->res != nullptr && pays() && buffers();
    d->res_tried = true;
    const int N = p.nx - 2, P = p.ny * p.nz;
    auto lds_of = [&](const Form &f) { return f.lds + (flat ? 0 : (size_t)(f.PL | 1) * 2 * p.ny * d->tsize); };
    const Form *best = nullptr;
    int bg = 0;
    double cost = 1e300;
    for (const Form &f : FORMS) {
        if (f.flat != flat || f.f64 != (d->precision == CASIM_FP64) || (flat ? 2 * P + 36 > 448 : P > f.PS)) continue;
        const int H = f.PL / 2, dmax = std::min(3, std::min(H - 1, f.PL - 2 - H));
        if (lds_of(f) > 160 * 1024) continue;
        for (int G = 1; G <= 16; ++G) {
            // planes of the fullest and the emptiest slab
            int hi = (N + G - 1) / G, lo = N / G;
            if (flat) hi = (hi + 1) / 2, lo = lo / 2;
            if (hi > f.PL || f.PL - lo > dmax || lo < H + 1) continue;
            const int groups = std::min(p.S, RES_CUS / G);
            const double c = (p.S + groups - 1) / groups * (f.us0 + f.us1 * f.PL);
            if (c < cost) cost = c, best = &f, bg = G;
        }
    }
    if (!best) return false;
    auto *res = new Resident();
    d->res = res;
    res->f = best;
    res->lds = lds_of(*best);
    ResArgs &a = res->a;
    a.G = bg;
    a.groups = std::min(p.S, RES_CUS / bg);
    a.units = a.groups * bg;
    a.nw = ((flat ? 2 * P + 36 : P) + 63) / 64;
    return pays() && buffers();
}

// Steps of one launch, with a cytosol box too: at most 2048, and about half a
// second on the chip, far below the limit of a wait, since a slab whose partners
// found every CU taken by another handle's launch waits until that one ends.
int resident_most(const CasimDyad *d) {
    const Resident &r = *d->res;
    const double rounds = (d->P.S + r.a.groups - 1) / r.a.groups;
    return (int)std::min(2048.0, std::max(16.0, 5e5 / (rounds * (r.f->us0 + r.f->us1 * r.f->PL))));
}

void resident_steps(CasimDyad *d, double dt, int k, bool carry) {
    ResArgs a = d->res->a;
    a.carry = carry;
    a.limit = (long long)(d->wait_limit * 1e8);
    const Channels &c = d->Ch;
    const Pools &q = d->Q;
    a.K = k;
    a.off = c.off, a.perm = c.perm, a.snode = c.snode, a.type = c.type, a.state = c.state;
    a.rng = c.rng, a.jump = c.jump, a.jsr = c.jsr, a.totals = c.totals, a.stats = c.stats;
    a.kin = d->res->kin;
    a.trace = c.trace, a.trace_every = c.trace_every, a.trace_bins = c.trace_bins, a.M = c.M, a.ca = c.ca;
    a.pool = q.on, a.jsr_const = q.jsr_const;
    a.cq = q.cq, a.Vjsr = q.Vjsr, a.Velem = q.Velem, a.nCQ = q.nCQ[0], a.KCQ = q.KCQ[0], a.tau = q.tau[0];
    a.jions = q.jions, a.jnew = q.jnew, a.IjSR = q.IjSR, a.jnsr = q.jnsr, a.nsr = q.nsr;
    BoxLinks b{};
    if (d->box) (void)box_links(d, &b);
    a.ne = b.ne, a.nlink = b.nlink, a.link_fac = b.fac, a.acc = b.acc;
    for (int e = 0; e < 3; ++e) a.exD[e] = b.D[e];
    d->res->f->launch(d, dt, a, d->res->lds);
    d->cur ^= 1;
}

void resident_check(const CasimDyad *d) {
    if (d->res && d->res->ready && *(volatile int *)d->res->a.err)
        throw Err(CASIM_E_DEVICE,
                  "a step kernel gave up waiting for a workgroup of its site; the state is invalid (casim_dyad_reset)");
}

void resident_reset(CasimDyad *d) {
    if (!d->res || !d->res->ready || !*(volatile int *)d->res->a.err) return;
    clear_flags(d, d->res->a);
    HIPCK(hipStreamSynchronize(d->stream));
    *(volatile int *)d->res->a.err = 0;
}

void resident_free(CasimDyad *d) {
    if (!d->res) return;
    ResArgs &a = d->res->a;
    for (void *q : {(void *)d->res->kin, (void *)a.mflag, (void *)a.eflag, (void *)a.ticket, a.edge, (void *)a.mouth})
        if (q) (void)hipFree(q);
    if (a.err) (void)hipHostFree(a.err);
    delete d->res;
    d->res = nullptr;
}

}  // namespace casim
