// resident2d.hip -- k_site2d: the steps of casim_dyad_step for 2D sites that
// fit one CU, one workgroup per site with the state in LDS over all K steps.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "dyad_internal.hpp"
#include "dyad_kernels.hpp"
#include "site_stream.hpp"

namespace casim {
namespace {

constexpr int S2_CH = 128;            // channels per site (padded)
constexpr int S2_KIN = NPAR + MAXI + 1;  // a type's parameters, conductances, model
constexpr int S2_THREADS = 1024;
constexpr size_t S2_LDS = 156 * 1024;

struct Site2DArgs {
    int K, nw;  // steps; waves that hold nodes (two each lane), two more run the channels and the compartments
    const int *off, *node, *perm, *snode, *type;
    int *state;
    uint32_t *rng;
    const uint32_t *jump;
    const double *jsr, *kin;
    double *totals, *stats;
    uint8_t *trace;
    int trace_every, trace_bins, M, ca, mg;
    double gm, sxm, sym;  // see k_efflux
    // compartments (Pools)
    int pool, jsr_const, cyto, nbc, nBc;
    double cq, Vjsr, Velem, nCQ[MAXI], KCQ[MAXI], tau[MAXI];
    double *jions, *jnew, *IjSR, *jnsr;
    const double *nsr;
    double *cions, *cbuf, *cfree, *cbb;
    int serca[MAXI];
    double jmax[MAXI], kup[MAXI], conet_i[MAXI], cbg[MAXI];
    const double *cb;  // [MAXCB][4] ckoff, ckon, conet_b, cinit
    const int *ci;     // [MAXCB][6] ion, buffer, efflux slot, rim slot (-1: none); then [MAXI][MAXCU] cbind
    const double *ctot;
};

template <int NI>
struct Site2DLds {
    double pg[2][NI][S2_CH], jv[NI][S2_CH], jvp[2][NI];  // as in k_resident, per ion
    double jn[36];
    double rim[MAXI + MAXB];  // rim value of each grid field
};

// y-neighbours of a node in an LDS plane per field; 2D has no z
template <typename T>
struct PlaneNbr {
    static constexpr bool regs = false;
    const T *L;  // the node in field 0
    int P;
    __device__ __forceinline__ T yl(int g) const { return L[g * P - 1]; }
    __device__ __forceinline__ T yr(int g) const { return L[g * P + 1]; }
    __device__ __forceinline__ T zl(int) const { return (T)0; }
    __device__ __forceinline__ T zr(int) const { return (T)0; }
};

// A step: between two barriers the node waves form the new values from the LDS
// planes, one wave gates the channels and advances the jSR, one forms the
// effluxes and advances the cytosol; then, after the barrier, the new values
// and the new rim are stored.  The operations are those of k_sweep
// (node_update), k_channels, k_efflux, pool_update_site, pool_advance_site and
// k_rim in their order, so the values are the same bits.
// What bounds it: the slowest of the three roles between the barriers (100 sites
// of 31 x 41 nodes with two ions and every compartment: 7.2 us per step, 9.1
// with the species layout read at run time, 6.6 without the grid update; four
// launches of 107 us together before).  A site's state does not leave the CU
// and there is no launch per step, so any number of steps and sites gains.
template <typename T, int NI, int NB, int LY, int NT>
__global__ __launch_bounds__(NT) void k_site2d(const T *__restrict__ gin, T *__restrict__ gout, const Params p,
                                                       const Site2DArgs a, double dt_) {
    constexpr int NG = NI + NB, SL = 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    Site2DLds<NI> &S = *reinterpret_cast<Site2DLds<NI> *>(smem);
    T *const U = reinterpret_cast<T *>(smem + sizeof(Site2DLds<NI>));  // [NG][P]
    const int s = blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nx = p.nx, ny = p.ny, P = p.NS, S1 = p.S;
    const size_t fs = (size_t)S1 * P;
    const T *gs = gin + (size_t)s * P;
    const int off = a.off[s], n = a.off[s + 1] - off;
    const int *sn = a.snode + off;
    const bool pool = a.pool != 0, cyto = a.cyto != 0;
    for (int i = threadIdx.x; i < P; i += blockDim.x)
#pragma unroll
        for (int g = 0; g < NG; ++g) U[g * P + i] = gs[g * fs + i];

    if (wave < a.nw) {
        // ---- node waves ----
        const int nin = (nx - 2) * (ny - 2), nt = a.nw * 64;
        const T ihx2 = (T)p.ihx2, ihy2 = (T)p.ihy2, dt = (T)dt_;
        int c[SL], me[SL];  // node, mouth entry or -1
#pragma unroll
        for (int k = 0; k < SL; ++k) {
            const int i = threadIdx.x + k * nt;
            c[k] = -1;
            me[k] = -1;
            if (i < nin) {
                const int x = i / (ny - 2);
                c[k] = (x + 1) * ny + 1 + i - x * (ny - 2);
                const int e = first_channel_at(sn, 0, n, c[k] + 1) - 1;  // the last channel on a node wins
                if (e >= 0 && sn[e] == c[k]) me[k] = e;
            }
        }
        __syncthreads();  // state loaded, tables and rim set
        __syncthreads();
        for (int k = 0; k < a.K; ++k) {
            const int par = k & 1;
            T G[SL][NG];
#pragma unroll
            for (int q = 0; q < SL; ++q) {
                if (c[q] < 0) continue;
                const T *L = U + c[q];
                T Cm[NG], C0[NG], Cp[NG], J[NI], F[1] = {(T)0}, Fo[1];
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    Cm[g] = L[g * P - ny];
                    C0[g] = L[g * P];
                    Cp[g] = L[g * P + ny];
                }
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    J[j] = (T)0;
                    if (me[q] >= 0) {
                        const double jv = pool ? S.jvp[par][j] : S.jv[j][me[q]];
                        J[j] = (T)(S.pg[par][j][me[q]] * (jv - (double)C0[j]));
                    }
                }
                node_update<T, 2, NI, NB, NG, 1, LY>(p, Cm, C0, Cp, PlaneNbr<T>{L, P}, 0, false, F, J, dt, ihx2, ihy2, (T)0,
                                                    G[q], Fo);
            }
            lds_barrier();
#pragma unroll
            for (int q = 0; q < SL; ++q)
                if (c[q] >= 0)
#pragma unroll
                    for (int g = 0; g < NG; ++g) U[g * P + c[q]] = G[q][g];
            lds_barrier();
        }
    } else if (wave == a.nw) {
        // ---- channels and jSR, as in k_resident ----
        int st[2], nd[2], pos_e[2], typ[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int i = lane + 64 * c;
            st[c] = nd[c] = pos_e[c] = typ[c] = 0;
            if (i < n) {
                const int e = pos_e[c] = a.perm[off + i];
                typ[c] = a.type[off + i];
                st[c] = a.state[off + i];
                nd[c] = a.node[off + i];
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    S.pg[0][j][e] = S.pg[1][j][e] = (double)st[c] * a.kin[typ[c] * S2_KIN + NPAR + j];
                    if (!pool) S.jv[j][e] = a.jsr[i + (size_t)a.M * (s + (size_t)j * S1)];
                }
            }
        }
        if (lane < 18) {
            const uint32_t v = a.jump[n * 18 + lane];
            S.jn[2 * lane] = (double)(v >> 16);
            S.jn[2 * lane + 1] = (double)(v & 0xffffu);
        }
        double jions[NI], jnew[NI], IjSR[NI], jnsr[NI], nsr[NI], tot[NI];
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            jions[j] = jnew[j] = IjSR[j] = jnsr[j] = nsr[j] = 0.0;
            tot[j] = a.totals[s + j * S1];
            if (pool) {
                jions[j] = a.jions[s + j * S1];
                jnew[j] = a.jnew[s + j * S1];
                IjSR[j] = a.IjSR[s + j * S1];
                jnsr[j] = a.jnsr[s + j * S1];
                nsr[j] = a.nsr[s + j * S1];
                S.jvp[0][j] = jnew[j];
            }
        }
        __syncthreads();
        double L6[2][6], u[2];
        auto lane_states = [&](const uint32_t(&S6)[6]) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if (c && 64 * c >= n) break;  // the first chunk holds the stream, also of a site without channels
                uint32_t o[6];
                const uint32_t *J = a.jump + (size_t)(lane + 64 * c) * 18;
                mrg::matvec(J, S6, o, mrg::C1, mrg::M1);
                mrg::matvec(J + 9, S6 + 3, o + 3, mrg::C2, mrg::M2);
                (void)mrg::step(o);
#pragma unroll
                for (int i = 0; i < 6; ++i) L6[c][i] = (double)o[i];
            }
        };
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
            for (int i = 0; i < 6; ++i) S6[i] = a.rng[s * 6 + i];
            lane_states(S6);
        }
        draws();
        const double *stp = a.stats + (size_t)s * NSTAT;
        double q_steps = stp[ST_STEPS], q_n = stp[ST_NOPEN], q_amp = stp[ST_AMP], q_ttp = stp[ST_TTP],
               q_tte = stp[ST_TTE], q_q = stp[ST_Q];
        const long long m0 = (long long)q_steps + 1;  // a step's count + 1 selects its time bin
        int bin_in = a.trace ? (int)(a.trace_every - m0 % a.trace_every) : 0;
        long long bin = a.trace ? m0 / a.trace_every + 1 : 0;
        int stale = 0;
        __syncthreads();
        for (int k = 0; k < a.K; ++k) {
            const int par = k & 1;
            double ion[2][NI];
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int j = 0; j < NI; ++j) ion[c][j] = (double)U[j * P + nd[c]];
            // totals of the currents in channel order; the first step keeps the
            // last update's, the first ion's is formed anew, the others add up
            if (k > 0 && (pool || NI > 1)) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    if (j == 0) tot[j] = 0.0;
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        if (64 * c >= n) break;
                        const int i = lane + 64 * c;
                        double J = 0.0;
                        if (i < n) {
                            const double jv = pool ? jnew[j] : S.jv[j][pos_e[c]];
                            J = (double)st[c] * (a.kin[typ[c] * S2_KIN + NPAR + j] * (jv - ion[c][j]));
                        }
                        unsigned long long m = __ballot(!(J == 0.0));
                        while (m) {  // zero terms leave the sum as it is
                            const int l = __builtin_ctzll(m);
                            m &= m - 1;
                            tot[j] += __shfl(J, l);
                        }
                    }
                }
            }
            if (pool && !a.jsr_const) {  // SRPool::Update, SRPool::Run (SRPool.cpp:55-89)
#pragma clang fp contract(off)
                double beta = 1;
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    IjSR[j] = tot[j] * a.Velem;
                    jnsr[j] = nsr[j];
                    jions[j] = jnew[j];
                    const double c = jions[j];
                    beta += a.nCQ[j] * a.KCQ[j] * a.cq / ((a.KCQ[j] + c) * (a.KCQ[j] + c));
                }
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const double c = jions[j];
                    const double Iref = 1 / a.tau[j] * (jnsr[j] - c);
                    jnew[j] = c + dt_ / beta * (Iref - IjSR[j] / a.Vjsr);
                }
            }
            // DyadChannels::RunMC: a channel can toggle only where its draw's first
            // value is below its threshold (the draw adds up to 2^-24, less 1 at 1)
            double thr[2];
            bool may = false;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                thr[c] = -1.0;
                if (64 * c >= n) break;
                if (lane + 64 * c < n) {
                    double ca = 0.0, mg = 0.0;
#pragma unroll
                    for (int j = 0; j < NI; ++j) {
                        if (j == a.ca) ca = ion[c][j];
                        if (j == a.mg) mg = ion[c][j];
                    }
                    const double *q = a.kin + typ[c] * S2_KIN;
                    thr[c] = channel_rate((int)q[S2_KIN - 1], q, st[c], ca, mg) * dt_;
                    may = may || !(u[c] >= thr[c]) || u[c] > 0.9999999;
                }
            }
            int pos = n;
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
                    const int end = n < c0 + 64 ? n : c0 + 64;
                    int first = c0;
                    while (first < end) {
                        const bool active = i < n && i >= first;
                        const double uu = active ? draw_at(a.jump, S6, pos + (i - first)) : 2.0;
                        const unsigned long long m = __ballot(active && uu < thr[c]);
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
                    if (lane + 64 * c < n)
#pragma unroll
                        for (int j = 0; j < NI; ++j)
                            S.pg[par ^ 1][j][pos_e[c]] = (double)st[c] * a.kin[typ[c] * S2_KIN + NPAR + j];
                stale = toggled;
            }
            if (pool)
#pragma unroll
                for (int j = 0; j < NI; ++j) S.jvp[par ^ 1][j] = jnew[j];
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
            if (a.trace && --bin_in == 0) {
                if (lane == 0 && bin < a.trace_bins) a.trace[(size_t)bin * S1 + s] = (uint8_t)(q_n < 254.0 ? q_n : 254.0);
                ++bin;
                bin_in = a.trace_every;
            }
            // streams and draws of the next step
            if (pos == n) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    if (c && 64 * c >= n) break;
                    jump53(S.jn, L6[c]);
                }
            } else {
                uint32_t S6[6], o6[6];
                site_state(S6);
                const uint32_t *J = a.jump + (size_t)pos * 18;
                mrg::matvec(J, S6, o6, mrg::C1, mrg::M1);
                mrg::matvec(J + 9, S6 + 3, o6 + 3, mrg::C2, mrg::M2);
                lane_states(o6);
            }
            draws();
            lds_barrier();
            lds_barrier();
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
            if (lane + 64 * c < n) a.state[off + lane + 64 * c] = st[c];
        uint32_t S6[6];
        site_state(S6);
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < 6; ++i) a.rng[s * 6 + i] = S6[i];
            double *so = a.stats + (size_t)s * NSTAT;
            so[ST_STEPS] = q_steps;
            so[ST_NOPEN] = q_n;
            so[ST_AMP] = q_amp;
            so[ST_TTP] = q_ttp;
            so[ST_TTE] = q_tte;
            so[ST_Q] = q_q;
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                a.totals[s + j * S1] = tot[j];
                if (pool) {
                    a.jions[s + j * S1] = jions[j];
                    a.jnew[s + j * S1] = jnew[j];
                    a.IjSR[s + j * S1] = IjSR[j];
                    a.jnsr[s + j * S1] = jnsr[j];
                }
            }
        }
    } else {
        // ---- effluxes, cytosol and rim: lane b holds bound field b of the
        // cytosol, lane u its buffer u's free concentration, every lane the ions
        const int b = lane < MAXCB ? lane : 0;
        const int *ci = a.ci + b * 6;
        const bool bound = cyto && lane < a.nBc;
        const int jb = ci[0], ub = ci[1], ke = ci[2], kr = ci[3];
        const double koff = a.cb[b * 4], kon = a.cb[b * 4 + 1], conet = a.cb[b * 4 + 2], cinit = a.cb[b * 4 + 3];
        const int *cbind = a.ci + MAXCB * 6;  // [MAXI][MAXCU]
        const bool buf = cyto && lane < a.nbc;
        int bj[NI];  // bound field of buffer `lane` and each ion
        double ctot = 0.0, cfree = 0.0, cb = 0.0, ions[NI];
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            bj[j] = buf ? cbind[j * MAXCU + lane] : -1;
            ions[j] = cyto ? a.cions[s + j * S1] : 0.0;
        }
        if (buf) {
            ctot = a.ctot[lane];
            cfree = a.cfree[s + lane * S1];
        }
        if (bound) cb = a.cbuf[s + lane * S1];
        auto rim_values = [&](double rb) {  // rb: rim value of lane's bound field, if it has one
            if (lane == 0)
#pragma unroll
                for (int j = 0; j < NI; ++j) S.rim[j] = ions[j];
            if (bound && kr >= 0 && kr < NB) S.rim[NI + kr] = rb;
        };
        auto rim_store = [&] {
            const int nr = 2 * ny + 2 * (nx - 2);
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const T v = (T)S.rim[g];
                for (int i = lane; i < nr; i += 64) {
                    int c = i;  // x = 0, then x = nx - 1, then the ends of the planes between
                    if (i >= ny) c = (nx - 1) * ny + i - ny;
                    if (i >= 2 * ny) {
                        const int r = i - 2 * ny;
                        c = (1 + (r >> 1)) * ny + (r & 1) * (ny - 1);
                    }
                    U[g * P + c] = v;
                }
            }
        };
        __syncthreads();  // the state is in LDS
        if (cyto) {
            rim_values(bound && kr >= 0 ? a.cbb[s + kr * S1] : 0.0);
            __builtin_amdgcn_wave_barrier();
            rim_store();
        }
        __syncthreads();
        for (int k = 0; k < a.K; ++k) {
            if (cyto) {
#pragma clang fp contract(off)
                // _GetGradients, k_efflux's terms, lanes and sum
                double eff[NG];  // ions, then bound fields
#pragma unroll
                for (int f = 0; f < NG; ++f) {
                    const double D = f < NI ? p.Dion[f] : p.Db[f < NI ? 0 : f - NI];
                    const T *uf = U + f * P;  // without face buffers bound field b is grid field NI + b
                    const double tx = D * a.gm * a.sxm, ty = D * a.gm * a.sym;
                    double acc = 0.0;
                    const int per_x = ny - 2;
                    for (int t = lane; t < 2 * per_x; t += 64) {
                        const int side = t >= per_x;
                        const int y = 1 + t - side * per_x, x = side ? nx - 1 : 0, d = side ? -ny : ny;
                        const T *q = uf + x * ny + y;
                        acc += tx * (2 * (double)q[d] - 1.5 * (double)q[0] - 0.5 * (double)q[2 * d]);
                    }
                    for (int t = lane; t < 2 * nx; t += 64) {
                        const int side = t >= nx;
                        const int x = t - side * nx, y = side ? ny - 1 : 0, d = side ? -1 : 1;
                        const T *q = uf + x * ny + y;
                        acc += ty * (2 * (double)q[d] - 1.5 * (double)q[0] - 0.5 * (double)q[2 * d]);
                    }
                    eff[f] = acc;
                }
#pragma unroll
                for (int o = 32; o > 0; o >>= 1)
#pragma unroll
                    for (int f = 0; f < NG; ++f) eff[f] += __shfl_down(eff[f], o, 64);
                double ef = 0.0;  // the efflux of lane's bound field
#pragma unroll
                for (int f = 0; f < NG; ++f) {
                    eff[f] = __shfl(eff[f], 0);
                    if (f >= NI && ke == f - NI) ef = eff[f];
                }
                // CytosolPool::RunRD (CytosolPool.cpp:217-268)
                double cj = 0.0;
#pragma unroll
                for (int j = 0; j < NI; ++j)
                    if (jb == j) cj = ions[j];
                const double R1 = koff * cb - kon * cj * __shfl(cfree, ub);
                double evo_b = -R1;
                if (ke >= 0) evo_b += ef;
                int ks = 0;
                double evo_i[NI];
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    double react = 0;
                    for (int v = 0; v < a.nbc; ++v) {
                        const int bb = cbind[j * MAXCU + v];
                        if (bb >= 0) react += __shfl(R1, bb);
                    }
                    evo_i[j] = react + eff[j];
                    if (a.serca[j]) {
                        const double c = ions[j];
                        const double ions2 = c * c;
                        const double K2 = a.kup[j] * a.kup[j];
                        double bg = a.cbg[0];  // indexed by the SERCA counter, as the reference
#pragma unroll
                        for (int q = 1; q < NI; ++q)
                            if (ks == q) bg = a.cbg[q];
                        const double b2 = bg * bg;
                        evo_i[j] -= a.jmax[j] * (ions2 / (ions2 + K2) - b2 / (b2 + K2));
                        ++ks;
                    }
                }
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const double c = ions[j];
                    evo_i[j] -= a.conet_i[j] * (c - a.cbg[j]);
                    ions[j] = c + evo_i[j] * dt_;
                }
                evo_b -= conet * (cb - cinit);
                cb = cb + evo_b * dt_;
                cfree = ctot;
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const double v = __shfl(cb, bj[j] >= 0 ? bj[j] : 0);
                    if (bj[j] >= 0) cfree -= v;
                }
                rim_values(cb);
            }
            lds_barrier();
            if (cyto) rim_store();
            lds_barrier();
        }
        if (cyto) {
            if (lane == 0)
#pragma unroll
                for (int j = 0; j < NI; ++j) a.cions[s + j * S1] = ions[j];
            if (buf) a.cfree[s + lane * S1] = cfree;
            if (bound) {
                a.cbuf[s + lane * S1] = cb;
                if (kr >= 0) a.cbb[s + kr * S1] = cb;
            }
        }
    }
    // every wave is past the last barrier: the state is complete
    T *os = gout + (size_t)s * P;
    for (int i = threadIdx.x; i < P; i += blockDim.x)
#pragma unroll
        for (int g = 0; g < NG; ++g) os[g * fs + i] = U[g * P + i];
}

template <typename T, int NI, int NB, int LY>
void launch(CasimDyad *d, double dt, const Site2DArgs &a, size_t lds) {
    // up to twelve waves leave 168 registers each, which the two-ion form uses
    auto *k = a.nw + 2 <= 12 ? k_site2d<T, NI, NB, LY, 768> : k_site2d<T, NI, NB, LY, S2_THREADS>;
    HIPCK(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k, dim3(d->P.S), dim3((a.nw + 2) * 64), lds, d->stream, (const T *)d->g[d->cur],
                       (T *)d->g[d->cur ^ 1], d->P, a, dt);
    HIPCK(hipGetLastError());
}

size_t lds_bytes(const CasimDyad *d) {
    const Params &p = d->P;
    return (p.ni == 1 ? sizeof(Site2DLds<1>) : sizeof(Site2DLds<2>)) + (size_t)p.n_grid * p.NS * d->tsize;
}

}  // namespace

struct Site2D {
    int pools = 0;  // made with pools attached
    double *kin = nullptr, *cb = nullptr, *ctot = nullptr;
    int *ci = nullptr;
};

bool site2d_ok(const CasimDyad *d) {
    const Params &p = d->P;
    if (p.dim != 2 || d->box || d->steps_per_pass < 2 || !d->use_sweep || d->M >= S2_CH || p.n_face) return false;
    if (!(layout_id(p) == 2 || (p.ni == 2 && p.nb == 4))) return false;
    return (p.nx - 2) * (p.ny - 2) <= (S2_THREADS / 64 - 2) * 128 && lds_bytes(d) <= S2_LDS;
}

void site2d_free(CasimDyad *d) {
    if (!d->s2d) return;
    for (void *q : {(void *)d->s2d->kin, (void *)d->s2d->cb, (void *)d->s2d->ctot, (void *)d->s2d->ci})
        if (q) (void)hipFree(q);
    delete d->s2d;
    d->s2d = nullptr;
}

namespace {

// Tables of the channels' kinetics and the cytosol's fields in device memory,
// where a lane can index them.
void site2d_plan(CasimDyad *d) {
    if (d->s2d && d->s2d->pools == d->Q.on) return;
    if (d->s2d) HIPCK(hipStreamSynchronize(d->stream));
    site2d_free(d);
    auto *r = d->s2d = new Site2D();
    r->pools = d->Q.on;
    std::vector<double> kin((size_t)MAXT * S2_KIN), cb((size_t)MAXCB * 4), ct(MAXCU);
    std::vector<int> ci((size_t)MAXCB * 6 + MAXI * MAXCU, -1);
    for (int t = 0; t < MAXT; ++t) {
        for (int q = 0; q < NPAR; ++q) kin[t * S2_KIN + q] = d->Ch.par[t * NPAR + q];
        for (int j = 0; j < MAXI; ++j) kin[t * S2_KIN + NPAR + j] = d->Ch.g[t * MAXI + j];
        kin[t * S2_KIN + S2_KIN - 1] = d->Ch.model[t];
    }
    const Pools &q = d->Q;
    for (int b = 0; b < MAXCB; ++b) ci[b * 6] = ci[b * 6 + 1] = 0;
    if (q.on && q.cyto) {
        int ke = 0, kr = 0;
        for (int j = 0; j < d->P.ni; ++j)
            for (int u = 0; u < q.nbc; ++u) {
                const int b = q.cbind[j * q.nbc + u];
                ci[MAXCB * 6 + j * MAXCU + u] = b;
                if (b < 0) continue;
                ci[b * 6] = j;
                ci[b * 6 + 1] = u;
                if (q.cb_dyad[b]) ci[b * 6 + 2] = ke++;
            }
        for (int b = 0; b < q.nBc; ++b) {
            if (q.cb_dyad[b]) ci[b * 6 + 3] = kr++;
            cb[b * 4] = q.ckoff[b], cb[b * 4 + 1] = q.ckon[b], cb[b * 4 + 2] = q.conet_b[b], cb[b * 4 + 3] = q.cinit[b];
        }
        for (int u = 0; u < q.nbc; ++u) ct[u] = q.ctot[u];
    }
    auto up = [&](auto *&dst, const auto &src) {
        HIPCK(hipMalloc(&dst, sizeof(src[0]) * src.size()));
        HIPCK(hipMemcpyAsync(dst, src.data(), sizeof(src[0]) * src.size(), hipMemcpyHostToDevice, d->stream));
    };
    try {
        up(r->kin, kin);
        up(r->cb, cb);
        up(r->ctot, ct);
        up(r->ci, ci);
        HIPCK(hipStreamSynchronize(d->stream));  // the sources are locals
    } catch (...) {  // no plan without its tables: the next call makes it anew
        site2d_free(d);
        throw;
    }
}

}  // namespace

void site2d_steps(CasimDyad *d, double dt, int k) {
    site2d_plan(d);
    const Channels &c = d->Ch;
    const Pools &q = d->Q;
    const Params &p = d->P;
    Site2DArgs a{};
    a.K = k;
    a.nw = ((p.nx - 2) * (p.ny - 2) + 127) / 128;
    a.off = c.off, a.node = c.node, a.perm = c.perm, a.snode = c.snode, a.type = c.type, a.state = c.state;
    a.rng = c.rng, a.jump = c.jump, a.jsr = c.jsr, a.totals = c.totals, a.stats = c.stats;
    a.kin = d->s2d->kin;
    a.trace = c.trace, a.trace_every = c.trace_every, a.trace_bins = c.trace_bins, a.M = c.M, a.ca = c.ca, a.mg = c.mg;
    a.gm = d->grad_mult, a.sxm = d->sxm, a.sym = d->sym;
    a.pool = q.on, a.jsr_const = q.jsr_const, a.cyto = q.on && q.cyto, a.nbc = q.nbc, a.nBc = q.nBc;
    a.cq = q.cq, a.Vjsr = q.Vjsr, a.Velem = q.Velem;
    for (int j = 0; j < MAXI; ++j) {
        a.nCQ[j] = q.nCQ[j], a.KCQ[j] = q.KCQ[j], a.tau[j] = q.tau[j];
        a.serca[j] = q.serca[j], a.jmax[j] = q.jmax[j], a.kup[j] = q.kup[j], a.conet_i[j] = q.conet_i[j], a.cbg[j] = q.cbg[j];
    }
    a.jions = q.jions, a.jnew = q.jnew, a.IjSR = q.IjSR, a.jnsr = q.jnsr, a.nsr = q.nsr;
    a.cions = q.cions, a.cbuf = q.cbuf, a.cfree = q.cfree, a.cbb = q.cbb;
    a.cb = d->s2d->cb, a.ci = d->s2d->ci, a.ctot = d->s2d->ctot;
    const size_t lds = lds_bytes(d);
    const bool f64 = d->precision == CASIM_FP64;
    if (layout_id(p) == 3) {
        f64 ? launch<double, 2, 4, 3>(d, dt, a, lds) : launch<float, 2, 4, 3>(d, dt, a, lds);
    } else if (p.ni == 1) {
        f64 ? launch<double, 1, 3, 2>(d, dt, a, lds) : launch<float, 1, 3, 2>(d, dt, a, lds);
    } else {
        f64 ? launch<double, 2, 4, 0>(d, dt, a, lds) : launch<float, 2, 4, 0>(d, dt, a, lds);
    }
    d->cur ^= 1;
}

}  // namespace casim
