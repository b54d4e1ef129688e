// Per-evaluation theta-only work and the final assembly.
//
//  k_prep      params -> coefficient table: couplings v_a, c_a = v_a K_a, amplitude
//              numerators K_a and every propagator-denominator coefficient, each with
//              its first and second derivatives over the block's free parameters
//              (forward-mode jets).  One wave per item; runs in microseconds.
//  k_finalize  per-workgroup partial sums -> NLL and gradient in the fit-parameter
//              layout [Re p, Im p, theta], following the assembly of the reference's
//              NLLFunction::forward/backward (src/Analysis.cu:1134-1261): phase-space
//              mean, N_eff log term, NaN/Inf -> 1e30 with zero gradient, Gaussian
//              constraints (src/Parameters.cu:769-806).
//  k_amplitudes / k_intensity   per-event amplitudes and intensities (diagnostics,
//              event generation).
#include "device.hpp"

namespace ctpwa {

// ---------------------------------------------------------------------------
// forward-mode jet over a block's NLOC = 8 local variables, spread over a wave: every lane
// carries the value and the derivatives of one component, lane i d/dx_i, or with second
// derivatives lane 8 i + k d/dx_i, d/dx_k and d2/dx_i dx_k.  An item is one chain of
// dependent operations, and one thread with all components issued them one after the other
// (149 amplitudes with second derivatives: 69 us, now 11 us).
// ---------------------------------------------------------------------------
static_assert(NLOC == 8, "one wave holds the 8 x 8 second derivatives");
template <bool H> struct DJ { double v, g, gk, h; };
template <> struct DJ<false> { double v, g; };
template <bool H> __device__ __forceinline__ int jet_i() { return H ? threadIdx.x >> 3 : threadIdx.x; }
template <bool H>
__device__ inline DJ<H> jc(double c) {
    if constexpr (H) return {c, 0.0, 0.0, 0.0};
    else return {c, 0.0};
}
template <bool H>
__device__ inline DJ<H> jv(double c, int i) {
    DJ<H> r = jc<H>(c);
    r.g = jet_i<H>() == i ? 1.0 : 0.0;
    if constexpr (H) r.gk = (int)(threadIdx.x & 7) == i ? 1.0 : 0.0;
    return r;
}
template <bool H>
__device__ inline DJ<H> jadd(const DJ<H>& a, const DJ<H>& b) {
    DJ<H> r;
    r.v = a.v + b.v;
    r.g = a.g + b.g;
    if constexpr (H) { r.gk = a.gk + b.gk; r.h = a.h + b.h; }
    return r;
}
template <bool H>
__device__ inline DJ<H> jscale(const DJ<H>& a, double c) {
    DJ<H> r;
    r.v = a.v * c;
    r.g = a.g * c;
    if constexpr (H) { r.gk = a.gk * c; r.h = a.h * c; }
    return r;
}
template <bool H>
__device__ inline DJ<H> jsub(const DJ<H>& a, const DJ<H>& b) { return jadd(a, jscale(b, -1.0)); }
template <bool H>
__device__ inline DJ<H> jmul(const DJ<H>& a, const DJ<H>& b) {
    DJ<H> r;
    r.v = a.v * b.v;
    r.g = a.g * b.v + a.v * b.g;
    if constexpr (H) {
        r.gk = a.gk * b.v + a.v * b.gk;
        r.h = a.h * b.v + a.v * b.h + a.g * b.gk + a.gk * b.g;
    }
    return r;
}
// f(a) given f, f', f''
template <bool H>
__device__ inline DJ<H> jfun(const DJ<H>& a, double f, double d1, double d2) {
    DJ<H> r;
    r.v = f;
    r.g = d1 * a.g;
    if constexpr (H) { r.gk = d1 * a.gk; r.h = d1 * a.h + d2 * a.g * a.gk; }
    return r;
}
template <bool H>
__device__ inline DJ<H> jinv(const DJ<H>& a) { double x = a.v; return jfun(a, 1.0 / x, -1.0 / (x * x), 2.0 / (x * x * x)); }
template <bool H>
__device__ inline DJ<H> jdiv(const DJ<H>& a, const DJ<H>& b) { return jmul(a, jinv(b)); }
template <bool H>
__device__ inline DJ<H> jsqrt(const DJ<H>& a) { double s = sqrt(a.v); return jfun(a, s, 0.5 / s, -0.25 / (s * a.v)); }
template <bool H>
__device__ inline DJ<H> jlog(const DJ<H>& a) { return jfun(a, log(a.v), 1.0 / a.v, -1.0 / (a.v * a.v)); }
template <bool H>
__device__ inline DJ<H> jpowi(const DJ<H>& a, int n) {
    if (n == 0) return jc<H>(1.0);
    if (n == 1) return a;
    double x = a.v, xn2 = 1.0;
    for (int i = 0; i < n - 2; ++i) xn2 *= x;
    double xn1 = xn2 * x, xn = xn1 * x;
    return jfun(a, xn, n * xn1, n * (n - 1.0) * xn2);
}
// N_L(z) with z = q0 d as a jet in q0
template <bool H>
__device__ inline DJ<H> jbfpoly(int L, const DJ<H>& q0, double d) {
    double c[7];
    int deg = 0;
    switch (L) {
    case 1: c[0] = 1; c[1] = 1; deg = 1; break;
    case 2: c[0] = 9; c[1] = 3; c[2] = 1; deg = 2; break;
    case 3: c[0] = 225; c[1] = 45; c[2] = 6; c[3] = 1; deg = 3; break;
    case 4: c[0] = 11025; c[1] = 1575; c[2] = 135; c[3] = 10; c[4] = 1; deg = 4; break;
    case 5: c[0] = 893025; c[1] = 99225; c[2] = 6300; c[3] = 315; c[4] = 15; c[5] = 1; deg = 5; break;
    case 6: c[0] = 540326025; c[1] = 6185025; c[2] = 363825; c[3] = 17325; c[4] = 630; c[5] = 21; c[6] = 1; deg = 6; break;
    default: return jc<H>(1.0);
    }
    DJ<H> z = jscale(q0, d);
    DJ<H> z2 = jmul(z, z);
    DJ<H> r = jc<H>(c[deg]);          // Horner in z^2
    for (int i = deg - 1; i >= 0; --i) r = jadd(jmul(r, z2), jc<H>(c[i]));
    return r;
}
// breakup momentum (src/AmpGen.cu:2733-2737) and computeQ0AD (include/ResModel.cuh:88-97)
template <bool H>
__device__ inline DJ<H> jbreakup(const DJ<H>& m, const DJ<H>& m1, const DJ<H>& m2) {
    DJ<H> s = jadd(m1, m2), d = jsub(m1, m2);
    DJ<H> mm = jmul(m, m);
    DJ<H> q2 = jmul(jsub(mm, jmul(s, s)), jsub(mm, jmul(d, d)));
    if (q2.v <= 0.0) return jc<H>(0.0);
    return jdiv(jsqrt(q2), jscale(m, 2.0));
}
template <bool H>
__device__ inline DJ<H> jq0ad(const DJ<H>& m0, const DJ<H>& m1, const DJ<H>& m2) {
    DJ<H> s = jadd(m1, m2), d = jsub(m1, m2);
    DJ<H> m0s = jmul(m0, m0);
    DJ<H> q2 = jdiv(jmul(jsub(m0s, jmul(s, s)), jsub(m0s, jmul(d, d))), jscale(m0s, 4.0));
    if (q2.v < 0.0) return jc<H>(0.0);
    return jsqrt(q2);
}

// a model table in the constant address space (nothing writes it while a kernel reads it)
#define CTAB(T) __attribute__((address_space(4))) T
__device__ inline int local_index(const CTAB(DBlock)& B, int slot) {
    for (int i = 0; i < B.nloc; ++i) if (B.vars[i] == slot) return i;
    return -1;
}
template <bool H>
__device__ inline DJ<H> res_param(const CTAB(DRes)& R, int p, const CTAB(DBlock)& B, const double* theta) {
    if (p >= R.np) return jc<H>(0.0);
    int s = R.slot[p];
    if (s < 0) return jc<H>(R.p[p]);
    return jv<H>(theta[s], local_index(B, s));
}
// mass used in q0 for a daughter: configured mass, else the mass parameter of the
// block's resonance that occupies it (src/AmpGen.cu:1664-1731)
template <bool H>
__device__ inline DJ<H> q0_dmass(double cfg, int ref, const CTAB(DBlock)& B, const CTAB(DRes)* res, const double* theta) {
    if (cfg > 0) return jc<H>(cfg);
    // a final-state particle configured with mass 0: the reference falls back to the
    // event mass here, which is 0 for a massless particle (up to rounding)
    if (ref >= 0) return jc<H>(0.0);
    int kk = -ref - 1;
    for (int r = 0; r < B.nres; ++r) {
        const CTAB(DRes)& R = res[B.res0 + r];
        if (R.node == kk && R.np > 0) return res_param<H>(R, 0, B, theta);
    }
    return jc<H>(1.0);   // unreachable: the host rejects event-dependent q0
}
// the wave's lanes hold the record's components side by side
template <bool H>
__device__ inline void store(double* t, const DJ<H>& x) {
    const int lane = threadIdx.x;
    if (lane == 0) t[0] = x.v;
    if (H ? (lane & 7) == 0 : lane < NLOC) t[1 + jet_i<H>()] = x.g;
    if constexpr (H) t[1 + NLOC + lane] = x.h;
}

template <bool H>
__device__ __forceinline__ void prep_body(const double* __restrict__ gparams, double* __restrict__ table, PrepArgs a) {
    using J = DJ<H>;
    // the model's tables are read with wave-uniform, dependent indices: scalar loads.  (Each
    // workgroup copying all tables to LDS first took 21 us at 149 amplitudes, this 11 us; 8 us
    // at 10 amplitudes either way, which is the launch and cold instruction and table reads.)
    const double* params = gparams;
    const CTAB(DBlock)* blocks = (const CTAB(DBlock)*)a.blocks;
    const CTAB(DRes)* res = (const CTAB(DRes)*)a.res;
    const CTAB(DNode)* nodes = (const CTAB(DNode)*)a.nodes;
    const CTAB(DTopo)* topos = (const CTAB(DTopo)*)a.topos;
    const CTAB(DDen)* dens = (const CTAB(DDen)*)a.dens;
    const CTAB(DAmp)* amps = (const CTAB(DAmp)*)a.amps;
    const CTAB(int)* slcL = (const CTAB(int)*)a.slcL;
    const CTAB(int)* slc0 = (const CTAB(int)*)a.slc0;
    // one item (denominator or amplitude record) per workgroup: the items' chains of
    // dependent jet arithmetic then run on different compute units at the same time instead
    // of one after another in a single divergent wave
    int item = blockIdx.x;
    const double* __restrict__ theta = params + 2 * a.nfree;
    if (blockIdx.x == 0)
        for (int j = threadIdx.x; j < a.ntheta; j += blockDim.x) {
            table[a.off_th + j] = theta[j];
            if (a.remember) table[a.off_lth + j] = theta[j];
        }
    if (item < a.nden) {
        const CTAB(DDen)& D = dens[item];
        const CTAB(DBlock)& B = blocks[D.block];
        const CTAB(DRes)& R = res[B.res0 + D.res];
        const CTAB(DTopo)& T = topos[B.topo];
        const CTAB(DNode)& n = nodes[T.node0 + R.node];
        J m0 = (R.np > 0) ? res_param<H>(R, 0, B, theta) : jc<H>(1.0);
        J q0 = jq0ad(m0, q0_dmass<H>(n.md1, n.d1ref, B, res, theta), q0_dmass<H>(n.md2, n.d2ref, B, res, theta));
        double* t = table + a.off_rec + (long long)D.rec * REC;
        J m02 = jmul(m0, m0);
        switch (R.model) {
        case 0: {   // BWR: D = m0^2 - s - i g0 m0^2 N_L(q0 d')/q0^(2L+1) * E
            J g0 = res_param<H>(R, 1, B, theta);
            double dp = n.has_bf ? n.bf_d : 0.0;
            J N0 = (dp != 0.0) ? jbfpoly(n.lmin, q0, dp) : jc<H>(1.0);
            J b = jdiv(jmul(jmul(g0, m02), N0), jpowi(q0, 2 * n.lmin + 1));
            store(t, m02);
            store(t + REC, b);
            break;
        }
        case 1: {   // BW: D = m0^2 - s - i m0 g0
            J g0 = res_param<H>(R, 1, B, theta);
            store(t, m02);
            store(t + REC, jmul(m0, g0));
            break;
        }
        case 3: {   // Flatte: D = m0^2 - s + sum b_i rho_im,i - i sum b_i rho_re,i, b_i = m0 g_i / 2
            store(t, m02);
            for (int i = 0; i < R.nch; ++i) store(t + (1 + i) * REC, jscale(jmul(m0, res_param<H>(R, 1 + i, B, theta)), 0.5));
            break;
        }
        case 4: {   // Gounaris-Sakurai (src/ResModel.cu:484-561)
            const double pi = 3.14159265358979323846;
            J g0 = res_param<H>(R, 1, B, theta);
            double mpi = R.nch > 0 ? R.ch[0] : 0.1396;
            J q02 = jmul(q0, q0), q03 = jmul(q02, q0);
            J logA = jlog(jscale(jadd(m0, jscale(q0, 2.0)), 1.0 / (2.0 * mpi)));
            J h0 = jmul(jscale(jdiv(q0, m0), 2.0 / pi), logA);
            J dh0 = jadd(jmul(h0, jsub(jinv(jscale(q02, 8.0)), jinv(jscale(m02, 2.0)))), jinv(jscale(m02, 2.0 * pi)));
            J c1 = jdiv(jmul(g0, m02), q03);
            J c3 = jdiv(jmul(jmul(g0, m02), dh0), q0);
            J one_c3 = jadd(jc<H>(1.0), c3);
            store(t, jmul(one_c3, m02));
            store(t + REC, jscale(one_c3, -1.0));
            store(t + 2 * REC, c1);
            store(t + 3 * REC, jscale(jmul(c1, h0), -1.0));
            break;
        }
        default: break;
        }
        return;
    }
    item -= a.nden;
    if (item >= a.namp) return;
    const CTAB(DAmp)& A = amps[item];
    const CTAB(DBlock)& B = blocks[A.block];
    const CTAB(DTopo)& T = topos[B.topo];
    const CTAB(int)* Ls = slcL + (long long)(slc0[B.topo] + A.slc) * MAXNODE;
    J K = jc<H>(1.0);
    for (int k = 0; k < T.nn; ++k) {
        const CTAB(DNode)& n = nodes[T.node0 + k];
        int L = Ls[k];
        int r = -1;
        for (int i = 0; i < B.nres; ++i) if (res[B.res0 + i].node == k) { r = i; break; }
        J m1 = q0_dmass<H>(n.md1, n.d1ref, B, res, theta), m2 = q0_dmass<H>(n.md2, n.d2ref, B, res, theta);
        if (k == 0 || r < 0) {
            if (n.has_bf && L >= 1 && L <= 6) {
                J q0 = jbreakup(jc<H>(n.mm > 0 ? n.mm : 1.0), m1, m2);
                K = jmul(K, jsqrt(jbfpoly(L, q0, n.bf_d)));
            }
            continue;
        }
        const CTAB(DRes)& R = res[B.res0 + r];
        // BW, Custom and the table lineshapes (Hist, Interp) carry no automatic barrier
        if (R.model == 1 || R.model == 5 || R.model == 6 || R.model == 7) continue;
        J m0 = (R.np > 0) ? res_param<H>(R, 0, B, theta) : jc<H>(1.0);
        J q0 = jq0ad(m0, m1, m2);
        if (n.has_bf && L >= 1 && L <= 6) K = jmul(K, jsqrt(jbfpoly(L, q0, n.bf_d)));
        if (R.model == 4) {                                // GS numerator 1 + d(m0) g0 / m0
            const double pi = 3.14159265358979323846;
            J g0 = res_param<H>(R, 1, B, theta);
            double mpi = R.nch > 0 ? R.ch[0] : 0.1396;
            J q02 = jmul(q0, q0), q03 = jmul(q02, q0);
            J logA = jlog(jscale(jadd(m0, jscale(q0, 2.0)), 1.0 / (2.0 * mpi)));
            J dv = jadd(jsub(jmul(jscale(jdiv(jc<H>(mpi * mpi), q02), 3.0 / pi), logA), jmul(jc<H>(mpi * mpi / pi), jdiv(m0, q03))),
                         jdiv(m0, jscale(q0, 2.0 * pi)));
            K = jmul(K, jadd(jc<H>(1.0), jdiv(jmul(dv, g0), m0)));
        }
    }
    store(table + a.off_rec + (long long)A.rec * REC, K);
    if (threadIdx.x != 0) return;
    double pr = params[A.freeidx] * A.ratio, pi_ = params[a.nfree + A.freeidx] * A.ratio;
    table[a.off_v + 2 * item] = pr;
    table[a.off_v + 2 * item + 1] = pi_;
    table[a.off_c + 2 * item] = pr * K.v;
    table[a.off_c + 2 * item + 1] = pi_ * K.v;
}

template <bool H>
__global__ void __launch_bounds__(64) k_prep(const double* __restrict__ params, double* __restrict__ table, PrepArgs a) {
    prep_body<H>(params, table, a);
}

// many likelihoods that share a fused kernel: blockIdx.y selects the likelihood, its
// parameters, its coefficient table and its own handle's model tables (args: a kernel's
// source does not hold fixed masses and the like).  hdr (graph replays; NULL otherwise):
// hdr[0] is the number of jobs, rows at or beyond it leave at once.  The grid has as many
// items as the largest job.
__global__ void __launch_bounds__(64) k_prep_batch(const double* const* __restrict__ params, double* const* __restrict__ tables,
                                                   const PrepArgs* __restrict__ args, const int* __restrict__ hdr) {
    if (hdr && (int)blockIdx.y >= hdr[0]) return;
    PrepArgs a = args[blockIdx.y];
    a.remember = 1;                 // NLL evaluations: each table keeps its theta as the last evaluated one
    prep_body<false>(params[blockIdx.y], tables[blockIdx.y], a);
}

// ---------------------------------------------------------------------------
// final assembly
// ---------------------------------------------------------------------------

constexpr int ASM_THREADS = 1024;

// this lane's share of class c's total of accumulator column col: the class's
// workgroup partials in a fixed order, or, for the phase space with a stored Gram (no free
// resonance parameter), the column from G and c_a = v_a K_a:
//   col 0: sum_a Re(conj(c_a) (G c)_a) = sum_e I(e);  col 1 + 2a / 2 + 2a: Re / Im (G c)_a
// (sum_e conj(Psi_a sl_a) S, the fused kernel's accX_a); a butterfly over the wave follows, so
// the result depends neither on timing nor on the kernel that sums
__device__ __forceinline__ double class_share(const FinArgs& f, int c, int col) {
    const int lane = threadIdx.x & 63;
    if (c == 0 && f.gram) {
        double s = 0.0;
        const int n = f.namp;
        const double2* cv = (const double2*)(f.table + f.off_c);
        if (col == 0) {
            for (int a = lane; a < n; a += 64) {
                double gr = 0.0, gi = 0.0;
                for (int b = 0; b < n; ++b) {
                    const double2 G = f.gram[(long long)a * n + b], cb = cv[b];
                    gr += G.x * cb.x - G.y * cb.y;
                    gi += G.x * cb.y + G.y * cb.x;
                }
                const double2 ca = cv[a];
                s += ca.x * gr + ca.y * gi;
            }
        } else {
            const int a = (col - 1) >> 1, im = (col - 1) & 1;
            for (int b = lane; b < n; b += 64) {
                const double2 G = f.gram[(long long)a * n + b], cb = cv[b];
                s += im ? (G.x * cb.y + G.y * cb.x) : (G.x * cb.x - G.y * cb.y);
            }
        }
        return s;
    }
    // four loads in flight per lane
    const double* src = f.part + (long long)col * f.nwg;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int g = f.g0[c] + lane;
    for (; g + 192 < f.g1[c]; g += 256) {
        s0 += src[g];
        s1 += src[g + 64];
        s2 += src[g + 128];
        s3 += src[g + 192];
    }
    for (; g < f.g1[c]; g += 64) s0 += src[g];
    return (s0 + s1) + (s2 + s3);
}
// the wave's (class, column) pair of the totals, the sum in every lane
__device__ __forceinline__ double pair_total(const FinArgs& f, int pair) {
    const int c = pair / f.nacc, col = pair - c * f.nacc;
    double s = class_share(f, c, col);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s;
}

// NLL and gradient from the class totals.  Every global read happens first, in
// parallel over the threads: the gradient entries' weights (scale times their table
// coefficient), accumulator indices and row pointers (assemble_prefill, which needs no
// totals and so runs in k_finalize before a workgroup's reduction, off the last
// workgroup's path), then the class-combined accumulators.  The gradient rows are then
// fixed-order sums over LDS (one wave per theta with a butterfly sum), so no thread waits
// on a chain of dependent global loads.
// LDS layout: assemble_lds_bytes (device.hpp)
struct AsmLds {
    double *C, *wcp, *wth, *vre, *vim;
    int *icp, *ith, *cpp, *thp;
};
__device__ __forceinline__ AsmLds asm_lds(const FinArgs& f) {
    extern __shared__ double smem_asm[];
    AsmLds L;
    L.C = smem_asm;                          // [nacc] = -data + bkg + cp * phsp
    L.wcp = L.C + f.nacc;
    L.wth = L.wcp + f.ncpe;
    L.vre = L.wth + f.nthe;
    L.vim = L.vre + f.nthe;
    L.icp = (int*)(L.vim + f.nthe);
    L.ith = L.icp + f.ncpe;
    L.cpp = L.ith + f.nthe;
    L.thp = L.cpp + f.nfree + 1;
    return L;
}
__device__ __forceinline__ void assemble_prefill(const FinArgs& f) {
    const AsmLds L = asm_lds(f);
    const int tid = threadIdx.x;
    // coupling entries: weight r_a K_a, accumulator pair (1 + 2a, 2 + 2a)
    for (int k = tid; k < f.ncpe; k += ASM_THREADS) {
        DGEnt e = f.cpe[k];
        L.wcp[k] = e.scale * f.table[f.off_rec + e.rec];
        L.icp[k] = e.idx;
    }
    // theta entries: idx >= 0 -> w C[idx]; idx < 0 -> w (vr C[1 + 2a] + vi C[2 + 2a])
    for (int k = tid; k < f.nthe; k += ASM_THREADS) {
        DGEnt e = f.the[k];
        double d = (e.rec < 0) ? 1.0 : f.table[f.off_rec + e.rec];
        L.wth[k] = e.scale * d;
        L.ith[k] = e.idx;
        if (e.idx < 0) {
            int a = -e.idx - 1;
            L.vre[k] = f.table[f.off_v + 2 * a];
            L.vim[k] = f.table[f.off_v + 2 * a + 1];
        }
    }
    for (int k = tid; k <= f.nfree; k += ASM_THREADS) L.cpp[k] = f.cpp[k];
    for (int k = tid; k <= f.ntheta; k += ASM_THREADS) L.thp[k] = f.thp[k];
}
// the assembly proper, after assemble_prefill and a barrier; the totals come from other
// workgroups of this launch (coherent loads)
__device__ __forceinline__ void assemble_main(const FinArgs& f) {
    const AsmLds L = asm_lds(f);
    double* C = L.C;
    const double* wcp = L.wcp;
    const double* wth = L.wth;
    const double* vre = L.vre;
    const double* vim = L.vim;
    const int* icp = L.icp;
    const int* ith = L.ith;
    const int* cpp = L.cpp;
    const int* thp = L.thp;
    int tid = threadIdx.x;
    auto tot = [&](int i) {                  // i = c * nacc + col
        return __hip_atomic_load(f.totals + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    double Np = f.Np, Neff = f.Wd - f.Wb;
    double pf = (Np > 0) ? tot(0) / Np : 0.0;
    if (!(pf > 1e-30) || isinf(pf)) pf = 1e-30;
    double cp = (Np > 0) ? Neff / (pf * Np) : 0.0;
    const double* theta = f.params + 2 * f.nfree;
    for (int col = tid; col < f.nacc; col += ASM_THREADS)
        C[col] = -tot(f.nacc + col) + tot(2 * f.nacc + col) + cp * tot(col);
    double loss = -tot(f.nacc) + tot(2 * f.nacc) + Neff * log(pf);
    for (int g = 0; g < f.ngauss; ++g) {
        double d = theta[f.g_slot[g]] - f.g_mu[g];
        loss += d * d / (2.0 * f.g_sig[g] * f.g_sig[g]);
    }
    bool reset = isnan(loss) || isinf(loss);
    __syncthreads();
    double* out = f.out;
    if (tid == 0) out[0] = reset ? 1e30 : loss;
    // coupling gradient: dL/dp_f* = sum_a r_a K_a X_a, X_a = (C[1 + 2a], C[2 + 2a]);
    // output [2 Re, 2 Im]
    for (int fi = tid; fi < f.nfree; fi += ASM_THREADS) {
        double gr = 0.0, gi = 0.0;
        for (int k = cpp[fi]; k < cpp[fi + 1]; ++k) {
            double w = wcp[k];
            gr += w * C[1 + 2 * icp[k]];
            gi += w * C[2 + 2 * icp[k]];
        }
        out[1 + fi] = reset ? 0.0 : 2.0 * gr;
        out[1 + f.nfree + fi] = reset ? 0.0 : 2.0 * gi;
    }
    // theta gradient: propagator part -2 sum_t dcoef_t/dtheta_j C_t plus numerator part
    // 2 Re sum_a v_a dK_a/dtheta_j conj(X_a)
    const int lane = tid & 63, nw = ASM_THREADS / 64;
    for (int j = tid >> 6; j < f.ntheta; j += nw) {
        double g = 0.0;
        for (int k = thp[j] + lane; k < thp[j + 1]; k += 64) {
            int idx = ith[k];
            if (idx >= 0) {
                g += wth[k] * C[idx];
            } else {
                int a = -idx - 1;
                g += wth[k] * (vre[k] * C[1 + 2 * a] + vim[k] * C[2 + 2 * a]);
            }
        }
        for (int o = 32; o > 0; o >>= 1) g += __shfl_xor(g, o);
        if (lane == 0) {
            for (int q = 0; q < f.ngauss; ++q)
                if (f.g_slot[q] == j) g += (theta[j] - f.g_mu[q]) / (f.g_sig[q] * f.g_sig[q]);
            out[1 + 2 * f.nfree + j] = reset ? 0.0 : g;
        }
    }
}

// Reduction and assembly in one launch: every wave sums one (class, accumulator) over the
// class's workgroup partials, and the workgroup that finishes last, found by a device-scope
// counter, runs the assembly on the totals and resets the counter for the next evaluation.
// Bound by latency: cold reads of the partials and tables, and the handover.  Sixteen waves to
// a workgroup (one workgroup and one count per sum, each with the assembly's inputs, took
// 37 us at 149 amplitudes, 11 us at 10; now 12 and 9); the totals go through relaxed
// agent-scope stores and loads and a wait instead of agent-scope fences, which write back and
// invalidate the L2 cache.  That rests on this target and not on the language's memory model:
// agent-scope stores write through to where every compute unit's agent-scope loads look, and
// after s_waitcnt vmcnt(0) they have arrived, so they precede the wave's barrier and the count.
__device__ __forceinline__ void finalize_body(const FinArgs& f) {
    __shared__ int last;
    const int pair = blockIdx.x * (ASM_THREADS / 64) + (threadIdx.x >> 6);
    // the assembly's inputs that need no totals, loaded by every workgroup while its
    // reduction loads are in flight (any workgroup may turn out to be the last)
    assemble_prefill(f);
    if (pair < 3 * f.nacc) {
        const double tot = pair_total(f, pair);
        if ((threadIdx.x & 63) == 0) __hip_atomic_store(f.totals + pair, tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's total is visible before the count
    __syncthreads();
    if (threadIdx.x == 0) last = atomicAdd(f.done, 1u) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    assemble_main(f);
    if (threadIdx.x == 0) *f.done = 0u;
}
__global__ void __launch_bounds__(ASM_THREADS) k_finalize(FinArgs f) { finalize_body(f); }
// many likelihoods, one per blockIdx.y.  (Separate launches for the sums and the assemblies
// took 4.7 + 6.2 us for 24 likelihoods of 10 amplitudes, together 9.5 us.)

__global__ void __launch_bounds__(ASM_THREADS) k_finalize_batch(const FinArgs* __restrict__ fins, const int* __restrict__ hdr) {
    if (hdr && (int)blockIdx.y >= hdr[0]) return;
    finalize_body(fins[blockIdx.y]);
}

// ---------------------------------------------------------------------------
// generic per-event amplitudes and intensities
// ---------------------------------------------------------------------------

// The model's tables are the same for every event, and nothing writes them while these
// kernels run: reads through the constant address space become scalar loads, shared by the
// wave and free of the vector memory counter.  As vector loads, each of a block's five
// dependent table reads waited behind the kernel's own output stores.  With them, one pass
// over all polarisations instead of one each, and one-wave workgroups, the partial amplitudes
// of 1M events (11 waves, 120 MB read, 352 MB written) take 140 us instead of 197: 3.4 TB/s,
// bound by writing eleven streams to memory (half the events, which the last-level cache
// takes, 45 us).  Two or four events per thread, which walk the tables once, and nontemporal
// stores change nothing.
__device__ __forceinline__ int uni(const int* p) { return *(const __attribute__((address_space(4))) int*)(unsigned long long)p; }
__device__ __forceinline__ double uni(const double* p) { return *(const __attribute__((address_space(4))) double*)(unsigned long long)p; }

__device__ __forceinline__ double post_inv(const EvStore& s, int i, long long e) {
    if (s.mixed) {
        const int m = uni(s.imap + i);
        return (m >= 0) ? s.inv[(long long)m * s.ld + e] : (double)s.invf[(long long)(-m - 1) * s.ld + e];
    }
    return s.inv[(long long)i * s.ld + e];
}
__device__ __forceinline__ double2 post_sl(const EvStore& s, int u, int p, int npol, long long e) {
    if (p < s.nps) return ev_sl_row(s, (long long)u * s.nps + p, e);
    const double2 m = ev_sl_row(s, (long long)u * s.nps + (npol - 1 - p), e);
    const double g = (double)uni(s.psign + u);
    return make_double2(g * m.x, -g * m.y);
}

__device__ __forceinline__ double2 block_psi(const AuxArgs& a, int b, long long e) {
    const DBlock* B = a.blocks + b;
    double pr = 1.0, pi = 0.0;
    const int nden = uni(&B->nden), den0 = uni(&B->den0);
    for (int d = den0; d < den0 + nden; ++d) {
        const int rec = uni(&a.dens[d].rec);
        const DDenTerms* DT = a.dterms + d;
        const int nre = uni(&DT->nre), nt = nre + uni(&DT->nim), t0 = uni(&DT->t0);
        double dr = 0.0, di = 0.0;
        for (int t = 0; t < nt; ++t) {
            const DTerm* T = a.terms + t0 + t;
            const int coef = uni(&T->coef), inv = uni(&T->inv);
            const double c = (coef < 0) ? uni(&T->cval) : uni(a.table + a.off_rec + (long long)(rec + coef) * REC);
            const double x = (inv < 0) ? 1.0 : post_inv(a.st, inv, e);
            if (t < nre) dr += c * x; else di += c * x;
        }
        double xr = dr, xi = di;                          // table lineshape: the factor itself
        if (!uni(&DT->stat)) {
            const double q = 1.0 / (dr * dr + di * di);
            xr = dr * q;                                  // 1 / (dr - i di)
            xi = di * q;
        }
        double nr = pr * xr - pi * xi, ni = pr * xi + pi * xr;
        pr = nr; pi = ni;
    }
    // Custom lineshape factors (written for this parameter point by the Custom kernel)
    for (int q = uni(a.bcp + b); q < uni(a.bcp + b + 1); ++q) {
        const double* f = a.cfb + (long long)uni(a.bcl + q) * a.ncf * a.cld + e;
        const double fr = f[0], fi = f[a.cld];
        const double nr = pr * fr - pi * fi, ni = pr * fi + pi * fr;
        pr = nr; pi = ni;
    }
    return make_double2(pr, pi);
}

// polarisation arrays of a compile-time length stay in registers, their loops unrolled
template <int NP> struct PolArr { double r[NP], i[NP]; };

// w += P_b(e, p0 + p) of NP polarisations (those below npol)
template <int NP>
__device__ __forceinline__ void add_block(const AuxArgs& a, int b, long long e, int p0, int npol, PolArr<NP>& w) {
    const int nsl = uni(&a.blocks[b].nsl), site = uni(&a.blocks[b].site);
    if (nsl <= 0) return;
    const double2 psi = block_psi(a, b, e);
    PolArr<NP> y;
#pragma unroll
    for (int p = 0; p < NP; ++p) { y.r[p] = 0.0; y.i[p] = 0.0; }
    for (int am = site; am < site + nsl; ++am) {
        const double cr = uni(a.table + a.off_c + 2 * am), ci = uni(a.table + a.off_c + 2 * am + 1);
        const int u = uni(&a.amps[am].u);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            if (p0 + p >= npol) continue;
            const double2 s = post_sl(a.st, u, p0 + p, npol, e);
            y.r[p] += cr * s.x - ci * s.y;
            y.i[p] += cr * s.y + ci * s.x;
        }
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        w.r[p] += psi.x * y.r[p] - psi.y * y.i[p];
        w.i[p] += psi.x * y.i[p] + psi.y * y.r[p];
    }
}

// A[e][p][a] = K_a Psi_b(e) sl_u,p(e)  (interleaved complex), events [e0, e0 + n)
__global__ void __launch_bounds__(128) k_amplitudes(AuxArgs a, long long e0, long long n, double* __restrict__ out) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    long long e = e0 + i;
    int block = -1;
    double2 psi = make_double2(0.0, 0.0);
    for (int am = 0; am < a.namp; ++am) {
        const DAmp* A = a.amps + am;
        if (uni(&A->block) != block) {
            block = uni(&A->block);
            psi = block_psi(a, block, e);
        }
        const double K = uni(a.table + a.off_rec + (long long)uni(&A->rec) * REC);
        const int u = uni(&A->u);
        for (int p = 0; p < a.npol; ++p) {
            double2 s = post_sl(a.st, u, p, a.npol, e);
            double r = K * (psi.x * s.x - psi.y * s.y), im = K * (psi.x * s.y + psi.y * s.x);
            long long o = ((i * a.npol + p) * a.namp + am) * 2;
            out[o] = r;
            out[o + 1] = im;
        }
    }
}

// per-event partial-wave intensities: out[b][i] = sum_p |P_b(e, p)|^2 for the nblock
// partial waves (blocks) and out[nblock][i] = I(e) = sum_p |sum_b P_b|^2, with
// P_b = Psi_b sum_{a in b} c_a sl_u(a),p and c_a = v_a K_a (src/ComputeResults.cu:57-190)
// partial wave w = blocks wblk[wptr[w] .. wptr[w+1]) (a block and its identical-particle
// permuted copies): out[w][i] = sum_pol |sum over the wave's blocks P_b|^2,
// out[nwave][i] = the total intensity.
// MORE: more than NP polarisations, NP at a time, each sum carried on in out (in the order of
// one pass over all).  Arrays of any length instead, indexed by a loop variable, lie in
// scratch: six polarisations, 500k events, 10 amplitudes, 926 us, now 125.
template <int NP, bool MORE>
__global__ void __launch_bounds__(64) k_partial_int(AuxArgs a, const int* __restrict__ wptr, const int* __restrict__ wblk, int nwave,
                                                     long long e0, long long n, double* __restrict__ out) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long long e = e0 + i;
    const int npol = MORE ? a.npol : NP;
    double I = 0.0;
    for (int p0 = 0; p0 < npol; p0 += NP) {
        PolArr<NP> S, W;
#pragma unroll
        for (int p = 0; p < NP; ++p) { S.r[p] = 0.0; S.i[p] = 0.0; }
        for (int w = 0; w < nwave; ++w) {
#pragma unroll
            for (int p = 0; p < NP; ++p) { W.r[p] = 0.0; W.i[p] = 0.0; }
            for (int k = uni(wptr + w); k < uni(wptr + w + 1); ++k) add_block<NP>(a, uni(wblk + k), e, p0, npol, W);
            double v = MORE && p0 ? out[(long long)w * n + i] : 0.0;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                v += W.r[p] * W.r[p] + W.i[p] * W.i[p];
                S.r[p] += W.r[p];
                S.i[p] += W.i[p];
            }
            out[(long long)w * n + i] = v;
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) I += S.r[p] * S.r[p] + S.i[p] * S.i[p];
    }
    out[(long long)nwave * n + i] = I;
}

// coherent partial-wave amplitudes: out[w][i][p] = sum over the wave's blocks of P_b
// (couplings applied), interleaved complex, events [e0, e0 + n)
template <int NP, bool MORE>
__global__ void __launch_bounds__(64) k_partial_amp(AuxArgs a, const int* __restrict__ wptr, const int* __restrict__ wblk, int nwave,
                                                     long long e0, long long n, double2* __restrict__ out) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long long e = e0 + i;
    const int npol = MORE ? a.npol : NP;
    for (int w = 0; w < nwave; ++w)
        // (one wave's groups one after the other: they fill the same lines of out)
        for (int p0 = 0; p0 < npol; p0 += NP) {
            PolArr<NP> W;
#pragma unroll
            for (int p = 0; p < NP; ++p) { W.r[p] = 0.0; W.i[p] = 0.0; }
            for (int k = uni(wptr + w); k < uni(wptr + w + 1); ++k) add_block<NP>(a, uni(wblk + k), e, p0, npol, W);
#pragma unroll
            for (int p = 0; p < NP; ++p)
                if (p0 + p < npol) out[((long long)w * n + i) * npol + p0 + p] = make_double2(W.r[p], W.i[p]);
        }
}

template <int NP, bool MORE>
__global__ void __launch_bounds__(64) k_intensity(AuxArgs a, int nblock, long long e0, long long n, double* __restrict__ out) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int npol = MORE ? a.npol : NP;
    double I = 0.0;
    for (int p0 = 0; p0 < npol; p0 += NP) {
        PolArr<NP> S;
#pragma unroll
        for (int p = 0; p < NP; ++p) { S.r[p] = 0.0; S.i[p] = 0.0; }
        for (int b = 0; b < nblock; ++b) add_block<NP>(a, b, e0 + i, p0, npol, S);
#pragma unroll
        for (int p = 0; p < NP; ++p) I += S.r[p] * S.r[p] + S.i[p] * S.i[p];
    }
    out[i] = I;
}

}  // namespace ctpwa

template <bool H>
static hipError_t launch_prep_t(const double* params, double* table, const ctpwa::PrepArgs* a, int remember,
                                hipStream_t stream) {
    int items = a->nden + a->namp;
    ctpwa::PrepArgs b = *a;
    b.remember = remember;
    hipLaunchKernelGGL((ctpwa::k_prep<H>), dim3(items), dim3(64), 0, stream, params, table, b);
    return hipGetLastError();
}

// flags: bit 0 also second
// derivatives (Hessian), bit 1 theta is also stored as the last evaluated theta (the
// NLL and Hessian entry points; the per-event outputs leave it)
extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_prep(const double* params, double* table,
                                                                              const ctpwa::PrepArgs* a, int flags,
                                                                              hipStream_t stream) {
    const int hess = flags & 1, rem = (flags >> 1) & 1;
    return hess ? launch_prep_t<true>(params, table, a, rem, stream) : launch_prep_t<false>(params, table, a, rem, stream);
}

// args: the jobs' prep arguments on the device; items: the largest job's coefficient records;
// rows: workgroup rows launched (the job count, or with hdr a bound on the job count hdr[0] on
// the device, extra rows leave)
extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_prep_batch(const double* const* params,
                                                                                    double* const* tables,
                                                                                    const ctpwa::PrepArgs* args, int items,
                                                                                    int rows, const int* hdr,
                                                                                    hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(ctpwa::k_prep_batch, dim3(items, rows), dim3(64), 0, stream, params, tables, args, hdr);
    return hipGetLastError();
}

// fins: device array of the jobs' arguments; rows and hdr as above; max_nacc: the largest
// accumulator count among the jobs
extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_finalize_batch(const ctpwa::FinArgs* fins, int rows,
                                                                                        int max_nacc, size_t lds_bytes,
                                                                                        const int* hdr, hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(ctpwa::k_finalize_batch, dim3((3 * max_nacc + 15) / 16, rows), dim3(ctpwa::ASM_THREADS), lds_bytes, stream,
                       fins, hdr);
    return hipGetLastError();
}

extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_finalize(const ctpwa::FinArgs* f, hipStream_t stream) {
    hipLaunchKernelGGL(ctpwa::k_finalize, dim3((3 * f->nacc + 15) / 16), dim3(ctpwa::ASM_THREADS), ctpwa::assemble_lds_bytes(*f),
                       stream, *f);
    return hipGetLastError();
}

// the polarisation count at compile time up to four; more: four at a time
#define POST_LAUNCH(K, npol, n, ...)                                                                     \
    do {                                                                                                 \
        const dim3 g_((unsigned)((n + 63) / 64)), b_(64);                                                \
        switch (npol) {                                                                                  \
        case 1: hipLaunchKernelGGL((ctpwa::K<1, false>), g_, b_, 0, stream, __VA_ARGS__); break;         \
        case 2: hipLaunchKernelGGL((ctpwa::K<2, false>), g_, b_, 0, stream, __VA_ARGS__); break;         \
        case 3: hipLaunchKernelGGL((ctpwa::K<3, false>), g_, b_, 0, stream, __VA_ARGS__); break;         \
        case 4: hipLaunchKernelGGL((ctpwa::K<4, false>), g_, b_, 0, stream, __VA_ARGS__); break;         \
        default: hipLaunchKernelGGL((ctpwa::K<4, true>), g_, b_, 0, stream, __VA_ARGS__);                \
        }                                                                                                \
    } while (0)

extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_partial_int(const ctpwa::AuxArgs* a, const int* wptr,
                                                                                     const int* wblk, int nwave,
                                                                                     long long e0, long long n, double* out,
                                                                                     hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    POST_LAUNCH(k_partial_int, a->npol, n, *a, wptr, wblk, nwave, e0, n, out);
    return hipGetLastError();
}

extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_partial_amp(const ctpwa::AuxArgs* a, const int* wptr,
                                                                                     const int* wblk, int nwave,
                                                                                     long long e0, long long n, double* out,
                                                                                     hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    POST_LAUNCH(k_partial_amp, a->npol, n, *a, wptr, wblk, nwave, e0, n, (double2*)out);
    return hipGetLastError();
}

extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_aux(const ctpwa::AuxArgs* a, int nblock, long long e0,
                                                                             long long n, double* out, int intensity,
                                                                             hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    if (intensity) POST_LAUNCH(k_intensity, a->npol, n, *a, nblock, e0, n, out);
    else hipLaunchKernelGGL(ctpwa::k_amplitudes, dim3((unsigned)((n + 127) / 128)), dim3(128), 0, stream, *a, e0, n, out);
    return hipGetLastError();
}
