// Source generator for the per-event kernel of the Hessian (replaces the per-event part of
// analysis::getHessian, src/Analysis.cu:2689-3378, src/AmpGen.cu:3020-3540,
// src/ComputeHessian.cu:411-1170) and of the amplitude Gram.
//
// Like the fused likelihood kernel, the code is specialised to one model: every
// denominator, block product and amplitude is a straight line of register arithmetic.  Per
// event it forms
//   J      the Jacobian rows: for every polarisation p the complex columns
//          A_a,p = F_a sl_u(a),p (amplitudes) and dS_p/dtheta_j (free parameters),
//          real parts in columns [0, C), imaginary parts in [C, 2C);
//   u      dI/dx (x = Re v, Im v, theta), whose weighted Gram is the -w/I^2 part of the
//          second derivative of w ln I (data and background);
//   alpha = w / I and beta = -w / I^2 (data, background) or 1 and 0 (phase space);
// and the sums over events of the alpha-weighted second-part scalars <S, dA_a/dtheta_i>,
// sum_a Re(v_a d2F_a/dtheta_i dtheta_k conj(T_u)), alpha I, and of u.
//
// With psi_d = 1 / D_d, the log-derivatives L_i = sum_d psi_d dD_d/dtheta_i and
// M_ik = sum_d (psi_d d2D_d - psi_d^2 dD_i dD_k) give the block product's derivatives
// P1 = -dPsi = Psi L, P2 = d2Psi = Psi (L L^T - M); Custom factors multiply in by the
// product rule from their per-event value, first and second derivative rows.
//
// Wave groups.  The G waves of a workgroup take the same 64 events; each evaluates its own
// blocks (contiguous in an order that keeps the blocks of one parameter set together) and
// they exchange their shares of S through LDS.  One wave with all of a model's blocks holds
// every dS_j of both polarisations next to the block's derivatives: 576 bytes per lane of
// scratch at 10 amplitudes, 7 KB at 149.  A parameter whose blocks lie in several groups is
// summed through LDS slots in group order by one of them.
//
// Three forms:
//  * fused (FP64 Jacobian of up to 64 real columns): J and u of the 64 events go into an LDS
//    tile and straight into the FP64 matrix cores, whose tile pairs are shared out among the
//    waves; nothing per event is written.  Written to memory and read back by the Gram
//    kernel, the 40-column Jacobian of 3.05M events moved 3.9 GB (getHessian 1.31 ms,
//    fused 0.79 ms).
//  * rows: J (FP64, or FP32 in the mixed form), u and the weights are written to memory,
//    column-major, for the Gram kernels.
//  * split rows, for more than 24 amplitudes.  A workgroup of eight waves that runs the code
//    of all 149 amplitudes for its 64 events fetches 600 KB of instructions per step (64 KB
//    cache for two CUs), and each wave's 19 amplitudes spill: 6.9 ms for 600k events.  Here
//    ctpwa_hess_sum forms S and the weights (eight wave groups, 0.2 ms); then every workgroup
//    is one wave with one set of about eleven amplitudes (blockIdx.y), whose 30-50 KB of code
//    stay cached while all workgroups of the set run (1.5 ms, of which 0.8 ms are the FP64
//    instructions); then ctpwa_hess_theta adds up the parameters that several sets share
//    (0.4 ms).  Sets of 7 to 15 amplitudes are within 3 %, single blocks 6 % slower: more
//    parameters are shared then.
#include <algorithm>
#include <map>
#include <set>
#include <sstream>
#include <stdexcept>
#include <string>

#include "model.hpp"

namespace ctpwa {

static std::string DH(double x) {
    std::ostringstream s;
    s.precision(17);
    s << x;
    std::string r = s.str();
    if (r.find_first_of(".eEn") == std::string::npos) r += ".0";
    return r;
}

static const char* HR_PREAMBLE = R"(
typedef double d4 __attribute__((ext_vector_type(4)));
struct HessPieces { int n; int cls[4]; int wg0[5]; int spw[4]; long long e0[4], cnt[4], row0[4], w0[4]; int glo[4], ghi[4]; };
__device__ __forceinline__ double frcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, r, 1.0); r = __builtin_fma(r, e, r);
  e = __builtin_fma(-x, r, 1.0); return __builtin_fma(r, e, r);
}
// column c of a 64-event LDS tile, event at byte offset r8: columns are 66 doubles apart, so
// that the 16 columns x 2 rows that half a wave reads lie in different banks and every
// address is a lane offset plus a constant
__device__ __forceinline__ double& xe(double* xs, int c, int r8) { return *(double*)((char*)xs + (c * 528 + r8)); }
// element of a column at a lane's byte offset
template <typename T> __device__ __forceinline__ T& at(T* col, unsigned off) { return *(T*)((char*)col + off); }
__device__ __forceinline__ void wsync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// column sums over a wave's 64 lanes, SW columns at a time staged in the wave's LDS slab:
// this lane's part of the sum, column lane / (64 / SW), SW rows in row order
__device__ __forceinline__ double col_part(const double* xs, int lane) {
  wsync();
  const int c = lane / (64 / SW), r0 = (lane % (64 / SW)) * SW;
  double s = 0.0;
#pragma unroll
  for (int t = 0; t < SW; ++t) s += xs[c * 66 + r0 + t];
  wsync();
  return s;
}
)";

int hess_nz(const Model_& M) {
    int nz = 1;
    for (size_t b = 0; b < M.P.blocks.size(); ++b) {
        if (M.P.blocks[b].nsl == 0) continue;
        const int nl = (int)M.bvars[b].size();
        nz += M.P.blocks[b].nsl * 2 * nl + nl * (nl + 1) / 2;
    }
    return nz;
}

// a block's code in FP64 instructions, about (nl: its free parameters)
static double block_cost(const Model_& M, int b, int nl) {
    return 40.0 + 30.0 * nl + 15.0 * nl * (nl + 1) + M.P.blocks[b].nsl * (30.0 + 35.0 * nl + 6.0 * nl * (nl + 1));
}

// shape of the generated kernel: wave groups, their blocks, LDS layout
HessShape hess_shape(const Model_& M, bool amps_only) {
    const Plan& P = M.P;
    HessShape H;
    const int NT = amps_only ? 0 : P.ntheta;
    H.C = P.namp + NT;
    H.NU = amps_only ? 0 : 2 * P.namp + NT;
    H.f32 = M.mixed && !amps_only;
    const int NP = P.npol;
    std::vector<int> bl;
    for (size_t b = 0; b < P.blocks.size(); ++b) if (P.blocks[b].nsl > 0) bl.push_back((int)b);
    auto pars = [&](int b) {
        std::vector<int> v;
        if (!amps_only) v = M.bvars[b];
        std::sort(v.begin(), v.end());
        return v;
    };
    std::stable_sort(bl.begin(), bl.end(), [&](int x, int y) { return pars(x) < pars(y); });
    const int n = (int)bl.size();
    int sets = 1;
    for (int k = 1; k < n; ++k) sets += pars(bl[k]) != pars(bl[k - 1]);
    // about five amplitudes to a group.  FP64, 10 amplitudes, 3.05M events: four groups 818 us,
    // two 827; amplitude Gram, 1M events: 108 against 124.  FP32 rows hold less per event: 10
    // amplitudes, 305k events: two 126 us, four 134; 20 amplitudes, 360k events: two 492, four 445
    int G = P.namp <= 4 ? 1 : P.namp <= (H.f32 ? 12 : 8) ? 2 : P.namp <= 24 ? 4 : 8;
    H.fused = !H.f32 && 2 * H.C <= 64;
    H.split = !H.fused && P.namp > 24;
    if (H.split) G = (P.namp + 10) / 11;
    for (;; G /= 2) {
        G = std::max(1, std::min(G, n));
        // cuts: the largest group's cost (FP64 instructions) as small as possible; between
        // different parameter sets where there are enough of them
        std::vector<double> cost(n + 1, 0.0);
        for (int k = 0; k < n; ++k) cost[k + 1] = cost[k] + block_cost(M, bl[k], (int)pars(bl[k]).size());
        std::vector<std::vector<double>> best;
        std::vector<std::vector<int>> cut;
        auto solve = [&](bool at_sets) {
            best.assign(G + 1, std::vector<double>(n + 1, 1e300));
            cut.assign(G + 1, std::vector<int>(n + 1, -1));
            best[0][0] = 0.0;
            for (int g = 1; g <= G; ++g)
                for (int j = g; j <= n; ++j) {
                    if (at_sets && j < n && pars(bl[j]) == pars(bl[j - 1])) continue;
                    for (int i = g - 1; i < j; ++i) {
                        const double v = std::max(best[g - 1][i], cost[j] - cost[i]);
                        if (v < best[g][j]) { best[g][j] = v; cut[g][j] = i; }
                    }
                }
            return best[G][n];
        };
        // (shared parameters cost the slots and an idle wait less than a tenth of a group)
        const double any = solve(false);
        if (!amps_only && sets >= 2 * G && solve(true) > 1.1 * any) solve(false);
        H.blocks.assign(G, {});
        for (int g = G, j = n; g > 0; --g) {
            for (int k = cut[g][j]; k < j; ++k) H.blocks[g - 1].push_back(bl[k]);
            j = cut[g][j];
        }
        // parameters of several groups: one slot of [2 npol][64] doubles per group
        std::vector<std::set<int>> of(P.ntheta);
        for (int g = 0; g < G; ++g)
            for (int b : H.blocks[g])
                if (!amps_only) for (int j : M.bvars[b]) of[j].insert(g);
        H.nslot = 0;
        H.slot.assign(P.ntheta, {});
        H.owner.assign(P.ntheta, -1);
        std::vector<int> load(G, 0);
        for (int j = 0; j < P.ntheta; ++j) {
            if (of[j].empty()) continue;
            if (of[j].size() == 1) { H.owner[j] = *of[j].begin(); continue; }
            for (int g : of[j]) H.slot[j].push_back({g, H.nslot++});
            int o = *of[j].begin();
            for (int g : of[j]) if (load[g] < load[o]) o = g;
            H.owner[j] = o;
            load[o]++;
        }
        H.G = G;
        if (H.split) {
            H.SW = 16;
            H.lds = amps_only ? 0 : H.SW * 66;
            // the summing kernel's wave groups: the same order of blocks, cut by amplitudes
            // (as many as have room to exchange their shares of S in LDS)
            H.sum_blocks.assign(std::min({8, n, std::max(1, 159 / NP)}), {});
            for (int k = 0, a = 0; k < n; a += P.blocks[bl[k++]].nsl)
                H.sum_blocks[std::min<size_t>(H.sum_blocks.size() - 1, (size_t)a * H.sum_blocks.size() / P.namp)].push_back(bl[k]);
            return H;
        }
        const long long X = G > 1 && !amps_only ? (long long)G * 2 * NP * 64 : 0, T = (long long)H.nslot * 2 * NP * 64;
        // (the fused tile: a column of weights, then J of every polarisation, or u)
        const int GTn = (2 * H.C + 15) / 16;
        const long long comb = H.fused && G > 1 ? (long long)GTn * (GTn + 1) / 2 * 256 : 0;     // the waves' tiles at the end
        const long long tile = H.fused ? std::max(comb, (1 + std::max((long long)NP * 2 * H.C, (long long)H.NU)) * 66) : 0;
        for (H.SW = 16; H.SW >= 8; H.SW /= 2) {
            H.oX = 0;
            H.oT = X;
            H.oZ = X + T;
            H.lds = std::max(X + T + (amps_only ? 0 : (long long)G * H.SW * 66), tile);
            if (H.lds * 8 <= 160 * 1024) return H;
        }
        H.SW = 8;
        if (H.fused && tile * 8 > 160 * 1024) {         // many polarisations: rows instead
            H.fused = false;
            H.lds = X + T + (amps_only ? 0 : (long long)G * H.SW * 66);
            if (H.lds * 8 <= 160 * 1024) return H;
        }
        if (G == 1) throw std::runtime_error("Hessian generator: too many polarisation states for the LDS exchange");
    }
}

// amps_only: the Gram of the amplitudes alone (no couplings, weights 1; withK 0 leaves out
// the theta coefficients K_a).  perm (when given) receives, for every summed column in the
// order of zpart, its index in the assembly's order [Z (plan block order), alpha I, u].
std::string generate_hess_kernel(const Model_& M, std::vector<int>* perm, bool amps_only) {
    const Plan& P = M.P;
    const HessShape H = hess_shape(M, amps_only);
    const bool fused = H.fused, ahead = fused && 2 * H.C <= 48;
    const int NP = P.npol, NA = P.namp, NT = amps_only ? 0 : P.ntheta;
    const int C = H.C, NUX = H.NU, SW = H.SW;
    const int GT = (2 * C + 15) / 16, UT = (NUX + 15) / 16;     // tiles of the two Grams
    const int NG2 = GT * (GT + 1) / 2, NU2 = UT * (UT + 1) / 2;
    std::ostringstream src;
    src << "// generated: " << (amps_only ? "amplitude Gram" : "Hessian") << (fused ? ", fused" : ", rows") << "\n";
    src << "#define OFFR " << M.off_rec() << "LL\n#define OFFV " << M.off_v() << "LL\n#define REC " << Model_::REC << "\n"
        << "#define SW " << SW << "\n" << HR_PREAMBLE;
    const char* SLT = M.mixed ? "float2" : "double2";
    const char* JT = H.f32 ? "float" : "double";
    const std::vector<int> imap = M.imap();
    // component of the second derivative (i, k) in a coefficient record
    auto hidx = [](int i, int k) { return 1 + Model_::NLOC + i * Model_::NLOC + k; };
    const int NPS = M.npstore(), ncv = M.customs.empty() ? 0 : M.ncv(), nh = ncv * (ncv + 1) / 2;
    const int ncfr = M.customs.empty() ? 0 : amps_only ? M.ncf() : M.ncf2();     // rows per Custom factor
    // canonical column of every summed value: Z in plan block order, then alpha I, then u
    std::vector<int> zoff(P.blocks.size(), 0);
    int NZ = 0;
    for (size_t b = 0; b < P.blocks.size(); ++b) {
        zoff[b] = NZ;
        if (P.blocks[b].nsl == 0) continue;
        const int nl = (int)M.bvars[b].size();
        NZ += P.blocks[b].nsl * 2 * nl + nl * (nl + 1) / 2;
    }
    if (NZ + 1 != hess_nz(M)) throw std::runtime_error("Hessian generator: second-part sum count mismatch");
    const int col_I = NZ, col_u0 = NZ + 1;
    // Gram tile pairs (I <= J) of each wave
    auto pair_of = [](int q, int T) {
        int I = 0;
        while (q >= T - I) { q -= T - I; ++I; }
        return std::make_pair(I, I + q);
    };
    const std::string SIG =
        "    const double* __restrict__ tab, const void* __restrict__ slv, const double* __restrict__ inv,\n"
        "    const float* __restrict__ invf, long long ld, const double* __restrict__ wts, double w1, double w2,\n"
        "    int pw1, int pw2, HessPieces H, " + std::string(JT) + "* __restrict__ J, long long ldJ, double* __restrict__ U, double* __restrict__ W, double* __restrict__ D,\n"
        "    long long ldc, double* __restrict__ gpart, double* __restrict__ upart, double* __restrict__ zpart, int nwg,\n"
        "    const double* __restrict__ cfr, long long cld, int withK";
    const std::string CALL = "tab, slv, inv, invf, ld, wts, w1, w2, pw1, pw2, H, J, ldJ, U, W, D, ldc, gpart, upart, zpart, nwg, cfr, cld, withK";
    bool branch_u = NA <= 12;
    for (size_t b = 0; b < P.blocks.size(); ++b)
        if (P.blocks[b].nsl > 0 && block_cost(M, (int)b, (int)M.bvars[b].size()) > 1000.0) branch_u = false;
    std::vector<int> order_cols;
    std::ostringstream bodies;
    // the generated functions: the groups, and in the split form the sets, the parameter
    // columns and the groups of the summing kernel
    enum Kind { GROUP, SET, THETA, SUM };
    struct Body { Kind kind; int g, waves; std::vector<int> blocks; };
    std::vector<Body> todo;
    for (int g = 0; g < H.G; ++g) todo.push_back({H.split ? SET : GROUP, g, H.split ? 1 : H.G, H.blocks[g]});
    if (H.split && !amps_only) {
        todo.push_back({THETA, 0, 1, {}});
        for (size_t g = 0; g < H.sum_blocks.size(); ++g) todo.push_back({SUM, (int)g, (int)H.sum_blocks.size(), H.sum_blocks[g]});
    }
    for (const Body& body : todo) {
        std::ostringstream o;
        const std::vector<int>& blocks = body.blocks;
        const int g = body.g, G = body.waves;
        const Kind kind = body.kind;
        const int col0 = (int)order_cols.size();           // this wave's first summed column
        auto nput = [&]() { return (int)order_cols.size() - col0; };
        // what the group reads
        std::vector<char> xu(M.inv.size(), 0), su(M.us.size(), 0);
        for (int b : blocks) {
            for (int d : M.block_dens[b]) {
                for (const Term& t : M.dens[d].re) if (t.inv >= 0) xu[t.inv] = 1;
                for (const Term& t : M.dens[d].im) if (t.inv >= 0) xu[t.inv] = 1;
            }
            for (int c = 0; c < P.blocks[b].nsl; ++c) su[M.amps[P.blocks[b].site + c].u] = 1;
        }
        // Every per-event input of an iteration is loaded before its first store: on this target
        // a wait for a load issued after stores also waits for those stores, so loads placed
        // among the Jacobian stores would serialise the kernel on store completion.  The fused
        // form loads the next iteration's inputs (in their stored types) while the tile's
        // products run: the current event's values are dead by then, so it costs no registers
        // up to three tiles.  The ten pair sums of four tiles leave none (22 amplitudes at
        // 600k events: 503 us, without 479 us).
        struct Input { std::string type, name, src; };
        std::vector<Input> inputs;
        for (size_t i = 0; i < M.inv.size(); ++i) {
            if (!xu[i]) continue;
            const bool f = imap[i] < 0;
            inputs.push_back({f ? "float" : "double", "nx" + std::to_string(i),
                              (f ? "invf[" + std::to_string(-imap[i] - 1) : "inv[" + std::to_string(imap[i])) + "LL * ld + e]"});
        }
        for (size_t u = 0; u < M.us.size(); ++u)
            for (int p = 0; su[u] && p < NPS; ++p)
                inputs.push_back({SLT, "ng" + std::to_string(u) + "_" + std::to_string(p),
                                  "sl[" + std::to_string((long long)u * NPS + p) + "LL * ld + e]"});
        // Custom factor rows (value and, for the Hessian, first and second derivatives)
        for (int b : blocks)
            for (int c : M.block_customs[b])
                for (int k = 0; k < (amps_only ? 2 : ncfr); ++k)
                    inputs.push_back({"double", "ncf" + std::to_string(c) + "_" + std::to_string(k),
                                      "cfr[" + std::to_string((long long)c * ncfr + k) + "LL * cld + e]"});
        if (!amps_only && (kind == GROUP || kind == SUM)) inputs.push_back({"double", "nwload", "(cls != 0 && wvar) ? wts[e] : wconst"});
        for (const Input& in : inputs) {
            if (!ahead) o << "  const " << in.type << " " << in.name << " = " << in.src << ";\n";
            if (in.type == SLT) continue;
            o << "  const double " << in.name.substr(1) << " = (double)" << in.name << ";\n";
        }
        auto load_next = [&]() {
            o << "  {\n    const long long t1 = t0 + 64 + lane, e = pe0 + (t1 < b1 ? t1 : b1 - 1);\n";
            for (const Input& in : inputs) o << "    " << in.name << " = " << in.src << ";\n";
            o << "  }\n";
        };
        // stored polarisations per SL tensor; a polarisation past them is the signed
        // conjugate of its mirror image
        for (size_t u = 0; u < M.us.size(); ++u) {
            if (!su[u]) continue;
            for (int p = 0; p < NP; ++p) {
                std::string nm = std::to_string(u) + "_" + std::to_string(p);
                if (p >= NPS) {
                    const std::string mm = std::to_string(u) + "_" + std::to_string(NP - 1 - p);
                    const bool neg = M.psign[u] < 0;
                    o << "  const double s" << nm << "x = " << (neg ? "-" : "") << "s" << mm << "x, s" << nm << "y = " << (neg ? "" : "-")
                      << "s" << mm << "y;\n";
                    continue;
                }
                o << "  const double s" << nm << "x = (double)ng" << nm << ".x, s" << nm << "y = (double)ng" << nm << ".y;\n";
            }
        }
        auto cf = [&](int c, int k) { return "cf" + std::to_string(c) + "_" + std::to_string(k); };
        // Each phase reads the wave-uniform coefficients at its own offset of the table
        // pointer, a zero passed through an empty asm statement: the compiler then reloads
        // them (scalar loads) where the second phase needs them instead of keeping the first
        // phase's values live in registers.
        auto phase_vars = [&](int ph, bool inner) {
            o << "    long long z_" << ph << " = 0;\n    asm volatile(\"\" : \"+s\"(z_" << ph << "));\n"
              << "    const double* __restrict__ tb_" << ph << " = tab + z_" << ph << ";\n"
              << (inner ? "    int l8 = lane * 8;\n" : "    l8 = lane * 8;\n") << "    asm volatile(\"\" : \"+v\"(l8));\n    (void)l8;\n";
            if (!fused) o << "    lj = ldJ; lc = ldc; lu = cls != 0 ? ldc : 0;\n    asm volatile(\"\" : \"+s\"(lj), \"+s\"(lc), \"+s\"(lu));\n";
        };
        auto rec = [&](int ph, long long rr, int comp) {
            std::ostringstream q;
            q << "tb_" << ph << "[OFFR + " << rr << "LL * REC + " << comp << "]";
            return q.str();
        };
        // the propagators of block b (psi_d = pr + i pi) and the block product (br + i bi)
        auto emit_block_value = [&](int ph, int b, const char* ind) {
            const std::vector<int>& ds = M.block_dens[b];
            for (int d : ds) {
                const DenSpec& Dn = M.dens[d];
                auto term = [&](const Term& t) {
                    std::string c = (t.coef < 0) ? DH(t.cval) : rec(ph, Dn.coef_base + t.coef, 0);
                    return t.inv < 0 ? c : c + " * x" + std::to_string(t.inv);
                };
                o << ind << "double dr" << d << " = 0.0, di" << d << " = 0.0;\n";
                for (const Term& t : Dn.re) o << ind << "dr" << d << " += " << term(t) << ";\n";
                for (const Term& t : Dn.im) o << ind << "di" << d << " += " << term(t) << ";\n";
                if (Dn.stat) {
                    o << ind << "const double pr" << d << " = dr" << d << ", pi" << d << " = di" << d << ";\n";
                } else {
                    o << ind << "const double q" << d << " = frcp(dr" << d << " * dr" << d << " + di" << d << " * di" << d << ");\n";
                    o << ind << "const double pr" << d << " = dr" << d << " * q" << d << ", pi" << d << " = di" << d << " * q" << d << ";\n";
                }
            }
            o << ind << "double br = 1.0, bi = 0.0;\n";
            for (int d : ds)
                o << ind << "{ const double tr = br * pr" << d << " - bi * pi" << d << "; bi = br * pi" << d << " + bi * pr" << d
                  << "; br = tr; }\n";
        };
        auto sn = [&](int u, int p) { return "s" + std::to_string(u) + "_" + std::to_string(p); };
        auto jstore = [&](int col, int p, const std::string& v, const char* ind) {
            o << ind << "at(J" << p << " + " << col << "LL * lj, ro * (unsigned)sizeof(" << JT << ")) = (" << JT << ")(" << v << ");\n";
        };
        auto gsync = [&]() { o << (G > 1 ? "  __syncthreads();\n" : "  wsync();\n"); };

        // ---- phase 1: block products, amplitudes, S, I, weights ---------------------------
        const bool first = amps_only || kind == GROUP || kind == SUM, stores = !fused && kind != SUM;
        phase_vars(1, false);
        if (fused)
            for (int b : blocks)
                for (int c = 0; c < P.blocks[b].nsl; ++c)
                    o << "  double F" << P.blocks[b].site + c << "r, F" << P.blocks[b].site + c << "i;\n";
        if (!amps_only)
            for (int p = 0; p < NP; ++p)
                for (int c = 0; c < 2; ++c)
                    o << "  double S" << p << (c ? "i" : "r") << " = " << (first ? std::string("0.0") : "at(Wk + " + std::to_string(2 + 2 * p + c) + "LL * lc, wo)") << ";\n";
        for (int b : blocks) {
            if (!first) break;
            const PBlock& B = P.blocks[b];
            o << "  {\n";
            phase_vars(1, true);
            emit_block_value(1, b, "    ");
            for (int c : M.block_customs[b])
                o << "    { const double fr = " << cf(c, 0) << ", fi = " << cf(c, 1) << ";\n"
                  << "      const double tr = br * fr - bi * fi; bi = br * fi + bi * fr; br = tr; }\n";
            for (int cc = 0; cc < B.nsl; ++cc) {
                const int a = B.site + cc, u = M.amps[a].u;
                o << "    { const double K = " << (amps_only ? "withK ? " + rec(1, M.amps[a].coef_base, 0) + " : 1.0" : rec(1, M.amps[a].coef_base, 0)) << ";\n"
                  << "      const double Fr = K * br, Fi = K * bi;\n";
                if (fused) o << "      F" << a << "r = Fr; F" << a << "i = Fi;\n";
                if (!amps_only) o << "      const double vr = tb_1[OFFV + " << 2 * a << "], vi = tb_1[OFFV + " << 2 * a + 1 << "];\n";
                for (int p = 0; p < NP; ++p) {
                    if (amps_only && fused) continue;
                    o << "      { const double ar = Fr * " << sn(u, p) << "x - Fi * " << sn(u, p) << "y, ai = Fr * " << sn(u, p) << "y + Fi * "
                      << sn(u, p) << "x;\n";
                    if (!amps_only)
                        o << "        S" << p << "r += vr * ar - vi * ai; S" << p << "i += vr * ai + vi * ar;\n";
                    if (stores) {
                        jstore(a, p, "ar", "        ");
                        jstore(C + a, p, "ai", "        ");
                    }
                    o << "      }\n";
                }
                o << "    }\n";
            }
            o << "  }\n";
        }
        if (!amps_only) {
            if (G > 1) {
                // the groups' shares of S, added in group order by every wave
                o << "  double* xb = sm + " << H.oX << " + lane;\n";
                for (int p = 0; p < NP; ++p)
                    o << "  xb[" << (g * 2 * NP + 2 * p) * 64 << "] = S" << p << "r; xb[" << (g * 2 * NP + 2 * p + 1) * 64 << "] = S" << p << "i;\n";
                o << "  __syncthreads();\n";
                for (int p = 0; p < NP; ++p)
                    for (int c = 0; c < 2; ++c) {
                        o << "  S" << p << (c ? "i" : "r") << " = xb[" << (2 * p + c) * 64 << "]";
                        for (int h = 1; h < G; ++h) o << " + xb[" << (h * 2 * NP + 2 * p + c) * 64 << "]";
                        o << ";\n";
                    }
            }
            // a lane past the end: S = 0 makes every sum it hands in zero
            if (first) {
                o << "  if (!live) {";
                for (int p = 0; p < NP; ++p) o << " S" << p << "r = 0.0; S" << p << "i = 0.0;";
                o << " }\n";
            }
            o << "  double I = 0.0;\n";
            for (int p = 0; p < NP; ++p) o << "  I += S" << p << "r * S" << p << "r + S" << p << "i * S" << p << "i;\n";
            if (!first) o << "  const double alpha = at(Wk, wo);\n";
            else o << "  const double we = (cls == 0) ? 1.0 : wload;\n"
                 "  double alpha, beta;\n"
                 "  if (cls == 0) { alpha = 1.0; beta = 0.0; }\n"
                 "  else if (I == 0.0) { alpha = 0.0; beta = 0.0; }\n"
                 "  else { const double iI = frcp(I); alpha = we * iI; beta = -alpha * iI; }\n";
            if (!fused && first && g == 0) o << "  at(Wk, wo) = alpha; at(Wk + lc, wo) = beta;\n";
            if (kind == SUM) {
                for (int p = 0; p < NP && g == 0; ++p)
                    o << "  at(Wk + " << 2 + 2 * p << "LL * lc, wo) = S" << p << "r; at(Wk + " << 3 + 2 * p << "LL * lc, wo) = S" << p << "i;\n";
                if (G > 1) o << "  __syncthreads();\n";      // every wave has read the exchanged S
            }
        }
        if (!amps_only && kind != SUM) {

            // ---- phase 2: u, derivative columns and second-part scalars --------------------
            o << "  double* zs = sm + " << (H.split ? 0 : H.oZ + (long long)g * SW * 66) << ";\n";
            auto flush = [&](const char* ind) {
                o << ind << "zf" << (nput() - 1) / SW << " += col_part(zs, l8 >> 3);\n";
            };
            auto put = [&](const std::string& v, int col, const char* ind) {
                o << ind << "xe(zs, " << nput() % SW << ", l8) = " << v << ";\n";
                order_cols.push_back(col);
                if (nput() % SW == 0) flush(ind);
            };
            auto ustore = [&](const std::string& v, int x, const char* ind) {
                put(v, col_u0 + x, ind);
                if (!fused) o << ind << (kind == GROUP && branch_u ? "if (cls != 0) " : "") << "at(Uk + " << x << "LL * lu, wo) = " << v << ";\n";
            };
            // a parameter's finished derivative columns
            auto theta_cols = [&](int j) {
                o << "  const double ut" << j << " = 2.0 * (";
                for (int p = 0; p < NP; ++p)
                    o << (p ? " + " : "") << "(S" << p << "r * dS" << j << "_" << p << "r + S" << p << "i * dS" << j << "_" << p << "i)";
                o << ");\n";
                ustore("ut" + std::to_string(j), 2 * NA + j, "  ");
                if (fused) return;
                for (int p = 0; p < NP; ++p) {
                    const std::string d = "dS" + std::to_string(j) + "_" + std::to_string(p);
                    jstore(NA + j, p, d + "r", "  ");
                    jstore(C + NA + j, p, d + "i", "  ");
                }
            };
            phase_vars(2, false);
            if (g == 0 && kind != SET) put("alpha * I", col_I, "  ");
            std::vector<int> last(NT, -1);
            for (size_t k = 0; k < blocks.size(); ++k)
                for (int j : M.bvars[blocks[k]]) last[j] = (int)k;
            std::vector<char> open_(NT, 0);
            for (size_t kb = 0; kb < blocks.size(); ++kb) {
                const int b = blocks[kb];
                const PBlock& B = P.blocks[b];
                const std::vector<int>& vars = M.bvars[b];
                const int nl = (int)vars.size();
                for (int j : vars)
                    if (!open_[j]) {
                        open_[j] = 1;
                        for (int p = 0; p < NP; ++p) o << "  double dS" << j << "_" << p << "r = 0.0, dS" << j << "_" << p << "i = 0.0;\n";
                    }
                o << "  {\n";
                phase_vars(2, true);
                emit_block_value(2, b, "    ");
                o << "    double psr = br, psi_ = bi;\n";
                if (nl > 0) {
                    // log-derivatives of the propagators: l_i = psi dD_i, M_ik = sum (psi d2D_ik - l_i l_k)
                    for (int i = 0; i < nl; ++i) o << "    double Lr" << i << " = 0.0, Li" << i << " = 0.0;\n";
                    for (int i = 0; i < nl; ++i)
                        for (int k = i; k < nl; ++k) o << "    double Mr" << i << "_" << k << " = 0.0, Mi" << i << "_" << k << " = 0.0;\n";
                    for (int d : M.block_dens[b]) {
                        const DenSpec& Dn = M.dens[d];
                        if (Dn.stat) continue;
                        bool any = false;
                        for (const Term& t : Dn.re) if (t.coef >= 0) any = true;
                        for (const Term& t : Dn.im) if (t.coef >= 0) any = true;
                        if (!any) continue;
                        auto dsum = [&](const char* acc, int comp, const char* ind) {
                            for (const Term& t : Dn.re)
                                if (t.coef >= 0)
                                    o << ind << acc << "r += " << rec(2, Dn.coef_base + t.coef, comp) << (t.inv >= 0 ? " * x" + std::to_string(t.inv) : "") << ";\n";
                            for (const Term& t : Dn.im)
                                if (t.coef >= 0)
                                    o << ind << acc << "i += " << rec(2, Dn.coef_base + t.coef, comp) << (t.inv >= 0 ? " * x" + std::to_string(t.inv) : "") << ";\n";
                        };
                        o << "    {\n";
                        phase_vars(2, true);
                        // dD_i = gr - i gi; l_i = (pr + i pi)(gr - i gi)
                        for (int i = 0; i < nl; ++i) {
                            o << "      double g" << i << "r = 0.0, g" << i << "i = 0.0;\n";
                            dsum(("g" + std::to_string(i)).c_str(), 1 + i, "      ");
                            o << "      const double lr" << i << " = pr" << d << " * g" << i << "r + pi" << d << " * g" << i << "i, li" << i << " = pi" << d
                              << " * g" << i << "r - pr" << d << " * g" << i << "i;\n";
                            o << "      Lr" << i << " += lr" << i << "; Li" << i << " += li" << i << ";\n";
                        }
                        for (int i = 0; i < nl; ++i)
                            for (int k = i; k < nl; ++k) {
                                o << "      { double hr = 0.0, hi = 0.0;\n";
                                if (k == i && nl > 2) phase_vars(2, true);
                                dsum("h", hidx(i, k), "        ");
                                o << "        Mr" << i << "_" << k << " += pr" << d << " * hr + pi" << d << " * hi - (lr" << i << " * lr" << k << " - li" << i
                                  << " * li" << k << ");\n"
                                  << "        Mi" << i << "_" << k << " += pi" << d << " * hr - pr" << d << " * hi - (lr" << i << " * li" << k << " + li" << i
                                  << " * lr" << k << "); }\n";
                            }
                        o << "    }\n";
                    }
                    // P1 = Psi L, P2 = Psi (L L - M)
                    for (int i = 0; i < nl; ++i)
                        for (int k = i; k < nl; ++k)
                            o << "    double P2r" << i << "_" << k << ", P2i" << i << "_" << k << ";\n"
                              << "    { const double ar = Lr" << i << " * Lr" << k << " - Li" << i << " * Li" << k << " - Mr" << i << "_" << k << ", ai = Lr" << i
                              << " * Li" << k << " + Li" << i << " * Lr" << k << " - Mi" << i << "_" << k << ";\n"
                              << "      P2r" << i << "_" << k << " = psr * ar - psi_ * ai; P2i" << i << "_" << k << " = psr * ai + psi_ * ar; }\n";
                    for (int i = 0; i < nl; ++i)
                        o << "    double P1r" << i << " = psr * Lr" << i << " - psi_ * Li" << i << ", P1i" << i << " = psr * Li" << i << " + psi_ * Lr" << i << ";\n";
                }
                // Custom factors: d2(Psi F) = P2 F - P1_i F_k - P1_k F_i + Psi F_ik; -(Psi F)_i = P1_i F - Psi F_i
                for (int c : M.block_customs[b]) {
                    o << "    {\n      const double fr = " << cf(c, 0) << ", fi = " << cf(c, 1) << ";\n";
                    for (int i = 0; i < nl; ++i)
                        o << "      const double fr" << i << " = " << cf(c, 2 + i) << ", fi" << i << " = " << cf(c, 2 + ncv + i) << ";\n";
                    for (int i = 0; i < nl; ++i)
                        for (int k = i; k < nl; ++k) {
                            const int h = i * ncv - (i * (i - 1)) / 2 + (k - i);
                            o << "      { const double hr = " << cf(c, 2 + 2 * ncv + h) << ", hi = " << cf(c, 2 + 2 * ncv + nh + h) << ";\n"
                              << "        const double nr = P2r" << i << "_" << k << " * fr - P2i" << i << "_" << k << " * fi - (P1r" << i << " * fr" << k
                              << " - P1i" << i << " * fi" << k << ") - (P1r" << k << " * fr" << i << " - P1i" << k << " * fi" << i << ") + (psr * hr - psi_ * hi);\n"
                              << "        const double ni = P2r" << i << "_" << k << " * fi + P2i" << i << "_" << k << " * fr - (P1r" << i << " * fi" << k
                              << " + P1i" << i << " * fr" << k << ") - (P1r" << k << " * fi" << i << " + P1i" << k << " * fr" << i << ") + (psr * hi + psi_ * hr);\n"
                              << "        P2r" << i << "_" << k << " = nr; P2i" << i << "_" << k << " = ni; }\n";
                        }
                    for (int i = 0; i < nl; ++i)
                        o << "      { const double nr = P1r" << i << " * fr - P1i" << i << " * fi - (psr * fr" << i << " - psi_ * fi" << i << ");\n"
                          << "        const double ni = P1r" << i << " * fi + P1i" << i << " * fr - (psr * fi" << i << " + psi_ * fr" << i << ");\n"
                          << "        P1r" << i << " = nr; P1i" << i << " = ni; }\n";
                    o << "      { const double tr = psr * fr - psi_ * fi; psi_ = psr * fi + psi_ * fr; psr = tr; }\n    }\n";
                }
                // sums over the block's amplitudes of w = v conj(T_u) times K, K_i and K_ik
                if (nl > 0) o << "    double W0r = 0.0, W0i = 0.0;\n";
                for (int i = 0; i < nl; ++i) {
                    o << "    double W" << i << "_r = 0.0, W" << i << "_i = 0.0;\n";
                    for (int k = i; k < nl; ++k) o << "    double W" << i << "_" << k << "r = 0.0, W" << i << "_" << k << "i = 0.0;\n";
                }
                std::vector<char> loaded(M.us.size(), 0);
                for (int cc = 0; cc < B.nsl; ++cc) {
                    const int a = B.site + cc, u = M.amps[a].u;
                    const long long ra = M.amps[a].coef_base;
                    if (!loaded[u]) {
                        // T_u = sum_p conj(sl_u,p) S_p
                        o << "    double t" << u << "r = 0.0, t" << u << "i = 0.0;\n";
                        for (int p = 0; p < NP; ++p)
                            o << "    t" << u << "r += " << sn(u, p) << "x * S" << p << "r + " << sn(u, p) << "y * S" << p << "i; t" << u << "i += " << sn(u, p)
                              << "x * S" << p << "i - " << sn(u, p) << "y * S" << p << "r;\n";
                    }
                    loaded[u] = 1;
                    o << "    {\n";
                    phase_vars(2, true);
                    o << "      const double K = " << rec(2, ra, 0) << ";\n"
                      << "      const double vr = tb_2[OFFV + " << 2 * a << "], vi = tb_2[OFFV + " << 2 * a + 1 << "];\n"
                      << "      const double Fr = K * psr, Fi = K * psi_;\n"
                      // g_a = conj(F_a) T_u: dI/dRe v_a = 2 Re g, dI/dIm v_a = 2 Im g
                      << "      const double gr = Fr * t" << u << "r + Fi * t" << u << "i, gi = Fr * t" << u << "i - Fi * t" << u << "r;\n";
                    for (int p = 0; p < NP && kind == SET; ++p) {
                        jstore(a, p, "Fr * " + sn(u, p) + "x - Fi * " + sn(u, p) + "y", "      ");
                        jstore(C + a, p, "Fr * " + sn(u, p) + "y + Fi * " + sn(u, p) + "x", "      ");
                    }
                    ustore("2.0 * gr", a, "      ");
                    ustore("2.0 * gi", NA + a, "      ");
                    for (int i = 0; i < nl; ++i) {
                        // dF_i = K_i Psi - K P1_i; q = dF_i conj(T_u) = <S, dA_a/dtheta_i>
                        o << "      const double Kg" << i << " = " << rec(2, ra, 1 + i) << ";\n"
                          << "      const double dFr" << i << " = Kg" << i << " * psr - K * P1r" << i << ", dFi" << i << " = Kg" << i << " * psi_ - K * P1i" << i << ";\n"
                          << "      const double qr" << i << " = dFr" << i << " * t" << u << "r + dFi" << i << " * t" << u << "i, qi" << i << " = dFi" << i << " * t" << u
                          << "r - dFr" << i << " * t" << u << "i;\n";
                        put("alpha * qr" + std::to_string(i), zoff[b] + cc * 2 * nl + 2 * i, "      ");
                        put("alpha * qi" + std::to_string(i), zoff[b] + cc * 2 * nl + 2 * i + 1, "      ");
                        o << "      { const double vdr = vr * dFr" << i << " - vi * dFi" << i << ", vdi = vr * dFi" << i << " + vi * dFr" << i << ";\n";
                        for (int p = 0; p < NP; ++p)
                            o << "        dS" << vars[i] << "_" << p << "r += vdr * " << sn(u, p) << "x - vdi * " << sn(u, p) << "y; dS" << vars[i] << "_" << p << "i += vdr * "
                              << sn(u, p) << "y + vdi * " << sn(u, p) << "x;\n";
                        o << "      }\n";
                    }
                    if (nl > 0) {
                        o << "      {\n";
                        phase_vars(2, true);
                        o << "      const double wr_ = vr * t" << u << "r + vi * t" << u << "i, wi_ = vi * t" << u << "r - vr * t" << u << "i;\n"
                          << "      W0r += K * wr_; W0i += K * wi_;\n";
                        for (int i = 0; i < nl; ++i) {
                            o << "      W" << i << "_r += Kg" << i << " * wr_; W" << i << "_i += Kg" << i << " * wi_;\n";
                            for (int k = i; k < nl; ++k)
                                o << "      { const double Kh = " << rec(2, ra, hidx(i, k)) << "; W" << i << "_" << k << "r += Kh * wr_; W" << i
                                  << "_" << k << "i += Kh * wi_; }\n";
                        }
                        o << "      }\n";
                    }
                    o << "    }\n";
                    // (regions of one amplitude: scheduling a whole block at once takes the
                    // compiler five times as long and keeps no fewer registers)
                    if (kind == SET) o << "    __builtin_amdgcn_sched_barrier(0);\n";
                }
                // R_ik = sum_a Re(v_a d2F_ik conj(T_u)), d2F_ik = K_ik Psi - K_i P1_k - K_k P1_i + K P2_ik
                {
                    int z = zoff[b] + B.nsl * 2 * nl;
                    for (int i = 0; i < nl; ++i)
                        for (int k = i; k < nl; ++k) {
                            std::ostringstream v;
                            v << "alpha * (psr * W" << i << "_" << k << "r - psi_ * W" << i << "_" << k << "i - (P1r" << k << " * W" << i << "_r - P1i" << k
                              << " * W" << i << "_i) - (P1r" << i << " * W" << k << "_r - P1i" << i << " * W" << k << "_i) + (P2r" << i << "_" << k
                              << " * W0r - P2i" << i << "_" << k << " * W0i))";
                            put(v.str(), z++, "    ");
                        }
                }
                o << "  }\n";
                // parameters whose last block of this group this was: their columns, or the
                // group's share of them into its slot
                for (int j : vars) {
                    if (last[j] != (int)kb) continue;
                    if (H.slot[j].empty()) { theta_cols(j); continue; }
                    for (const auto& s : H.slot[j])
                        if (s.first == g && kind == SET)
                            for (int p = 0; p < NP; ++p)
                                o << "  at(Dk + " << s.second * 2 * NP + 2 * p << "LL * lc, wo) = dS" << j << "_" << p << "r; at(Dk + " << s.second * 2 * NP + 2 * p + 1
                                  << "LL * lc, wo) = dS" << j << "_" << p << "i;\n";
                        else if (s.first == g)
                            for (int p = 0; p < NP; ++p)
                                o << "  sm[" << H.oT + ((long long)s.second * 2 * NP + 2 * p) * 64 << " + lane] = dS" << j << "_" << p << "r; sm["
                                  << H.oT + ((long long)s.second * 2 * NP + 2 * p + 1) * 64 << " + lane] = dS" << j << "_" << p << "i;\n";
                }
            }
            // shared parameters, summed in group order by their owner.  (The barrier also
            // ends every wave's reads of the exchanged S before the next iteration writes it;
            // the slots are written again only after the next iteration's first barrier.)
            if (G > 1) o << "  __syncthreads();\n";
            for (int j = 0; j < NT; ++j) {
                if (H.slot[j].empty() || (H.split ? kind != THETA : H.owner[j] != g)) continue;
                if (H.split) phase_vars(3 + j, false);
                for (int p = 0; p < NP; ++p)
                    for (int c = 0; c < 2; ++c) {
                        o << "  " << (open_[j] ? "" : "double ") << "dS" << j << "_" << p << (c ? "i" : "r") << " = ";
                        for (size_t k = 0; k < H.slot[j].size(); ++k)
                            if (H.split) o << (k ? " + " : "") << "at(Dk + " << H.slot[j][k].second * 2 * NP + 2 * p + c << "LL * lc, wo)";
                            else o << (k ? " + " : "") << "sm[" << H.oT + ((long long)H.slot[j][k].second * 2 * NP + 2 * p + c) * 64 << " + lane]";
                        o << ";\n";
                    }
                theta_cols(j);
            }
            // parameters of no block with waves: zero columns
            if (g == 0 && kind != SET)
                for (int j = 0; j < NT; ++j)
                    if (H.owner[j] < 0 && H.slot[j].empty()) {
                        for (int p = 0; p < NP; ++p) o << "  const double dS" << j << "_" << p << "r = 0.0, dS" << j << "_" << p << "i = 0.0;\n";
                        theta_cols(j);
                    }
            if (nput() % SW) flush("  ");
        }
        if (fused) {
            // u (data, background), then the Jacobian of both polarisations, through the
            // workgroup's LDS tile into the matrix cores; the waves share out the tile's rows
            // and each holds every tile pair's sums.  (Sharing out the pairs instead has every
            // wave run the whole row loop, with its address arithmetic, and left the waves
            // unevenly loaded.)  A lane's operand serves as A (times the weight) and as B:
            // A[i][k] is in lane 16 k + i, B[k][j] in lane 16 k + j.  Columns past the last one
            // repeat it (their products are dropped).
            auto col = [&](int c, const std::string& v, const char* ind) {
                o << ind << "xe(sm, " << 1 + c << ", l8) = " << v << ";\n";
            };
            // rows [rb, re) (multiples of 4) of the tile's columns base .. base + nc
            auto pass = [&](int base, int T, int nc, bool weighted, const char* acc, int rb, int re) {
                if (rb >= re) return;
                o << "#pragma unroll 8\n  for (int k0 = " << rb << "; k0 < " << re << "; k0 += 4) {\n";
                if (weighted) o << "    const double wr = sm[k0 + (lane >> 4)];\n";
                for (int I = 0; I < T; ++I) {
                    const bool whole = 16 * I + 16 <= nc;
                    o << "    const double x" << I << " = sm[" << (1 + base + 16 * I) * 66 << " + "
                      << (whole ? "(lane & 15)" : "((lane & 15) < " + std::to_string(nc - 16 * I) + " ? (lane & 15) : " + std::to_string(nc - 16 * I - 1) + ")")
                      << " * 66 + (lane >> 4) + k0];\n";
                }
                int q = 0;
                for (int I = 0; I < T; ++I) {
                    o << "    const double a" << I << " = " << (weighted ? "wr * " : "") << "x" << I << ";\n";
                    for (int Jt = I; Jt < T; ++Jt, ++q)
                        o << "    " << acc << q << " = __builtin_amdgcn_mfma_f64_16x16x4f64(a" << I << ", x" << Jt << ", " << acc << q << ", 0, 0, 0);\n";
                }
                o << "  }\n";
            };
            if (!amps_only) {
                gsync();                        // slabs and slots are consumed
                o << "  if (cls != 0) {\n";
                std::vector<char> td(M.us.size(), 0);
                for (int b : blocks)
                    for (int c = 0; c < P.blocks[b].nsl; ++c) {
                        const int a = P.blocks[b].site + c, u = M.amps[a].u;
                        if (!td[u]) {
                            td[u] = 1;
                            o << "    double t" << u << "r = 0.0, t" << u << "i = 0.0;\n";
                            for (int p = 0; p < NP; ++p)
                                o << "    t" << u << "r += " << sn(u, p) << "x * S" << p << "r + " << sn(u, p) << "y * S" << p << "i; t" << u << "i += " << sn(u, p)
                                  << "x * S" << p << "i - " << sn(u, p) << "y * S" << p << "r;\n";
                        }
                        const std::string f = "F" + std::to_string(a), t = "t" + std::to_string(u);
                        col(a, "2.0 * (" + f + "r * " + t + "r + " + f + "i * " + t + "i)", "    ");
                        col(NA + a, "2.0 * (" + f + "r * " + t + "i - " + f + "i * " + t + "r)", "    ");
                    }
                for (int j = 0; j < NT; ++j)
                    if (H.owner[j] == g || (g == 0 && H.owner[j] < 0)) col(2 * NA + j, "ut" + std::to_string(j), "    ");
                if (g == 0) o << "    xe(sm, 0, l8) = live ? beta : 0.0;\n";
                gsync();
                pass(0, UT, NUX, true, "au", 64 * g / G / 4 * 4, 64 * (g + 1) / G / 4 * 4);
                gsync();
                o << "  }\n";
            }
            for (int p = 0; p < NP; ++p) {
                for (int b : blocks)
                    for (int c = 0; c < P.blocks[b].nsl; ++c) {
                        const int a = P.blocks[b].site + c, u = M.amps[a].u;
                        const std::string f = "F" + std::to_string(a);
                        // (amplitude Gram: lanes past the end must add nothing; no weight is applied)
                        col(p * 2 * C + a, (amps_only ? "live ? " : "") + (f + "r * " + sn(u, p) + "x - " + f + "i * " + sn(u, p) + "y") + (amps_only ? " : 0.0" : ""), "  ");
                        col(p * 2 * C + C + a, (amps_only ? "live ? " : "") + (f + "r * " + sn(u, p) + "y + " + f + "i * " + sn(u, p) + "x") + (amps_only ? " : 0.0" : ""), "  ");
                    }
                for (int j = 0; j < NT; ++j) {
                    if (!(H.owner[j] == g || (g == 0 && H.owner[j] < 0))) continue;
                    const std::string d = "dS" + std::to_string(j) + "_" + std::to_string(p);
                    col(p * 2 * C + NA + j, d + "r", "  ");
                    col(p * 2 * C + C + NA + j, d + "i", "  ");
                }
            }
            if (!amps_only && g == 0) o << "  xe(sm, 0, l8) = live ? alpha : 0.0;\n";
            if (ahead) load_next();
            gsync();
            // the npol 64-row tiles one after the other, cut into G ranges
            for (int p = 0; p < NP; ++p)
                pass(p * 2 * C, GT, 2 * C, !amps_only, "ag", std::max(0, std::min(64, NP * 64 * g / G / 4 * 4 - 64 * p)),
                     std::max(0, std::min(64, NP * 64 * (g + 1) / G / 4 * 4 - 64 * p)));
            gsync();                            // the tile is consumed
        }
        // the function: declarations, the loop over the workgroup's events, the partial sums
        const int ncols = nput(), nflush = (ncols + SW - 1) / SW;
        static const char* const fname[] = {"hess_g", "hess_g", "hess_t", "hess_s"};
        bodies << "__device__ __forceinline__ void " << fname[kind] << g << "(\n" << SIG << ", double* __restrict__ sm)\n{\n"
               << "  const " << SLT << "* __restrict__ sl = (const " << SLT << "*)slv;\n"
               << "  const int lane = threadIdx.x & 63, wg = blockIdx.x;\n"
                  "  int k = 0;\n  while (k + 1 < H.n && wg >= H.wg0[k + 1]) ++k;\n"
                  "  const int cls = H.cls[k];\n"
                  "  const long long cnt = H.cnt[k], pe0 = H.e0[k];\n"
                  "  const long long b0 = (long long)(wg - H.wg0[k]) * H.spw[k] * 64, b1_ = b0 + (long long)H.spw[k] * 64;\n"
                  "  const long long b1 = b1_ < cnt ? b1_ : cnt;\n"
                  "  const double wconst = cls == 1 ? w1 : w2;\n"
                  "  const bool wvar = cls == 1 ? pw1 != 0 : cls == 2 && pw2 != 0;\n";
        for (int f = 0; f < nflush; ++f) bodies << "  double zf" << f << " = 0.0;\n";
        if (!fused) {
            // rows: uniform column addresses plus a 32-bit lane offset.  The column strides pass
            // through empty asm statements (phase_vars), or hundreds of column addresses are
            // formed before the loop and kept in spilled registers.  Phase space has no u.  Its
            // stores go to one column that nothing reads: a branch around each store cuts a
            // block's code into pieces that the compiler schedules and allocates badly (2.5 KB
            // of scratch per lane in the sets; 600k events, mixed: 12 amplitudes in blocks of
            // 1600 instructions 477 us, without branches 265; 8 in blocks of up to 1400, 299
            // and 206).  Only where every block is small is the branch the better one: 10
            // amplitudes in blocks of 330 instructions 208 and 231 us, 8 in blocks of up to 460
            // 136 and 154, 6 in blocks of up to 730 116 and 121; 13 in blocks of 330 the same.
            bodies << "  long long lj = ldJ, lc = ldc, lu = ldc;\n  (void)lj; (void)lc; (void)lu;\n";
            for (int p = 0; p < NP; ++p) bodies << "  " << JT << "* __restrict__ J" << p << " = J + H.row0[k] + " << p << " * cnt;\n";
            if (!amps_only) bodies << "  double *__restrict__ Uk = U + H.w0[k], *__restrict__ Wk = W + H.w0[k], *__restrict__ Dk = D + H.w0[k];\n";
        }
        if (fused) {
            for (int q = 0; q < NG2; ++q) bodies << "  d4 ag" << q << " = (d4){0.0, 0.0, 0.0, 0.0};\n";
            for (int q = 0; q < NU2; ++q) bodies << "  d4 au" << q << " = (d4){0.0, 0.0, 0.0, 0.0};\n";
        }
        if (ahead) {
            bodies << "  if (b0 >= cnt) return;\n  const long long e = pe0 + (b0 + lane < b1 ? b0 + lane : b1 - 1);\n";
            for (const Input& in : inputs) bodies << "  " << in.type << " " << in.name << " = " << in.src << ";\n";
        }
        bodies << "  for (long long t0 = b0; t0 < b1; t0 += 64) {\n"
                  // a copy of the lane index the optimiser cannot see through, here and in every
                  // scope: the dozens of LDS addresses made from it are then formed where they
                  // are used instead of being kept in registers across the loop
                  "  int l8 = lane * 8;\n  asm volatile(\"\" : \"+v\"(l8));\n"
                  // a lane past the end takes the last event: its row stores repeat that event's
                  // own values (no guard around each), its sums get weight 0
                  "  const bool live = t0 + lane < b1;\n"
                  "  const long long r = live ? t0 + lane : b1 - 1;\n"
                  "  const long long e = pe0 + r;\n  (void)e;\n";
        if (!fused) {
            // (the u and weight entries of lanes past the end go to the piece's padding)
            bodies << "  const unsigned ro = (unsigned)r;\n";
            if (!amps_only) bodies << "  const unsigned wo = (unsigned)(t0 + lane) * 8u;\n";
        }
        bodies << o.str() << "  }\n";
        if (fused) {
            // element 16 i + j of a tile pair: D[4 r + q][j] is component r of lane 16 q + j; the
            // waves add their tiles in LDS, one after the other, a pair's tile at a time
            auto combine = [&](const char* acc, int n, const char* out) {
                bodies << "  {\n    double* o = sm + (lane >> 4) * 16 + (lane & 15);\n";
                for (int h = 0; h < G; ++h) {
                    if (h == g)
                        for (int q = 0; q < n; ++q)
                            for (int r = 0; r < 4; ++r) {
                                const std::string at = "[" + std::to_string(q * 256 + r * 64) + "]", v = acc + std::to_string(q) + "[" + std::to_string(r) + "]";
                                if (h + 1 < G) bodies << "    o" << at << " = " << (h ? "o" + at + " + " : "") << v << ";\n";
                                else bodies << "    " << out << "[((long long)wg * " << n << " + " << q << ") * 256 + " << r * 64 << " + lane] = "
                                            << (h ? "o" + at + " + " : "") << v << ";\n";
                            }
                    if (h + 1 < G) bodies << "    __syncthreads();\n";
                }
                bodies << "  }\n";
            };
            combine("ag", NG2, "gpart");
            if (!amps_only) {
                if (G > 1) bodies << "  __syncthreads();\n";
                bodies << "  if (cls != 0) ";
                combine("au", NU2, "upart");
            }
        }
        for (int f = 0; f < nflush; ++f) {
            for (int s = 1; s < 64 / SW; s *= 2) bodies << "  zf" << f << " += __shfl_xor(zf" << f << ", " << s << ", 64);\n";
            bodies << "  if (lane % " << 64 / SW << " == 0 && lane / " << 64 / SW << " < " << std::min(SW, ncols - SW * f) << ") zpart[(" << col0 + SW * f
                   << "LL + lane / " << 64 / SW << ") * nwg + wg] = zf" << f << ";\n";
        }
        bodies << "}\n";
    }
    if (!amps_only && (int)order_cols.size() != NZ + 1 + NUX) throw std::runtime_error("Hessian generator: summed-column count mismatch");
    if (perm) *perm = order_cols;
    src << bodies.str();
    // a kernel of n functions, one per wave of the workgroup or (sets) per blockIdx.y
    auto kernel = [&](const char* name, const char* fn, int n, bool sets, long long lds, const char* bounds) {
        src << "extern \"C\" __global__ void __launch_bounds__(" << (sets ? 64 : 64 * n) << bounds << ") " << name << "(\n" << SIG << ")\n{\n"
            << "  __shared__ __attribute__((aligned(16))) double sm[" << std::max<long long>(lds, 2) << "];\n";
        if (n == 1) {
            src << "  " << fn << "0(" << CALL << ", sm);\n}\n";
            return;
        }
        src << "  switch (" << (sets ? "blockIdx.y" : "__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))") << ") {\n";
        for (int g = 0; g < n; ++g)
            src << "  " << (g + 1 < n ? "case " + std::to_string(g) : std::string("default")) << ": " << fn << g << "(" << CALL << ", sm); break;\n";
        src << "  }\n}\n";
    };
    kernel(amps_only ? "ctpwa_amp_gram" : fused ? "ctpwa_hess_fused" : "ctpwa_hess_rows", "hess_g", H.G, H.split, H.lds,
           H.split || (H.G < 8 && (!fused || 2 * C <= 48)) ? ", 2" : "");
    if (H.split && !amps_only) {
        kernel("ctpwa_hess_theta", "hess_t", 1, true, H.lds, "");
        kernel("ctpwa_hess_sum", "hess_s", (int)H.sum_blocks.size(), false, (long long)H.sum_blocks.size() * 2 * NP * 64, "");
    }
    return src.str();
}

}  // namespace ctpwa
