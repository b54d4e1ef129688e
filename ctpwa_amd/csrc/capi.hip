// C ABI of the native likelihood library: handle construction (plan -> device
// layout -> one-time SL/invariant kernels -> generated fused kernel via hipRTC) and
// the per-evaluation entry points.  See include/ctpwa_amd.h for the contract.
#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/ctpwa_amd.h"
#include "device.hpp"
#include "model.hpp"

namespace ctpwa {
std::string generate_eval_kernel(const Model_& M);
std::string generate_custom2_kernel(const Model_& M);
std::string generate_hess_kernel(const Model_& M, std::vector<int>* perm, bool amps_only);
}

extern "C" hipError_t ctpwa_launch_init(const double*, long long, int, const ctpwa::DTopo*, int, const ctpwa::DNode*,
                                         const ctpwa::DKin*, int, const ctpwa::DU*, int, const double*, const int*, int,
                                         const ctpwa::DInv*, int, const double*, double2*, double*, long long, long long,
                                         hipStream_t);
extern "C" hipError_t ctpwa_launch_to_mixed(const double2*, const double*, long long, int, int, const int*, float2*,
                                             double*, float*, long long, long long, hipStream_t);
extern "C" hipError_t ctpwa_launch_polsym(const double2*, long long, long long, long long, int, unsigned long long*,
                                          hipStream_t);
extern "C" hipError_t ctpwa_launch_prep(const double*, double*, const ctpwa::PrepArgs*, int, hipStream_t);
extern "C" hipError_t ctpwa_launch_finalize(const ctpwa::FinArgs*, hipStream_t);
extern "C" hipError_t ctpwa_launch_prep_batch(const double* const*, double* const*, const ctpwa::PrepArgs*, int, int,
                                              const int*, hipStream_t);
extern "C" hipError_t ctpwa_launch_finalize_batch(const ctpwa::FinArgs*, int, int, size_t, const int*, hipStream_t);
extern "C" hipError_t ctpwa_launch_aux(const ctpwa::AuxArgs*, int, long long, long long, double*, int, hipStream_t);


extern "C" hipError_t ctpwa_launch_zero(double*, long long, hipStream_t);
extern "C" int ctpwa_gram_tables(int, int2*, ctpwa::GramPair*, int*, int*);
extern "C" int ctpwa_gram_nwg(int, int);
extern "C" hipError_t ctpwa_launch_gram_panels(const void*, int, int, long long, const ctpwa::HessPieces*, int, const double*,
                                                double*, hipStream_t);
extern "C" hipError_t ctpwa_launch_gram_wide(const void*, int, int, long long, long long, long long, const double*,
                                              const ctpwa::GramPair*, int, const int2*, const int*, int, int, double*, double*,
                                              int, hipStream_t);
extern "C" hipError_t ctpwa_launch_hess_accum(const ctpwa::HessPieces*, const ctpwa::HessPieces*, const ctpwa::HessTotals*,
                                               const double*, int, const int2*, int, const double*, int, const int2*, int,
                                               const double*, int, int, const int*, hipStream_t);
extern "C" hipError_t ctpwa_launch_partial_int(const ctpwa::AuxArgs*, const int*, const int*, int, long long, long long,
                                               double*, hipStream_t);
extern "C" hipError_t ctpwa_launch_partial_amp(const ctpwa::AuxArgs*, const int*, const int*, int, long long, long long,
                                               double*, hipStream_t);
extern "C" hipError_t ctpwa_launch_gram_to_complex(const double*, int, double*, hipStream_t);
extern "C" hipError_t ctpwa_launch_hess_assemble(const ctpwa::HessAsm*, hipStream_t);

using namespace ctpwa;

static thread_local std::string g_err;

static int fail(const std::string& msg) {
    g_err = msg;
    return 1;
}

#define HIPCHECK(x)                                                                          \
    do {                                                                                     \
        hipError_t e_ = (x);                                                                 \
        if (e_ != hipSuccess) throw std::runtime_error(std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

// ---------------------------------------------------------------------------
// host angular-momentum algebra for the Clebsch-Gordan x Y_lm table
// ---------------------------------------------------------------------------
// factorial with the reference's semantics (src/Amplitude.cu:5-91): exact for
// integers and half-integers up to 11.5, Stirling with two correction terms for
// integers >= 12
static double host_fact(double n) {
    if (n < 0) return 0.0;
    double ri = std::round(n);
    bool is_int = std::fabs(n - ri) < 1e-10;
    if (is_int && ri <= 11) {
        double f = 1.0;
        for (int i = 2; i <= (int)ri; ++i) f *= i;
        return f;
    }
    if (is_int) {
        int m = (int)ri;
        return std::sqrt(2.0 * M_PI * m) * std::pow(m / M_E, m) * (1.0 + 1.0 / (12.0 * m) + 1.0 / (288.0 * m * m));
    }
    if (std::fabs(2 * n - std::round(2 * n)) < 1e-10 && n <= 11.5) {
        int k = (int)std::round(n - 0.5);
        double df = 1.0;
        for (int i = 1; i <= 2 * k + 1; i += 2) df *= i;
        return df / std::pow(2.0, k + 1) * std::sqrt(M_PI);
    }
    return std::tgamma(n);
}

// <j1 m1 j2 m2 | J M> (Racah), arguments as 2j+1 and 2m
static double host_cg(int dj1, int m1x2, int dj2, int m2x2, int dJ, int Mx2) {
    double j1 = (dj1 - 1) / 2.0, j2 = (dj2 - 1) / 2.0, J = (dJ - 1) / 2.0;
    double m1 = m1x2 / 2.0, m2 = m2x2 / 2.0, M = Mx2 / 2.0;
    if (std::fabs(M - m1 - m2) > 1e-10) return 0.0;
    if (J < std::fabs(j1 - j2) || J > j1 + j2) return 0.0;
    if (std::fabs(m1) > j1 || std::fabs(m2) > j2 || std::fabs(M) > J) return 0.0;
    double pre = std::sqrt((2 * J + 1) * host_fact(j1 + j2 - J) * host_fact(j1 - j2 + J) * host_fact(-j1 + j2 + J) /
                           host_fact(j1 + j2 + J + 1));
    pre *= std::sqrt(host_fact(J + M) * host_fact(J - M) * host_fact(j1 - m1) * host_fact(j1 + m1) *
                     host_fact(j2 - m2) * host_fact(j2 + m2));
    int kmin = (int)std::ceil(std::max(0.0, std::max(j2 - J - m1, j1 - J + m2)));
    int kmax = (int)std::floor(std::min(j1 + j2 - J, std::min(j1 - m1, j2 + m2)));
    double s = 0;
    for (int k = kmin; k <= kmax; ++k) {
        double den = host_fact(k) * host_fact(j1 + j2 - J - k) * host_fact(j1 - m1 - k) * host_fact(j2 + m2 - k) *
                     host_fact(J - j2 + m1 + k) * host_fact(J - j1 - m2 + k);
        if (std::fabs(den) > 1e-15) s += ((k & 1) ? -1.0 : 1.0) / den;
    }
    return pre * s;
}

// table entry for amp[s][s1][s2] = qs^L / sqrt(2j+1) <j1 s1 j2 s2|S s1+s2> <S s1+s2 L M|j s>
//   N_LM phase(M) P_L^|M|(cos) e^{-iM phi}:  everything but qs^L, P and the phase factor
static void node_cg_table(const PNode& n, int S, int L, std::vector<double>& out) {
    for (int si = 0; si < n.dj; ++si)
        for (int s1i = 0; s1i < n.dj1; ++s1i)
            for (int s2i = 0; s2i < n.dj2; ++s2i) {
                int s = n.dj - 1 - 2 * si, s1 = n.dj1 - 1 - 2 * s1i, s2 = n.dj2 - 1 - 2 * s2i;
                int Mx2 = s - s1 - s2;
                double v = 0.0;
                if (Mx2 % 2 == 0) {
                    int M = Mx2 / 2, am = std::abs(M);
                    if (am <= L) {
                        double cg1 = host_cg(n.dj1, s1, n.dj2, s2, S, s1 + s2);
                        double cg2 = host_cg(S, s1 + s2, 2 * L + 1, Mx2, n.dj, s);
                        double norm = (L == 0) ? 0.5 * std::sqrt(1.0 / M_PI)
                                               : std::sqrt((2.0 * L + 1.0) * host_fact(L - am) / (4.0 * M_PI * host_fact(L + am)));
                        double ph = (M < 0 && (am & 1)) ? -1.0 : 1.0;
                        v = cg1 * cg2 * norm * ph / std::sqrt((double)n.dj);
                    }
                }
                out.push_back(v);
            }
}

// ---------------------------------------------------------------------------
// generated-kernel cache (one module per device and source text)
// ---------------------------------------------------------------------------
static std::mutex g_mod_mu;
static std::map<std::pair<int, std::string>, hipModule_t> g_mods;

// hipRTC options of the generated kernels: gfx950, and no packed FP32 instructions
// (the same target-feature switch as the library's own hipcc build)
static const char* RTC_OPTS[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=fast",
                                 "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
static const int RTC_NOPTS = (int)(sizeof(RTC_OPTS) / sizeof(RTC_OPTS[0]));

static hipModule_t compile_eval(int device, const std::string& src) {
    std::lock_guard<std::mutex> lk(g_mod_mu);
    auto key = std::make_pair(device, src);
    auto it = g_mods.find(key);
    hipModule_t mod;
    if (it != g_mods.end()) {
        mod = it->second;
    } else {
        hiprtcProgram prog;
        if (hiprtcCreateProgram(&prog, src.c_str(), "ctpwa_eval.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS)
            throw std::runtime_error("hiprtcCreateProgram failed");
        hiprtcResult r = hiprtcCompileProgram(prog, RTC_NOPTS, RTC_OPTS);
        if (r != HIPRTC_SUCCESS) {
            size_t ls = 0;
            hiprtcGetProgramLogSize(prog, &ls);
            std::string log(ls + 1, '\0');
            hiprtcGetProgramLog(prog, &log[0]);
            hiprtcDestroyProgram(&prog);
            throw std::runtime_error("hipRTC compile of the fused kernel failed: " + log);
        }
        size_t cs = 0;
        hiprtcGetCodeSize(prog, &cs);
        std::vector<char> code(cs);
        hiprtcGetCode(prog, code.data());
        hiprtcDestroyProgram(&prog);
        HIPCHECK(hipModuleLoadData(&mod, code.data()));
        g_mods[key] = mod;
    }
    return mod;
}

// ---------------------------------------------------------------------------
// handle
// ---------------------------------------------------------------------------
// upload staging, one per device for the process lifetime: two pinned host buffers and
// two device buffers of STAGE_BYTES (momenta chunks), the mixed form's FP64 batch (grown
// on demand), a stream of default priority and an event per buffer.  Handle creations on
// one device take turns on it.
static const size_t STAGE_BYTES = (size_t)32 << 20;
struct Staging {
    std::mutex mu;
    char* host[2] = {nullptr, nullptr};
    double* dev[2] = {nullptr, nullptr};
    double2* sl64 = nullptr;
    double* inv64 = nullptr;
    size_t n_sl64 = 0, n_inv64 = 0;
    hipStream_t s = nullptr;
    hipEvent_t copied[2] = {nullptr, nullptr};    // the DMA out of host[k] has finished
    void reserve_mixed(size_t nsl, size_t ninv) {
        if (nsl > n_sl64) {
            if (sl64) HIPCHECK(hipFree(sl64));
            sl64 = nullptr;
            HIPCHECK(hipMalloc(&sl64, nsl * sizeof(double2)));
            n_sl64 = nsl;
        }
        if (ninv > n_inv64) {
            if (inv64) HIPCHECK(hipFree(inv64));
            inv64 = nullptr;
            HIPCHECK(hipMalloc(&inv64, ninv * sizeof(double)));
            n_inv64 = ninv;
        }
    }
};
static std::mutex g_stage_mu;
static std::map<int, Staging*> g_stage;
static Staging* staging(int device) {          // called with `device` current
    std::lock_guard<std::mutex> lk(g_stage_mu);
    auto it = g_stage.find(device);
    if (it != g_stage.end()) return it->second;
    Staging* S = new Staging();
    for (int k = 0; k < 2; ++k) {
        HIPCHECK(hipHostMalloc((void**)&S->host[k], STAGE_BYTES, hipHostMallocDefault));
        HIPCHECK(hipMalloc((void**)&S->dev[k], STAGE_BYTES));
        HIPCHECK(hipEventCreateWithFlags(&S->copied[k], hipEventDisableTiming));
    }
    HIPCHECK(hipStreamCreateWithFlags(&S->s, hipStreamNonBlocking));
    for (int k = 0; k < 2; ++k) HIPCHECK(hipEventRecord(S->copied[k], S->s));
    g_stage[device] = S;
    return S;
}

// ---------------------------------------------------------------------------
// matrix-core Gram of ncol columns: tile-pair list, workgroups, partials buffer; more than 64
// columns: panel pairs and each tile pair's panel pair
struct GramTabs {
    int ncol = 0, npp = 0, ntp = 0, nwg = 0;
    GramPair* pp = nullptr;
    int2* tiles = nullptr;
    int* tpair = nullptr;
    double* part = nullptr;
};

// serial numbers of handles: a handle created after another was destroyed may reuse its
// address, never its serial
static std::atomic<unsigned long long> g_handle_serial{0};
// Workspace of a generated per-event kernel with a Gram (the Hessian; the amplitude Gram):
// the kernel, its shape, Jacobian rows of one pass (rows form), u rows, weights, the sums'
// per-workgroup partials, and the Gram partials of the Jacobian (2C columns) and of u
struct GramWS {
    bool ready = false;
    HessShape S;
    hipModule_t mod = nullptr;
    hipFunction_t fn = nullptr, fn_sum = nullptr, fn_theta = nullptr;
    int nz = 0;                          // summed columns
    int* perm = nullptr;                 // put order -> [Z | u] order
    int target = 0;                      // workgroups of the per-event kernel
    long long chunk = 0, cap = 0;        // events of a class per pass, events per pass
    long long ldJ = 0, ldc = 0;
    void* J = nullptr;
    double *U = nullptr, *W = nullptr, *D = nullptr, *z = nullptr;
    GramTabs gJ, gU;
};

struct ctpwa_handle {
    int device = 0;
    const unsigned long long serial = ++g_handle_serial;
    Model_ M;
    long long n[3] = {0, 0, 0}, off[3] = {0, 0, 0}, ntot = 0;
    double Wd = 0, Wb = 0;
    int pw[3] = {0, 0, 0};
    double wc[3] = {1.0, 1.0, 1.0};
    std::vector<void*> allocs;
    double2* sl = nullptr;
    double* inv = nullptr;
    double* wts = nullptr;
    double* table = nullptr;
    double* part = nullptr;
    int nwg = 0, g0[3] = {0, 0, 0}, g1[3] = {0, 0, 0};
    int* wg_cls = nullptr;
    long long* wg_rng = nullptr;
    int nacc = 0;
    int noalloc_nwg = 0;            // workgroups that the no-alloc entry point's limit counts
    PrepArgs prep{};
    FinArgs fin{};
    AuxArgs aux{};
    hipModule_t mod = nullptr;
    hipFunction_t fn_eval = nullptr;       // one likelihood
    hipFunction_t fn_group = nullptr;      // many likelihoods of this model in one launch
    hipFunction_t fn_group_p = nullptr;    // the same, persistent form (graph replays)
    hipFunction_t fn_aux = nullptr;        // amplitudes / intensities (models with Custom lineshapes)
    hipFunction_t fn_custom = nullptr;     // Custom factors and derivatives per event (models with Custom lineshapes)
    double* cfb = nullptr;                 // their per-event rows, [ncustom * ncf][ntot]
    int* wave_ptr = nullptr;               // partial wave w = blocks wave_blk[wave_ptr[w] .. wave_ptr[w+1])
    int* wave_blk = nullptr;
    std::string src;
    // Hessian workspace (allocated on the first ctpwa_hessian call)
    GramWS hess;
    int hnG = 0, hnUu = 0, hNZ = 0;
    double* htot = nullptr;
    int *hzvt = nullptr, *http = nullptr, *httl = nullptr;   // second-part sums of the assembly (HessAsm)
    int *hmap_ptr = nullptr, *hmap_x = nullptr;   // fit parameter -> extended entries (CSR)
    double* hmap_r = nullptr;
    // models with Custom lineshapes: second-order factor rows for the Hessian, from a
    // module compiled on the first Hessian call
    hipModule_t mod2 = nullptr;
    hipFunction_t fn_custom2 = nullptr;
    double* cfb2 = nullptr;
    int *hbcp = nullptr, *hbcl = nullptr;   // per-block Custom factor lists (CSR)
    // amplitude-Gram workspace (allocated on the first ctpwa_amplitude_gram call)
    GramWS agram;
    double* gtot = nullptr;
    // no free resonance parameter: the phase-space amplitude Gram without couplings or
    // theta coefficients, built once at creation; the evaluations then scan data and
    // background only (fin.gram points here)
    double2* d_gram = nullptr;
    std::vector<int> used_inv;
    // storage precision (0 FP64, 1 mixed) and the FP32 stores of the mixed form
    int mixed = 0;
    float2* slf = nullptr;
    float* invf = nullptr;
    int* d_imap = nullptr;
    const void* slp = nullptr;      // the SL store the fused kernel reads
    int* d_psign = nullptr;         // [NU] signs of the mirrored polarisation (folded store)
    unsigned int* fin_done = nullptr;   // finishing-workgroup counter of the final assembly (zero between calls)
    EvStore store() const { return EvStore{sl, slf, inv, invf, d_imap, ntot, mixed, M.npstore(), d_psign}; }

    template <class T>
    T* alloc(size_t count) {
        void* p = nullptr;
        if (count == 0) count = 1;
        // 256 bytes of slack after every buffer: whole 16-byte chunks never end past it
        HIPCHECK(hipMalloc(&p, count * sizeof(T) + 256));
        allocs.push_back(p);
        return (T*)p;
    }
    template <class T>
    T* upload(const std::vector<T>& v) {
        T* p = alloc<T>(v.size());
        if (!v.empty()) HIPCHECK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
        return p;
    }
    ~ctpwa_handle() {
        int prev = 0;
        (void)hipGetDevice(&prev);
        (void)hipSetDevice(device);
        // the modules belong to the process-wide compile cache (shared by handles of one
        // model), not to the handle
        for (void* p : allocs) (void)hipFree(p);
        (void)hipSetDevice(prev);
    }
};

// code-generation options for the fused kernel (tuning; defaults are the measured best)
// code-generation options; the environment overrides them for measurements
static void apply_codegen_env(Model_& M) {
    // next-event loads in registers: measured 4 % faster on the mixed form of a model of
    // about ten amplitudes over four SL tensors (216 of 256 VGPRs without); a larger model
    // has no registers to spare (a 20-amplitude four-body model spills with it)
    M.prefetch_sl = (M.mixed && M.P.namp <= 12 && (int)M.us.size() * M.P.npol <= 8) ? 1 : 0;
    if (const char* e = std::getenv("CTPWA_EVAL_WAVES")) M.min_waves = std::atoi(e);
    if (const char* e = std::getenv("CTPWA_EVAL_LDS")) M.lds_pipe = std::atoi(e) != 0;
    if (const char* e = std::getenv("CTPWA_EVAL_INVTREE")) M.inv_tree = std::atoi(e) != 0;
    if (const char* e = std::getenv("CTPWA_EVAL_PREFETCH")) {
        int d = std::atoi(e);
        if (d < 0 || d > 2) throw std::runtime_error("CTPWA_EVAL_PREFETCH must be 0, 1 or 2");
        M.prefetch_sl = d;
    }
    if (const char* e = std::getenv("CTPWA_EVAL_WGS")) {
        int w = std::atoi(e);
        if (w != 64 && w != 128 && w != 256) throw std::runtime_error("CTPWA_EVAL_WGS must be 64, 128 or 256");
        if (M.groups == 1) M.wgs = w;
    }
}

static void build_tables(ctpwa_handle* h, std::vector<DTopo>& topos, std::vector<DNode>& nodes,
                         std::vector<DKin>& kins, std::vector<DU>& us, std::vector<double>& cgtab,
                         std::vector<DInv>& invs) {
    const Model_& M = h->M;
    const Plan& P = M.P;
    if ((int)M.kin.size() > MAXKIN) throw std::runtime_error("too many distinct kinematic nodes");
    if (P.npol > MAXPOL) throw std::runtime_error("too many polarisation states");
    if (P.nfinal + 1 + MAXNODE > MAXPART) throw std::runtime_error("too many final-state particles");
    kins.resize(M.kin.size());
    for (size_t i = 0; i < M.kin.size(); ++i)
        kins[i] = DKin{M.kin[i].mset, M.kin[i].d1set, M.kin[i].d2set, -1, -1, 0};
    for (size_t t = 0; t < P.topos.size(); ++t) {
        const PTopo& T = P.topos[t];
        DTopo dt{};
        dt.nn = (int)T.nodes.size();
        dt.node0 = (int)nodes.size();
        // daughters-first order of the intermediates
        std::vector<int> order;
        std::function<void(int)> visit = [&](int ref) {
            if (ref >= 0) return;
            int k = -ref - 1;
            visit(T.nodes[k].d1ref);
            visit(T.nodes[k].d2ref);
            if (std::find(order.begin(), order.end(), k) == order.end()) order.push_back(k);
        };
        visit(T.nodes[0].d1ref);
        visit(T.nodes[0].d2ref);
        if ((int)order.size() != dt.nn - 1) throw std::runtime_error("topology has unreachable nodes");
        for (size_t i = 0; i < order.size(); ++i) dt.order[i] = order[i];
        topos.push_back(dt);
        for (size_t k = 0; k < T.nodes.size(); ++k) {
            const PNode& n = T.nodes[k];
            int kin = M.topo_kin[t][k];
            nodes.push_back(DNode{n.dj, n.dj1, n.dj2, n.d1ref, n.d2ref, n.has_bf, n.lmin, kin, n.bf_d, n.mm, n.md1, n.md2});
            if (kins[kin].owner_topo < 0) { kins[kin].owner_topo = (int)t; kins[kin].owner_node = (int)k; }
            if (n.dj1 > 5 || n.dj2 > 5) throw std::runtime_error("daughter spin above 2 is not built");
            // an intermediate daughter's q0 mass must come from a configured mass or a
            // resonance mass parameter (otherwise q0 would depend on the event)
        }
    }
    for (const USpec& U : M.us) {
        DU du{};
        du.topo = U.topo;
        du.mask = (int)U.mask;
        const PTopo& T = P.topos[U.topo];
        for (size_t k = 0; k < T.nodes.size(); ++k) {
            du.S[k] = T.slc[U.slc][k].first;
            du.L[k] = T.slc[U.slc][k].second;
            if (du.L[k] > 7) throw std::runtime_error("orbital angular momentum above 7 is not built");
            du.cg[k] = (int)cgtab.size();
            node_cg_table(T.nodes[k], du.S[k], du.L[k], cgtab);
        }
        us.push_back(du);
    }
    for (const InvSpec& s : M.inv) invs.push_back(DInv{s.kin, s.kind, s.L, 0, s.d, s.ma, s.mb});
}

static void check_q0_masses(const Model_& M) {
    const Plan& P = M.P;
    for (const PBlock& B : P.blocks) {
        if (B.nsl == 0) continue;
        const PTopo& T = P.topos[B.topo];
        for (const PNode& n : T.nodes) {
            for (int side = 0; side < 2; ++side) {
                double cfg = side ? n.md2 : n.md1;
                int ref = side ? n.d2ref : n.d1ref;
                if (cfg > 0) continue;
                if (ref >= 0 && cfg == 0.0) continue;    // massless final-state particle: q0 mass 0
                bool ok = false;
                // an occupying resonance gives its mass parameter, or 1 when it has none
                // (src/AmpGen.cu:1504-1527)
                if (ref < 0)
                    for (const PRes& r : B.res) if (r.node == -ref - 1) ok = true;
                if (!ok) throw std::runtime_error("a daughter without a configured mass and without a resonance mass "
                                                  "parameter makes q0 event-dependent; not built");
            }
        }
    }
}

// Workgroup ranges of the fused kernel: `target` workgroups shared out among the classes by
// event count times cost, each a whole number of `step`-event iterations of one class.
// scan_phsp == false (phase-space term from the stored Gram): the phase space gets none.
// at_most: no more than `target` workgroups in all.
struct Partition {
    std::vector<int> cls;
    std::vector<long long> rng;
    int g0[3] = {0, 0, 0}, g1[3] = {0, 0, 0};
};
static Partition partition(const ctpwa_handle* h, bool scan_phsp, long long target, long long step, double wcost, bool at_most) {
    Partition R;
    const double weff = (scan_phsp ? (double)h->n[0] : 0.0) + wcost * (double)(h->n[1] + h->n[2]);
    for (int c = 0; c < 3; ++c) {
        R.g0[c] = (int)R.cls.size();
        const long long n = (c == 0 && !scan_phsp) ? 0 : h->n[c];
        if (n > 0) {
            const double share = (double)target * ((c == 0 ? 1.0 : wcost) * (double)n) / weff;
            const long long want = std::max<long long>(1, at_most ? (long long)share : (long long)std::llround(share));
            long long chunk = (n + want - 1) / want;
            chunk = ((chunk + step - 1) / step) * step;
            const long long nw = (n + chunk - 1) / chunk;
            for (long long g = 0; g < nw; ++g) {
                R.cls.push_back(c);
                R.rng.push_back(h->off[c] + g * chunk);
                R.rng.push_back(h->off[c] + std::min(n, (g + 1) * chunk));
            }
        }
        R.g1[c] = (int)R.cls.size();
    }
    return R;
}

// scratch of ctpwa_nll_grad_noalloc in doubles, and what its contract (include/ctpwa_amd.h)
// counts for a handle: accumulators of every propagator, workgroups of 256 events.  What it
// accepts is a matter of the model and the event counts, not of the kernel's split.
static const size_t NOALLOC_DOUBLES = (size_t)1 << 18;
static size_t noalloc_contract(const ctpwa_handle* h) {
    const size_t nacc = 1 + 2 * (size_t)h->M.P.namp + (size_t)h->M.nth_all + h->M.cterms.size();
    return nacc * (size_t)std::max(1, h->noalloc_nwg) + 3 * nacc;
}

// The fused kernel's workgroups.  One wave per event (groups == 1): about 1024 (four
// 128-thread workgroups per CU), at least 256 events each.  Wave groups: as many as the chip
// holds at once by the compiled kernel's registers and LDS, at least 128 events each.  Two
// groups of at most 256 registers (25 to 32 amplitudes) fit four times on a CU: one workgroup
// per CU left half of the SIMDs idle (1.4M events, FP64: 26 amplitudes 147 us, four per CU
// 94; 3M events of 25 amplitudes 270 and 144; as one wave 101 and 181).  More of them than
// fit run as further rounds: 31 amplitudes, whose 302 registers allow two per CU, 200 us with
// four and 193 with two; 149 amplitudes, one per CU, 512 us with four and 496 with one, which
// also leaves a quarter of the partial sums to add up.
static void setup_partition(ctpwa_handle* h, bool scan_phsp) {
    const long long nev = (scan_phsp ? h->n[0] : 0) + h->n[1] + h->n[2];
    // relative cost of a data or background event: the workgroups of each class get events
    // in inverse proportion, so that the classes finish together.  A phase-space event costs
    // about 20 FP64 instructions per amplitude (sums and gradient accumulators), 10 per
    // propagator and 8 per SL tensor and polarisation; a data event of a constant-weight
    // class adds the two frexp of the product of intensities, the reciprocal of I and the
    // clamps, about 40 (a class with per-event weights takes a logarithm per event, about
    // 100 more, as the first form of the kernel did for every data event: there the fastest
    // split of the 3-pion model was at 1.3-1.4).  Environment CTPWA_DATA_COST overrides it.
    const Model_& M = h->M;
    const double base = 20.0 * M.P.namp + 10.0 * (double)M.dens.size() + 8.0 * (double)M.us.size() * M.P.npol + 40.0;
    const bool any_pw = (h->n[1] > 0 && h->pw[1]) || (h->n[2] > 0 && h->pw[2]);
    double wcost = 1.0 + (any_pw ? 140.0 : 40.0) / base;
    if (const char* e = std::getenv("CTPWA_DATA_COST")) wcost = std::atof(e);
    if (!(wcost >= 0.25 && wcost <= 4.0)) throw std::runtime_error("CTPWA_DATA_COST must lie in [0.25, 4]");
    const long long t1 = std::min<long long>(1024, std::max<long long>(1, (nev + 255) / 256));
    Partition R;
    if (M.groups > 1) {
        int ncu = 0, per_cu = 0;
        HIPCHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, h->device));
        HIPCHECK(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, h->fn_eval, M.wgs, 0));
        const int fit = ncu * std::max(1, per_cu);
        long long t = std::min<long long>(std::max(4, std::min(fit, 1024)), std::max<long long>(1, (nev + 127) / 128));
        h->noalloc_nwg = (int)partition(h, scan_phsp, t1, 128, wcost, false).cls.size();
        // (some hundred amplitudes: a handle within the contract has to fit into the scratch)
        if (noalloc_contract(h) <= NOALLOC_DOUBLES) t = std::min<long long>(t, (long long)NOALLOC_DOUBLES / h->nacc - 3);
        // (a class too small for a workgroup of its own still gets one)
        for (long long k = t;; --k) {
            R = partition(h, scan_phsp, k, M.ev_step(), wcost, true);
            if ((long long)R.cls.size() <= t || k <= 1) break;
        }
    } else {
        R = partition(h, scan_phsp, t1, M.ev_step(), wcost, false);
        h->noalloc_nwg = (int)R.cls.size();
    }
    for (int c = 0; c < 3; ++c) { h->g0[c] = R.g0[c]; h->g1[c] = R.g1[c]; }
    h->nwg = (int)R.cls.size();
    h->wg_cls = h->upload(R.cls);
    h->wg_rng = h->upload(R.rng);
}

static bool constant_weights(const double* w, long long n, double* c) {
    if (!w || n == 0) { *c = 1.0; return true; }
    for (long long i = 1; i < n; ++i) if (w[i] != w[0]) return false;
    *c = w[0];
    return true;
}

// ---------------------------------------------------------------------------
// ctpwa_nll_grad_noalloc: the per-workgroup partial sums and the class totals of an
// evaluation live in `scratch`, a file-scope device array of NOALLOC_DOUBLES doubles
// (2 MiB) that every GPU the library runs on holds until the process ends, instead of
// the handle's buffers.  Host code never passes the array's name to a kernel (it is a
// host-side stand-in there): each device's own address comes from hipGetSymbolAddress,
// taken once per device with the device current (at ctpwa_create) and kept in g_scratch.
// Every evaluation overwrites what it reads (each workgroup writes its partial row, the
// reduction writes the totals), so nothing needs clearing between calls; calls that
// overlap on one GPU share the array and race.
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];
static std::mutex g_scratch_mu;
static std::map<int, double*> g_scratch;

// the device's copy of `scratch` (call with the device current)
static double* scratch_setup(int device) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto it = g_scratch.find(device);
    if (it != g_scratch.end()) return it->second;
    double* ptr = nullptr;
    hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        throw std::runtime_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch[device] = ptr;
    return ptr;
}
static double* scratch_lookup(int device) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto it = g_scratch.find(device);
    return it == g_scratch.end() ? nullptr : it->second;
}

// After the SL tensors are built: when both polarisations of every SL tensor are mirror
// images over all events (polarisation 1 = sign_u conj(polarisation 0) to 1e-12 of the
// tensor's largest component; spin-0 final states of a J/psi with M = +1, -1), keep only
// polarisation 0 ([NU][1][ld]) and the signs: the kernels then read half the SL bytes.
static void fold_polarisations(ctpwa_handle* h, const unsigned long long* d_sym, int nu, hipStream_t s) {
    std::vector<unsigned long long> raw((size_t)4 * nu);
    HIPCHECK(hipMemcpy(raw.data(), d_sym, raw.size() * sizeof(unsigned long long), hipMemcpyDeviceToHost));
    std::vector<int> sign((size_t)nu, 1);
    for (int u = 0; u < nu; ++u) {
        double dp, dm, m0;
        std::memcpy(&dp, &raw[4 * u + 0], 8);
        std::memcpy(&dm, &raw[4 * u + 1], 8);
        std::memcpy(&m0, &raw[4 * u + 2], 8);
        if (!(std::min(dp, dm) <= 1e-12 * m0) && !(dp == 0.0 || dm == 0.0)) return;   // not mirror images
        sign[u] = (dp <= dm) ? 1 : -1;
    }
    const size_t es = h->mixed ? sizeof(float2) : sizeof(double2);
    void* old = h->mixed ? (void*)h->slf : (void*)h->sl;
    void* neu = h->alloc<unsigned char>((size_t)nu * h->ntot * es);
    for (int u = 0; u < nu; ++u)
        HIPCHECK(hipMemcpyAsync((char*)neu + (size_t)u * h->ntot * es, (const char*)old + (size_t)2 * u * h->ntot * es,
                                (size_t)h->ntot * es, hipMemcpyDeviceToDevice, s));
    HIPCHECK(hipStreamSynchronize(s));
    HIPCHECK(hipFree(old));
    h->allocs.erase(std::remove(h->allocs.begin(), h->allocs.end(), old), h->allocs.end());
    if (h->mixed) h->slf = (float2*)neu; else h->sl = (double2*)neu;
    h->slp = neu;
    h->M.nps = 1;
    h->M.psign = sign;
    h->d_psign = h->upload(sign);
}

static bool fixed_gram_applies(const ctpwa_handle* h);
static void build_fixed_gram(ctpwa_handle* h);

extern "C" int ctpwa_create(const char* plan_text, const double* phsp, long long n_phsp, const double* w_phsp,
                            const double* data, long long n_data, const double* w_data,
                            const double* bkg, long long n_bkg, const double* w_bkg, int precision, int device,
                            ctpwa_handle** out) {
    if (!out) return fail("ctpwa_create: out is NULL");
    *out = nullptr;
    ctpwa_handle* h = nullptr;
    int prev = 0;
    (void)hipGetDevice(&prev);
    try {
        if (!plan_text) throw std::runtime_error("plan_text is NULL");
        if (n_phsp < 0 || n_data < 0 || n_bkg < 0) throw std::runtime_error("negative event count");
        if (n_phsp == 0) throw std::runtime_error("phase-space sample is empty");
        int ndev = 0;
        if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) throw std::runtime_error("no HIP device available");
        if (device < 0 || device >= ndev) throw std::runtime_error("device index out of range");
        HIPCHECK(hipSetDevice(device));
        scratch_setup(device);     // this device's address of the no-alloc entry point's scratch
        h = new ctpwa_handle();
        h->device = device;
        if (precision != 0 && precision != 1) throw std::runtime_error("precision must be 0 (FP64) or 1 (mixed)");
        h->M = derive(parse_plan(plan_text));
        h->M.mixed = precision;
        h->mixed = precision;
        apply_codegen_env(h->M);
        check_q0_masses(h->M);
        const Model_& M = h->M;
        const Plan& P = M.P;
        const double* moms[3] = {phsp, data, bkg};
        const double* ws[3] = {w_phsp, w_data, w_bkg};
        long long ns[3] = {n_phsp, n_data, n_bkg};
        for (int c = 0; c < 3; ++c) {
            h->n[c] = ns[c];
            // class offsets and the leading dimension are multiples of 64 events, so
            // every row of a tile starts 16-byte aligned (the pipelined kernel copies
            // 16-byte chunks)
            h->off[c] = (h->ntot + 63) / 64 * 64;
            h->ntot = h->off[c] + ns[c];
            if (ns[c] > 0 && !moms[c]) throw std::runtime_error("event array is NULL");
        }
        h->ntot = (h->ntot + 63) / 64 * 64;
        // weights: constant per class unless they vary
        std::vector<double> wall;
        bool any_var = false;
        for (int c = 1; c < 3; ++c) {
            double cst;
            if (!constant_weights(ws[c], ns[c], &cst)) { any_var = true; h->pw[c] = 1; }
            h->wc[c] = cst;
        }
        if (ws[0] && n_phsp > 0) {
            double cst;
            if (!constant_weights(ws[0], n_phsp, &cst) || cst != 1.0)
                throw std::runtime_error("phase-space weights are not built (the reference's phase-space mean is unweighted)");
        }
        h->Wd = 0;
        for (long long i = 0; i < n_data; ++i) h->Wd += w_data ? w_data[i] : 1.0;
        h->Wb = 0;
        for (long long i = 0; i < n_bkg; ++i) h->Wb += w_bkg ? w_bkg[i] : 1.0;
        if (any_var) {
            wall.assign(h->ntot, 1.0);
            for (int c = 1; c < 3; ++c)
                if (ws[c]) std::copy(ws[c], ws[c] + ns[c], wall.begin() + h->off[c]);
            h->wts = h->upload(wall);
        }

        std::vector<DTopo> topos;
        std::vector<DNode> nodes;
        std::vector<DKin> kins;
        std::vector<DU> us;
        std::vector<double> cgtab;
        std::vector<DInv> invs;
        build_tables(h, topos, nodes, kins, us, cgtab, invs);
        int nu = (int)us.size(), ninv = (int)invs.size();
        std::vector<int> imap = M.imap();
        int nind = 0, ninf = 0;
        for (int m : imap) (m >= 0 ? nind : ninf)++;
        if (h->mixed) {
            h->slf = h->alloc<float2>((size_t)std::max(1, nu) * P.npol * h->ntot);
            h->inv = h->alloc<double>((size_t)std::max(1, nind) * h->ntot);
            h->invf = h->alloc<float>((size_t)std::max(1, ninf) * h->ntot);
            h->d_imap = h->upload(imap);
            h->slp = h->slf;
        } else {
            h->sl = h->alloc<double2>((size_t)std::max(1, nu) * P.npol * h->ntot);
            h->inv = h->alloc<double>((size_t)std::max(1, ninv) * h->ntot);
            h->slp = h->sl;
        }
        {
            DTopo* d_topos = h->upload(topos);
            DNode* d_nodes = h->upload(nodes);
            DKin* d_kins = h->upload(kins);
            DU* d_us = h->upload(us);
            double* d_cg = h->upload(cgtab);
            int* d_pol = h->upload(P.polmap);
            DInv* d_invs = h->upload(invs);
            const double* d_tabs = h->upload(M.tabs);
            // events class by class, in chunks through the device's staging pool: the
            // host copy of a chunk into pinned memory overlaps the DMA and the init
            // kernel of the previous one; only the pool's stream is waited for
            Staging* S = staging(device);
            std::lock_guard<std::mutex> lk(S->mu);
            const size_t ev_bytes = (size_t)P.nfinal * 4 * sizeof(double);
            const long long chunk = std::max<long long>(1, (long long)(STAGE_BYTES / ev_bytes));
            if (h->mixed) S->reserve_mixed((size_t)std::max(1, nu) * P.npol * chunk, (size_t)std::max(1, ninv) * chunk);
            // two polarisations: check over every event whether they are mirror images
            unsigned long long* d_sym = nullptr;
            if (P.npol == 2 && nu > 0) {
                d_sym = h->alloc<unsigned long long>((size_t)4 * nu);
                HIPCHECK(hipMemsetAsync(d_sym, 0, (size_t)4 * nu * sizeof(unsigned long long), S->s));
            }
            int b = 0;
            for (int c = 0; c < 3; ++c) {
                for (long long s0 = 0; s0 < ns[c]; s0 += chunk) {
                    long long cnt = std::min(chunk, ns[c] - s0);
                    HIPCHECK(hipEventSynchronize(S->copied[b]));      // host[b] free again
                    std::memcpy(S->host[b], moms[c] + (size_t)s0 * P.nfinal * 4, (size_t)cnt * ev_bytes);
                    HIPCHECK(hipMemcpyAsync(S->dev[b], S->host[b], (size_t)cnt * ev_bytes, hipMemcpyHostToDevice, S->s));
                    HIPCHECK(hipEventRecord(S->copied[b], S->s));
                    if (h->mixed) {
                        HIPCHECK(ctpwa_launch_init(S->dev[b], cnt, P.nfinal, d_topos, (int)topos.size(), d_nodes, d_kins,
                                                   (int)kins.size(), d_us, nu, d_cg, d_pol, P.npol, d_invs, ninv, d_tabs,
                                                   S->sl64, S->inv64, cnt, 0, S->s));
                        if (d_sym) HIPCHECK(ctpwa_launch_polsym(S->sl64, cnt, 0, cnt, nu, d_sym, S->s));
                        HIPCHECK(ctpwa_launch_to_mixed(S->sl64, S->inv64, cnt, nu * P.npol, ninv, h->d_imap, h->slf,
                                                       h->inv, h->invf, h->ntot, h->off[c] + s0, S->s));
                    } else {
                        HIPCHECK(ctpwa_launch_init(S->dev[b], cnt, P.nfinal, d_topos, (int)topos.size(), d_nodes, d_kins,
                                                   (int)kins.size(), d_us, nu, d_cg, d_pol, P.npol, d_invs, ninv, d_tabs,
                                                   h->sl, h->inv, h->ntot, h->off[c] + s0, S->s));
                        if (d_sym) HIPCHECK(ctpwa_launch_polsym(h->sl, h->ntot, h->off[c] + s0, cnt, nu, d_sym, S->s));
                    }
                    b ^= 1;
                }
            }
            HIPCHECK(hipStreamSynchronize(S->s));
            if (d_sym) fold_polarisations(h, d_sym, nu, S->s);
        }

        // model tables for prep / finalize / aux
        std::vector<DBlock> blocks;
        std::vector<DRes> res;
        std::vector<int> slcL, slc0;
        std::vector<DDen> dens;
        std::vector<DAmp> amps;
        std::vector<DDenTerms> dterms;
        std::vector<DTerm> terms;
        for (size_t t = 0; t < P.topos.size(); ++t) {
            slc0.push_back((int)(slcL.size() / MAXNODE));
            for (const auto& row : P.topos[t].slc) {
                for (int k = 0; k < MAXNODE; ++k) slcL.push_back(k < (int)row.size() ? row[k].second : 0);
            }
        }
        for (size_t b = 0; b < P.blocks.size(); ++b) {
            const PBlock& B = P.blocks[b];
            DBlock db{};
            db.topo = B.topo;
            db.nloc = (int)M.bvars[b].size();
            db.nres = (int)B.res.size();
            db.res0 = (int)res.size();
            db.nsl = B.nsl;
            db.site = B.site;
            db.nden = (int)M.block_dens[b].size();
            db.den0 = db.nden ? M.block_dens[b][0] : 0;
            for (int i = 0; i < NLOC; ++i) db.vars[i] = i < db.nloc ? M.bvars[b][i] : -1;
            for (size_t k = 1; k < M.block_dens[b].size(); ++k)
                if (M.block_dens[b][k] != db.den0 + (int)k) throw std::runtime_error("denominators of a block are not contiguous");
            blocks.push_back(db);
            for (const PRes& r : B.res) {
                DRes dr{};
                dr.node = r.node;
                dr.model = r.model;
                dr.np = (int)r.params.size();
                dr.nch = (int)r.ch.size() / 2;
                if (dr.np > 6 || dr.nch > 4) throw std::runtime_error("too many lineshape parameters or channels");
                for (int i = 0; i < dr.np; ++i) { dr.p[i] = r.params[i]; dr.slot[i] = r.slots[i]; }
                for (int i = 0; i < 2 * dr.nch; ++i) dr.ch[i] = r.ch[i];
                res.push_back(dr);
            }
        }
        for (const DenSpec& D : M.dens) {
            dens.push_back(DDen{D.block, D.res, D.coef_base, D.ncoef});
            DDenTerms dt{(int)D.re.size(), (int)D.im.size(), (int)terms.size(), D.stat ? 1 : 0};
            for (const Term& t : D.re) terms.push_back(DTerm{t.inv, t.coef, t.cval});
            for (const Term& t : D.im) terms.push_back(DTerm{t.inv, t.coef, t.cval});
            dterms.push_back(dt);
        }
        for (int a = 0; a < P.namp; ++a) {
            const AmpSpec& A = M.amps[a];
            amps.push_back(DAmp{A.block, A.slc, P.amap[a], A.coef_base, A.u, 0, P.aratio[a]});
        }
        DBlock* d_blocks = h->upload(blocks);
        DRes* d_res = h->upload(res);
        DNode* d_nodes2 = h->upload(nodes);
        DTopo* d_topos2 = h->upload(topos);
        int* d_slcL = h->upload(slcL);
        int* d_slc0 = h->upload(slc0);
        DDen* d_dens = h->upload(dens);
        DAmp* d_amps = h->upload(amps);
        DDenTerms* d_dterms = h->upload(dterms);
        DTerm* d_terms = h->upload(terms);
        int* d_gslot = h->upload(P.g_slot);
        double* d_gmu = h->upload(P.g_mu);
        double* d_gsig = h->upload(P.g_sig);
        h->table = h->alloc<double>(M.table_size());
        HIPCHECK(hipMemset(h->table, 0, M.table_size() * sizeof(double)));

        h->src = generate_eval_kernel(M);
        h->mod = compile_eval(device, h->src);
        HIPCHECK(hipModuleGetFunction(&h->fn_eval, h->mod, "ctpwa_eval"));
        HIPCHECK(hipModuleGetFunction(&h->fn_group, h->mod, "ctpwa_eval_group"));
        HIPCHECK(hipModuleGetFunction(&h->fn_group_p, h->mod, "ctpwa_eval_group_persist"));

        h->nacc = M.nacc();
        const bool use_gram = fixed_gram_applies(h);
        setup_partition(h, !use_gram);
        h->part = h->alloc<double>((size_t)h->nacc * std::max(1, h->nwg));
        h->fin_done = h->alloc<unsigned int>(1);
        HIPCHECK(hipMemset(h->fin_done, 0, sizeof(unsigned int)));

        h->prep = PrepArgs{d_blocks, d_res, d_nodes2, d_topos2, d_slcL, d_slc0, d_dens, d_amps,
                           (int)dens.size(), P.namp, P.nfree, P.ntheta,
                           (long long)M.off_v(), (long long)M.off_c(), (long long)M.off_rec(),
                           (long long)M.off_th(), (long long)M.off_lth(), 0};
        h->fin = FinArgs{};
        h->fin.part = h->part;
        h->fin.done = h->fin_done;
        h->fin.nwg = h->nwg;
        h->fin.nacc = h->nacc;
        for (int c = 0; c < 3; ++c) { h->fin.g0[c] = h->g0[c]; h->fin.g1[c] = h->g1[c]; }
        h->fin.table = h->table;
        h->fin.off_v = (long long)M.off_v();
        h->fin.off_rec = (long long)M.off_rec();
        h->fin.amps = d_amps;
        h->fin.blocks = d_blocks;
        {
            std::vector<DThTerm> th;
            for (const ThTerm& t : M.thterms) th.push_back(DThTerm{M.dens[t.den].block, M.dens[t.den].coef_base + t.coef});
            h->fin.thterms = h->upload(th);
            h->fin.nth = (int)th.size();
            // CSR lists of the gradient contractions (see DGEnt)
            auto local = [&](int b, int j) {
                for (int i = 0; i < blocks[b].nloc; ++i) if (blocks[b].vars[i] == j) return i;
                return -1;
            };
            std::vector<int> thp{0}, cpp{0};
            std::vector<DGEnt> the, cpe;
            for (int j = 0; j < P.ntheta; ++j) {
                for (size_t t = 0; t < th.size(); ++t) {
                    int li = local(th[t].block, j);
                    if (li >= 0) the.push_back(DGEnt{1 + 2 * P.namp + (int)t, th[t].rec * REC + 1 + li, -2.0});
                }
                for (int a = 0; a < P.namp; ++a) {
                    int li = local(amps[a].block, j);
                    if (li >= 0) the.push_back(DGEnt{-a - 1, amps[a].rec * REC + 1 + li, 2.0});
                }
                // Custom factors: accumulated Re(z dPsi/dtheta_j) directly (no coefficient record)
                for (size_t t = 0; t < M.cterms.size(); ++t) {
                    const CTerm& T = M.cterms[t];
                    if (M.bvars[M.customs[T.custom].block][T.local] == j)
                        the.push_back(DGEnt{1 + 2 * P.namp + (int)th.size() + (int)t, -1, 2.0});
                }
                thp.push_back((int)the.size());
            }
            for (int fi = 0; fi < P.nfree; ++fi) {
                for (int a = 0; a < P.namp; ++a)
                    if (amps[a].freeidx == fi) cpe.push_back(DGEnt{a, amps[a].rec * REC, amps[a].ratio});
                cpp.push_back((int)cpe.size());
            }
            if (the.empty()) the.push_back(DGEnt{0, 0, 0.0});
            if (cpe.empty()) cpe.push_back(DGEnt{0, 0, 0.0});
            h->fin.thp = h->upload(thp);
            h->fin.the = h->upload(the);
            h->fin.cpp = h->upload(cpp);
            h->fin.cpe = h->upload(cpe);
            h->fin.nthe = (int)the.size();
            h->fin.ncpe = (int)cpe.size();
            h->fin.nacc = h->nacc;
            h->fin.nfree = P.nfree;
            h->fin.ntheta = P.ntheta;
            if (assemble_lds_bytes(h->fin) > 60 * 1024)
                throw std::runtime_error("too many gradient accumulators for the assembly kernel");
        }
        h->fin.namp = P.namp;
        h->fin.nfree = P.nfree;
        h->fin.ntheta = P.ntheta;
        h->fin.ngauss = (int)P.g_slot.size();
        h->fin.g_slot = d_gslot;
        h->fin.g_mu = d_gmu;
        h->fin.g_sig = d_gsig;
        h->fin.Np = (double)n_phsp;
        h->fin.Wd = h->Wd;
        h->fin.Wb = h->Wb;
        h->fin.totals = h->alloc<double>((size_t)3 * h->nacc);
        h->aux = AuxArgs{h->store(), h->table, (long long)M.off_c(), (long long)M.off_rec(),
                         d_amps, d_blocks, d_dens, d_dterms, d_terms, P.namp, P.npol};
        {
            std::vector<int> bcp(1, 0), bcl;
            for (size_t b = 0; b < P.blocks.size(); ++b) {
                for (int c : M.block_customs[b]) bcl.push_back(c);
                bcp.push_back((int)bcl.size());
            }
            h->hbcp = h->upload(bcp);
            h->hbcl = h->upload(bcl);
            h->aux.bcp = h->hbcp;
            h->aux.bcl = h->hbcl;
            h->aux.cld = h->ntot;
            h->aux.ncf = M.customs.empty() ? 0 : M.ncf();
        }
        {
            std::vector<int> wptr(P.nwave + 1, 0), wblk;
            for (int w = 0; w < P.nwave; ++w) {
                for (size_t b = 0; b < P.blocks.size(); ++b)
                    if (P.bwave[b] == w) wblk.push_back((int)b);
                wptr[w + 1] = (int)wblk.size();
            }
            h->wave_ptr = h->upload(wptr);
            h->wave_blk = h->upload(wblk);
        }

        if (!M.customs.empty()) {
            HIPCHECK(hipModuleGetFunction(&h->fn_aux, h->mod, "ctpwa_aux"));
            HIPCHECK(hipModuleGetFunction(&h->fn_custom, h->mod, "ctpwa_custom"));
            h->cfb = h->alloc<double>((size_t)M.customs.size() * M.ncf() * h->ntot);
            h->aux.cfb = h->cfb;
        }
        h->used_inv.assign(M.inv.size(), 0);
        for (const DenSpec& D : M.dens) {
            for (const Term& t : D.re) if (t.inv >= 0) h->used_inv[t.inv] = 1;
            for (const Term& t : D.im) if (t.inv >= 0) h->used_inv[t.inv] = 1;
        }
        if (use_gram) build_fixed_gram(h);
        HIPCHECK(hipStreamSynchronize(nullptr));
        (void)hipSetDevice(prev);
        *out = h;
        return 0;
    } catch (const std::exception& e) {
        delete h;
        (void)hipSetDevice(prev);
        return fail(std::string("ctpwa_create: ") + e.what());
    }
}

extern "C" void ctpwa_destroy(ctpwa_handle* h) { delete h; }

extern "C" int ctpwa_dims(const ctpwa_handle* h, int* n_amp, int* n_free, int* n_theta, int* n_pol) {
    if (!h) return fail("ctpwa_dims: NULL handle");
    if (n_amp) *n_amp = h->M.P.namp;
    if (n_free) *n_free = h->M.P.nfree;
    if (n_theta) *n_theta = h->M.P.ntheta;
    if (n_pol) *n_pol = h->M.P.npol;
    return 0;
}

extern "C" int ctpwa_param_info(const ctpwa_handle* h, double* init, double* lower, double* upper) {
    if (!h) return fail("ctpwa_param_info: NULL handle");
    const Plan& P = h->M.P;
    for (int j = 0; j < P.ntheta; ++j) {
        if (init) init[j] = P.th_init[j];
        if (lower) lower[j] = P.th_lo[j];
        if (upper) upper[j] = P.th_hi[j];
    }
    return 0;
}

// Custom factors of every stored event at the parameter point the table holds
static hipError_t launch_custom(ctpwa_handle* h, hipStream_t s) {
    if (!h->fn_custom) return hipSuccess;
    void* args[] = {&h->table, &h->inv, &h->invf, &h->ntot, &h->cfb};
    unsigned grid = (unsigned)std::min<long long>(4096, (h->ntot + 255) / 256);
    return hipModuleLaunchKernel(h->fn_custom, grid, 1, 1, 256, 1, 1, 0, s, args, nullptr);
}

static hipError_t launch_eval(ctpwa_handle* h, hipStream_t s, double* part = nullptr) {
    if (h->nwg <= 0) return hipSuccess;       // stored phase-space Gram and no data events
    double* pp = part ? part : h->part;
    void* args[] = {&h->table, &h->slp, &h->inv, &h->invf, &h->wts, &pp, &h->wg_cls, &h->wg_rng, &h->ntot,
                    &h->nwg, &h->wc[1], &h->wc[2], &h->pw[1], &h->pw[2], &h->cfb};
    return hipModuleLaunchKernel(h->fn_eval, h->nwg, 1, 1, h->M.wgs, 1, 1, 0, s, args, nullptr);
}


struct DeviceGuard {
    int prev = 0;
    explicit DeviceGuard(int dev) { (void)hipGetDevice(&prev); (void)hipSetDevice(dev); }
    ~DeviceGuard() { (void)hipSetDevice(prev); }
};

extern "C" int ctpwa_nll_grad(ctpwa_handle* h, const double* params_dev, double* out_dev, void* stream) {
    if (!h || !params_dev || !out_dev) return fail("ctpwa_nll_grad: NULL argument");
    DeviceGuard g(h->device);
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = ctpwa_launch_prep(params_dev, h->table, &h->prep, 2, s);
    if (e == hipSuccess) e = launch_custom(h, s);
    if (e == hipSuccess) e = launch_eval(h, s);
    if (e == hipSuccess) {
        h->fin.params = params_dev;
        h->fin.out = out_dev;
        e = ctpwa_launch_finalize(&h->fin, s);
    }
    if (e != hipSuccess) return fail(std::string("ctpwa_nll_grad: ") + hipGetErrorString(e));
    return 0;
}

extern "C" int ctpwa_nll_grad_noalloc(ctpwa_handle* h, const double* params_dev, double* out_dev, void* stream) {
    if (!h || !params_dev || !out_dev) return fail("ctpwa_nll_grad_noalloc: NULL argument");
    const size_t need = std::max(noalloc_contract(h), (size_t)h->nacc * (size_t)std::max(1, h->nwg) + 3 * (size_t)h->nacc);
    if (need > NOALLOC_DOUBLES)
        return fail("ctpwa_nll_grad_noalloc: the evaluation needs " + std::to_string(need) +
                    " doubles of scratch, more than the " + std::to_string(NOALLOC_DOUBLES) + " it holds");
    DeviceGuard g(h->device);
    double* scr = scratch_lookup(h->device);
    if (!scr) return fail("ctpwa_nll_grad_noalloc: no scratch address for this device");
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = ctpwa_launch_prep(params_dev, h->table, &h->prep, 2, s);
    if (e == hipSuccess) e = launch_custom(h, s);
    if (e == hipSuccess) e = launch_eval(h, s, scr);
    if (e == hipSuccess) {
        FinArgs f = h->fin;
        f.part = scr;
        f.totals = scr + (size_t)h->nacc * (size_t)std::max(1, h->nwg);
        f.params = params_dev;
        f.out = out_dev;
        e = ctpwa_launch_finalize(&f, s);
    }
    if (e != hipSuccess) return fail(std::string("ctpwa_nll_grad_noalloc: ") + hipGetErrorString(e));
    return 0;
}


// bytes of rows per pass: 2 GiB of Jacobian rows, 256 MiB of the amplitude Gram's, which a
// handle keeps besides (environment CTPWA_HESS_JBYTES overrides it for measurements)
static long long hess_jbytes(bool amps_only) {
    const long long most = amps_only ? 256LL << 20 : 2LL << 30;
    if (const char* e = std::getenv("CTPWA_HESS_JBYTES")) {
        long long v = std::atoll(e);
        if (v >= (1LL << 20)) return amps_only ? std::min(v, most) : v;
    }
    return most;
}
static long long up(long long x, long long m) { return (x + m - 1) / m * m; }
// Sizes of a GramWS for the classes' event counts: events of one class per pass (chunk, a
// multiple of 256), events of all classes per pass (cap), workgroups (occ: of the compiled
// kernel on a CU, 0 for an estimate), and the buffers in doubles
struct GramSizes {
    long long chunk, cap, ldJ, ldc, J, U, W, D, z, part;     // ldJ, ldc: rows of J and of U, W, D
    int target, nz;
};
// the partials of a Gram: ncol <= 64 at least one workgroup per piece; more columns: two
// workgroups per CU shared out among the panel pairs by a wave's tile pairs
static long long gram_plan(int ncol, bool f32, int ncu, std::vector<GramPair>* pairs, int* nwg) {
    int np = 0;
    const int ntp = ctpwa_gram_tables(ncol, nullptr, nullptr, &np, nullptr);
    if (ncol <= 64) {
        *nwg = ctpwa_gram_nwg(f32, ncol);
        return (long long)*nwg * ntp * 256;
    }
    std::vector<GramPair> pp((size_t)np);
    ctpwa_gram_tables(ncol, nullptr, pp.data(), &np, nullptr);
    const int budget = std::max(2 * ncu, np);
    int cost = 0;
    for (const GramPair& p : pp) cost += p.nq;
    long long off = 0;
    int s0 = 0;
    for (GramPair& p : pp) {
        p.s0 = s0;
        p.ns = std::max(1, (int)((long long)budget * p.nq / cost));
        p.off = off;
        s0 += p.ns;
        off += (long long)p.ns * p.nt;
    }
    *nwg = s0;
    if (pairs) *pairs = pp;
    return off * 256;
}
static GramSizes gram_sizes(const Model_& M, const HessShape& S, const long long n3[3], int ncu, int occ) {
    GramSizes z{};
    const long long row = (long long)M.P.npol * 2 * S.C * 8;
    // (a row's byte offset in its column is a 32-bit number in the generated kernel)
    z.chunk = std::max<long long>(256, std::min<long long>(1 << 28, hess_jbytes(S.NU == 0) / row / 256 * 256));
    const long long all = n3[0] + n3[1] + n3[2];
    z.cap = std::max<long long>(1, std::min(all, z.chunk));
    // (split rows: one-wave workgroups, as many times over as there are sets; 2 or 8 per CU and
    // set are 2 % slower)
    // (rows: what the compiled kernel's registers and LDS allow, or for an estimate the LDS and 32
    // waves.  With no more than two waves per SIMD, 3M events, mixed: 7 amplitudes, six workgroups
    // of two waves, 627 us, now 570; 13 amplitudes, three of four, 1092 and 1018.  Fused: two
    // waves per SIMD; 49 to 64 columns take 512 registers and run one wave at a time, in two
    // rounds of half the events, which is no slower than one round)
    const int fit = (int)std::min<long long>((S.fused ? 8 : 32) / S.G, 160 * 1024 / std::max<long long>(1, S.lds * 8));
    const int per_cu = S.split ? 4 : std::max(1, occ > 0 && !S.fused ? occ : fit);
    // never more than fit on the chip at once (four workgroups over, for classes smaller than
    // a share, ran as a second round: the mixed form's Gram of 3.05M events 611 us, not 310);
    // at least one for each of up to four pieces
    z.target = (int)std::max<long long>(4, std::min<long long>((long long)ncu * per_cu, (all + 63) / 64 + 3));
    z.nz = S.NU > 0 ? hess_nz(M) + S.NU : 0;
    z.z = (long long)z.nz * z.target;
    if (S.fused) {
        z.chunk = std::max<long long>(1, all);
        z.cap = all;
        const int gt = (2 * S.C + 15) / 16, ut = (S.NU + 15) / 16;
        z.part = (long long)z.target * (gt * (gt + 1) / 2 + ut * (ut + 1) / 2) * 256;
        return z;
    }
    z.ldJ = up((long long)M.P.npol * z.cap + 4 * 32, 32);
    z.ldc = up(z.cap + 4 * 64, 64);
    z.J = z.ldJ * 2 * S.C;
    z.U = z.ldc * S.NU;
    z.W = z.ldc * (S.split && S.NU > 0 ? 2 + 2 * M.P.npol : 2);
    z.D = S.split ? z.ldc * S.nslot * 2 * M.P.npol : 0;
    int nwg = 0;
    z.part = gram_plan(2 * S.C, S.f32, ncu, nullptr, &nwg) + (S.NU > 0 ? gram_plan(S.NU, false, ncu, nullptr, &nwg) : 0);
    return z;
}
static int device_cus(int device) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0) return 256;
    return n;
}
static long long hess_workspace_bytes(const Model_& M0, const long long n3[3], long long ntot) {
    long long most = 0;
    for (int mixed = 0; mixed < 2; ++mixed) {       // the larger of the two storage forms
        Model_ M = M0;
        M.mixed = mixed;
        const HessShape S = hess_shape(M, false);
        const GramSizes z = gram_sizes(M, S, n3, 256, 0);
        const long long nG = (long long)(2 * S.C) * (2 * S.C + 1) / 2, nUu = (long long)S.NU * (S.NU + 1) / 2;
        long long w = 3 * (nG + nUu + z.nz) + (S.f32 ? z.J / 2 : z.J) + z.U + z.W + z.D + z.z + z.part;
        w += (long long)M.P.ntheta * M.P.ntheta * 4 + (long long)M.P.namp * M.P.ntheta;      // index tables
        w += (long long)M.customs.size() * M.ncf2() * ntot;   // second-order Custom factor rows
        most = std::max(most, w);
    }
    return most * 8 + 64 * 1024;    // + the smaller tables and allocation slack
}

// the amplitude Gram's workspace for classes of up to n events
static long long agram_workspace_bytes(const Model_& M, long long n) {
    const long long n3[3] = {n, 0, 0};
    const HessShape S = hess_shape(M, true);
    const GramSizes z = gram_sizes(M, S, n3, 256, 0);
    return (z.J + z.U + z.W + z.D + z.z + z.part + (long long)M.P.namp * (2 * M.P.namp + 1)) * 8;
}

// nwg > 0: the fused form's workgroups, each with its tile pairs' sums
static void gram_setup(ctpwa_handle* h, GramTabs& g, int ncol, bool f32, int nwg) {
    g.ncol = ncol;
    g.ntp = ctpwa_gram_tables(ncol, nullptr, nullptr, &g.npp, nullptr);
    std::vector<int2> tiles((size_t)g.ntp);
    std::vector<int> tpair((size_t)g.ntp);
    ctpwa_gram_tables(ncol, tiles.data(), nullptr, &g.npp, tpair.data());
    std::vector<GramPair> pp;
    long long part = gram_plan(ncol, f32, device_cus(h->device), &pp, &g.nwg);
    if (nwg > 0) {
        g.nwg = nwg;
        part = (long long)nwg * g.ntp * 256;
    }
    g.pp = h->upload(pp);
    g.tiles = h->upload(tiles);
    g.tpair = h->upload(tpair);
    g.part = h->alloc<double>((size_t)part);
}

static void gramws_setup(ctpwa_handle* h, GramWS& w, bool amps_only, const long long n3[3]) {
    const Model_& M = h->M;
    w.S = hess_shape(M, amps_only);
    std::vector<int> perm;
    w.mod = compile_eval(h->device, generate_hess_kernel(M, &perm, amps_only));
    HIPCHECK(hipModuleGetFunction(&w.fn, w.mod, amps_only ? "ctpwa_amp_gram" : w.S.fused ? "ctpwa_hess_fused" : "ctpwa_hess_rows"));
    if (w.S.split && !amps_only) {
        HIPCHECK(hipModuleGetFunction(&w.fn_sum, w.mod, "ctpwa_hess_sum"));
        HIPCHECK(hipModuleGetFunction(&w.fn_theta, w.mod, "ctpwa_hess_theta"));
    }
    int occ = 0;
    HIPCHECK(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&occ, w.fn, w.S.split ? 64 : 64 * w.S.G, 0));
    const GramSizes z = gram_sizes(M, w.S, n3, device_cus(h->device), occ);
    if ((int)perm.size() != z.nz) throw std::runtime_error("Hessian: summed-column count mismatch");
    w.perm = h->upload(perm);
    w.nz = z.nz;
    w.target = z.target;
    w.chunk = z.chunk;
    w.cap = z.cap;
    w.ldJ = z.ldJ;
    w.ldc = z.ldc;
    w.z = h->alloc<double>((size_t)z.z);
    if (!w.S.fused) {
        w.J = h->alloc<unsigned char>((size_t)z.J * (w.S.f32 ? sizeof(float) : sizeof(double)));
        w.U = h->alloc<double>((size_t)z.U);
        w.D = h->alloc<double>((size_t)z.D);
        // the amplitude Gram weights every row by one
        w.W = amps_only ? h->upload(std::vector<double>((size_t)z.W, 1.0)) : h->alloc<double>((size_t)z.W);
    }
    gram_setup(h, w.gJ, 2 * w.S.C, w.S.f32, w.S.fused ? z.target : 0);
    if (w.S.NU > 0) gram_setup(h, w.gU, w.S.NU, false, w.S.fused ? z.target : 0);
    w.ready = true;
}

// shares out `target` workgroups among k pieces of the given costs, at least one each, at
// most `target` in all (target >= k)
static std::vector<int> share_out(const std::vector<double>& cost, int target) {
    double all = 0.0;
    for (double c : cost) all += c;
    std::vector<int> n(cost.size(), 1);
    const int spare = target - (int)cost.size();
    for (size_t k = 0; k < cost.size(); ++k) n[k] += (int)(spare * (all > 0 ? cost[k] / all : 0.0));
    return n;
}

// Runs a GramWS over the classes with use[c]: passes of up to four pieces (a piece: up to
// `chunk` events of one class), each the per-event kernel, in the rows form the Gram kernels
// over its rows, and the sums, which go to T
static void gramws_run(ctpwa_handle* h, GramWS& w, const bool use[3], HessTotals T, const double* cfr, int withK, hipStream_t s) {
    const Model_& M = h->M;
    const int NP = M.P.npol;
    struct Piece { int c; long long s0, cnt; };
    std::vector<Piece> todo;
    for (int c = 0; c < 3; ++c)
        for (long long s0 = 0; use[c] && s0 < h->n[c]; s0 += w.chunk) todo.push_back({c, s0, std::min(w.chunk, h->n[c] - s0)});
    bool seen[3] = {false, false, false};
    for (size_t at = 0; at < todo.size();) {
        HessPieces H{}, HU{};
        long long ev = 0, row = 0, wr = 0;
        while (at < todo.size() && H.n < 4 && (H.n == 0 || ev + todo[at].cnt <= w.cap)) {
            const Piece& p = todo[at];
            const int k = H.n;
            // (a class may have one piece per pass: its sums then have one writer)
            if (k > 0 && H.cls[k - 1] == p.c) break;
            H.cls[k] = p.c;
            H.e0[k] = h->off[p.c] + p.s0;
            H.cnt[k] = p.cnt;
            H.row0[k] = row;
            H.w0[k] = wr;
            ev += p.cnt;
            row += up(NP * p.cnt, 32);          // every piece's rows start 16-byte aligned
            wr += up(p.cnt, 64);           // (a last wave's idle lanes write there)
            ++H.n;
            ++at;
        }
        if (!w.S.fused && (row > w.ldJ || wr > w.ldc)) throw std::runtime_error("Hessian: a pass exceeds its buffers");
        // data and background events also have a u row (and in the fused form its Gram)
        std::vector<double> ce, cr, cu;
        for (int k = 0; k < H.n; ++k) {
            ce.push_back((double)H.cnt[k] * (H.cls[k] != 0 ? 1.2 : 1.0));
            cr.push_back((double)H.cnt[k]);
        }
        const std::vector<int> we = share_out(ce, w.target);
        const std::vector<int> gs = w.S.fused ? we : share_out(cr, w.gJ.nwg);
        int g0 = 0;
        for (int k = 0; k < H.n; ++k) {
            const long long steps = (H.cnt[k] + 63) / 64;
            H.spw[k] = (int)((steps + we[k] - 1) / we[k]);
            H.wg0[k + 1] = H.wg0[k] + (int)((steps + H.spw[k] - 1) / H.spw[k]);
            if (w.S.fused) {
                H.glo[k] = H.wg0[k];
                H.ghi[k] = H.wg0[k + 1];
            } else {
                H.glo[k] = g0;
                g0 += gs[k];
                H.ghi[k] = g0;
            }
        }
        for (int k = 0; k < H.n && w.S.NU > 0; ++k) {
            if (H.cls[k] == 0) continue;
            const int q = HU.n++;
            HU.cls[q] = H.cls[k];
            HU.cnt[q] = H.cnt[k];
            HU.row0[q] = HU.w0[q] = H.w0[k];
            HU.glo[q] = H.glo[k];
            HU.ghi[q] = H.ghi[k];
            cu.push_back((double)H.cnt[k]);
        }
        if (!w.S.fused && HU.n > 0) {
            const std::vector<int> us = share_out(cu, w.gU.nwg);
            for (int q = 0, u0 = 0; q < HU.n; ++q) {
                HU.glo[q] = u0;
                u0 += us[q];
                HU.ghi[q] = u0;
            }
        }
        int nwg = H.wg0[H.n];
        if (nwg > w.target) throw std::runtime_error("Hessian: more workgroups than partials");
        double* gp = w.gJ.part;
        double* upart = w.gU.part;
        void* args[] = {&h->table, (void*)&h->slp, &h->inv, &h->invf, &h->ntot, &h->wts, &h->wc[1], &h->wc[2], &h->pw[1], &h->pw[2],
                        &H, &w.J, &w.ldJ, &w.U, &w.W, &w.D, &w.ldc, &gp, &upart, &w.z, &nwg, (void*)&cfr, &h->ntot, &withK};
        if (w.fn_sum) HIPCHECK(hipModuleLaunchKernel(w.fn_sum, nwg, 1, 1, 64 * (unsigned)w.S.sum_blocks.size(), 1, 1, 0, s, args, nullptr));
        if (w.S.split) HIPCHECK(hipModuleLaunchKernel(w.fn, nwg, w.S.G, 1, 64, 1, 1, 0, s, args, nullptr));
        else HIPCHECK(hipModuleLaunchKernel(w.fn, nwg, 1, 1, 64 * w.S.G, 1, 1, 0, s, args, nullptr));
        if (w.fn_theta) HIPCHECK(hipModuleLaunchKernel(w.fn_theta, nwg, 1, 1, 64, 1, 1, 0, s, args, nullptr));
        for (int c = 0; c < 3; ++c) T.first[c] = !seen[c];
        for (int k = 0; k < H.n; ++k) seen[H.cls[k]] = true;
        // Grams of up to 64 columns: one launch for all pieces, summed with the columns below;
        // wider ones: a launch and its sums per piece
        const bool jw = !w.S.fused && w.gJ.ncol > 64, uw = !w.S.fused && w.gU.ncol > 64;
        const size_t es = w.S.f32 ? sizeof(float) : sizeof(double);
        if (jw) {
            for (int k = 0; k < H.n; ++k)
                HIPCHECK(ctpwa_launch_gram_wide((const char*)w.J + (size_t)H.row0[k] * es, w.S.f32, w.gJ.ncol, w.ldJ, NP * H.cnt[k],
                                                H.cnt[k], w.W + H.w0[k], w.gJ.pp, w.gJ.npp, w.gJ.tiles, w.gJ.tpair, w.gJ.ntp,
                                                w.gJ.nwg, w.gJ.part, T.G[H.cls[k]], T.first[H.cls[k]], s));
        } else if (!w.S.fused) {
            HIPCHECK(ctpwa_launch_gram_panels(w.J, w.S.f32, w.gJ.ncol, w.ldJ, &H, NP, w.W, w.gJ.part, s));
        }
        if (uw) {
            for (int q = 0; q < HU.n; ++q)
                HIPCHECK(ctpwa_launch_gram_wide(w.U + HU.row0[q], 0, w.gU.ncol, w.ldc, HU.cnt[q], HU.cnt[q], w.W + w.ldc + HU.w0[q],
                                                w.gU.pp, w.gU.npp, w.gU.tiles, w.gU.tpair, w.gU.ntp, w.gU.nwg, w.gU.part,
                                                T.Uu[HU.cls[q]], T.first[HU.cls[q]], s));
        } else if (!w.S.fused && HU.n > 0) {
            HIPCHECK(ctpwa_launch_gram_panels(w.U, 0, w.gU.ncol, w.ldc, &HU, 1, w.W + w.ldc, w.gU.part, s));
        }
        if (jw && w.nz == 0 && (uw || w.S.NU == 0)) continue;
        HIPCHECK(ctpwa_launch_hess_accum(&H, &HU, &T, w.gJ.part, jw ? 0 : w.gJ.ntp, w.gJ.tiles, w.gJ.ncol, w.gU.part,
                                         uw || w.S.NU == 0 ? 0 : w.gU.ntp, w.gU.tiles, w.S.NU, w.z, w.nz, nwg, w.perm, s));
    }
}

static void hess_setup(ctpwa_handle* h) {
    const Model_& M = h->M;
    const Plan& P = M.P;
    if (P.ntheta > 64) throw std::runtime_error("Hessian: more than 64 free resonance parameters is not built");
    gramws_setup(h, h->hess, false, h->n);
    const HessShape& S = h->hess.S;
    h->hNZ = hess_nz(M);
    h->hnG = 2 * S.C * (2 * S.C + 1) / 2;
    h->hnUu = S.NU * (S.NU + 1) / 2;
    h->hess.ready = false;              // until the tables below exist
    // totals: per class G, Uu, Z, g
    h->htot = h->alloc<double>((size_t)3 * (h->hnG + h->hnUu + h->hNZ + S.NU));
    // second-part sums: per block its (amplitude, local parameter) pairs of reals, then its
    // upper triangle of parameter pairs
    {
        const int n = P.namp, T = P.ntheta;
        std::vector<int> zvt((size_t)n * T, -1), ttp(1, 0), ttl;
        std::vector<std::vector<int>> tt((size_t)T * T);
        int z = 0;
        for (size_t b = 0; b < P.blocks.size(); ++b) {
            if (P.blocks[b].nsl == 0) continue;
            const std::vector<int>& v = M.bvars[b];
            const int nl = (int)v.size();
            for (int a = P.blocks[b].site; a < P.blocks[b].site + P.blocks[b].nsl; ++a)
                for (int i = 0; i < nl; ++i, z += 2) zvt[(size_t)a * T + v[i]] = z;
            for (int i = 0; i < nl; ++i)
                for (int k = i; k < nl; ++k, ++z) {
                    tt[(size_t)v[i] * T + v[k]].push_back(z);
                    if (v[i] != v[k]) tt[(size_t)v[k] * T + v[i]].push_back(z);
                }
        }
        if (z != h->hNZ - 1) throw std::runtime_error("Hessian: second-part sum count mismatch");
        for (const std::vector<int>& l : tt) {
            ttl.insert(ttl.end(), l.begin(), l.end());
            ttp.push_back((int)ttl.size());
        }
        h->hzvt = h->upload(zvt);
        h->http = h->upload(ttp);
        h->httl = h->upload(ttl);
    }
    // fit parameter -> extended entries: [Re p_f] -> Re v_a, [Im p_f] -> Im v_a with
    // v_a = r_a p_f(a); theta_j -> theta_j
    {
        const int nf = P.nfree, np = 2 * nf + P.ntheta;
        std::vector<int> ptr(np + 1, 0), xs;
        std::vector<double> rs;
        for (int q = 0; q < np; ++q) {
            if (q >= 2 * nf) {
                xs.push_back(2 * P.namp + (q - 2 * nf));
                rs.push_back(1.0);
            } else {
                const int f = q < nf ? q : q - nf, off = q < nf ? 0 : P.namp;
                for (int a = 0; a < P.namp; ++a)
                    if (P.amap[a] == f) {
                        xs.push_back(off + a);
                        rs.push_back(P.aratio[a]);
                    }
            }
            ptr[q + 1] = (int)xs.size();
        }
        h->hmap_ptr = h->upload(ptr);
        h->hmap_x = h->upload(xs);
        h->hmap_r = h->upload(rs);
    }
    if (!M.customs.empty()) {
        h->mod2 = compile_eval(h->device, generate_custom2_kernel(M));
        HIPCHECK(hipModuleGetFunction(&h->fn_custom2, h->mod2, "ctpwa_custom2"));
        h->cfb2 = h->alloc<double>((size_t)M.customs.size() * M.ncf2() * h->ntot);
    }
    h->hess.ready = true;
}

// Gram of class cls's amplitude rows at the parameter point the table holds, to out
// [namp][namp][2]: with the theta coefficients K_a (withK = 1) or without them (0)
static void class_gram(ctpwa_handle* h, int cls, int withK, double* out, hipStream_t s) {
    const Plan& P = h->M.P;
    if (!h->agram.ready) {
        // one class per call: buffers for the largest
        const long long n3[3] = {std::max(h->n[0], std::max(h->n[1], h->n[2])), 0, 0};
        h->gtot = h->alloc<double>((size_t)P.namp * (2 * P.namp + 1));
        gramws_setup(h, h->agram, true, n3);
    }
    bool use[3] = {false, false, false};
    use[cls] = true;
    HessTotals T{};
    for (int c = 0; c < 3; ++c) T.G[c] = h->gtot;
    if (h->n[cls] > 0) gramws_run(h, h->agram, use, T, h->cfb, withK, s);
    else HIPCHECK(ctpwa_launch_zero(h->gtot, (long long)P.namp * (2 * P.namp + 1), s));
    HIPCHECK(ctpwa_launch_gram_to_complex(h->gtot, P.namp, out, s));
}

// No free resonance parameter: the amplitudes without couplings, A'_a = Psi_b sl_u, do
// not change between evaluations, so the phase-space sum of I = sum_p |sum_a c_a A'_a|^2
// is the quadratic form c^H G c of their Gram G, and the phase-space gradient sums
// sum_e conj(A'_a) S are (G c)_a (the reference's stored phase-space matrix and
// quadratic form, src/Analysis.cu:808-826, src/ComputeNLL.cu:575-597).  G is built once
// here in FP64 on the matrix cores; the final reduction forms the phase-space totals from
// it and the fused kernel scans data and background only.  Environment CTPWA_FIXED_GRAM=0
// keeps the per-event phase-space scan (for comparisons).
static bool fixed_gram_applies(const ctpwa_handle* h) {
    const Plan& P = h->M.P;
    if (P.ntheta != 0 || h->nacc != 1 + 2 * P.namp || h->n[0] <= 0) return false;
    const char* e = std::getenv("CTPWA_FIXED_GRAM");
    return !(e && std::string(e) == "0");
}
static void build_fixed_gram(ctpwa_handle* h) {
    const Plan& P = h->M.P;
    hipStream_t s = nullptr;
    // the table's coefficient records depend on theta only (none free): any couplings do
    double* p0 = h->upload(std::vector<double>((size_t)std::max(1, 2 * P.nfree), 0.0));
    double2* G = h->alloc<double2>((size_t)P.namp * P.namp);
    HIPCHECK(ctpwa_launch_prep(p0, h->table, &h->prep, 0, s));
    HIPCHECK(launch_custom(h, s));
    class_gram(h, 0, 0, (double*)G, s);
    h->d_gram = G;
    h->fin.gram = G;
    h->fin.off_c = (long long)h->M.off_c();
}

extern "C" int ctpwa_amplitude_gram(ctpwa_handle* h, const double* params_dev, int cls, double* out_dev, void* stream) {
    if (!h || !params_dev || !out_dev) return fail("ctpwa_amplitude_gram: NULL argument");
    if (cls < 0 || cls > 2) return fail("ctpwa_amplitude_gram: class must be 0 (phsp), 1 (data) or 2 (bkg)");
    DeviceGuard g(h->device);
    hipStream_t s = (hipStream_t)stream;
    try {
        HIPCHECK(ctpwa_launch_prep(params_dev, h->table, &h->prep, 0, s));
        HIPCHECK(launch_custom(h, s));
        class_gram(h, cls, 1, out_dev, s);
        return 0;
    } catch (const std::exception& e) {
        return fail(std::string("ctpwa_amplitude_gram: ") + e.what());
    }
}

extern "C" int ctpwa_partial_intensities(ctpwa_handle* h, const double* params_dev, int cls, double* out_dev, void* stream) {
    if (!h || !params_dev || !out_dev) return fail("ctpwa_partial_intensities: NULL argument");
    if (cls < 0 || cls > 2) return fail("ctpwa_partial_intensities: class must be 0 (phsp), 1 (data) or 2 (bkg)");
    DeviceGuard g(h->device);
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = ctpwa_launch_prep(params_dev, h->table, &h->prep, 0, s);
    if (e == hipSuccess) e = launch_custom(h, s);
    if (e == hipSuccess)
        e = ctpwa_launch_partial_int(&h->aux, h->wave_ptr, h->wave_blk, h->M.P.nwave, h->off[cls], h->n[cls],
                                     out_dev, s);
    if (e != hipSuccess) return fail(std::string("ctpwa_partial_intensities: ") + hipGetErrorString(e));
    return 0;
}

extern "C" int ctpwa_partial_amplitudes(ctpwa_handle* h, const double* params_dev, int cls, double* out_dev, void* stream) {
    if (!h || !params_dev || !out_dev) return fail("ctpwa_partial_amplitudes: NULL argument");
    if (cls < 0 || cls > 2) return fail("ctpwa_partial_amplitudes: class must be 0 (phsp), 1 (data) or 2 (bkg)");
    DeviceGuard g(h->device);
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = ctpwa_launch_prep(params_dev, h->table, &h->prep, 0, s);
    if (e == hipSuccess) e = launch_custom(h, s);
    if (e == hipSuccess)
        e = ctpwa_launch_partial_amp(&h->aux, h->wave_ptr, h->wave_blk, h->M.P.nwave, h->off[cls], h->n[cls],
                                     out_dev, s);
    if (e != hipSuccess) return fail(std::string("ctpwa_partial_amplitudes: ") + hipGetErrorString(e));
    return 0;
}

extern "C" int ctpwa_last_theta(ctpwa_handle* h, double* theta_host, void* stream) {
    if (!h || (!theta_host && h->M.P.ntheta > 0)) return fail("ctpwa_last_theta: NULL argument");
    if (h->M.P.ntheta == 0) return 0;
    DeviceGuard g(h->device);
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = hipMemcpyAsync(theta_host, h->table + h->M.off_lth(), (size_t)h->M.P.ntheta * sizeof(double),
                                  hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return fail(std::string("ctpwa_last_theta: ") + hipGetErrorString(e));
    return 0;
}

extern "C" int ctpwa_hessian(ctpwa_handle* h, const double* params_dev, double* hess_dev, void* stream) {
    if (!h || !params_dev || !hess_dev) return fail("ctpwa_hessian: NULL argument");
    DeviceGuard g(h->device);
    hipStream_t s = (hipStream_t)stream;
    try {
        if (!h->hess.ready) hess_setup(h);
        const Model_& M = h->M;
        const Plan& P = M.P;
        const HessShape& S = h->hess.S;
        HIPCHECK(ctpwa_launch_prep(params_dev, h->table, &h->prep, 3, s));
        if (h->fn_custom2) {
            void* args[] = {&h->table, &h->inv, &h->invf, &h->ntot, &h->cfb2};
            unsigned grid = (unsigned)std::min<long long>(16384, (h->ntot + 63) / 64);
            HIPCHECK(hipModuleLaunchKernel(h->fn_custom2, grid, 1, 1, 64, 1, 1, 0, s, args, nullptr));
        }
        const size_t per_class = (size_t)h->hnG + h->hnUu + h->hNZ + S.NU;
        HessAsm as{};
        HessTotals T{};
        bool use[3];
        for (int c = 0; c < 3; ++c) {
            double* base = h->htot + c * per_class;
            as.G[c] = T.G[c] = base;
            as.Uu[c] = T.Uu[c] = base + h->hnG;
            as.Zs[c] = T.Z[c] = base + h->hnG + h->hnUu;
            as.gs[c] = base + h->hnG + h->hnUu + h->hNZ;        // the u sums follow Z
            use[c] = h->n[c] > 0;
            as.live[c] = use[c];
        }
        gramws_run(h, h->hess, use, T, h->cfb2, 1, s);
        as.C = S.C; as.NU = S.NU; as.NZ = h->hNZ;
        as.namp = P.namp; as.nfree = P.nfree; as.ntheta = P.ntheta;
        as.zvt = h->hzvt; as.ttp = h->http; as.ttl = h->httl;
        as.Np = (double)h->n[0]; as.Wd = h->Wd; as.Wb = h->Wb;
        as.ngauss = (int)P.g_slot.size(); as.g_slot = h->fin.g_slot; as.g_sig = h->fin.g_sig;
        as.map_ptr = h->hmap_ptr; as.map_x = h->hmap_x; as.map_r = h->hmap_r;
        as.out = hess_dev;
        HIPCHECK(ctpwa_launch_hess_assemble(&as, s));
        return 0;
    } catch (const std::exception& e) {
        return fail(std::string("ctpwa_hessian: ") + e.what());
    }
}

static int aux_call(ctpwa_handle* h, const double* params_dev, int cls, double* out_dev, void* stream, int intensity) {
    if (!h || !params_dev || !out_dev) return fail("NULL argument");
    if (cls < 0 || cls > 2) return fail("event class must be 0, 1 or 2");
    DeviceGuard g(h->device);
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = ctpwa_launch_prep(params_dev, h->table, &h->prep, 0, s);
    if (e == hipSuccess) e = launch_custom(h, s);
    if (e == hipSuccess && h->fn_aux) {
        // generated kernel of the model (Custom lineshapes)
        long long e0 = h->off[cls], n = h->n[cls];
        if (n > 0) {
            int flag = intensity;
            void* args[] = {&h->table, &h->slp, &h->inv, &h->invf, &h->ntot, &e0, &n, &out_dev, &flag, &h->cfb};
            e = hipModuleLaunchKernel(h->fn_aux, (unsigned)((n + 255) / 256), 1, 1, 256, 1, 1, 0, s, args, nullptr);
        }
    } else if (e == hipSuccess) {
        e = ctpwa_launch_aux(&h->aux, (int)h->M.P.blocks.size(), h->off[cls], h->n[cls], out_dev, intensity, s);
    }
    if (e != hipSuccess) return fail(hipGetErrorString(e));
    return 0;
}

extern "C" int ctpwa_intensity(ctpwa_handle* h, const double* params_dev, int cls, double* out_dev, void* stream) {
    return aux_call(h, params_dev, cls, out_dev, stream, 1);
}

extern "C" int ctpwa_amplitudes(ctpwa_handle* h, const double* params_dev, int cls, double* out_dev, void* stream) {
    return aux_call(h, params_dev, cls, out_dev, stream, 0);
}

extern "C" int ctpwa_time_eval_kernel(ctpwa_handle* h, const double* params_dev, int iters, void* stream, double* avg_ms) {
    if (!h || !params_dev || !avg_ms || iters <= 0 || iters > 10000) return fail("ctpwa_time_eval_kernel: bad argument");
    DeviceGuard g(h->device);
    hipStream_t s = (hipStream_t)stream;
    // one event pair around every launch: the average is over the kernels' own durations,
    // not over the gaps between back-to-back launches
    std::vector<hipEvent_t> ev(2 * (size_t)iters, nullptr);
    hipError_t e = hipSuccess;
    for (size_t i = 0; i < ev.size() && e == hipSuccess; ++i) e = hipEventCreate(&ev[i]);
    if (e == hipSuccess) e = ctpwa_launch_prep(params_dev, h->table, &h->prep, 0, s);
    if (e == hipSuccess) e = launch_custom(h, s);
    for (int i = 0; i < iters && e == hipSuccess; ++i) {
        e = hipEventRecord(ev[2 * i], s);
        if (e == hipSuccess) e = launch_eval(h, s);
        if (e == hipSuccess) e = hipEventRecord(ev[2 * i + 1], s);
    }
    if (e == hipSuccess) e = hipEventSynchronize(ev.back());
    double total = 0.0;
    for (int i = 0; i < iters && e == hipSuccess; ++i) {
        float ms = 0.f;
        e = hipEventElapsedTime(&ms, ev[2 * i], ev[2 * i + 1]);
        total += ms;
    }
    for (hipEvent_t x : ev)
        if (x) (void)hipEventDestroy(x);
    if (e != hipSuccess) return fail(std::string("ctpwa_time_eval_kernel: ") + hipGetErrorString(e));
    *avg_ms = total / iters;
    return 0;
}

// ---------------------------------------------------------------------------
// many likelihoods of one model in one set of launches (continuous batching)
// ---------------------------------------------------------------------------
// mirrors `struct EvalJob` of the generated source (codegen.cpp)
struct EvalJob {
    const double* tab; const void* sl; const double* inv; const float* invf; const double* wts;
    double* part; const int* wg_cls; const long long* wg_rng; const double* cf; long long ld; double w1, w2;
    int nwg, pw1, pw2, wg_begin;
};

struct ctpwa_batch {
    int device = 0;
    int cap = 0;
    size_t bytes = 0;
    char* host = nullptr;          // pinned staging of the descriptors
    // device copy: [header: job count, task count | task counters][EvalJob cap][FinArgs cap]
    // [params ptr cap][table ptr cap][PrepArgs cap]
    char* dev = nullptr;
    hipEvent_t copied = nullptr;   // the staging buffer may be rewritten once this completes
    bool pending = false;
    size_t o_hdr = 0, o_ctr = 0, o_jobs = 0, o_fins = 0, o_params = 0, o_tables = 0, o_preps = 0;
    int max_nacc = 0;              // of the uploaded list
    int max_items = 0;             // coefficient records of a job's prep
    size_t max_lds = 0;
    // Graph replays (opt-in, environment CTPWA_BATCH_GRAPH=1): the descriptors on the device
    // belong to `key`, a list of (handle serial, params, out); a call with the same list
    // reuses them without an upload (serials, not handle addresses: a new handle may take a
    // destroyed one's address) and replays a captured graph of the launches, one per
    // power-of-two row bucket per model module.  Every argument a captured launch holds is
    // in the descriptors or is a constant of the model (each job's prep arguments included:
    // they point into that job's own handle).
    bool use_graphs = false;
    std::vector<unsigned long long> key;
    int rows = 0;
    hipStream_t cs = nullptr;      // capture stream
    hipModule_t gmod = nullptr;
    std::map<std::pair<int, int>, hipGraphExec_t> execs;   // by (rows, max_items)
    int persist = 0;               // workgroups of the persistent grouped kernel
};

static size_t align256(size_t x) { return (x + 255) / 256 * 256; }

extern "C" int ctpwa_batch_create(int device, int max_jobs, ctpwa_batch** out) {
    if (!out) return fail("ctpwa_batch_create: out is NULL");
    *out = nullptr;
    if (max_jobs <= 0 || max_jobs > 65535) return fail("ctpwa_batch_create: max_jobs must be in [1, 65535]");
    ctpwa_batch* b = new ctpwa_batch();
    DeviceGuard g(device);
    try {
        b->device = device;
        b->cap = max_jobs;
        b->o_hdr = 0;
        b->o_ctr = 256;
        b->o_jobs = 512;
        b->o_fins = b->o_jobs + align256(sizeof(EvalJob) * max_jobs);
        b->o_params = b->o_fins + align256(sizeof(FinArgs) * max_jobs);
        b->o_tables = b->o_params + align256(sizeof(void*) * max_jobs);
        b->o_preps = b->o_tables + align256(sizeof(void*) * max_jobs);
        b->bytes = b->o_preps + align256(sizeof(PrepArgs) * max_jobs);
        const char* e = std::getenv("CTPWA_BATCH_GRAPH");
        b->use_graphs = e && std::string(e) == "1";
        HIPCHECK(hipSetDevice(device));
        HIPCHECK(hipHostMalloc((void**)&b->host, b->bytes, hipHostMallocDefault));
        std::memset(b->host, 0, b->bytes);
        HIPCHECK(hipMalloc((void**)&b->dev, b->bytes));
        // the task counters start at zero; the persistent grouped kernel leaves them at zero
        HIPCHECK(hipMemset(b->dev, 0, 512));
        HIPCHECK(hipEventCreateWithFlags(&b->copied, hipEventDisableTiming));
        if (b->use_graphs) HIPCHECK(hipStreamCreateWithFlags(&b->cs, hipStreamNonBlocking));
        *out = b;
        return 0;
    } catch (const std::exception& e) {
        if (b->host) (void)hipHostFree(b->host);
        if (b->dev) (void)hipFree(b->dev);
        if (b->copied) (void)hipEventDestroy(b->copied);
        delete b;
        return fail(std::string("ctpwa_batch_create: ") + e.what());
    }
}

static void batch_drop_graphs(ctpwa_batch* b) {
    for (auto& kv : b->execs) (void)hipGraphExecDestroy(kv.second);
    b->execs.clear();
}

extern "C" void ctpwa_batch_destroy(ctpwa_batch* b) {
    if (!b) return;
    DeviceGuard g(b->device);
    if (!b->execs.empty()) (void)hipDeviceSynchronize();   // no replay still reads the buffers
    else if (b->pending) (void)hipEventSynchronize(b->copied);
    batch_drop_graphs(b);
    if (b->cs) (void)hipStreamDestroy(b->cs);
    (void)hipEventDestroy(b->copied);
    (void)hipHostFree(b->host);
    (void)hipFree(b->dev);
    delete b;
}

// graph replays: the launches over the uploaded descriptors with the job and task counts
// read on the device, `rows` (>= the job count) workgroup rows of prep and reduction, the
// persistent grouped kernel, each job's own prep arguments
static void batch_launches_graph(ctpwa_batch* b, const ctpwa_handle* h0, int rows, hipStream_t s) {
    const int* d_hdr = (const int*)(b->dev + b->o_hdr);
    unsigned int* d_ctr = (unsigned int*)(b->dev + b->o_ctr);
    HIPCHECK(ctpwa_launch_prep_batch((const double* const*)(b->dev + b->o_params), (double* const*)(b->dev + b->o_tables),
                                     (const PrepArgs*)(b->dev + b->o_preps), b->max_items, rows, d_hdr, s));
    const EvalJob* d_jobs = (const EvalJob*)(b->dev + b->o_jobs);
    void* args[] = {&d_jobs, &d_hdr, &d_ctr};
    HIPCHECK(hipModuleLaunchKernel(h0->fn_group_p, b->persist, 1, 1, h0->M.wgs, 1, 1, 0, s, args, nullptr));
    HIPCHECK(ctpwa_launch_finalize_batch((const FinArgs*)(b->dev + b->o_fins), rows, b->max_nacc, b->max_lds, d_hdr, s));
}

extern "C" int ctpwa_batch_nll_grad(ctpwa_batch* b, ctpwa_handle* const* hs, const double* const* params_dev,
                                    double* const* out_dev, int n, void* stream) {
    if (!b || !hs || !params_dev || !out_dev) return fail("ctpwa_batch_nll_grad: NULL argument");
    if (n <= 0) return 0;
    if (n > b->cap) return fail("ctpwa_batch_nll_grad: more likelihoods than the batch was created for");
    DeviceGuard g(b->device);
    hipStream_t s = (hipStream_t)stream;
    try {
        const ctpwa_handle* h0 = hs[0];
        for (int j = 0; j < n; ++j) {
            const ctpwa_handle* h = hs[j];
            if (!h || !params_dev[j] || !out_dev[j]) throw std::runtime_error("NULL handle, parameter or output pointer");
            if (h->device != b->device) throw std::runtime_error("a handle lives on another device than the batch");
            if (h->mod != h0->mod) throw std::runtime_error("the handles of one batch must share one model and precision");
        }
        // graph replays only for models without Custom lineshapes (those launch one factor
        // kernel per job)
        const bool graph = b->use_graphs && h0->M.customs.empty();
        std::vector<unsigned long long> key;
        if (graph) {
            key.resize((size_t)3 * n);
            for (int j = 0; j < n; ++j) {
                key[3 * j] = hs[j]->serial;
                key[3 * j + 1] = (unsigned long long)(uintptr_t)params_dev[j];
                key[3 * j + 2] = (unsigned long long)(uintptr_t)out_dev[j];
            }
        }
        int wg = 0;
        if (!graph || key != b->key) {
            {
                // a handle holds one coefficient table and one set of partial sums
                std::vector<const ctpwa_handle*> seen(hs, hs + n);
                std::sort(seen.begin(), seen.end());
                if (std::adjacent_find(seen.begin(), seen.end()) != seen.end())
                    throw std::runtime_error("a handle appears twice in one batch (each job needs a handle of its own)");
            }
            b->key.clear();
            // the staging buffer is reused: wait for the previous upload from it
            if (b->pending) HIPCHECK(hipEventSynchronize(b->copied));
            int* hdr = (int*)(b->host + b->o_hdr);
            EvalJob* jobs = (EvalJob*)(b->host + b->o_jobs);
            FinArgs* fins = (FinArgs*)(b->host + b->o_fins);
            const double** pp = (const double**)(b->host + b->o_params);
            double** tp = (double**)(b->host + b->o_tables);
            PrepArgs* pa = (PrepArgs*)(b->host + b->o_preps);
            int max_nacc = 0, max_items = 0;
            size_t max_lds = 0;
            for (int j = 0; j < n; ++j) {
                ctpwa_handle* h = hs[j];
                max_nacc = std::max(max_nacc, h->nacc);
                max_items = std::max(max_items, h->prep.nden + h->prep.namp);
                max_lds = std::max(max_lds, assemble_lds_bytes(h->fin));
                jobs[j] = EvalJob{h->table, h->slp, h->inv, h->invf, h->wts, h->part, h->wg_cls, h->wg_rng, h->cfb,
                                  h->ntot, h->wc[1], h->wc[2], h->nwg, h->pw[1], h->pw[2], wg};
                wg += h->nwg;
                fins[j] = h->fin;
                fins[j].params = params_dev[j];
                fins[j].out = out_dev[j];
                pp[j] = params_dev[j];
                tp[j] = h->table;
                pa[j] = h->prep;
            }
            hdr[0] = n;
            hdr[1] = wg;
            // header and descriptors (the task counters stay as the kernel left them)
            HIPCHECK(hipMemcpyAsync(b->dev + b->o_hdr, b->host + b->o_hdr, 2 * sizeof(int), hipMemcpyHostToDevice, s));
            HIPCHECK(hipMemcpyAsync(b->dev + b->o_jobs, b->host + b->o_jobs, b->bytes - b->o_jobs, hipMemcpyHostToDevice, s));
            HIPCHECK(hipEventRecord(b->copied, s));
            b->pending = true;
            b->max_nacc = max_nacc;
            b->max_items = max_items;
            b->max_lds = max_lds;
            if (graph) {
                b->key.swap(key);
                int rows = 1;
                while (rows < n) rows <<= 1;
                b->rows = std::min(rows, b->cap);
            }
        }
        if (!graph) {
            // one batched prep launch, each job's Custom factors, one grouped launch whose
            // workgroups are shared out among the jobs, one batched reduction and assembly.
            // Every job's coefficients come from its own handle's model tables: handles that
            // share a kernel may differ in fixed masses, widths, ratios and constraints, which
            // the kernel's source does not hold.
            HIPCHECK(ctpwa_launch_prep_batch((const double* const*)(b->dev + b->o_params),
                                             (double* const*)(b->dev + b->o_tables),
                                             (const PrepArgs*)(b->dev + b->o_preps), b->max_items, n, nullptr, s));
            for (int j = 0; j < n; ++j) HIPCHECK(launch_custom(hs[j], s));
            const EvalJob* d_jobs = (const EvalJob*)(b->dev + b->o_jobs);
            void* args[] = {&d_jobs, &n};
            if (wg > 0) HIPCHECK(hipModuleLaunchKernel(h0->fn_group, wg, 1, 1, h0->M.wgs, 1, 1, 0, s, args, nullptr));
            HIPCHECK(ctpwa_launch_finalize_batch((const FinArgs*)(b->dev + b->o_fins), n, b->max_nacc, b->max_lds, nullptr,
                                                 s));
            return 0;
        }
        if (b->gmod != h0->mod) {
            // a new model: its grouped kernel's persistent grid, and no graph of another model
            batch_drop_graphs(b);
            int per_cu = 0, ncu = 0;
            HIPCHECK(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, h0->fn_group_p, h0->M.wgs, 0));
            HIPCHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, b->device));
            b->persist = std::max(1, per_cu) * std::max(1, ncu);
            b->gmod = h0->mod;
        }
        const auto shape = std::make_pair(b->rows, b->max_items);
        auto it = b->execs.find(shape);
        if (it == b->execs.end()) {
            hipGraph_t graph_ = nullptr;
            hipGraphExec_t exec = nullptr;
            HIPCHECK(hipStreamBeginCapture(b->cs, hipStreamCaptureModeThreadLocal));
            try {
                batch_launches_graph(b, h0, b->rows, b->cs);
            } catch (...) {
                (void)hipStreamEndCapture(b->cs, &graph_);
                if (graph_) (void)hipGraphDestroy(graph_);
                throw;
            }
            HIPCHECK(hipStreamEndCapture(b->cs, &graph_));
            hipError_t e = hipGraphInstantiate(&exec, graph_, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph_);
            HIPCHECK(e);
            it = b->execs.emplace(shape, exec).first;
        }
        HIPCHECK(hipGraphLaunch(it->second, s));
        return 0;
    } catch (const std::exception& e) {
        b->key.clear();                    // upload again on the next call
        return fail(std::string("ctpwa_batch_nll_grad: ") + e.what());
    }
}

// per-event bytes of the SL tensors and the invariants a model stores at a precision
static long long event_bytes(const Model_& M, const std::vector<int>* used) {
    std::vector<int> imap = M.imap();
    long long b = (long long)M.us.size() * M.npstore() * (M.mixed ? 8 : 16);
    for (size_t i = 0; i < M.inv.size(); ++i)
        if (!used || (*used)[i]) b += (imap[i] >= 0) ? 8 : 4;
    b += (long long)M.customs.size() * M.ncf() * 8;      // Custom factor rows
    return b;
}

extern "C" long long ctpwa_footprint_bytes(const char* plan_text, long long n_phsp, long long n_data, long long n_bkg,
                                           int precision) {
    try {
        if (precision != 0 && precision != 1) throw std::runtime_error("precision must be 0 (FP64) or 1 (mixed)");
        Model_ M = derive(parse_plan(plan_text));
        M.mixed = precision;
        long long nt = n_phsp + n_data + n_bkg;
        long long b = nt * event_bytes(M, nullptr);
        b += (long long)M.table_size() * 8 + (long long)(1 + 2 * M.P.namp + M.P.ntheta) * 1024 * 8;
        b += nt * (long long)M.customs.size() * M.ncf() * 8;     // Custom factor rows
        // no free resonance parameter: the stored phase-space Gram and its build workspace
        if (M.P.ntheta == 0)
            b += (long long)M.P.namp * M.P.namp * 16 + agram_workspace_bytes(M, std::max(n_phsp, std::max(n_data, n_bkg)));
        // (the upload staging is one pool per device for the process, not per handle)
        return b;
    } catch (const std::exception& e) {
        g_err = std::string("ctpwa_footprint_bytes: ") + e.what();
        return -1;
    }
}

extern "C" long long ctpwa_hessian_workspace_bytes(const char* plan_text, long long n_phsp, long long n_data,
                                                   long long n_bkg) {
    try {
        Model_ M = derive(parse_plan(plan_text));
        const long long n3[3] = {n_phsp, n_data, n_bkg};
        return hess_workspace_bytes(M, n3, n_phsp + n_data + n_bkg);
    } catch (const std::exception& e) {
        g_err = std::string("ctpwa_hessian_workspace_bytes: ") + e.what();
        return -1;
    }
}

extern "C" int ctpwa_layout(const ctpwa_handle* h, long long* n_events3, long long* bytes_per_eval, int* n_sl, int* n_inv,
                            int* n_wg, int* n_pol_stored) {
    if (!h) return fail("ctpwa_layout: NULL handle");
    if (n_events3) for (int c = 0; c < 3; ++c) n_events3[c] = h->n[c];
    int used = 0;
    for (int u : h->used_inv) used += u;
    if (bytes_per_eval) {
        // with the stored phase-space Gram an evaluation reads data and background only
        long long b = ((h->d_gram ? 0 : h->n[0]) + h->n[1] + h->n[2]) * event_bytes(h->M, &h->used_inv);
        for (int c = 1; c < 3; ++c) if (h->pw[c]) b += h->n[c] * 8;
        *bytes_per_eval = b;
    }
    if (n_sl) *n_sl = (int)h->M.us.size();
    if (n_inv) *n_inv = used;
    if (n_wg) *n_wg = h->nwg;
    if (n_pol_stored) *n_pol_stored = h->M.npstore();
    return 0;
}

extern "C" const char* ctpwa_kernel_source(const ctpwa_handle* h) { return h ? h->src.c_str() : ""; }

// source of the fused kernel for a plan, without a device (buf may be NULL to query the size)
extern "C" long long ctpwa_generate_source(const char* plan_text, int precision, char* buf, long long cap) {
    try {
        if (precision != 0 && precision != 1) throw std::runtime_error("precision must be 0 (FP64) or 1 (mixed)");
        Model_ M = derive(parse_plan(plan_text));
        M.mixed = precision;
        apply_codegen_env(M);
        std::string src = generate_eval_kernel(M);
        if (buf && cap > 0) {
            long long n = std::min<long long>(cap - 1, (long long)src.size());
            std::memcpy(buf, src.data(), (size_t)n);
            buf[n] = '\0';
        }
        return (long long)src.size() + 1;
    } catch (const std::exception& e) {
        g_err = std::string("ctpwa_generate_source: ") + e.what();
        return -1;
    }
}

// source of the generated Hessian kernel for a plan, without a device
extern "C" long long ctpwa_generate_hessian_source(const char* plan_text, int precision, char* buf, long long cap) {
    try {
        if (precision != 0 && precision != 1) throw std::runtime_error("precision must be 0 (FP64) or 1 (mixed)");
        Model_ M = derive(parse_plan(plan_text));
        M.mixed = precision;
        std::string src = generate_hess_kernel(M, nullptr, false);
        // the amplitude Gram's module follows, and for models with Custom lineshapes the
        // second-order factors'
        src += "\n// ---- module: ctpwa_amp_gram ----\n" + generate_hess_kernel(M, nullptr, true);
        if (!M.customs.empty()) src += "\n// ---- module: ctpwa_custom2 ----\n" + generate_custom2_kernel(M);
        if (buf && cap > 0) {
            long long n = std::min<long long>(cap - 1, (long long)src.size());
            std::memcpy(buf, src.data(), (size_t)n);
            buf[n] = '\0';
        }
        return (long long)src.size() + 1;
    } catch (const std::exception& e) {
        g_err = std::string("ctpwa_generate_hessian_source: ") + e.what();
        return -1;
    }
}

// compile a plan's generated kernels with hipRTC (no device needed); returns the
// code objects' size in bytes, or -1 with the compiler log in ctpwa_last_error()
extern "C" long long ctpwa_compile_check(const char* plan_text, int precision) {
    try {
        if (precision != 0 && precision != 1) throw std::runtime_error("precision must be 0 (FP64) or 1 (mixed)");
        Model_ M = derive(parse_plan(plan_text));
        M.mixed = precision;
        apply_codegen_env(M);
        auto compile = [](const std::string& src) -> long long {
            hiprtcProgram prog;
            if (hiprtcCreateProgram(&prog, src.c_str(), "ctpwa_eval.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS)
                throw std::runtime_error("hiprtcCreateProgram failed");
            hiprtcResult r = hiprtcCompileProgram(prog, RTC_NOPTS, RTC_OPTS);
            size_t ls = 0;
            hiprtcGetProgramLogSize(prog, &ls);
            std::string log(ls + 1, '\0');
            hiprtcGetProgramLog(prog, &log[0]);
            size_t cs = 0;
            if (r == HIPRTC_SUCCESS) hiprtcGetCodeSize(prog, &cs);
            hiprtcDestroyProgram(&prog);
            if (r != HIPRTC_SUCCESS) throw std::runtime_error(log);
            return (long long)cs;
        };
        long long cs = compile(generate_eval_kernel(M));
        cs += compile(generate_hess_kernel(M, nullptr, false));
        cs += compile(generate_hess_kernel(M, nullptr, true));
        // models with Custom lineshapes: also the Hessian's second-order factor module
        if (!M.customs.empty()) cs += compile(generate_custom2_kernel(M));
        return cs;
    } catch (const std::exception& e) {
        g_err = std::string("ctpwa_compile_check: ") + e.what();
        return -1;
    }
}
extern "C" const char* ctpwa_last_error(void) { return g_err.c_str(); }
extern "C" const char* ctpwa_version(void) { return "ctpwa_amd 0.1.0 (gfx950)"; }
