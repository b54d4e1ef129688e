// Hessian of the likelihood (replaces analysis::getHessian, src/Analysis.cu:2689-3378).
//
// With S_p = sum_a v_a A_a(p), I = sum_p |S_p|^2 and real parameters x = (Re v, Im v,
// theta), every event needs
//   dI/dx           = 2 Re <S, dS/dx>
//   d2I/dx dy       = 2 Re sum_p [conj(dS/dy) dS/dx + conj(S) d2S/dx dy]
// The first part of d2I is the real embedding of the complex Gram of the Jacobian
// columns J = [A_1..A_n, dS/dtheta_1..dS/dtheta_P] (rows: event x polarisation), so
// the sum over events is a weighted Gram  sum_e alpha_e J^H J  (a K = N*nPol tall-skinny
// contraction).  The second part only couples (v, theta) and (theta, theta) and reduces
// to per-event scalars: <S, dA_a/dtheta> = dF_a/dtheta conj(T_u) and
// <S, d2S> = sum_a v_a d2F_a conj(T_u), T_u = sum_p conj(sl'_u,p) S_p.
//
// Per class the device forms
//   G   = sum_e alpha_e Jhat^T Jhat      (Jhat = [Re J | Im J])
//   U   = sum_e beta_e u u^T,  u = dI/dx
//   Z   = sum_e alpha_e z,     z = second-part scalars and I
//   g   = sum_e u
// with alpha = w/I, beta = -w/I^2 (data, background: second derivative of w ln I) and
// alpha = 1, beta = 0 (phase space), then assembles
//   H = -H_data + H_bkg + N_eff [ A2 / (N_p pf) - g g^T / (N_p pf)^2 ] (+ Gaussian terms)
// and maps it to the fit parameters (v_a = r_a p_f(a)).
//
// Events are processed in chunks; every sum is a fixed-order reduction.
#include <algorithm>
#include <cstdlib>

#include "device.hpp"

namespace ctpwa {

// Weighted Gram of a column-major matrix X[column][row] (column stride ldx) on the matrix
// cores:
//   G[a][b] = sum_rows w(row) X[a][row] X[b][row],  w(row) = Wt[row mod nev]
// (rows p * nev + r share event r's weight).  The rows of a pass's pieces lie one after the
// other; share x of the workgroups belongs to one piece, so that one launch serves every event
// class.  (Rows in blocks of 32, each block's columns together, do not speed this kernel or
// k_gram_wide up, and the FP32 writer's stores take 25 % longer.)  This kernel takes up to 64
// columns (four 16-column tiles); k_gram_wide takes more.  Each of a workgroup's four waves
// owns a contiguous range of the share, stages R-row slabs of the columns in its own LDS
// region (register prefetch of the next slab, column stride padded by one element against
// bank conflicts) and accumulates the 16x16 tile products I <= J in registers with
// v_mfma_f64_16x16x4 (T = double) or v_mfma_f32_16x16x4 (T = float: the mixed form's FP32
// Jacobian, products summed in FP32 over one slab, then added into FP64 accumulators).  The
// waves combine their tiles through LDS in wave order and the workgroup writes one partial
// per tile pair; k_hess_accum sums the partials in a fixed order.
// Lane layouts (16x16x4, one block): A[i][k] in lane 16 k + i, B[k][j] in lane 16 k + j;
// D[4 r + q][j] (f64) or D[4 q + r][j] (f32) in component r of lane 16 q + j.
constexpr int GP_WAVES = 4;
template <typename T> struct GP;
template <> struct GP<double> {
    static constexpr int R = 16;
    typedef double acc_t __attribute__((ext_vector_type(4)));
    __device__ static inline int row(int lane, int r) { return 4 * r + (lane >> 4); }
};
template <> struct GP<float> {
    static constexpr int R = 32;
    typedef float acc_t __attribute__((ext_vector_type(4)));
    __device__ static inline int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};
typedef double gp_acc64 __attribute__((ext_vector_type(4)));

// LDS bytes of k_gram_panels<T, NT>: per wave a slab of the columns, or the combined tile pairs
inline size_t gram_panels_lds(bool f32, int NT) {
    const int R = f32 ? 32 : 16;
    const size_t es = f32 ? 4 : 8;
    const int npair = NT * (NT + 1) / 2;
    size_t slabs = (size_t)GP_WAVES * NT * 16 * (R + 1) * es;
    size_t comb = (size_t)npair * 256 * sizeof(double);
    return std::max(slabs, comb);
}

// NT: tiles of the columns; the NT (NT + 1) / 2 tile pairs I <= J.  With the pair count fixed
// at compile time every pair's product is unconditional.
template <typename T, int NT>
__global__ void __launch_bounds__(64 * GP_WAVES, sizeof(T) == 4 && NT < 4 ? 3 : 2)
k_gram_panels(const T* __restrict__ X0, int ncol, long long ldx, HessPieces H, int rpe, const double* __restrict__ Wt0,
              double* __restrict__ part) {
    constexpr int R = GP<T>::R, ST = R + 1;
    constexpr int NPAIR = NT * (NT + 1) / 2;
    typedef typename GP<T>::acc_t acc_t;
    extern __shared__ __attribute__((aligned(16))) unsigned char gp_smem[];
    __shared__ double wsh[GP_WAVES][R];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    constexpr int NCOLS = NT * 16;
    T* xs = (T*)gp_smem + (size_t)wave * NCOLS * ST;
    double* ws = wsh[wave];
    int pk = 0;
    while (pk + 1 < H.n && (int)blockIdx.x >= H.ghi[pk]) ++pk;
    const long long nev = H.cnt[pk], nrows = nev * rpe;      // rpe rows per event
    const T* X = X0 + H.row0[pk];
    const double* Wt = Wt0 + H.w0[pk];
    // this wave's rows: the piece's waves split [0, nrows) into ranges of whole slabs
    const long long nw = (long long)(H.ghi[pk] - H.glo[pk]) * GP_WAVES;
    const long long gw = (long long)((int)blockIdx.x - H.glo[pk]) * GP_WAVES + wave;
    const long long per = ((nrows + nw - 1) / nw + R - 1) / R * R;
    const long long r0 = gw * per < nrows ? gw * per : nrows;
    const long long r1 = r0 + per < nrows ? r0 + per : nrows;
    gp_acc64 acc[NPAIR];
#pragma unroll
    for (int q = 0; q < NPAIR; ++q) acc[q] = (gp_acc64){0.0, 0.0, 0.0, 0.0};
    // 16-byte loads: lane l carries rows VW (l mod LPC) .. + VW - 1 of column CPI it + l / LPC
    // (pieces start at multiples of 4 rows and ldx is one, so every such run is aligned).
    // Every lane loads: a column past the last takes the last one (its products are not used),
    // rows past the last lie in the piece's padding and are set to 0 on the way to LDS.  With a
    // guard on each load the lanes of missing columns took its other arm, which waits for all
    // loads before it (5M rows of 50 FP32 columns 505 us, now 303, 3.3 TB/s; 6M of 40 columns
    // 304 and 255).
    constexpr int VW = 16 / (int)sizeof(T), LPC_ = R / VW, CPI = 64 / LPC_;
    constexpr int NLD = NCOLS / CPI;
    typedef T vec_t __attribute__((ext_vector_type(VW)));
    const int rr0 = (lane % LPC_) * VW, ch = lane / LPC_;
    const int rw = lane % R;
    // event of row t + rw is (t + rw) mod nev: one division for the wave's first slab, then
    // the base of the next slab to load advances by R with subtractions (no 64-bit division
    // per slab)
    long long eload = r0 < r1 ? r0 % nev : 0;
    auto load = [&](vec_t (&pre)[NLD], double& wpre, long long t0) {
        const T* Xb = X + t0 + rr0;
#pragma unroll
        for (int it = 0; it < NLD; ++it) pre[it] = *(const vec_t*)(Xb + (long long)min(CPI * it + ch, ncol - 1) * ldx);
        long long ev = eload + rw;
        while (ev >= nev) ev -= nev;              // rows that wrap to the next polarisation
        wpre = Wt[ev];
        eload += R;
        while (eload >= nev) eload -= nev;        // once at most unless nev < R
    };
    // one slab: its registers to the wave's LDS region, the refill of those registers with
    // the slab at tnext (loads in flight during this slab's products), then the products
    auto slab = [&](vec_t (&pre)[NLD], double& wpre, long long t0) {
        const long long tnext = t0 + R;
        if (tnext > r1) {
            const int nt = (int)(r1 - t0);
#pragma unroll
            for (int it = 0; it < NLD; ++it)
#pragma unroll
                for (int v = 0; v < VW; ++v) pre[it][v] = rr0 + v < nt ? pre[it][v] : (T)0;
            wpre = rw < nt ? wpre : 0.0;
        }
#pragma unroll
        for (int it = 0; it < NLD; ++it) {
            const int c = CPI * it + ch;
#pragma unroll
            for (int v = 0; v < VW; ++v) xs[c * ST + rr0 + v] = pre[it][v];
        }
        if (lane < R) ws[rw] = wpre;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        if (tnext < r1) load(pre, wpre, tnext);
        const int li = lane & 15;
        if constexpr (sizeof(T) == 8) {
#pragma unroll
            for (int k0 = 0; k0 < R; k0 += 4) {
                const int kr = k0 + (lane >> 4);
                const double w = ws[kr];
                int q = 0;
#pragma unroll
                for (int I = 0; I < NT; ++I) {
                    const double av = w * (double)xs[(I * 16 + li) * ST + kr];
#pragma unroll
                    for (int J = I; J < NT; ++J, ++q)
                        acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, (double)xs[(J * 16 + li) * ST + kr], acc[q],
                                                                      0, 0, 0);
                }
            }
        } else {
            acc_t t[NPAIR];
#pragma unroll
            for (int q = 0; q < NPAIR; ++q) t[q] = (acc_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k0 = 0; k0 < R; k0 += 4) {
                const int kr = k0 + (lane >> 4);
                const float w = (float)ws[kr];
                int q = 0;
#pragma unroll
                for (int I = 0; I < NT; ++I) {
                    const float av = w * xs[(I * 16 + li) * ST + kr];
#pragma unroll
                    for (int J = I; J < NT; ++J, ++q)
                        t[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, (float)xs[(J * 16 + li) * ST + kr], t[q], 0, 0, 0);
                }
            }
#pragma unroll
            for (int q = 0; q < NPAIR; ++q) {
                acc[q][0] += (double)t[q][0];
                acc[q][1] += (double)t[q][1];
                acc[q][2] += (double)t[q][2];
                acc[q][3] += (double)t[q][3];
            }
        }
        // the slab is consumed before the next one overwrites it
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    // one register buffer: the next slab's loads are in flight while this one is consumed
    // (a second buffer, two slabs ahead, measured no faster at two waves per SIMD)
    vec_t pre[NLD];
    double wpre = 0.0;
    if (r0 < r1) load(pre, wpre, r0);
    for (long long t0 = r0; t0 < r1; t0 += R) slab(pre, wpre, t0);
    // combine the waves in wave order in LDS (the slab regions are free once every wave
    // has finished), element e = 16 i + j of tile pair q at comb[q * 256 + e]
    double* comb = (double*)gp_smem;
    __syncthreads();
    for (int w = 0; w < GP_WAVES; ++w) {
        if (wave == w) {
#pragma unroll
            for (int q = 0; q < NPAIR; ++q) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int e = q * 256 + GP<T>::row(lane, r) * 16 + (lane & 15);
                    comb[e] = (w == 0) ? acc[q][r] : comb[e] + acc[q][r];
                }
            }
        }
        __syncthreads();
    }
    double* o = part + (size_t)blockIdx.x * NPAIR * 256;
    for (int e = threadIdx.x; e < NPAIR * 256; e += 64 * GP_WAVES) o[e] = comb[e];
}

// The same Gram for more than 64 columns, one piece per launch.  Panels of 128 columns (eight
// tiles); a workgroup of eight waves takes a panel pair and a share of the rows and stages
// slabs of R rows of the pair's 256 columns in LDS (two buffers, one barrier per slab, the next
// slab's loads in flight during the products).  Wave i holds the tile pairs of row i: all of an
// off-diagonal panel pair's (A read and weighted once per step), (i, i + q mod T) for
// q <= T / 2 on the diagonal, so every wave of a workgroup has the same work and the shares
// are dealt out by it.  Bound by the matrix cores (64 cycles per FP64 product); every column
// is read 3.3 times for 346 columns.  Registers should not spill: a reload between the loads
// waits for all of them (7.3 instead of 3.5 ms for 1.2M rows of 346 and 100k rows of 322
// columns, which meet none; of the FP64 forms an off-diagonal pair of seven tiles reloads two
// values per slab, of the FP32 forms one of eight tiles four).  Panels of 64 columns read every column 7.8 times
// and computed full tile squares on the diagonal (7.5 ms).
// LDS column strides: 16 columns x 2 rows (FP64) or x 4 rows (FP32) of a read lie in different
// banks, and 16-byte stores stay aligned.
constexpr int GW_WAVES = 8;
template <typename T> struct GWS { static constexpr int ST = sizeof(T) == 8 ? 18 : 36; };
template <typename T>
inline size_t gram_wide_lds() { return (size_t)2 * 256 * GWS<T>::ST * sizeof(T); }

template <typename T, int NQ, bool DIAG>
__device__ __forceinline__ void gram_wide_rows(const T* __restrict__ X, int ncol, long long ldx, const GramPair& G, long long r0,
                                               long long r1, int nev, const double* __restrict__ Wt, T* xs, double (*wsh)[GP<T>::R],
                                               double* __restrict__ o) {
    constexpr int R = GP<T>::R, ST = GWS<T>::ST;
    typedef typename GP<T>::acc_t acc_t;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int TQ = (min(128, ncol - 128 * G.Q) + 15) / 16, I = DIAG ? min(wave, TQ - 1) : wave;
    gp_acc64 acc[NQ];
    const int tl = li * ST + lk;
    int tb[NQ];                                   // first element of the B tiles
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        acc[q] = (gp_acc64){0.0, 0.0, 0.0, 0.0};
        tb[q] = (DIAG ? (I + q) % TQ : 8 + q) * 16 * ST;
    }
    // 16-byte loads, eight lanes to a column's slab: loads 0, 1 take panel P, loads 2, 3 panel Q
    // (a diagonal pair stages its panel once).  A column past the last takes the last one: its
    // products are not used.  Rows past the last lie in the matrix's padding and are set to 0.
    constexpr int VW = 16 / (int)sizeof(T), CPI = 64;
    static_assert(R / VW == 8, "eight lanes per column");
    typedef T vec_t __attribute__((ext_vector_type(VW)));
    const int rr0 = (threadIdx.x % 8) * VW, ch = threadIdx.x / 8;
    // row r0 + R k + thread's event (rows that wrap to the next polarisation start again)
    int ev = (int)((r0 + (int)threadIdx.x % R) % nev);
    const int evstep = R % nev;
    constexpr int NL = DIAG ? 2 : 4;
    vec_t pre[NL];
    double wpre = 0.0;
    const T* Xr = X + r0;
    auto load = [&]() {
        // the column's address is formed anew for each load, from a column index the optimiser
        // cannot see through: four addresses kept across the loop spill
        int c0 = ch;
        asm volatile("" : "+v"(c0));
        if ((int)threadIdx.x < R) {
            wpre = Wt[ev];
            ev += evstep;
            if (ev >= nev) ev -= nev;
        }
#pragma unroll
        for (int it = 0; it < NL; ++it)
            pre[it] = *(const vec_t*)(Xr + (long long)min(ncol - 1, 128 * (it < 2 ? G.P : G.Q) + CPI * (it & 1) + c0) * ldx + rr0);
        Xr += R;
    };
    auto store = [&](int b, long long t0) {
        T* xb = xs + b * 256 * ST + ch * ST + rr0;
        if (t0 + R > r1) {
            const int nt = (int)(r1 - t0);
#pragma unroll
            for (int it = 0; it < NL; ++it)
#pragma unroll
                for (int v = 0; v < VW; ++v) pre[it][v] = rr0 + v < nt ? pre[it][v] : (T)0;
            wpre = (int)threadIdx.x < nt ? wpre : 0.0;
        }
        if ((int)threadIdx.x < R) wsh[b][threadIdx.x] = wpre;
#pragma unroll
        for (int it = 0; it < NL; ++it) *(vec_t*)(xb + CPI * it * ST) = pre[it];
    };
    if (r0 < r1) {
        load();
        store(0, r0);
    }
    __syncthreads();
    int b = 0;
    for (long long t0 = r0; t0 < r1; t0 += R, b ^= 1) {
        const bool more = t0 + R < r1;
        if (more) load();
        const T* xb = xs + b * 256 * ST + tl;
        const T* xa = xb + I * 16 * ST;
        const double* ws = wsh[b] + lk;
        if constexpr (sizeof(T) == 8) {
#pragma unroll
            for (int k0 = 0; k0 < R; k0 += 4) {
                const double av = ws[k0] * xa[k0];
#pragma unroll
                for (int q = 0; q < NQ; ++q) acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, xb[tb[q] + k0], acc[q], 0, 0, 0);
            }
        } else {
            // a slab's products are summed in FP32, then added into the FP64 sums
            float av[R / 4];
#pragma unroll
            for (int k = 0; k < R / 4; ++k) av[k] = (float)ws[4 * k] * xa[4 * k];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                acc_t t = (acc_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int k = 0; k < R / 4; ++k) t = __builtin_amdgcn_mfma_f32_16x16x4f32(av[k], xb[tb[q] + 4 * k], t, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[q][r] += (double)t[r];
            }
        }
        if (more) store(b ^ 1, t0 + R);
        __syncthreads();             // the slab is consumed and the next one is in place
    }
    // the tile pairs in the order of the tile list; a wrapped diagonal pair (J < I) is the
    // transpose of (J, I), and (I, I + T / 2) comes twice for an even T
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int J = DIAG ? (I + q) % TQ : q;
        const int i = DIAG ? min(I, J) : I, j = DIAG ? max(I, J) : J;
        if (DIAG && (wave >= TQ || (2 * q == TQ && wave >= q))) continue;
        double* oq = o + (DIAG ? i * TQ - i * (i - 1) / 2 + (j - i) : i * TQ + j) * 256;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int a = GP<T>::row(lane, r);
            oq[DIAG && J < I ? li * 16 + a : a * 16 + li] = acc[q][r];
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(64 * GW_WAVES, 4)
k_gram_wide(const T* __restrict__ X, int ncol, long long ldx, long long nrows, int nev, const double* __restrict__ Wt,
            const GramPair* __restrict__ pairs, int npair, double* __restrict__ part) {
    constexpr int R = GP<T>::R;
    extern __shared__ __attribute__((aligned(16))) unsigned char gp_smem[];
    __shared__ double wsh[2][R];
    int y = 0;
    while (y + 1 < npair && (int)blockIdx.x >= pairs[y + 1].s0) ++y;
    const GramPair G = pairs[y];
    const int share = (int)blockIdx.x - G.s0;
    const long long slabs = (nrows + R - 1) / R;
    const long long per = (slabs + G.ns - 1) / G.ns;
    const long long r0 = min(nrows, share * per * R), r1 = min(nrows, r0 + per * R);
    // tile pair q of the panel pair at part[(off + share nt + q) 256]
    double* o = part + (G.off + (long long)share * G.nt) * 256;
#define GW_ROWS(NQ, D) gram_wide_rows<T, NQ, D>(X, ncol, ldx, G, r0, r1, nev, Wt, (T*)gp_smem, wsh, o); break
    switch (G.P == G.Q ? G.nq : 8 + G.nq) {
    case 1: GW_ROWS(1, true);
    case 2: GW_ROWS(2, true);
    case 3: GW_ROWS(3, true);
    case 4: GW_ROWS(4, true);
    case 5: GW_ROWS(5, true);
    case 9: GW_ROWS(1, false);
    case 10: GW_ROWS(2, false);
    case 11: GW_ROWS(3, false);
    case 12: GW_ROWS(4, false);
    case 13: GW_ROWS(5, false);
    case 14: GW_ROWS(6, false);
    case 15: GW_ROWS(7, false);
    case 16: GW_ROWS(8, false);
#undef GW_ROWS
    }
}

// tot (packed upper triangle) = or += the Gram from k_gram_wide's partials: 64 elements of one
// tile pair per workgroup, tpair its panel pair; sixteen waves as in k_hess_accum
constexpr int HA_WAVES = 16;
__global__ void __launch_bounds__(64 * HA_WAVES)
k_accum_wide(const double* __restrict__ part, const GramPair* __restrict__ pairs, const int2* __restrict__ tiles,
             const int* __restrict__ tpair, int ncol, double* __restrict__ tot, int first) {
    __shared__ double sh[HA_WAVES][64];
    const int tq = blockIdx.x >> 2, e = (blockIdx.x & 3) * 64 + (threadIdx.x & 63), wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const GramPair G = pairs[tpair[tq]];
    const double* p = part + (G.off + (tq - G.tile0)) * 256 + e;
    double s = 0.0, s1 = 0.0;
    int g = wave;
    for (; g + HA_WAVES < G.ns; g += 2 * HA_WAVES) {
        s += p[(size_t)g * G.nt * 256];
        s1 += p[(size_t)(g + HA_WAVES) * G.nt * 256];
    }
    if (g < G.ns) s += p[(size_t)g * G.nt * 256];
    sh[wave][lane] = s + s1;
    __syncthreads();
    if (wave == 0) {
        double v = sh[0][lane];
        for (int w = 1; w < HA_WAVES; ++w) v += sh[w][lane];
        const int2 t = tiles[tq];
        const int a = t.x * 16 + (e >> 4), b = t.y * 16 + (e & 15);
        if (a < ncol && b < ncol && a <= b) {
            double* o = tot + ((long long)a * ncol - (long long)a * (a - 1) / 2 + (b - a));
            *o = first ? v : *o + v;
        }
    }
}

// The sums of a pass, one launch: blockIdx.y is the piece; the first nG workgroups along x
// add the Gram partials of 64 tile elements each (tiles[q] = (I, J): the 16-column tiles of
// tile pair q; result in the packed upper triangle, row-major), the next nU those of the u
// Gram (pieces of HU), the rest the summed columns, one per wave (zpart[c * nwg + w], result
// at Z[perm[c]]).  Sixteen waves per workgroup add every sixteenth partial in four
// interleaved sums, joined in a fixed order: with four waves the 40-column Gram's 1000
// partials were a chain of 30 dependent loads (18 us per class).
__device__ inline void accum_tiles(const double* __restrict__ part, int lo, int hi, int ntp, const int2* __restrict__ tiles,
                                   int ncol, double* __restrict__ tot, bool first, int blk, double (*sh)[64]) {
    const long long E = (long long)ntp * 256;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long e = (long long)blk * 64 + lane;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    int g = lo + wave;
    for (; g + 3 * HA_WAVES < hi; g += 4 * HA_WAVES) {
#pragma unroll
        for (int k = 0; k < 4; ++k) s[k] += part[(size_t)(g + k * HA_WAVES) * E + e];
    }
    for (; g < hi; g += HA_WAVES) s[0] += part[(size_t)g * E + e];
    sh[wave][lane] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    if (wave == 0) {
        double v = sh[0][lane];
        for (int w = 1; w < HA_WAVES; ++w) v += sh[w][lane];
        const int2 t = tiles[e >> 8];
        const int a = t.x * 16 + (int)((e >> 4) & 15), b = t.y * 16 + (int)(e & 15);
        if (a < ncol && b < ncol && a <= b) {
            double* o = tot + ((long long)a * ncol - (long long)a * (a - 1) / 2 + (b - a));
            *o = first ? v : *o + v;
        }
    }
}
__global__ void __launch_bounds__(64 * HA_WAVES)
k_hess_accum(HessPieces H, HessPieces HU, HessTotals T, const double* __restrict__ gpart, int ntp, const int2* __restrict__ tiles,
             int ncol, const double* __restrict__ upart, int utp, const int2* __restrict__ utiles, int ucol,
             const double* __restrict__ zpart, int nz, int nwg, const int* __restrict__ perm) {
    __shared__ double sh[HA_WAVES][64];
    const int nG = ntp * 4, nU = utp * 4, k = blockIdx.y;
    int blk = blockIdx.x;
    if (blk < nG) {
        if (k >= H.n) return;
        accum_tiles(gpart, H.glo[k], H.ghi[k], ntp, tiles, ncol, T.G[H.cls[k]], T.first[H.cls[k]], blk, sh);
        return;
    }
    blk -= nG;
    if (blk < nU) {
        if (k >= HU.n) return;
        accum_tiles(upart, HU.glo[k], HU.ghi[k], utp, utiles, ucol, T.Uu[HU.cls[k]], T.first[HU.cls[k]], blk, sh);
        return;
    }
    blk -= nU;
    const int c = blk * HA_WAVES + (threadIdx.x >> 6);
    if (k >= H.n || c >= nz) return;
    const double* p = zpart + (long long)c * nwg;
    double s = 0.0;
    for (int w = H.wg0[k] + (threadIdx.x & 63); w < H.wg0[k + 1]; w += 64) s += p[w];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) {
        double* o = T.Z[H.cls[k]] + perm[c];
        *o = T.first[H.cls[k]] ? s : *o + s;
    }
}

__device__ inline double gram_at(const double* G, int n2, int k, int l) {
    // index of (min, max) in the row-major upper-triangle list of an n2 x n2 matrix
    int a = k < l ? k : l, b = k < l ? l : k;
    long long idx = (long long)a * n2 - (long long)a * (a - 1) / 2 + (b - a);
    return G[idx];
}

// sum_e alpha d2I[x][y] for one class from its Gram and second-part sums
__device__ double d2I_sum(const HessAsm& h, int c, int x, int y) {
    const int n = h.namp, C = h.C, C2 = 2 * C;
    const double* G = h.G[c];
    // complex Gram entry G[l][k] = sum conj(J_l) J_k
    auto Gre = [&](int l, int k) { return gram_at(G, C2, l, k) + gram_at(G, C2, C + l, C + k); };
    auto Gim = [&](int l, int k) { return gram_at(G, C2, l, C + k) - gram_at(G, C2, C + l, k); };
    // column index and factor (1 or i) of a real parameter
    auto col = [&](int p, int& k, bool& im) {
        if (p < n) { k = p; im = false; }
        else if (p < 2 * n) { k = p - n; im = true; }
        else { k = n + (p - 2 * n); im = false; }
    };
    int kx, ly;
    bool ix, iy;
    col(x, kx, ix);
    col(y, ly, iy);
    // 2 Re(conj(c_y) c_x G[ly][kx])
    double gr = Gre(ly, kx), gi = Gim(ly, kx);
    double v;
    if (!ix && !iy) v = 2.0 * gr;
    else if (!ix && iy) v = 2.0 * gi;
    else if (ix && !iy) v = -2.0 * gi;
    else v = 2.0 * gr;
    return v;
}

// complex Gram Q[l][k] = sum conj(A_l) A_k (n x n, interleaved) from the packed real Gram G
// of the 2n columns [Re A | Im A]
__global__ void k_gram_to_complex(const double* __restrict__ G, int n, double* __restrict__ Q) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n * n) return;
    const int l = q / n, k = q - l * n, n2 = 2 * n;
    Q[2 * q] = gram_at(G, n2, l, k) + gram_at(G, n2, n + l, n + k);
    Q[2 * q + 1] = gram_at(G, n2, l, n + k) - gram_at(G, n2, n + l, k);
}

// Hessian assembly in one launch: entry (r, c) of the fit-parameter Hessian
// [Re p, Im p, theta] is the sum over the extended parameters (Re v, Im v, theta) that r and
// c stand for (v_a = r_a p_f(a)) of
//   H = -H_data + H_bkg + N_eff [A2 / (N_p pf) - g g^T / (N_p pf)^2] + diag(1 / sigma^2),
// each class's part from its Gram, its u Gram and its second-part sums (zvt: the sum of
// <S, dA_a/dtheta_j>; ttp/ttl: the sums of Re(v d2F conj(T)) of a parameter pair over the
// blocks, in block order).  Every entry is one thread's, with no intermediate matrix.  As
// separate kernels the second-part terms of 149 amplitudes were one workgroup's serial
// work (137 us), and the three kernels of a 10-amplitude Hessian took 33 us.
__device__ inline void hess_pf(const HessAsm& h, double& cp, double& cq) {
    double Np = h.Np, Neff = h.Wd - h.Wb;
    double pf = (Np > 0) ? h.Zs[0][h.NZ - 1] / Np : 0.0;
    if (!(pf > 1e-30) || isinf(pf)) pf = 1e-30;
    cp = (Np > 0) ? Neff / (Np * pf) : 0.0;
    cq = (Np > 0) ? -Neff / (Np * pf * Np * pf) : 0.0;
}

__device__ inline double hess_ext(const HessAsm& h, double cp, double cq, int x, int y) {
    const int n = h.namp, P = h.ntheta;
    const bool tx = x >= 2 * n, ty = y >= 2 * n;
    const double sc[3] = {cp, -1.0, 1.0};
    double H = 0.0;
    for (int c = 0; c < 3; ++c) {
        if (!h.live[c]) continue;
        double v = d2I_sum(h, c, x, y);
        if (c != 0) v += gram_at(h.Uu[c], h.NU, x, y);
        // d2S/dRe v_a dtheta = dA_a/dtheta: 2 Re <S, dA>; d2S/dIm v_a dtheta = i dA: -2 Im <S, dA>
        if (tx != ty) {
            const int p = tx ? y : x, j = (tx ? x : y) - 2 * n;
            const int a = p < n ? p : p - n;
            const int z = h.zvt[a * P + j];
            if (z >= 0) v += p < n ? 2.0 * h.Zs[c][z] : -2.0 * h.Zs[c][z + 1];
        } else if (tx) {
            const int q = (x - 2 * n) * P + (y - 2 * n);
            for (int k = h.ttp[q]; k < h.ttp[q + 1]; ++k) v += 2.0 * h.Zs[c][h.ttl[k]];
        }
        H += sc[c] * v;
        if (c == 0) H += cq * h.gs[0][x] * h.gs[0][y];
    }
    if (tx && x == y)
        for (int g = 0; g < h.ngauss; ++g)
            if (h.g_slot[g] == x - 2 * n) H += 1.0 / (h.g_sig[g] * h.g_sig[g]);
    return H;
}

__global__ void __launch_bounds__(256) k_hess_out(HessAsm h) {
    const int np = 2 * h.nfree + h.ntheta;
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long long)np * np) return;
    double cp, cq;
    hess_pf(h, cp, cq);
    // the elements (r, c) and (c, r) are the same sum: the matrix is exactly symmetric
    const int qr = (int)(q / np), qc = (int)(q - (long long)qr * np), r = min(qr, qc), c = max(qr, qc);
    double H = 0.0;
    for (int u = h.map_ptr[r]; u < h.map_ptr[r + 1]; ++u)
        for (int w = h.map_ptr[c]; w < h.map_ptr[c + 1]; ++w)
            H += h.map_r[u] * h.map_r[w] * hess_ext(h, cp, cq, h.map_x[u], h.map_x[w]);
    h.out[q] = H;
}

}  // namespace ctpwa

using namespace ctpwa;

__global__ void k_zero(double* __restrict__ p, long long n) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = 0.0;
}

// zero fill by a kernel (not hipMemsetAsync: the call may be captured in a graph)
extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_zero(double* p, long long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    unsigned nb = (unsigned)std::min<long long>(1024, (n + 255) / 256);
    hipLaunchKernelGGL(k_zero, dim3(nb), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

// Tile pairs (I, J) of the Gram of ncol columns, returned count; more than 64 columns: also
// the panel pairs (their workgroups and partials set by the caller) and each tile pair's panel
// pair
extern "C" __attribute__((visibility("hidden"))) int ctpwa_gram_tables(int ncol, int2* tiles, GramPair* pairs, int* npair,
                                                                      int* tpair) {
    const int T = (ncol + 15) / 16;
    const bool wide = ncol > 64;
    const int np = wide ? (T + 7) / 8 : 1;
    int q = 0, y = 0;
    for (int P = 0; P < np; ++P)
        for (int Q = P; Q < np; ++Q, ++y) {
            const int i1 = wide ? std::min(T, 8 * P + 8) : T, j1 = wide ? std::min(T, 8 * Q + 8) : T, q0 = q;
            for (int I = 8 * P; I < i1; ++I)
                for (int J = P == Q ? I : 8 * Q; J < j1; ++J, ++q) {
                    if (tiles) tiles[q] = make_int2(I, J);
                    if (tpair) tpair[q] = y;
                }
            if (pairs) pairs[y] = GramPair{P, Q, q0, q - q0, P == Q ? (j1 - 8 * P) / 2 + 1 : j1 - 8 * Q, 0, 0, 0};
        }
    if (npair) *npair = y;
    return q;
}

// workgroups of a Gram of up to 64 columns (environment CTPWA_GRAM_WGS overrides it for
// measurements): as many as fit on the chip at once by their registers, three per CU for up to
// three tiles of FP32 columns, else two.  One more runs as a second round (four over 512: 611 us
// for the FP32 rows of 3.05M events, 378 us without, with three per CU 325 us).
extern "C" __attribute__((visibility("hidden"))) int ctpwa_gram_nwg(int f32, int ncol) {
    static const int n = [] {
        const char* e = std::getenv("CTPWA_GRAM_WGS");
        return e ? std::max(32, std::atoi(e) / 4) : 0;
    }();
    return n ? n : f32 && ncol <= 48 ? 768 : 512;
}

// weighted Gram on the matrix cores of the pieces' rows (rpe rows per event), up to 64 columns:
// partials [ghi of the last piece][tile pairs][256]; FP64 input, or FP32 input (f32 = 1)
extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_gram_panels(const void* X, int f32, int ncol, long long ldx, const HessPieces* H,
                                                                                     int rpe, const double* Wt, double* part,
                                                                                     hipStream_t s) {
    if (ncol <= 0 || H->n <= 0) return hipSuccess;
    if (ncol > 64) return hipErrorInvalidValue;
    const dim3 g(H->ghi[H->n - 1]), b(64 * GP_WAVES);
#define GP_LAUNCH(TT, NTT)                                                                                            \
    hipLaunchKernelGGL((k_gram_panels<TT, NTT>), g, b, gram_panels_lds(f32 != 0, NTT), s, (const TT*)X, ncol, ldx, *H, rpe, \
                       Wt, part)
    switch ((ncol + 15) / 16 + (f32 ? 4 : 0)) {
    case 1: GP_LAUNCH(double, 1); break;
    case 2: GP_LAUNCH(double, 2); break;
    case 3: GP_LAUNCH(double, 3); break;
    case 4: GP_LAUNCH(double, 4); break;
    case 5: GP_LAUNCH(float, 1); break;
    case 6: GP_LAUNCH(float, 2); break;
    case 7: GP_LAUNCH(float, 3); break;
    default: GP_LAUNCH(float, 4); break;
    }
#undef GP_LAUNCH
    return hipGetLastError();
}

// more than 64 columns, one piece: rows X[col ldx + row], nwg workgroups as set in pairs, then
// the sums into tot (first: set, else add)
extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_gram_wide(const void* X, int f32, int ncol, long long ldx, long long nrows, long long nev, const double* Wt,
                                                                                   const GramPair* pairs, int npair, const int2* tiles,
                                                                                   const int* tpair, int ntp, int nwg, double* part,
                                                                                   double* tot, int first, hipStream_t s) {
    const dim3 g(nwg), b(64 * GW_WAVES);
    if (f32)
        hipLaunchKernelGGL(k_gram_wide<float>, g, b, gram_wide_lds<float>(), s, (const float*)X, ncol, ldx, nrows, (int)nev, Wt, pairs,
                           npair, part);
    else
        hipLaunchKernelGGL(k_gram_wide<double>, g, b, gram_wide_lds<double>(), s, (const double*)X, ncol, ldx, nrows, (int)nev, Wt, pairs,
                           npair, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_accum_wide, dim3(4 * ntp), dim3(64 * HA_WAVES), 0, s, part, pairs, tiles, tpair, ncol, tot, first);
    return hipGetLastError();
}

// a pass's sums (k_hess_accum)
extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_hess_accum(
    const HessPieces* H, const HessPieces* HU, const HessTotals* T, const double* gpart, int ntp, const int2* tiles, int ncol,
    const double* upart, int utp, const int2* utiles, int ucol, const double* zpart, int nz, int nwg, const int* perm,
    hipStream_t s) {
    const unsigned nx = (unsigned)(4 * ntp + 4 * utp + (nz + HA_WAVES - 1) / HA_WAVES);
    hipLaunchKernelGGL(k_hess_accum, dim3(nx, (unsigned)std::max(H->n, HU->n)), dim3(64 * HA_WAVES), 0, s, *H, *HU, *T, gpart,
                       ntp, tiles, ncol, upart, utp, utiles, ucol, zpart, nz, nwg, perm);
    return hipGetLastError();
}

extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_gram_to_complex(const double* G, int n, double* Q,
                                                                                        hipStream_t s) {
    hipLaunchKernelGGL(k_gram_to_complex, dim3((n * n + 255) / 256), dim3(256), 0, s, G, n, Q);
    return hipGetLastError();
}

extern "C" __attribute__((visibility("hidden"))) hipError_t ctpwa_launch_hess_assemble(const HessAsm* h, hipStream_t s) {
    const int np = 2 * h->nfree + h->ntheta;
    const long long nm = (long long)np * np;
    hipLaunchKernelGGL(k_hess_out, dim3((unsigned)((nm + 255) / 256)), dim3(256), 0, s, *h);
    return hipGetLastError();
}
