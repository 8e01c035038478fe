// m3d_basic.hpp -- basic (Moulinec-Suquet) scheme with mixed control and the
// J2 / damage constitutive updates: runAnalysis "ep" / "ed",
// src/3d/FFT_analysis3D.cpp:796-853.
//
// Per iteration (one stage = four kernels; m3d_basic.hip and
// m3d_flex_basic.hip hold them, the finalisers run inside the y passes):
//   z    : c2r along z of eps^ (6 comps) -> eps;  constitutive() -> sigma
//          (elastoPlastic :640-691 or elastoDamage :619-638, per voxel,
//          history in HBM); FP64 partial sums of every component of sigma and
//          eps (updateE :583-594 needs the means); r2c along z of sigma (and,
//          in the start stage, of eps)
//   fin1 : itNo, diff_sum_field (:399, with the E of the Green step that made
//          this iterate), updateE -> E for the next Green step
//   y    : forward FFT along y
//   x    : forward FFT along x; eqVar partials from sigma^ (convergenceCheck
//          :351-389 -- the reference transforms sigma once more for it, here it
//          is the spectrum the next Green step uses anyway); Green step
//          t3 = eps^ - Gamma0:sigma^ (multiplyGF :323-338), DC = E N; inverse
//          FFT along x of the 6 output components
//   fin2 : eqVar, diff_avr_eqVar, stop rule (:820-826)
//   y    : inverse FFT along y (6 components)
// The reference medium is always the strain-based Gamma0 with arithmetic
// means of lambda and mu (:517-521).
#pragma once
#include "m3d_kernels.hpp"

namespace m3d {

enum { BEH_EP = 1, BEH_ED = 2 };
// FINAL: the fields and state of the last iterate
// of an increment, recomputed from the Green output its z pass read (the
// FP64 iterations do not write them)
enum { BMODE_START = 0, BMODE_ITER = 1, BMODE_RESTART = 2, BMODE_FINAL = 3 };
constexpr int NBSUM = 12; // sums per solve in the z pass: sigma_c, eps_c

template <typename T>
struct BPtr {
    T* eps;          // 6N per solve (sU stride)
    T* sig;          // 6N
    T* sig_old;      // 6N  ("ep")
    T* eps_old;      // 6N
    T* ep;           // N   equivalent plastic strain ("ep") / damage d ("ed")
    T* phi;          // N   yield function of the last constitutive call ("ep")
    T* dep;          // N   plastic multiplier increment ("ep")
    T* seff;         // N   von Mises stress after the return map ("ep")
    T* sig_star;     // 6N  sigma_old - C eps_old, once per increment ("ep", FP64)
    double* pfin;    // [14][nbz] block sums of the fused FINAL pass ("ep", FP64)
    long long sU;    // per-solve stride of the 6N fields
    long long sN;    // per-solve stride of the N fields
    cx<T>* S6;       // Green output, 6 components (read by the z pass)
    cx<T>* S12;      // [sigma^ | eps^], 12 components (START) or sigma^, 6 components (ITER)
    cx<T>* S6w;      // Green output written by the x pass (the other S6 buffer)
    cx<T>* Eh;       // eps^ after the Green step (specialised x pass: in its tile order)
    long long sS6, sS12;
    const uint8_t* ph;
    const double* mat; // per phase {la, mu, Sy, H, n, P, Y0, 0}
    const cx<T>* twz;
    const cx<T>* twy;
    const cx<T>* twx;
    double* psum;    // [nsolve][NBSUM][nbz]
    double* pchk;    // [nsolve][nbx + 1]
    Ctl* ctl;
};

// von Mises stress and deviator, sigma_eff_calculator :597-606
template <typename T>
__device__ __forceinline__ T vm_eff(const T* s, T* sd)
{
    const T sm = (s[0] + s[1] + s[2]) / T(3);
#pragma unroll
    for (int c = 0; c < 6; ++c) sd[c] = s[c] - (c < 3 ? sm : T(0));
    return sqrt(T(1.5)) * sqrt(sd[0] * sd[0] + sd[1] * sd[1] + sd[2] * sd[2] + T(2) * sd[3] * sd[3] +
                               T(2) * sd[4] * sd[4] + T(2) * sd[5] * sd[5]);
}

// isotropic C d with C = lambda tr I + 2 mu (tensor shears)
template <typename T>
__device__ __forceinline__ void iso_C(T la, T mu, const T* d, T* o)
{
    const T tr = d[0] + d[1] + d[2];
#pragma unroll
    for (int c = 0; c < 6; ++c) o[c] = T(2) * mu * d[c] + (c < 3 ? la * tr : T(0));
}

// elastoPlastic for one voxel.  Returns false when the Newton iteration for
// the plastic multiplier produces NaN (the reference terminates) or does not
// reach |res| < 1e-5 within 200 steps.
// LIN: every phase has hardening exponent n = 1, where pow(a, 1) = a and
// pow(a, 0) = 1 exactly, so the same arithmetic runs without the pow code
// (and its registers)
// STAR: the trial stress sigma_old + C (eps - eps_old) is formed as
// sig_star + C eps with sig_star = sigma_old - C eps_old kept per increment
// (passed in sig_old; eps_old unused): one 6-vector read instead of two
template <typename T, bool LIN = false, bool STAR = false>
__device__ __forceinline__ bool j2_update(const double* m, const T* eps, const T* eps_old, const T* sig_old, T ep_eff,
                                          T* sig, T& phi, T& dep, T& seff)
{
    const T la = T(m[0]), mu = T(m[1]), Sy = T(m[2]), H = T(m[3]), n = T(m[4]);
    T d[6], c[6], sd[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) d[k] = STAR ? eps[k] : eps[k] - eps_old[k];
    iso_C(la, mu, d, c);
#pragma unroll
    for (int k = 0; k < 6; ++k) sig[k] = sig_old[k] + c[k];
    seff = vm_eff(sig, sd);
    auto pw = [&](T a, T e) {
        if constexpr (LIN) return e == T(0) ? T(1) : a; // e is n or n - 1 with n = 1
        else return pow(a, e);
    };
    phi = seff - Sy - H * pw(ep_eff, n);
    if (phi > T(0)) {
        T x = 0, x_o = 0, res;
        bool ok = false;
        if (sizeof(T) == 4 && n == T(1)) {
            // FP32 phase, linear hardening: the root of
            // seff - 3 mu x - Sy - H (ep + x) = 0 (the reference's first Newton
            // step from x = 0 is this root)
            x = phi / (T(3) * mu + H);
            ok = true;
        } else {
            // FP32: |res| < 1e-5 is below the resolution of stresses in FP32,
            // so the FP32 phase stops at a residual relative to the yield
            // stress; the FP64 polish applies the reference's absolute rule
            const T rtol = sizeof(T) == 4 ? T(1e-6) * (Sy + seff) : T(1e-5);
            for (int iter = 0; iter < 200; ++iter) {
                x = x_o - (seff - T(3) * mu * x_o - Sy - H * pw(ep_eff + x_o, n)) /
                              (-T(3) * mu - H * n * pw(ep_eff + x_o, n - T(1)));
                x_o = x;
                res = seff - T(3) * mu * x - Sy - H * pw(ep_eff + x, n);
                if (isnan(x)) break;
                if (fabs(res) < rtol) { ok = true; break; }
            }
        }
        if (!ok) return false;
        dep = x;
        // sigma -= (1.5 x / seff) C sd; C sd = 2 mu sd for the deviator
        const T f = T(1.5) * x / seff;
        iso_C(la, mu, sd, c);
#pragma unroll
        for (int k = 0; k < 6; ++k) sig[k] -= f * c[k];
        seff = vm_eff(sig, sd);
    } else {
        dep = T(0);
    }
    return true;
}

// elastoDamage for one voxel; d is read (previous iterate) and updated
template <typename T>
__device__ __forceinline__ void damage_update(const double* m, const T* eps, T& d, T* sig)
{
    const T la = T(m[0]), mu = T(m[1]), P = T(m[5]), Y0 = T(m[6]);
    T c[6];
    iso_C(la, mu, eps, c);
    const T Y = sqrt(c[0] * eps[0] + c[1] * eps[1] + c[2] * eps[2] + T(2) * c[3] * eps[3] + T(2) * c[4] * eps[4] +
                     T(2) * c[5] * eps[5]);
    const T d_old = d;
    if (Y > Y0) {
        const T dn = T(1) - exp(-P * (Y - Y0));
        d = dn > d_old ? dn : d_old;
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) sig[k] = (T(1) - d) * c[k];
}

// ----------------------------------------------------------- finalisers
// S0 u for the isotropic reference medium: S0 = (1/3K0) J + (1/2mu0) Kdev
__device__ __forceinline__ void s0_apply(double la0, double mu0, const double* u, double* o)
{
    const double K0 = la0 + 2.0 * mu0 / 3.0;
    const double a = 1.0 / (3.0 * K0), b = 1.0 / (2.0 * mu0);
    const double t = (u[0] + u[1] + u[2]) / 3.0;
    for (int c = 0; c < 6; ++c) o[c] = b * u[c] + (c < 3 ? (a - b) * t : 0.0);
}

__device__ __forceinline__ double prod6(const double* a, const double* b)
{
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + 2 * a[3] * b[3] + 2 * a[4] * b[4] + 2 * a[5] * b[5];
}

// updateE, FFT_analysis3D.cpp:583-594, from the means of sigma and eps
__device__ __forceinline__ void update_E(Ctl& c, const double* sbar, const double* ebar)
{
    double S0s[6], y[6], x[6];
    s0_apply(c.la0, c.mu0, sbar, S0s);
    for (int i = 0; i < 6; ++i) x[i] = S0s[i] - ebar[i];
    s0_apply(c.la0, c.mu0, c.X0, y);
    const double k = (c.dEsum * c.incNo + prod6(x, c.X0)) / prod6(y, c.X0);
    for (int i = 0; i < 6; ++i) c.E[i] = k * y[i] - S0s[i] + ebar[i];
}

// MODE_START: after the increment's first constitutive call (:809):
//   sum_field_old = sum(sigma^0); E <- updateE(sigma^0, eps^0); itNo = 0
// MODE_ITER : itNo += 1, diff_sum_field with the E that produced this
//   iterate (:399), sum_field_old for the next check, E <- updateE
// MODE_RESTART: the iterate itNo recomputed in FP64 from its FP32 strain
//   (end of an FP32 phase): sum_field_old and E as in MODE_ITER, itNo kept;
//   the check after it records eqVar without a stop decision
//
// Both finalisers are one workgroup's work and nothing in a y pass depends on
// them (the x pass needs the new E, the next z pass the stop flag), so they run
// as the first workgroup of the y passes instead of as launches of their own:
// at 64^3 three launches of 4.6, 12 and 4.7 us per iteration less, of 77 us.
// They finish well inside the y pass from 32^3 (1024 partial sums each) to
// 192^3 (18 432).  The sums are taken in a fixed order, so the result does not
// depend on timing.
struct BFin {
    int kind;           // 0: none, 1: after the z pass, 2: after the x pass
    int mode;           // kind 1: BMODE_START, BMODE_ITER or BMODE_RESTART
    int n;              // partial sums (per sum)
    double invN;
    const double* part; // kind 1: [NBSUM][n]; kind 2: [n + 1]
    unsigned long long* hs; // kind 2: the iterations' published state (publish)
};

// kind 1: the NBSUM sums, then itNo, diff_sum_field and E
__device__ __forceinline__ void bfin1(Ctl& c, const BFin& f, double (*red)[NBSUM])
{
    double m[NBSUM];
#pragma unroll
    for (int q = 0; q < NBSUM; ++q) m[q] = 0;
#pragma unroll 2
    for (int i = threadIdx.x; i < f.n; i += blockDim.x)
#pragma unroll
        for (int q = 0; q < NBSUM; ++q) m[q] += f.part[(long long)q * f.n + i];
#pragma unroll
    for (int q = 0; q < NBSUM; ++q) {
        const double v = wave_sum(m[q]);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][q] = v;
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    double mq = 0; // lane q: sum q
    if (threadIdx.x < NBSUM)
        for (int w = 0; w < (int)blockDim.x >> 6; ++w) mq += red[w][threadIdx.x];
#pragma unroll
    for (int q = 0; q < NBSUM; ++q) m[q] = __shfl(mq, q, 64);
    if (threadIdx.x == 0) {
        double sbar[6], ebar[6], S = 0;
        for (int q = 0; q < 6; ++q) {
            sbar[q] = m[q] * f.invN;
            ebar[q] = m[6 + q] * f.invN;
            S += m[q];
        }
        if (f.mode == BMODE_ITER) {
            c.it += 1;
            double es = 0;
            for (int q = 0; q < 6; ++q) es += c.E[q];
            c.dsum = fabs((S - c.sum_prev) / (c.nc * es));
            c.first = 0;
        } else if (f.mode == BMODE_RESTART) {
            c.first = 2;
        } else {
            c.it = 0;
            c.first = 1;
        }
        c.sum_prev = S;
        update_E(c, sbar, ebar);
    }
}

// Stop rule (:820-826).  It runs beside the tiles of the inverse y pass, which
// test `done`, so the decision goes to `stop`: a word of its own that only later
// launches test.  The next z pass tests it alone and, in its first workgroup,
// sets `done` for the y and x passes after it.  So no launch writes a word that
// decides whether its own workgroups run, and all waves of a workgroup agree.
__host__ __device__ inline void bstop_rule(Ctl& c)
{
    if (c.err) c.stop = 3;
    else if (c.it > 1 && fabs(c.deq) < c.tol_eq && fabs(c.dsum) < c.tol_f) c.stop = 1;
    else if (c.it > c.cap) c.stop = 2;
}
// a z pass's workgroup has nothing to do; first: the launch's first thread
__host__ __device__ inline bool bz_skip(Ctl& c, bool first)
{
    if (!c.stop) return false;
    if (first) c.done = c.stop;
    return true;
}

// kind 2: eqVar of this iterate, diff_avr_eqVar, stop rule
__device__ __forceinline__ void bfin2(Ctl& c, const BFin& f, double* red)
{
    const double cc = ordered_sum(f.part, f.n, red);
    if (threadIdx.x == 0) {
        if (c.first == 1) return; // the stage after the increment start checks nothing
        const double eq = cc / f.part[f.n] * f.invN;
        if (c.first == 2) {
            // restart stage: eqVar of the recomputed iterate, no stop decision
            c.eq_val = eq;
            c.eqvar = eq;
            c.first = 0;
            return;
        }
        c.deq = fabs(eq - c.eq_val);
        c.eq_val = eq;
        c.eqvar = eq;
        bstop_rule(c);
        publish(c, f.hs, 0);
    }
}

// a y pass's first workgroup; it writes nothing that the others read
__device__ __forceinline__ void bfin_block(Ctl& c, const BFin& f, double (*red)[NBSUM])
{
    if (c.done) {
        if (f.kind == 2 && threadIdx.x == 0) publish(c, f.hs, 0);
        return;
    }
    if (f.kind == 1) bfin1(c, f, red);
    else if (f.kind == 2) bfin2(c, f, &red[0][0]);
}

// sums for export_homogen_var (:722-746): eps_c, sigma_c, seff|d, ep (14 per solve)
template <typename T, int BEH>
__global__ void __launch_bounds__(256) k_bsums(Geo g, BPtr<T> p, double* out, int nblk)
{
    __shared__ double red[256 / 64];
    const int s = blockIdx.y;
    double a[14];
    for (int q = 0; q < 14; ++q) a[q] = 0;
    for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < g.N; v += (long long)gridDim.x * blockDim.x) {
        for (int c = 0; c < 6; ++c) {
            a[c] += (double)p.eps[(long long)s * p.sU + v * 6 + c];
            a[6 + c] += (double)p.sig[(long long)s * p.sU + v * 6 + c];
        }
        if (BEH == BEH_EP) {
            a[12] += (double)p.seff[(long long)s * p.sN + v];
            a[13] += (double)p.ep[(long long)s * p.sN + v];
        } else {
            a[12] += (double)p.ep[(long long)s * p.sN + v];
        }
    }
    for (int q = 0; q < 14; ++q) {
        const double b = block_sum(a[q], red);
        if (threadIdx.x == 0) out[((long long)s * 14 + q) * nblk + blockIdx.x] = b;
    }
}

// update_old_Variable, FFT_analysis3D.cpp:693-719
template <typename T, int BEH>
__global__ void k_bupdate(Geo g, BPtr<T> p, int nsolve)
{
    // element-wise over the 6N tensors and the N scalars (consecutive
    // threads, consecutive values)
    const long long st = (long long)gridDim.x * blockDim.x;
    const long long i0 = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    for (int s = 0; s < nsolve; ++s) {
        const long long b6 = (long long)s * p.sU, b1 = (long long)s * p.sN;
        for (long long i = i0; i < 6 * g.N; i += st) {
            if (BEH == BEH_EP) p.sig_old[b6 + i] = p.sig[b6 + i];
            const T e = p.eps[b6 + i], tmp = p.eps_old[b6 + i];
            p.eps_old[b6 + i] = e;
            p.eps[b6 + i] = e + (e - tmp);
        }
        if (BEH == BEH_EP)
            for (long long v = i0; v < g.N; v += st)
                if (p.phi[b1 + v] > T(0)) p.ep[b1 + v] += p.dep[b1 + v];
    }
}

// the 14 export sums of the fused FINAL pass: its block sums pfin[q][nbz],
// added in nblk contiguous shares (fixed order), out[q][b] as k_bsums writes
template <int U = 0> // a template so that every unit including this header may instantiate it
__global__ void __launch_bounds__(256) k_bfsums(Geo g, const double* pfin, double* out, int nblk)
{
    __shared__ double red[256 / 64];
    const int q = blockIdx.y, b = blockIdx.x;
    const int per = (g.nbz + nblk - 1) / nblk;
    const int i0 = b * per, i1 = min(g.nbz, i0 + per);
    double v = 0;
    for (int i = i0 + threadIdx.x; i < i1; i += blockDim.x) v += pfin[(long long)q * g.nbz + i];
    v = block_sum(v, red);
    if (threadIdx.x == 0) out[(long long)q * nblk + b] = v;
}

// sigma_star = sigma_old - C eps_old for the next increment's start stage
// ("ep", FP64), after k_bupdate (one solve)
template <typename T>
__global__ void k_bstar(Geo g, BPtr<T> p)
{
    for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < g.N; v += (long long)gridDim.x * blockDim.x) {
        const double* mt = p.mat + p.ph[v] * 8;
        T eo[6], ce[6];
        for (int c = 0; c < 6; ++c) eo[c] = p.eps_old[v * 6 + c];
        iso_C(T(mt[0]), T(mt[1]), eo, ce);
        for (int c = 0; c < 6; ++c) p.sig_star[v * 6 + c] = p.sig_old[v * 6 + c] - ce[c];
    }
}

// copy fields between the FP64 and FP32 states of a solve; what: 1 eps,
// 2 sig, 4 sig_old, 8 eps_old, 16 ep|d, 32 phi, dep and seff, 64 the Green
// output spectrum S6 (6 x H complex)
enum { BC_EPS = 1, BC_SIG = 2, BC_SIGOLD = 4, BC_EPSOLD = 8, BC_EP = 16, BC_PHI = 32, BC_S6 = 64 };
template <typename TS, typename TD>
__global__ void k_bcopy(Geo g, BPtr<TS> a, BPtr<TD> b, int what)
{
    const long long n6 = 6 * g.N, n1 = g.N, h6 = 6 * g.H;
    const long long i0 = blockIdx.x * (long long)blockDim.x + threadIdx.x, st = (long long)gridDim.x * blockDim.x;
    for (long long i = i0; i < n6; i += st) {
        if (what & BC_EPS) b.eps[i] = TD(a.eps[i]);
        if (what & BC_SIG) b.sig[i] = TD(a.sig[i]);
        if (what & BC_SIGOLD) b.sig_old[i] = TD(a.sig_old[i]);
        if (what & BC_EPSOLD) b.eps_old[i] = TD(a.eps_old[i]);
    }
    for (long long i = i0; i < n1; i += st) {
        if (what & BC_EP) b.ep[i] = TD(a.ep[i]);
        if (what & BC_PHI) {
            b.phi[i] = TD(a.phi[i]);
            b.dep[i] = TD(a.dep[i]);
            b.seff[i] = TD(a.seff[i]);
        }
    }
    if (what & BC_S6)
        for (long long i = i0; i < h6; i += st) b.S6[i] = cx<TD>{TD(a.S6[i].re), TD(a.S6[i].im)};
}

template <typename T>
__global__ void k_binit(Geo g, BPtr<T> p, int nsolve, int beh)
{
    for (int s = 0; s < nsolve; ++s) {
        const Ctl& c = p.ctl[s];
        for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < g.N; v += (long long)gridDim.x * blockDim.x) {
            const long long i6 = (long long)s * p.sU + v * 6, i1 = (long long)s * p.sN + v;
            for (int k = 0; k < 6; ++k) {
                p.eps[i6 + k] = T(c.E[k]); // setLoad(dE, X0) (:799)
                p.eps_old[i6 + k] = T(0);
                if (beh == BEH_EP) p.sig_old[i6 + k] = T(0);
                if (beh == BEH_EP && p.sig_star) p.sig_star[i6 + k] = T(0); // sigma_old - C eps_old
            }
            p.ep[i1] = beh == BEH_EP ? T(.000000001236547) : T(0); // :67-69 / :89-90
        }
    }
}

} // namespace m3d
