// m3d_kernels.hpp -- gfx950 kernels of the FFT homogenization loop.
//
// One accelerated (Eyre-Milton) iteration of src/3d/FFT_analysis3D.cpp:751-794
// (and src/3dTherm/FFT_thermal3D.cpp:446-485) is realised as four passes over
// HBM, all working in place on one half-spectrum buffer per solve:
//
//   zpass  (MODE_IUF): c2r along z of the Green output  -> u_c
//                      u <- u + A(x)(u_c - u)            (update,  :283-295)
//                      v  = M(x) u, FP64 partial sums    (multipCx :236-247, sum_field)
//                      tau = (M(x) - M0) u               (polarisation :757-767)
//                      r2c along z of tau
//   ypass  (fwd)     : complex FFT along y
//   xgreen           : complex FFT along x, u_c^ = -G0(xi) tau^ / N, DC = E
//                      (multiplyGF :297-348 with the Nyquist projection that
//                      FFTW's c2r applies), inverse FFT along x
//   ypass  (inv)     : inverse complex FFT along y
//
// The equilibrium check (convergenceCheck :351-416) needs the spectrum of
// sigma.  It is only needed when the stop rule can fire, i.e. when
// |diff_sum_field| < tol_field, so it runs on demand (zpass MODE_CHK, ypass,
// xcheck) and is skipped otherwise; the stop decision is the reference's.
//
// Layouts (AoS, the reference's own, FFT_analysis3D.cpp:110-150):
//   real field  U[((x*Ny + y)*Nz + z)*C + c]
//   spectrum    S[((x*Ny + y)*Nzh + kz)*C + c],  Nzh = Nz/2 + 1
// Tensor index 0 is the z axis, 1 is y, 2 is x (FFT_analysis3D.cpp:211).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "m3d_fft.hpp"

namespace m3d {

constexpr int NCOEF = 8; // per-phase coefficients

// z-pass modes: forward only, update (inverse, update, forward), check FFT of
// the current / previous iterate, update of an anchored FP32 correction (adds
// r), the FP64 anchor iteration of the polish (inverse and update only;
// writes r = u_new - u_old and the first correction e = r in FP32), and the
// FP64 start of the polish from the FP32 iterate (forward only; reads the
// FP32 ring, writes the promoted FP64 iterate).
enum { MODE_FWD = 0, MODE_IUF = 1, MODE_CHK_CUR = 2, MODE_CHK_PREV = 3, MODE_IUFR = 4, MODE_IUA = 5, MODE_FWDP = 6 };
enum { BUF_MAIN = 0, BUF_CHK_CUR = 2, BUF_CHK_PREV = 3, BUF_K = 4 };

// per-solve control block, read and written on the device only
struct Ctl {
    int it;        // itNo
    int done;      // 0 running, 1 converged, 2 iteration cap
    int need_cur;  // equilibrium check of the current iterate needed
    int need_prev; // ... and of the previous iterate
    int eq_it;     // iterate index eq_val belongs to (-1: none)
    int cap;       // iteration cap (reference: 2000 / 500)
    int first;     // basic scheme: 1 while the stage after the increment start runs
    int err;       // basic scheme: constitutive update failed (Newton NaN / no convergence)
    int sb;        // elastic: 1 strain base, 0 stress base; thermal: 1 gradient base
    // anchored polish: the iterate is A + e with the FP64 anchor A (iterate
    // anc_it of the FP64 ring) and an FP32 correction e (FP32 ring); the
    // FP32 passes iterate e <- r + M e (r = T(A) - A, load term dropped)
    int corr;
    int anc_it;
    // 1: the iterate needs a check that the launched sequence does not hold;
    // the solve stands still until one that does (k_finA)
    int wait;
    int tick; // states published to the host since the loop began (publish)
    int stop; // basic scheme: value of `done` that the stop rule decided on (bstop_rule)
    double sum_anchor; // sum of the dual field of the anchor (FP64)
    double sum_prev;  // sum of the dual field at iterate `it`
    double eq_val;    // eqVar at iterate eq_it
    double dsum, deq, eqvar;
    double tol_f, tol_eq;
    double norm;      // N * (M[0]_00/2 + M[1]_00/2) * sum(E)
    double E[6];      // macroscopic load (DC of the Green output)
    // basic scheme with mixed control (updateE, FFT_analysis3D.cpp:583-594)
    double X0[6];     // stress direction
    double dEsum;     // dE.sum()
    double incNo;     // increment number (1-based)
    double nc;        // N * (C[0]_00/2 + C[1]_00/2): Delta-sum normalisation without sum(E)
    double la0, mu0;  // reference medium (S0 = C0^-1 applied in closed form)
    double dsum_hist[16]; // dsum of iterate i at [i % 16] (how far an FP32 switch rolls back)
};

struct Geo {
    int Nx, Ny, Nz, Nzh, C;
    long long N, H;
    FftAxis az, ay, ax; // radix plans of the run-time-length passes (m3d_flex.hpp)
    int zeven;
    int TY, nty;        // z tiles: TY lines (y) per tile, Ny/TY tiles per x plane
    int TKy, nky;       // y tiles: TKy kz values, ceil(Nzh/TKy) tiles
    int TKx, nkx;       // x tiles
    int nsolve;
    int nbz, nbx;       // blocks per solve of the z pass and the x pass
    int TKc, nbc;       // x pass of the equilibrium check: kz tile, partial sums per solve
    double invN;
    // spectrum layout: the half-spectrum row
    // (x, y) (Nzh*C complex values) starts at
    //   (x >> lxb) * sxa + (x & xbm) * sxb + y * sy
    // plain rows: lxb = 0, xbm = 0, sxa = Ny*Nzh*C (+ padding), sy = Nzh*C;
    // x planes in blocks of 2^lxb: sxa = Ny*2^lxb*Nzh*C, sxb = Nzh*C, sy = 2^lxb*Nzh*C
    int lxb, xbm;
    long long sxa, sxb, sy;
    long long spec;     // complex values of one solve's spectrum (rows + padding)
    int fz, fy, fx;     // host only: compile-time specialised kernel used for this axis
};

template <typename T>
struct Ptr {
    T* U;                   // ring of `ring` iterate buffers, each holding every solve
    long long sU;           // per-solve stride of U (reals)
    long long sB;           // stride between ring buffers (reals)
    int ring;               // iterate j lives in buffer j mod ring
    cx<T>* S;               // main spectrum
    cx<T>* K;               // check spectrum
    long long sS;           // per-solve stride of S and K (complex)
    const uint8_t* ph;      // phase ids, per RVE
    long long sPh;
    const int* rve_of;      // solve -> RVE index
    const T* coef;          // per RVE: [maxph][NCOEF]
    int sCoef;
    const cx<T>* twz;
    const cx<T>* twy;
    const cx<T>* twx;
    double* psum;           // z-pass partial sums, [nsolve][nbz]
    double* pchk;           // check partials, [nsolve][2][nbc + 1]
    Ctl* ctl;
    // anchored polish (solves with ctl.corr): FP32 passes add R to the
    // update; FP64 passes read the iterate as U[anc_it] + e, e from the FP32
    // ring eU (stride eB between ring buffers, `ering` buffers)
    const float* R;
    const float* eU;
    long long eB;
    int ering;
};

// ----------------------------------------------------------------- physics
// Elastic: isotropic maps M u = a tr(u)/3 I + b dev(u) on Voigt vectors with
// tensor shears ([11,22,33,23,13,12], FFT_analysis3D.cpp:457-462).
struct Elastic {
    static constexpr int C = 6;
    // workgroups of a check-pass launch: the check is rarely needed (Δsum
    // reaches its tolerance near the stop), so the launches that leave at
    // once dominate and a smaller grid wins (measured: 8192 against 32768,
    // 256^3 headline -1.5%, 64-RVE batch -2.3%)
    static constexpr int chk_grid = 8192;
    template <typename T>
    __device__ static __forceinline__ void iso(T a, T b, const T* u, T* o)
    {
        const T t = (u[0] + u[1] + u[2]) * T(1.0 / 3.0);
        const T q = (a - b) * t;
        o[0] = b * u[0] + q;
        o[1] = b * u[1] + q;
        o[2] = b * u[2] + q;
        o[3] = b * u[3];
        o[4] = b * u[4];
        o[5] = b * u[5];
    }
    // coef: [a_v,b_v, a_t,b_t, a_a,b_a]
    template <typename T>
    __device__ static __forceinline__ void dual(const T* k, const T* u, T* o) { iso(k[0], k[1], u, o); }
    template <typename T>
    __device__ static __forceinline__ void polar(const T* k, const T* u, T* o) { iso(k[2], k[3], u, o); }
    template <typename T>
    __device__ static __forceinline__ void accel(const T* k, const T* u, T* o) { iso(k[4], k[5], u, o); }
    // frequency map, FFT_analysis3D.cpp:202-209
    __device__ static __forceinline__ int fmap(int k, int N) { return k <= (N - 1) / 2 ? k : -(N - k); }
    __device__ static __forceinline__ int fmapx(int k, int Nx, int Ny) { return fmap(k, Nx); }
};

// Thermal: scalar conductivities, 3 components (FFT_thermal3D.cpp:180-268).
struct Thermal {
    static constexpr int C = 3;
    // at high conductivity contrast the check runs in most iterations (the
    // 512^3 three-phase workload: every one), where 32768 workgroups beat 8192
    // by 2.5%
    static constexpr int chk_grid = 32768;
    // coef: [k_v, k_t, k_a]
    template <typename T>
    __device__ static __forceinline__ void dual(const T* k, const T* u, T* o)
    {
        o[0] = k[0] * u[0]; o[1] = k[0] * u[1]; o[2] = k[0] * u[2];
    }
    template <typename T>
    __device__ static __forceinline__ void polar(const T* k, const T* u, T* o)
    {
        o[0] = k[1] * u[0]; o[1] = k[1] * u[1]; o[2] = k[1] * u[2];
    }
    template <typename T>
    __device__ static __forceinline__ void accel(const T* k, const T* u, T* o)
    {
        o[0] = k[2] * u[0]; o[1] = k[2] * u[1]; o[2] = k[2] * u[2];
    }
};

// ------------------------------------------------------- Green operators
// per-solve constants of the isotropic Green operators, computed once per
// tile instead of per frequency (same values and operation order as the
// per-frequency expressions they replace)
template <typename T>
struct GreenK {
    T la0, mu0;
    T d2;   // (la0 + mu0) / (mu0 (la0 + 2 mu0))
    T c3;   // 2 la0 mu0 / (la0 + 2 mu0)
    T m2;   // 2 mu0
    T h2mu; // 1 / (2 mu0): FP32 multiplies by it where FP64 divides
    T k0;   // thermal reference conductivity
};

template <typename T>
__device__ __forceinline__ GreenK<T> green_k(T la0, T mu0)
{
    GreenK<T> K;
    K.la0 = la0;
    K.mu0 = mu0;
    K.d2 = (la0 + mu0) / (mu0 * (la0 + T(2) * mu0));
    K.c3 = T(2) * la0 * mu0 / (la0 + T(2) * mu0);
    K.m2 = T(2) * mu0;
    K.h2mu = T(1) / (T(2) * mu0);
    K.k0 = T(0);
    return K;
}

// the constants of a solve's medium: elastic prm = {la0, mu0}, thermal {k0}
template <typename T, int C>
__device__ __forceinline__ GreenK<T> green_k_of(const T* prm)
{
    if constexpr (C == 6) return green_k<T>(prm[0], prm[1]);
    GreenK<T> K{};
    K.k0 = prm[0];
    return K;
}

// Strain base, Gamma0 (FFT_analysis3D.cpp:223-224) contracted with a
// symmetric tau (all shear pairs summed): closed form
//   (G:t)_ij = (xi_i (t xi)_j + xi_j (t xi)_i) / (2 mu0 |xi|^2)
//              - (la0+mu0)/(mu0(la0+2mu0)) xi_i xi_j (xi.t.xi) / |xi|^4
// Stress base, Delta0 (:226-228): with P = I - n n, n = xi/|xi|,
//   (D:t)_ij = c3 P_ij tr(P t) + 2 mu0 (P t P)_ij,  c3 = 2 la0 mu0/(la0+2mu0)
// Returns G:t (complex, per Voigt component).
template <typename T>
__device__ __forceinline__ void green_elastic_k(const T xi[3], const cx<T> t[6], cx<T> o[6], int strain_base,
                                                const GreenK<T>& K)
{
    const T n2 = xi[0] * xi[0] + xi[1] * xi[1] + xi[2] * xi[2];
    // FP32: the hardware reciprocal (1 ulp) in place of the IEEE division
    // sequence; FP32 iterates are refined in FP64, whose path divides exactly
    T inv;
    if constexpr (sizeof(T) == 4) inv = __builtin_amdgcn_rcpf(n2);
    else inv = T(1) / n2;
    // w = t xi, tensor from Voigt: 0:(0,0) 1:(1,1) 2:(2,2) 3:(1,2) 4:(0,2) 5:(0,1)
    cx<T> w0 = cscale(t[0], xi[0]) + cscale(t[5], xi[1]) + cscale(t[4], xi[2]);
    cx<T> w1 = cscale(t[5], xi[0]) + cscale(t[1], xi[1]) + cscale(t[3], xi[2]);
    cx<T> w2 = cscale(t[4], xi[0]) + cscale(t[3], xi[1]) + cscale(t[2], xi[2]);
    cx<T> s = cscale(w0, xi[0]) + cscale(w1, xi[1]) + cscale(w2, xi[2]);
    const cx<T> w[3] = {w0, w1, w2};
    const int pi[6] = {0, 1, 2, 1, 0, 0};
    const int pj[6] = {0, 1, 2, 2, 2, 1};
    if (strain_base) {
        T a;
        if constexpr (sizeof(T) == 4) a = inv * K.h2mu;
        else a = inv / (T(2) * K.mu0);
        const T b = K.d2 * inv * inv;
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const int i = pi[q], j = pj[q];
            cx<T> r = cscale(cscale(w[j], xi[i]) + cscale(w[i], xi[j]), a);
            o[q] = r - cscale(s, b * xi[i] * xi[j]);
        }
    } else {
        // n n = xi xi / n2 ; s/n2 = n.t.n ; w/|xi| = t n ; with
        // (P t P)_ij = t_ij - n_i w'_j - w'_i n_j + sn n_i n_j (w' = t n) and
        // P_ij = delta_ij - xi_i xi_j / n2 the output collects into
        //   o_ij = 2mu0 t_ij - (2mu0/n2)(xi_i w_j + xi_j w_i) + xi_i xi_j G + delta_ij D
        // with D = c3 tr(P t) and G = (2mu0 sn - D) / n2, formed once per frequency
        const cx<T> trt = t[0] + t[1] + t[2];
        const cx<T> sn = cscale(s, inv); // n.t.n
        const cx<T> D = cscale(trt - sn, K.c3);
        const cx<T> G = cscale(cscale(sn, K.m2) - D, inv);
        const T a = K.m2 * inv;
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const int i = pi[q], j = pj[q];
            const cx<T> x = cscale(w[j], xi[i]) + cscale(w[i], xi[j]);
            cx<T> r = cscale(t[q], K.m2) - cscale(x, a) + cscale(G, xi[i] * xi[j]);
            if (i == j) r = r + D;
            o[q] = r;
        }
    }
}

template <typename T>
__device__ __forceinline__ void green_elastic(const T xi[3], const cx<T> t[6], cx<T> o[6], int strain_base,
                                              T la0, T mu0)
{
    green_elastic_k<T>(xi, t, o, strain_base, green_k<T>(la0, mu0));
}

// Thermal flux base:     D_ij = k0 (delta_ij - xi_i xi_j/|xi|^2) (:161-169)
template <typename T>
__device__ __forceinline__ void green_thermal(const T xi[3], const cx<T> t[3], cx<T> o[3], int grad_base, T k0)
{
    const T n2 = xi[0] * xi[0] + xi[1] * xi[1] + xi[2] * xi[2];
    cx<T> s = cscale(t[0], xi[0]) + cscale(t[1], xi[1]) + cscale(t[2], xi[2]);
    // FP32: hardware reciprocal, as in green_elastic
    auto rcp = [](T x) {
        if constexpr (sizeof(T) == 4) return __builtin_amdgcn_rcpf(x);
        else return T(1) / x;
    };
    if (grad_base) {
        const T a = rcp(k0 * n2);
#pragma unroll
        for (int c = 0; c < 3; ++c) o[c] = cscale(s, a * xi[c]);
    } else {
        const T a = rcp(n2);
#pragma unroll
        for (int c = 0; c < 3; ++c) o[c] = cscale(t[c] - cscale(s, a * xi[c]), k0);
    }
}

// ------------------------------------------------------------ reductions
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// deterministic block sum (fixed tree); result valid in thread 0
__device__ __forceinline__ double block_sum(double v, double* red)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0) {
        const int nw = (blockDim.x + 63) >> 6;
        for (int i = 0; i < nw; ++i) r += red[i];
    }
    return r;
}

template <typename T>
__device__ __forceinline__ T* u_buf(const Ptr<T>& p, int it, int s)
{
    int b = it % p.ring;
    if (b < 0) b += p.ring;
    return p.U + (long long)b * p.sB + (long long)s * p.sU;
}

// FP32 correction e of iterate `it` of an anchored solve
template <typename T>
__device__ __forceinline__ const float* e_buf(const Ptr<T>& p, int it, int s)
{
    int b = it % p.ering;
    if (b < 0) b += p.ering;
    return p.eU + (long long)b * p.eB + (long long)s * p.sU;
}

// ------------------------------------------------ x pass with Green step
// frequency vector (tensor order z, y, x) of spectrum index (kx, ky, kz)
__device__ __forceinline__ void freq_el(const Geo& g, int kx, int ky, int kz, int f[3])
{
    f[0] = Elastic::fmap(kz, g.Nz);
    f[1] = Elastic::fmap(ky, g.Ny);
    f[2] = Elastic::fmap(kx, g.Nx);
}

// thermal maps: gradient base and check use the N/2-positive map
// (FFT_thermal3D.cpp:113-120); flux base the (N-1)/2 map with -(Ny-x) for x (:150-151)
__device__ __forceinline__ int fmap_t(int k, int N) { return k <= N / 2 ? k : -(N - k); }
__device__ __forceinline__ void freq_th(const Geo& g, int sb, int kx, int ky, int kz, int f[3])
{
    if (sb) {
        f[0] = fmap_t(kz, g.Nz);
        f[1] = fmap_t(ky, g.Ny);
        f[2] = fmap_t(kx, g.Nx);
    } else {
        f[0] = Elastic::fmap(kz, g.Nz);
        f[1] = Elastic::fmap(ky, g.Ny);
        f[2] = kx <= (g.Nx - 1) / 2 ? kx : -(g.Ny - kx);
    }
}

template <typename T, typename PH>
__device__ __forceinline__ void green_apply_k(const Geo& g, int sb, const GreenK<T>& K, int kx, int ky, int kz, cx<T>* v)
{
    constexpr int C = PH::C;
    int f[3];
    if constexpr (C == 6) freq_el(g, kx, ky, kz, f);
    else freq_th(g, sb, kx, ky, kz, f);
    T xi[3] = {T(f[0]), T(f[1]), T(f[2])};
    cx<T> in[C], o[C];
#pragma unroll
    for (int c = 0; c < C; ++c) in[c] = v[c];
    if constexpr (C == 6) green_elastic_k<T>(xi, in, o, sb, K);
    else green_thermal<T>(xi, in, o, sb, K.k0);
    // c2r of a multi-dimensional half spectrum keeps only the Hermitian part
    // of the kz=0 and kz=Nz/2 planes: average with the operator of the
    // conjugate-partner index when its frequency vector is not -xi.
    const bool plane = (kz == 0) || (g.zeven && kz == g.Nz / 2);
    if (plane) {
        const int px = (g.Nx - kx) % g.Nx, py = (g.Ny - ky) % g.Ny;
        int fp[3];
        if constexpr (C == 6) freq_el(g, px, py, kz, fp);
        else freq_th(g, sb, px, py, kz, fp);
        if (fp[0] != -f[0] || fp[1] != -f[1] || fp[2] != -f[2]) {
            T xp[3] = {T(fp[0]), T(fp[1]), T(fp[2])};
            cx<T> o2[C];
            if constexpr (C == 6) green_elastic_k<T>(xp, in, o2, sb, K);
            else green_thermal<T>(xp, in, o2, sb, K.k0);
#pragma unroll
            for (int c = 0; c < C; ++c) o[c] = cscale(o[c] + o2[c], T(0.5));
        }
    }
    const T sc = T(-g.invN);
#pragma unroll
    for (int c = 0; c < C; ++c) v[c] = cscale(o[c], sc);
}

// ---------------------------------------------- x pass of the check FFT
// eqVar partials: mechanical sums kz >= 1 of sqrt|sum_c |s_c|^2 W_c| with
// W = (xi0^2, xi1^2, xi2^2, 2xi1+2xi2, 2xi0+2xi2, 2xi0+2xi1) (FFT_analysis3D.cpp:366-389);
// thermal sums kz >= 0 of sqrt(sum_c |q_c|^2 xi_c^2) (FFT_thermal3D.cpp:315-335).
// The term of frequency (kx, y, kz) with values v; a2: |v_c|^2.  The passes
// of compile-time lengths (fast::xy_tile, bfast::kxb) hold the same sum in
// place: through this function they come out with an addition of zero for
// kz = 0 and in another order.
template <typename T, int C>
__device__ __forceinline__ double eq_term(const Geo& g, int kx, int y, int kz, const cx<T>* v, double (&a2)[C])
{
#pragma unroll
    for (int c = 0; c < C; ++c) a2[c] = (double)v[c].re * (double)v[c].re + (double)v[c].im * (double)v[c].im;
    if constexpr (C == 6) {
        if (kz < 1) return 0.0;
        const double z0 = Elastic::fmap(kz, g.Nz), z1 = Elastic::fmap(y, g.Ny), z2 = Elastic::fmap(kx, g.Nx);
        const double q = a2[0] * z0 * z0 + a2[1] * z1 * z1 + a2[2] * z2 * z2 + a2[3] * ((z1 + z1) + (z2 + z2)) +
                         a2[4] * ((z0 + z0) + (z2 + z2)) + a2[5] * ((z0 + z0) + (z1 + z1));
        return sqrt(fabs(q));
    } else {
        const double z0 = fmap_t(kz, g.Nz), z1 = fmap_t(y, g.Ny), z2 = fmap_t(kx, g.Nx);
        return sqrt(a2[0] * z0 * z0 + a2[1] * z1 * z1 + a2[2] * z2 * z2);
    }
}

// the norm of the mean field from its |v_c|^2 at the zero frequency
template <int C>
__device__ __forceinline__ double eq_mean(const double (&a2)[C])
{
    if constexpr (C == 6) return sqrt(a2[0] + a2[1] + a2[2] + 2 * a2[3] + 2 * a2[4] + 2 * a2[5]);
    else return sqrt(a2[0] + a2[1] + a2[2]);
}

// ---------------------------------------------------------- finalizers
constexpr int FTHREADS = 256;
// the accelerated scheme's finalisers: one workgroup per solve over up to
// Nx*Ny/TY (z pass) or Ny*Nzh/TK (check x pass) partial sums, 65536 at 512^3
constexpr int ATHREADS = 1024;

// sum of a[0..n) by one workgroup in a fixed order: every thread keeps 8
// partial sums of its strided elements (8 loads in flight, not one chain of
// dependent adds), combined pairwise, then the workgroup's tree
__device__ __forceinline__ double ordered_sum(const double* a, int n, double* red)
{
    double p0 = 0, p1 = 0, p2 = 0, p3 = 0, p4 = 0, p5 = 0, p6 = 0, p7 = 0;
    const int st = blockDim.x;
    int i = threadIdx.x;
    for (; i + 7 * st < n; i += 8 * st) {
        p0 += a[i];
        p1 += a[i + st];
        p2 += a[i + 2 * st];
        p3 += a[i + 3 * st];
        p4 += a[i + 4 * st];
        p5 += a[i + 5 * st];
        p6 += a[i + 6 * st];
        p7 += a[i + 7 * st];
    }
    for (; i < n; i += st) p0 += a[i];
    return block_sum(((p0 + p1) + (p2 + p3)) + ((p4 + p5) + (p6 + p7)), red);
}

// after the forward-only z pass: sum of the dual field at the start iterate
template <int C>
__global__ void __launch_bounds__(ATHREADS) k_fin0(Geo g, Ctl* ctl, const double* psum)
{
    __shared__ double red[ATHREADS / 64];
    const int s = blockIdx.x;
    Ctl& c = ctl[s];
    const int done = c.done;
    __syncthreads();
    if (done) return;
    const double S = ordered_sum(psum + (long long)s * g.nbz, g.nbz, red);
    if (threadIdx.x == 0) {
        // anchored solves sum e; the anchor's sum completes the iterate's
        if (c.corr) c.sum_prev = S + c.sum_anchor;
        else {
            c.sum_prev = S;
            c.sum_anchor = S;
        }
        c.eq_it = -1;
        c.need_cur = 0;
        c.need_prev = 0;
        c.wait = 0;
    }
}

// check passes that follow the update pass in a launched iteration: none, the
// current iterate's, or also the previous iterate's (which only the first
// checked iterate of a solve needs)
enum { CHECKS_NONE = 0, CHECKS_CUR = 1, CHECKS_BOTH = 2 };

// What the host's loop knows of a solve: one word per solve in pinned host
// memory, (tick << 8) | flags, stored by the last finaliser of an iteration.
// One relaxed 64-bit store needs no fence, and reading it costs the stream
// nothing; a copy of the control blocks left the device idle for 18 us each
// time (9 us before the copy, 4 us of it, 5 us after).
enum { ST_DONE = 1, ST_WAIT = 2, ST_NEAR = 4, ST_CHECKED = 8 };
// "Near its stop": Delta-sum below this many tolerances.  Six load cases of
// 32^3 to 128^3, 64^3 and 96^3 thermal and a mixed batch, both precisions, a
// homogenization against 3: 10 within 1% (one thermal case 4% slower); 1.7 the
// same but for two cases 5% faster; 1 (a solve near its stop always waits once)
// up to 13% faster below 64^3 and within 2% above; checks in every iteration
// 1-14% slower.
constexpr double NEAR_TOL = 3.0;

__device__ __forceinline__ void publish(Ctl& c, unsigned long long* hs, int s)
{
    if (!hs) return;
    c.tick += 1;
    unsigned long long v = (unsigned long long)c.tick << 8;
    if (c.done || c.stop) v |= ST_DONE;
    if (c.wait) v |= ST_WAIT;
    if (c.it >= 1 && c.dsum < NEAR_TOL * c.tol_f) v |= ST_NEAR;
    if (c.eq_it == c.it) v |= ST_CHECKED;
    __hip_atomic_store(hs + s, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// after the update pass: itNo += 1, diff_sum_field, decide whether the
// equilibrium check is needed (FFT_analysis3D.cpp:392-416, stop rule :785-792).
// checks: what this iteration's launches hold.  A solve that needs more waits:
// every pass of it is skipped until an iteration that holds its checks, which
// then goes on from the same iterate (its update pass and this decision are
// not repeated).
template <int C>
__global__ void __launch_bounds__(ATHREADS) k_finA(Geo g, Ctl* ctl, const double* psum, int checks, unsigned long long* hs)
{
    __shared__ double red[ATHREADS / 64];
    const int s = blockIdx.x;
    Ctl& c = ctl[s];
    const int done = c.done, wait = c.wait;
    if (checks != CHECKS_NONE) hs = nullptr; // k_finB publishes
    __syncthreads();
    if (done || wait) {
        if (threadIdx.x == 0) {
            if (wait && checks >= (c.need_prev ? CHECKS_BOTH : CHECKS_CUR)) c.wait = 0;
            publish(c, hs, s);
        }
        return;
    }
    const double S0 = ordered_sum(psum + (long long)s * g.nbz, g.nbz, red);
    if (threadIdx.x == 0) {
        const double S = c.corr ? S0 + c.sum_anchor : S0;
        c.it += 1;
        c.dsum = fabs((S - c.sum_prev) / c.norm);
        c.dsum_hist[c.it & 15] = c.dsum;
        c.sum_prev = S;
        const int need = (c.it > 1) && (fabs(c.dsum) < c.tol_f);
        c.need_cur = need;
        c.need_prev = need && (c.eq_it != c.it - 1);
        c.wait = need && checks < (c.need_prev ? CHECKS_BOTH : CHECKS_CUR);
        if (!need && c.it > c.cap) c.done = 2;
        publish(c, hs, s);
    }
}

// after the check FFTs: eqVar, diff_avr_eqVar and the stop decision
template <int C>
__global__ void __launch_bounds__(ATHREADS) k_finB(Geo g, Ctl* ctl, const double* pchk, unsigned long long* hs)
{
    __shared__ double red[ATHREADS / 64];
    const int s = blockIdx.x;
    Ctl& c = ctl[s];
    const int done = c.done, need_cur = c.need_cur && !c.wait, need_prev = c.need_prev;
    __syncthreads();
    if (done || !need_cur) {
        if (threadIdx.x == 0) publish(c, hs, s);
        return;
    }
    const double* pc = pchk + (long long)s * 2 * (g.nbc + 1);
    const double cc = ordered_sum(pc, g.nbc, red);
    double ccp = 0;
    if (need_prev) ccp = ordered_sum(pc + g.nbc + 1, g.nbc, red);
    if (threadIdx.x == 0) {
        const double eq = cc / pc[g.nbc] * g.invN;
        const double eqp = need_prev ? (ccp / pc[2 * g.nbc + 1] * g.invN) : c.eq_val;
        c.eqvar = eq;
        c.deq = fabs(eq - eqp);
        c.eq_val = eq;
        c.eq_it = c.it;
        if (fabs(c.deq) < c.tol_eq) c.done = 1;
        else if (c.it > c.cap) c.done = 2;
        c.need_cur = 0;
        c.need_prev = 0;
        publish(c, hs, s);
    }
}

// --------------------------------------------------------------- utility
template <typename T, int C>
__global__ void k_fill_load(Geo g, Ptr<T> p, int buf)
{
    const long long n = g.N * C;
    for (int s = 0; s < g.nsolve; ++s) {
        T* U = u_buf(p, buf, s);
        const Ctl& c = p.ctl[s];
        for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
            U[i] = T(c.E[i % C]);
    }
}

// FP32 -> FP64 state transfer at the precision switch: the FP64 iterate
// `it` <- the FP32 iterate `it` (solves that are done are skipped)
template <int C>
__global__ void k_promote(Geo g, Ptr<float> p32, Ptr<double> p64, const Ctl* ctl)
{
    const long long n = g.N * C;
    for (int s = 0; s < g.nsolve; ++s) {
        if (ctl[s].done) continue;
        const int it = ctl[s].it;
        const float* src = u_buf(p32, it, s);
        double* dst = u_buf(p64, it, s);
        for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
            dst[i] = (double)src[i];
    }
}

// means of u and of the dual field v = M(x) u at the final iterate; output
// per solve [2*C] partial sums per block
template <typename T, typename PH>
__global__ void __launch_bounds__(256) k_means(Geo g, Ptr<T> p, double* out, int nblk)
{
    __shared__ double red[256 / 64];
    constexpr int C = PH::C;
    const int s = blockIdx.y;
    const Ctl& ctl = p.ctl[s];
    const bool corr = sizeof(T) == 8 && ctl.corr;
    const T* U = u_buf(p, corr ? ctl.anc_it : ctl.it, s);
    const float* E = corr ? e_buf(p, ctl.it, s) : nullptr;
    const int rv = p.rve_of[s];
    const uint8_t* ph = p.ph + (long long)rv * p.sPh;
    const T* coef = p.coef + (long long)rv * p.sCoef;
    double su[C], sv[C];
#pragma unroll
    for (int c = 0; c < C; ++c) { su[c] = 0; sv[c] = 0; }
    for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < g.N; v += (long long)gridDim.x * blockDim.x) {
        T u[C], o[C];
#pragma unroll
        for (int c = 0; c < C; ++c) u[c] = U[v * C + c];
        if (E) {
#pragma unroll
            for (int c = 0; c < C; ++c) u[c] += (T)E[v * C + c];
        }
        PH::dual(coef + (int)ph[v] * NCOEF, u, o);
#pragma unroll
        for (int c = 0; c < C; ++c) { su[c] += (double)u[c]; sv[c] += (double)o[c]; }
    }
    for (int c = 0; c < C; ++c) {
        double a = block_sum(su[c], red);
        if (threadIdx.x == 0) out[((long long)s * 2 * C + c) * nblk + blockIdx.x] = a;
        double bsum = block_sum(sv[c], red);
        if (threadIdx.x == 0) out[((long long)s * 2 * C + C + c) * nblk + blockIdx.x] = bsum;
    }
}

// final fields in the reference order: eps/sigma (or gradient/flux) FP64 AoS
template <typename T, typename PH>
__global__ void k_fields(Geo g, Ptr<T> p, int s, double* uo, double* vo)
{
    constexpr int C = PH::C;
    const Ctl& ctl = p.ctl[s];
    const bool corr = sizeof(T) == 8 && ctl.corr;
    const T* U = u_buf(p, corr ? ctl.anc_it : ctl.it, s);
    const float* E = corr ? e_buf(p, ctl.it, s) : nullptr;
    const int rv = p.rve_of[s];
    const uint8_t* ph = p.ph + (long long)rv * p.sPh;
    const T* coef = p.coef + (long long)rv * p.sCoef;
    for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < g.N; v += (long long)gridDim.x * blockDim.x) {
        T u[C], o[C];
#pragma unroll
        for (int c = 0; c < C; ++c) u[c] = U[v * C + c];
        if (E) {
#pragma unroll
            for (int c = 0; c < C; ++c) u[c] += (T)E[v * C + c];
        }
        PH::dual(coef + (int)ph[v] * NCOEF, u, o);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            uo[v * C + c] = (double)u[c];
            vo[v * C + c] = (double)o[c];
        }
    }
}

} // namespace m3d
