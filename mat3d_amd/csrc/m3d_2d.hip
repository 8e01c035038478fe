// m3d_2d.hip -- FFT_Analysis2D (src/2d/FFT_analysis2D.cpp) on the GPU, FP64:
// the basic scheme on complex 2D fields [E11, E22, E12] (tensor shear) with
// a fixed 25 iterations per runAnalysis.
//
// Per iteration (two launches):
//   row : one x row in LDS: backward FFT along y (p4), eps = t / xy of the
//         previous iteration (FFTBCKWRD_epsilon :143-148); sigma = C(phase) eps
//         (multipCx, :96-106); tau = sigma - C0 eps (:240); forward FFT along y
//         of the three interleaved components (p3).  The first row pass reads
//         eps, the last one ends after eps; sigma is stored by the last
//         iteration only (nothing else reads it)
//   x   : forward FFT along x, then t = -G(xi) t with the reference's
//         6-entry Green operator per frequency (setGF :53-93, recomputed
//         here; x > (Nx-1)/2 maps to -(Ny - x) as in the reference), DC =
//         E xy (multiplyGF :114-141), then the backward FFT along x
// convergenceCheck (:150-187) only prints, and its sum reads past the two-entry
// frequency vector; its iteration counter is kept, its transform is not.
// The x pass is that of m3d_fast.hpp on a three-component view: x lines are
// rows Ny*3 values apart with the y index in the role of the contiguous kz tile.
// The 75 iterations of a homogenization are a chain of dependent launches, bound
// by their latency up to 512^2: with four launches per iteration (62 us) and the
// means taken on the host from 75 MB of copied fields a 512^2 homogenization
// took 11.7 ms, with two launches and row sums taken on the device 2.7 ms.
#include "m3d_engine.hpp"

#include <cstring>
#include <string>
#include <vector>

namespace m3d {
namespace p2 {

struct Comp3 {
    static constexpr int C = 3;
    // the x pass with the Green step on the view of an Nx x Ny grid as
    // g.Nx x 1 x g.Nzh (kx: x frequency, kz: y frequency); prm = {la0, mu0},
    // ctl.E = the load as (re, im) pairs
    template <typename T>
    static __device__ void green(const Geo& g, const Ctl& ctl, const T* prm, int kx, int, int kz, cx<T>* v);
};

// threads of the row pass and of the x pass (128, 192 and 512 within 3-10%)
constexpr int NTR = 256, NTX = 256;

struct Mat {
    double Cm[9], Ci[9], C0[9];
    double la0, mu0;
};

// FIRST: eps is read (no backward transform), LAST: ends after storing eps.
// psum: the row's sums of the real parts, [6][Nx] (eps by the LAST pass, sigma
// by the pass that stores it)
template <int L, bool FIRST, bool LAST>
__global__ void __launch_bounds__(NTR) k_row(const uint8_t* ph, Mat m, cx<double>* eps, cx<double>* sig, cx<double>* t,
                                             const cx<double>* twg, double xy, int store_sig, double* psum)
{
    __shared__ __align__(16) cx<double> sl[3 * L];
    __shared__ cx<double> tw[L];
    __shared__ double red[NTR / 64];
    const int x = blockIdx.x, nx = gridDim.x;
    const long long row = (long long)x * L;
    const cx<double>* src = (FIRST ? eps : t) + 3 * row;
    constexpr int PER = (3 * L + NTR - 1) / NTR;
    {
        fast::vd2 r[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if ((3 * L) % NTR == 0 || (int)threadIdx.x + i * NTR < 3 * L)
                r[i] = *reinterpret_cast<const fast::vd2*>(src + threadIdx.x + i * NTR);
        for (int i = threadIdx.x; i < L; i += NTR) tw[i] = twg[i];
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if ((3 * L) % NTR == 0 || (int)threadIdx.x + i * NTR < 3 * L)
                *reinterpret_cast<fast::vd2*>(sl + threadIdx.x + i * NTR) = r[i];
    }
    __syncthreads();
    if constexpr (!FIRST) fast::fft<double, L, 3, NTR, 1, 1>(sl, tw);
    double se[3] = {0, 0, 0}, ss[3] = {0, 0, 0};
    for (int y = threadIdx.x; y < L; y += NTR) {
#pragma clang fp contract(off)
        cx<double> e[3];
        for (int c = 0; c < 3; ++c) {
            e[c] = sl[3 * y + c];
            if (!FIRST) e[c] = cx<double>{e[c].re / xy, e[c].im / xy};
        }
        if constexpr (LAST) {
            for (int c = 0; c < 3; ++c) {
                eps[3 * (row + y) + c] = e[c];
                se[c] += e[c].re;
            }
            continue;
        }
        const double* C = ph[row + y] ? m.Cm : m.Ci;
        for (int r = 0; r < 3; ++r) {
            const cx<double> sg{(C[3 * r] * e[0].re + C[3 * r + 1] * e[1].re) + C[3 * r + 2] * e[2].re,
                                (C[3 * r] * e[0].im + C[3 * r + 1] * e[1].im) + C[3 * r + 2] * e[2].im};
            const cx<double> c0{(m.C0[3 * r] * e[0].re + m.C0[3 * r + 1] * e[1].re) + m.C0[3 * r + 2] * e[2].re,
                                (m.C0[3 * r] * e[0].im + m.C0[3 * r + 1] * e[1].im) + m.C0[3 * r + 2] * e[2].im};
            if (store_sig) {
                sig[3 * (row + y) + r] = sg;
                ss[r] += sg.re;
            }
            sl[3 * y + r] = cx<double>{sg.re - c0.re, sg.im - c0.im};
        }
    }
    if (LAST || store_sig) {
        for (int c = 0; c < 3; ++c) {
            const double v = block_sum(LAST ? se[c] : ss[c], red);
            if (threadIdx.x == 0) psum[(long long)(LAST ? c : 3 + c) * nx + x] = v;
        }
    }
    if constexpr (LAST) return;
    __syncthreads();
    fast::fft<double, L, 3, NTR, -1, 1>(sl, tw);
    cx<double>* dst = t + 3 * row;
#pragma unroll
    for (int i = 0; i < PER; ++i)
        if ((3 * L) % NTR == 0 || (int)threadIdx.x + i * NTR < 3 * L) dst[threadIdx.x + i * NTR] = sl[threadIdx.x + i * NTR];
}

// setLoad: eps = E at every point
__global__ void k_fill_eps(cx<double>* eps, cx<double> e0, cx<double> e1, cx<double> e2, long long xy)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < xy; i += (long long)gridDim.x * blockDim.x) {
        eps[3 * i] = e0;
        eps[3 * i + 1] = e1;
        eps[3 * i + 2] = e2;
    }
}

__device__ __forceinline__ double dl(int i, int j) { return i == j ? 1.0 : 0.0; }

// the Green step at frequency (x, y) of the Nx x Ny grid on its three values
// v (multiplyGF, :114-141): DC = E xy, else v = -G(xi) v with the shear
// weighted twice; E as (re, im) pairs
__device__ __forceinline__ void green2d(int x, int y, int Nx, int Ny, double la0, double mu0, const double* E,
                                        cx<double>* v)
{
#pragma clang fp contract(off)
    if (x == 0 && y == 0) {
        const double n = (double)((long long)Nx * Ny);
        for (int c = 0; c < 3; ++c) v[c] = cx<double>{E[2 * c] * n, E[2 * c + 1] * n};
        return;
    }
    const double d1 = 1 / (4 * mu0);
    const double d2 = (la0 + mu0) / (mu0 * (la0 + 2 * mu0));
    const int q[6][4] = {{0, 0, 0, 0}, {0, 0, 1, 1}, {0, 0, 0, 1}, {1, 1, 1, 1}, {1, 1, 0, 1}, {0, 1, 0, 1}};
    const int w[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
    const int x1 = (x <= (Nx - 1) / 2) ? x : -(Ny - x);
    const int y1 = (y <= (Ny - 1) / 2) ? y : -(Ny - y);
    const double zet[2] = {x1 * 1.0, y1 * 1.0};
    const double n2 = zet[0] * zet[0] + zet[1] * zet[1];
    double G[6];
    for (int r = 0; r < 6; ++r) {
        const int a = q[r][0], b = q[r][1], k = q[r][2], h = q[r][3];
        G[r] = (d1 / n2) * (((dl(k, a) * zet[h] * zet[b] + dl(h, a) * zet[k] * zet[b]) + dl(k, b) * zet[h] * zet[a]) +
                            dl(h, b) * zet[k] * zet[a]) -
               (d2 * zet[a] * zet[b] * zet[k] * zet[h]) / (n2 * n2);
    }
    const cx<double> a0 = v[0], a1 = v[1], a2 = v[2];
    for (int j = 0; j < 3; ++j) {
        const double re = -((G[w[j][0]] * a0.re + G[w[j][1]] * a1.re) + G[w[j][2]] * a2.re * 2);
        const double im = -((G[w[j][0]] * a0.im + G[w[j][1]] * a1.im) + G[w[j][2]] * a2.im * 2);
        v[j] = cx<double>{re, im};
    }
}

template <typename T>
__device__ void Comp3::green(const Geo& g, const Ctl& ctl, const T* prm, int kx, int, int kz, cx<T>* v)
{
    green2d(kx, kz, g.Nx, g.Nzh, prm[0], prm[1], ctl.E, v);
}

static_assert(fast::has_green_hook<Comp3>::value, "the 2D Green step must replace the 3D one in the x pass");

inline bool fast_len(int L)
{
    return L == 32 || L == 48 || L == 64 || L == 96 || L == 128 || L == 192 || L == 256 || L == 512;
}

struct Solver {
    int Nx, Ny;
    long long xy;
    hipStream_t st = nullptr;
    cx<double>*eps = nullptr, *sig = nullptr, *t = nullptr;
    uint8_t* ph = nullptr;
    Ctl* ctl = nullptr; // never done: gates nothing in the passes; E holds the load
    cx<double>*twx = nullptr, *twy = nullptr;
    double* dprm = nullptr; // {la0, mu0} for the Green step
    int* drve = nullptr;    // {0}: the one solve's parameter row
    double* psum = nullptr; // [6][Nx] row sums of the real parts of eps and sigma
    Geo gx1{};
    Mat m{};
    cx<double> E[3] = {{0, 0}, {0, 0}, {0, 0}};
    bool have_mat = false;
    int itNo = 0;

    template <typename P>
    void alloc(P** p, size_t bytes)
    {
        hipError_t e = hipMalloc((void**)p, bytes);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            *p = nullptr;
            throw ArgError{M3D_ERR_OOM, "device allocation of " + std::to_string(bytes) + " bytes failed"};
        }
    }

    Solver(int nx, int ny) : Nx(nx), Ny(ny)
    {
        xy = (long long)nx * ny;
        if (!fast_len(nx) || !fast_len(ny))
            throw ArgError{M3D_ERR_UNSUPPORTED, "FFT_Analysis2D: Nx and Ny must be 32, 48, 64, 96, 128, 192, 256 or 512"};
        HCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
        alloc(&eps, sizeof(cx<double>) * 3 * xy);
        alloc(&sig, sizeof(cx<double>) * 3 * xy);
        alloc(&t, sizeof(cx<double>) * 3 * xy);
        alloc(&ph, (size_t)xy);
        alloc(&ctl, sizeof(Ctl));
        alloc(&dprm, sizeof(double) * 2);
        alloc(&drve, sizeof(int));
        alloc(&psum, sizeof(double) * 6 * nx);
        HCHK(hipMemset(drve, 0, sizeof(int)));
        HCHK(hipMemset(eps, 0, sizeof(cx<double>) * 3 * xy));
        HCHK(hipMemset(sig, 0, sizeof(cx<double>) * 3 * xy));
        HCHK(hipMemset(ctl, 0, sizeof(Ctl)));
        auto tx = twiddles<double>(nx), ty = twiddles<double>(ny);
        alloc(&twx, sizeof(cx<double>) * nx);
        alloc(&twy, sizeof(cx<double>) * ny);
        HCHK(hipMemcpy(twx, tx.data(), sizeof(cx<double>) * nx, hipMemcpyHostToDevice));
        HCHK(hipMemcpy(twy, ty.data(), sizeof(cx<double>) * ny, hipMemcpyHostToDevice));
        // x lines with the Green step: the grid as nx x 1 x ny, rows x at
        // stride ny*3, the y points in the role of the kz tile
        std::memset(&gx1, 0, sizeof gx1);
        gx1.Nx = nx; gx1.Ny = 1; gx1.Nz = 1; gx1.Nzh = ny; gx1.C = 3; gx1.nsolve = 1;
        gx1.sy = (long long)ny * 3; gx1.sxa = (long long)ny * 3; gx1.sxb = 0; gx1.lxb = 0; gx1.xbm = 0;
    }

    ~Solver()
    {
        if (st) (void)hipStreamSynchronize(st);
        for (void* p : {(void*)eps, (void*)sig, (void*)t, (void*)ph, (void*)ctl, (void*)dprm, (void*)drve, (void*)psum,
                        (void*)twx, (void*)twy})
            if (p) (void)hipFree(p);
        if (st) (void)hipStreamDestroy(st);
    }

    template <int L, bool FIRST, bool LAST>
    bool row_at(int store_sig)
    {
        if (Ny != L) return false;
        hipLaunchKernelGGL((k_row<L, FIRST, LAST>), dim3(Nx), dim3(NTR), 0, st, ph, m, eps, sig, t, twy, (double)xy, store_sig,
                           psum);
        return true;
    }
    template <bool FIRST, bool LAST>
    void row(int store_sig)
    {
        if (!(row_at<512, FIRST, LAST>(store_sig) || row_at<256, FIRST, LAST>(store_sig) ||
              row_at<192, FIRST, LAST>(store_sig) || row_at<128, FIRST, LAST>(store_sig) ||
              row_at<96, FIRST, LAST>(store_sig) || row_at<64, FIRST, LAST>(store_sig) ||
              row_at<48, FIRST, LAST>(store_sig) || row_at<32, FIRST, LAST>(store_sig)))
            throw ArgError{M3D_ERR_UNSUPPORTED, "FFT_Analysis2D: no y kernel"};
    }
    // x lines: forward FFT, the Green step (Comp3::green), inverse FFT in one
    // pass over each tile
    template <int L>
    bool xg_at()
    {
        if (gx1.Nx != L) return false;
        // one y point per tile: as many workgroups as rows (tiles of the 3D
        // width left 16 workgroups for a 128^2 plate)
        constexpr int TK = 1;
        const int nkt = (gx1.Nzh + TK - 1) / TK;
        const size_t sm = ((size_t)L * TK * 3 + L) * sizeof(cx<double>);
        if (sm > 65536) throw ArgError{M3D_ERR_UNSUPPORTED, "FFT_Analysis2D: x tile too large"};
        Ptr<double> p;
        std::memset(&p, 0, sizeof p);
        p.S = t;
        p.K = t;
        p.twx = twx;
        p.ctl = ctl;
        p.rve_of = drve;
        hipLaunchKernelGGL((fast::kxy<double, Comp3, 1, -1, BUF_MAIN, L, TK, NTX>), dim3(nkt), dim3(NTX), sm, st, gx1, p,
                           (const double*)dprm);
        return true;
    }
    void xgreen()
    {
        if (!(xg_at<512>() || xg_at<256>() || xg_at<192>() || xg_at<128>() || xg_at<96>() || xg_at<64>() ||
              xg_at<48>() || xg_at<32>()))
            throw ArgError{M3D_ERR_UNSUPPORTED, "FFT_Analysis2D: no x kernel"};
    }

    // material(properties, RVE1), :189-221
    void material(const double* q, const double* rve)
    {
        const double Em = q[0], vm = q[1], Ei = q[2], vi = q[3];
        const double mum = Em / (1 + vm) / 2, lam = vm * Em / (1 + vm) / (1 - 2 * vm);
        const double mui = Ei / (1 + vi) / 2, lai = vi * Ei / (1 + vi) / (1 - 2 * vi);
        const double cm[9] = {lam + 2 * mum, lam, 0, lam, lam + 2 * mum, 0, 0, 0, 2 * mum};
        const double ci[9] = {lai + 2 * mui, lai, 0, lai, lai + 2 * mui, 0, 0, 0, 2 * mui};
        const double alf = 1;
        for (int k = 0; k < 9; ++k) {
            m.Cm[k] = cm[k];
            m.Ci[k] = ci[k];
            m.C0[k] = alf * (cm[k] + ci[k]) / 2.;
        }
        m.la0 = alf * (lai + lam) / 2.;
        m.mu0 = alf * (mui + mum) / 2.;
        const double lm[2] = {m.la0, m.mu0};
        HCHK(hipMemcpy(dprm, lm, sizeof lm, hipMemcpyHostToDevice));
        std::vector<uint8_t> p((size_t)xy);
        for (long long i = 0; i < xy; ++i) p[(size_t)i] = rve[i] == 1 ? 1 : 0; // RVE(i)==1: matrix (:99-103)
        HCHK(hipMemcpy(ph, p.data(), (size_t)xy, hipMemcpyHostToDevice));
        have_mat = true;
    }

    // runAnalysis, :232-246, without waiting for it; e_ri: the load, alive
    // until the stream is synchronised
    void run_async(const double* e_ri)
    {
        if (!have_mat) throw ArgError{M3D_ERR_STATE, "runAnalysis: material() first"};
        HCHK(hipMemcpyAsync(reinterpret_cast<char*>(ctl) + offsetof(Ctl, E), e_ri, 6 * sizeof(double), hipMemcpyHostToDevice, st));
        for (int it = 0; it < 25; ++it) {
            if (it == 0) row<true, false>(0);
            else row<false, false>(it == 24);
            xgreen();
            itNo += 1;
        }
        row<false, true>(0);
        HCHK(hipGetLastError());
    }
    void run()
    {
        double e_ri[6];
        for (int c = 0; c < 3; ++c) {
            e_ri[2 * c] = E[c].re;
            e_ri[2 * c + 1] = E[c].im;
        }
        run_async(e_ri);
        HCHK(hipStreamSynchronize(st));
    }
};

} // namespace p2
} // namespace m3d

using namespace m3d;

struct m3d_2d {
    p2::Solver* s = nullptr;
    std::string err;
};

namespace {

template <typename F>
int guarded(m3d_2d* h, F&& f)
{
    if (!h) return M3D_ERR_ARG;
    try {
        return f();
    } catch (const HipError& e) {
        h->err = std::string("HIP error in ") + e.what + ": " + hipGetErrorString(e.e);
        (void)hipGetLastError();
        return M3D_ERR_HIP;
    } catch (const ArgError& e) {
        h->err = e.msg;
        return e.code;
    } catch (const std::bad_alloc&) {
        h->err = "host allocation failed";
        return M3D_ERR_OOM;
    } catch (const std::exception& e) {
        h->err = e.what();
        return M3D_ERR_UNSUPPORTED;
    }
}

// 3x3 column-major inverse by Gauss-Jordan with partial pivoting (Eigen's inverse())
bool inv3(const double* A, double* X)
{
    double M[9];
    std::memcpy(M, A, sizeof M);
    for (int k = 0; k < 9; ++k) X[k] = (k % 4 == 0) ? 1.0 : 0.0;
    for (int c = 0; c < 3; ++c) {
        int piv = c;
        for (int r = c + 1; r < 3; ++r)
            if (std::fabs(M[r + 3 * c]) > std::fabs(M[piv + 3 * c])) piv = r;
        if (M[piv + 3 * c] == 0) return false;
        if (piv != c)
            for (int k = 0; k < 3; ++k) {
                std::swap(M[c + 3 * k], M[piv + 3 * k]);
                std::swap(X[c + 3 * k], X[piv + 3 * k]);
            }
        const double d = M[c + 3 * c];
        for (int k = 0; k < 3; ++k) {
            M[c + 3 * k] /= d;
            X[c + 3 * k] /= d;
        }
        for (int r = 0; r < 3; ++r) {
            if (r == c) continue;
            const double f = M[r + 3 * c];
            for (int k = 0; k < 3; ++k) {
                M[r + 3 * k] -= f * M[c + 3 * k];
                X[r + 3 * k] -= f * X[c + 3 * k];
            }
        }
    }
    return true;
}

} // namespace

int m3d_2d_create(int nx, int ny, m3d_2d** out)
{
    if (!out || nx < 1 || ny < 1) return M3D_ERR_ARG;
    *out = nullptr;
    m3d_2d* h = new (std::nothrow) m3d_2d;
    if (!h) return M3D_ERR_OOM;
    const int rc = guarded(h, [&]() {
        h->s = new p2::Solver(nx, ny);
        return M3D_OK;
    });
    if (rc != M3D_OK) {
        delete h->s;
        delete h;
        return rc;
    }
    *out = h;
    return M3D_OK;
}

int m3d_2d_destroy(m3d_2d* h)
{
    if (!h) return M3D_ERR_ARG;
    delete h->s;
    delete h;
    return M3D_OK;
}

const char* m3d_2d_last_error(m3d_2d* h) { return h ? h->err.c_str() : "null handle"; }

int m3d_2d_material(m3d_2d* h, const double* properties, const double* rve)
{
    return guarded(h, [&]() {
        if (!properties || !rve) throw ArgError{M3D_ERR_ARG, "material: null argument"};
        h->s->material(properties, rve);
        return M3D_OK;
    });
}

int m3d_2d_set_load(m3d_2d* h, const double* E_ri)
{
    return guarded(h, [&]() {
        if (!E_ri) throw ArgError{M3D_ERR_ARG, "setLoad: null argument"};
        p2::Solver& s = *h->s;
        for (int c = 0; c < 3; ++c) s.E[c] = cx<double>{E_ri[2 * c], E_ri[2 * c + 1]};
        hipLaunchKernelGGL(p2::k_fill_eps, dim3(256), dim3(256), 0, s.st, s.eps, s.E[0], s.E[1], s.E[2], s.xy);
        HCHK(hipGetLastError());
        // the fields' copies do not follow this stream, and a failed fill is this call's error
        HCHK(hipStreamSynchronize(s.st));
        return M3D_OK;
    });
}

int m3d_2d_run(m3d_2d* h, int* itNo)
{
    return guarded(h, [&]() {
        h->s->run();
        if (itNo) *itNo = h->s->itNo;
        return M3D_OK;
    });
}

int m3d_2d_homogenization(m3d_2d* h, double* CHomo, double* epHomo, double* sigHomo)
{
    return guarded(h, [&]() {
        p2::Solver& s = *h->s;
        double ep[9], sg[9], loads[3][6];
        std::vector<double> sums((size_t)3 * 6 * s.Nx);
        // the three load cases follow each other on the device; their row sums
        // come back together
        for (int w = 0; w < 3; ++w) {
            for (int c = 0; c < 3; ++c) {
                s.E[c] = cx<double>{c == w ? 0.005 : 0.0, 0.0};
                loads[w][2 * c] = s.E[c].re;
                loads[w][2 * c + 1] = 0.0;
            }
            s.run_async(loads[w]);
            HCHK(hipMemcpyAsync(sums.data() + (size_t)w * 6 * s.Nx, s.psum, sizeof(double) * 6 * s.Nx, hipMemcpyDeviceToHost,
                                s.st));
        }
        HCHK(hipStreamSynchronize(s.st));
        for (int w = 0; w < 3; ++w)
            for (int c = 0; c < 3; ++c) {
                double se = 0, ss = 0;
                for (int x = 0; x < s.Nx; ++x) {
                    se += sums[((size_t)w * 6 + c) * s.Nx + x];
                    ss += sums[((size_t)w * 6 + 3 + c) * s.Nx + x];
                }
                ep[w + 3 * c] = se / (double)s.xy;
                sg[c + 3 * w] = ss / (double)s.xy;
            }
        double inv[9];
        if (!inv3(ep, inv)) throw ArgError{M3D_ERR_NUMERIC, "homogenization: singular epHomo"};
        double C[9];
        for (int c = 0; c < 3; ++c)
            for (int r = 0; r < 3; ++r) {
                double a = 0;
                for (int k = 0; k < 3; ++k) a += inv[r + 3 * k] * sg[k + 3 * c];
                C[r + 3 * c] = a;
            }
        if (CHomo) std::memcpy(CHomo, C, sizeof C);
        if (epHomo) std::memcpy(epHomo, ep, sizeof ep);
        if (sigHomo) std::memcpy(sigHomo, sg, sizeof sg);
        return M3D_OK;
    });
}

int m3d_2d_get_fields(m3d_2d* h, double* eps_ri, double* sig_ri)
{
    return guarded(h, [&]() {
        p2::Solver& s = *h->s;
        if (eps_ri) HCHK(hipMemcpy(eps_ri, s.eps, sizeof(cx<double>) * 3 * s.xy, hipMemcpyDeviceToHost));
        if (sig_ri) HCHK(hipMemcpy(sig_ri, s.sig, sizeof(cx<double>) * 3 * s.xy, hipMemcpyDeviceToHost));
        return M3D_OK;
    });
}
