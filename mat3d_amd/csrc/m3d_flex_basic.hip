// m3d_flex_basic.hip -- the basic scheme ("ep" / "ed", FFT_analysis3D.cpp:796-853)
// in FP64 on grids without the compile-time kernels of m3d_basic.hip: the same
// passes (sigma-only transforms in the iterations, eps^ kept by the x pass,
// FINAL recomputation of an increment's last iterate) on the run-time-length
// transforms of m3d_flex.hpp.
//
// One solve of a small grid is bound by latency: at 50^3 (250 to 450
// workgroups) z 69 -> 17, x 63 -> 17, y 38 + 29 -> 9 + 10 us per iteration
// against passes that transformed [sigma | eps] (12 components) in every
// iteration; a 50^3 damage path of 2076 iterations 463 -> 112 ms (with the
// finalisers inside the y passes and the tiles of kz_most).
#include "m3d_basic_fast.hpp"
#include "m3d_flex.hpp"

#include <algorithm>
#include <stdexcept>
#include <string>

namespace m3d {
namespace bflex {

using flex::NT0;
using flex::NT1;
using flex::fdiv;
using flex::mul24;
using T = double;
constexpr int VPT = 2; // voxels per thread of the z pass at most

// ------------------------------------------------------------------ z pass
// Modes, buffers and results as bfast::kzb (m3d_basic.hip); one voxel at a
// time, its two transform columns being pairs of components.
//   START: [sigma | eps] of a row in 6 columns; ITER, FINAL: sigma in 3.
template <int BEH, int MODE, bool LIN, int NT>
__global__ void __launch_bounds__(NT) k_zb(Geo g, BPtr<T> p)
{
    constexpr bool FIN = MODE == BMODE_FINAL;
    constexpr bool START = MODE == BMODE_START;
    constexpr bool STAR = BEH == BEH_EP; // sigma_star = sigma_old - C eps_old in place of both
    constexpr bool FUSE = FIN && STAR;   // FINAL of "ep" also ends the increment
    constexpr int C = START ? 12 : 6, HC = C / 2;
    constexpr int NW = NT / 64;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double red[NBSUM + 2][NW];
    cx<T>* sl = reinterpret_cast<cx<T>*>(smem_raw);
    Ctl& ctl = p.ctl[0];
    if (bz_skip(ctl, blockIdx.x == 0 && threadIdx.x == 0)) return;
    const int t = fast::xcd_remap(blockIdx.x, gridDim.x);
    const int x = t / g.nty, y0 = (t - x * g.nty) * g.TY;
    const int ny = min(g.TY, g.Ny - y0), Nz = g.Nz;
    const int W = ny * HC, ws = W | 1;
    const int tid = threadIdx.x;
    const long long vox0 = ((long long)x * g.Ny + y0) * Nz;
    const long long row0 = ((long long)x * g.Ny + y0) * g.Nzh;
    const cx<T>* tw = flex::stage_twiddles<T, NT>(sl + (size_t)Nz * ((g.TY * HC) | 1), p.twz, Nz);
    const int nv = ny * Nz;
    const float inv_nz = 1.0f / (float)Nz;

    using V6 = flex::Vox<T, 6>;
    // the iterations' voxel data (history and phases; START: eps) before the
    // transform, so that it arrives during it
    V6 hs[VPT];
    T hep[VPT];
    int hph[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int v = tid + i * NT;
        if (v < nv) {
            if constexpr (STAR) hs[i] = *reinterpret_cast<const V6*>(p.sig_star + (vox0 + v) * 6);
            hep[i] = p.ep[vox0 + v];
            hph[i] = p.ph[vox0 + v];
        }
    }
    if constexpr (!START) {
        constexpr int PER = flex::ept<T, NT>() / 2 + 1;
        cx<T> ca[PER], cb[PER];
        const flex::ZPairs<6> zp(Nz, g.Nzh, ny);
        zp.template issue<T, NT, PER>(p.S6 + row0 * 6, (long long)g.Nzh * 6, ca, cb);
        zp.template commit<T, NT, PER>(sl, ws, ca, cb);
        __syncthreads();
        flex::fft<T, 1, NT>(sl, tw, g.az, W, ws, 1.0f / (float)W);
    } else {
        __syncthreads();
    }

    T* sr = reinterpret_cast<T*>(sl);
    double acc[NBSUM + 2]; // sigma, eps; FUSE: sigma_eff, eps_p
#pragma unroll
    for (int q = 0; q < NBSUM + 2; ++q) acc[q] = 0.0;
    bool bad = false;
    const int vt = fast::lane_tid();
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int v = vt + i * NT;
        if (v < nv) {
            const int yl = fdiv(v, inv_nz), m = v - mul24(yl, Nz);
            T* rp = sr + 2 * (mul24(m, ws) + yl * HC);
            const long long vg = vox0 + v;
            const double* mt = p.mat + hph[i] * 8;
            T e[6], sg[6];
            if constexpr (!START) {
#pragma unroll
                for (int c = 0; c < 6; ++c) e[c] = rp[c];
            } else {
                const V6 f = *reinterpret_cast<const V6*>(p.eps + vg * 6);
#pragma unroll
                for (int c = 0; c < 6; ++c) e[c] = f.v[c];
            }
            V6 out;
            if constexpr (BEH == BEH_EP) {
                T so[6], eo[6], phi, dep, seff;
#pragma unroll
                for (int c = 0; c < 6; ++c) so[c] = hs[i].v[c];
                if (!j2_update<T, LIN, true>(mt, e, eo, so, hep[i], sg, phi, dep, seff)) bad = true;
                if constexpr (FUSE) {
                    // export sums of this iterate, then update_old_Variable and the next sigma_star
                    acc[NBSUM] += seff;
                    acc[NBSUM + 1] += hep[i];
                    p.seff[vg] = seff;
                    p.ep[vg] = phi > T(0) ? hep[i] + dep : hep[i];
                    T ce[6];
                    iso_C(T(mt[0]), T(mt[1]), e, ce);
                    const V6 prev = *reinterpret_cast<const V6*>(p.eps_old + vg * 6);
                    V6 a, b;
#pragma unroll
                    for (int c = 0; c < 6; ++c) {
                        a.v[c] = e[c] + (e[c] - prev.v[c]);
                        b.v[c] = e[c];
                        out.v[c] = sg[c];
                    }
                    *reinterpret_cast<V6*>(p.eps + vg * 6) = a;
                    *reinterpret_cast<V6*>(p.eps_old + vg * 6) = b;
                    *reinterpret_cast<V6*>(p.sig_old + vg * 6) = out;
#pragma unroll
                    for (int c = 0; c < 6; ++c) a.v[c] = sg[c] - ce[c];
                    *reinterpret_cast<V6*>(p.sig_star + vg * 6) = a;
                } else if constexpr (START) {
                    p.phi[vg] = phi;
                    p.dep[vg] = dep;
                    p.seff[vg] = seff;
                }
            } else {
                T d = hep[i];
                damage_update<T>(mt, e, d, sg);
                p.ep[vg] = d;
                if constexpr (FIN) {
#pragma unroll
                    for (int c = 0; c < 6; ++c) out.v[c] = e[c];
                    *reinterpret_cast<V6*>(p.eps + vg * 6) = out;
                }
            }
            if constexpr (FIN || START) {
#pragma unroll
                for (int c = 0; c < 6; ++c) out.v[c] = sg[c];
                *reinterpret_cast<V6*>(p.sig + vg * 6) = out;
            }
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                acc[c] += sg[c];
                acc[6 + c] += e[c];
                if constexpr (!FIN) rp[c] = sg[c];
                if constexpr (START) rp[6 + c] = e[c];
            }
        }
    }
    if (bad) ctl.err = 1;
    if (FIN && !FUSE) return;
    // fixed-order block sums of the 12 means (FUSE: the 14 export sums, in the
    // order eps, sigma, sigma_eff, eps_p)
    {
        constexpr int NQ = FUSE ? NBSUM + 2 : NBSUM;
        const int lane = tid & 63, wid = tid >> 6;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const double v = wave_sum(acc[q]);
            if (lane == 0) red[q][wid] = v;
        }
        __syncthreads();
        if (tid < NQ) {
            double r = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) r += red[tid][w];
            if constexpr (FUSE) {
                const int o = tid < 6 ? tid + 6 : (tid < 12 ? tid - 6 : tid);
                p.pfin[(long long)o * g.nbz + t] = r;
            } else {
                p.psum[(long long)tid * g.nbz + t] = r;
            }
        }
    }
    if constexpr (FUSE) return;
    __syncthreads();
    flex::fft<T, -1, NT>(sl, tw, g.az, W, ws, 1.0f / (float)W);
    const flex::ZPairs<C> zp(Nz, g.Nzh, ny);
    zp.template store<T, NT>(sl, ws, p.S12 + row0 * C, (long long)g.Nzh * C);
}

// ------------------------------------------------------------------ x pass
// bfast::kxb with run-time lengths; one frequency per thread.  Eh holds eps^
// as [y][kx][kz][c], whatever the tiles of the start stage and of the
// iterations.
template <bool E6, int NT>
__global__ void __launch_bounds__(NT) k_xb(Geo g, BPtr<T> p)
{
    constexpr int C = E6 ? 6 : 12;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double red[NT / 64];
    cx<T>* sl = reinterpret_cast<cx<T>*>(smem_raw);
    const Ctl& ctl = p.ctl[0];
    if (ctl.done) return;
    const int t = fast::xcd_remap(blockIdx.x, gridDim.x);
    const int y = t / g.nkx, kz0 = (t - y * g.nkx) * g.TKx;
    const int nk = min(g.TKx, g.Nzh - kz0), w = nk * C;
    const int tid = threadIdx.x;
    const cx<T>* tw = flex::stage_twiddles<T, NT>(sl + (size_t)g.Nx * g.TKx * C, p.twx, g.Nx);
    flex::load_tile<T, NT>(sl, p.S12 + ((long long)y * g.Nzh + kz0) * C, (long long)g.Ny * g.Nzh * C, g.Nx, w);
    const int kx = fdiv(tid, 1.0f / (float)nk), kzl = tid - mul24(kx, nk), kz = kz0 + kzl;
    const bool on = tid < g.Nx * nk;
    cx<T>* eo = p.Eh + (((long long)y * g.Nx + kx) * g.Nzh + kz) * 6;
    cx<T> ev[6];
    if (E6 && on) {
#pragma unroll
        for (int c = 0; c < 6; ++c) ev[c] = eo[c];
    }
    __syncthreads();
    flex::fft<T, -1, NT>(sl, tw, g.ax, w, w, 1.0f / (float)w);

    double acc = 0.0;
    cx<T> v6[6];
    if (on) {
        const cx<T>* v = sl + (mul24(kx, w) + kzl * C);
        cx<T> sg[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) sg[c] = v[c];
        double a2[6];
        acc = eq_term<T, 6>(g, kx, y, kz, sg, a2);
        if (kx == 0 && y == 0 && kz == 0) {
            p.pchk[g.nbx] = eq_mean<6>(a2);
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                v6[c] = cx<T>{T(ctl.E[c]), T(0)};
                eo[c] = cx<T>{T(ctl.E[c] / g.invN), T(0)};
            }
        } else {
            if constexpr (!E6) {
#pragma unroll
                for (int c = 0; c < 6; ++c) ev[c] = v[6 + c];
            }
            const T la0 = T(ctl.la0), mu0 = T(ctl.mu0), sc = T(g.invN);
            const int fz = Elastic::fmap(kz, g.Nz), fy = Elastic::fmap(y, g.Ny), fx = Elastic::fmap(kx, g.Nx);
            const T xi[3] = {T(fz), T(fy), T(fx)};
            cx<T> o[6];
            green_elastic<T>(xi, sg, o, 1, la0, mu0);
            // kz = 0 and Nz/2 planes: Hermitian part of the Gamma0 term
            if (kz == 0 || (g.zeven && kz == g.Nz / 2)) {
                const int px = kx ? g.Nx - kx : 0, py = y ? g.Ny - y : 0;
                const int gy = Elastic::fmap(py, g.Ny), gx = Elastic::fmap(px, g.Nx);
                if (fz != -fz || gy != -fy || gx != -fx) {
                    const T xp[3] = {T(fz), T(gy), T(gx)};
                    cx<T> o2[6];
                    green_elastic<T>(xp, sg, o2, 1, la0, mu0);
#pragma unroll
                    for (int c = 0; c < 6; ++c) o[c] = cscale(o[c] + o2[c], T(0.5));
                }
            }
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                const cx<T> n = ev[c] - o[c];
                eo[c] = n;
                v6[c] = cscale(n, sc);
            }
        }
    }
    const double bs = block_sum(acc, red); // synchronises: every tile value has been read
    if (tid == 0) p.pchk[t] = bs;
    const int w6 = nk * 6;
    if (on) {
#pragma unroll
        for (int c = 0; c < 6; ++c) sl[mul24(kx, w6) + kzl * 6 + c] = v6[c];
    }
    __syncthreads();
    flex::fft<T, 1, NT>(sl, tw, g.ax, w6, w6, 1.0f / (float)w6);
    flex::store_tile<T, NT>(sl, p.S6w + ((long long)y * g.Nzh + kz0) * 6, (long long)g.Ny * g.Nzh * 6, g.Nx, w6);
}

// ------------------------------------------------------------------ y pass
// flex::k_y with the finaliser f as its first workgroup
template <int DIR, int NT>
__global__ void __launch_bounds__(NT) k_yb(Geo g, Ptr<T> p, int which, BFin f)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double red[NT / 64][NBSUM];
    if (blockIdx.x == 0) {
        bfin_block(p.ctl[0], f, red);
        return;
    }
    cx<T>* sl = reinterpret_cast<cx<T>*>(smem_raw);
    flex::y_tile<T, DIR, NT>(g, p, which, fast::xcd_remap(blockIdx.x - 1, gridDim.x - 1), sl, sl + (size_t)g.Ny * g.TKy * g.C);
}

// ---------------------------------------------------------------- planning
namespace {

// a z tile of 2 voxels per thread and an x tile of one frequency per thread,
// within the transform's values (and the z tile's loaded pairs) per thread
int z_rows(int Nz, int C, int nt)
{
    const int E = flex::ept<T, NT0>(), hc = C / 2;
    return std::min({E * nt / (Nz * hc), VPT * nt / Nz, (E / 2 + 1) * nt / ((Nz / 2 + 1) * hc)});
}
int x_cols(int Nx, int C, int nt) { return std::min(flex::ept<T, NT0>() * nt / (C * Nx), nt / Nx); }

int even(int n, int most)
{
    const int parts = (n + most - 1) / most;
    return (n + parts - 1) / parts;
}

// kz values of an x or y tile that leave 384 workgroups (3 for 2 CUs): one load
// case of a grid of up to ~60^3 makes fewer of full tiles, and the launch then
// waits for workgroups that run alone on their CU.  Per load path, full tiles
// against this bound: 20^3 damage 10.1 / 8.4 ms, 36^3 19.4 / 17.2, 50^3 117.9 /
// 112.3, J2 40^3 13.5 / 11.6, 70^3 28.6 / 28.3, 100^3 69.4 / 68.6.  Bounds of 512
// and 768 cut to single kz (96-byte rows) earlier: 40^3 13.2, 50^3 110.8 and 140.7.
int kz_most(const Geo& g, int planes) { return std::max(1, (int)((long long)planes * g.Nzh / 384)); }

template <typename K, typename... A>
void go(K* k, int blocks, int nt, size_t sm, hipStream_t st, const A&... args)
{
    if (sm > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
        if (e != hipSuccess) throw std::runtime_error(std::string("LDS size: ") + hipGetErrorString(e));
    }
    hipLaunchKernelGGL(k, dim3(blocks), dim3(nt), sm, st, args...);
}

template <int BEH, int MODE, bool LIN>
void z_at(const Geo& g, const BPtr<T>& p, hipStream_t st)
{
    constexpr int HC = MODE == BMODE_START ? 6 : 3;
    const size_t W = (size_t)(g.TY * HC) | 1;
    if (z_rows(g.Nz, 2 * HC, NT0) >= 1) go(&k_zb<BEH, MODE, LIN, NT0>, g.nbz, NT0, g.Nz * (W + 1) * sizeof(cx<T>), st, g, p);
    else go(&k_zb<BEH, MODE, LIN, NT1>, g.nbz, NT1, g.Nz * W * sizeof(cx<T>), st, g, p);
}

template <int BEH, bool LIN>
void z_beh(int mode, const Geo& g, const BPtr<T>& p, hipStream_t st)
{
    if (mode == BMODE_START) z_at<BEH, BMODE_START, LIN>(g, p, st);
    else if (mode == BMODE_FINAL) z_at<BEH, BMODE_FINAL, LIN>(g, p, st);
    else z_at<BEH, BMODE_ITER, LIN>(g, p, st);
}

} // namespace

void plan(Geo& g)
{
    const int znt = z_rows(g.Nz, g.C, NT0) >= 1 ? NT0 : NT1, xnt = x_cols(g.Nx, g.C, NT0) >= 1 ? NT0 : NT1;
    const int ty = z_rows(g.Nz, g.C, znt), tk = x_cols(g.Nx, g.C, xnt);
    if (ty < 1 || tk < 1) throw std::length_error("line too long for one workgroup");
    g.TY = even(g.Ny, ty);
    g.nty = (g.Ny + g.TY - 1) / g.TY;
    g.nbz = g.Nx * g.nty;
    g.TKx = even(g.Nzh, std::min(tk, kz_most(g, g.Ny)));
    g.nkx = (g.Nzh + g.TKx - 1) / g.TKx;
    g.nbx = g.Ny * g.nkx;
    g.TKy = even(g.Nzh, std::min(g.TKy, kz_most(g, g.Nx)));
    g.nky = (g.Nzh + g.TKy - 1) / g.TKy;
}

void launch_z(int beh, int mode, const Geo& g, const BPtr<T>& p, hipStream_t st, bool lin)
{
    if (beh == BEH_EP && lin) z_beh<BEH_EP, true>(mode, g, p, st);
    else if (beh == BEH_EP) z_beh<BEH_EP, false>(mode, g, p, st);
    else z_beh<BEH_ED, false>(mode, g, p, st);
}

void launch_y(int dir, int which, const Geo& g, const Ptr<T>& p, const BFin& f, hipStream_t st)
{
    const long tile = (long)g.Ny * g.TKy * g.C;
    const bool lg = tile > (long)flex::ept<T, NT0>() * NT0;
    const size_t sm = (size_t)(tile + (lg ? 0 : g.Ny)) * sizeof(cx<T>);
    const int blocks = g.Nx * g.nky + 1;
    if (dir < 0) {
        if (lg) go(&k_yb<-1, NT1>, blocks, NT1, sm, st, g, p, which, f);
        else go(&k_yb<-1, NT0>, blocks, NT0, sm, st, g, p, which, f);
    } else {
        if (lg) go(&k_yb<1, NT1>, blocks, NT1, sm, st, g, p, which, f);
        else go(&k_yb<1, NT0>, blocks, NT0, sm, st, g, p, which, f);
    }
}

void launch_x(const Geo& g, const BPtr<T>& p, hipStream_t st, bool e6)
{
    const size_t tile = (size_t)g.Nx * g.TKx * g.C;
    const bool lg = x_cols(g.Nx, g.C, NT0) < 1;
    const size_t sm = (tile + (lg ? 0 : g.Nx)) * sizeof(cx<T>);
    if (e6) {
        if (lg) go(&k_xb<true, NT1>, g.nbx, NT1, sm, st, g, p);
        else go(&k_xb<true, NT0>, g.nbx, NT0, sm, st, g, p);
    } else {
        if (lg) go(&k_xb<false, NT1>, g.nbx, NT1, sm, st, g, p);
        else go(&k_xb<false, NT0>, g.nbx, NT0, sm, st, g, p);
    }
}

} // namespace bflex
} // namespace m3d
