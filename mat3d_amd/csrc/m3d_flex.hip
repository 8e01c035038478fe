// m3d_flex.hip -- planning and launchers of the passes of m3d_flex.hpp for the
// elastic and thermal solvers.
#include "m3d_flex.hpp"

#include <algorithm>
#include <stdexcept>
#include <vector>

namespace m3d {
namespace flex {

bool make_axis(int L, FftAxis& a)
{
    a = FftAxis{};
    a.L = L;
    // best radix sequence of every divisor of L: fewest passes, then smallest sum
    struct Best {
        int n = 0, cost = 0, radix = 0;
    };
    std::vector<Best> best(L + 1);
    for (int d = 2; d <= L; ++d) {
        if (L % d) continue;
        for (int r = 2; r <= 16; ++r) {
            if (d % r || (d != r && !best[d / r].radix)) continue;
            const int n = (d == r ? 0 : best[d / r].n) + 1, cost = (d == r ? 0 : best[d / r].cost) + r;
            if (!best[d].radix || n < best[d].n || (n == best[d].n && cost < best[d].cost)) best[d] = Best{n, cost, r};
        }
    }
    if (L > 1 && !best[L].radix) return false;
    std::vector<int> r;
    for (int d = L; d > 1; d /= best[d].radix) r.push_back(best[d].radix);
    if ((int)r.size() > 16) return false;
    std::sort(r.rbegin(), r.rend());
    a.np = (int)r.size();
    for (int i = 0; i < a.np; ++i) a.rad |= (unsigned long long)(r[i] - 1) << (4 * i);
    return true;
}

namespace {

int ept_of(size_t csz, int nt) { return nt == NT1 ? 8 : (csz == 8 ? ept<float, NT0>() : ept<double, NT0>()); }
int zcols_of(int C, int ny) { return C % 2 == 0 ? ny * (C / 2) : C * ((ny + 1) / 2); }

bool z_fits(const Geo& g, size_t csz, int ty, int nt)
{
    const int E = ept_of(csz, nt), W = zcols_of(g.C, ty);
    const long npair = (long)(g.C % 2 == 0 ? ty * (g.C / 2) : g.C * ((ty + 1) / 2)) * g.Nzh;
    const size_t lds = ((size_t)g.Nz * (W | 1) + (nt == NT0 ? g.Nz : 0)) * csz;
    return (long)g.Nz * W <= (long)E * nt && npair <= (long)(E / 2 + 1) * nt && lds <= (nt == NT0 ? 65536u : 160u * 1024u - 1024u);
}

int xy_tile(const Geo& g, size_t csz, int L)
{
    for (int nt : {NT0, NT1}) {
        const int tk = (int)((long)ept_of(csz, nt) * nt / ((long)g.C * L));
        if (tk >= 1) {
            // as wide as the workgroup holds, then evened out over the tiles
            const int n = (g.Nzh + tk - 1) / tk;
            return (g.Nzh + n - 1) / n;
        }
    }
    throw std::length_error("x/y line too long for one workgroup");
}

bool xy_long(const Geo& g, size_t csz, int L, int tk) { return (long)g.C * L * tk > (long)ept_of(csz, NT0) * NT0; }
bool z_long(const Geo& g, size_t csz) { return (long)g.Nz * zcols_of(g.C, g.TY) > (long)ept_of(csz, NT0) * NT0; }

// dynamic LDS above 64 KB has to be opted into
template <typename K>
void opt_in(K* kernel, size_t sm)
{
    if (sm > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
        if (e != hipSuccess) throw std::runtime_error(std::string("LDS size: ") + hipGetErrorString(e));
    }
}

template <typename T, typename PH, int MODE>
void z_mode(int which, const Geo& g, const Ptr<T>& p, hipStream_t st)
{
    const int W = zcols_of(g.C, g.TY) | 1;
    const long long total = (long long)g.nsolve * g.nbz;
    const unsigned grid = (unsigned)(MODE == MODE_CHK_CUR ? std::min<long long>(total, PH::chk_grid) : total);
    if (z_long(g, sizeof(cx<T>))) {
        const size_t sm = (size_t)g.Nz * W * sizeof(cx<T>);
        opt_in(&k_z<T, PH, MODE, NT1>, sm);
        hipLaunchKernelGGL((k_z<T, PH, MODE, NT1>), dim3(grid), dim3(NT1), sm, st, g, p, which);
    } else {
        const size_t sm = (size_t)g.Nz * (W + 1) * sizeof(cx<T>);
        hipLaunchKernelGGL((k_z<T, PH, MODE, NT0>), dim3(grid), dim3(NT0), sm, st, g, p, which);
    }
}

} // namespace

void plan(Geo& g, size_t csz)
{
    g.TY = 0;
    for (int nt : {NT0, NT1}) {
        for (int ty = g.Ny; ty >= 1 && !g.TY; --ty)
            if (z_fits(g, csz, ty, nt)) g.TY = ty;
        if (g.TY) {
            // rows evened out over the tiles; an even number of rows per tile
            // where rows are transformed in pairs
            g.nty = (g.Ny + g.TY - 1) / g.TY;
            int ty = (g.Ny + g.nty - 1) / g.nty;
            if (g.C % 2 && ty % 2 && z_fits(g, csz, ty + 1, nt)) ++ty;
            g.TY = ty;
            break;
        }
    }
    if (!g.TY) throw std::length_error("z line too long for one workgroup");
    g.nty = (g.Ny + g.TY - 1) / g.TY;
    g.nbz = g.Nx * g.nty;
    g.TKy = xy_tile(g, csz, g.Ny);
    g.nky = (g.Nzh + g.TKy - 1) / g.TKy;
    g.TKx = g.TKc = xy_tile(g, csz, g.Nx);
    g.nkx = (g.Nzh + g.TKx - 1) / g.TKx;
    g.nbx = g.nbc = g.Ny * g.nkx;
}

template <typename T, typename PH>
void launch_z(int mode, const Geo& g, const Ptr<T>& p, hipStream_t st)
{
    switch (mode) {
    case MODE_FWD: z_mode<T, PH, MODE_FWD>(BUF_MAIN, g, p, st); return;
    case MODE_IUF: z_mode<T, PH, MODE_IUF>(BUF_MAIN, g, p, st); return;
    case MODE_CHK_CUR: z_mode<T, PH, MODE_CHK_CUR>(BUF_CHK_CUR, g, p, st); return;
    case MODE_CHK_PREV: z_mode<T, PH, MODE_CHK_CUR>(BUF_CHK_PREV, g, p, st); return;
    default: break;
    }
    if constexpr (sizeof(T) == 4) {
        if (mode == MODE_IUFR) return z_mode<T, PH, MODE_IUFR>(BUF_MAIN, g, p, st);
    } else {
        if (mode == MODE_IUA) return z_mode<T, PH, MODE_IUA>(BUF_MAIN, g, p, st);
        if (mode == MODE_FWDP) return z_mode<T, PH, MODE_FWDP>(BUF_MAIN, g, p, st);
    }
    throw std::runtime_error("z pass mode");
}

template <typename T>
void launch_y(int dir, int which, unsigned cap, const Geo& g, const Ptr<T>& p, hipStream_t st)
{
    const long long total = (long long)g.nsolve * g.Nx * g.nky;
    const bool chk = which == BUF_CHK_CUR || which == BUF_CHK_PREV;
    const dim3 grid((unsigned)(chk ? std::min<long long>(total, cap) : total));
    const bool lg = xy_long(g, sizeof(cx<T>), g.Ny, g.TKy);
    const size_t sm = ((size_t)g.Ny * g.TKy * g.C + (lg ? 0 : g.Ny)) * sizeof(cx<T>);
    auto go = [&](auto* k, int nt) {
        opt_in(k, sm);
        hipLaunchKernelGGL(k, grid, dim3(nt), sm, st, g, p, which);
    };
    if (dir < 0) {
        if (lg) go(&k_y<T, -1, NT1>, NT1);
        else go(&k_y<T, -1, NT0>, NT0);
    } else {
        if (lg) go(&k_y<T, 1, NT1>, NT1);
        else go(&k_y<T, 1, NT0>, NT0);
    }
}

template <typename T, typename PH>
void launch_xgreen(const Geo& g, const Ptr<T>& p, const T* prm, hipStream_t st)
{
    const bool lg = xy_long(g, sizeof(cx<T>), g.Nx, g.TKx);
    const size_t sm = ((size_t)g.Nx * g.TKx * g.C + (lg ? 0 : g.Nx)) * sizeof(cx<T>);
    const dim3 grid((unsigned)((long long)g.nsolve * g.nbx));
    if (lg) {
        opt_in(&k_xg<T, PH, NT1>, sm);
        hipLaunchKernelGGL((k_xg<T, PH, NT1>), grid, dim3(NT1), sm, st, g, p, prm);
    } else {
        hipLaunchKernelGGL((k_xg<T, PH, NT0>), grid, dim3(NT0), sm, st, g, p, prm);
    }
}

template <typename T, typename PH>
void launch_xcheck(int which, const Geo& g, const Ptr<T>& p, hipStream_t st)
{
    const bool lg = xy_long(g, sizeof(cx<T>), g.Nx, g.TKc);
    const size_t sm = ((size_t)g.Nx * g.TKc * g.C + (lg ? 0 : g.Nx)) * sizeof(cx<T>);
    const dim3 grid((unsigned)std::min<long long>((long long)g.nsolve * g.nbc, PH::chk_grid));
    if (lg) {
        opt_in(&k_xc<T, PH, NT1>, sm);
        hipLaunchKernelGGL((k_xc<T, PH, NT1>), grid, dim3(NT1), sm, st, g, p, which);
    } else {
        hipLaunchKernelGGL((k_xc<T, PH, NT0>), grid, dim3(NT0), sm, st, g, p, which);
    }
}

#define M3D_FLEX(T)                                                                          \
    template void launch_z<T, Elastic>(int, const Geo&, const Ptr<T>&, hipStream_t);         \
    template void launch_z<T, Thermal>(int, const Geo&, const Ptr<T>&, hipStream_t);         \
    template void launch_y<T>(int, int, unsigned, const Geo&, const Ptr<T>&, hipStream_t);   \
    template void launch_xgreen<T, Elastic>(const Geo&, const Ptr<T>&, const T*, hipStream_t); \
    template void launch_xgreen<T, Thermal>(const Geo&, const Ptr<T>&, const T*, hipStream_t); \
    template void launch_xcheck<T, Elastic>(int, const Geo&, const Ptr<T>&, hipStream_t);    \
    template void launch_xcheck<T, Thermal>(int, const Geo&, const Ptr<T>&, hipStream_t);
M3D_FLEX(float)
M3D_FLEX(double)

} // namespace flex
} // namespace m3d
