// m3d_basic_fast.hpp -- interface of the compile-time specialised kernels of
// the basic scheme ("ep" / "ed", FFT_analysis3D.cpp:796-853), defined in
// m3d_basic.hip: z pass with the constitutive update, y pass on 12 (start
// stage) or 6 components, x pass with eqVar partials and the Green step, y pass
// on 6, with every FFT length and tile a template constant.
#pragma once
#include "m3d_basic.hpp"
#include "m3d_fast.hpp"

namespace m3d {
namespace bfast {

#ifndef M3D_BZ_THREADS
#define M3D_BZ_THREADS 256
#endif
#ifndef M3D_BZ_TILE
#define M3D_BZ_TILE 2304
#endif
#ifndef M3D_BZ_PAD
#define M3D_BZ_PAD 0 // complex values of padding per LDS row of the z pass
#endif
#ifndef M3D_BX_TILE
#define M3D_BX_TILE 6144
#endif
// minimum waves per SIMD the register allocator must leave room for in the
// z and x passes (0: no constraint)
#ifndef M3D_BZ_WAVES
#define M3D_BZ_WAVES 0
#endif
#ifndef M3D_BX_WAVES
#define M3D_BX_WAVES 0
#endif
#if M3D_BZ_WAVES > 0
#define M3D_BZ_ATTR __attribute__((amdgpu_waves_per_eu(M3D_BZ_WAVES)))
#else
#define M3D_BZ_ATTR
#endif
#if M3D_BX_WAVES > 0
#define M3D_BX_ATTR __attribute__((amdgpu_waves_per_eu(M3D_BX_WAVES)))
#else
#define M3D_BX_ATTR
#endif
constexpr int ZNT = M3D_BZ_THREADS; // threads of the z pass
// x pass: lines of up to 128 points on half tiles of 256 threads (two more
// workgroups per CU to overlap), longer ones on full tiles of 512.  Measured per
// J2 load path, half against full: 32^3 15.3 / 16.1 ms, 48^3 25.2 / 25.7, 64^3
// 49.9 / 50.9, 96^3 82.8 / 91.7, 128^3 190 / 193, 192^3 670 / 648.
constexpr int xthreads(int L) { return L <= 128 ? 256 : 512; }

// z tile: TY lines (y) of 12 components each, TY*12*LZ <= M3D_BZ_TILE complex
constexpr int zlines(int LZ, int Ny)
{
    int ty = 1;
    while (ty < 8 && (ty * 2) * 12 * LZ <= M3D_BZ_TILE && Ny % (ty * 2) == 0) ty *= 2;
    return ty;
}
// x tile: TK kz values of 12 components (TK * L <= M3D_BX_TILE / 12, half of it
// for short lines)
constexpr int xtile(int L)
{
    const int tk = (L <= 128 ? M3D_BX_TILE / 2 : M3D_BX_TILE) / (12 * L);
    return tk < 1 ? 1 : tk;
}
// y tiles (the generic fast y pass with 12 / 6 components)
constexpr int ytile12(int L) { return fast::xytile<double>(L, 12); }
constexpr int ytile6(int L) { return fast::xytile<double>(L, 6); }

// line lengths with specialised basic kernels: z half-lengths and x/y lengths
inline bool z_supported(int LZ) { return LZ == 16 || LZ == 24 || LZ == 32 || LZ == 48 || LZ == 64 || LZ == 96 || LZ == 128; }
inline bool xy_supported(int L) { return L == 32 || L == 48 || L == 64 || L == 96 || L == 128 || L == 192 || L == 256; }
inline bool supported(int Nx, int Ny, int Nz)
{
    return Nz % 2 == 0 && z_supported(Nz / 2) && xy_supported(Nx) && xy_supported(Ny) && Ny % zlines(Nz / 2, Ny) == 0 &&
           zlines(Nz / 2, Ny) == zlines(Nz / 2, Nz);
}

// host launchers (m3d_basic.hip); g carries Nx..Nzh, N, H, invN, nbz, nbx
// of the tiles above, TY, TKx; the y launch takes the 12- or 6-component
// view of the spectra in p (S: 6-component Green output, K: 12-component) and
// the finaliser to run beside them
// (T = double or float)
// lin: every phase has hardening exponent n = 1 (FP64 "ep" then runs the
// return map without pow, bit for bit the same arithmetic)
template <typename T>
void launch_z(int beh, int mode, const Geo& g, const BPtr<T>& p, hipStream_t st, bool lin = false);
template <typename T>
void launch_y12(const Geo& g, const Ptr<T>& p, const BFin& f, hipStream_t st);
// forward y pass of the 6-component sigma^ spectrum that an ITER z pass
// leaves in the K view
template <typename T>
void launch_y6_fwd(const Geo& g, const Ptr<T>& p, const BFin& f, hipStream_t st);
// e6: the x pass after an ITER z pass (sigma^ with 6 components, eps^ from Eh)
template <typename T>
void launch_x(const Geo& g, const BPtr<T>& p, hipStream_t st, bool e6);
template <typename T>
void launch_y6(const Geo& g, const Ptr<T>& p, const BFin& f, hipStream_t st);

} // namespace bfast

// The same passes for every other grid, in FP64 (m3d_flex_basic.hip): g is a
// run-time plan of 12 (start stage) or 6 components (iterations, FINAL) whose
// z and x tiles plan() has set.
namespace bflex {
void plan(Geo& g);
void launch_z(int beh, int mode, const Geo& g, const BPtr<double>& p, hipStream_t st, bool lin);
void launch_y(int dir, int which, const Geo& g, const Ptr<double>& p, const BFin& f, hipStream_t st);
void launch_x(const Geo& g, const BPtr<double>& p, hipStream_t st, bool e6);
} // namespace bflex
} // namespace m3d
