// m3d_flex.hpp -- passes for line lengths without a compile-time kernel (any
// product of primes up to 13).
//
// Same dataflow, tiles and LDS layout (lines interleaved: element e of line l
// at e*ws + l) as m3d_fast.hpp, with the line length and the tile width as
// run-time values.  What makes that cheap:
//   * radices 2..16 with compile-time butterflies (100 = 10*10, 65 = 13*5: two
//     LDS round trips), one switch per pass on a uniform radix;
//   * divisions of indexes by run-time widths through a float reciprocal (two
//     full-rate instructions, exact for the tile's index range) and 24-bit
//     multiplies instead of the quarter-rate 32-bit ones;
//   * the loads of a tile are issued together before the first LDS store;
//   * twiddle tables in LDS (in global memory for the 1024-thread form).
//
// The z pass transforms two real lines as one complex line of the full length
// Nz (odd lengths need no special case): Z = A + iB is formed while the half
// spectra A, B are loaded and taken apart while they are stored, so neither
// needs a pass over LDS of its own.  With an even number of components the
// pair is two components of one row, and a voxel's C components are adjacent
// in LDS; with three components it is one component of two rows.
//
// Bound: HBM (or the memory-side cache, which a 100^3 batch of six solves
// fits) for large batches, latency below about 50^3.  Measured per launch,
// six solves, against the run-time-planned passes this replaces (one voxel
// per thread through scalar loads, odd radices as direct DFTs with twiddles
// from global memory, integer divisions by run-time widths):
//   100^3 FP32     z update 835 -> 129 us, x with the Green step 378 -> 74, y
//                  238 -> 48 (averages of a homogenization; while all six
//                  solves run 151 us, 3.9 TB/s, 84, 3.5, and 55, 5.3)
//   45x50x56 FP64  z 237 -> 42, x 131 -> 31, y 82 -> 21 us
//   96^3 thermal   (three solves, FP64) z 103 -> 74, x 88 -> 39, y 54 -> 27 us
// A homogenization, with the check passes left out where no solve needs them:
// 100^3 FP32 101 -> 24 ms, 45x50x56 FP64 16.9 -> 3.9, 96^3 thermal 10.4 -> 5.2.
#pragma once
#include "m3d_fast.hpp"

namespace m3d {
namespace flex {

// A workgroup holds at most EPT complex values per thread.  256 threads
// where a tile of one line group fits (every elastic line up to 512 points in
// FP32 and 341 in FP64), 1024 for longer lines.
constexpr int NT0 = 256, NT1 = 1024;
template <typename T, int NT>
constexpr int ept()
{
    return NT == NT1 ? 8 : (sizeof(T) == 4 ? 12 : 8);
}

// floor(x / d) for 0 <= x < 2^14, inv = 1.0f / d: the relative error of the
// product is below 2^-23, so the absolute one is below 2^-9 / d, while x + 1/2
// is at least 1 / (2 d) away from the next multiple of d
__device__ __forceinline__ int fdiv(int x, float inv) { return (int)(((float)x + 0.5f) * inv); }
__device__ __forceinline__ int mul24(int a, int b) { return (int)__umul24((unsigned)a, (unsigned)b); }

// One in-place Stockham pass of radix R over W interleaved lines of length L
// (LDS row stride ws >= W); rem = L / Ns before the pass.  Returns rem / R.
template <typename T, int R, int DIR, int NT>
__device__ __forceinline__ int pass(cx<T>* __restrict__ s, const cx<T>* __restrict__ tw, int L, int W, int ws, float invW,
                                    int Ns, int rem)
{
    constexpr int IPT = (ept<T, NT>() + R - 1) / R;
    const int nR = (int)((unsigned)L / (unsigned)R);
    const int items = nR * W;
    const int tstep = (int)((unsigned)rem / (unsigned)R);
    const int sr = nR * ws, sw = Ns * ws;
    const float invNs = 1.0f / (float)Ns;
    const int tid = fast::lane_tid();
    cx<T> v[IPT][R];
    int o[IPT];
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
        const int it = tid + i * NT;
        if (it < items) {
            const int j = fdiv(it, invW), l = it - mul24(j, W);
            const cx<T>* a = s + (mul24(j, ws) + l);
#pragma unroll
            for (int r = 0; r < R; ++r) v[i][r] = a[r * sr];
            if (Ns == 1) {
                o[i] = mul24(j, R * ws) + l;
            } else {
                const int q = fdiv(j, invNs), k = j - mul24(q, Ns);
                o[i] = mul24(mul24(q, Ns * R) + k, ws) + l;
                const int kt = mul24(k, tstep);
                int m = kt;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    v[i][r] = fast::twmul<DIR>(v[i][r], tw[m]);
                    m += kt;
                }
            }
            butterfly<T, R, DIR>(v[i]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
        const int it = tid + i * NT;
        if (it < items) {
#pragma unroll
            for (int r = 0; r < R; ++r) s[o[i] + r * sw] = v[i][r];
        }
    }
    __syncthreads();
    return tstep;
}

template <typename T, int DIR, int NT>
__device__ __forceinline__ void fft(cx<T>* __restrict__ s, const cx<T>* __restrict__ tw, const FftAxis& ax, int W, int ws,
                                    float invW)
{
    int Ns = 1, rem = ax.L;
    for (int p = 0; p < ax.np; ++p) {
        const int R = ax.radix(p);
        switch (R) {
        case 2: rem = pass<T, 2, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 3: rem = pass<T, 3, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 4: rem = pass<T, 4, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 5: rem = pass<T, 5, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 6: rem = pass<T, 6, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 7: rem = pass<T, 7, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 8: rem = pass<T, 8, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 9: rem = pass<T, 9, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 10: rem = pass<T, 10, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 11: rem = pass<T, 11, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 12: rem = pass<T, 12, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 13: rem = pass<T, 13, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 14: rem = pass<T, 14, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        case 15: rem = pass<T, 15, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        default: rem = pass<T, 16, DIR, NT>(s, tw, ax.L, W, ws, invW, Ns, rem); break;
        }
        Ns *= R;
    }
}

// twiddle table: a copy in LDS, or the global table itself (1024 threads)
template <typename T, int NT>
__device__ __forceinline__ const cx<T>* stage_twiddles(cx<T>* lds, const cx<T>* __restrict__ table, int n)
{
    if constexpr (NT == NT1) return table;
    for (int i = threadIdx.x; i < n; i += NT) lds[i] = table[i];
    return lds;
}

// ------------------------------------------------------------- tile movers
// Rows of w contiguous complex values (row r at base + r*stride) <-> LDS,
// rows back to back.  G complex values per access (2: 16 bytes in FP32).
template <typename T, int NT, int G>
struct Rows {
    using V = typename std::conditional<G == 2, fast::vf4, typename std::conditional<sizeof(T) == 4, fast::vf2, fast::vd2>::type>::type;
    static constexpr int PER = (ept<T, NT>() + G - 1) / G;
};

template <typename T, int NT, int G, typename F>
__device__ __forceinline__ void rows_each(long long stride, int rows, int w, F&& f)
{
    // byte offsets by one 24-bit multiply where they fit, else in 64 bits
    const int wg = w / G, n = rows * wg;
    const float inv = 1.0f / (float)wg;
    const int tid = fast::lane_tid();
    const long long sb = stride * (long long)sizeof(cx<T>);
    if (sb < (1ll << 24) && sb * rows < (1ll << 32)) {
#pragma unroll
        for (int i = 0; i < Rows<T, NT, G>::PER; ++i) {
            const int e = tid + i * NT;
            if (e < n) {
                const int r = fdiv(e, inv), j = e - mul24(r, wg);
                f(i, e, (long long)(fast::mul_u24((unsigned)r, (unsigned)sb) + (unsigned)j * (unsigned)(G * sizeof(cx<T>))));
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < Rows<T, NT, G>::PER; ++i) {
            const int e = tid + i * NT;
            if (e < n) {
                const int r = fdiv(e, inv), j = e - mul24(r, wg);
                f(i, e, (long long)r * sb + (long long)j * (long long)(G * sizeof(cx<T>)));
            }
        }
    }
}

template <typename T, int NT, int G>
__device__ __forceinline__ void load_rows(cx<T>* __restrict__ sl, const cx<T>* __restrict__ base, long long stride, int rows,
                                          int w)
{
    using V = typename Rows<T, NT, G>::V;
    V r[Rows<T, NT, G>::PER];
    const char* bb = reinterpret_cast<const char*>(base);
    rows_each<T, NT, G>(stride, rows, w, [&](int i, int, long long o) { r[i] = *reinterpret_cast<const V*>(bb + o); });
    const int n = rows * (w / G);
    const int tid = fast::lane_tid();
#pragma unroll
    for (int i = 0; i < Rows<T, NT, G>::PER; ++i) {
        const int e = tid + i * NT;
        if (e < n) *reinterpret_cast<V*>(sl + e * G) = r[i];
    }
}

template <typename T, int NT, int G>
__device__ __forceinline__ void store_rows(const cx<T>* __restrict__ sl, cx<T>* __restrict__ base, long long stride, int rows,
                                           int w)
{
    using V = typename Rows<T, NT, G>::V;
    char* bb = reinterpret_cast<char*>(base);
    rows_each<T, NT, G>(stride, rows, w, [&](int, int e, long long o) {
        *reinterpret_cast<V*>(bb + o) = *reinterpret_cast<const V*>(sl + e * G);
    });
}

// 16-byte accesses to FP32 rows: even row width and pitch, aligned base
template <typename T>
__device__ __forceinline__ bool pairs_ok(const cx<T>* base, long long stride, int w)
{
    return sizeof(T) == 4 && (w & 1) == 0 && (stride & 1) == 0 && (reinterpret_cast<unsigned long long>(base) & 15) == 0;
}

template <typename T, int NT>
__device__ __forceinline__ void load_tile(cx<T>* sl, const cx<T>* base, long long stride, int rows, int w)
{
    if constexpr (sizeof(T) == 4) {
        if (pairs_ok<T>(base, stride, w)) {
            load_rows<T, NT, 2>(sl, base, stride, rows, w);
            return;
        }
    }
    load_rows<T, NT, 1>(sl, base, stride, rows, w);
}

template <typename T, int NT>
__device__ __forceinline__ void store_tile(const cx<T>* sl, cx<T>* base, long long stride, int rows, int w)
{
    if constexpr (sizeof(T) == 4) {
        if (pairs_ok<T>(base, stride, w)) {
            store_rows<T, NT, 2>(sl, base, stride, rows, w);
            return;
        }
    }
    store_rows<T, NT, 1>(sl, base, stride, rows, w);
}

// ------------------------------------------------------------ y and x passes
__host__ __device__ __forceinline__ bool active(const Ctl& c, int which)
{
    return !c.done && !c.wait && (which != BUF_CHK_CUR || c.need_cur) && (which != BUF_CHK_PREV || c.need_prev);
}

// any solve takes part in a check pass (called by the whole workgroup)
__device__ __forceinline__ bool any_active(const Geo& g, const Ctl* ctl, int which)
{
    int mine = 0;
    for (int s = threadIdx.x; s < g.nsolve; s += blockDim.x) mine |= active(ctl[s], which);
    return __syncthreads_or(mine) != 0;
}

// complex FFT along y in place; which selects the spectrum (BUF_MAIN: S, else K)
template <typename T, int DIR, int NT>
__device__ __forceinline__ void y_tile(const Geo& g, const Ptr<T>& p, int which, int b, cx<T>* sl, cx<T>* twl)
{
    const int per = g.Nx * g.nky;
    const int s = b / per, t = b - s * per;
    if (!active(p.ctl[s], which)) return;
    const int x = t / g.nky, kz0 = (t - x * g.nky) * g.TKy;
    const int w = min(g.TKy, g.Nzh - kz0) * g.C;
    cx<T>* base = (which == BUF_MAIN ? p.S : p.K) + (long long)s * p.sS + (long long)x * g.sxa + (long long)kz0 * g.C;
    const cx<T>* tw = stage_twiddles<T, NT>(twl, p.twy, g.Ny);
    load_tile<T, NT>(sl, base, g.sy, g.Ny, w);
    __syncthreads();
    fft<T, DIR, NT>(sl, tw, g.ay, w, w, 1.0f / (float)w);
    store_tile<T, NT>(sl, base, g.sy, g.Ny, w);
}

// The check passes run a capped grid that loops over the tiles and leaves at
// once when no solve needs the check; the main passes one workgroup per tile.
template <typename T, int DIR, int NT>
__global__ void __launch_bounds__(NT) k_y(Geo g, Ptr<T> p, int which)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* sl = reinterpret_cast<cx<T>*>(smem_raw);
    cx<T>* twl = sl + (size_t)g.Ny * g.TKy * g.C;
    if ((which == BUF_CHK_CUR || which == BUF_CHK_PREV) && !any_active(g, p.ctl, which)) return;
    const int total = g.nsolve * g.Nx * g.nky;
    for (int b = blockIdx.x; b < total; b += gridDim.x) {
        y_tile<T, DIR, NT>(g, p, which, fast::xcd_split(b, total, g.Nx * g.nky), sl, twl);
        __syncthreads();
    }
}

// x FFT, Green step (DC = E), inverse x FFT
template <typename T, typename PH, int NT>
__global__ void __launch_bounds__(NT) k_xg(Geo g, Ptr<T> p, const T* __restrict__ prm_all)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int C = PH::C;
    cx<T>* sl = reinterpret_cast<cx<T>*>(smem_raw);
    cx<T>* twl = sl + (size_t)g.Nx * g.TKx * C;
    const int per = g.Ny * g.nkx;
    const int b = fast::xcd_split(blockIdx.x, gridDim.x, per);
    const int s = b / per, t = b - s * per;
    const Ctl& ctl = p.ctl[s];
    if (ctl.done || ctl.wait) return;
    const int y = t / g.nkx, kz0 = (t - y * g.nkx) * g.TKx;
    const int nk = min(g.TKx, g.Nzh - kz0), w = nk * C;
    cx<T>* base = p.S + (long long)s * p.sS + (long long)y * g.sy + (long long)kz0 * C;
    const cx<T>* tw = stage_twiddles<T, NT>(twl, p.twx, g.Nx);
    load_tile<T, NT>(sl, base, g.sxa, g.Nx, w);
    __syncthreads();
    const float invw = 1.0f / (float)w;
    fft<T, -1, NT>(sl, tw, g.ax, w, w, invw);
    const GreenK<T> K = green_k_of<T, C>(prm_all + 2 * p.rve_of[s]);
    const float invk = 1.0f / (float)nk;
    for (int f = fast::lane_tid(); f < g.Nx * nk; f += NT) {
        const int kx = fdiv(f, invk), kzl = f - mul24(kx, nk), kz = kz0 + kzl;
        cx<T>* v = sl + (mul24(kx, w) + kzl * C);
        if (kx == 0 && y == 0 && kz == 0) {
#pragma unroll
            for (int c = 0; c < C; ++c) v[c] = cx<T>{T(ctl.E[c]), T(0)};
        } else {
            green_apply_k<T, PH>(g, ctl.sb, K, kx, y, kz, v);
        }
    }
    __syncthreads();
    fft<T, 1, NT>(sl, tw, g.ax, w, w, invw);
    store_tile<T, NT>(sl, base, g.sxa, g.Nx, w);
}

// x FFT of the check spectrum and the equilibrium partial sums
template <typename T, typename PH, int NT>
__global__ void __launch_bounds__(NT) k_xc(Geo g, Ptr<T> p, int which)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double red[NT / 64];
    constexpr int C = PH::C;
    cx<T>* sl = reinterpret_cast<cx<T>*>(smem_raw);
    cx<T>* twl = sl + (size_t)g.Nx * g.TKc * C;
    if (!any_active(g, p.ctl, which)) return;
    const int nkc = g.nbc / g.Ny, total = g.nsolve * g.nbc;
    const cx<T>* tw = stage_twiddles<T, NT>(twl, p.twx, g.Nx);
    for (int bb = blockIdx.x; bb < total; bb += gridDim.x) {
        const int b = fast::xcd_split(bb, total, g.nbc);
        const int s = b / g.nbc, t = b - s * g.nbc;
        if (!active(p.ctl[s], which)) continue; // uniform for the workgroup
        const int y = t / nkc, kz0 = (t - y * nkc) * g.TKc;
        const int nk = min(g.TKc, g.Nzh - kz0), w = nk * C;
        load_tile<T, NT>(sl, p.K + (long long)s * p.sS + (long long)y * g.sy + (long long)kz0 * C, g.sxa, g.Nx, w);
        __syncthreads();
        fft<T, -1, NT>(sl, tw, g.ax, w, w, 1.0f / (float)w);
        double* pc = p.pchk + ((long long)s * 2 + (which == BUF_CHK_CUR ? 0 : 1)) * (g.nbc + 1);
        const float invk = 1.0f / (float)nk;
        double acc = 0.0;
        for (int f = fast::lane_tid(); f < g.Nx * nk; f += NT) {
            const int kx = fdiv(f, invk), kzl = f - mul24(kx, nk), kz = kz0 + kzl;
            const cx<T>* v = sl + (mul24(kx, w) + kzl * C);
            double a2[C];
            acc += eq_term<T, C>(g, kx, y, kz, v, a2);
            if (kx == 0 && y == 0 && kz == 0) pc[g.nbc] = eq_mean<C>(a2);
        }
        const double bs = block_sum(acc, red);
        if (threadIdx.x == 0) pc[t] = bs;
        __syncthreads();
    }
}

// ------------------------------------------------------------------ z pass
// columns of a z tile of ny rows: pairs of components (even C) or of rows
template <int C>
__host__ __device__ constexpr int zcols(int ny)
{
    return C % 2 == 0 ? ny * (C / 2) : C * ((ny + 1) / 2);
}

// The pairs (A, B) of half-spectrum values of a z tile's rows, flat over
// their memory order: even C: (kz, 2q), (kz, 2q + 1) of one row; odd C:
// (kz, q) of rows 2a and 2a + 1 (B = 0 where an odd tile has no second row).
template <int C>
struct ZPairs {
    static constexpr bool CP = C % 2 == 0;
    static constexpr int HC = CP ? C / 2 : C; // columns per row (CP) or per pair of rows
    int Nz, ny, rowi, n;
    float inv;
    __device__ __forceinline__ ZPairs(int Nz_, int Nzh, int ny_) : Nz(Nz_), ny(ny_)
    {
        rowi = Nzh * HC;
        n = (CP ? ny : (ny + 1) / 2) * rowi;
        inv = 1.0f / (float)rowi;
    }
    __device__ __forceinline__ void at(int e, int& yr, int& kz, int& q) const
    {
        yr = fdiv(e, inv);
        const int r = e - mul24(yr, rowi);
        kz = (int)((unsigned)r / (unsigned)HC);
        q = r - kz * HC;
    }
    // global -> registers; sy: row stride
    template <typename T, int NT, int PER>
    __device__ __forceinline__ void issue(const cx<T>* __restrict__ src, long long sy, cx<T> (&ca)[PER], cx<T> (&cb)[PER]) const
    {
        const int tid = fast::lane_tid();
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = tid + i * NT;
            if (e < n) {
                int yr, kz, q;
                at(e, yr, kz, q);
                if constexpr (CP) {
                    const cx<T>* a = src + (long long)yr * sy + (kz * C + 2 * q);
                    if constexpr (sizeof(T) == 4) {
                        const fast::vf4 f = *reinterpret_cast<const fast::vf4*>(a);
                        ca[i] = cx<T>{f.x, f.y};
                        cb[i] = cx<T>{f.z, f.w};
                    } else {
                        ca[i] = a[0];
                        cb[i] = a[1];
                    }
                } else {
                    const cx<T>* a = src + (long long)(2 * yr) * sy + (kz * C + q);
                    ca[i] = a[0];
                    cb[i] = 2 * yr + 1 < ny ? a[sy] : cx<T>{T(0), T(0)};
                }
            }
        }
    }
    // registers -> LDS: Z[k] = A + iB, Z[Nz-k] = conj(A) + i conj(B); kz = 0
    // and Nz/2 keep the real parts of A and B (what a c2r transform reads)
    template <typename T, int NT, int PER>
    __device__ __forceinline__ void commit(cx<T>* __restrict__ sl, int ws, const cx<T> (&ca)[PER], const cx<T> (&cb)[PER]) const
    {
        const int tid = fast::lane_tid();
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = tid + i * NT;
            if (e < n) {
                int yr, kz, q;
                at(e, yr, kz, q);
                const int col = yr * HC + q;
                const cx<T> A = ca[i], B = cb[i];
                if (kz == 0 || 2 * kz == Nz) {
                    sl[mul24(kz, ws) + col] = cx<T>{A.re, B.re};
                } else {
                    sl[mul24(kz, ws) + col] = cx<T>{A.re - B.im, A.im + B.re};
                    sl[mul24(Nz - kz, ws) + col] = cx<T>{A.re + B.im, B.re - A.im};
                }
            }
        }
    }
    // LDS -> global: A = (Z[k] + conj Z[Nz-k]) / 2, B = (Z[k] - conj Z[Nz-k]) / 2i
    template <typename T, int NT>
    __device__ __forceinline__ void store(const cx<T>* __restrict__ sl, int ws, cx<T>* __restrict__ dst, long long sy) const
    {
        for (int e = fast::lane_tid(); e < n; e += NT) {
            int yr, kz, q;
            at(e, yr, kz, q);
            const int col = yr * HC + q;
            const cx<T> zk = sl[mul24(kz, ws) + col], zc = cconj(sl[mul24(kz == 0 ? 0 : Nz - kz, ws) + col]);
            const cx<T> A = cscale(zk + zc, T(0.5)), B = cscale(rot90<-1>(zk - zc), T(0.5));
            if constexpr (CP) {
                cx<T>* a = dst + (long long)yr * sy + (kz * C + 2 * q);
                if constexpr (sizeof(T) == 4) {
                    *reinterpret_cast<fast::vf4*>(a) = fast::vf4{A.re, A.im, B.re, B.im};
                } else {
                    a[0] = A;
                    a[1] = B;
                }
            } else {
                cx<T>* a = dst + (long long)(2 * yr) * sy + (kz * C + q);
                a[0] = A;
                if (2 * yr + 1 < ny) a[sy] = B;
            }
        }
    }
};

// a voxel's C values of one field, contiguous in memory (4- or 8-byte aligned)
template <typename T, int C>
struct __attribute__((packed, aligned(sizeof(T)))) Vox {
    T v[C];
};

// Modes and buffers as in fast::kz_tile; which = BUF_CHK_CUR / BUF_CHK_PREV
// selects the iterate of MODE_CHK_CUR.
template <typename T, typename PH, int MODE, int NT>
__device__ __forceinline__ void z_tile(const Geo& g, const Ptr<T>& p, int which, int b, cx<T>* sl, cx<T>* twl, double* red)
{
    constexpr int C = PH::C;
    constexpr bool CP = C % 2 == 0;
    constexpr int HC = ZPairs<C>::HC;
    constexpr int E = ept<T, NT>();
    constexpr bool IUF = MODE == MODE_IUF || MODE == MODE_IUFR || MODE == MODE_IUA;
    constexpr bool ANC = MODE == MODE_IUA;
    constexpr bool CHK = MODE == MODE_CHK_CUR;
    constexpr bool FWD = MODE == MODE_FWD || MODE == MODE_FWDP;
    const int s = b / g.nbz, t = b - s * g.nbz;
    const Ctl& ctl = p.ctl[s];
    if (ctl.done || ctl.wait || (CHK && !active(ctl, which))) return;
    const int it = ctl.it;
    const int x = t / g.nty, y0 = (t - x * g.nty) * g.TY;
    const int ny = min(g.TY, g.Ny - y0);
    const int Nz = g.Nz, Nzh = g.Nzh;
    const int W = zcols<C>(ny), ws = W | 1; // odd LDS row stride: voxel rows spread over the banks
    const int tid = threadIdx.x;

    const long long vox0 = ((long long)x * g.Ny + y0) * Nz;
    const long long spec0 = (long long)x * g.sxa + (long long)y0 * g.sy;
    const int rv = p.rve_of[s];
    const uint8_t* ph = p.ph + (long long)rv * p.sPh + vox0;
    const T* coef = p.coef + (long long)rv * p.sCoef;
    const T* Uin;
    T* Uout = nullptr;
    const float* Ein = nullptr; // FP64 check of an anchored solve: anchor + FP32 correction
    if constexpr (CHK) {
        const int ci = which == BUF_CHK_CUR ? it : it - 1;
        Uin = u_buf(p, ci, s);
        if (sizeof(T) == 8 && ctl.corr) {
            Uin = u_buf(p, ctl.anc_it, s);
            Ein = e_buf(p, ci, s) + vox0 * C;
        }
    } else {
        Uin = u_buf(p, it, s);
    }
    if constexpr (IUF) Uout = u_buf(p, it + 1, s) + vox0 * C;
    Uin += vox0 * C;
    const float* Rin = MODE == MODE_IUFR ? p.R + (long long)s * p.sU + vox0 * C : nullptr;

    const cx<T>* tw = stage_twiddles<T, NT>(twl, p.twz, Nz);

    const ZPairs<C> zp(Nz, Nzh, ny);
    constexpr int PER = E / 2 + 1;
    cx<T> ca[IUF ? PER : 1], cb[IUF ? PER : 1];
    if constexpr (IUF) zp.template issue<T, NT, PER>(p.S + (long long)s * p.sS + spec0, g.sy, ca, cb);
    // voxels: flat over the tile's rows
    constexpr int VPT = (2 * E + C - 1) / C; // an odd last row makes fewer voxels per column
    const int nv = ny * Nz;
    const float inv_nz = 1.0f / (float)Nz;
    T u[VPT][C];
    float rr[MODE == MODE_IUFR ? VPT : 1][C];
    uint8_t pv[VPT];
    using VT = Vox<T, C>;
    using VF = Vox<float, C>;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int v = tid + i * NT;
        if (v < nv) {
            if constexpr (MODE == MODE_FWDP) {
                const VF f = *reinterpret_cast<const VF*>(e_buf(p, it, s) + (vox0 + v) * C);
                VT d;
#pragma unroll
                for (int c = 0; c < C; ++c) u[i][c] = d.v[c] = (T)f.v[c];
                *reinterpret_cast<VT*>(u_buf(p, it, s) + (vox0 + v) * C) = d;
            } else {
                const VT f = *reinterpret_cast<const VT*>(Uin + (long long)v * C);
#pragma unroll
                for (int c = 0; c < C; ++c) u[i][c] = f.v[c];
            }
            if constexpr (MODE == MODE_IUFR) {
                const VF f = *reinterpret_cast<const VF*>(Rin + (long long)v * C);
#pragma unroll
                for (int c = 0; c < C; ++c) rr[i][c] = f.v[c];
            }
            pv[i] = ph[v];
            if constexpr (CHK && sizeof(T) == 8) {
                if (Ein) {
                    const VF f = *reinterpret_cast<const VF*>(Ein + (long long)v * C);
#pragma unroll
                    for (int c = 0; c < C; ++c) u[i][c] += (T)f.v[c];
                }
            }
        }
    }

    if constexpr (IUF) {
        zp.template commit<T, NT, PER>(sl, ws, ca, cb);
        __syncthreads();
        fft<T, 1, NT>(sl, tw, g.az, W, ws, 1.0f / (float)W);
    } else {
        __syncthreads();
    }

    // per voxel: slot m of a column holds (A, B) of sample m
    T* sr = reinterpret_cast<T*>(sl);
    double acc = 0.0;
    const int vt = fast::lane_tid(); // addresses recomputed here, not kept across the transform
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int v = vt + i * NT;
        if (v < nv) {
            const int yl = fdiv(v, inv_nz), m = v - mul24(yl, Nz);
            // component c of the voxel at rp[c * RS]
            constexpr int RSC = CP ? 1 : 2;
            T* rp = CP ? sr + 2 * (mul24(m, ws) + yl * HC) : sr + 2 * (mul24(m, ws) + (yl >> 1) * HC) + (yl & 1);
            const T* kp = coef + (int)pv[i] * NCOEF;
            T w[C], o[C];
#pragma unroll
            for (int c = 0; c < C; ++c) w[c] = u[i][c];
            if constexpr (IUF) {
                T d[C], a[C];
#pragma unroll
                for (int c = 0; c < C; ++c) d[c] = rp[c * RSC] - w[c];
                PH::accel(kp, d, a);
                VT un;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    w[c] += a[c];
                    if constexpr (MODE == MODE_IUFR) w[c] += rr[i][c];
                    un.v[c] = w[c];
                }
                *reinterpret_cast<VT*>(Uout + (long long)v * C) = un;
                if constexpr (ANC) {
                    // r = T(A) - A in FP64, kept in FP32, and the first correction e = r
                    VF f;
#pragma unroll
                    for (int c = 0; c < C; ++c) f.v[c] = (float)(w[c] - u[i][c]);
                    *reinterpret_cast<VF*>(const_cast<float*>(p.R) + (long long)s * p.sU + (vox0 + v) * C) = f;
                    *reinterpret_cast<VF*>(const_cast<float*>(e_buf(p, it + 1, s)) + (vox0 + v) * C) = f;
                }
            }
            if constexpr (FWD || IUF) {
                PH::dual(kp, w, o);
#pragma unroll
                for (int c = 0; c < C; ++c) acc += (double)o[c];
                if constexpr (!ANC) PH::polar(kp, w, o);
            } else if (ctl.sb) {
                PH::dual(kp, w, o);
            } else {
#pragma unroll
                for (int c = 0; c < C; ++c) o[c] = w[c];
            }
            if constexpr (!ANC) {
#pragma unroll
                for (int c = 0; c < C; ++c) rp[c * RSC] = o[c];
                // the missing row of an odd last pair
                if constexpr (!CP) {
                    if (yl == ny - 1 && (ny & 1)) {
#pragma unroll
                        for (int c = 0; c < C; ++c) rp[c * RSC + 1] = T(0);
                    }
                }
            }
        }
    }
    if constexpr (FWD || IUF) {
        const double bs = block_sum(acc, red);
        if (tid == 0) p.psum[(long long)s * g.nbz + t] = bs;
    }
    if constexpr (ANC) return;
    __syncthreads();

    fft<T, -1, NT>(sl, tw, g.az, W, ws, 1.0f / (float)W);
    zp.template store<T, NT>(sl, ws, ((FWD || IUF) ? p.S : p.K) + (long long)s * p.sS + spec0, g.sy);
}

template <typename T, typename PH, int MODE, int NT>
__global__ void __launch_bounds__(NT) k_z(Geo g, Ptr<T> p, int which)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double red[NT / 64];
    cx<T>* sl = reinterpret_cast<cx<T>*>(smem_raw);
    cx<T>* twl = sl + (size_t)g.Nz * (zcols<PH::C>(g.TY) | 1);
    constexpr bool CHK = MODE == MODE_CHK_CUR;
    if (CHK && !any_active(g, p.ctl, which)) return;
    const int total = g.nsolve * g.nbz;
    for (int b = blockIdx.x; b < total; b += gridDim.x) {
        z_tile<T, PH, MODE, NT>(g, p, which, fast::xcd_split(b, total, g.nbz), sl, twl, red);
        __syncthreads();
    }
}

// --------------------------------------------------------------- planning
// radices of a line of L points: the fewest passes, then the smallest sum;
// the largest radix first (the first pass has no twiddles).  False if L has a
// prime factor above 13.
bool make_axis(int L, FftAxis& a);

// tile shapes of the passes of g (C components, complex values of csz bytes)
void plan(Geo& g, size_t csz);

// ---------------------------------------------------------------- launchers
// (m3d_flex.hip; PH = Elastic or Thermal, T = float or double)
template <typename T, typename PH>
void launch_z(int mode, const Geo& g, const Ptr<T>& p, hipStream_t st);
template <typename T>
void launch_y(int dir, int which, unsigned cap, const Geo& g, const Ptr<T>& p, hipStream_t st);
template <typename T, typename PH>
void launch_xgreen(const Geo& g, const Ptr<T>& p, const T* prm, hipStream_t st);
template <typename T, typename PH>
void launch_xcheck(int which, const Geo& g, const Ptr<T>& p, hipStream_t st);

} // namespace flex
} // namespace m3d
