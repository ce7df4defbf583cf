#pragma once
// spectral_mag.hpp -- the x transforms of the magnetic part fused with the
// spectral algebra of mag_deriv and bandj (src/magnetic.f90), for gfx950.
//
// On the double-halfcomplex layout d/dx and d/dy are index swaps, i -> nx - i
// and j -> ny - j.  Here a transform packs the rows j and ny - j of a plane
// (j = 0 and ny/2 alone) as A + i B, so its complex spectrum Z at mode k holds
// all four partners of a swap: d/dx is i kx Z, d/dy is i ky Z, and the
// derivatives cost registers instead of passes over HBM.
//
//   emf_x    forward: rows of E (physical x, halfcomplex y) -> the spectra
//            C = dEx/dy - dEy/dx, D = dEx/dx + dEy/dy and Ez
//   bandj_x  inverse: pol, tor and d pol/dz -> the rows of Bx, By, Bz, Jz,
//            dBz/dx and, in FP32, dBz/dy in physical x, halfcomplex y.  With `skip` the 2/3 band of
//            pol and tor is known to be zero: its modes are not read, its rows
//            neither transformed nor written (the y pass takes them as zero).
//
// Both are bound by HBM (about 4.5 TB/s of the fields they read and write at
// 256^2 x 160).  emf_x follows a y pass that forms u x B; with the x pass first,
// C and D took a kernel of their own: 135 + 94 + 66 -> 171 + 100 us FP64, 70 + 51
// + 36 -> 97 + 49 FP32 (x, y, C and D).  bandj_x reads 3 fields on the modes that
// are not zero (44 % of a plane) and writes 5 on the rows that are not (67 %),
// where a spectral kernel wrote 6 fields and the x pass read and wrote 6; dBz/dy
// comes from the y pass's spectrum (FP32: it is a sixth field): 163 + 184 + 226 -> 96
// + 175 us FP64, 105 + 79 + 98 -> 72 + 86 FP32 (spectral, x, y).
#include "spectral_impl.hpp"

namespace mhd {

// plan with the smaller radix last: the spectra of an item live in registers
// as the last radix's points
template <int N>
struct MagPlan {
    using type = FftPlan<N>;
};
template <> struct MagPlan<32> { using type = Plan<32, 8, 4>; };
template <> struct MagPlan<128> { using type = Plan<128, 8, 4, 4>; };
template <> struct MagPlan<512> { using type = Plan<512, 8, 4, 4, 4>; };

// the row pairs of a launch: items (plane k, row p), p < np
struct RowPair {
    long a, b;     // element 0 of the rows p and ny - p
    int k, p;
    bool ok, two;  // within the launch; row ny - p is another row
};
__device__ __forceinline__ RowPair row_pair(const Geom& g, int np, long item)
{
    RowPair R;
    const long total = (long)g.nz * np;
    R.ok = item < total;
    const long i = R.ok ? item : total - 1;
    R.k = (int)(i / np);
    R.p = (int)(i - (long)R.k * np);
    R.two = R.p != 0 && 2 * R.p != g.ny;
    R.a = (long)R.k * g.nxy + (long)R.p * g.nx;
    R.b = R.two ? (long)R.k * g.nxy + (long)(g.ny - R.p) * g.nx : R.a;
    return R;
}

template <typename TC, typename PL, int B>
struct MagBase {
    using Args = MagSpecArgs;
    static constexpr int N = PL::N;
    static constexpr int NT = B * plan_tpt<PL>();
    static constexpr bool WAVE_LOCAL = NT <= 64 || (plan_tpt<PL>() <= 64 && 64 % plan_tpt<PL>() == 0);
    using F = RegFFT<TC, PL, WAVE_LOCAL>;
    static constexpr int NB0 = F::NB0, NBL = F::NBL, R0 = F::R0, RL = F::RL;
    static constexpr bool full0 = NB0 == plan_tpt<PL>();
    // signed wavenumber and -wavenumber^2 of mode kk
    static __device__ __forceinline__ double kx1(int kk, double cx)
    {
        if (kk == 0 || kk == N / 2) return 0.0;
        return kk < N / 2 ? (double)kk * cx : -((double)(N - kk) * cx);
    }
    static __device__ __forceinline__ double k2(int kk, double cx, int p, double cy)
    {
        const int m = kk <= N / 2 ? kk : N - kk;
        return -((double)m * (double)m * cx * cx) - ((double)p * (double)p * cy * cy);
    }
};

template <typename TC, typename PL, int B>
struct EmfXK : MagBase<TC, PL, B> {
    using M = MagBase<TC, PL, B>;
    using F = typename M::F;
    using Args = MagSpecArgs;
    static constexpr int NT = M::NT;
    static __device__ __forceinline__ void body(const MagSpecArgs& a, uint3 bid, uint3 gdim)
    {
        constexpr int R0 = M::R0, RL = M::RL, NB0 = M::NB0, NBL = M::NBL;
        const Geom g = a.g;
        extern __shared__ __align__(16) unsigned char smem[];
        cpx<TC>* twl = reinterpret_cast<cpx<TC>*>(smem);
        F::stage_twiddles(twl, reinterpret_cast<const cpx<TC>*>(a.tw), threadIdx.x, NT);
        const int j_ = threadIdx.x % plan_tpt<PL>(), t = threadIdx.x / plan_tpt<PL>();
        cpx<TC>* lds = twl + F::TWN + t * F::SP;
        const int np = g.ny / 2 + 1;
        const long ngrp = ((long)g.nz * np + B - 1) / B;
        __syncthreads();
        auto load = [&](const void* p, const RowPair& R, int j, cpx<TC>* dst) {
            const TC* __restrict__ s = (const TC*)p;
            const int j0 = M::full0 || j < NB0 ? j : 0;
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                dst[r].x = s[R.a + j0 + r * NB0];
                dst[r].y = s[R.b + j0 + r * NB0];
            }
        };
        long grp = bid.x;
        if (grp >= ngrp) return;
        cpx<TC> fx[R0], fy[R0], fz[R0];
        RowPair C = row_pair(g, np, grp * B + t);
        load(a.ex, C, j_, fx);
        load(a.ey, C, j_, fy);
        load(a.ez, C, j_, fz);
        for (;;) {
            const int j = F::own(j_);
            const RowPair R = C;
            grp += gdim.x;
            const bool more = grp < ngrp;
            if (more) C = row_pair(g, np, grp * B + t);
            auto take = [&](const cpx<TC>* f, cpx<TC>* v) {
#pragma unroll
                for (int r = 0; r < R0; ++r) v[r] = {f[r].x, R.two ? f[r].y : (TC)0};
            };
            cpx<TC> v[F::RMAX], x[RL], c[RL];
            take(fx, v);
            if (more) load(a.ex, C, j, fx);
            F::forward(v, j, lds, twl);
#pragma unroll
            for (int r = 0; r < RL; ++r) x[r] = v[r];
            take(fy, v);
            if (more) load(a.ey, C, j, fy);
            F::forward(v, j, lds, twl);
            if (R.ok && R.p == 0 && j == 0) {
                // the plane means' numerators, where mean_emf reads them
                ((TC*)a.ex)[R.a] = x[0].x;
                ((TC*)a.ey)[R.a] = v[0].x;
            }
            const double ky = R.two ? (double)R.p * a.cy : 0.0;
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                const double kx = M::kx1(j + r * NBL, a.cx);
                const double xr = (double)x[r].x, xi = (double)x[r].y, yr = (double)v[r].x, yi = (double)v[r].y;
                c[r] = {(TC)(kx * yi - ky * xi), (TC)(ky * xr - kx * yr)};
                x[r] = {(TC)(-kx * xi - ky * yi), (TC)(kx * xr + ky * yr)};
            }
            for (int o = 0; o < 3; ++o) {
                if (o == 2) {
                    take(fz, v);
                    if (more) load(a.ez, C, j, fz);
                    F::forward(v, j, lds, twl);
                } else {
#pragma unroll
                    for (int r = 0; r < RL; ++r) v[r] = o == 0 ? c[r] : x[r];
                }
                store(v, j, lds, R, (TC*)(o == 0 ? a.cc : o == 1 ? a.d : a.ez));
            }
            if (!more) break;
        }
    }
    // packed spectrum -> the two rows' halfcomplex lines
    static __device__ __forceinline__ void store(const cpx<TC>* v, int j, cpx<TC>* lds, const RowPair& R,
                                                 TC* __restrict__ out)
    {
        constexpr int N = M::N, R0 = M::R0, RL = M::RL, NB0 = M::NB0, NBL = M::NBL;
        if (j < NBL) {
#pragma unroll
            for (int r = 0; r < RL; ++r) lds[F::pad(j + r * NBL)] = v[r];
        }
        F::sync();
        if (R.ok && j < NB0) {
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                const int n = j + r * NB0;
                const int kk = (n <= N / 2) ? n : N - n;
                const cpx<TC> zk = lds[F::pad(kk)];
                const cpx<TC> zn = lds[F::pad((N - kk) % N)];
                TC p, q;
                if (n <= N / 2) { p = (TC)0.5 * (zk.x + zn.x); q = (TC)0.5 * (zk.y + zn.y); }
                else { p = (TC)0.5 * (zk.y - zn.y); q = (TC)0.5 * (zn.x - zk.x); }
                out[R.a + n] = p;
                if (R.two) out[R.b + n] = q;
            }
        }
        F::sync();
    }
};

template <typename TC, typename PL, int B>
struct BandjXK : MagBase<TC, PL, B> {
    using M = MagBase<TC, PL, B>;
    using F = typename M::F;
    using Args = MagSpecArgs;
    static constexpr int NT = M::NT;
    // halfcomplex elements of the two rows at this thread's modes
    template <typename T>
    struct Raw {
        T ar[M::RL], ai[M::RL], br[M::RL], bi[M::RL];
    };
    static __device__ __forceinline__ void body(const MagSpecArgs& a, uint3 bid, uint3 gdim)
    {
        constexpr int N = M::N, R0 = M::R0, RL = M::RL, NB0 = M::NB0, NBL = M::NBL;
        const Geom g = a.g;
        extern __shared__ __align__(16) unsigned char smem[];
        cpx<TC>* twl = reinterpret_cast<cpx<TC>*>(smem);
        F::stage_twiddles(twl, reinterpret_cast<const cpx<TC>*>(a.tw), threadIdx.x, NT);
        const int j_ = threadIdx.x % plan_tpt<PL>(), t = threadIdx.x / plan_tpt<PL>();
        cpx<TC>* lds = twl + F::TWN + t * F::SP;
        const int np = a.skip ? g.ny / 2 - a.icuty : g.ny / 2 + 1;
        const int mlim = a.skip ? N / 2 - a.icutx : N;   // modes of the rows that are not zero
        const long ngrp = ((long)g.nz * np + B - 1) / B;
        __syncthreads();
        auto load = [&](const auto* __restrict__ s, const RowPair& R, int j, auto& w) {
            const auto* __restrict__ sa = s + R.a;
            const auto* __restrict__ sb = s + R.b;
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                const int kk = j + r * NBL;
                const int m0 = kk <= N / 2 ? kk : N - kk;
                const int m = m0 >= 0 && m0 < mlim ? m0 : 0;   // zero modes: any element, dropped by pack
                const int im = m == 0 ? 0 : N - m;
                w.ar[r] = sa[m];
                w.ai[r] = sa[im];
                w.br[r] = sb[m];
                w.bi[r] = sb[im];
            }
        };
        long grp = bid.x;
        if (grp >= ngrp) return;
        RowPair C = row_pair(g, np, grp * B + t);
        Raw<TC> wz;
        Raw<double> wt, wp;
        load((const TC*)a.polz, C, j_, wz);
        load(a.tor, C, j_, wt);
        for (;;) {
            const int j = F::own(j_);
            const RowPair R = C;
            // pol's rows fly during the first three outputs, the next item's
            // other rows during the last two
            load(a.pol, R, j, wp);
            const double ky = R.two ? (double)R.p * a.cy : 0.0;
            auto pack = [&](const auto& w, int r) -> cpx<double> {
                const int kk = j + r * NBL;
                if ((kk <= N / 2 ? kk : N - kk) >= mlim) return {0.0, 0.0};
                const double ar = (double)w.ar[r], br = R.two ? (double)w.br[r] : 0.0;
                if (kk == 0 || kk == N / 2) return {ar, br};
                const double s = kk < N / 2 ? 1.0 : -1.0;
                return {ar - s * (R.two ? (double)w.bi[r] : 0.0), s * (double)w.ai[r] + br};
            };
            auto finish = [&](cpx<TC>* v, void* o) {
                F::inverse(v, j, lds, twl);
                if (R.ok && (M::full0 || j < NB0)) {
                    TC* __restrict__ out = (TC*)o;
#pragma unroll
                    for (int r = 0; r < R0; ++r) {
                        const int n = j + r * NB0;
                        out[R.a + n] = v[r].x * (TC)(1.0 / N);
                        if (R.two) out[R.b + n] = v[r].y * (TC)(1.0 / N);
                    }
                }
            };
            cpx<double> z[RL], q[RL];
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                z[r] = pack(wz, r);
                q[r] = pack(wt, r);
            }
            for (int o = 0; o < 3; ++o) {
                cpx<TC> v[F::RMAX];
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const int kk = j + r * NBL;
                    if (o < 2) {
                        // i kx z + i ky q, or i ky z - i kx q
                        const double kx = M::kx1(kk, a.cx);
                        const double ca = o == 0 ? kx : ky, cb = o == 0 ? ky : -kx;
                        v[r] = {(TC)(-(ca * z[r].y + cb * q[r].y)), (TC)(ca * z[r].x + cb * q[r].x)};
                    } else {
                        const double k2 = M::k2(kk, a.cx, R.p, a.cy);
                        v[r] = {(TC)(-1.0 * q[r].x * k2), (TC)(-1.0 * q[r].y * k2)};
                    }
                }
                finish(v, a.out[o]);
            }
            grp += gdim.x;
            const bool more = grp < ngrp;
            cpx<double> b[RL];
#pragma unroll
            for (int r = 0; r < RL; ++r) {
                const double k2 = M::k2(j + r * NBL, a.cx, R.p, a.cy);
                const cpx<double> p = pack(wp, r);
                b[r] = {-1.0 * p.x * k2, -1.0 * p.y * k2};
            }
            if (more) {
                C = row_pair(g, np, grp * B + t);
                load((const TC*)a.polz, C, j, wz);
                load(a.tor, C, j, wt);
            }
            for (int o = 3; o < (sizeof(TC) == 4 ? 6 : 5); ++o) {
                cpx<TC> v[F::RMAX];
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const double kx = M::kx1(j + r * NBL, a.cx);
                    const double kd = o == 4 ? kx : ky;
                    if (o == 3) v[r] = {(TC)b[r].x, (TC)b[r].y};
                    else v[r] = {(TC)(-kd * b[r].y), (TC)(kd * b[r].x)};
                }
                finish(v, a.out[o]);
            }
            if (!more) break;
        }
    }
};

template <typename K>
static int launch_mag_x(const MagSpecArgs& a, size_t lds, int np, int B, hipStream_t s)
{
    static_assert(K::NT <= 1024, "workgroup too large");
    auto kern = single_kernel<K>;
    static int per_cu = 0;
    if (per_cu == 0) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, K::NT, lds) != hipSuccess || n < 1) n = 1;
        per_cu = n;
    }
    long grid = ((long)a.g.nz * np + B - 1) / B;
    const long resident = (long)per_cu * a.ncu;
    if (a.ncu > 0 && grid > resident) grid = resident;
    return mhd_launch<K>(dim3((unsigned)grid), dim3(K::NT), lds, s, a);
}

// which: 0 emf_x, 1 bandj_x
template <typename TC, int N>
static int launch_mag_n(int which, const MagSpecArgs& a, hipStream_t s)
{
    using PL = typename MagPlan<N>::type;
    constexpr int B = spec_b<TC, PL, 0>();
    constexpr size_t lds = spec_lds_bytes<TC, PL, B>();
    static_assert(lds <= 65536, "row transforms fit in 64 KB of LDS");
    if (which == 0) return launch_mag_x<EmfXK<TC, PL, B>>(a, lds, a.g.ny / 2 + 1, B, s);
    return launch_mag_x<BandjXK<TC, PL, B>>(a, lds, a.skip ? a.g.ny / 2 - a.icuty : a.g.ny / 2 + 1, B, s);
}

}  // namespace mhd
