#pragma once
// spectral_expand.hpp -- one direction of expand (interpolate/fft.F90:832-927)
// in one pass, for gfx950.
//
// Doubling a line by zero-padding its spectrum gives, at the even fine points,
// the coarse values plus the Nyquist term once more (the reference keeps the
// coarse Nyquist coefficient whole, as a cosine of the fine grid, where the
// coarse transform holds half of it twice):
//   f(2n) = x(n) + (-1)^n X_{N/2} / N,
// and at the odd ones the line shifted by half a cell, where that cosine is 0:
//   f(2n+1) = 1/N sum_{|k| < N/2} X_k exp(i pi k / N) exp(2 pi i k n / N).
// So a transform of the coarse length and its inverse with the multiplier
// exp(i pi k / N) do, between one read of the line and one write of the fine
// one: 3 coarse-field units instead of the 9 of a forward transform, a padding
// kernel and an inverse transform of length 2N.  128^2 x 96, device arrays: 82 ->
// 31 us a call (both directions and the twiddles; latency and the memory-side
// cache bound it, 88 MB in 26 us).
#include "spectral_impl.hpp"

namespace mhd {

template <typename PL, int DIR, int B>
struct ExpandK {
    using Args = ExpandArgs;
    using TC = double;
    static constexpr int N = PL::N;
    static constexpr int NT = B * plan_tpt<PL>();
    static constexpr bool WAVE_LOCAL =
        NT <= 64 || (DIR == 0 && plan_tpt<PL>() <= 64 && 64 % plan_tpt<PL>() == 0);
    using F = RegFFT<TC, PL, WAVE_LOCAL>;
    static __device__ __forceinline__ void body(const ExpandArgs& a, uint3 bid, uint3 gdim)
    {
        using LN = Lines<PL, DIR, B>;
        constexpr int NB0 = F::NB0, NBL = F::NBL, R0 = F::R0, RL = F::RL;
        const Geom g = a.g;
        extern __shared__ __align__(16) unsigned char smem[];
        cpx<TC>* twl = reinterpret_cast<cpx<TC>*>(smem);
        F::stage_twiddles(twl, reinterpret_cast<const cpx<TC>*>(a.tw), threadIdx.x, NT);
        int t, j;
        LN::lane(threadIdx.x, t, j);
        cpx<TC>* lds = twl + F::TWN + t * F::SP;
        const long ngrp = LN::groups(g);
        // exp(i pi k / N) / N of this thread's modes (signed k), 0 at N/2
        cpx<TC> m[RL];
#pragma unroll
        for (int r = 0; r < RL; ++r) {
            const int kk = j + r * NBL;
            double s, c;
            sincospi((double)(kk < N / 2 ? kk : kk - N) / N, &s, &c);
            m[r] = kk == N / 2 ? cpx<TC>{0.0, 0.0} : cpx<TC>{c / N, s / N};
        }
        __syncthreads();
        auto fetch = [&](long grp, cpx<TC>* dst) {
            long ia, ib, st;
            int k;
            const bool ok = LN::base(g, grp, t, ia, ib, st, k);
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                dst[r] = {0.0, 0.0};
                if (ok && j < NB0) {
                    const long n = (long)(j + r * NB0) * st;
                    if constexpr (DIR != 0) dst[r] = ld_pair(a.in, ia + n);
                    else dst[r] = {a.in[ia + n], a.in[ib + n]};
                }
            }
        };
        cpx<TC> nxt[R0];
        long grp = bid.x;
        if (grp < ngrp) fetch(grp, nxt);
        for (; grp < ngrp; grp += gdim.x) {
            cpx<TC> x[R0], v[F::RMAX];
#pragma unroll
            for (int r = 0; r < R0; ++r) x[r] = v[r] = nxt[r];
            if (grp + gdim.x < ngrp) fetch(grp + gdim.x, nxt);
            F::forward(v, j, lds, twl);
            // the Nyquist coefficient to every thread, through the slot the
            // exchanges leave free
#pragma unroll
            for (int r = 0; r < RL; ++r)
                if (j < NBL && j + r * NBL == N / 2) lds[F::SP - 1] = v[r];
            F::sync();
            const cpx<TC> q = lds[F::SP - 1];
            F::sync();
#pragma unroll
            for (int r = 0; r < RL; ++r) v[r] = cmul(v[r], m[r]);
            F::inverse(v, j, lds, twl);
            long ia, ib, st;
            int k;
            const bool ok = LN::base(g, grp, t, ia, ib, st, k);
            if (ok && j < NB0) {
#pragma unroll
                for (int r = 0; r < R0; ++r) {
                    const int n = j + r * NB0;
                    const TC s = n % 2 ? -1.0 / N : 1.0 / N;
                    const cpx<TC> e = {x[r].x + s * q.x, x[r].y + s * q.y};
                    if constexpr (DIR == 0) {
                        // rows of 2N: elements 2n and 2n + 1
                        st_pair(a.out, 2 * (ia + n), e.x, v[r].x);
                        st_pair(a.out, 2 * (ib + n), e.y, v[r].y);
                    } else {
                        // rows 2n and 2n + 1 of a plane of 2N rows
                        const long col = ia - (long)k * g.nxy, base = 2 * (long)k * g.nxy + col;
                        st_pair(a.out, base + 2L * n * st, e.x, e.y);
                        st_pair(a.out, base + (2L * n + 1) * st, v[r].x, v[r].y);
                    }
                }
            }
        }
    }
};

template <typename PL, int DIR, int B>
static int launch_expand_one(const ExpandArgs& a, hipStream_t s)
{
    using K = ExpandK<PL, DIR, B>;
    constexpr size_t lds = spec_lds_bytes<double, PL, B>();
    auto kern = single_kernel<K>;
    static int lds_ok = lds <= 65536 ? 1 : 0;
    if (!lds_ok) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return -22;
        lds_ok = 1;
    }
    static int per_cu = 0;
    if (per_cu == 0) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, K::NT, lds) != hipSuccess || n < 1) n = 1;
        per_cu = n;
    }
    long grid = Lines<PL, DIR, B>::groups(a.g);
    const long resident = (long)per_cu * a.ncu;
    if (a.ncu > 0 && grid > resident) grid = resident;
    return mhd_launch<K>(dim3((unsigned)grid), dim3(K::NT), lds, s, a);
}

template <int N>
static int launch_expand_n(const ExpandArgs& a, hipStream_t s)
{
    using PL = FftPlan<N>;
    if (a.dir == 0) return launch_expand_one<PL, 0, spec_b<double, PL, 0>()>(a, s);
    constexpr int B = spec_b<double, PL, 1>();
    if (a.g.nx % (2 * B) == 0) return launch_expand_one<PL, 1, B>(a, s);
    return launch_expand_one<PL, 2, B>(a, s);
}

}  // namespace mhd
