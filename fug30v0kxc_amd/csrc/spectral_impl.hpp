#pragma once
// spectral_impl.hpp -- horizontal transform kernels for gfx950 (template
// definitions; spectral_g*.hip instantiate them per transform length).
//
// One kernel template covers the four horizontal operator families of the
// reference (src/fft.F90): spectral derivatives (d1bydx/d1bydy/d2bydx/d2bydy),
// the 2/3 dealias, and the two halves of the 2-D real transforms
// (forwardfft: r2hc per line; inversefft: hc2r per line).
//
// A workgroup owns B transforms of one job; each transform packs two real
// lines (rows for dir=x, adjacent columns for dir=y) as a + i b.  Because
// every operator here multiplies each mode by a Hermitian-symmetric factor
// m(N-k) = conj(m(k)), one complex FFT, one multiply and one inverse FFT
// return the operator applied to a in the real part and to b in the
// imaginary part; real<->halfcomplex conversions separate / merge the pair
// through one extra LDS round trip.  Each line is read once from HBM and each
// output written once, straight from registers (see fft_reg.hpp).
//
// Rows (dir=x): the TPT threads of a transform read TPT consecutive elements
// of each of its two rows per load.  Columns (dir=y): consecutive threads
// belong to consecutive column pairs, so one load reads 2*B adjacent columns
// of one row (2*B*sizeof(T) bytes).
#include <type_traits>

#include "fft_reg.hpp"
#include "launch.hpp"
#include "spectral.hpp"

namespace mhd {

// Adjacent pairs (i, i+1) with i even: the two columns of a y transform.
// One 8-byte (float) or 16-byte (double) access instead of two.
template <typename TC>
using vec2_t = typename std::conditional<sizeof(TC) == 4, float2, double2>::type;
template <typename TC>
__device__ __forceinline__ cpx<TC> ld_pair(const TC* __restrict__ p, long i)
{
    const vec2_t<TC> v = *reinterpret_cast<const vec2_t<TC>*>(p + i);
    return {(TC)v.x, (TC)v.y};
}
template <typename TC>
__device__ __forceinline__ void st_pair(TC* __restrict__ p, long i, TC a, TC b)
{
    vec2_t<TC> v;
    v.x = a;
    v.y = b;
    *reinterpret_cast<vec2_t<TC>*>(p + i) = v;
}
// derivative outputs are read back only by later kernels, after the step has
// streamed other fields through the caches: stored non-temporally
template <typename TC>
__device__ __forceinline__ void st_pair_nt(TC* __restrict__ p, long i, TC a, TC b)
{
    using v2 = TC __attribute__((ext_vector_type(2)));
    v2 v;
    v.x = a;
    v.y = b;
    __builtin_nontemporal_store(v, reinterpret_cast<v2*>(p + i));
}
template <typename TC>
__device__ __forceinline__ void st_nt(TC* __restrict__ p, long i, TC a)
{
    __builtin_nontemporal_store(a, p + i);
}

// Input loaders, fixed at compile time per launch; inputs have the compute type.
template <typename TC, int LOP>
struct Loader {
    const TC* __restrict__ a;
    const TC* __restrict__ b;
    const TC* __restrict__ c;
    const TC* __restrict__ d;
    TC m0, m1, m2, m3;   // per-plane means of the factors (0 when absent)
    const TC* __restrict__ jj;   // LD_CROSS: current density component, or null
    TC jc;                       // its per-plane coefficient
    __device__ __forceinline__ Loader(const SpecJob& J, int k)
    {
        a = (const TC*)J.in[0];
        b = (const TC*)J.in[1];
        c = (const TC*)J.in[2];
        d = (const TC*)J.in[3];
        m0 = m1 = m2 = m3 = (TC)0;
        jj = nullptr;
        jc = (TC)0;
        if constexpr (LOP == LD_CROSS) {
            if (J.jin) {
                jj = (const TC*)J.jin;
                jc = (TC)J.jcoef[k];
            }
            if (J.mean[0]) m0 = (TC)J.mean[0][k];
            if (J.mean[1]) m1 = (TC)J.mean[1][k];
            if (J.mean[2]) m2 = (TC)J.mean[2][k];
            if (J.mean[3]) m3 = (TC)J.mean[3][k];
        }
    }
    // elements i and i+1 (i even)
    __device__ __forceinline__ cpx<TC> pair(long i) const
    {
        if constexpr (LOP == LD_PLAIN) return ld_pair(a, i);
        else return cross_pair(ld_pair(a, i), ld_pair(b, i), ld_pair(c, i), ld_pair(d, i), i);
    }
    // LD_CROSS from factor values already loaded (x = in0, y = in1, z = in2,
    // w = in3 at element i), the extra term loaded here
    __device__ __forceinline__ TC cross(TC x, TC y, TC z, TC w, long i) const
    {
        TC r = x * y - z * w + (x * m1 + m0 * y) - (z * m3 + m2 * w);
        if (jj) r = r - jc * jj[i];
        return r;
    }
    __device__ __forceinline__ cpx<TC> cross_pair(cpx<TC> x, cpx<TC> y, cpx<TC> z, cpx<TC> w, long i) const
    {
        cpx<TC> r = {x.x * y.x - z.x * w.x + (x.x * m1 + m0 * y.x) - (z.x * m3 + m2 * w.x),
                     x.y * y.y - z.y * w.y + (x.y * m1 + m0 * y.y) - (z.y * m3 + m2 * w.y)};
        if (jj) {
            const cpx<TC> q = ld_pair(jj, i);
            r.x = r.x - jc * q.x;
            r.y = r.y - jc * q.y;
        }
        return r;
    }
    __device__ __forceinline__ TC operator()(long i) const
    {
        if constexpr (LOP == LD_PLAIN) return a[i];
        else return cross(a[i], b[i], c[i], d[i], i);
    }
};

// A job's auxiliary line (SpecJob::aux) of one plane: the Maxwell-stress load
// from field components x = b_ai, y = b_aj, z = b_al (l the third; AUX_MAXW
// only) and the further term's q, with the components' per-plane means.
// (s*x)*y is the reference's product; the mean terms drop its constant.
template <typename TC>
struct AuxLoad {
    TC s, mi, mj, ml, xc;
    int op, ai, aj, al;
    bool xin;
    __device__ __forceinline__ AuxLoad(const SpecLaunch& L, const SpecJob& J, int k)
    {
        op = J.aux;
        ai = op ? J.ai : 0;
        aj = op == AUX_PROD ? J.aj : (ai == 0 ? 1 : 0);
        al = 3 - ai - aj;
        s = (TC)J.ascale;
        xin = sizeof(TC) == 8 && op && J.xin;
        xc = (TC)J.xcoef;
        mi = ml = mj = (TC)0;
        if (!op) return;
        mi = L.bmean[ai] ? (TC)L.bmean[ai][k] : (TC)0;
        mj = L.bmean[aj] ? (TC)L.bmean[aj][k] : (TC)0;
        ml = L.bmean[al] ? (TC)L.bmean[al][k] : (TC)0;
    }
    // from the three components of an element
    __device__ __forceinline__ TC pick(TC b0, TC b1, TC b2, TC q) const
    {
        return one(ai == 0 ? b0 : ai == 1 ? b1 : b2, aj == 0 ? b0 : aj == 1 ? b1 : b2, al == 0 ? b0 : al == 1 ? b1 : b2,
                   q);
    }
    __device__ __forceinline__ TC one(TC x, TC y, TC z, TC q) const
    {
        TC v;
        if (op == AUX_PROD) v = (s * x) * y + s * (x * mj + mi * y);
        else v = s * x * x - s * y * y - s * z * z + (TC)2 * s * (mi * x - mj * y - ml * z);
        return xin ? v + xc * q : v;
    }
};

// spectral multiplier of mode k (full complex spectrum index), folded with
// 1/N.  The wavenumbers are those of src/fft.F90:196-221: mode m = min(k,N-k)
// has akx1 = m*cx and akx2 = -(m*m*cx*cx), Nyquist included in akx2 only.
template <typename TC, int N>
__device__ __forceinline__ cpx<TC> apply_mul(int kind, cpx<TC> z, int k, double cx, int icut,
                                              const double* mc)
{
    constexpr double invN = 1.0 / N;
    const int m = (k < N - k) ? k : N - k;
    if (kind == MUL_D1) {
        if (k == 0 || k == N / 2) return {(TC)0, (TC)0};
        const TC a = (TC)(((double)m * cx) * invN);
        // +i*a for k < N/2; the negative frequency N-k carries -i*a
        if (k < N / 2) return {-a * z.y, a * z.x};
        return {a * z.y, -a * z.x};
    } else if (kind == MUL_D2 || kind == MUL_D2C) {
        double f = -((double)m * (double)m * cx * cx);
        if (kind == MUL_D2C) f *= (k == N / 2) ? mc[0] : mc[0] + mc[1];
        const TC a = (TC)(f * invN);
        return {a * z.x, a * z.y};
    } else {
        if (m < N / 2 - icut) return {z.x * (TC)invN, z.y * (TC)invN};
        return {(TC)0, (TC)0};
    }
}

// DIR: 0 along x, 1 along y, 2 along y where B does not divide the column pairs
// of a row: the last group of each row is partly filled.  (Those boxes ran groups
// of one pair, workgroups of 15 threads and 16-byte row segments at 30 x 30: the
// y passes of a step, second derivatives, EMF and inverse, went from 17.4, 9.3 and
// 10.4 us to 11.9, 8.1 and 8.2 at 60 planes FP64.  A kernel of its own, so that
// full groups carry no mask.)
template <typename PL, int DIR, int B>
struct Lines {
    static constexpr int N = PL::N;
    static constexpr int TPT = plan_tpt<PL>();
    // (transform t, butterfly j) of this thread
    static __device__ __forceinline__ void lane(int tid, int& t, int& j)
    {
        if constexpr (DIR == 0) { j = tid % TPT; t = tid / TPT; }
        else { t = tid % B; j = tid / B; }
    }
    // line groups per job: B complex lines each
    static __host__ __device__ __forceinline__ long groups(const Geom& g)
    {
        if constexpr (DIR == 0) return ((long)g.nz * g.ny / 2 + B - 1) / B;
        else return (long)g.nz * row_groups(g);
    }
    static __host__ __device__ __forceinline__ int row_groups(const Geom& g)
    {
        return DIR == 2 ? (g.nx / 2 + B - 1) / B : g.nx / (2 * B);
    }
    // global index of element 0 of the transform's lines a and b in group grp
    static __device__ __forceinline__ bool base(const Geom& g, long grp, int t, long& ia, long& ib, long& step,
                                                int& k)
    {
        if constexpr (DIR == 0) {
            const long cl = grp * B + t;
            const long row = 2 * cl;
            k = (int)(row / g.ny);
            ia = row * N;
            ib = ia + N;
            step = 1;
            return cl < (long)g.nz * g.ny / 2;
        } else {
            const int tpp = row_groups(g);
            k = (int)(grp / tpp);
            const int x0 = (int)(grp - (long)k * tpp) * 2 * B;
            ia = (long)k * g.nxy + x0 + 2 * t;
            ib = ia + 1;
            step = g.nx;
            return DIR == 1 || x0 + 2 * t < g.nx;
        }
    }
};

// Persistent, software-pipelined kernel: workgroup w handles the items
// (job, line group) w, w + gridDim.x, ...  The pass-0 inputs of the next item
// are loaded into registers before the current item is transformed, and the
// transform touches only registers and LDS (twiddles are staged in LDS), so
// the loads of item i+1 are in flight while item i is computed and stored.
//
// SM_DERIV2 runs body_deriv2 instead: an item is every job of one line group
// (or, with L.split, one job of one group).
// LOP = LD_CROSS3 (SM_R2HC, three jobs forming one cross product) runs
// body_cross3 instead: an item is one line group, whose six factor lines are
// loaded once and combined into the three jobs' inputs.
template <typename TC, typename PL, int DIR, int B, int MODE, int LOP>
struct SpecK {
    using Args = SpecLaunch;
    static constexpr int NT = B * plan_tpt<PL>();
    // each transform within one wavefront: rows with at most 64 butterflies
    // per transform, or a workgroup of one wave
    static constexpr bool WAVE_LOCAL =
        NT <= 64 || (DIR == 0 && plan_tpt<PL>() <= 64 && 64 % plan_tpt<PL>() == 0);
    using F = RegFFT<TC, PL, WAVE_LOCAL>;
    static __device__ __forceinline__ void body(const SpecLaunch& L, uint3 bid, uint3 gdim)
    {
        if constexpr (LOP == LD_CROSS3) body_cross3(L, bid, gdim);
        else if constexpr (MODE == SM_DERIV2) body_deriv2(L, bid, gdim);
        else body_jobs(L, bid, gdim);
    }
    static __device__ __forceinline__ void body_deriv2(const SpecLaunch& L, uint3 bid, uint3 gdim);
    static __device__ __forceinline__ void body_jobs(const SpecLaunch& L, uint3 bid, uint3 gdim);
    static __device__ __forceinline__ void body_cross3(const SpecLaunch& L, uint3 bid, uint3 gdim);
    // Column groups narrower than a 128-byte line (y, 2 B sizeof(TC) < 128
    // bytes) share each line with the next group.  Within every 16 items, item
    // c (< 8) takes group 2c and item c + 8 group 2c + 1: workgroups w and w + 8
    // run on the same XCD (they are dealt round-robin over 8) at the same time,
    // so a line is fetched once.  Identity otherwise.
    static __device__ __forceinline__ long paired_group(long item, long G, long ngrp)
    {
        constexpr bool half_line = DIR != 0 && 2 * B * (int)sizeof(TC) < 128;
        if constexpr (half_line) {
            if (G % 16 == 0 && ngrp % 16 == 0) {
                const long c = item & 15;
                return item - c + (c < 8 ? 2 * c : 2 * (c - 8) + 1);
            }
        }
        return item;
    }
    // forward spectrum in v -> the two halfcomplex lines of the pair, stored
    static __device__ __forceinline__ void r2hc_store(cpx<TC>* v, int j, cpx<TC>* lds, bool ok, TC* __restrict__ out0,
                                                      long ia, long ib, long st);
};

template <typename TC, typename PL, int DIR, int B, int MODE, int LOP>
__device__ __forceinline__ void SpecK<TC, PL, DIR, B, MODE, LOP>::r2hc_store(cpx<TC>* v, int j, cpx<TC>* lds, bool ok,
                                                                             TC* __restrict__ out0, long ia, long ib,
                                                                             long st)
{
    constexpr int N = PL::N;
    constexpr int NB0 = F::NB0, NBL = F::NBL, R0 = F::R0, RL = F::RL;
    // spectrum -> LDS, then separate the pair into two halfcomplex lines
    if (j < NBL) {
#pragma unroll
        for (int r = 0; r < RL; ++r) lds[F::pad(j + r * NBL)] = v[r];
    }
    F::sync();
    if (ok && j < NB0) {
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const int n = j + r * NB0;
            const int kk = (n <= N / 2) ? n : N - n;
            const cpx<TC> zk = lds[F::pad(kk)];
            const cpx<TC> zn = lds[F::pad((N - kk) % N)];
            TC a, b;
            if (n <= N / 2) { a = (TC)0.5 * (zk.x + zn.x); b = (TC)0.5 * (zk.y + zn.y); }
            else { a = (TC)0.5 * (zk.y - zn.y); b = (TC)0.5 * (zn.x - zk.x); }
            if constexpr (DIR != 0) st_pair(out0, ia + n * st, a, b);
            else {
                out0[ia + n * st] = a;
                out0[ib + n * st] = b;
            }
        }
    }
    F::sync();
}

template <typename TC, typename PL, int DIR, int B, int MODE, int LOP>
__device__ __forceinline__ void SpecK<TC, PL, DIR, B, MODE, LOP>::body_cross3(const SpecLaunch& L, uint3 bid,
                                                                              uint3 gdim)
{
    using LN = Lines<PL, DIR, B>;
    constexpr int NB0 = F::NB0, R0 = F::R0;
    const Geom g = L.g;
    extern __shared__ __align__(16) unsigned char smem[];
    cpx<TC>* twl = reinterpret_cast<cpx<TC>*>(smem);
    const cpx<TC>* __restrict__ twg = reinterpret_cast<const cpx<TC>*>(L.tw);
    F::stage_twiddles(twl, twg, threadIdx.x, NT);
    int t, j;
    LN::lane(threadIdx.x, t, j);
    cpx<TC>* lds = twl + F::TWN + t * F::SP;
    const long ngrp = LN::groups(g);
    const long G = gdim.x;
    // the factors: job q loads {a_{q+1}, b_{q+2}, a_{q+2}, b_{q+1}}
    const TC* __restrict__ a0 = (const TC*)L.job[2].in[0];
    const TC* __restrict__ a1 = (const TC*)L.job[0].in[0];
    const TC* __restrict__ a2 = (const TC*)L.job[1].in[0];
    const TC* __restrict__ b0 = (const TC*)L.job[1].in[1];
    const TC* __restrict__ b1 = (const TC*)L.job[2].in[1];
    const TC* __restrict__ b2 = (const TC*)L.job[0].in[1];
    __syncthreads();

    // the three jobs' pass-0 inputs of line group grp
    auto fetch = [&](long grp, cpx<TC> (*dst)[R0]) {
        long ia, ib, st;
        int k;
        const bool ok = LN::base(g, grp, t, ia, ib, st, k);
        const Loader<TC, LD_CROSS> l0(L.job[0], ok ? k : 0), l1(L.job[1], ok ? k : 0), l2(L.job[2], ok ? k : 0);
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const int n = j + r * NB0;
            dst[0][r] = dst[1][r] = dst[2][r] = {(TC)0, (TC)0};
            if (ok && j < NB0) {
                const long i = ia + n * st;
                const cpx<TC> x0 = ld_pair(a0, i), x1 = ld_pair(a1, i), x2 = ld_pair(a2, i);
                const cpx<TC> y0 = ld_pair(b0, i), y1 = ld_pair(b1, i), y2 = ld_pair(b2, i);
                dst[0][r] = l0.cross_pair(x1, y2, x2, y1, i);
                dst[1][r] = l1.cross_pair(x2, y0, x0, y2, i);
                dst[2][r] = l2.cross_pair(x0, y1, x1, y0, i);
            }
        }
    };

    cpx<TC> nxt[3][R0];
    long item = bid.x;
    if (item < ngrp) fetch(paired_group(item, G, ngrp), nxt);
    for (; item < ngrp; item += G) {
        const long grp = paired_group(item, G, ngrp);
        cpx<TC> cur[3][R0];
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int r = 0; r < R0; ++r) cur[q][r] = nxt[q][r];
        long ia, ib, st;
        int k;
        const bool ok = LN::base(g, grp, t, ia, ib, st, k);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            // the next group's loads fly during the last job's transform
            if (q == 2 && item + G < ngrp) fetch(paired_group(item + G, G, ngrp), nxt);
            cpx<TC> v[F::RMAX];
#pragma unroll
            for (int r = 0; r < R0; ++r) v[r] = cur[q][r];
            F::forward(v, j, lds, twl);
            r2hc_store(v, j, lds, ok, (TC*)L.job[q].out[0], ia, ib, st);
        }
    }
}

// First and second derivatives (SM_DERIV2), with the auxiliary lines of
// SpecJob::aux.  An item is one line group: its field components b0, b1, b2 are
// loaded once, then its jobs run back to back, each with its line (and extra
// term) loaded during the job before it, and the next item's components during
// the jobs without an auxiliary line, which come last.  With L.split an item is
// one job of one line group (boxes with too few line groups to fill the device).
//
// What bounds it: HBM through the few waves its registers allow (FP64 210: two
// per SIMD), LDS busy 35-46 % and the VALU 23-31 % of the time.  The auxiliary
// lines replace a launch of their own per direction (three first derivatives
// from one load of b) and, in y FP64, two single-output jobs: at 256^2 x 160 FP64 x
// 241 + 104 -> 318 us, y 324 + 151 -> 449, and hydro_col reads 18 arrays for 26 (855
// -> 723 us).  FP32, whose stresses stay outputs of their own (AuxOp): 132 + 72 ->
// 179 and 209 + 91 -> 296.  Reloading b per job (three waves per SIMD) measured
// slower: x 336, y 460 us FP64.
template <typename TC, typename PL, int DIR, int B, int MODE, int LOP>
__device__ __forceinline__ void SpecK<TC, PL, DIR, B, MODE, LOP>::body_deriv2(const SpecLaunch& L, uint3 bid,
                                                                              uint3 gdim)
{
    constexpr int N = PL::N;
    using LN = Lines<PL, DIR, B>;
    constexpr int NB0 = F::NB0, NBL = F::NBL, R0 = F::R0, RL = F::RL;
    const Geom g = L.g;
    extern __shared__ __align__(16) unsigned char smem[];
    cpx<TC>* twl = reinterpret_cast<cpx<TC>*>(smem);
    const cpx<TC>* __restrict__ twg = reinterpret_cast<const cpx<TC>*>(L.tw);
    F::stage_twiddles(twl, twg, threadIdx.x, NT);
    int t, j;
    LN::lane(threadIdx.x, t, j);
    cpx<TC>* lds = twl + F::TWN + t * F::SP;
    const long ngrp = LN::groups(g);
    const long G = gdim.x;
    const int nj = L.njobs;
    const bool split = L.split != 0;
    const long nitems = split ? ngrp * nj : ngrp;
    const double cx = L.cx;
    const int icut = L.icut;
    __syncthreads();

    // first job and line group of an item
    auto decode = [&](long item, int& q0, long& grp) {
        q0 = split ? (int)(item / ngrp) : 0;
        grp = paired_group(item - (long)q0 * ngrp, G, ngrp);
    };
    auto load = [&](const TC* __restrict__ p, long grp, cpx<TC>* dst) {
        long ia, ib, st;
        int k;
        const bool ok = LN::base(g, grp, t, ia, ib, st, k);
#pragma unroll
        for (int r = 0; r < R0; ++r) {
            const long n = (long)(j + r * NB0) * st;
            dst[r] = {(TC)0, (TC)0};
            if (ok && j < NB0) {
                if constexpr (DIR != 0) dst[r] = ld_pair(p, ia + n);
                else dst[r] = {p[ia + n], p[ib + n]};
            }
        }
    };
    constexpr bool SUM = sizeof(TC) == 8;   // AuxOp
    cpx<TC> f[R0], x[SUM ? R0 : 1], b0[R0], b1[R0], b2[R0];
    auto load_job = [&](int q, long grp) {
        load((const TC*)L.job[q].in[0], grp, f);
        if constexpr (SUM)
            if (L.job[q].xin) load((const TC*)L.job[q].xin, grp, x);
    };
    auto load_b = [&](long grp) {
        load((const TC*)L.bf[0], grp, b0);
        load((const TC*)L.bf[1], grp, b1);
        load((const TC*)L.bf[2], grp, b2);
    };

    long item = bid.x;
    int q0 = 0;
    long grp = 0;
    if (item < nitems) {
        decode(item, q0, grp);
        load_job(q0, grp);
        if (L.job[q0].aux) load_b(grp);
    }
    while (item < nitems) {
        long ia, ib, st;
        int k;
        const bool ok = LN::base(g, grp, t, ia, ib, st, k);
        const int q1 = split ? q0 + 1 : nj;
        int nq0 = 0;
        long ngroup = 0;
        const long next = item + G;
        if (next < nitems) decode(next, nq0, ngroup);
        bool b_next = next < nitems && L.job[nq0].aux != AUX_NONE;   // components still to be loaded
        for (int q = q0; q < q1; ++q) {
            const SpecJob& J = L.job[q];
            cpx<TC> v[F::RMAX], a[R0];
#pragma unroll
            for (int r = 0; r < R0; ++r) v[r] = f[r];
            if (J.aux) {
                const AuxLoad<TC> al(L, J, ok ? k : 0);
#pragma unroll
                for (int r = 0; r < R0; ++r) {
                    const cpx<TC> q_ = SUM ? x[SUM ? r : 0] : cpx<TC>{(TC)0, (TC)0};
                    a[r].x = al.pick(b0[r].x, b1[r].x, b2[r].x, q_.x);
                    a[r].y = al.pick(b0[r].y, b1[r].y, b2[r].y, q_.y);
                }
            }
            if (q + 1 < q1) load_job(q + 1, grp);
            else if (next < nitems) load_job(nq0, ngroup);
            if (b_next && (q + 1 == q1 || !L.job[q + 1].aux)) {
                load_b(ngroup);
                b_next = false;
            }
            F::forward(v, j, lds, twl);
            cpx<TC> z[RL], w[RL];
#pragma unroll
            for (int r = 0; r < RL; ++r) z[r] = v[r];
            // the auxiliary line's spectrum
            auto aux_to = [&](cpx<TC>* d) {
#pragma unroll
                for (int r = 0; r < R0; ++r) v[r] = a[r];
                F::forward(v, j, lds, twl);
#pragma unroll
                for (int r = 0; r < RL; ++r) d[r] = v[r];
            };
            if (SUM && J.aux) aux_to(w);
            for (int o = 0; o < (SUM ? 2 : 3); ++o) {
                // a first-derivative job, a job without an auxiliary line (uniform)
                if (o == 1 && !J.out[1]) break;
                if (o == 2) {
                    if (!J.aux) break;
                    aux_to(z);
                }
                const int mul = o == 2 ? (int)MUL_D1 : J.mul[o == 0 ? 0 : 1];
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const int kk = j + r * NBL;
                    v[r] = apply_mul<TC, N>(mul, z[r], kk, cx, icut, J.mc);
                    if (SUM && o == 1 && J.aux)
                        v[r] = cadd(v[r], apply_mul<TC, N>(MUL_D1, w[r], kk, cx, icut, J.mc));
                }
                F::inverse(v, j, lds, twl);
                if (ok && j < NB0) {
                    TC* __restrict__ out = (TC*)J.out[o];
#pragma unroll
                    for (int r = 0; r < R0; ++r) {
                        const int n = j + r * NB0;
                        if constexpr (DIR != 0) st_pair_nt(out, ia + n * st, v[r].x, v[r].y);
                        else {
                            st_nt(out, ia + n * st, v[r].x);
                            st_nt(out, ib + n * st, v[r].y);
                        }
                    }
                }
            }
        }
        item = next;
        q0 = nq0;
        grp = ngroup;
    }
}

template <typename TC, typename PL, int DIR, int B, int MODE, int LOP>
__device__ __forceinline__ void SpecK<TC, PL, DIR, B, MODE, LOP>::body_jobs(const SpecLaunch& L, uint3 bid,
                                                                            uint3 gdim)
{
    constexpr int N = PL::N;
    using LN = Lines<PL, DIR, B>;
    constexpr int NB0 = F::NB0, NBL = F::NBL, R0 = F::R0, RL = F::RL;
    const Geom g = L.g;
    extern __shared__ __align__(16) unsigned char smem[];
    cpx<TC>* twl = reinterpret_cast<cpx<TC>*>(smem);
    const cpx<TC>* __restrict__ twg = reinterpret_cast<const cpx<TC>*>(L.tw);
    F::stage_twiddles(twl, twg, threadIdx.x, NT);
    int t, j;
    LN::lane(threadIdx.x, t, j);
    cpx<TC>* lds = twl + F::TWN + t * F::SP;
    const long ngrp = LN::groups(g);
    const long G = gdim.x;
    const long nitems = ngrp * L.njobs;
    const double cx = L.cx;
    const int icut = L.icut;
    __syncthreads();

    // Column groups narrower than a 128-byte line (y direction, 2 B elements of
    // sizeof(TC) < 128 bytes: the 512-point lengths) share each line with the
    // next group.  Within every 16 items, item c (< 8) takes group 2c and item
    // c + 8 group 2c + 1: workgroups w and w + 8 run on the same XCD (they are
    // dealt round-robin over 8) at the same time, so a line is fetched once.
    constexpr bool half_line = DIR != 0 && 2 * B * (int)sizeof(TC) < 128;
    const bool pair = half_line && (G % 16 == 0) && (ngrp % 16 == 0);
    // (job, line group) of an item
    auto decode = [&](long item, int& jb, long& grp) {
        if (pair) {
            const long c = item & 15;
            item = item - c + (c < 8 ? 2 * c : 2 * (c - 8) + 1);
        }
        jb = (int)(item / ngrp);
        grp = item - (long)jb * ngrp;
    };

    // pass-0 inputs of one item (zeros for lines past the end)
    auto fetch = [&](long item, cpx<TC>* dst) {
        int jb;
        long grp;
        decode(item, jb, grp);
        const SpecJob& J = L.job[jb];
        long ia, ib, st;
        int k;
        const bool ok = LN::base(g, grp, t, ia, ib, st, k);
        if constexpr (MODE == SM_HC2R) {
            const TC* __restrict__ src = (const TC*)J.in[0];
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                const int n = j + r * NB0;
                dst[r] = {(TC)0, (TC)0};
                if (ok && j < NB0 && !(L.skip && n >= N / 2 - icut && n <= N / 2 + icut)) {
                    if constexpr (DIR != 0) dst[r] = ld_pair(src, ia + n * st);
                    else dst[r] = {src[ia + n * st], src[ib + n * st]};
                }
            }
        } else {
            const Loader<TC, LOP> ld(J, ok ? k : 0);
#pragma unroll
            for (int r = 0; r < R0; ++r) {
                const int n = j + r * NB0;
                dst[r] = {(TC)0, (TC)0};
                if (ok && j < NB0) {
                    if constexpr (DIR != 0) dst[r] = ld.pair(ia + n * st);
                    else dst[r] = {ld(ia + n * st), ld(ib + n * st)};
                }
            }
        }
    };

    cpx<TC> nxt[R0];
    long item = bid.x;
    if (item < nitems) fetch(item, nxt);
    for (; item < nitems; item += G) {
        cpx<TC> v[F::RMAX];
#pragma unroll
        for (int r = 0; r < R0; ++r) v[r] = nxt[r];
        if (item + G < nitems) fetch(item + G, nxt);

        int jb;
        long grp;
        decode(item, jb, grp);
        const SpecJob& J = L.job[jb];
        long ia, ib, st;
        int k;
        const bool ok = LN::base(g, grp, t, ia, ib, st, k);
        TC* __restrict__ out0 = (TC*)J.out[0];
        // epilogue constant of this line pair (one plane): the mean parts of B
        const TC add = (J.addk && ok ? (TC)J.addk[k] : (TC)0) + (TC)J.adds;

        if constexpr (MODE == SM_HC2R) {
            // raw halfcomplex lines -> LDS (natural order), then Z = A + iB
            if (j < NB0) {
#pragma unroll
                for (int r = 0; r < R0; ++r) lds[F::pad(j + r * NB0)] = v[r];
            }
            F::sync();
            if (j < NBL) {
#pragma unroll
                for (int r = 0; r < RL; ++r) {
                    const int kk = j + r * NBL;
                    const cpx<TC> u = lds[F::pad(kk)];
                    const cpx<TC> m = lds[F::pad((N - kk) % N)];
                    cpx<TC> A, Bv;
                    if (kk == 0 || kk == N / 2) { A = {u.x, (TC)0}; Bv = {u.y, (TC)0}; }
                    else if (kk < N / 2) { A = {u.x, m.x}; Bv = {u.y, m.y}; }
                    else { A = {m.x, -u.x}; Bv = {m.y, -u.y}; }
                    v[r] = {A.x - Bv.y, A.y + Bv.x};
                }
            }
            F::sync();
            cpx<TC> z[RL];
#pragma unroll
            for (int r = 0; r < RL; ++r) z[r] = v[r];
            for (int o = 0;; ++o) {
                F::inverse(v, j, lds, twl);
                if (ok && j < NB0) {
                    TC* __restrict__ out = (TC*)J.out[o];
                    const TC sc = o == 0 ? (TC)(1.0 / N) : (TC)1, ad = o == 0 ? add : (TC)0;
#pragma unroll
                    for (int r = 0; r < R0; ++r) {
                        const int n = j + r * NB0;
                        const TC xa = v[r].x * sc + ad, xb = v[r].y * sc + ad;
                        if constexpr (DIR != 0) st_pair(out, ia + n * st, xa, xb);
                        else {
                            out[ia + n * st] = xa;
                            out[ib + n * st] = xb;
                        }
                    }
                }
                if (sizeof(TC) == 4 || o == 1 || !J.out[1]) break;
#pragma unroll
                for (int r = 0; r < RL; ++r)
                    v[r] = apply_mul<TC, N>(J.mul[1], z[r], j + r * NBL, cx, icut, J.mc);
            }
        } else {
            F::forward(v, j, lds, twl);
            if constexpr (MODE == SM_R2HC) {
                r2hc_store(v, j, lds, ok, out0, ia, ib, st);
            } else {
                if (j < NBL) {
#pragma unroll
                    for (int r = 0; r < RL; ++r)
                        v[r] = apply_mul<TC, N>(J.mul[0], v[r], j + r * NBL, cx, icut, J.mc);
                }
                F::inverse(v, j, lds, twl);
                if (ok && j < NB0) {
#pragma unroll
                    for (int r = 0; r < R0; ++r) {
                        const int n = j + r * NB0;
                        if constexpr (DIR != 0) st_pair_nt(out0, ia + n * st, v[r].x + add, v[r].y + add);
                        else {
                            st_nt(out0, ia + n * st, v[r].x + add);
                            st_nt(out0, ib + n * st, v[r].y + add);
                        }
                    }
                }
            }
        }
    }
}


// ---------------------------------------------------------------------------
// host dispatch
// ---------------------------------------------------------------------------
// transforms per workgroup: about 256 threads along x; along y, 8 (FP64) or
// 16 (FP32) column pairs = 128-byte row segments.  LDS per workgroup: up to
// 64 KB, and up to 160 KB (gfx950's limit) for FP64 along y, so that the
// 512-point FP64 lengths keep full-line column groups (about 78 KB; the 4-field
// pass at 512^2 x 256 went from 2.15 to 1.48 ms).  In FP32 the 64 KB groups
// (half lines, paired onto one XCD) measured faster than full-line ones.
constexpr int SPEC_LDS_X = 65536, SPEC_LDS_Y = 163840;
template <typename TC, typename PL, int DIR>
constexpr int spec_b()
{
    constexpr int tpt = plan_tpt<PL>();
    constexpr int sp = RegFFT<TC, PL>::SP * (int)sizeof(cpx<TC>);
    constexpr int twb = RegFFT<TC, PL>::TWN * (int)sizeof(cpx<TC>);
    constexpr int lim = (DIR != 0 && sizeof(TC) == 8) ? SPEC_LDS_Y : SPEC_LDS_X;
    // FP64 y groups of 8 pairs (128-byte rows); 16 (256-byte rows) where a
    // transform takes at most 16 threads, so the group stays at 256 threads
    int b = DIR == 0 ? (128 / tpt > 0 ? 128 / tpt : 1) : (sizeof(TC) == 8 ? (tpt <= 16 ? 16 : 8) : 16);
    while (b > 1 && (b * tpt > 1024 || twb + b * sp > lim)) b /= 2;
    return b;
}

template <typename TC, typename PL, int B>
constexpr size_t spec_lds_bytes()
{
    return (size_t)(RegFFT<TC, PL>::TWN + B * RegFFT<TC, PL>::SP) * sizeof(cpx<TC>);
}

template <typename TC, typename PL, int DIR, int B, int MODE, int LOP>
static int launch_one(const SpecLaunch& L, hipStream_t s)
{
    using K = SpecK<TC, PL, DIR, B, MODE, LOP>;
    constexpr int NT = K::NT;
    constexpr size_t lds = spec_lds_bytes<TC, PL, B>();
    static_assert(lds <= (size_t)SPEC_LDS_Y, "transform workgroup exceeds 160 KB of LDS");
    auto kern = single_kernel<K>;
    const long ngrp = Lines<PL, DIR, B>::groups(L.g);
    // more than 64 KB of dynamic LDS is opted into once per kernel
    static int lds_ok = lds <= 65536 ? 1 : 0;
    if (!lds_ok) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) !=
            hipSuccess)
            return -22;
        lds_ok = 1;
    }
    // persistent grid: the workgroups that fit on the device at once
    static int per_cu = 0;
    if (per_cu == 0) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, NT, lds) != hipSuccess || n < 1) n = 1;
        per_cu = n;
    }
    const long resident = (long)per_cu * L.ncu * (L.grid_mult > 1 ? L.grid_mult : 1);
    SpecLaunch La = L;
    // items: the (job, line group) pairs, or line groups whose jobs share loads;
    // second derivatives share them where the line groups alone fill the device
    if (MODE == SM_DERIV2) La.split = L.njobs == 1 || ngrp < resident;
    const bool shared = LOP == LD_CROSS3 || (MODE == SM_DERIV2 && !La.split);
    long grid = ngrp * (shared ? 1 : L.njobs);
    if (L.ncu > 0 && grid > resident) grid = resident;
    return mhd_launch<K>(dim3((unsigned)grid), dim3(NT), lds, s, La);
}

// (mode, load op) pairs the solver uses besides second derivatives and the EMF's
// cross products; every job of L has the same load op
template <typename TC, typename PL, int DIR, int B>
static int launch_mode(const SpecLaunch& L, hipStream_t s)
{
    switch (L.mode * 8 + L.job[0].load_op) {
    case SM_DERIV1 * 8 + LD_PLAIN: return launch_one<TC, PL, DIR, B, SM_DERIV1, LD_PLAIN>(L, s);
    case SM_R2HC * 8 + LD_PLAIN: return launch_one<TC, PL, DIR, B, SM_R2HC, LD_PLAIN>(L, s);
    case SM_HC2R * 8 + LD_PLAIN: return launch_one<TC, PL, DIR, B, SM_HC2R, LD_PLAIN>(L, s);
    }
    return -23;
}

// along y with groups of B column pairs, partly filled ones where B does not
// divide a row's
template <typename TC, typename PL, int B, int MODE, int LOP>
static int launch_y(const SpecLaunch& L, hipStream_t s)
{
    return L.g.nx % (2 * B) == 0 ? launch_one<TC, PL, 1, B, MODE, LOP>(L, s) : launch_one<TC, PL, 2, B, MODE, LOP>(L, s);
}

// Second derivatives.  Half groups along y where a full one has 512 threads
// (FP64) or 1024 (FP32), so that two or more workgroups share a CU (256 points FP64:
// y 449 against 458 us; FP32: 293 against 276 at 256^2 x 160 and 317 against 284 at 256
// x 384 x 64, but 50 against 58 at 256^2 x 24 and 118 against 138 at 192^2 x 96).
// In FP64 also where the full group is 4 pairs (480, 640, 768 and 1024 points,
// 640 to 1024 threads): those spill 150 to 210 registers, 2 pairs and their 32-byte
// row segments do not (y pass 1478 -> 645 us at 256 x 480 x 64, 1712 -> 872 at
// 256 x 640 x 64, 1412 -> 763 at 256 x 768 x 48).  FP32 groups of 4 pairs stay: their
// halves read 16 bytes a row (a step of 256 x 1024 x 48: 2.7 -> 4.2 ms).
template <typename TC, typename PL>
static int launch_d2(const SpecLaunch& L, hipStream_t s)
{
    if (L.job[0].load_op != LD_PLAIN) return -23;
    if (L.dir == 0) return launch_one<TC, PL, 0, spec_b<TC, PL, 0>(), SM_DERIV2, LD_PLAIN>(L, s);
    constexpr int B0 = spec_b<TC, PL, 1>();
    constexpr int B2 = B0 >= (sizeof(TC) == 4 ? 8 : 4) && B0 * plan_tpt<PL>() >= (sizeof(TC) == 4 ? 1024 : 512)
                           ? B0 / 2 : B0;
    return launch_y<TC, PL, B2, SM_DERIV2, LD_PLAIN>(L, s);
}

template <typename TC, typename PL>
static int launch_plan(const SpecLaunch& L, hipStream_t s)
{
    if (L.dir == 0) return launch_mode<TC, PL, 0, spec_b<TC, PL, 0>()>(L, s);
    constexpr int B0 = spec_b<TC, PL, 1>();
    // the EMF's cross products: 3 lines and their 6 factors per thread, so half
    // groups in FP64, also of 4 pairs above 512 threads (they spill)
    constexpr int BC = sizeof(TC) == 8 && (B0 >= 8 || (B0 == 4 && B0 * plan_tpt<PL>() > 512)) ? B0 / 2 : B0;
    if (L.cross3) return launch_y<TC, PL, BC, SM_R2HC, LD_CROSS3>(L, s);
    // FP32 only, where a full group would be a 1024-thread workgroup (one per
    // CU): at 256 points 8 pairs beat 16 for the first derivatives (76, 72, 45 us
    // against 81, 83, 48); in FP64 4 pairs lose to 8.  The other FP32 modes keep
    // 16 pairs (8 pairs: hc2r 125 against 109, r2hc 63 against 58)
    constexpr int BH = (sizeof(TC) == 4 && B0 >= 8 && B0 * plan_tpt<PL>() >= 1024) ? B0 / 2 : B0;
    if (BH != B0 && L.mode == SM_DERIV1 && L.g.nx % (2 * BH) == 0)
        return launch_one<TC, PL, 1, BH, SM_DERIV1, LD_PLAIN>(L, s);
    if (L.g.nx % (2 * B0) == 0) return launch_mode<TC, PL, 1, B0>(L, s);
    return launch_mode<TC, PL, 2, B0>(L, s);
}

template <typename TC, int N>
static int launch_n(const SpecLaunch& L, hipStream_t s)
{
    const bool d2 = L.mode == SM_DERIV2;
    if constexpr (!std::is_void<typename AltPlan<N>::type>::value) {
        using PL = typename AltPlan<N>::type;
        if (L.variant == 1) return d2 ? launch_d2<TC, PL>(L, s) : launch_plan<TC, PL>(L, s);
    }
    if constexpr (!std::is_void<typename AltPlan2<N>::type>::value) {
        using PL = typename AltPlan2<N>::type;
        if (L.variant == 2) return d2 ? launch_d2<TC, PL>(L, s) : launch_plan<TC, PL>(L, s);
    }
    return d2 ? launch_d2<TC, typename D2Plan<N, TC>::type>(L, s) : launch_plan<TC, FftPlan<N>>(L, s);
}

}  // namespace mhd

// Defines launch_spectral_<group>(n, L, f32, s) for the lengths in SIZES.
#define MHD_SPECTRAL_GROUP(name, SIZES)                                        \
    namespace mhd {                                                            \
    int name(int n, const SpecLaunch& L, int f32, hipStream_t s)               \
    {                                                                          \
        switch (n) {                                                           \
            SIZES(MHD_SPEC_CASE)                                               \
        }                                                                      \
        return -20;                                                            \
    }                                                                          \
    int name##_mag(int n, int which, const MagSpecArgs& a, int f32, hipStream_t s) \
    {                                                                          \
        switch (n) {                                                           \
            SIZES(MHD_MAG_CASE)                                                \
        }                                                                      \
        (void)which; (void)a; (void)f32; (void)s;                              \
        return -20;                                                            \
    }                                                                          \
    int name##_expand(int n, const ExpandArgs& a, hipStream_t s)               \
    {                                                                          \
        switch (n) {                                                           \
            SIZES(MHD_EXPAND_CASE)                                             \
        }                                                                      \
        (void)a; (void)s;                                                      \
        return -20;                                                            \
    }                                                                          \
    }
#define MHD_EXPAND_CASE(n_)                                                    \
    case n_:                                                                   \
        return launch_expand_n<n_>(a, s);
#define MHD_MAG_CASE(n_)                                                       \
    case n_:                                                                   \
        return f32 ? launch_mag_n<float, n_>(which, a, s) : launch_mag_n<double, n_>(which, a, s);
#define MHD_SPEC_CASE(n_)                                                      \
    case n_:                                                                   \
        return f32 ? launch_n<float, n_>(L, s) : launch_n<double, n_>(L, s);
