// spectral_generic.hip -- the horizontal transform kernels for any even
// length that has no register-blocked plan (fft_reg.hpp), as the reference
// plans FFTW for any even nx, ny (src/fft.F90:101-136).
//
// A workgroup holds `nlb` complex lines (two real lines each, as in
// spectral_impl.hpp) in LDS and runs a self-sorting (Stockham) FFT whose
// radices are the length's factors, found at run time: 4s (and one 8 where the
// power of two is odd), then 3, 5, 7 and any larger prime.  In a pass with radix
// R up to 13 a thread owns one butterfly: it reads its R points, multiplies them
// by the twiddles of one LDS table W_N^t and writes the R outputs
//   dst[(j / Ns) Ns R + (j mod Ns) + m Ns], m < R,
// ping-ponging between two LDS buffers.  Larger primes compute every output
// point directly, N R multiply-adds per line and pass.  Loads (every LoadOp),
// spectral multipliers, the halfcomplex packing and the stores are those of
// spec_kernel.
//
// What bounds it: the latency of the passes (a barrier each) at the three
// workgroups per CU that three LDS buffers leave.  The transforms of a step on
// lengths 100 (4 5 5) and 144 (4 4 3 3), 61 planes FP64: 507 us with one output
// point per thread (R reads and twiddles each, a 64-bit division per point for
// its line), 445 with a butterfly per thread.
#include "spectral_impl.hpp"

namespace mhd {

namespace {

constexpr int GNT = 256;
constexpr int GEN_MAX_LINES = 64;

template <typename TC>
__device__ __forceinline__ cpx<TC> apply_mul_rt(int kind, cpx<TC> z, int k, int N, double cx, int icut,
                                                 const double* mc)
{
    const double invN = 1.0 / N;
    const int m = (k < N - k) ? k : N - k;
    if (kind == MUL_D1) {
        if (k == 0 || 2 * k == N) return {(TC)0, (TC)0};
        const TC a = (TC)(((double)m * cx) * invN);
        if (2 * k < N) return {-a * z.y, a * z.x};
        return {a * z.y, -a * z.x};
    } else if (kind == MUL_D2 || kind == MUL_D2C) {
        double f = -((double)m * (double)m * cx * cx);
        if (kind == MUL_D2C) f *= (2 * k == N) ? mc[0] : mc[0] + mc[1];
        const TC a = (TC)(f * invN);
        return {a * z.x, a * z.y};
    } else {
        if (m < N / 2 - icut) return {z.x * (TC)invN, z.y * (TC)invN};
        return {(TC)0, (TC)0};
    }
}

// q / d for 0 <= q < 2^16, inv = 1.0f / d
__device__ __forceinline__ int fdiv(int q, float inv) { return (int)(((float)q + 0.5f) * inv); }

// R-point DFT in registers; odd primes from 7 on take their roots of unity
// W_R^t = tw[t N / R] from the table (uniform reads)
template <typename TC, int R, bool INV>
__device__ __forceinline__ void gen_dft(cpx<TC>* v, const cpx<TC>* __restrict__ tw, int NR)
{
    if constexpr (R <= 5 || R == 8) {
        (void)tw;
        (void)NR;
        dft_r<TC, R, INV>(v);
    } else {
        constexpr int H = (R - 1) / 2;
        cpx<TC> s[H], d[H], o[R];
#pragma unroll
        for (int r = 0; r < H; ++r) {
            s[r] = cadd(v[r + 1], v[R - 1 - r]);
            d[r] = csub(v[r + 1], v[R - 1 - r]);
        }
        o[0] = v[0];
#pragma unroll
        for (int r = 0; r < H; ++r) o[0] = cadd(o[0], s[r]);
#pragma unroll
        for (int m = 1; m <= H; ++m) {
            cpx<TC> a = v[0], b = {(TC)0, (TC)0};
#pragma unroll
            for (int r = 1; r <= H; ++r) {
                const cpx<TC> w = tw[(r * m % R) * NR];   // cos, -sin
                a.x += w.x * s[r - 1].x;
                a.y += w.x * s[r - 1].y;
                b.x -= w.y * d[r - 1].x;
                b.y -= w.y * d[r - 1].y;
            }
            // a -+ i b
            const cpx<TC> ib = cmul_i<TC, INV ? 1 : -1>(b);
            o[m] = cadd(a, ib);
            o[R - m] = csub(a, ib);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = o[r];
    }
}

// one pass over the workgroup's nlb lines, src -> dst, one butterfly per thread
template <typename TC, int R, bool INV>
__device__ __forceinline__ void gen_pass_r(const cpx<TC>* __restrict__ src, cpx<TC>* __restrict__ dst,
                                           const cpx<TC>* __restrict__ tw, int N, int nlb, int Ns)
{
    const int NB = N / R, ts = NB / Ns;   // twiddle of butterfly kk, point r: W_N^(r kk ts)
    const float iNB = 1.0f / (float)NB, iNs = 1.0f / (float)Ns;
    for (int q = threadIdx.x; q < nlb * NB; q += GNT) {
        const int b = fdiv(q, iNB), j = q - b * NB;
        const int blk = fdiv(j, iNs), kk = j - blk * Ns;
        const cpx<TC>* s = src + b * N + j;
        cpx<TC> v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = s[r * NB];
        const int e = kk * ts;
#pragma unroll
        for (int r = 1; r < R; ++r) {
            const cpx<TC> w = tw[r * e];   // r kk ts < N
            v[r] = INV ? cmulc(v[r], w) : cmul(v[r], w);
        }
        gen_dft<TC, R, INV>(v, tw, NB);
        cpx<TC>* d = dst + b * N + blk * Ns * R + kk;
#pragma unroll
        for (int r = 0; r < R; ++r) d[r * Ns] = v[r];
    }
    __syncthreads();
}

// any radix, one output point per thread
template <typename TC, bool INV>
__device__ __forceinline__ void gen_pass(const cpx<TC>* __restrict__ src, cpx<TC>* __restrict__ dst,
                                         const cpx<TC>* __restrict__ tw, int N, int nlb, int Ns, int R)
{
    const int NB = N / R;
    const int tstride = N / (Ns * R);
    const int NsR = Ns * R;
    for (int q = threadIdx.x; q < nlb * N; q += GNT) {
        const int b = q / N, o = q - b * N;
        const int blk = o / NsR, rem = o - blk * NsR;
        const int m = rem / Ns, kk = rem - m * Ns;
        const int j = blk * Ns + kk;
        const int estep = (tstride * (kk + m * Ns)) % N;
        const cpx<TC>* s = src + b * N;
        cpx<TC> acc = s[j];
        int e = 0;
        for (int r = 1; r < R; ++r) {
            e += estep;
            if (e >= N) e -= N;
            const cpx<TC> x = s[j + r * NB];
            acc = cadd(acc, INV ? cmulc(x, tw[e]) : cmul(x, tw[e]));
        }
        dst[b * N + o] = acc;
    }
    __syncthreads();
}

// the transform of the lines in *a (b is scratch of the same size); returns
// the buffer holding the result
template <typename TC, bool INV>
__device__ __forceinline__ cpx<TC>* gen_fft(cpx<TC>* a, cpx<TC>* b, const cpx<TC>* tw, const SpecLaunch& L,
                                            int N, int nlb)
{
    int Ns = 1;
    for (int p = 0; p < L.gen_npass; ++p) {
        const int R = L.gen_radix[p];
        switch (L.direct ? 0 : R) {
        case 2: gen_pass_r<TC, 2, INV>(a, b, tw, N, nlb, Ns); break;
        case 3: gen_pass_r<TC, 3, INV>(a, b, tw, N, nlb, Ns); break;
        case 4: gen_pass_r<TC, 4, INV>(a, b, tw, N, nlb, Ns); break;
        case 5: gen_pass_r<TC, 5, INV>(a, b, tw, N, nlb, Ns); break;
        case 7: gen_pass_r<TC, 7, INV>(a, b, tw, N, nlb, Ns); break;
        case 8: gen_pass_r<TC, 8, INV>(a, b, tw, N, nlb, Ns); break;
        case 11: gen_pass_r<TC, 11, INV>(a, b, tw, N, nlb, Ns); break;
        case 13: gen_pass_r<TC, 13, INV>(a, b, tw, N, nlb, Ns); break;
        default: gen_pass<TC, INV>(a, b, tw, N, nlb, Ns, R);
        }
        cpx<TC>* t = a;
        a = b;
        b = t;
        Ns *= R;
    }
    return a;
}

template <int DIR>
struct GenLines {
    // line groups of nlb complex lines per job
    static __host__ __device__ long groups(const Geom& g, int nlb)
    {
        if constexpr (DIR == 0) return ((long)g.nz * g.ny / 2 + nlb - 1) / nlb;
        else return (long)g.nz * ((g.nx / 2 + nlb - 1) / nlb);
    }
    // element 0 of the lines a, b of line b_ in group grp; false past the end
    static __device__ __forceinline__ bool base(const Geom& g, int nlb, long grp, int b_, long& ia, long& ib,
                                                long& st, int& k)
    {
        if constexpr (DIR == 0) {
            const long cl = grp * nlb + b_;
            const long row = 2 * cl;
            k = (int)(row / g.ny);
            ia = row * g.nx;
            ib = ia + g.nx;
            st = 1;
            return cl < (long)g.nz * g.ny / 2;
        } else {
            const int gpp = (g.nx / 2 + nlb - 1) / nlb;
            k = (int)(grp / gpp);
            const int cp = (int)(grp - (long)k * gpp) * nlb + b_;
            ia = (long)k * g.nxy + 2 * cp;
            ib = ia + 1;
            st = g.nx;
            return 2 * cp < g.nx;
        }
    }
};

template <typename TC, int DIR, int MODE, int LOP>
struct GenK {
    using Args = SpecLaunch;
    static constexpr int NT = GNT;
    static __device__ __forceinline__ void body(const SpecLaunch& L, uint3 bid, uint3 gdim);
};

template <typename TC, int DIR, int MODE, int LOP>
__device__ __forceinline__ void GenK<TC, DIR, MODE, LOP>::body(const SpecLaunch& L, uint3 bid, uint3 gdim)
{
    const Geom g = L.g;
    const int N = DIR == 0 ? g.nx : g.ny;
    const int nlb = L.gen_nlb;
    extern __shared__ __align__(16) unsigned char smem[];
    // the lines of the item: elements 0 of lines a and b (a < 0: past the end), plane
    long* line_a = reinterpret_cast<long*>(smem);
    long* line_b = line_a + GEN_MAX_LINES;
    int* line_k = reinterpret_cast<int*>(line_b + GEN_MAX_LINES);
    cpx<TC>* twl = reinterpret_cast<cpx<TC>*>(line_k + GEN_MAX_LINES);
    cpx<TC>* buf0 = twl + N;
    cpx<TC>* buf1 = buf0 + nlb * N;
    cpx<TC>* buf2 = buf1 + nlb * N;   // two-output jobs only (gen_lds_bytes)
    const cpx<TC>* __restrict__ twg = reinterpret_cast<const cpx<TC>*>(L.tw);
    for (int i = threadIdx.x; i < N; i += GNT) twl[i] = twg[i];
    const long ngrp = GenLines<DIR>::groups(g, nlb);
    const long nitems = ngrp * L.njobs;
    const int P = nlb * N;
    const float iN = 1.0f / (float)N, iL = 1.0f / (float)nlb;
    const long st = DIR == 0 ? 1 : g.nx;
    __syncthreads();

    for (long item = bid.x; item < nitems; item += gdim.x) {
        const int jb = (int)(item / ngrp);
        const long grp = item - (long)jb * ngrp;
        const SpecJob& J = L.job[jb];
        // point q of the workgroup: line b, element n (rows: n fastest;
        // columns: the line fastest, so a row of adjacent column pairs is one
        // contiguous load)
        auto point = [&](int q, int& b, int& n) {
            if constexpr (DIR == 0) { b = fdiv(q, iN); n = q - b * N; }
            else { n = fdiv(q, iL); b = q - n * nlb; }
        };
        if ((int)threadIdx.x < nlb) {
            long ia, ib, s1;
            int k;
            const bool ok = GenLines<DIR>::base(g, nlb, grp, threadIdx.x, ia, ib, s1, k);
            line_a[threadIdx.x] = ok ? ia : -1;
            line_b[threadIdx.x] = ib;
            line_k[threadIdx.x] = k;
        }
        __syncthreads();
        // load
        for (int q = threadIdx.x; q < P; q += GNT) {
            int b, n;
            point(q, b, n);
            const long ia = line_a[b], ib = line_b[b];
            const int k = line_k[b];
            cpx<TC> v = {(TC)0, (TC)0};
            if (ia >= 0) {
                if constexpr (MODE == SM_HC2R) {
                    const TC* __restrict__ src = (const TC*)J.in[0];
                    if (!(L.skip && n >= N / 2 - L.icut && n <= N / 2 + L.icut))
                        v = {src[ia + n * st], src[ib + n * st]};
                } else {
                    const Loader<TC, LOP> ld(J, k);
                    v = {ld(ia + n * st), ld(ib + n * st)};
                }
            }
            buf0[b * N + n] = v;
        }
        __syncthreads();

        TC* __restrict__ out0 = (TC*)J.out[0];
        TC* __restrict__ out1 = (TC*)J.out[1];
        auto store = [&](const cpx<TC>* res, TC* __restrict__ out, TC scale, bool plus = true) {
            for (int q = threadIdx.x; q < P; q += GNT) {
                int b, n;
                point(q, b, n);
                const long ia = line_a[b], ib = line_b[b];
                if (ia < 0) continue;
                const int k = line_k[b];
                const TC add = plus ? (J.addk ? (TC)J.addk[k] : (TC)0) + (TC)J.adds : (TC)0;
                const cpx<TC> v = res[b * N + n];
                out[ia + n * st] = v.x * scale + add;
                out[ib + n * st] = v.y * scale + add;
            }
        };

        if constexpr (MODE == SM_HC2R) {
            // two halfcomplex lines -> the spectrum of z = a + i b
            for (int q = threadIdx.x; q < P; q += GNT) {
                const int b = fdiv(q, iN), kk = q - b * N;
                const cpx<TC> u = buf0[b * N + kk];
                const cpx<TC> m = buf0[b * N + (N - kk) % N];
                cpx<TC> A, Bv;
                if (kk == 0 || 2 * kk == N) { A = {u.x, (TC)0}; Bv = {u.y, (TC)0}; }
                else if (2 * kk < N) { A = {u.x, m.x}; Bv = {u.y, m.y}; }
                else { A = {m.x, -u.x}; Bv = {m.y, -u.y}; }
                buf1[b * N + kk] = {A.x - Bv.y, A.y + Bv.x};
            }
            __syncthreads();
            if (out1) {
                // the derivative output first, from a copy of the spectrum
                for (int q = threadIdx.x; q < P; q += GNT)
                    buf0[q] = apply_mul_rt<TC>(J.mul[1], buf1[q], q - fdiv(q, iN) * N, N, L.cx, L.icut, J.mc);
                __syncthreads();
                const cpx<TC>* der = gen_fft<TC, true>(buf0, buf2, twl, L, N, nlb);
                store(der, out1, (TC)1, false);
                __syncthreads();
            }
            const cpx<TC>* res = gen_fft<TC, true>(buf1, buf0, twl, L, N, nlb);
            store(res, out0, (TC)(1.0 / N));
        } else {
            cpx<TC>* spec = gen_fft<TC, false>(buf0, buf1, twl, L, N, nlb);
            cpx<TC>* other = spec == buf0 ? buf1 : buf0;
            if constexpr (MODE == SM_R2HC) {
                for (int q = threadIdx.x; q < P; q += GNT) {
                    int b, n;
                    point(q, b, n);
                    const long ia = line_a[b], ib = line_b[b];
                    if (ia < 0) continue;
                    const int kk = (2 * n <= N) ? n : N - n;
                    const cpx<TC> zk = spec[b * N + kk];
                    const cpx<TC> zn = spec[b * N + (N - kk) % N];
                    TC a, bb;
                    if (2 * n <= N) { a = (TC)0.5 * (zk.x + zn.x); bb = (TC)0.5 * (zk.y + zn.y); }
                    else { a = (TC)0.5 * (zk.y - zn.y); bb = (TC)0.5 * (zn.x - zk.x); }
                    out0[ia + n * st] = a;
                    out0[ib + n * st] = bb;
                }
            } else {
                constexpr bool SUM = sizeof(TC) == 8;   // AuxOp
                constexpr int NOUT = (MODE == SM_DERIV2) ? (SUM ? 2 : 3) : 1;
                for (int o = 0; o < NOUT; ++o) {
                    // a first-derivative job, a job without an auxiliary line (uniform)
                    if (o == 1 && out1 == nullptr) break;
                    if (o == 2 && !J.aux) break;
                    cpx<TC>* aux = nullptr;
                    // a job with one output needs no third buffer
                    cpx<TC>* work = out1 ? buf2 : spec;
                    if (o == (SUM ? 1 : 2) && J.aux) {
                        // the auxiliary line's spectrum
                        for (int q = threadIdx.x; q < P; q += GNT) {
                            int b, n;
                            point(q, b, n);
                            const long ia = line_a[b], ib = line_b[b];
                            const int k = line_k[b];
                            cpx<TC> v = {(TC)0, (TC)0};
                            if (ia >= 0) {
                                const AuxLoad<TC> al(L, J, k);
                                const TC* __restrict__ p0 = (const TC*)L.bf[al.ai];
                                const TC* __restrict__ p1 = (const TC*)L.bf[al.aj];
                                const TC* __restrict__ p2 = (const TC*)L.bf[al.al];
                                const TC* __restrict__ px = SUM ? (const TC*)J.xin : nullptr;
                                const long i = ia + n * st, e = ib + n * st;
                                const bool mw = J.aux == AUX_MAXW;
                                v = {al.one(p0[i], p1[i], mw ? p2[i] : (TC)0, px ? px[i] : (TC)0),
                                     al.one(p0[e], p1[e], mw ? p2[e] : (TC)0, px ? px[e] : (TC)0)};
                            }
                            other[b * N + n] = v;
                        }
                        __syncthreads();
                        aux = gen_fft<TC, false>(other, buf2, twl, L, N, nlb);
                        work = aux == other ? buf2 : other;
                    }
                    // multiplied spectrum into `dst`, inverse through `work`
                    cpx<TC>* dst = aux ? aux : other;
                    for (int q = threadIdx.x; q < P; q += GNT) {
                        const int kk = q - fdiv(q, iN) * N;
                        cpx<TC> m = o == 2 ? cpx<TC>{(TC)0, (TC)0}
                                           : apply_mul_rt<TC>(J.mul[o == 0 ? 0 : 1], spec[q], kk, N, L.cx, L.icut, J.mc);
                        if (aux) {
                            const cpx<TC> d = apply_mul_rt<TC>(MUL_D1, aux[q], kk, N, L.cx, L.icut, J.mc);
                            m = o == 2 ? d : cadd(m, d);
                        }
                        dst[q] = m;
                    }
                    __syncthreads();
                    const cpx<TC>* res = gen_fft<TC, true>(dst, work, twl, L, N, nlb);
                    store(res, (TC*)J.out[o], (TC)1);
                    __syncthreads();   // the buffers are reused by the next output
                }
            }
        }
        __syncthreads();   // LDS reused by the next item
    }
}

// the table of lines, twiddles, the two buffers of the passes and, where a
// spectrum outlives them (two outputs), a third
size_t gen_lds_bytes(int N, int nlb, size_t csz, bool keep)
{
    return GEN_MAX_LINES * (2 * sizeof(long) + sizeof(int)) + (size_t)(N + (keep ? 3 : 2) * nlb * N) * csz;
}
bool gen_keeps(const SpecLaunch& L)
{
    for (int q = 0; q < L.njobs; ++q)
        if (L.job[q].out[1]) return true;
    return false;
}

template <typename TC, int DIR, int MODE, int LOP>
int gen_launch(const SpecLaunch& L, hipStream_t s)
{
    const size_t lds = gen_lds_bytes(L.dir == 0 ? L.g.nx : L.g.ny, L.gen_nlb, sizeof(cpx<TC>), gen_keeps(L));
    using K = GenK<TC, DIR, MODE, LOP>;
    auto kern = single_kernel<K>;
    // more than 64 KB of dynamic LDS is opted into once per kernel
    static int lds_max = 65536;
    if ((int)lds > lds_max) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 163840) !=
            hipSuccess)
            return -22;
        lds_max = 163840;
    }
    const long items = GenLines<DIR>::groups(L.g, L.gen_nlb) * L.njobs;
    long grid = items;
    const long cap = (long)(L.ncu > 0 ? L.ncu : 256) * 8;
    if (grid > cap) grid = cap;
    return mhd_launch<K>(dim3((unsigned)grid), dim3(GNT), lds, s, L);
}

template <typename TC, int DIR>
int gen_mode(const SpecLaunch& L, hipStream_t s)
{
    switch (L.mode * 8 + L.job[0].load_op) {
    case SM_DERIV1 * 8 + LD_PLAIN: return gen_launch<TC, DIR, SM_DERIV1, LD_PLAIN>(L, s);
    case SM_DERIV2 * 8 + LD_PLAIN: return gen_launch<TC, DIR, SM_DERIV2, LD_PLAIN>(L, s);
    case SM_R2HC * 8 + LD_PLAIN: return gen_launch<TC, DIR, SM_R2HC, LD_PLAIN>(L, s);
    case SM_R2HC * 8 + LD_CROSS: return gen_launch<TC, DIR, SM_R2HC, LD_CROSS>(L, s);
    case SM_HC2R * 8 + LD_PLAIN: return gen_launch<TC, DIR, SM_HC2R, LD_PLAIN>(L, s);
    }
    return -23;
}

}  // namespace

bool generic_plan(int n, int radix[SPEC_GEN_MAX_PASSES], int* npass, bool direct)
{
    if (n < 2 || n % 2 || n > SPEC_GEN_MAX_N) return false;
    int p = 0, m = n;
    // one 8 where the power of two is odd and at least 8 (point by point: only
    // 4s and a 2), then 4s
    int e2 = 0;
    while (m % (2 << e2) == 0) ++e2;
    if (!direct && e2 >= 3 && e2 % 2) { radix[p++] = 8; m /= 8; }
    while (m % 4 == 0 && p < SPEC_GEN_MAX_PASSES) { radix[p++] = 4; m /= 4; }
    for (int f = 2; m > 1 && p < SPEC_GEN_MAX_PASSES; ++f)
        while (m % f == 0 && p < SPEC_GEN_MAX_PASSES) { radix[p++] = f; m /= f; }
    *npass = p;
    return m == 1;
}

int launch_spectral_generic(const SpecLaunch& L0, int f32, hipStream_t s)
{
    SpecLaunch L = L0;
    const int N = L.dir == 0 ? L.g.nx : L.g.ny;
    if (!generic_plan(N, L.gen_radix, &L.gen_npass, L.direct != 0)) return -20;
    // lines per workgroup: about 1024 points, at most 64 KB of LDS where one
    // line fits in that
    const size_t csz = f32 ? sizeof(cpx<float>) : sizeof(cpx<double>);
    const bool keep = gen_keeps(L);
    int nlb = 1024 / N;
    if (nlb < 1) nlb = 1;
    if (nlb > GEN_MAX_LINES) nlb = GEN_MAX_LINES;
    while (nlb > 1 && gen_lds_bytes(N, nlb, csz, keep) > 65536) --nlb;
    L.gen_nlb = nlb;
    if (f32) return L.dir == 0 ? gen_mode<float, 0>(L, s) : gen_mode<float, 1>(L, s);
    return L.dir == 0 ? gen_mode<double, 0>(L, s) : gen_mode<double, 1>(L, s);
}

}  // namespace mhd
