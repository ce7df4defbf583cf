// spectral.hpp -- host-side interface of the horizontal (x/y) transform
// kernels: spectral derivatives (src/fft.F90 d1bydx/d1bydy/d2bydx/d2bydy),
// 2/3 dealiasing (dealias), and the real<->halfcomplex 2-D transform passes
// (forwardfft/inversefft) in FFTW-2 halfcomplex order.
#pragma once

#include "common.hpp"

namespace mhd {

enum SpecMode { SM_DERIV1 = 0, SM_DERIV2 = 1, SM_R2HC = 2, SM_HC2R = 3 };
// MUL_D2C: mc[0] * d2 + mc[1] * d1(d1(.)); the two differ at the Nyquist
// mode only, which d2 keeps (akx2) and d1 zeroes.
enum MulKind { MUL_D1 = 0, MUL_D2 = 1, MUL_MASK = 2, MUL_D2C = 3 };
// Inputs have the compute type.  Products take optional per-plane means m_i of
// their factors (the mixed path stores B without its means): the load is the
// product of (in_i + m_i) minus its per-plane constant, which no horizontal
// derivative sees.
//   LD_CROSS (in0+m0)*(in1+m1) - (in2+m2)*(in3+m3)
enum LoadOp { LD_PLAIN = 0, LD_CROSS = 1,
              // kernel template value only: three LD_CROSS jobs that are the
              // components of one cross product a x b, job q loading
              // {a_{q+1}, b_{q+2}, a_{q+2}, b_{q+1}} (indices mod 3); the six
              // factor lines of a line group are loaded once for all three
              LD_CROSS3 = 2 };
// A second-derivative job may carry a second, auxiliary line a:
//   AUX_PROD  a = ascale*(b_i+m_i)*(b_j+m_j) + xcoef*xin     (i, j = ai, aj)
//   AUX_MAXW  a = ascale*((b_i+m_i)^2 - (b_j+m_j)^2 - (b_l+m_l)^2) + xcoef*xin
// with b the launch's three field components (SpecLaunch::bf, bmean).
// FP64: its first derivative joins the second output, out[1] = mul[1](in) +
// d1(a).  The multipliers are linear, so the Maxwell stress and the composite
// viscous flux of a momentum component need no transform back, store and re-read
// of their own: one inverse transform returns the sum.
// FP32: it is an output of its own, out[2] = d1(a), and there is no xin.  The
// column kernel adds the stresses in FP64; summed in FP32 spectra, a small viscous
// term next to large stresses that cancel in the equation would be rounded away.
enum AuxOp { AUX_NONE = 0, AUX_PROD = 1, AUX_MAXW = 2 };

constexpr int SPEC_MAX_JOBS = 8;
// lengths without a register-blocked plan: run-time radix plans up to this length
constexpr int SPEC_GEN_MAX_N = 2048;
constexpr int SPEC_GEN_MAX_PASSES = 12;

// One transform job: one input field (or a fused product of fields) and up
// to two outputs.  Element types: *_f32 = 1 for float arrays, 0 for double.
struct SpecJob {
    const void* in[4];
    int in_f32;
    int load_op;      // LoadOp
    const double* mean[4]; // optional per-plane means of in[0..3] (nz entries)
    // LD_CROSS only: the load also subtracts jcoef[k] * jin (the eta(z) term
    // -(eta - eta_0) J of the EMF), when jin is set
    const void* jin;
    const double* jcoef;
    double mc[2];     // MUL_D2C coefficients
    int aux;          // AuxOp (SM_DERIV2 with out[1])
    int ai, aj;       // its field components
    double ascale;
    const void* xin;  // FP64: its further term xcoef * xin, or null
    double xcoef;
    // SM_DERIV2: out[1] may be null (the job's first derivative only); out[2] see
    // AuxOp.
    // SM_HC2R in FP64: out[1], when set, takes mul[1] of the same line (d/dx or
    // d/dy of the output, from the spectrum in registers)
    void* out[3];
    int out_f32;
    int mul[2];       // MulKind for out[0], out[1] (SM_DERIV*)
    const double* addk; // optional per-plane value added on store (nz entries)
    double adds;        // scalar added on store
};

struct SpecLaunch {
    Geom g;
    int dir;          // 0: along x (rows), 1: along y (columns)
    int mode;         // SpecMode
    int njobs;
    SpecJob job[SPEC_MAX_JOBS];
    // SM_DERIV2: field components of the jobs' auxiliary lines and their
    // per-plane means (null: none); jobs with an auxiliary line come first
    const void* bf[3];
    const double* bmean[3];
    int split;        // SM_DERIV2, set by the launcher: an item is one job of a line group, not all
    double cx;        // 2*pi/xmax (dir x) or 2*pi/ymax (dir y): mode m has wavenumber m*cx
    const void* tw;   // W_N^t table in the compute type
    int icut;         // dealias cut-off (n/2)/3
    int ncu;          // compute units: the persistent grid is occupancy x ncu workgroups
    int grid_mult;    // ... times this (>= 1; 0 = 1), a tunable launch shape
    int variant;      // radix plan: 0 the default, 1 and 2 the length's alternatives (if any)
    // SM_DERIV1: lines without a register plan, and those of the eight lengths
    // from 36 to 216 that gained theirs last (spectral_len_direct), are
    // transformed output point by output point in the run-time radix kernel
    int direct;
    int skip;         // SM_HC2R: the rows within icut of N/2 are zero and not read (magdealias's band)
    int cross3;       // set by the launcher: the three jobs form one cross product (LD_CROSS3)
    // set by the launcher for lengths without a register-blocked plan: the
    // run-time radices and the complex lines per workgroup
    int gen_radix[SPEC_GEN_MAX_PASSES];
    int gen_npass;
    int gen_nlb;
};

// x transforms of the magnetic part over row pairs (j, ny - j), with
// mag_deriv's and bandj's spectral algebra (spectral_mag.hpp)
struct MagSpecArgs {
    Geom g;
    const void* tw;          // W_nx^t table in the working precision
    double cx, cy;           // 2 pi / xmax, 2 pi / ymax
    int icutx, icuty;
    int skip;                // bandj_x: pol and tor are zero in the 2/3 band
    int ncu;
    void *ex, *ey, *ez;      // emf_x: E along physical x, halfcomplex y; ez in place
    void *cc, *d;
    const double *pol, *tor; // bandj_x
    const void* polz;
    // Bx, By, Jz, Bz, dBz/dx; FP32 also dBz/dy, so that both derivatives come from
    // the FP64 spectrum of pol (FP64 takes it from Bz's spectrum in the y pass)
    void* out[6];
};
// register-blocked lengths nx only (spectral_len_fixed), else -20
int launch_emf_x(const MagSpecArgs& a, int f32, hipStream_t s);
int launch_bandj_x(const MagSpecArgs& a, int f32, hipStream_t s);

// one direction of expand on an FP64 box g: out has 2 g.nx columns (dir 0) or
// 2 g.ny rows (dir 1); spectral_len_fixed lengths only (spectral_expand.hpp)
struct ExpandArgs {
    Geom g;
    int dir, ncu;
    const void* tw;          // W_n^t table of the doubled direction's length n
    const double* in;
    double* out;
};
int launch_expand(const ExpandArgs& a, hipStream_t s);

// What the kernels take for granted of a launch's jobs: an auxiliary line
// (AuxOp) belongs to a second-derivative job with both outputs, in FP32 with its
// own third output and no further term; it takes two different field components
// out of three that are there (AuxLoad indexes bf and bmean by them); the jobs
// that have one come first (body_deriv2 reloads the components during the
// others).  The second output of an inverse transform is FP64 only.
inline bool spec_launch_ok(const SpecLaunch& L, int f32)
{
    if (L.njobs < 0 || L.njobs > SPEC_MAX_JOBS) return false;
    for (int q = 0; q < L.njobs; ++q) {
        const SpecJob& J = L.job[q];
        if (L.mode == SM_HC2R && f32 && J.out[1]) return false;
        if (J.aux == AUX_NONE) continue;
        if (L.mode != SM_DERIV2 || !J.out[1]) return false;
        if (f32 && (!J.out[2] || J.xin)) return false;
        if (!L.bf[0] || !L.bf[1] || !L.bf[2] || J.ai < 0 || J.ai > 2) return false;
        if (J.aux == AUX_PROD) {
            if (J.aj < 0 || J.aj > 2 || J.aj == J.ai) return false;
        } else if (J.aux != AUX_MAXW) {
            return false;
        }
        if (q > 0 && L.job[q - 1].aux == AUX_NONE) return false;
    }
    return true;
}

// Returns 0 or a negative code (-20: unsupported length, -23: jobs that
// spec_launch_ok refuses).
int launch_spectral(const SpecLaunch& L, int compute_f32, hipStream_t s);

// every even length from 2 to SPEC_GEN_MAX_N: register-blocked kernels for
// the lengths of fft_reg.hpp, run-time radix kernels for the others
bool spectral_len_supported(int n);
// the length has a register-blocked plan
bool spectral_len_fixed(int n);
// run-time radix plan of an even length (false: odd or too long)
bool generic_plan(int n, int radix[SPEC_GEN_MAX_PASSES], int* npass, bool direct = false);
int launch_spectral_generic(const SpecLaunch& L, int compute_f32, hipStream_t s);
// radix plans of the length: SpecLaunch::variant runs from 0 to this - 1
int spectral_variants(int n);
// threads of a transform in the FP32 second-derivative passes (0: no plan)
int spectral_d2_threads(int n);

}  // namespace mhd
