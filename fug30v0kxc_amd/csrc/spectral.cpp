// spectral.cpp -- dispatch of the horizontal transform kernels by length.
#include <type_traits>

#include "fft_reg.hpp"
#include "spectral.hpp"

namespace mhd {

#define MHD_DECL(f)                                                              \
    int f(int n, const SpecLaunch& L, int f32, hipStream_t s);                    \
    int f##_mag(int n, int which, const MagSpecArgs& a, int f32, hipStream_t s);  \
    int f##_expand(int n, const ExpandArgs& a, hipStream_t s);
MHD_DECL(launch_spectral_g0)
MHD_DECL(launch_spectral_g1)
MHD_DECL(launch_spectral_g2)
MHD_DECL(launch_spectral_g3)
MHD_DECL(launch_spectral_g4)
MHD_DECL(launch_spectral_g5)
MHD_DECL(launch_spectral_g6)
MHD_DECL(launch_spectral_g7)
#undef MHD_DECL

#define MHD_ALL_SIZES(X) X(8) X(12) X(16) X(20) X(24) X(30) X(32) X(36) X(40) X(48) X(60) X(64) X(72) X(80) X(96) X(100) X(108) X(120) X(128) X(144) X(160) X(180) X(192) X(200) X(216) X(240) X(256) X(320) X(384) X(480) X(512) X(640) X(768) X(1024)

bool spectral_len_fixed(int n)
{
    switch (n) {
#define X(n_) case n_: return true;
        MHD_ALL_SIZES(X)
#undef X
    }
    return false;
}

bool spectral_len_supported(int n)
{
    if (spectral_len_fixed(n)) return true;
    int r[SPEC_GEN_MAX_PASSES], np = 0;
    return generic_plan(n, r, &np);
}

int spectral_variants(int n)
{
    switch (n) {
#define X(n_)                                                                  \
    case n_:                                                                   \
        return std::is_void<AltPlan<n_>::type>::value ? 1 : std::is_void<AltPlan2<n_>::type>::value ? 2 : 3;
        MHD_ALL_SIZES(X)
#undef X
    }
    return 1;
}

int spectral_d2_threads(int n)
{
    switch (n) {
#define X(n_) case n_: return plan_tpt<typename D2Plan<n_, float>::type>();
        MHD_ALL_SIZES(X)
#undef X
    }
    return 0;
}

// the file that instantiates a length's kernels
static int size_group(int n)
{
    switch (n) {
    case 36: case 72: case 100: case 108: return 6;
    case 144: case 180: case 200: case 216: return 7;
    }
    return n <= 60 ? 0 : n <= 128 ? 1 : n <= 256 ? 2 : n <= 480 ? 3 : n <= 640 ? 4 : 5;
}
// lengths with a plan that direct launches do not use (SpecLaunch::direct)
static bool spectral_len_direct(int n) { return size_group(n) >= 6; }
#define MHD_GROUP_FNS(k)                                                                                  \
    launch_spectral_g0##k, launch_spectral_g1##k, launch_spectral_g2##k, launch_spectral_g3##k,           \
        launch_spectral_g4##k, launch_spectral_g5##k, launch_spectral_g6##k, launch_spectral_g7##k

static int launch_group(const SpecLaunch& L, int compute_f32, hipStream_t s)
{
    static constexpr decltype(&launch_spectral_g0) fn[] = {MHD_GROUP_FNS()};
    const int n = (L.dir == 0) ? L.g.nx : L.g.ny;
    if (!spectral_len_fixed(n) || (L.direct && spectral_len_direct(n))) return launch_spectral_generic(L, compute_f32, s);
    return fn[size_group(n)](n, L, compute_f32, s);
}

static int launch_mag_x(int which, const MagSpecArgs& a, int f32, hipStream_t s)
{
    static constexpr decltype(&launch_spectral_g0_mag) fn[] = {MHD_GROUP_FNS(_mag)};
    const int n = a.g.nx;
    if (!spectral_len_fixed(n)) return -20;
    return fn[size_group(n)](n, which, a, f32, s);
}
int launch_emf_x(const MagSpecArgs& a, int f32, hipStream_t s) { return launch_mag_x(0, a, f32, s); }
int launch_bandj_x(const MagSpecArgs& a, int f32, hipStream_t s) { return launch_mag_x(1, a, f32, s); }

int launch_expand(const ExpandArgs& a, hipStream_t s)
{
    static constexpr decltype(&launch_spectral_g0_expand) fn[] = {MHD_GROUP_FNS(_expand)};
    const int n = a.dir == 0 ? a.g.nx : a.g.ny;
    if (!spectral_len_fixed(n)) return -20;
    return fn[size_group(n)](n, a, s);
}
#undef MHD_GROUP_FNS

// Three LD_CROSS jobs whose factors are the components of two vectors a, b
// with job q = a_{q+1} b_{q+2} - a_{q+2} b_{q+1}: the EMF u x B.
static bool is_cross_product(const SpecLaunch& L)
{
    if (L.njobs != 3) return false;
    const SpecJob* J = L.job;
    for (int q = 0; q < 3; ++q)
        if (J[q].load_op != LD_CROSS || J[q].in_f32 != J[0].in_f32) return false;
    // a_{q+1} = J[q].in[0], b_{q+2} = J[q].in[1]
    const void *a[3], *b[3];
    for (int q = 0; q < 3; ++q) {
        a[(q + 1) % 3] = J[q].in[0];
        b[(q + 2) % 3] = J[q].in[1];
    }
    for (int q = 0; q < 3; ++q)
        if (J[q].in[2] != a[(q + 2) % 3] || J[q].in[3] != b[(q + 1) % 3]) return false;
    return true;
}

// The load operation is a compile-time parameter of the kernels, so jobs are
// launched in groups of equal load operation -- except, on the
// register-blocked lengths, the three components of a cross product along y,
// which share their six factor loads (LD_CROSS3).
int launch_spectral(const SpecLaunch& L, int compute_f32, hipStream_t s)
{
    if (L.njobs == 0) return 0;
    if (!spec_launch_ok(L, compute_f32)) return -23;
    if (L.mode == SM_R2HC && L.dir == 1 && spectral_len_fixed(L.g.ny) && is_cross_product(L)) {
        SpecLaunch G = L;
        G.cross3 = 1;
        return launch_group(G, compute_f32, s);
    }
    bool done[SPEC_MAX_JOBS] = {};
    for (int i = 0; i < L.njobs; ++i) {
        if (done[i]) continue;
        SpecLaunch G = L;
        G.njobs = 0;
        for (int j = i; j < L.njobs; ++j)
            if (!done[j] && L.job[j].load_op == L.job[i].load_op) {
                G.job[G.njobs++] = L.job[j];
                done[j] = true;
            }
        const int e = launch_group(G, compute_f32, s);
        if (e) return e;
    }
    return 0;
}

}  // namespace mhd
