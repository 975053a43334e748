// qvti_kernels.hip -- instantiates the pencil kernels of one build group of
// axis lengths (qvti_lengths.h) and defines their launch records
// (qvti_launch.h).  Compiled once per group with -DQVTI_GROUP=g.
#include "qvti_launch.h"

#ifndef QVTI_GROUP
#error "compile with -DQVTI_GROUP=<build group>"
#endif

namespace qvti {
namespace {

template <class G, int MODE, bool NT>
void l_deriv(dim3 grid, hipStream_t st, const StridedPair& a)
{
    hipLaunchKernelGGL((k2_deriv_strided<G, MODE, NT>), grid, dim3(G::T), 0, st, a);
}
template <class G, bool NT>
void l_stress_xy(dim3 grid, hipStream_t st, const StressXYPair& a)
{
    hipLaunchKernelGGL((k2_stress_xy<G, NT>), grid, dim3(G::T), 0, st, a);
}
template <class G, int DIR, bool NT>
void l_cfft(dim3 grid, hipStream_t st, const CStridedArgs& a)
{
    hipLaunchKernelGGL((k2_cfft_strided<G, DIR, NT>), grid, dim3(G::T), 0, st, a);
}
template <class G, bool KS, bool NT>
void l_xpass(dim3 grid, hipStream_t st, const XPassArgs& a)
{
    hipLaunchKernelGGL((k2_xpass<G, KS, NT>), grid, dim3(G::T), 0, st, a);
}
template <class G, bool INJ>
void l_vel_z(dim3 grid, hipStream_t st, const VelZArgs& a)
{
    hipLaunchKernelGGL((k2_vel_z<G, INJ>), grid, dim3(kThreads), 0, st, a);
}
template <class G, bool NT>
void l_zrows(dim3 grid, hipStream_t st, const ZRowsArgs& a)
{
    hipLaunchKernelGGL((k2_zrows<G, NT>), grid, dim3(kThreads), 0, st, a);
}
template <class G, bool VTI, int NT>
void l_stress_z(dim3 grid, hipStream_t st, const StressZArgs& a)
{
    hipLaunchKernelGGL((k2_stress_z<G, VTI, NT>), grid, dim3(StressTile<G>::T), 0, st, a);
}
template <class G>
void l_deriv_rows(dim3 grid, hipStream_t st, const RowDerivArgs& a)
{
    hipLaunchKernelGGL(k2_deriv_rows<G>, grid, dim3(kThreads), 0, st, a);
}

// Tile width PW of the strided kernels exists for n >= 64 while the tile fits in LDS.
template <int A, int B, int PW>
constexpr bool pw_ok()
{
    if constexpr (PW == 1) return true;
    else return A * B >= 64 && L2<A, B, PW>::kFits;
}

// A non-temporal variant exists where the tile is made of whole 128-byte
// lines, `cols` floats per pencil; elsewhere its entry is the plain kernel.
template <int A, int B, int PW, int COLS>
constexpr bool lines()
{
    return L2<A, B, PW>::P * COLS % 32 == 0;
}

using DerivFn = void (*)(dim3, hipStream_t, const StridedPair&);
using StressXYFn = void (*)(dim3, hipStream_t, const StressXYPair&);
using CfftFn = void (*)(dim3, hipStream_t, const CStridedArgs&);
using XpassFn = void (*)(dim3, hipStream_t, const XPassArgs&);

template <int A, int B, int PW, int MODE, bool NT>
DerivFn deriv_fn()
{
    if constexpr (pw_ok<A, B, PW>()) return &l_deriv<L2<A, B, PW>, MODE, NT && lines<A, B, PW, 2>()>;
    else return nullptr;
}
template <int A, int B, int PW, bool NT>
StressXYFn stress_xy_fn()
{
    if constexpr (pw_ok<A, B, PW>()) return &l_stress_xy<L2<A, B, PW>, NT && lines<A, B, PW, 1>()>;
    else return nullptr;
}
template <int A, int B, int PW, int DIR, bool NT>
CfftFn cfft_fn()
{
    if constexpr (pw_ok<A, B, PW>()) return &l_cfft<L2<A, B, PW>, DIR, NT && lines<A, B, PW, 2>()>;
    else return nullptr;
}
template <int A, int B, int PW, bool KS, bool NT>
XpassFn xpass_fn()
{
    if constexpr (pw_ok<A, B, PW>()) return &l_xpass<L2<A, B, PW>, KS, NT && lines<A, B, PW, 2>()>;
    else return nullptr;
}
template <int A, int B, int PW>
constexpr int pencils()
{
    if constexpr (pw_ok<A, B, PW>()) return L2<A, B, PW>::P;
    else return 0;
}

// tile widths PW of width index 0, 1, 2
constexpr int kW0 = 1, kW1 = 2, kW2 = 4;

// Built at load time (dynamic initialisation), so that every launch function
// whose address the record holds is instantiated and emitted.
template <int A, int B>
LenOps make_ops()
{
    using G = L2<A, B, 1>;
    constexpr int kNt = A * B % 32 == 0 ? 1 : 0;  // rows of whole 128-byte lines
#define QVTI_WIDTHS(fn, ...) {fn<A, B, kW0, __VA_ARGS__>(), fn<A, B, kW1, __VA_ARGS__>(), fn<A, B, kW2, __VA_ARGS__>()}
#define QVTI_WIDTHS_NT(fn, ...) {QVTI_WIDTHS(fn, __VA_ARGS__, false), QVTI_WIDTHS(fn, __VA_ARGS__, true)}
    return LenOps{
        A * B, A, B, G::P, StressTile<G>::R,
        {pencils<A, B, kW0>(), pencils<A, B, kW1>(), pencils<A, B, kW2>()},
        {L2<A, B, kW0>::T, L2<A, B, kW1>::T, L2<A, B, kW2>::T},
        deriv_fn<A, B, kW0, MODE_STORE, false>(),
        QVTI_WIDTHS_NT(deriv_fn, MODE_VEL),
        {QVTI_WIDTHS(stress_xy_fn, false), QVTI_WIDTHS(stress_xy_fn, true)},
        {QVTI_WIDTHS_NT(cfft_fn, -1), QVTI_WIDTHS_NT(cfft_fn, 1)},
        {QVTI_WIDTHS_NT(xpass_fn, false), QVTI_WIDTHS_NT(xpass_fn, true)},
        {&l_vel_z<G, false>, &l_vel_z<G, true>},
        {&l_zrows<G, false>, &l_zrows<G, kNt != 0>},
        {{&l_stress_z<G, false, 0>, &l_stress_z<G, false, kNt * 1>, &l_stress_z<G, false, kNt * 2>},
         {&l_stress_z<G, true, 0>, &l_stress_z<G, true, kNt * 1>, &l_stress_z<G, true, kNt * 2>}},
        &l_deriv_rows<G>,
    };
#undef QVTI_WIDTHS
#undef QVTI_WIDTHS_NT
}

}  // namespace

#define QVTI_DEFINE_IN_GROUP(n, a, b, g) QVTI_DEFINE_IN_GROUP_##g(n, a, b)
#define QVTI_DEFINE_LEN(n, a, b) const LenOps kLenOps_##n = make_ops<a, b>();
#define QVTI_SKIP_LEN(n, a, b)
#if QVTI_GROUP == 0
#define QVTI_DEFINE_IN_GROUP_0 QVTI_DEFINE_LEN
#else
#define QVTI_DEFINE_IN_GROUP_0 QVTI_SKIP_LEN
#endif
#if QVTI_GROUP == 1
#define QVTI_DEFINE_IN_GROUP_1 QVTI_DEFINE_LEN
#else
#define QVTI_DEFINE_IN_GROUP_1 QVTI_SKIP_LEN
#endif
#if QVTI_GROUP == 2
#define QVTI_DEFINE_IN_GROUP_2 QVTI_DEFINE_LEN
#else
#define QVTI_DEFINE_IN_GROUP_2 QVTI_SKIP_LEN
#endif
#if QVTI_GROUP == 3
#define QVTI_DEFINE_IN_GROUP_3 QVTI_DEFINE_LEN
#else
#define QVTI_DEFINE_IN_GROUP_3 QVTI_SKIP_LEN
#endif
#if QVTI_GROUP == 4
#define QVTI_DEFINE_IN_GROUP_4 QVTI_DEFINE_LEN
#else
#define QVTI_DEFINE_IN_GROUP_4 QVTI_SKIP_LEN
#endif
#if QVTI_GROUP == 5
#define QVTI_DEFINE_IN_GROUP_5 QVTI_DEFINE_LEN
#else
#define QVTI_DEFINE_IN_GROUP_5 QVTI_SKIP_LEN
#endif
#if QVTI_GROUP == 6
#define QVTI_DEFINE_IN_GROUP_6 QVTI_DEFINE_LEN
#else
#define QVTI_DEFINE_IN_GROUP_6 QVTI_SKIP_LEN
#endif
#if QVTI_GROUP == 7
#define QVTI_DEFINE_IN_GROUP_7 QVTI_DEFINE_LEN
#else
#define QVTI_DEFINE_IN_GROUP_7 QVTI_SKIP_LEN
#endif

QVTI_LENGTHS(QVTI_DEFINE_IN_GROUP)

#define QVTI_ALT_IN_GROUP(n, a, b, g) QVTI_DEFINE_IN_GROUP_##g(Alt_##n, a, b)
QVTI_ALT_LENGTHS(QVTI_ALT_IN_GROUP)

}  // namespace qvti
