// qvti_layout.h -- HBM layout constants shared by the setup kernels and the
// pencil kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace qvti {

// Blocked field groups.  A group of nf per-cell fields is stored as 64-cell
// blocks with the fields interleaved: element (f, ip) sits at
// ((ip >> 6) * nf + f) * 64 + (ip & 63).  A thread reaches every field of its
// cell from one address with immediate offsets f * 256 bytes, and the fields
// of 64 neighbouring cells form one contiguous run of nf * 256 bytes.
// A group of N cells takes blk_len(N) floats per field: N rounded up to whole
// blocks (N need not be a multiple of 64: axis lengths such as 18 or 90 are
// supported).
constexpr int kBlk = 64;
__host__ __device__ __forceinline__ long long blk_len(long long n) { return (n + kBlk - 1) / kBlk * kBlk; }
__host__ __device__ __forceinline__ long long blk_index(long long ip, int nf, int f)
{
    return ((ip >> 6) * nf + f) * kBlk + (ip & 63);
}
// Stress family: per velocity component the four fields {A1 w, A2 v, A3 v,
// A2 w} whose derivatives the stress update weighs with the Q coefficients
// (k_coefficients in qvti_aux.h).
constexpr int kFam = 4;
// Medium fields from which the stress update forms the coefficients of the
// moduli sets P, S, H and D (set_coeffs in qvti_aux.h): the speeds c = v
// cos(pi g/2), the low bits of two of them, the gammas and the density in one
// blocked group per cell (the last two: VTI); in natural order the four
// coefficients of S-bar (8-corner averages) and, VTI, the low bits of the other
// two speeds (a ninth field in the group would pass 4 GiB at 512^3).
enum { GM_CP, GM_CS, GM_LOW, GM_GP, GM_GS, GM_RHO, GM_CH, GM_CD };
constexpr int kGM(bool vti) { return vti ? 8 : 6; }
constexpr int kGS(bool vti) { return vti ? kFam + 1 : kFam; }
// constants of the medium and the run (q_coeffs), on the device
struct MediumConst {
    double k0, k2, k3, s4;
    float wa, wb;  // alpha, alpha kappa
};
// x- (y-) derivatives that the stress update reads: the four of the family
// whose component is the axis, and the two S-bar-weighted shear sums
constexpr int kDer = kFam + 2;

// Global memory through a uniform row pointer and a per-lane byte offset.  The
// empty asm keeps the row's address a value of its own in SGPRs, so that the
// access is one instruction with one 32-bit offset register shared by all rows
// (global_load v, v, s[:]; imm, a compile-time byte offset, rides along).  Without it the compiler folds the lane offset into
// the base and keeps a 64-bit address register pair, made by a 64-bit add, for
// every row.  Offsets stay below 4 GiB: within one shot's field (512^3
// floats) or blocked group of at most 8 fields.
typedef __attribute__((address_space(1))) char gchar;
typedef float vfloat2 __attribute__((ext_vector_type(2)));
struct Row {
    gchar* p;
};
template <class T>
__device__ __forceinline__ Row row_at(const T* base, long long elem)
{
    unsigned long long u = reinterpret_cast<unsigned long long>(base + elem);
    asm("" : "+s"(u));
    return Row{(gchar*)u};
}
// The lane offset, made opaque where it is used: the 32-to-64-bit extension
// then sits next to the accesses and folds into them, instead of being hoisted
// out of loops into a register pair.
__device__ __forceinline__ unsigned lane_off(unsigned off)
{
    asm volatile("" : "+v"(off));
    return off;
}
// NT: non-temporal access, for streams that no later kernel finds in a cache
// anyway (kStreamBytes); the caches then keep what is read again soon.  Only
// for whole 128-byte lines: a line that two tiles share must stay in L2 until
// the second one has used it.
template <bool NT = false>
__device__ __forceinline__ float ld1(Row r, unsigned off, int imm = 0)
{
    const auto p = (__attribute__((address_space(1))) const float*)(r.p + off + imm);
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
template <bool NT = false>
__device__ __forceinline__ float2 ld2(Row r, unsigned off, int imm = 0)
{
    const auto p = (__attribute__((address_space(1))) const vfloat2*)(r.p + off + imm);
    vfloat2 v;
    if constexpr (NT) v = __builtin_nontemporal_load(p);
    else v = *p;
    return make_float2(v.x, v.y);
}
template <bool NT = false>
__device__ __forceinline__ void st1(Row r, unsigned off, float v, int imm = 0)
{
    const auto p = (__attribute__((address_space(1))) float*)(r.p + off + imm);
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}
template <bool NT = false>
__device__ __forceinline__ void st2(Row r, unsigned off, float2 v, int imm = 0)
{
    const auto p = (__attribute__((address_space(1))) vfloat2*)(r.p + off + imm);
    vfloat2 w;
    w.x = v.x;
    w.y = v.y;
    if constexpr (NT) __builtin_nontemporal_store(w, p);
    else *p = w;
}
// Bytes a step touches beyond which its fields no longer stay in the 256 MB
// Infinity Cache from one kernel to the next.  A plain copy of 2 GiB runs at
// 5.65 TB/s, a non-temporal one at 5.95 - 6.3; a working set of 64 MB at 7.9
// against 6.4.
constexpr long long kStreamBytes = 256LL << 20;

}  // namespace qvti
