// qvti_pencils.h -- pencil kernels of the time step on the two-level register
// FFT (qvti_fft2l.h).  Every kernel is a template over the split G = L2<N1,N2,PW>
// of its axis length; the row (z) kernels run 256 threads, the strided-axis
// (x, y) kernels up to 256*PW (the tile width the autotuner picks).
//
// Per step (reference loop: cuviscoelas_3D.cu:1255-1605):
//   velocity half-step   k2_deriv_strided (x and y; advances the step counter)
//                        -> k2_vel_z (z-derivatives, velocity update, forward z-FFTs of v and w)
//   stress half-step     k2_cfft_strided(y, fwd) -> k2_xpass -> k2_cfft_strided(y, inv)
//                        -> k2_zrows (inverse z; receivers) -> k2_stress_xy (x and y)
//                        -> k2_stress_z (z-derivatives, stress update, source injection)
// The x and the y derivatives are independent: one launch takes both where the
// two axes have one length (and so one kernel), two launches elsewhere.
//
// Algebra used (exact in exact arithmetic; only rounding differs from the
// reference's C2C + `.x / ntp` formulation):
//  * every spectral operator of the scheme is Hermitian (real |k|^p times a
//    1-D shift-derivative whose Nyquist symbol is taken as its real part,
//    which is what `.x` of the C2C result keeps), so two real fields packed
//    as a + ib go through ONE complex transform and come back as op(a) + i op(b);
//  * an operator acting along one axis only (all nine velocity-step
//    derivatives and the A2 = 1 stress terms) is a 1-D transform along that
//    axis: the other two axes' forward and inverse transforms cancel;
//  * A_j D_a V = D_a (A_j V): the 45 stress terms are 1-D derivatives of the
//    12 fields {A1 w, v, A3 v, w} per component, w = alpha (v + kappa dv) with
//    dv = v - v_prev in real space (v_prev: the previous step's pre-injection
//    velocity): the coefficients of A1 v and A1 dv are in one ratio kappa
//    everywhere (q_coeffs in qvti_aux.h), so only A1 w and A3 v need the full
//    3-D transform - three forward and four inverse complex transforms.  With
//    five fields {A1 v, v, A3 v, A1 dv, dv} per component it was three and
//    five, and 248 floats per cell and step instead of 188 (VTI, with the
//    coefficients of set_coeffs and the shear sums of k2_stress_xy, each field
//    of a launch counted once; 196 with the second reads of S-bar there).
//    Fields that share a complex transform are scaled (alpha and the length
//    scale of A1 and A3, powers of two) so that the FP32 rounding of one does
//    not swamp the other where it matters (q_coeffs).
#pragma once
#include "qvti_aux.h"
#include "qvti_fft2l.h"
#include "qvti_layout.h"

namespace qvti {

constexpr int kThreads = 256;
#ifndef QVTI_STRIDED_WAVES
#define QVTI_STRIDED_WAVES 1
#endif
#ifndef QVTI_XPASS_WAVES
#define QVTI_XPASS_WAVES 1
#endif
// minimum waves per SIMD the z-row kernels are compiled for (1: no bound on
// their registers; 4 caps them at 128 VGPRs, the occupancy their LDS allows;
// the stress update takes 137 without at n = 160, 192, 288 and 320, none of its
// lengths spills with: 160^3 188 -> 174 us, 192^3 287 -> 269 us)
#ifndef QVTI_VELZ_WAVES
#define QVTI_VELZ_WAVES 1
#endif
#ifndef QVTI_STRESSZ_WAVES
#define QVTI_STRESSZ_WAVES 4
#endif
enum { MODE_STORE = 0, MODE_VEL = 1 };

// Elements per chunk of the C-PML epilogues: a divisor of the thread's N1
// elements, about 4 (more would hold more loads in registers than they overlap).
constexpr int vel_chunk(int n1)
{
    return n1 % 4 == 0 ? 4 : (n1 % 5 == 0 ? 5 : (n1 % 3 == 0 ? 3 : 1));
}

// XCD-aware placement of (row tile, shot) on a 1-D grid of
// ceil(ntiles / (8 run)) * 8 run * nshots workgroups.  Workgroup ids are dealt
// round-robin to the 8 XCDs; id = ((c run + k) nshots + shot) 8 + x runs tile
// (8 c + x) run + k on XCD x.  So
//  * the shots of one row tile run on the same XCD (same L2), dispatched
//    close together, and the model fields they all read (coefficients,
//    buoyancies) come from cache after the first shot;
//  * `run` consecutive row tiles run on one XCD, one after another, so the
//    128-byte lines (and 64-cell blocks) that neighbouring tiles share when a
//    tile does not end on a line or block boundary are fetched from HBM once.
// Returns tile = -1 for the padding workgroups.
struct TileShot {
    int tile, shot;
};
__device__ __forceinline__ TileShot tile_shot(int ntiles, int nshots, int run)
{
    const int id = blockIdx.x;
    const int x = id & 7, q = id >> 3;
    const int ck = q / nshots, shot = q - ck * nshots;
    const int c = ck / run, k = ck - c * run;
    const int t = (c * 8 + x) * run + k;
    return {t < ntiles ? t : -1, shot};
}

// (plane, z-tile) of a strided-axis workgroup.  run = 0: blockIdx.x =
// plane * ztiles + tile.  run >= 1: XCD-aware placement on a 1-D grid of
// ceil(nplanes / (8 run)) * 8 run * ztiles workgroups, id = ((c run + k)
// ztiles + zt) 8 + x running (plane (8 c + x) run + k, z-tile zt) on XCD x:
// the z-tiles of one plane, and `run` consecutive planes, run on the same XCD
// (same L2) one after another, so the 128-byte lines that neighbouring tiles
// share - within a row when a tile's rows do not end on a line boundary, and
// between the end of a row and the start of the next plane's row - are
// fetched from HBM once.  plane = -1 for the padding workgroups.
struct PlaneTile {
    int plane, zt;
};
__device__ __forceinline__ PlaneTile plane_tile(int ztiles, int nplanes, int run, int id)
{
    if (!run) {
        const int pl = id / ztiles;
        return {pl, id - pl * ztiles};
    }
    const int x = id & 7, q = id >> 3;
    const int pk = q / ztiles, zt = q - pk * ztiles;
    const int c = pk / run, k = pk - c * run;
    const int pl = (c * 8 + x) * run + k;
    return {pl < nplanes ? pl : -1, zt};
}

template <class G>
__device__ __forceinline__ void load_twiddles(float2* tws, const float2* tw)
{
    for (int t = threadIdx.x; t < G::TWN; t += G::T) twiddle_entry<G>(tws, tw, t);
}

// ------------------------------------------------------------------------
// 1-D shift-derivatives of real fields along a strided axis (x or y).  Tile:
// G::P complex pencils = 2*G::P adjacent real z-columns at one value of the
// other in-plane index, loaded as float2 (two real pencils per complex one).
// Modes: STORE out = d (standalone derivative); VEL out = d + phi, with the
// velocity C-PML memory variable phi updated on the axis' face slabs
// (cuviscoelas_3D.cu:1049-1074).  A launch takes one or two axes (of one
// length), which fill the chip together: at 64^3 an axis' 192 workgroups leave
// a quarter of the CUs without one.
struct DJob {
    const float* in;
    float* out;
    float* phi;
    int sym;   // 0: D+, 1: D-
    int half;  // 1: half-cell averaged C-PML a, b
};

struct StridedArgs {
    int nx, ny, nz, pml;
    long long sx, sy;
    int axis;  // 0: x (stride sx), 1: y (stride sy)
    int ztiles, nplanes, run;  // workgroup placement: plane_tile()
    int mode;
    float dt;
    long long shot_stride, slab_stride;
    const float2* tw;
    const float2* sym[2];
    const float *pa, *pb, *pah, *pbh;
    int njobs;
    // step counter advanced by this launch (the first kernel of a step), or null
    int* tick;
    DJob job[3];
};
struct StridedPair {
    StridedArgs a[2];
    int jz;  // workgroups per tile and axis; grid z: (axis, job)
};

// NT: non-temporal loads and stores (stream_nt)
template <class G, int MODE, bool NT>
__global__ __launch_bounds__(G::T) __attribute__((amdgpu_waves_per_eu(QVTI_STRIDED_WAVES)))
void k2_deriv_strided(StridedPair pr)
{
    const int sel = blockIdx.z / pr.jz, jb0 = blockIdx.z - sel * pr.jz;
    const StridedArgs& a = pr.a[sel];
    __shared__ float2 lds[G::P * G::PS];
    __shared__ float2 tws[G::TWN];
    const int tid = threadIdx.x, shot = blockIdx.y;
    // one thread of the grid advances the step counter; the kernels of the
    // step that read it run after this one
    if (a.tick != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && tid == 0) *a.tick = *a.tick + 1;
    const PlaneTile pt = plane_tile(a.ztiles, a.nplanes, a.run, blockIdx.x);
    if (pt.plane < 0) return;
    const int other = pt.plane;
    const int p = tid % G::P, jj = tid / G::P;
    const int zc = pt.zt * 2 * G::P + 2 * p;
    // scalars of the chosen axis in registers: read through `a` they would be
    // loaded again at every use below
    const int nx = a.nx, ny = a.ny, nz = a.nz, axis = a.axis, pml = a.pml;
    const float dt = a.dt;
    const bool zok = zc < nz;
    // columns past nz (last tile of a ragged z) load a valid column and are
    // never stored, so the loads need no branch
    const int zl = zok ? zc : nz - 2;
    const bool act1 = jj < G::N2, act2 = jj < G::N1;
    // uniform per-block base (SGPRs) + 32-bit per-thread element offsets
    const int astride = (int)(axis == 0 ? a.sx : a.sy);
    const long long poff = axis == 0 ? (long long)other * a.sy : (long long)other * a.sx;  // plane offset in the shot
    const long long ubase = (long long)shot * a.shot_stride + poff;
    const unsigned lvoff = 4u * (unsigned)(jj * astride + zl);  // lane byte offset from a uniform row
    float2* pen = lds + p * G::PS;
    load_twiddles<G>(tws, a.tw);
    for (int jb = jb0; jb < a.njobs; jb += pr.jz) {
        const DJob J = a.job[jb];
        __syncthreads();
        if (act1) {
            float2 v[G::N1];
            const unsigned o = lane_off(lvoff);
#pragma unroll
            for (int j1 = 0; j1 < G::N1; ++j1)
                v[j1] = ld2<NT>(row_at(J.in, ubase + (long long)(j1 * G::N2) * astride), o);
            fwd_l1<G>(v, pen, tws, jj);
        }
        __syncthreads();
        float2 b[G::N2];
        if (act2) {
            fwd_l2<G>(b, pen, jj);
            const Row S = row_at(a.sym[J.sym], 0);
            const unsigned o = lane_off(8u * jj);
#pragma unroll
            for (int k2 = 0; k2 < G::N2; ++k2) b[k2] = c_mul(b[k2], ld2(S, o, 8 * G::N1 * k2));
        }
        __syncthreads();
        if (act2) inv_la<G>(b, pen, tws + G::T2OFF, jj);
        __syncthreads();
        if (MODE == MODE_STORE) {
            if (act1 && zok) {
                float2 d[G::N1];
                inv_lb<G>(d, pen, jj);
                const unsigned o = lane_off(lvoff);
#pragma unroll
                for (int j1 = 0; j1 < G::N1; ++j1)
                    st2(row_at(J.out, ubase + (long long)(G::N2 * j1) * astride), o, d[j1]);
            }
        } else {
            // The C-PML branch differs per element: park the pencil's result in
            // its own LDS slots (natural order) and finish element by element,
            // which keeps the register footprint at the FFT's.
            float2 d[G::N1];
            if (act1 && zok) inv_lb<G>(d, pen, jj);
            __syncthreads();
            if (act1 && zok) {
#pragma unroll
                for (int j1 = 0; j1 < G::N1; ++j1) pen[jj + G::N2 * j1] = d[j1];
                constexpr int n = G::N;
                // an opaque copy of the lane's row index: keeps the per-element
                // C-PML indices and table loads inside the job loop instead of
                // being hoisted (and held in registers through the FFTs)
                int jl = jj;
                asm volatile("" : "+v"(jl));
                const unsigned o = lane_off(lvoff);  // (zok: zl == zc)
                const Row pa = row_at(J.half ? a.pah : a.pa, 0), pb = row_at(J.half ? a.pbh : a.pb, 0);
                const Row phs = row_at(J.phi, (long long)shot * a.slab_stride);
                // Chunks of CH elements: every load of a chunk (unconditional
                // and in bounds - a non-slab element reads slab plane 0) before
                // its stores, so the chunk's memory round trips overlap.
                constexpr int CH = vel_chunk(G::N1);
#pragma unroll
                for (int c0 = 0; c0 < G::N1; c0 += CH) {
                    float2 rr[CH], q[CH];
                    unsigned sidx[CH];
                    bool upd[CH];
#pragma unroll
                    for (int jc = 0; jc < CH; ++jc) {
                        const int j1 = c0 + jc;
                        const int i = jl + G::N2 * j1;
                        float2 r = pen[i];
                        const int ix = axis == 0 ? i : other;
                        const int iy = axis == 0 ? other : i;
                        upd[jc] = (i < pml || i >= n - pml) && ix < nx - 1 && iy < ny - 1;
                        const int si = i < pml ? i : (i >= n - pml ? i - (n - 2 * pml) : 0);
                        sidx[jc] = 4u * (unsigned)((axis == 0 ? si * ny + iy : ix * 2 * pml + si) * nz + zc);
                        const float2 q0 = ld2(phs, sidx[jc]);
                        const float A = ld1(pa, 4u * jl, 4 * G::N2 * j1), B = ld1(pb, 4u * jl, 4 * G::N2 * j1);
                        q[jc] = q0;
                        if (upd[jc]) {
                            if (zc < nz - 1) { q[jc].x = q0.x + dt * (-A * q0.x - B * r.x); r.x = r.x + q[jc].x; }
                            if (zc + 1 < nz - 1) { q[jc].y = q0.y + dt * (-A * q0.y - B * r.y); r.y = r.y + q[jc].y; }
                        }
                        rr[jc] = r;
                    }
#pragma unroll
                    for (int jc = 0; jc < CH; ++jc)
                        if (upd[jc]) st2(phs, sidx[jc], q[jc]);
#pragma unroll
                    for (int jc = 0; jc < CH; ++jc)
                        st2<NT>(row_at(J.out, ubase + (long long)(G::N2 * (c0 + jc)) * astride), o, rr[jc]);
                    asm volatile("" ::: "memory");  // the next chunk's loads stay after this chunk
                }
            }
        }
    }
}

// ------------------------------------------------------------------------
// Stress half-step: derivatives of the family fields along a strided axis.
// Tile: G::P adjacent z-columns at one value of the other in-plane index, one
// complex pencil per column: a pass transforms two fields of one component,
// (A1 w + i A2 w) or (A2 v + i A3 v).  A job of one pass stores the two
// derivatives; a job of two passes stores the one real field
//   sum_j S-bar_j D(in_j)
// of the component's four derivatives, the only form in which the stress
// update uses the shear derivatives: six fields per axis go to HBM and back
// instead of twelve, for four coefficient fields that each of the two sums
// reads (24 -> 26 floats per cell and axis here, 22 with S-bar counted once;
// 61 -> 49 in the stress update).  Pairing fields, and not two columns of one
// field as k2_deriv_strided does, halves the passes of a sum and the
// accumulators that live through the transforms (N1 instead of 2 N1 registers).
struct SJob {
    const float* re[2];
    const float* im[2];
    int n;    // passes: 1 or 2
    int sym;  // 0: D+, 1: D-
    int out[2];  // n = 1: fields of the output group; n = 2: out[0] the sum's field
};

struct StressXYArgs {
    int nz;
    long long sx, sy;
    int axis;  // 0: x (stride sx), 1: y (stride sy)
    int ztiles, nplanes, run;  // workgroup placement: plane_tile()
    long long shot_stride;
    const float2* tw;
    const float2* sym[2];
    const float* gs;  // S-bar coefficients [kFam][N]
    long long N;
    float* out;       // blocked group [shot][N/64][kDer][64]
    // per-shot length of a blocked group's field: N rounded up to whole 64-cell blocks
    long long blk_stride;
    int njobs;
    SJob job[4];
};
struct StressXYPair {
    StressXYArgs a[2];  // one or two axes of one length
    int jz;             // workgroups per tile and axis; grid z: (axis, job)
    int nshots;         // shots interleaved on grid x, or 1
};

// NT: non-temporal field loads and stores (stream_nt).
// What bounds it: 52 floats per cell for both axes (each sum reads S-bar).
// 256^3: 680 us, 5.1 TB/s, the rate of the memory at 20 streams; 400x400x200:
// 1790 us, 3.7 TB/s, 3 waves per SIMD and rows that end mid-line.  The bounds:
// one axis at 256^3, before the streaming, took 370-375 us with 2, 3 and 4
// waves per SIMD; at 400x400x200 3 waves were best (985 us; 1045 us with 2).
// Some splits spill under them: 256 and 240 up to 6 VGPRs, 480 to 512 from 5 to
// 73 by tile width; other bounds were not timed there.  A whole step of
// 480x480x32, 500x500x32, 512x512x128 takes 1.39, 1.68, 6.76 ms (1.96, 2.12,
// 7.77 ms when every derivative was stored).
template <class G, bool NT>
__global__ __launch_bounds__(G::T) __attribute__((amdgpu_waves_per_eu(G::NMAX <= 16 ? 4 : 3)))
void k2_stress_xy(StressXYPair pr)
{
    const int sel = blockIdx.z / pr.jz, jb0 = blockIdx.z - sel * pr.jz;
    const StressXYArgs& a = pr.a[sel];
    __shared__ float2 lds[G::P * G::PS];
    __shared__ float2 tws[G::TWN];
    const int tid = threadIdx.x;
    // pr.nshots > 1: the shots of one tile follow each other on one XCD (as
    // tile_shot), so the S-bar values are read from its L2 after the first
    // shot; 1: the shots are on grid y (stress_xy_shots)
    const int q = (int)(blockIdx.x >> 3) / pr.nshots, shot = (int)blockIdx.y + (int)(blockIdx.x >> 3) - q * pr.nshots;
    const PlaneTile pt = plane_tile(a.ztiles, a.nplanes, a.run, q * 8 + (int)(blockIdx.x & 7));
    if (pt.plane < 0) return;
    const int other = pt.plane;
    const int p = tid % G::P, jj = tid / G::P;
    const int zc = pt.zt * G::P + p;
    const int nz = a.nz;
    const bool zok = zc < nz;
    // columns past nz (last tile of a ragged z) load a valid column and are
    // never stored, so the loads need no branch
    const int zl = zok ? zc : nz - 1;
    const bool act1 = jj < G::N2, act2 = jj < G::N1;
    const int astride = (int)(a.axis == 0 ? a.sx : a.sy);
    const long long poff = a.axis == 0 ? (long long)other * a.sy : (long long)other * a.sx;
    const long long ubase = (long long)shot * a.shot_stride + poff;
    const unsigned lvoff = 4u * (unsigned)(jj * astride + zl);  // lane byte offset from a uniform row
    float2* pen = lds + p * G::PS;
    load_twiddles<G>(tws, a.tw);
    for (int jb = jb0; jb < a.njobs; jb += pr.jz) {
        const int np = a.job[jb].n;
        float acc[G::N1];
#pragma unroll
        for (int j1 = 0; j1 < G::N1; ++j1) acc[j1] = 0.f;
#pragma unroll 1
        for (int f = 0; f < np; ++f) {
            const float* re = a.job[jb].re[f] + ubase;
            const float* im = a.job[jb].im[f] + ubase;
            __syncthreads();
            if (act1) {
                float2 v[G::N1];
                const unsigned o = lane_off(lvoff);
#pragma unroll
                for (int j1 = 0; j1 < G::N1; ++j1) {
                    const long long row = (long long)(j1 * G::N2) * astride;
                    v[j1] = make_float2(ld1<NT>(row_at(re, row), o), ld1<NT>(row_at(im, row), o));
                }
                fwd_l1<G>(v, pen, tws, jj);
            }
            __syncthreads();
            float2 b[G::N2];
            if (act2) {
                fwd_l2<G>(b, pen, jj);
                const Row S = row_at(a.sym[a.job[jb].sym], 0);
                const unsigned o = lane_off(8u * jj);
#pragma unroll
                for (int k2 = 0; k2 < G::N2; ++k2) b[k2] = c_mul(b[k2], ld2(S, o, 8 * G::N1 * k2));
            }
            __syncthreads();
            if (act2) inv_la<G>(b, pen, tws + G::T2OFF, jj);
            // The S-bar values of a sum are loaded here, ahead of the last
            // exchange: their round trip overlaps the barrier and the inverse
            // transform.  Fields of the pass: (0, 3) for (A1 w, A2 w), (1, 2)
            // for (A2 v, A3 v).
            float2 c[G::N1];
            if (np > 1 && act1) {
                const float* g0 = a.gs + f * a.N + poff;
                const float* g1 = a.gs + (kFam - 1 - f) * a.N + poff;
                const unsigned o = lane_off(lvoff);
#pragma unroll
                for (int j1 = 0; j1 < G::N1; ++j1) {
                    const long long row = (long long)(j1 * G::N2) * astride;
                    c[j1] = make_float2(ld1(row_at(g0, row), o), ld1(row_at(g1, row), o));
                }
            }
            __syncthreads();
            if (act1 && zok) {
                float2 d[G::N1];
                inv_lb<G>(d, pen, jj);
                if (np == 1) {
                    const Row ore = row_at(a.out, (long long)shot * kDer * a.blk_stride + a.job[jb].out[0] * kBlk);
                    const Row oim = row_at(a.out, (long long)shot * kDer * a.blk_stride + a.job[jb].out[1] * kBlk);
                    const unsigned ip0 = lane_off((unsigned)(poff + jj * astride + zc));
#pragma unroll
                    for (int j1 = 0; j1 < G::N1; ++j1) {
                        const unsigned ip = ip0 + (unsigned)(G::N2 * j1 * astride);
                        const unsigned o = 4u * ((ip >> 6) * (unsigned)(kBlk * kDer) + (ip & 63u));
                        st1<NT>(ore, o, d[j1].x);
                        st1<NT>(oim, o, d[j1].y);
                    }
                } else {
#pragma unroll
                    for (int j1 = 0; j1 < G::N1; ++j1) acc[j1] += c[j1].x * d[j1].x + c[j1].y * d[j1].y;
                }
            }
        }
        if (np > 1 && act1 && zok) {
            const Row ob = row_at(a.out, (long long)shot * kDer * a.blk_stride + a.job[jb].out[0] * kBlk);
            const unsigned ip0 = lane_off((unsigned)(poff + jj * astride + zc));
#pragma unroll
            for (int j1 = 0; j1 < G::N1; ++j1) {
                const unsigned ip = ip0 + (unsigned)(G::N2 * j1 * astride);
                st1<NT>(ob, 4u * ((ip >> 6) * (unsigned)(kBlk * kDer) + (ip & 63u)), acc[j1]);
            }
        }
    }
}

// ------------------------------------------------------------------------
// Velocity update (cuviscoelas_3D.cu:1018-1101) fused with the z-derivatives
// and with the first (z) pass of the stress step's 3-D transform:
//   v += b * (acc_xy + dz sigma + phi_z);  dv = v_new - v_old + src_prev;
//   w = alpha v + (alpha kappa) dv;
//   P0 = FFT_z(wx + i wy), P1 = FFT_z(wz + i vz), P2 = FFT_z(vx + i vy)
// Two workgroups per tile (grid y): vx and vy with P0 and P2, and vz with P1.
// They share nothing but the twiddles, and the chain of dependent transforms,
// which bounds the kernel where a grid has few tiles, is a third shorter:
// 64^3 20 -> 15 us, 160x160x128 78 -> 73 us, 256^3 349 -> 343 us (27 floats per
// cell, 5.3 TB/s: the memory bounds it there), 400x400x200 751 -> 738 us.
// dv is the change since the previous step's pre-injection velocity (the
// reference's V - V_prev, cuviscoelas_3D.cu:517-522, 1124-1131, without 1/dt).
// Tile: G::P rows (z-pencils).
struct VelZArgs {
    int nx, ny, nz, pml;
    int ntiles, nshots, run;  // grid: tile_shot()
    long long nrows;
    float dt;
    long long shot_stride, slab_stride;
    const float2* tw;
    const float2 *symp, *symm;
    const float *pa, *pb, *pah, *pbh;
    const float *pxz, *pyz, *pzz;
    const float *accx[3], *accy[3];  // x and y derivatives (+ phi)
    float* v[3];
    float* w[3];
    const MediumConst* med;
    float2* P[3];
    const float* buoy[3];
    float* phi[3];  // z-slab: phi_pxz_z (node), phi_pyz_z (node), phi_pzz_z (half)
    const int* src_kind;
    const long long* src_ip;
    const float* rik;
    const int* it;
    // extra point sources added to v after the previous step (the receiver
    // side of a reverse-time migration): dense [3][shot][N], zero away from
    // the injection cells; they enter dv like the shot's own source
    // (k2_vel_z<G, true> only)
    const float* inj[3];
};

// Velocity update of one component on the thread's level-1 elements of one
// row (iz = j + N2*j1), from its z-derivative d (real or imaginary part):
// C-PML memory variable on the z-slab, v += b * (acc + dz + phi), dv = v_new
// - v_old (+ the previous step's source at the injection cell), w = wa v +
// wb dv.  Writes v and w (rows with rowdom / ok1 only), returns (v_new, w).
// v, w, accx, accy, bu, inj: uniform tile bases, `row` the byte offset of the lane's
// row in them; ph: the shot's z-slabs, phrow the byte offset of the row's
// 2*pml values.
template <class G, bool INJ>
__device__ __forceinline__ void vz_component(float2 (&out)[G::N1], const float2 (&d)[G::N1], const bool imag,
                                             const Row v, const Row w, const float wa, const float wb, const Row accx,
                                             const Row accy, const Row bu, const Row ph, const unsigned phrow, const Row pa,
                                             const Row pb, const unsigned row, const int j, const int pml,
                                             const float dt, const bool rowdom, const bool ok1, const int src_iz,
                                             const float sprev, const Row inj)
{
    constexpr int n = G::N;
    // opaque per call: nothing is shared (and held) across components
    const int jl = (int)lane_off((unsigned)j);
    const unsigned o = lane_off(row + 4u * j);
    // all loads and arithmetic first (every load unconditional and in bounds:
    // ph is a valid slab row even where it is not used), all stores after, so
    // no load waits behind a store or a branch
    // (in chunks, to bound the registers in flight: up to 10 elements at once
    // - n = 128: 53 -> 51 us at 128^3 against chunks of 4 - else as vel_chunk,
    // 355 us at 256^3 against 368 us with all 16 at once)
    constexpr int CH = G::N1 <= 10 ? G::N1 : vel_chunk(G::N1);
#pragma unroll
    for (int c0 = 0; c0 < G::N1; c0 += CH) {
    float qn[CH];
#pragma unroll
    for (int jc = 0; jc < CH; ++jc) {
        const int j1 = c0 + jc, im = 4 * G::N2 * j1;
        const int iz = jl + G::N2 * j1;
        const float vold = ld1(v, o, im), bb = ld1(bu, o, im);
        const float ac = ld1(accx, o, im) + ld1(accy, o, im);
        const bool slab = iz < pml || iz >= n - pml;
        const int si = iz < pml ? iz : (iz >= n - pml ? iz - (n - 2 * pml) : 0);
        const float q0 = ld1(ph, phrow + 4u * si), A = ld1(pa, 4u * jl, im), B = ld1(pb, 4u * jl, im);
        const bool upd = rowdom && iz < n - 1;
        float dz = imag ? d[j1].y : d[j1].x;
        qn[jc] = q0 + dt * (-A * q0 - B * dz);
        if (upd && slab) dz = dz + qn[jc];
        const float vnew = upd ? vold + bb * (ac + dz) : vold;
        float dvv = vnew - vold;
        if (iz == src_iz) dvv += sprev;
        if constexpr (INJ) dvv += ld1(inj, o, im);
        out[j1] = make_float2(vnew, wa * vnew + wb * dvv);
    }
#pragma unroll
    for (int jc = 0; jc < CH; ++jc) {
        const int j1 = c0 + jc, im = 4 * G::N2 * j1;
        const int iz = jl + G::N2 * j1;
        const bool upd = rowdom && iz < n - 1;
        if (upd && (iz < pml || iz >= n - pml)) st1(ph, phrow + 4u * (iz < pml ? iz : iz - (n - 2 * pml)), qn[jc]);
        if (upd) st1(v, o, out[j1].x, im);
        if (ok1) st1(w, o, out[j1].y, im);
    }
    asm volatile("" ::: "memory");  // the next chunk's loads stay after this chunk
    }
}

template <class G, bool INJ>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(QVTI_VELZ_WAVES))) void k2_vel_z(VelZArgs a)
{
    __shared__ float2 lds[G::P * G::PS];
    __shared__ float2 tws[G::TWN];
    constexpr int n = G::N;
    const TileShot ts = tile_shot(a.ntiles, a.nshots, a.run);
    if (ts.tile < 0) return;  // padding workgroup (whole workgroup, before any barrier)
    const int tid = threadIdx.x, shot = ts.shot;
    // level 1/B mapping (column j fastest) and level 2/A mapping (row k1 fastest)
    const int j = tid % G::N2, p1 = tid / G::N2;
    const int k1 = tid % G::N1, p2 = tid / G::N1;
    const bool act1 = p1 < G::P, act2 = p2 < G::P;
    const long long r0 = (long long)ts.tile * G::P;
    const long long r1 = r0 + p1, r2 = r0 + p2;
    const bool ok1 = act1 && r1 < a.nrows, ok2 = act2 && r2 < a.nrows;
    // uniform block base (shot + first row) and unsigned 32-bit lane offsets;
    // rows past the end (ragged last block) read row r0 and store nothing
    const long long ubase = (long long)shot * a.shot_stride + r0 * n;
    const unsigned lrow1 = ok1 ? 4u * (unsigned)(p1 * n) : 0u;
    float2* pen1 = lds + p1 * G::PS;
    float2* pen2 = lds + p2 * G::PS;
    load_twiddles<G>(tws, a.tw);

    // derivative of (fa + i fb) along z with symbol S, result in d (level-1 layout)
    auto deriv = [&](const float* fa, const float* fb, const float2* S, float2 (&d)[G::N1]) {
        __syncthreads();
        if (act1) {
            float2 v[G::N1];
            const unsigned o = lane_off(lrow1 + 4u * j);
            const Row ra = row_at(fa, ubase), rb = row_at(fb ? fb : fa, ubase);
#pragma unroll
            for (int j1 = 0; j1 < G::N1; ++j1)
                v[j1] = make_float2(ld1(ra, o, 4 * G::N2 * j1), fb ? ld1(rb, o, 4 * G::N2 * j1) : 0.f);
            fwd_l1<G>(v, pen1, tws, j);
        }
        __syncthreads();
        float2 b[G::N2];
        if (act2) {
            fwd_l2<G>(b, pen2, k1);
            const Row sy = row_at(S, 0);
            const unsigned o = lane_off(8u * k1);
#pragma unroll
            for (int k2 = 0; k2 < G::N2; ++k2) b[k2] = c_mul(b[k2], ld2(sy, o, 8 * G::N1 * k2));
        }
        __syncthreads();
        if (act2) inv_la<G>(b, pen2, tws + G::T2OFF, k1);
        __syncthreads();
        if (act1) inv_lb<G>(d, pen1, j);
    };

    const int it = *a.it;
    const int kind = a.src_kind[shot];
    const long long sip = a.src_ip[shot];
    const float sprev = it > 0 ? a.rik[it - 1] : 0.f;
    const float wa = a.med->wa, wb = a.med->wb;
    const int ix = (int)(r1 / a.ny), iy = (int)(r1 - (long long)ix * a.ny);
    const bool rowdom = ok1 && ix < a.nx - 1 && iy < a.ny - 1;
    const unsigned slab_row = ok1 ? (unsigned)(r1 * 2 * a.pml) * 4u : 0u;

    // component c on this thread's elements of its row
    auto update = [&](float2 (&out)[G::N1], const float2 (&d)[G::N1], int c, bool imag) {
        const int src_iz = (kind == c && sip >= r1 * n && sip < (r1 + 1) * n) ? (int)(sip - r1 * n) : -1;
        const bool h = c == 2;
        const Row v = row_at(a.v[c], ubase);
        vz_component<G, INJ>(out, d, imag, v, row_at(a.w[c], ubase), wa, wb, row_at(a.accx[c], ubase),
                        row_at(a.accy[c], ubase),
                        row_at(a.buoy[c], r0 * n), row_at(a.phi[c], (long long)shot * a.slab_stride), slab_row,
                        row_at(h ? a.pah : a.pa, 0), row_at(h ? a.pbh : a.pb, 0), lrow1, j, a.pml, a.dt, rowdom, ok1,
                        src_iz, sprev, INJ ? row_at(a.inj[c], ubase) : v);
    };
    // forward z-FFT of x (first pass of the 3-D transform) into dst
    auto fft_store = [&](float2 (&x)[G::N1], float2* dstp) {
        __syncthreads();
        if (act1) fwd_l1<G>(x, pen1, tws, j);
        __syncthreads();
        if (ok2) {
            float2 b[G::N2];
            fwd_l2<G>(b, pen2, k1);
            const Row dst = row_at(dstp, ubase);
            const unsigned o = lane_off(8u * (unsigned)(p2 * n + k1));
#pragma unroll
            for (int k2 = 0; k2 < G::N2; ++k2) st2(dst, o, b[k2], 8 * G::N1 * k2);
        }
    };

    // Packing of the stress step's transforms: P0 = F(wx + i wy),
    // P1 = F(wz + i vz), P2 = F(vx + i vy).  A1 is needed on P0 and P1, A3 on
    // P1 and P2.
    if (blockIdx.y == 0) {
        float2 d[G::N1];
        deriv(a.pxz, a.pyz, a.symp, d);  // dz pxz (vx) + i dz pyz (vy), D+
        float2 u[G::N1];
        update(u, d, 0, false);
        // park (vx, wx) in this thread's own pencil slots while vy is updated
        __syncthreads();  // every thread has read the pencil buffer (inv_lb)
        if (act1) {  // (threads past the last pencil own no slots)
#pragma unroll
            for (int j1 = 0; j1 < G::N1; ++j1) pen1[j + G::N2 * j1] = u[j1];
        }
        update(u, d, 1, true);
        float2 x0[G::N1], x1[G::N1];
#pragma unroll
        for (int j1 = 0; j1 < G::N1; ++j1) {
            const float2 ux = act1 ? pen1[j + G::N2 * j1] : make_float2(0.f, 0.f);
            x0[j1] = make_float2(ux.y, u[j1].y);
            x1[j1] = make_float2(ux.x, u[j1].x);
        }
        fft_store(x0, a.P[0]);
        fft_store(x1, a.P[2]);
    } else {
        float2 d[G::N1];
        deriv(a.pzz, nullptr, a.symm, d);  // dz pzz (vz), D-
        float2 x2[G::N1];
        update(x2, d, 2, false);
#pragma unroll
        for (int j1 = 0; j1 < G::N1; ++j1) x2[j1] = make_float2(x2[j1].y, x2[j1].x);
        fft_store(x2, a.P[1]);
    }
}

// ------------------------------------------------------------------------
// In-place complex transforms along a strided axis (y: stride sy, x: stride
// sx) for up to 6 complex fields.  Tile: G::P adjacent complex z-columns.
// DIR -1: forward (natural-order input, natural-order spectrum out);
// DIR +1: inverse.
struct CStridedArgs {
    int nz;
    long long sx, sy;
    int axis, ztiles, nplanes, run;  // workgroup placement: plane_tile()
    long long shot_stride;
    const float2* tw;
    int nfields;
    float2* f[8];
};

// NT: non-temporal loads (stream_nt); the stores feed the next kernel's rows
template <class G, int DIR, bool NT>
__global__ __launch_bounds__(G::T) void k2_cfft_strided(CStridedArgs a)
{
    __shared__ float2 lds[G::P * G::PS];
    __shared__ float2 tws[G::TWN];
    const int tid = threadIdx.x, shot = blockIdx.y;
    const PlaneTile pt = plane_tile(a.ztiles, a.nplanes, a.run, blockIdx.x);
    if (pt.plane < 0) return;
    const int other = pt.plane;
    const int p = tid % G::P, jj = tid / G::P;
    const int zc = pt.zt * G::P + p;
    const bool zok = zc < a.nz;
    const bool act1 = jj < G::N2 && zok, act2 = jj < G::N1 && zok;
    const int astride = (int)(a.axis == 0 ? a.sx : a.sy);
    // uniform tile base (shot, plane, first column) + unsigned lane offset
    const long long tbase = (long long)shot * a.shot_stride +
                            (a.axis == 0 ? (long long)other * a.sy : (long long)other * a.sx) +
                            (long long)pt.zt * G::P;
    const unsigned voff = 8u * (unsigned)(jj * astride + p);
    float2* pen = lds + p * G::PS;
    load_twiddles<G>(tws, a.tw);
    for (int f = blockIdx.z; f < a.nfields; f += gridDim.z) {
        float2* const fb = a.f[f] + tbase;
        const unsigned o = lane_off(voff);
        __syncthreads();
        if (DIR < 0) {
            if (act1) {
                float2 v[G::N1];
#pragma unroll
                for (int j1 = 0; j1 < G::N1; ++j1)
                    v[j1] = ld2<NT>(row_at(fb, (long long)(j1 * G::N2) * astride), o);
                fwd_l1<G>(v, pen, tws, jj);
            }
            __syncthreads();
            if (act2) {
                float2 b[G::N2];
                fwd_l2<G>(b, pen, jj);
#pragma unroll
                for (int k2 = 0; k2 < G::N2; ++k2) st2(row_at(fb, (long long)(G::N1 * k2) * astride), lane_off(voff), b[k2]);
            }
        } else {
            if (act2) {
                float2 b[G::N2];
#pragma unroll
                for (int k2 = 0; k2 < G::N2; ++k2)
                    b[k2] = ld2<NT>(row_at(fb, (long long)(G::N1 * k2) * astride), o);
                inv_la<G>(b, pen, tws + G::T2OFF, jj);
            }
            __syncthreads();
            if (act1) {
                float2 d[G::N1];
                inv_lb<G>(d, pen, jj);
#pragma unroll
                for (int j1 = 0; j1 < G::N1; ++j1) st2(row_at(fb, (long long)(G::N2 * j1) * astride), lane_off(voff), d[j1]);
            }
        }
    }
}

// ------------------------------------------------------------------------
// x-pass of the 3-D transform: forward x-FFT of P (already z- and
// y-transformed), multiply by A1 = |k|^-1 / L and A3 = L |k| over N (|k|^2 = kx^2+ky^2+kz^2
// from the folded 1-D |K| tables, evaluated in FP64 and rounded once,
// cuviscoelas_3D.cu:72, 188-190; the DC symbol of |k|^-1 is 0 because every
// use is followed by a derivative that vanishes there), inverse x-FFT,
// write Q1, Q3.
//
// KS (opt-in k-space correction and wavenumber filter): every stress
// operator A_j, A2 = 1 included, is multiplied by
//   F(|k|) = sinc^2(vh |k|) * W(|k|),  sinc(x) = sin(x)/x,  vh = vref dt / 2
// (the disabled sinc2nd of cuviscoelas_3D.cu:183-190), with W the radial
// Tukey taper: 1 for |k| <= k0, (1 + cos(pi (|k| - k0) / (kc - k0))) / 2 up
// to kc, 0 beyond (the filter the reference declares but never builds,
// Myfunctions.h:69, viscoelas_3D.cpp:111-112).  A2 F is no longer a 1-D
// operator, so a third product F P / N is inverse-transformed into Q2.
struct XPassArgs {
    int ny, nz;
    long long sx, sy;
    int ztiles, run;  // planes: ny; workgroup placement: plane_tile()
    long long shot_stride;
    const float2* tw;
    const float *kfx, *kfy, *kfz;
    double invN, invN1, invN3;  // 1/N, 1/(N L), L/N
    int ncomp;
    const float2* P[3];
    float2* Q1[3];           // null: A1 P_c is not used
    float2* Q3[3];           // null: A3 P_c is not used
    float2* Q2[3];           // KS only
    float ks_vh;             // vref dt / 2 (0: no sinc^2 factor)
    float ks_k0, ks_kc;      // taper start and cut-off (kc = 0: no filter)
    float ks_pw;             // pi / (kc - k0) (0 when k0 == kc)
};

// F(|k|) of the KS mode, in FP32.
__device__ __forceinline__ float kspace_factor(const XPassArgs& a, float k)
{
    float f = 1.f;
    if (a.ks_vh > 0.f) {
        const float x = a.ks_vh * k;
        const float sx = x > 0.f ? sinf(x) / x : 1.f;
        f = sx * sx;
    }
    if (a.ks_kc > 0.f) {
        if (k > a.ks_kc) f = 0.f;
        else if (k > a.ks_k0) f *= 0.5f * (1.f + cosf(a.ks_pw * (k - a.ks_k0)));
    }
    return f;
}

// NT: non-temporal loads and stores (stream_nt)
template <class G, bool KS, bool NT>
__global__ __launch_bounds__(G::T) __attribute__((amdgpu_waves_per_eu(QVTI_XPASS_WAVES))) void k2_xpass(XPassArgs a)
{
    __shared__ float2 lds[G::P * G::PS];
    __shared__ float2 tws[G::TWN];
    const int tid = threadIdx.x, shot = blockIdx.y;
    const PlaneTile pt = plane_tile(a.ztiles, a.ny, a.run, blockIdx.x);
    if (pt.plane < 0) return;
    const int iy = pt.plane;
    const int p = tid % G::P, jj = tid / G::P;
    const int zc = pt.zt * G::P + p;
    const bool zok = zc < a.nz;
    const bool act1 = jj < G::N2 && zok, act2 = jj < G::N1 && zok;
    // uniform tile base (shot, plane, first column) + unsigned lane offset
    const long long tbase = (long long)shot * a.shot_stride + (long long)iy * a.sy +
                            (long long)pt.zt * G::P;
    const int sxi = (int)a.sx;
    const unsigned voff = 8u * (unsigned)(jj * sxi + p);
    float2* pen = lds + p * G::PS;
    load_twiddles<G>(tws, a.tw);
    const double ky = a.kfy[iy];
    const double kz = a.kfz[zok ? zc : 0];
    const double kyz = ky * ky + kz * kz;
    for (int comp = blockIdx.z; comp < a.ncomp; comp += gridDim.z) {
        const float2* const src = a.P[comp] + tbase;
        __syncthreads();
        if (act1) {
            float2 v[G::N1];
            const unsigned o = lane_off(voff);
#pragma unroll
            for (int j1 = 0; j1 < G::N1; ++j1) v[j1] = ld2<NT>(row_at(src, (long long)(j1 * G::N2) * sxi), o);
            fwd_l1<G>(v, pen, tws, jj);
        }
        __syncthreads();
        float2 b[G::N2];
        if (act2) fwd_l2<G>(b, pen, jj);
        int jl = jj;  // opaque copy: the |k| symbols are computed here, not hoisted and held
        asm volatile("" : "+v"(jl));
        if (KS && act2) {
            // F multiplies every operator: apply it to the spectrum once (one
            // more FP32 rounding than folding it into each symbol)
#pragma unroll
            for (int k2 = 0; k2 < G::N2; ++k2) {
                const double kx = a.kfx[jl + G::N1 * k2];
                const float F = kspace_factor(a, sqrtf((float)(kx * kx + kyz)));
                b[k2] = make_float2(b[k2].x * F, b[k2].y * F);
            }
        }
        // ops: 0 A1 -> Q1, 1 A3 -> Q3 (where used), 2 A2 -> Q2 (KS only)
#pragma unroll
        for (int op = 0; op < (KS ? 3 : 2); ++op) {
            float2* const q = op == 0 ? a.Q1[comp] : (op == 1 ? a.Q3[comp] : a.Q2[comp]);
            if (!q) continue;  // uniform: this product is not used
            __syncthreads();
            if (act2) {
                float2 c[G::N2];
#pragma unroll
                for (int k2 = 0; k2 < G::N2; ++k2) {
                    const double kx = a.kfx[jl + G::N1 * k2];
                    const double k2s = kx * kx + kyz;
                    // 1/sqrt(k2s): the FP32 hardware estimate (relative
                    // error below 2^-23) and one FP64 Newton step (below
                    // 2^-45), so the FP32 rounding below is that of the
                    // exact value except within 2^-45 of a rounding boundary
                    double y = __builtin_amdgcn_rsqf((float)k2s);
                    y = fma(y, fma(-0.5 * k2s * y, y, 0.5), y);
                    const double s = KS && op == 2 ? a.invN  // A2 = 1 (F already applied)
                                                   : (op == 0 ? a.invN1 * y : a.invN3 * (k2s * y));
                    float fs = (float)s;
                    // k = 0 only at element 0 (k2 = 0, jl = 0), where the
                    // estimate is inf and y NaN: both symbols are 0 there,
                    // |k|^-1 by the convention above
                    if (k2 == 0 && !(KS && op == 2) && !(k2s > 0.0)) fs = 0.f;
                    c[k2] = make_float2(b[k2].x * fs, b[k2].y * fs);
                }
                inv_la<G>(c, pen, tws + G::T2OFF, jj);
            }
            __syncthreads();
            if (act1) {
                float2 d[G::N1];
                inv_lb<G>(d, pen, jj);
                float2* const dst = q + tbase;
                const unsigned o = lane_off(voff);
#pragma unroll
                for (int j1 = 0; j1 < G::N1; ++j1) st2<NT>(row_at(dst, (long long)(G::N2 * j1) * sxi), o, d[j1]);
            }
        }
    }
}

// ------------------------------------------------------------------------
// z-direction complex transforms on rows.
//  mode 1 (inverse, stress step end): re_out + i im_out = IFFT_z(cin)   (either may be null)
//  mode 2 (plain, standalone transforms): cout = FFT_z^DIR(cin), in place allowed
// A last grid-z slice (rec.nt > 0) takes the receivers of the step: the
// velocities are final since k2_vel_z except for the source, whose sample the
// stress update adds to its cell after this kernel and record_sample adds here
// (the same FP32 sum).  A launch of its own cost 3.9 us a step.
struct ZRowsArgs {
    long long nrows;
    long long shot_stride;
    const float2* tw;
    int mode, dir, nfields;
    const float2* cin[8];
    float2* cout[8];
    float* re_out[8];
    float* im_out[8];
    RecArgs rec;
};

// NT: non-temporal loads (stream_nt)
template <class G, bool NT>
__global__ __launch_bounds__(kThreads) void k2_zrows(ZRowsArgs a)
{
    __shared__ float2 lds[G::P * G::PS];
    __shared__ float2 tws[G::TWN];
    constexpr int n = G::N;
    const int tid = threadIdx.x, shot = blockIdx.y;
    if (a.rec.nt > 0 && blockIdx.z == gridDim.z - 1) {
        record_samples(a.rec, shot, blockIdx.x * kThreads + tid, gridDim.x * kThreads);
        return;
    }
    const int fz = a.rec.nt > 0 ? gridDim.z - 1 : gridDim.z;  // grid-z slices of the transforms
    const int j = tid % G::N2, p1 = tid / G::N2;
    const int k1 = tid % G::N1, p2 = tid / G::N1;
    const long long r0 = (long long)blockIdx.x * G::P, r1 = r0 + p1, r2 = r0 + p2;
    const bool ok1 = p1 < G::P && r1 < a.nrows, ok2 = p2 < G::P && r2 < a.nrows;
    const long long soff = (long long)shot * a.shot_stride;
    float2* pen1 = lds + p1 * G::PS;
    float2* pen2 = lds + p2 * G::PS;
    load_twiddles<G>(tws, a.tw);
    for (int f = blockIdx.z; f < a.nfields; f += fz) {
        __syncthreads();
        if (a.mode == 2 && a.dir < 0) {
            if (ok1) {
                float2 v[G::N1];
                const Row src = row_at(a.cin[f], soff + r0 * n);
                const unsigned o = lane_off(8u * (unsigned)(p1 * n + j));
#pragma unroll
                for (int j1 = 0; j1 < G::N1; ++j1) v[j1] = ld2(src, o, 8 * G::N2 * j1);
                fwd_l1<G>(v, pen1, tws, j);
            }
            __syncthreads();
            if (ok2) {
                float2 b[G::N2];
                fwd_l2<G>(b, pen2, k1);
                const Row dst = row_at(a.cout[f], soff + r0 * n);
                const unsigned o = lane_off(8u * (unsigned)(p2 * n + k1));
#pragma unroll
                for (int k2 = 0; k2 < G::N2; ++k2) st2(dst, o, b[k2], 8 * G::N1 * k2);
            }
        } else {
            if (ok2) {
                float2 b[G::N2];
                const Row src = row_at(a.cin[f], soff + r0 * n);
                const unsigned o = lane_off(8u * (unsigned)(p2 * n + k1));
#pragma unroll
                for (int k2 = 0; k2 < G::N2; ++k2) b[k2] = ld2<NT>(src, o, 8 * G::N1 * k2);
                inv_la<G>(b, pen2, tws + G::T2OFF, k1);
            }
            __syncthreads();
            if (ok1) {
                float2 d[G::N1];
                inv_lb<G>(d, pen1, j);
                if (a.mode == 2) {
                    const Row dst = row_at(a.cout[f], soff + r0 * n);
                    const unsigned o = lane_off(8u * (unsigned)(p1 * n + j));
#pragma unroll
                    for (int j1 = 0; j1 < G::N1; ++j1) st2(dst, o, d[j1], 8 * G::N2 * j1);
                } else {
                    const unsigned o = lane_off(4u * (unsigned)(p1 * n + j));
                    if (a.re_out[f]) {
                        const Row re = row_at(a.re_out[f], soff + r0 * n);
#pragma unroll
                        for (int j1 = 0; j1 < G::N1; ++j1) st1(re, o, d[j1].x, 4 * G::N2 * j1);
                    }
                    if (a.im_out[f]) {
                        const Row im = row_at(a.im_out[f], soff + r0 * n);
#pragma unroll
                        for (int j1 = 0; j1 < G::N1; ++j1) st1(im, o, d[j1].y, 4 * G::N2 * j1);
                    }
                }
            }
        }
    }
}

// ------------------------------------------------------------------------
// 1-D shift-derivative along z of one real field (standalone entry point).
// Tile: G::P complex pencils = 2*G::P rows.
struct RowDerivArgs {
    long long nrows;
    const float2* tw;
    const float2* sym;
    const float* in;
    float* out;
};

template <class G>
__global__ __launch_bounds__(kThreads) void k2_deriv_rows(RowDerivArgs a)
{
    __shared__ float2 lds[G::P * G::PS];
    __shared__ float2 tws[G::TWN];
    constexpr int n = G::N;
    const int tid = threadIdx.x;
    const int j = tid % G::N2, p1 = tid / G::N2;
    const int k1 = tid % G::N1, p2 = tid / G::N1;
    const long long ra = (long long)blockIdx.x * 2 * G::P + 2 * p1;  // rows ra, ra+1
    const bool act1 = p1 < G::P, act2 = p2 < G::P;
    float2* pen1 = lds + p1 * G::PS;
    float2* pen2 = lds + p2 * G::PS;
    load_twiddles<G>(tws, a.tw);
    __syncthreads();
    if (act1) {
        float2 v[G::N1];
#pragma unroll
        for (int j1 = 0; j1 < G::N1; ++j1) {
            const int i = j1 * G::N2 + j;
            v[j1] = make_float2(ra < a.nrows ? a.in[ra * n + i] : 0.f, ra + 1 < a.nrows ? a.in[(ra + 1) * n + i] : 0.f);
        }
        fwd_l1<G>(v, pen1, tws, j);
    }
    __syncthreads();
    float2 b[G::N2];
    if (act2) {
        fwd_l2<G>(b, pen2, k1);
#pragma unroll
        for (int k2 = 0; k2 < G::N2; ++k2) b[k2] = c_mul(b[k2], a.sym[k1 + G::N1 * k2]);
    }
    __syncthreads();
    if (act2) inv_la<G>(b, pen2, tws + G::T2OFF, k1);
    __syncthreads();
    if (act1) {
        float2 d[G::N1];
        inv_lb<G>(d, pen1, j);
#pragma unroll
        for (int j1 = 0; j1 < G::N1; ++j1) {
            const int i = j + G::N2 * j1;
            if (ra < a.nrows) a.out[ra * n + i] = d[j1].x;
            if (ra + 1 < a.nrows) a.out[(ra + 1) * n + i] = d[j1].y;
        }
    }
}

// ------------------------------------------------------------------------
// Stress update (cuviscoelas_3D.cu:800-1015, generalised to VTI moduli) fused
// with the z-derivatives of the 12 family fields, the stress C-PML memory
// variables on the face slabs, and the source injection
// (cuviscoelas_3D.cu:771-777).  Tile: R rows (StressTile); 6 complex pencils
// per row carry the 12 fields (two per pencil, same z-symbol); their
// derivatives are staged in LDS, then every thread updates R*nz/T cells.
struct StressZArgs {
    int nx, ny, nz, pml;
    int ntiles, nshots, run;  // grid: tile_shot()
    long long nrows;
    float dt;
    long long shot_stride, slabx_stride, slaby_stride, slabz_stride;
    const float2* tw;
    const float2* symp;  // D+ symbols; the D- ones follow symm_off bytes on
    unsigned symm_off;
    const float *pax, *pbx, *paxh, *pbxh;
    const float *pay, *pby, *payh, *pbyh;
    const float *paz, *pbz, *pazh, *pbzh;
    // [component][A1 w, A2 v, A3 v, A2 w]; A2 = 1 (the fields v and w
    // themselves) unless the k-space correction is on
    const float* fam[3][kFam];
    float* vel[3];  // vx vy vz: force sources are added here
    // x- and y-derivatives, blocked groups [shot][N/64][kDer][64]:
    //   dxb: ex 0-3 (dx vx-family), sum_j S-bar_j dx of the vz family 4, of the vy family 5
    //   dyb: ey 0-3 (dy vy-family), sum_j S-bar_j dy of the vz family 4, of the vx family 5
    const float *dxb, *dyb;
    long long blk_stride;  // per-shot field length of the blocked groups (N rounded up to 64)
    const float *gm, *gs;  // medium fields: the blocked group; in natural order
    long long N;
    const MediumConst* med;
    float* sig[6];  // pxx pyy pzz pxy pxz pyz
    float* phx[5];
    float* phy[5];
    float* phz[4];
    const int* src_kind;
    const long long* src_ip;
    const float* rik;
    const int* it;
};

// Workgroup tile of the stress update: R rows of 6 pencils on T threads (both
// transform levels take one pass: 6 R NMAX <= T).
//  * rows that end on a 128-byte line: T = 192 or 256, whichever leaves fewer
//    threads idle in the transforms (256 = 16 x 16: 12 pencils on 192 threads;
//    at 256^3 1001 us against 1081 us on 384 and 1269 us on 512 threads (646
//    us since the shear sums left it and with streaming): more, smaller
//    workgroups overlap their load and transform phases better; 384 threads at
//    n = 128: 109 us against 91 us at 128^3);
//  * long rows that end mid-line share their last line and 64-cell block with
//    the next tile, so fewer, larger tiles: T = 512 (400x400x200: 4 rows,
//    1980 us, against 2211 us with 2 rows on 256 threads; 1365 us since the
//    shear sums left it).
template <class G>
struct StressTile {
    static constexpr int R256 = 256 / (6 * G::NMAX), R192 = 192 / (6 * G::NMAX);
    static constexpr int T = G::N % 32 != 0 && G::N >= 128 ? 512 : (4 * R192 >= 3 * R256 ? 192 : 256);
    static constexpr int R = T / (6 * G::NMAX);
    static constexpr int NP = 6 * R;  // pencils
};

// pencil kind -> (component, family member of the real part, of the imaginary part)
// staging field index = 2*kind (+1 for the imaginary part)
//   c     (0-2): A1 w_c + i A2 w_c    3 + c (3-5): A2 v_c + i A3 v_c
// (c = 2: D+, else D-)
// NT (stream_nt): 1 loads the derivatives non-temporally, 2 (one shot) the
// coefficients and stresses as well - with several shots the coefficients are
// read again for the next shot of the tile.  49 floats per cell bound it: 256^3
// 714 -> 657 us (2; 654 us, 5.0 TB/s, with the early loads below and the FP64
// coefficients, 730 us with all 16 of them read), 32 shots of 160x160x128:
// 4234 -> 4192 us (1; 4260 with 2).
template <class G, bool VTI, int NT>
__global__ __launch_bounds__(StressTile<G>::T) __attribute__((amdgpu_waves_per_eu(QVTI_STRESSZ_WAVES))) void k2_stress_z(
    StressZArgs a)
{
    using T = StressTile<G>;
    constexpr int R = T::R, NP = T::NP;
    constexpr int n = G::N;
    static_assert(R >= 1, "tile too small");
    static_assert(G::PS >= n + 1, "staging must fit in the pencil buffer");
    __shared__ float2 lds[NP * G::PS];
    __shared__ float2 tws[G::TWN];
    const TileShot ts = tile_shot(a.ntiles, a.nshots, a.run);
    if (ts.tile < 0) return;  // padding workgroup (whole workgroup, before any barrier)
    const int tid = threadIdx.x, shot = ts.shot;
    // level 1: N2 lanes per pencil; level 2: N1 lanes per pencil
    const int j = tid % G::N2, q1 = tid / G::N2;
    const int k1 = tid % G::N1, q2 = tid / G::N1;
    const bool act1 = q1 < NP, act2 = q2 < NP;
    const long long r0 = (long long)ts.tile * R;
    const long long soff = (long long)shot * a.shot_stride;
    float2* pen1 = lds + q1 * G::PS;
    float2* pen2 = lds + q2 * G::PS;
    {
        const int kind1 = q1 % 6, rr1 = q1 / 6;
        float2 v[G::N1];  // on its way while the twiddle tables load (256^3: 665 -> 655 us)
        if (act1) {
            const long long row1 = r0 + rr1;
            const bool ok1 = row1 < a.nrows;
            const int c = kind1 < 3 ? kind1 : kind1 - 3;
            // rows past the end (last tile) read the tile's first row and are not used
            const long long g = soff + (ok1 ? row1 : r0) * n + j;
            const float* fre = a.fam[c][kind1 < 3 ? 0 : 1] + g;
            const float* fim = a.fam[c][kind1 < 3 ? 3 : 2] + g;
#pragma unroll
            for (int j1 = 0; j1 < G::N1; ++j1) v[j1] = make_float2(fre[j1 * G::N2], fim[j1 * G::N2]);
        }
        for (int t = tid; t < G::TWN; t += T::T) twiddle_entry<G>(tws, a.tw, t);
        __syncthreads();
        if (act1) fwd_l1<G>(v, pen1, tws, j);
        __syncthreads();
        float2 b[G::N2];
        if (act2) {
            fwd_l2<G>(b, pen2, k1);
            const int kind2 = q2 % 6;
            // both symbol tables sit in one allocation: a per-lane offset picks one
            const Row S = row_at(a.symp, 0);
            const unsigned o = lane_off(8u * k1 + (kind2 == 2 || kind2 == 5 ? 0u : a.symm_off));
#pragma unroll
            for (int k2 = 0; k2 < G::N2; ++k2) b[k2] = c_mul(b[k2], ld2(S, o, 8 * G::N1 * k2));
        }
        __syncthreads();
        if (act2) inv_la<G>(b, pen2, tws + G::T2OFF, k1);
        __syncthreads();
        float2 d[G::N1];
        if (act1) inv_lb<G>(d, pen1, j);
        __syncthreads();
        // stage: st[field][rr][iz] with rows padded to n + 1 floats (odd), so
        // the rows written by one wave fall in different banks, field = 2*kind + part
        float* st = reinterpret_cast<float*>(lds);
        if (act1) {
#pragma unroll
            for (int j1 = 0; j1 < G::N1; ++j1) {
                const int iz = j + G::N2 * j1;
                st[((2 * kind1) * R + rr1) * (n + 1) + iz] = d[j1].x;
                st[((2 * kind1 + 1) * R + rr1) * (n + 1) + iz] = d[j1].y;
            }
        }
        __syncthreads();
    }
    const float* st = reinterpret_cast<const float*>(lds);
    const int pml = a.pml;
    const float dt = a.dt;
    const MediumConst med = *a.med;
    const int it = *a.it;
    const int kind = a.src_kind[shot];
    const long long sip = a.src_ip[shot];
    // uniform block bases; per-cell offsets below are unsigned 32-bit
    const long long cbase = r0 * n;          // flat index of the tile's first cell
    const long long fbase = soff + cbase;    // per-shot natural fields
    const Row dxr = row_at(a.dxb, (long long)shot * kDer * a.blk_stride);
    const Row dyr = row_at(a.dyb, (long long)shot * kDer * a.blk_stride);
    const Row gmr = row_at(a.gm, 0);
    Row gsr[kGS(VTI)], sgr[6];
#pragma unroll
    for (int k = 0; k < kGS(VTI); ++k) gsr[k] = row_at(a.gs + k * a.N, cbase);
#pragma unroll
    for (int k = 0; k < 6; ++k) sgr[k] = row_at(a.sig[k], fbase);
    constexpr bool vti = VTI;  // G2 (H, D sets) present: a compile-time choice keeps the loads branch-free
    const long long sxb = (long long)shot * a.slabx_stride, syb = (long long)shot * a.slaby_stride,
                    szb = (long long)shot * a.slabz_stride;
#pragma unroll 1
    for (int cell = tid; cell < R * n; cell += T::T) {
        const int rr = cell / n, iz = cell - rr * n;
        const long long row = r0 + rr;
        if (row >= a.nrows) continue;
        const int ix = (int)(row / a.ny), iy = (int)(row - (long long)ix * a.ny);
        const unsigned o = (unsigned)cell;  // == rr * n + iz
        auto S = [&](int f) { return st[(f * R + rr) * (n + 1) + iz]; };
        if (ix < a.nx - 1 && iy < a.ny - 1 && iz < n - 1) {
            // staging fields of the family members (A1 w, v, A3 v, w)
            const int fz[kFam] = {4, 10, 11, 5};   // vz family (D+): normal dz vz
            const int fgx[kFam] = {0, 6, 7, 1};    // vx family (D-): dz vx for pxz
            const int fhy[kFam] = {2, 8, 9, 3};    // vy family (D-): dz vy for pyz
            // blocked addresses of the cell: one offset per group, the
            // fields at immediate offsets f*64 floats
            const unsigned ip = (unsigned)cbase + o;
            const unsigned blk = ip >> 6, in = ip & 63u;
            const unsigned od = lane_off(4u * (blk * (kBlk * kDer) + in));
            const unsigned om = lane_off(4u * (blk * (kBlk * kGM(VTI)) + in));
            const unsigned oc = lane_off(4u * o);
            constexpr int FB = 4 * kBlk;  // bytes between the fields of a block
            float oP[kFam], oS[kFam], oH[kFam], oD[kFam];
            {
                auto gm = [&](int f) { return ld1<(NT > 1)>(gmr, om, f * FB); };
                const int ps = __float_as_int(gm(GM_LOW));  // (the low half's sign is extended)
                const double rho = gm(GM_RHO), gp = gm(GM_GP);
                set_coeffs(oP, gm(GM_CP), (int)(short)ps, gp, rho, med);
                set_coeffs(oS, gm(GM_CS), ps >> 16, gm(GM_GS), rho, med);
                if (vti) {
                    const int hd = __float_as_int(ld1<(NT > 1)>(gsr[kFam], oc));
                    set_coeffs(oH, gm(GM_CH), (int)(short)hd, gp, rho, med);
                    set_coeffs(oD, gm(GM_CD), hd >> 16, gp, rho, med);
                }
            }
            float A[14];
#pragma unroll
            for (int k = 0; k < 14; ++k) A[k] = 0.f;
            A[9] = ld1<(NT > 0)>(dxr, od, kFam * FB);         // sb_zx  (dx vz)
            A[11] = ld1<(NT > 0)>(dxr, od, (kFam + 1) * FB);  // sb_yx  (dx vy)
            A[13] = ld1<(NT > 0)>(dyr, od, kFam * FB);        // sb_zy  (dy vz)
            A[10] = ld1<(NT > 0)>(dyr, od, (kFam + 1) * FB);  // sb_xy  (dy vx)
#pragma unroll
            for (int jf = 0; jf < kFam; ++jf) {
                const float ez = S(fz[jf]), gz = S(fgx[jf]), hz = S(fhy[jf]);
                const float ex = ld1<(NT > 0)>(dxr, od, jf * FB), ey = ld1<(NT > 0)>(dyr, od, jf * FB);
                const float c33 = oP[jf], cs = oS[jf], csb = ld1<(NT > 1)>(gsr[jf], oc);
                const float c11 = vti ? oH[jf] : c33, c13 = vti ? oD[jf] : c33;
                const float c12 = c11 - 2 * cs, c13d = c13 - 2 * cs;
                A[0] += c11 * ex;   // s11x
                A[1] += c12 * ex;   // s12x
                A[2] += c13d * ex;  // s13x
                A[3] += c12 * ey;   // s12y
                A[4] += c11 * ey;   // s11y
                A[5] += c13d * ey;  // s13y
                A[6] += c13d * ez;  // s13z
                A[7] += c33 * ez;   // s33z
                A[8] += csb * gz;   // sb_xz  (dz vx)
                A[12] += csb * hz;  // sb_yz  (dz vy)
            }
            // Every load of the cell is issued before its first store: the
            // stress and C-PML arrays are distinct, but the compiler cannot
            // know it, so loads placed after a store would each wait for it.
            float sg[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) sg[k] = ld1<(NT > 1)>(sgr[k], oc);
            const bool xs = ix < pml || ix >= a.nx - pml;
            const bool ys = iy < pml || iy >= a.ny - pml;
            const bool zs = iz < pml || iz >= n - pml;
            unsigned ox = 0, oy = 0, oz = 0;
            float qx[5], qy[5], qz[4];
            if (xs) {
                const int si = ix < pml ? ix : ix - (a.nx - 2 * pml);
                ox = (unsigned)(((long long)si * a.ny + iy) * n + iz);
#pragma unroll
                for (int k = 0; k < 5; ++k) qx[k] = a.phx[k][sxb + ox];
            }
            if (ys) {
                const int si = iy < pml ? iy : iy - (a.ny - 2 * pml);
                oy = (unsigned)(((long long)ix * 2 * pml + si) * n + iz);
#pragma unroll
                for (int k = 0; k < 5; ++k) qy[k] = a.phy[k][syb + oy];
            }
            if (zs) {
                const int si = iz < pml ? iz : iz - (n - 2 * pml);
                oz = (unsigned)(row * 2 * pml + si);
#pragma unroll
                for (int k = 0; k < 4; ++k) qz[k] = a.phz[k][szb + oz];
            }
            float fxx_x = 0.f, fxy_x = 0.f, fxz_x = 0.f, fzx = 0.f, fyx = 0.f;
            float fyx_y = 0.f, fyy_y = 0.f, fyz_y = 0.f, fxy = 0.f, fzy = 0.f;
            float fzx_z = 0.f, fzz_z = 0.f, fxz = 0.f, fyz = 0.f;
            if (xs) {
                const float Ax = a.pax[ix], Bx = a.pbx[ix], Ah = a.paxh[ix], Bh = a.pbxh[ix];
                fxx_x = qx[0] + dt * (-Ax * qx[0] - Bx * A[0]);
                fxy_x = qx[1] + dt * (-Ax * qx[1] - Bx * A[1]);
                fxz_x = qx[2] + dt * (-Ax * qx[2] - Bx * A[2]);
                fzx = qx[3] + dt * (-Ah * qx[3] - Bh * A[9]);
                fyx = qx[4] + dt * (-Ah * qx[4] - Bh * A[11]);
                a.phx[0][sxb + ox] = fxx_x;
                a.phx[1][sxb + ox] = fxy_x;
                a.phx[2][sxb + ox] = fxz_x;
                a.phx[3][sxb + ox] = fzx;
                a.phx[4][sxb + ox] = fyx;
            }
            if (ys) {
                const float Ay = a.pay[iy], By = a.pby[iy], Ah = a.payh[iy], Bh = a.pbyh[iy];
                fyx_y = qy[0] + dt * (-Ay * qy[0] - By * A[3]);
                fyy_y = qy[1] + dt * (-Ay * qy[1] - By * A[4]);
                fyz_y = qy[2] + dt * (-Ay * qy[2] - By * A[5]);
                fxy = qy[3] + dt * (-Ah * qy[3] - Bh * A[10]);
                fzy = qy[4] + dt * (-Ah * qy[4] - Bh * A[13]);
                a.phy[0][syb + oy] = fyx_y;
                a.phy[1][syb + oy] = fyy_y;
                a.phy[2][syb + oy] = fyz_y;
                a.phy[3][syb + oy] = fxy;
                a.phy[4][syb + oy] = fzy;
            }
            if (zs) {
                const float Az = a.paz[iz], Bz = a.pbz[iz], Ah = a.pazh[iz], Bh = a.pbzh[iz];
                fzx_z = qz[0] + dt * (-Az * qz[0] - Bz * A[6]);
                fzz_z = qz[1] + dt * (-Az * qz[1] - Bz * A[7]);
                fxz = qz[2] + dt * (-Ah * qz[2] - Bh * A[8]);
                fyz = qz[3] + dt * (-Ah * qz[3] - Bh * A[12]);
                a.phz[0][szb + oz] = fzx_z;
                a.phz[1][szb + oz] = fzz_z;
                a.phz[2][szb + oz] = fxz;
                a.phz[3][szb + oz] = fyz;
            }
            st1<(NT > 1)>(sgr[0], oc, sg[0] + dt * (A[0] + A[3] + A[6] + (fxx_x + fyx_y + fzx_z)));
            st1<(NT > 1)>(sgr[1], oc, sg[1] + dt * (A[1] + A[4] + A[6] + (fxy_x + fyy_y + fzx_z)));
            st1<(NT > 1)>(sgr[2], oc, sg[2] + dt * (A[2] + A[5] + A[7] + (fxz_x + fyz_y + fzz_z)));
            st1<(NT > 1)>(sgr[3], oc, sg[3] + dt * (A[10] + fxy + A[11] + fyx));
            st1<(NT > 1)>(sgr[4], oc, sg[4] + dt * (A[8] + fxz + A[9] + fzx));
            st1<(NT > 1)>(sgr[5], oc, sg[5] + dt * (A[12] + fyz + A[13] + fzy));
        }
        if (row * n + iz == sip) {
            // source after the stress update; no other workgroup of this
            // launch touches this row of v (at most this one read it, for its
            // z-derivative, staged above), so the write cannot race.
            const float s = a.rik[it];
            const long long g = fbase + o;
            if (kind == 3) {
                a.sig[0][g] += s;
                a.sig[1][g] += s;
                a.sig[2][g] += s;
            } else if (kind >= 0 && kind < 3) {
                a.vel[kind][g] += s;
            }
        }
    }
}

}  // namespace qvti
