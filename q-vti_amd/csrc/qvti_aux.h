// qvti_aux.h -- non-transform kernels of the engine: receivers, step
// counter, snapshots, blow-up probe and the once-per-model setup kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "qvti_layout.h"

namespace qvti {

// Receivers: rec[it][r] = v[cell_r] for the three components after the
// source injection, cuviscoelas_3D.cu:782-792.  Runs before the injection
// (k2_zrows), which adds rik[it] to one cell: a receiver there gets v + rik[it],
// the value the injection writes.
struct RecArgs {
    const float *vx, *vy, *vz;
    long long shot_stride;
    const long long* rec_ip;  // all shots' receivers back to back
    const int* rec_off;       // per shot: first receiver, [nshots+1]
    float *rx, *ry, *rz;      // records, per shot offset rec_off[s]*nt
    int nt;                   // 0: no receivers
    const int* it;
    const int* src_kind;
    const long long* src_ip;
    const float* rik;
};

// receivers first, first + stride, ... of one shot
__device__ __forceinline__ void record_samples(const RecArgs& a, int shot, int first, int stride)
{
    const int r0 = a.rec_off[shot], nr = a.rec_off[shot + 1] - r0;
    if (first >= nr) return;
    const int it = *a.it, kind = a.src_kind[shot];
    const long long sip = a.src_ip[shot];
    const float s = a.rik[it];
    for (int r = first; r < nr; r += stride) {
        const long long cell = a.rec_ip[r0 + r], ip = cell + (long long)shot * a.shot_stride;
        const long long o = (long long)r0 * a.nt + (long long)it * nr + r;
        const bool src = cell == sip;
        const float vx = a.vx[ip], vy = a.vy[ip], vz = a.vz[ip];
        a.rx[o] = src && kind == 0 ? vx + s : vx;
        a.ry[o] = src && kind == 1 ? vy + s : vy;
        a.rz[o] = src && kind == 2 ? vz + s : vz;
    }
}

// Snapshot of one field over the box [lo, hi) (ix slowest) when
// it % every == 0; snapshot k lands at out[k * W], W the box's cell count.
struct SnapArgs {
    const float* f;
    int ny, nz;
    int lo[3], hi[3];
    int every;
    const int* it;
    float* out;
    long long cap;
};

static __global__ __launch_bounds__(256) void k_snapshot(SnapArgs a)
{
    const int t = *a.it;
    if (a.every <= 0 || t % a.every != 0) return;
    const long long k = t / a.every;
    const int wx = a.hi[0] - a.lo[0], wy = a.hi[1] - a.lo[1], wz = a.hi[2] - a.lo[2];
    const long long W = (long long)wx * wy * wz;
    if ((k + 1) * W > a.cap) return;
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < W; q += (long long)gridDim.x * 256) {
        const int ix = (int)(q / ((long long)wy * wz));
        const long long rem = q - (long long)ix * wy * wz;
        const int iy = (int)(rem / wz), iz = (int)(rem - (long long)iy * wz);
        a.out[k * W + q] = a.f[((long long)(ix + a.lo[0]) * a.ny + iy + a.lo[1]) * a.nz + iz + a.lo[2]];
    }
}

// Blow-up probe: max |v| over a field (bit pattern of a non-negative float
// orders like an int; NaN sorts above Inf).  One atomic per workgroup, and none
// where the running maximum already covers it: with one per wave, all to one
// address, 64^3 took 50 us.
static __global__ __launch_bounds__(256) void k_probe(const float* f, long long N, int* out)
{
    __shared__ int wave[4];
    int m = 0;
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < N; q += (long long)gridDim.x * 256) {
        const int b = __float_as_int(fabsf(f[q]));
        m = b > m ? b : m;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const int o = __shfl_down(m, off);
        m = o > m ? o : m;
    }
    if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int k = 1; k < 4; ++k) m = wave[k] > m ? wave[k] : m;
    if (m > *out) atomicMax(out, m);  // (a stale read only costs an atomic: *out never falls during a run)
}

// ---- setup kernels (once per model) ------------------------------------

// Q coefficients (cuviscoelas_3D.cu:195-205) in FP64, rounded to FP32.
// set: 0 P (vp, gp), 1 S (vs, gs), 2 H (vp*sqrt(1+2eps), gp), 3 D (v_delta, gp).
// The reference's five terms act on A1 v, v, A3 v, A1 dv and dv, dv = v -
// v_prev (the tau terms carry the 1/dt of its (V - V_prev)/dt).  With c =
// v cos(pi g/2), M = rho c^2 they are
//   o0 = -rho c g w0, o1 = M, o2 = rho c^3 g / w0, o3 = rho c g pi / dt,
//   o4 = M g^2 pi / (w0 dt).
// o3 / o0 = -pi / (w0 dt) = kappa is one constant of the run, and A1 is
// linear, so with the field w = alpha (v + kappa dv)
//   o0 A1 v + o3 A1 dv = (o0 / alpha) A1 w,
//   o1 v + o4 dv       = (o1 - o4 / kappa) v + (o4 / (alpha kappa)) w,
// o4 / kappa = -M g^2: four terms per moduli set instead of five, exactly,
// and A1 acts on w alone.  alpha (qvti_set_model) and the length scale L of
// A1 = 1/(L |k|) and A3 = L |k| (qvti_create) are powers of two (they only
// shift exponents) that keep w and A3 v within a few times v at every
// frequency and wavenumber: v, whose coefficient is the largest by far, then
// takes little rounding from the field that shares a complex transform with
// it, and the others' coefficients are of order g.
//   o[0] = L o0 / alpha (A1 w), o[1] = M (1 + g^2) (v),
//   o[2] = o2 / L (A3 v),       o[3] = -M g^2 / alpha (w)
// o2 and o3 follow from o0, o1 and one field r = alpha / (rho w0^2 L^2):
//   o3 = -o0^2 r,  o2 = -o0 r M,  M = o1 + alpha o3
// (set_coeffs).  The stress update forms them per cell in FP32, so that it
// reads 13 coefficient fields instead of 20 (VTI; 9 instead of 12 isotropic).
// Their rounding (about 2^-23 relative) enters the stresses times g, of order
// 1e-2, so below that of o1 v.
// media (qvti_set_media, the reference's media_type, viscoelas_3D.cpp:57-60):
// 0 viscoelastic (as above); 1 dispersion only (tau terms dropped: kappa = 0,
// w = v, no fourth term); 2 lossless (gamma = 0); 3 Q-compensating (tau terms
// negated: the amplitude loss becomes a gain of the same size, the dispersion
// is kept; kappa changes sign, the four coefficients do not).
__device__ __forceinline__ void q_coeffs(double rho, double v, double g, double w0, double alpha, double L, int media,
                                         double* o)
{
    const double pi = 3.1415926;
    if (media == 2) g = 0.0;
    const double c = v * cos(g * pi / 2.0);
    const double M = rho * (c * c), Mg2 = media == 1 ? 0.0 : M * (g * g);
    o[0] = -rho * c * g * w0 * (L / alpha);
    o[1] = M + Mg2;
    o[2] = rho * pow(c, 3.0) * g / w0 / L;
    o[3] = -Mg2 / alpha;
}

// The four coefficients of one moduli set in the stress update from its
// stored o0, o1 and the cell's r; s4 = 0 where the medium has no tau terms
// (dispersion only), else 1.
__device__ __forceinline__ void set_coeffs(float (&o)[kFam], float o0, float o1, float r, float alpha, float s4)
{
    const float t = o0 * r;
    o[0] = o0;
    o[1] = o1;
    o[3] = -s4 * (o0 * t);
    o[2] = -t * (o1 + alpha * o[3]);
}

// (blocked field groups and coefficient group sizes: qvti_layout.h)

struct CoefArgs {
    long long N;
    int vti, media;
    double w0, alpha, L;
    const float *vp, *gp, *vs, *gs, *rho, *eps, *del;
    float* g1;  // blocked [N/64][kG1][64]
    float* g2;  // blocked [N/64][kG2][64] (VTI only)
    float* s;   // [kFam][N]: the S set, averaged by k_averages
};

static __global__ __launch_bounds__(256) void k_coefficients(CoefArgs a)
{
    for (long long ip = (long long)blockIdx.x * 256 + threadIdx.x; ip < a.N; ip += (long long)gridDim.x * 256) {
        double o[kFam];
        const double r = a.rho[ip];
        q_coeffs(r, a.vp[ip], a.gp[ip], a.w0, a.alpha, a.L, a.media, o);
        for (int j = 0; j < 2; ++j) a.g1[blk_index(ip, kG1, j)] = (float)o[j];
        q_coeffs(r, a.vs[ip], a.gs[ip], a.w0, a.alpha, a.L, a.media, o);
        for (int j = 0; j < 2; ++j) a.g1[blk_index(ip, kG1, 2 + j)] = (float)o[j];
        for (int j = 0; j < kFam; ++j) a.s[j * a.N + ip] = (float)o[j];
        // (rho = 0: every coefficient is 0)
        a.g1[blk_index(ip, kG1, 4)] = r != 0.0 ? (float)(a.alpha / (r * (a.w0 * a.w0) * (a.L * a.L))) : 0.f;
        if (a.vti) {
            const double e = a.eps[ip], dl = a.del[ip], vp = a.vp[ip], vs = a.vs[ip];
            const double vh = e == 0.0 ? vp : vp * sqrt(1.0 + 2.0 * e);
            q_coeffs(r, vh, a.gp[ip], a.w0, a.alpha, a.L, a.media, o);
            for (int j = 0; j < 2; ++j) a.g2[blk_index(ip, kG2, j)] = (float)o[j];
            double vd = vp;
            if (dl != 0.0) {
                const double c33 = r * vp * vp, c44 = r * vs * vs;
                const double prod = (c33 - c44) * (c33 * (1.0 + 2.0 * dl) - c44);
                vd = sqrt((sqrt(prod > 0.0 ? prod : 0.0) + c44) / r);
            }
            q_coeffs(r, vd, a.gp[ip], a.w0, a.alpha, a.L, a.media, o);
            for (int j = 0; j < 2; ++j) a.g2[blk_index(ip, kG2, 2 + j)] = (float)o[j];
        }
    }
}

// 8-corner cube average of the S set (cuviscoelas_3D.cu:903-907) and the
// buoyancies dt / (0.5 (rho + rho_next)) (cuviscoelas_3D.cu:1077-1092).
struct AvgArgs {
    int nx, ny, nz;
    long long sx, sy, N;
    float dt;
    const float* s;  // [kFam][N]: the S set
    float* gs;       // [kGS][N]: S-bar
    const float* rho;
    float* buoy;     // [3][N]
};

static __global__ __launch_bounds__(256) void k_averages(AvgArgs a)
{
    for (long long ip = (long long)blockIdx.x * 256 + threadIdx.x; ip < a.N; ip += (long long)gridDim.x * 256) {
        const int ix = (int)(ip / a.sx);
        const int iy = (int)((ip - (long long)ix * a.sx) / a.sy);
        const int iz = (int)(ip - (long long)ix * a.sx - (long long)iy * a.sy);
        const bool in = ix < a.nx - 1 && iy < a.ny - 1 && iz < a.nz - 1;
        for (int j = 0; j < kFam; ++j) {
            const float* c_ = a.s + j * a.N;
            auto c = [&](long long q) { return c_[q]; };
            float v = 0.f;
            if (in) {
                const float s8 = c(ip) + c(ip + 1) + c(ip + a.sy) + c(ip + 1 + a.sy) + c(ip + a.sx) + c(ip + a.sx + 1)
                               + c(ip + a.sx + a.sy) + c(ip + a.sx + 1 + a.sy);
                v = 0.125f * s8;
            }
            a.gs[j * a.N + ip] = v;
        }
        // rho + rho' is an FP32 sum in the reference, the rest FP64
        const float r = a.rho[ip];
        a.buoy[ip] = ix < a.nx - 1 ? (float)((double)a.dt / (0.5 * (double)(r + a.rho[ip + a.sx]))) : 0.f;
        a.buoy[a.N + ip] = iy < a.ny - 1 ? (float)((double)a.dt / (0.5 * (double)(r + a.rho[ip + a.sy]))) : 0.f;
        a.buoy[2 * a.N + ip] = iz < a.nz - 1 ? (float)((double)a.dt / (0.5 * (double)(r + a.rho[ip + 1]))) : 0.f;
    }
}

}  // namespace qvti
