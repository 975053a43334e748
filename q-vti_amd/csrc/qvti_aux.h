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
// The sets P, H and D share rho and g, so the stress update reads c of each
// set, g, rho and forms the four in FP64 per cell, each rounded once
// (set_coeffs): 9 fields instead of 16 (VTI; 6 instead of 8 isotropic).  c is
// held as an FP32 value and 16 bits more, exact to 2^-40, so that the four are
// rounded as from the FP64 c but for about one in 30000, which lies that close
// to a rounding boundary (with 8 bits it was one in 150).
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

// c as an FP32 value and 16 signed bits: c = hi (1 + low 2^-39)
__device__ __forceinline__ int low_bits(double c, float hi)
{
    const double x = rint((c - (double)hi) / (double)hi * 0x1p39);
    return fabs(x) <= 32768.0 ? (int)fmin(x, 32767.0) : 0;  // (0 or not finite: no low bits)
}

// The four coefficients of one moduli set in the stress update (q_coeffs).
__device__ __forceinline__ void set_coeffs(float (&o)[kFam], float hi, int low, double g, double rho,
                                           const MediumConst& k)
{
    const double h = hi;
    const double c = fma(h * 0x1p-39, (double)low, h);
    const double rc = rho * c, M = rc * c, Mg = M * g, Mg2 = Mg * g;
    o[0] = (float)(rc * g * k.k0);
    o[1] = (float)fma(Mg2, k.s4, M);
    o[2] = (float)(Mg * c * k.k2);
    o[3] = (float)(Mg2 * k.k3);
}

// (blocked field groups and coefficient group sizes: qvti_layout.h)

struct CoefArgs {
    long long N;
    int vti, media;
    double w0, alpha, L;
    const float *vp, *gp, *vs, *gs, *rho, *eps, *del;
    float* gm;   // blocked [N/64][kGM][64]
    float* low;  // [N]: low bits of H and D (VTI only)
    float* s;    // [kFam][N]: the coefficients of the set S, averaged by k_averages
};

static __global__ __launch_bounds__(256) void k_coefficients(CoefArgs a)
{
    for (long long ip = (long long)blockIdx.x * 256 + threadIdx.x; ip < a.N; ip += (long long)gridDim.x * 256) {
        const double r = a.rho[ip], half_pi = 3.1415926 / 2.0;
        const float gp = a.media == 2 ? 0.f : a.gp[ip], gs = a.media == 2 ? 0.f : a.gs[ip];
        const int nf = kGM(a.vti);
        auto put = [&](int f, float v) { a.gm[blk_index(ip, nf, f)] = v; };
        const double cosp = cos((double)gp * half_pi), coss = cos((double)gs * half_pi);
        // two speeds and the word of their low bits
        auto speeds = [&](int f0, double c0, int f1, double c1) {
            put(f0, (float)c0);
            put(f1, (float)c1);
            return __int_as_float((low_bits(c0, (float)c0) & 0xffff) | (low_bits(c1, (float)c1) << 16));
        };
        put(GM_LOW, speeds(GM_CP, a.vp[ip] * cosp, GM_CS, a.vs[ip] * coss));
        if (a.vti) {
            const double e = a.eps[ip], dl = a.del[ip], vp = a.vp[ip], vs = a.vs[ip];
            const double vh = e == 0.0 ? vp : vp * sqrt(1.0 + 2.0 * e);
            double vd = vp;
            if (dl != 0.0) {
                const double c33 = r * vp * vp, c44 = r * vs * vs;
                const double prod = (c33 - c44) * (c33 * (1.0 + 2.0 * dl) - c44);
                vd = sqrt((sqrt(prod > 0.0 ? prod : 0.0) + c44) / r);
            }
            a.low[ip] = speeds(GM_CH, vh * cosp, GM_CD, vd * cosp);
        }
        put(GM_GP, gp);
        put(GM_GS, gs);
        put(GM_RHO, a.rho[ip]);
        double o[kFam];
        q_coeffs(r, a.vs[ip], a.gs[ip], a.w0, a.alpha, a.L, a.media, o);
        for (int j = 0; j < kFam; ++j) a.s[j * a.N + ip] = (float)o[j];
    }
}

// 8-corner cube average of the S set (cuviscoelas_3D.cu:903-907) and the
// buoyancies dt / (0.5 (rho + rho_next)) (cuviscoelas_3D.cu:1077-1092).
struct AvgArgs {
    int nx, ny, nz;
    long long sx, sy, N;
    float dt;
    const float* s;  // [kFam][N]: the S set
    float* gs;       // [kFam][N]: S-bar
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
