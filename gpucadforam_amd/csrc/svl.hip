// Spatially variant lattice (SVL) synthesis: the step before the meshing path
// in the reference application (src/main.cu:3904-4037, spatial_lattice_run).
//
// The reference builds the lattice field as a sum of gratings: for each
// harmonic (i, j, k) of the unit cell's Fourier series it derives a phase
// field phi on a coarse grid by solving D^T D phi = D^T K with conjugate
// gradients (K: the spatially varying grating vector), samples e^{i phi} on a
// grid twice as fine and accumulates Re(c_ijk e^{i phi}).  This file holds
//   * the reference-shaped steps (period/angle data, normalise, finding_phi,
//     the operator, CG, refine/grating, svl accumulation, FFT fill/scale), each
//     with the reference's arithmetic, and
//   * the native form, gpucad_svl_field: the right-hand side of finding_phi
//     is linear in (i, j, k), so three solves (unit wave numbers) replace one
//     solve per harmonic; the three are solved together (one CG over three
//     right-hand sides, all scalars on the device, no per-iteration host
//     round trip) and one fused pass upsamples the three phase fields and
//     sums every harmonic per fine point as products of e^{i Phi_x},
//     e^{i Phi_y}, e^{i Phi_z}.
//   * the unit-cell Fourier coefficients by separable direct DFT (FP64 accumulation)
//     for exactly the (2r+1)^3 coefficients the reference keeps.
#include <cmath>

#include "gc_common.hpp"
#include "gc_math.hpp"

namespace gc {

int enqueue_minmax0(const float *in, uint64_t n, float2 *part, hipStream_t st);

namespace {

constexpr float kInv2Pi = (float)0.15915494309189533577;  // 1/(2 pi), binary32
constexpr double kTwoPi = 6.283185307179586476925286766559;

// cos/sin of an angle in radians through the revolution polynomials
__device__ __forceinline__ float cos_rad(float t) { return cos_rev(t * kInv2Pi); }
__device__ __forceinline__ float sin_rad(float t) { return sin_rev(t * kInv2Pi); }

// (x, y, z) of linear point t; grids have fewer than 2^32 points (checked
// at the entry points), so the divisions are 32-bit
__device__ __forceinline__ void point_xyz(uint64_t t, int nx, int ny, int *x, int *y, int *z) {
    const uint32_t tt = (uint32_t)t, plane = (uint32_t)nx * (uint32_t)ny;
    const uint32_t zz = tt / plane;
    const uint32_t r = tt - zz * plane;
    const uint32_t yy = r / (uint32_t)nx;
    *z = (int)zz;
    *y = (int)yy;
    *x = (int)(r - yy * (uint32_t)nx);
}

// n / d for n < 2^32 through a double reciprocal and one correction step
struct Div32 {
    uint32_t d;
    double inv;
};
inline Div32 make_div32(uint32_t d) { return Div32{d, 1.0 / (double)d}; }
__device__ __forceinline__ uint32_t div32(uint32_t n, const Div32 &f) {
    uint32_t q = (uint32_t)((double)n * f.inv);
    const int64_t r = (int64_t)n - (int64_t)q * f.d;
    if (r < 0) --q;
    else if (r >= (int64_t)f.d) ++q;
    return q;
}
__device__ __forceinline__ void point_xyz(uint32_t t, const Div32 &dnx, const Div32 &dplane,
                                          int *x, int *y, int *z) {
    const uint32_t zz = div32(t, dplane);
    const uint32_t r = t - zz * dplane.d;
    const uint32_t yy = div32(r, dnx);
    *z = (int)zz;
    *y = (int)yy;
    *x = (int)(r - yy * dnx.d);
}

// ---------------------------------------------------------------------------
// period and angle data (src/lattice_files/Gratings.cu:775-860)
// ---------------------------------------------------------------------------
__global__ void period_angle_kernel(float *out, int nx, int ny, int nz, float dx, float dy,
                                    float dz, float mx, float my, float mz, int axis, int angle) {
    const uint64_t n = (uint64_t)nx * ny * nz;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x) {
        int xx, yy, zz;
        point_xyz(t, nx, ny, &xx, &yy, &zz);
        const float x = ((float)xx - mx) * dx;
        const float y = ((float)yy - my) * dy;
        const float z = ((float)zz - mz) * dz;
        float v;
        if (angle) {
            v = axis == 'y' ? atan2_poly(z + 1.0f, x + 1.0f) : atan2_poly(y + 1.0f, x + 1.0f);
        } else {
            float u, w;
            if (axis == 'z') {
                u = x + 1.0f;
                w = y + 1.0f;
            } else if (axis == 'y') {
                u = x + 1.0f;
                w = z + 1.0f;
            } else {
                u = z + 1.0f;
                w = y + 1.0f;
            }
            v = __builtin_sqrtf(u * u + w * w);
        }
        out[t] = v;
    }
}

// k = (f - a)/(b - a); out = a1 + b1 k (three) or k (buffer); (a, b) = part[0]
__global__ void rescale_kernel(const float *in, float *out, uint64_t n, const float2 *ab,
                               float a1, float b1, int affine) {
    const float a = ab->x, b = ab->y;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x) {
        const float k = (in[t] - a) / (b - a);
        out[t] = affine ? a1 + b1 * k : k;
    }
}

// ---------------------------------------------------------------------------
// finding_phi: right-hand side D^T K of one harmonic (Gratings.cu:100-417)
// ---------------------------------------------------------------------------
struct PhiArgs {
    int nx, ny, nz;
    int i, j, k;
    float dx, dy, dz;
    int type;          // 'n' 'b' 'r' 's'
    int uniform_type;  // 0 const, 1 per axis, 2 period field
    float const_period, x_period, y_period, z_period;
    float lcon, lcon_1;
    int sinewave_zaxis;
};

// stencil weights and the two neighbours of coordinate c in [0, n)
__device__ __forceinline__ void axis_weights(int c, int n, float *w1, float *w2, int *c1, int *c2) {
    if (c == 0) {
        *w1 = -1.0f; *w2 = -0.5f; *c1 = c; *c2 = c + 1;
    } else if (c == 1) {
        *w1 = 1.0f; *w2 = -0.5f; *c1 = c - 1; *c2 = c + 1;
    } else if (c == n - 2) {
        *w1 = 0.5f; *w2 = -1.0f; *c1 = c - 1; *c2 = c + 1;
    } else if (c == n - 1) {
        *w1 = 0.5f; *w2 = 1.0f; *c1 = c - 1; *c2 = c;
    } else {
        *w1 = 0.5f; *w2 = -0.5f; *c1 = c - 1; *c2 = c + 1;
    }
}

// (2 pi / per) * w, the reference's double expression rounded to binary32
__device__ __forceinline__ float wave(float per, float w) {
    return (float)((kTwoPi / (double)per) * (double)w);
}

// lcon * sin(6.28 * lcon_1 * u): the product in double as the reference's
// double literal makes it, the sine of the binary32 argument
__device__ __forceinline__ float sine_angle(float lcon, float lcon_1, float u) {
    const float arg = (float)((6.28 * (double)lcon_1) * (double)u);
    return lcon * sin_rad(arg);
}

__global__ void finding_phi_kernel(float *phi, const float *period, PhiArgs p) {
    const uint64_t n = (uint64_t)p.nx * p.ny * p.nz;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x) {
        int x, y, z;
        point_xyz(t, p.nx, p.ny, &x, &y, &z);
        float a1, a2, b1, b2, c1, c2;
        int x1, x2, y1, y2, z1, z2;
        axis_weights(x, p.nx, &a1, &a2, &x1, &x2);
        axis_weights(y, p.ny, &b1, &b2, &y1, &y2);
        axis_weights(z, p.nz, &c1, &c2, &z1, &z2);
        float th1 = 0.f, th2 = 0.f, th3 = 0.f, th4 = 0.f, th5 = 0.f, th6 = 0.f, th7 = 0.f,
              th8 = 0.f;
        if (p.type == 'r' || p.type == 'b') {
            const float mx = p.type == 'r' ? (float)(p.nx + 1) / 2.0f : 0.f;
            const float my = p.type == 'r' ? (float)(p.ny + 1) / 2.0f : 0.f;
            const float yy = ((float)(y + 1) - my) * p.dx;
            th1 = atan2_poly(yy, ((float)(x1 + 1) - mx) * p.dx);
            th2 = atan2_poly(yy, ((float)(x2 + 1) - mx) * p.dx);
            const float xx = ((float)(x + 1) - mx) * p.dx;
            th3 = atan2_poly(((float)(y1 + 1) - my) * p.dx, xx);
            th4 = atan2_poly(((float)(y2 + 1) - my) * p.dx, xx);
        } else if (p.type == 's') {
            th1 = sine_angle(p.lcon, p.lcon_1, (float)(x1 + 1) * p.dx);
            th5 = sine_angle(p.lcon, p.lcon_1, (float)(z1 + 1) * p.dz);
            th2 = sine_angle(p.lcon, p.lcon_1, (float)(x2 + 1) * p.dx);
            th6 = sine_angle(p.lcon, p.lcon_1, (float)(z2 + 1) * p.dz);
            th3 = sine_angle(p.lcon, p.lcon_1, (float)(x + 1) * p.dx);
            th7 = sine_angle(p.lcon, p.lcon_1, (float)(z + 1) * p.dz);
            th4 = th3;
            th8 = th7;
        }
        float per1, per2, per3, per4, per5, per6;
        if (p.uniform_type == 0) {
            per1 = per2 = per3 = per4 = per5 = per6 = p.const_period;
        } else if (p.uniform_type == 1) {
            per1 = per2 = p.x_period;
            per3 = per4 = p.y_period;
            per5 = per6 = p.z_period;
        } else {
            const uint64_t row = (uint64_t)p.nx, plane = (uint64_t)p.nx * p.ny;
            const uint64_t c = (uint64_t)y * row + (uint64_t)z * plane;
            per1 = period[(uint64_t)x1 + c];
            per2 = period[(uint64_t)x2 + c];
            per3 = period[(uint64_t)x + (uint64_t)y1 * row + (uint64_t)z * plane];
            per4 = period[(uint64_t)x + (uint64_t)y2 * row + (uint64_t)z * plane];
            per5 = period[(uint64_t)x + (uint64_t)y * row + (uint64_t)z1 * plane];
            per6 = period[(uint64_t)x + (uint64_t)y * row + (uint64_t)z2 * plane];
        }
        const float fi = (float)p.i, fj = (float)p.j, fk = (float)p.k;
        float kx1 = wave(per1, fi * cos_rad(th1) - fj * sin_rad(th1));
        float kx2 = wave(per2, fi * cos_rad(th2) - fj * sin_rad(th2));
        float ky1 = wave(per3, fi * sin_rad(th3) + fj * cos_rad(th3));
        float ky2 = wave(per4, fi * sin_rad(th4) + fj * cos_rad(th4));
        float kz1 = wave(per5, fk);
        float kz2 = wave(per6, fk);
        float ph = (__builtin_fmaf(a1, kx1, a2 * kx2) + __builtin_fmaf(b1, ky1, b2 * ky2)) +
                   __builtin_fmaf(c1, kz1, c2 * kz2);
        if (p.type == 's' && p.sinewave_zaxis) {
            kz1 = wave(per5, fj * sin_rad(th5) + fk * cos_rad(th5));
            kz2 = wave(per6, fj * sin_rad(th6) + fk * cos_rad(th6));
            ky1 = wave(per3, fj * cos_rad(th7) - fk * sin_rad(th7));
            ky2 = wave(per4, fj * cos_rad(th8) - fk * sin_rad(th8));
            kx1 = wave(per1, fi);
            kx2 = wave(per2, fi);
            ph += (__builtin_fmaf(a1, kx1, a2 * kx2) + __builtin_fmaf(b1, ky1, b2 * ky2)) +
                  __builtin_fmaf(c1, kz1, c2 * kz2);
        }
        phi[t] = ph;
    }
}

// ---------------------------------------------------------------------------
// the operator D^T D of the phase solve (GPUMatvec_lattice_kernel,
// Gratings.cu:420-597): per axis a diagonal weight and two neighbour terms
// ---------------------------------------------------------------------------
// Coordinate c of n (n >= 4) along stride s:
//   c = 0:     w 1.25, t2 = -d(t+s),         t3 = -0.25 d(t+2s)
//   c = 1:     w 1.25, t2 = -d(t-s),         t3 = -0.25 d(t+2s)
//   c = n-2:   w 1.25, t2 = -0.25 d(t-2s),   t3 = -d(t+s)
//   c = n-1:   w 1.25, t2 = -0.25 d(t-2s),   t3 = -d(t-s)
//   otherwise: w 0.5,  t2 = -0.25 d(t-2s),   t3 = -0.25 d(t+2s)
// chosen by selects, so both loads are unconditional (every point's loads
// can be in flight together); -1 * v and -0.25 * v are the exact negation
// and quarter the cases name.
template <class G>
__device__ __forceinline__ void axis_terms(const G &get, int c, int n, int64_t t, int64_t s,
                                           float *w, float *t2, float *t3) {
    const bool lo = c <= 1, hi1 = c == n - 2, hi0 = c == n - 1;
    *w = (lo || hi1 || hi0) ? 1.25f : 0.5f;
    const int64_t o2 = c == 0 ? s : (c == 1 ? -s : -2 * s);
    const float k2 = lo ? -1.0f : -0.25f;
    const int64_t o3 = lo ? 2 * s : (hi1 ? s : (hi0 ? -s : 2 * s));
    const float k3 = lo ? -0.25f : ((hi1 || hi0) ? -1.0f : -0.25f);
    *t2 = k2 * get(t + o2);
    *t3 = k3 * get(t + o3);
}

// (wx + wy + wz) * d + x2 + x3 + y2 + y3 + z2 + z3 in this order, the first
// product and sum fused (the reference's contracted form)
template <class G>
__device__ __forceinline__ float apply_op(const G &get, int x, int y, int z, int nx, int ny,
                                          int nz, int64_t t) {
    float wx, x2, x3, wy, y2, y3, wz, z2, z3;
    axis_terms(get, x, nx, t, 1, &wx, &x2, &x3);
    axis_terms(get, y, ny, t, (int64_t)nx, &wy, &y2, &y3);
    axis_terms(get, z, nz, t, (int64_t)nx * ny, &wz, &z2, &z3);
    const float w = (wx + wy) + wz;
    float a = __builtin_fmaf(w, get(t), x2);
    a = a + x3;
    a = a + y2;
    a = a + y3;
    a = a + z2;
    a = a + z3;
    return a;
}

__global__ void matvec_kernel(const float *d, float *q, int nx, int ny, int nz) {
    const uint64_t n = (uint64_t)nx * ny * nz;
    auto get = [d](int64_t i) { return d[i]; };
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x) {
        int x, y, z;
        point_xyz(t, nx, ny, &x, &y, &z);
        q[t] = apply_op(get, x, y, z, nx, ny, nz, (int64_t)t);
    }
}

// ---------------------------------------------------------------------------
// conjugate gradients over m right-hand sides (GPUCG_lattice,
// Gratings.cu:875-974, scalars kept on the device)
// ---------------------------------------------------------------------------
constexpr int kCgThreads = 256;
constexpr int kCgBlocks = 512;  // blocks of the stand-alone dot product
constexpr int kCgResident = 1280;  // CG workgroups over all right-hand sides (5 per CU)
constexpr int kMaxRhs = 4;

struct CgState {
    float delta[2];  // r.r of the last two iterations (by iteration parity)
    int done;
    int iters;       // the reference's FinalIter
    float res;       // the reference's FinalRes = sqrt(r.r)
    uint32_t tiles;  // tiles whose part of the solution is written (cg_chip_kernel)
    int pad[2];
};

constexpr int kCgUnroll = 2;  // points per thread and step, all their loads in flight
constexpr int kCgStep = kCgThreads * kCgUnroll;

struct CgArgs {
    int nx, ny, nz, G;             // G: workgroups per right-hand side, a multiple of 8
    uint64_t n, C;                 // C: points per workgroup range, a multiple of kCgThreads
    Div32 dnx, dplane;
    float *phi, *r, *q, *d0, *d1;  // m vectors of n each (right-hand side s at s*n)
    double *pq, *prr;              // partial sums: pq[m][G], prr[2][m][G]
    CgState *st;
    int max_iter;
    float term;                    // end_res^2
};

__device__ __forceinline__ double block_sum(double v) {
    __shared__ double s[kCgThreads];
    __syncthreads();
    s[threadIdx.x] = v;
    __syncthreads();
    for (int w = kCgThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    return s[0];
}

// one step of the wave sum: v plus the DPP-moved v (0 where no lane is the source)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
    return v + __longlong_as_double((long long)((uint64_t)(uint32_t)hi << 32 | (uint32_t)lo));
}
// sum over the 64 lanes, the same in every lane (DPP moves: no LDS)
__device__ __forceinline__ double wave_sum_d(double v) {
    v = dpp_add<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8 within rows of 16 lanes
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15, 31: lane 63 holds the sum
    v = dpp_add<0x143, 0xc>(v);
    const long long b = __double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)b, 63);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}

// the same fixed-order sum of G partials in every block (so every block
// takes the same decisions without communicating)
__device__ __forceinline__ double sum_partials(const double *p, int G) {
    double v = 0.0;
    for (int i = threadIdx.x; i < G; i += kCgThreads) v += p[i];
    return block_sum(v);
}

// Points [lo, hi) of workgroup blockIdx.x.  Workgroups are dispatched to
// the 8 XCDs round robin, so range (b % 8) * (G / 8) + b / 8 gives each XCD
// one contiguous run of z planes: the operator's neighbours (two planes up
// and down) then sit in the L2 of the XCD that reads them.
__device__ __forceinline__ void cg_range(const CgArgs &a, uint64_t *lo, uint64_t *hi) {
    const uint32_t b = blockIdx.x;
    const uint64_t r = (uint64_t)((b & 7u) * ((uint32_t)a.G >> 3) + (b >> 3));
    *lo = r * a.C < a.n ? r * a.C : a.n;
    *hi = *lo + a.C < a.n ? *lo + a.C : a.n;
}

__global__ void cg_init_kernel(const float *b, CgArgs a) {
    const int s = blockIdx.y;
    const uint64_t off = (uint64_t)s * a.n;
    uint64_t lo, hi;
    cg_range(a, &lo, &hi);
    double acc = 0.0;
    for (uint64_t t = lo + threadIdx.x; t < hi; t += kCgThreads) {
        const float v = b[off + t];
        a.phi[off + t] = 0.0f;
        a.r[off + t] = v;
        a.d0[off + t] = v;
        acc += (double)v * (double)v;
    }
    const double tot = block_sum(acc);
    if (threadIdx.x == 0) a.prr[(uint64_t)s * a.G + blockIdx.x] = tot;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        CgState z = {};
        a.st[s] = z;
    }
}

// iteration it, first half: convergence test, d_it = r + beta d_{it-1}
// (recomputed for the stencil's neighbours), q = A d_it, partial d.q
__global__ void cg_a_kernel(CgArgs a, int it) {
    const int s = blockIdx.y;
    if (a.st[s].done) return;
    const uint64_t m_off = (uint64_t)s * a.n;
    const int m = gridDim.y;
    const double *prr = a.prr + ((uint64_t)(it & 1) * m + s) * a.G;
    const float delta = (float)sum_partials(prr, a.G);
    // the reference loops while (iCounter < iter && delta_new > term),
    // iCounter = it + 1
    if (!(it + 1 < a.max_iter && delta > a.term)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            a.st[s].iters = it + 1;
            a.st[s].res = sqrtf(delta);
            a.st[s].done = 1;
        }
        return;
    }
    const float beta = it == 0 ? 0.0f : delta / a.st[s].delta[(it + 1) & 1];
    if (blockIdx.x == 0 && threadIdx.x == 0) a.st[s].delta[it & 1] = delta;
    float *dcur = (it & 1 ? a.d1 : a.d0) + m_off;
    const float *r = a.r + m_off;
    const bool first = it == 0;
    // d = r + beta d_prev; the first direction is r itself (fma(0, r, r) = r
    // exactly), so one load pattern serves every iteration
    const float *dprev = first ? r : ((it - 1) & 1 ? a.d1 : a.d0) + m_off;
    const float bt = first ? 0.0f : beta;
    auto get = [=](int64_t i) { return __builtin_fmaf(bt, dprev[i], r[i]); };
    // points t0 + u * kCgThreads (u < kCgUnroll) per step: every load of the
    // step is issued before its stores; the partial sum adds a thread's points
    // in increasing order
    uint64_t lo, hi;
    cg_range(a, &lo, &hi);
    double acc = 0.0;
    for (uint64_t t0 = lo + threadIdx.x; t0 < hi; t0 += kCgStep) {
        float dv[kCgUnroll], qv[kCgUnroll];
#pragma unroll
        for (int u = 0; u < kCgUnroll; ++u) {
            const uint32_t t = (uint32_t)(t0 + u * kCgThreads < hi ? t0 + u * kCgThreads : t0);
            int x, y, z;
            point_xyz(t, a.dnx, a.dplane, &x, &y, &z);
            dv[u] = get((int64_t)t);
            qv[u] = apply_op(get, x, y, z, a.nx, a.ny, a.nz, (int64_t)t);
        }
#pragma unroll
        for (int u = 0; u < kCgUnroll; ++u) {
            const uint64_t t = t0 + u * kCgThreads;
            if (t < hi) {
                if (!first) dcur[t] = dv[u];
                a.q[m_off + t] = qv[u];
                acc += (double)dv[u] * (double)qv[u];
            }
        }
    }
    const double tot = block_sum(acc);
    if (threadIdx.x == 0) a.pq[(uint64_t)s * a.G + blockIdx.x] = tot;
}

// iteration it, second half: alpha = delta / d.q, phi += alpha d,
// r -= alpha q, partial r.r for the next test
__global__ void cg_b_kernel(CgArgs a, int it) {
    const int s = blockIdx.y;
    if (a.st[s].done) return;
    const uint64_t m_off = (uint64_t)s * a.n;
    const int m = gridDim.y;
    const float dq = (float)sum_partials(a.pq + (uint64_t)s * a.G, a.G);
    const float alpha = a.st[s].delta[it & 1] / dq;
    const float *d = (it & 1 ? a.d1 : a.d0) + m_off;
    float *phi = a.phi + m_off, *r = a.r + m_off;
    const float *q = a.q + m_off;
    uint64_t lo, hi;
    cg_range(a, &lo, &hi);
    double acc = 0.0;
    for (uint64_t t0 = lo + threadIdx.x; t0 < hi; t0 += kCgStep) {
        float dv[kCgUnroll], pv[kCgUnroll], qv[kCgUnroll], rv[kCgUnroll];
#pragma unroll
        for (int u = 0; u < kCgUnroll; ++u) {
            const uint32_t t = (uint32_t)(t0 + u * kCgThreads < hi ? t0 + u * kCgThreads : t0);
            dv[u] = d[t];
            pv[u] = phi[t];
            qv[u] = q[t];
            rv[u] = r[t];
        }
#pragma unroll
        for (int u = 0; u < kCgUnroll; ++u) {
            const uint64_t t = t0 + u * kCgThreads;
            if (t < hi) {
                phi[t] = __builtin_fmaf(alpha, dv[u], pv[u]);
                const float rn = __builtin_fmaf(-alpha, qv[u], rv[u]);
                r[t] = rn;
                acc += (double)rn * (double)rn;
            }
        }
    }
    const double tot = block_sum(acc);
    if (threadIdx.x == 0) a.prr[((uint64_t)((it + 1) & 1) * m + s) * a.G + blockIdx.x] = tot;
}

// ---------------------------------------------------------------------------
// The same iteration in one launch, for grids whose vectors fit on the chip
// ---------------------------------------------------------------------------
// The two-launch form moves ten vectors through memory per iteration and pays
// two launches.  Here a workgroup keeps a tile of one right-hand side for
// the whole solve: r, phi and q in registers (a thread owns a column of the
// tile, one (x, y), and its z run), d in LDS with two points around the tile.
// Tiles span the grid along x and split y and z.  Per iteration the tiles
// exchange r on their faces (two layers; each tile updates its halo of d by the
// same d = r + beta d as the owner, so d needs no exchange) and meet twice, in
// the sums d.q and r.r.  Every element sees the arithmetic of the two-launch
// form in the same order.  The sums are FP64 over the same products, in tiles'
// order instead of ranges', so alpha and beta are the same floats unless the two
// round to different ones (in none of 13 solves compared, of 4^3 to 162^3 with one
// and three right-hand sides, up to 391 iterations: all bits the same).
//
// There are no fences: an exchanged value travels in one 8-byte word with the
// number of its iteration, written and read by relaxed agent-scope atomics,
// so a word is valid as soon as its number is the expected one.  A face or sum
// word is written again only after its writer passed a sum that every reader
// posted to after reading the word's last value.
//
// All workgroups must be resident together: at most one per CU is launched.
// Every wait is bounded in time: should other work hold the CUs that long, the
// waiting workgroups leave.  A tile that leaves may have posted its sums, so
// others, the first one too, can still reach the end: the solution is complete
// only when every tile has counted itself after writing its part.  Otherwise
// the caller solves by the two-launch form; x has not been written.
//
// Measured (us per iteration of whole calls, two-launch form -> this): three
// right-hand sides of 120^3 50 -> 20.3 (41 in its kernels alone), of 100^3 35.6 -> 12.9;
// one of 162^3 45.4 -> 21.0, of 120^3 26.6 -> 12.4, of 61 x 57 x 70 13.7 -> 8.0, of 12^3
// (12 tiles) 12.1 -> 6.0, of 4^3 (one tile, nothing to wait for) 11.7 -> 4.2.
// What is left is latency: two exchanges of about 2 us each and the barriers of a
// workgroup that fills its CU.
constexpr int kChipThreads = 1024;            // most threads of a tile's workgroup
constexpr int kChipZ = 24;                    // longest z run of a tile
constexpr int kYPass = 3;                     // most passes over a halo layer of a y side
constexpr size_t kChipLds = 160 * 1024 - 1024;  // LDS of a tile's d (1 KB: the sums)
// Longest wait: 5 ms of the 100 MHz clock, about what a whole solve takes (1 ms
// for 61^3, 6 ms for three of 120^3) and less than the two-launch form adds to it.
constexpr int64_t kChipWaitTicks = 500000;
// After a solve gave up, the next ones on its device go straight to two
// launches: what held the CUs (another process, a long kernel of another
// stream, a CU mask) mostly still does, and a loop over 62 harmonics would wait
// in each.  One in 64 tries again, which costs such a loop 0.1 ms per solve.
constexpr int kChipPause = 64;
int g_chip_pause[64];  // solves left to take so, per device; under lock_device_calls()

struct ChipArgs {
    int nx, ny, nz, m, ty, tz, G;  // G = ty * tz tiles per right-hand side
    uint64_t n;
    const float *b;             // m right-hand sides
    float *phi;                 // their solutions, complete when each has G finished tiles
    uint64_t *faces;            // [m][G][4][face_words]: r, iteration
    uint64_t *sums;             // [m][2][G][2]: FP64 halves, iteration
    uint32_t face_words;
    uint32_t *abort;            // set by a workgroup whose wait ran out
    CgState *st;
    int max_iter;
    float term;
    // longest wait of a right-hand side's first tile and of the others, in ticks
    // of the 100 MHz clock; negative: the first wait ends at once
    int64_t wait_first, wait_others;
};

// The same value, unknown to the optimiser: what is computed from it inside the
// iteration stays there instead of being held in registers throughout.
__device__ __forceinline__ int here(int v) {
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ int here_uniform(int v) {
    asm volatile("" : "+s"(v));
    return v;
}

struct ChipShared {
    double part[kChipThreads / 64], total[kChipThreads / 64];
    int abort;
};

__device__ __forceinline__ void post_word(uint64_t *p, uint32_t value, uint32_t it) {
    __hip_atomic_store(p, (uint64_t)it << 32 | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t read_word(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A bounded wait: false once the time has run out or another workgroup gave up.
struct ChipWait {
    int64_t limit, start = 0;
    uint32_t turns = 0;
    __device__ __forceinline__ explicit ChipWait(int64_t ticks) : limit(ticks) {}
    __device__ __forceinline__ bool again(uint32_t *abort) {
        if (limit >= 0 && (++turns & 63u) != 0) return true;
        const int64_t now = (int64_t)wall_clock64();
        if (start == 0) start = now;
        if (now - start > limit)
            __hip_atomic_store(abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
    }
};

// Sum of v over the workgroups of a right-hand side, the same bits in every
// one (each sums all of them in the same order), in two halves: the
// workgroup's own sum is posted, and then all of them are collected (false
// when a wait ran out).  One barrier each.
__device__ __forceinline__ void chip_post(double v, uint64_t *slots, int g, uint32_t it,
                                          ChipShared &sh) {
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6, waves = (int)blockDim.x >> 6;
    v = wave_sum_d(v);
    if (lane == 0) sh.part[wave] = v;
    __syncthreads();
    if (wave == 0) {
        const double w = wave_sum_d(lane < waves ? sh.part[lane] : 0.0);
        if (lane == 0 && sh.abort == 0) {  // (a sum without its halo is not posted)
            const uint64_t bits = (uint64_t)__double_as_longlong(w);
            post_word(slots + 2 * g, (uint32_t)(bits >> 32), it);
            post_word(slots + 2 * g + 1, (uint32_t)bits, it);
        }
    }
}
__device__ __forceinline__ bool chip_collect(const uint64_t *slots, int G, uint32_t it,
                                             uint32_t *abort, int64_t limit, ChipShared &sh,
                                             double *total) {
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6, used = (G + 63) >> 6;
    if (wave < used) {
        double w = 0.0;
        bool ok = true;
        if (t < G) {
            ChipWait wait(limit);
            uint64_t hi, lo;
            for (;;) {
                hi = read_word(slots + 2 * t);
                lo = read_word(slots + 2 * t + 1);
                if (limit >= 0 && (uint32_t)(hi >> 32) == it && (uint32_t)(lo >> 32) == it) break;
                if (!wait.again(abort)) {
                    ok = false;
                    break;
                }
            }
            w = __longlong_as_double((long long)(hi << 32 | (lo & 0xffffffffull)));
        }
        if (!ok) sh.abort = 1;
        w = wave_sum_d(w);
        if (lane == 0) sh.total[wave] = w;
    }
    __syncthreads();
    double s = 0.0;
    for (int i = 0; i < used; ++i) s += sh.total[i];
    *total = s;
    return sh.abort == 0;
}

// the two neighbour terms of coordinate c of n (axis_terms): offsets in points and weights
struct AxisTerms {
    int o2, o3;
    float w, k2, k3;
};
__device__ __forceinline__ AxisTerms axis_terms_at(int c, int n) {
    const bool lo = c <= 1, hi1 = c == n - 2, hi0 = c == n - 1;
    AxisTerms a;
    a.w = (lo || hi1 || hi0) ? 1.25f : 0.5f;
    a.o2 = c == 0 ? 1 : (c == 1 ? -1 : -2);
    a.k2 = lo ? -1.0f : -0.25f;
    a.o3 = lo ? 2 : (hi1 ? 1 : (hi0 ? -1 : 2));
    a.k3 = lo ? -0.25f : ((hi1 || hi0) ? -1.0f : -0.25f);
    return a;
}

// A tile's z runs are held in registers: KZ is the tiles' longest run rounded
// up to 4, and every run is at least KZ - 4.  The z loops are unrolled over KZ
// with the arrays assigned in every step and no branch around a step (steps
// past the run compute on its last plane and are not stored, summed or sent):
// branches that merge the arrays made the compiler spill them.
template <int KZ>
__global__ void __launch_bounds__(kChipThreads) cg_chip_kernel(ChipArgs a) {
    extern __shared__ float lds_d[];
    __shared__ ChipShared sh;
    // workgroups are dispatched to the 8 XCDs round robin: each XCD gets a
    // contiguous run of tiles (y fastest), so most faces are exchanged through
    // its own L2
    const int tile = (int)((blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3));
    if (tile >= a.G * a.m) return;
    const int s = tile / a.G, g = tile - s * a.G, t = (int)threadIdx.x;
    const int iy = g % a.ty, iz = g / a.ty, nx = a.nx;
    const int y0 = (int)((int64_t)a.ny * iy / a.ty), y1 = (int)((int64_t)a.ny * (iy + 1) / a.ty);
    const int z0 = (int)((int64_t)a.nz * iz / a.tz), z1 = (int)((int64_t)a.nz * (iz + 1) / a.tz);
    const int by = y1 - y0, bz = z1 - z0;
    const bool ylo = iy > 0, yhi = iy + 1 < a.ty, zlo = iz > 0, zhi = iz + 1 < a.tz;
    const int rows = (int)blockDim.x / nx;  // tile rows a pass of the workgroup covers
    const int row = t / nx, x = t - row * nx;
    const bool own = row < by;              // (rows >= by)
    const int64_t limit = g == 0 ? a.wait_first : a.wait_others;
    const int ty = own ? row : 0;           // threads without a column follow column 0's
    const float *b = a.b + (uint64_t)s * a.n;
    if (t == 0) sh.abort = 0;
    __syncthreads();

    // d in LDS: the tile's planes with two rows before and after, then two
    // planes below and two above (by rows each)
    const int ps = (by + 4) * nx, zoff = bz * ps;
    // (point of column offset xy = y nx + x in plane z, or in layer l, 0 next
    // to the tile, of a z side)
    auto at = [=](int xy, int z) { return z * ps + 2 * nx + xy; };
    auto at_z = [=](int side, int l, int xy) { return zoff + (2 * side + l) * by * nx + xy; };
    // The column offset and the position within the grid are taken through
    // here() in every phase: what derives from them is computed there instead of
    // being held in registers over the whole iteration.
    const int column = ty * nx + x;
    auto face = [=](int tile, int f) {
        return a.faces + (((uint64_t)s * a.G + tile) * 4 + f) * a.face_words;
    };
    // Past the grid's ends along z the halo holds the point whose -d the
    // operator takes there (axis_terms: rows 0, 1, nz - 2, nz - 1 have -d(1),
    // -d(0), -d(nz - 1), -d(nz - 2) in the place of -0.25 d two planes off), so
    // every plane has the one form k d(-2) + k' d(+2).
    auto ghosts = [&](int n) {  // from the thread's own column
        const int xy = here(column), c = at(xy, 0), cz = at_z(0, 0, xy);
        if (!zlo && own) {
            lds_d[cz] = lds_d[c];
            lds_d[cz + by * nx] = lds_d[c + ps];
        }
        if (!zhi && own) {
            lds_d[cz + 2 * by * nx] = lds_d[c + (n - 1) * ps];
            lds_d[cz + 3 * by * nx] = lds_d[c + (n - 2) * ps];
        }
    };
    // step z exists: only the last four steps can be past the run
#define GC_IN_RUN(z, n) ((z) < KZ - 4 || (z) < (n))

    float r[KZ], phi[KZ], q[KZ];
    double acc = 0.0;
    {
        const float *bp = b + ((uint64_t)z0 * a.ny + (y0 + ty)) * nx + x;
        const uint64_t plane = (uint64_t)a.ny * nx;
#pragma unroll
        for (int z = 0; z < KZ; ++z) {
            phi[z] = 0.f;
            r[z] = bp[(uint64_t)min(z, bz - 1) * plane];
            if ((z & 3) == 3) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int z = 0; z < KZ; ++z)
            if (GC_IN_RUN(z, bz) && own) {
                lds_d[at(column, z)] = r[z];
                acc += (double)r[z] * (double)r[z];
            }
    }
    ghosts(bz);
    // The halo's rows: layer l of a y side has a row per z (thread row `row`
    // takes rows row + p * rows, p < kYPass), layer l of a z side a row per y (its
    // own column's).  Its first values come from b, later ones from the faces:
    // face 0 / 1 holds the tile's first / last two rows, 2 / 3 its first / last two
    // planes, layer by layer from the outside.
    if (row < rows) {
        for (int l = 0; l < 2; ++l)
            for (int z = row; z < bz; z += rows) {
                const float *p = b + ((uint64_t)(z0 + z) * a.ny + y0) * nx + x;
                if (ylo) lds_d[at((-1 - l) * nx + x, z)] = p[-(1 + l) * nx];
                if (yhi) lds_d[at((by + l) * nx + x, z)] = p[(by + l) * nx];
            }
        for (int l = 0; l < 2; ++l) {
            const float *p = b + ((uint64_t)z0 * a.ny + y0 + ty) * nx + x;
            const int64_t plane = (int64_t)a.ny * nx;
            if (own && zlo) lds_d[at_z(0, l, column)] = p[-(1 + l) * plane];
            if (own && zhi) lds_d[at_z(1, l, column)] = p[(bz + l) * plane];
        }
    }
    uint64_t *const sums_dq = a.sums + (uint64_t)s * 4 * a.G, *const sums_rr = sums_dq + 2 * a.G;
    const bool fetch = row < rows;

    double tot;
    chip_post(acc, sums_rr, g, 1u, sh);
    if (!chip_collect(sums_rr, a.G, 1u, a.abort, limit, sh, &tot)) return;
    float delta = (float)tot, delta_prev = 0.f, beta = 0.f;
    float hy[2][2][kYPass], hz[2][2];  // the halo's r: [side][layer][pass], [side][layer]
    int it = 0;
    for (;; ++it) {
        if (!(it + 1 < a.max_iter && delta > a.term)) break;
        if (it > 0) {
            // d = r + beta d: the tile's own points, then its halo
            const int n = here_uniform(bz), xy = here(column);
            float *d = lds_d + at(xy, 0);
            if (own) {
#pragma unroll
                for (int z = 0; z < KZ; ++z) {
                    if (GC_IN_RUN(z, n)) *d = __builtin_fmaf(beta, *d, r[z]);
                    d += ps;
                    if ((z & 3) == 3) __builtin_amdgcn_sched_barrier(0);
                }
            }
            ghosts(n);
            if (fetch) {
                const int hr = here(row), hx = here(x) + hr * ps;
#pragma unroll
                for (int side = 0; side < 2; ++side) {
                    if (!(side ? yhi : ylo)) continue;
#pragma unroll
                    for (int l = 0; l < 2; ++l) {
                        float *h = lds_d + at(hx + (side ? by + l : -1 - l) * nx, 0);
#pragma unroll
                        for (int p = 0; p < kYPass; ++p) {
                            if (hr + p * rows < n) *h = __builtin_fmaf(beta, *h, hy[side][l][p]);
                            h += rows * ps;
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (own) {
#pragma unroll
                for (int side = 0; side < 2; ++side) {
                    if (!(side ? zhi : zlo)) continue;
#pragma unroll
                    for (int l = 0; l < 2; ++l) {
                        float *h = lds_d + at_z(side, l, xy);
                        *h = __builtin_fmaf(beta, *h, hz[side][l]);
                    }
                }
            }
        }
        __syncthreads();
        // q = A d and d.q; the z terms from a run of five d values
        acc = 0.0;
        {
            const int n = here_uniform(bz), last = by * nx, xy = here(column);
            const int cz = at_z(1, 0, xy);
            int c = at(xy, 0);
            const AxisTerms ax = axis_terms_at(here(x), nx);
            const AxisTerms ay = axis_terms_at(y0 + here(ty), a.ny);
            const int ox2 = ax.o2, ox3 = ax.o3, oy2 = ay.o2 * nx, oy3 = ay.o3 * nx;
            const float wxy = ax.w + ay.w;
            const int lo_edge = here_uniform(zlo ? -1 : 2), hi_edge = here_uniform(zhi ? KZ : bz - 2);
            const float klo = lo_edge > 0 ? -1.0f : -0.25f;
            float dm2 = lds_d[at_z(0, 1, xy)], dm1 = lds_d[at_z(0, 0, xy)];
            float dc = lds_d[c], dp1 = lds_d[c + ps];
            // two planes up: in the tile, in its halo, then past both (not used)
            int up = n > 2 ? c + 2 * ps : cz;
#pragma unroll
            for (int z = 0; z < KZ; ++z) {
                const float dp2 = lds_d[up];
                const float wz = z < lo_edge || z >= hi_edge ? 1.25f : 0.5f;
                float v = __builtin_fmaf(wxy + wz, dc, ax.k2 * lds_d[c + ox2]);
                v = v + ax.k3 * lds_d[c + ox3];
                v = v + ay.k2 * lds_d[c + oy2];
                v = v + ay.k3 * lds_d[c + oy3];
                v = v + (z < 2 ? klo : -0.25f) * dm2;
                // (the last two planes of a run are past KZ - 7)
                v = v + (z >= KZ - 6 && z >= hi_edge ? -1.0f : -0.25f) * dp2;
                asm volatile("" : "+v"(v));  // (computed here, not where it is used)
                q[z] = v;
                if (GC_IN_RUN(z, n)) acc += (double)dc * (double)v;
                dm2 = dm1;
                dm1 = dc;
                dc = dp1;
                dp1 = dp2;
                c += GC_IN_RUN(z + 1, n) ? ps : 0;
                up = z + 3 < n ? up + ps : (z + 3 == n ? cz : cz + last);
                // (the later steps' reads stay behind: the state fills the registers)
                if (z & 1) __builtin_amdgcn_sched_barrier(0);
            }
            if (!own) acc = 0.0;
        }
        chip_post(acc, sums_dq, g, (uint32_t)it + 1u, sh);
        if (!chip_collect(sums_dq, a.G, (uint32_t)it + 1u, a.abort, limit, sh, &tot)) return;
        const float alpha = delta / (float)tot;
        // phi += alpha d, r -= alpha q, the new r on the faces, r.r
        acc = 0.0;
        const uint32_t tag = (uint32_t)it + 1u;
        {
            const int n = here_uniform(bz), fstep = by * nx, xy = here(column), y = here(ty);
            int c = at(xy, 0);
            const bool send_lo = own && y < 2 && ylo, send_hi = own && y >= by - 2 && yhi;
            // 32-bit offsets from the tile's faces
            uint64_t *const f = face(g, 0);
            const uint32_t fw = a.face_words, hx = (uint32_t)here(x), fz = 2 * fw + (uint32_t)xy;
            uint32_t lo = (uint32_t)(y * n * nx) + hx;
            uint32_t hi = fw + (uint32_t)((by - 1 - y) * n * nx) + hx;
#pragma unroll
            for (int z = 0; z < KZ; ++z) {
                const float d = lds_d[c];
                phi[z] = __builtin_fmaf(alpha, d, phi[z]);
                r[z] = __builtin_fmaf(-alpha, q[z], r[z]);
                asm volatile("" : "+v"(phi[z]), "+v"(r[z]));  // (not vectors of them)
                if (GC_IN_RUN(z, n)) {
                    acc += (double)r[z] * (double)r[z];
                    const uint32_t bits = __float_as_uint(r[z]);
                    if (send_lo) post_word(f + lo, bits, tag);
                    if (send_hi) post_word(f + hi, bits, tag);
                    if (z < 2 && zlo && own) post_word(f + (fz + (uint32_t)(z * fstep)), bits, tag);
                    if (z >= KZ - 6 && z >= n - 2 && zhi && own)
                        post_word(f + (fz + fw + (uint32_t)((n - 1 - z) * fstep)), bits, tag);
                }
                c += GC_IN_RUN(z + 1, n) ? ps : 0;
                lo += nx;
                hi += nx;
                if (z & 1) __builtin_amdgcn_sched_barrier(0);
            }
            if (!own) acc = 0.0;
        }
        chip_post(acc, sums_rr, g, (uint32_t)it + 2u, sh);
        // the neighbours' new r, all words in flight at once and together with
        // the sum's
        bool ok = true;
        {
            const int n = here_uniform(bz);
            uint64_t vy[2][2][kYPass], vz[2][2];
            const uint64_t none = (uint64_t)tag << 32;  // nothing to read: as read
            // (uniform addresses plus 32-bit lane offsets)
            const int hr = here(row);
            const uint32_t xr = (uint32_t)(hr * nx + here(x)), xy = (uint32_t)here(column);
            const uint64_t *py[2] = {face(ylo ? g - 1 : g, 1), face(yhi ? g + 1 : g, 0)};
            const uint64_t *pz[2] = {face(zlo ? g - a.ty : g, 3), face(zhi ? g + a.ty : g, 2)};
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const bool hasy = fetch && (side ? yhi : ylo), hasz = own && (side ? zhi : zlo);
#pragma unroll
                for (int l = 0; l < 2; ++l) {
#pragma unroll
                    for (int p = 0; p < kYPass; ++p)
                        vy[side][l][p] = hasy && hr + p * rows < n
                                             ? read_word(py[side] + (l * n + p * rows) * nx + xr)
                                             : none;
                    vz[side][l] = hasz ? read_word(pz[side] + l * by * nx + xy) : none;
                }
            }
            ChipWait wait(limit);
            auto settle = [&](uint64_t v, const uint64_t *w) {
                while ((uint32_t)(v >> 32) != tag) {
                    if (!wait.again(a.abort)) {
                        ok = false;
                        break;
                    }
                    v = read_word(w);
                }
                uint32_t bits = (uint32_t)v;
                asm volatile("" : "+v"(bits));  // (one register each, not vectors of them)
                return __uint_as_float(bits);
            };
#pragma unroll
            for (int side = 0; side < 2; ++side)
#pragma unroll
                for (int l = 0; l < 2; ++l) {
#pragma unroll
                    for (int p = 0; p < kYPass; ++p)
                        hy[side][l][p] =
                            settle(vy[side][l][p], py[side] + (l * n + p * rows) * nx + xr);
                    hz[side][l] = settle(vz[side][l], pz[side] + l * by * nx + xy);
                }
        }
        if (!ok) sh.abort = 1;  // (read after the next barrier)
        if (!chip_collect(sums_rr, a.G, (uint32_t)it + 2u, a.abort, limit, sh, &tot)) return;
        delta_prev = delta;
        delta = (float)tot;
        beta = delta / delta_prev;
    }
    if (own) {
        float *o = a.phi + (uint64_t)s * a.n + ((uint64_t)z0 * a.ny + (y0 + ty)) * nx + x;
        const uint64_t plane = (uint64_t)a.ny * nx;
#pragma unroll
        for (int z = 0; z < KZ; ++z)
            if (z < bz) o[z * plane] = phi[z];
    }
    if (g == 0 && t == 0) {
        a.st[s].iters = it + 1;
        a.st[s].res = sqrtf(delta);
    }
    if (t == 0)
        __hip_atomic_fetch_add(&a.st[s].tiles, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#undef GC_IN_RUN
}

// zeroes the exchange words (a stale iteration number must not be read) and
// the states and abort flag behind them
__global__ void chip_clear_kernel(uint64_t *p, uint64_t words) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words;
         i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = 0;
}

// The tiles of one right-hand side, or ty = 0 when the grid does not fit.
struct ChipPlan {
    int ty = 0, tz = 0, threads = 0;
    uint32_t face_words = 0;
    size_t lds = 0;
};

// Every tile at least two points along y and z (a halo reaches one tile), its
// columns one per thread, its z run in registers, its d in LDS, all tiles of
// all right-hand sides on `cus` workgroups.  Of these the split with the
// least work per iteration: a z step of the tile, the halo rows a pass of the
// workgroup fetches, and the sums' words (weights from timings).
ChipPlan chip_plan(int nx, int ny, int nz, int m, int cus) {
    ChipPlan best;
    double best_cost = 1e30;
    if (nx * 2 > kChipThreads) return best;
    for (int ty = 1; ty <= ny / 2 && ty * m <= cus; ++ty) {
        const int by = (ny + ty - 1) / ty;
        if (by * nx > kChipThreads) continue;
        const int threads = std::min(kChipThreads, std::max(256, (by * nx + 63) / 64 * 64));
        for (int tz = 1; tz <= nz / 2 && ty * tz * m <= cus; ++tz) {
            const int bz = (nz + tz - 1) / tz;
            if (bz > kChipZ) continue;
            const size_t lds = ((size_t)bz * (by + 4) + 4 * (size_t)by) * nx * sizeof(float);
            if (lds > kChipLds) continue;
            const int rows = threads / nx;
            if (ty > 1 && (bz + rows - 1) / rows > kYPass) continue;
            const int halo = (ty > 1 ? (4 * bz + rows - 1) / rows : 0) +
                             (tz > 1 ? (4 * by + rows - 1) / rows : 0);
            const double cost = 60.0 * bz * threads / 1024 + 40.0 * halo + 4.0 * ty * tz;
            if (cost < best_cost) {
                best_cost = cost;
                best.ty = ty;
                best.tz = tz;
                best.threads = threads;
                best.face_words = (uint32_t)(2 * std::max(by, bz) * nx);
                best.lds = lds;
            }
        }
    }
    return best;
}

int cg_cus(int *cus, int *device = nullptr) {
    int dev = 0;
    GC_HIP(hipGetDevice(&dev));
    GC_HIP(hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (device) *device = dev;
    return GPUCAD_OK;
}

struct ChipLayout {
    uint64_t faces, sums, state, bytes;  // offsets, the first word 0
};
ChipLayout chip_layout(const ChipPlan &p, int m) {
    const uint64_t G = (uint64_t)p.ty * p.tz;
    ChipLayout l;
    l.faces = 0;
    l.sums = l.faces + (uint64_t)m * G * 4 * p.face_words * 8;
    l.state = l.sums + (uint64_t)m * G * 4 * 8;
    l.bytes = l.state + kMaxRhs * sizeof(CgState) + 64;
    return l;
}

// Workspace of a solve: slots of m vectors, phi in slot 0, r in slot 1 (where
// the caller may have put b), q, d0 and d1 of the two-launch form in 2 to 4
// and its partial sums and states behind them; the chip form's exchange words
// begin at slot 2.
struct CgLayout {
    uint64_t slot, bytes;
    int G;
    uint64_t C;
};
CgLayout cg_layout(uint64_t n, int m) {
    CgLayout l;
    // about kCgResident workgroups in all (one wave of them, none waiting),
    // fewer when ranges of one step per thread cover the grid
    const uint64_t steps = (n + kCgStep - 1) / kCgStep;
    l.G = (int)std::min<uint64_t>((steps + 7) & ~uint64_t(7), std::max(8, (kCgResident / m) & ~7));
    l.C = ((n + l.G - 1) / l.G + kCgThreads - 1) / kCgThreads * kCgThreads;
    l.slot = (m * n * sizeof(float) + 255) & ~uint64_t(255);  // 256-byte aligned vectors
    l.bytes = 5 * l.slot + (uint64_t)m * l.G * 8 * 3 + kMaxRhs * sizeof(CgState) + 1024;
    return l;
}

// How a solve is made (gpucad_svl_cg_form) and, after it, how it was.
struct CgForm {
    enum { kAuto = 0, kTwoLaunch = 1, kChip = 2 };
    int form = kAuto;
    int64_t wait_first = kChipWaitTicks, wait_others = kChipWaitTicks;  // ChipArgs
    int solved_by = 0;
};

// The solve on the chip: m right-hand sides b, solutions into x (x may be b) or
// left in slot 0 of ws (x == ws).  *solved says whether every tile ran to its
// end.
int cg_chip_solve(const ChipPlan &p, const float *b, float *x, int m, int nx, int ny, int nz,
                  int max_iter, float end_res, const CgForm &f, CgState *h, void *ws, bool *solved,
                  hipStream_t st) {
    const ChipLayout l = chip_layout(p, m);
    const uint64_t n = (uint64_t)nx * ny * nz;
    char *w = (char *)ws + 2 * cg_layout(n, m).slot;
    ChipArgs a;
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.m = m;
    a.ty = p.ty;
    a.tz = p.tz;
    a.G = p.ty * p.tz;
    a.n = n;
    a.b = b;
    a.phi = (float *)ws;
    a.faces = (uint64_t *)(w + l.faces);
    a.sums = (uint64_t *)(w + l.sums);
    a.face_words = p.face_words;
    a.st = (CgState *)(w + l.state);
    a.abort = (uint32_t *)(w + l.state + kMaxRhs * sizeof(CgState));
    a.max_iter = max_iter;
    a.term = end_res * end_res;
    a.wait_first = f.wait_first;
    a.wait_others = f.wait_others;
    *solved = false;
    typedef void (*ChipKernel)(ChipArgs);
    const int bz = (nz + p.tz - 1) / p.tz;
    static_assert(kChipZ == 24, "one kernel per four planes");
    static const ChipKernel kernels[6] = {cg_chip_kernel<4>,  cg_chip_kernel<8>,
                                          cg_chip_kernel<12>, cg_chip_kernel<16>,
                                          cg_chip_kernel<20>, cg_chip_kernel<24>};
    const ChipKernel kernel = kernels[(bz + 3) / 4 - 1];
    GC_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)kChipLds));
    const uint64_t words = l.bytes / 8;
    hipLaunchKernelGGL(chip_clear_kernel, dim3((unsigned)std::min<uint64_t>((words + 255) / 256, 2048)),
                       dim3(256), 0, st, (uint64_t *)w, words);
    GC_CHECK_LAUNCH();
    hipLaunchKernelGGL(kernel, dim3((unsigned)((a.G * m + 7) / 8 * 8)), dim3(p.threads), p.lds, st, a);
    GC_CHECK_LAUNCH();
    GC_HIP(hipMemcpyAsync(h, a.st, m * sizeof(CgState), hipMemcpyDeviceToHost, st));
    GC_HIP(hipStreamSynchronize(st));
    for (int s = 0; s < m; ++s)
        if (h[s].tiles != (uint32_t)a.G) return GPUCAD_OK;
    if (x != a.phi)
        GC_HIP(hipMemcpyAsync(x, a.phi, m * n * sizeof(float), hipMemcpyDeviceToDevice, st));
    *solved = true;
    return GPUCAD_OK;
}

// b's place in the workspace ws of a solve, for a caller without its own
float *cg_rhs(void *ws, uint64_t n, int m) { return (float *)((char *)ws + cg_layout(n, m).slot); }

// Workspace of cg_solve.
size_t cg_bytes(int m, int nx, int ny, int nz) {
    const uint64_t n = (uint64_t)nx * ny * nz;
    int cus = 0;
    if (cg_cus(&cus)) cus = 0;
    const CgLayout l = cg_layout(n, m);
    size_t bytes = l.bytes;
    const ChipPlan p = chip_plan(nx, ny, nz, m, cus);
    if (p.ty) bytes = std::max<size_t>(bytes, 2 * l.slot + chip_layout(p, m).bytes);
    return bytes;
}

// Solves A x = b for m right-hand sides (b: m vectors of n, also at cg_rhs; x
// written over b when x == b, or left in ws when x == ws) in ws (cg_bytes).  On the chip when the grid fits there and no
// solve gave up lately; otherwise, or when this one gives up waiting, iterations
// of two launches in chunks between host checks of the done flags (a finished
// right-hand side leaves the kernels at their first test).  x is complete in
// stream order.
int cg_solve(const float *b, float *x, int m, int nx, int ny, int nz, int max_iter, float end_res,
             CgForm *f, int *iters, float *res, void *ws, hipStream_t st) {
    const uint64_t n = (uint64_t)nx * ny * nz;
    CgState h[kMaxRhs];
    int cus = 0, dev = 0;
    int rc = cg_cus(&cus, &dev);
    if (rc) return rc;
    const ChipPlan chip = chip_plan(nx, ny, nz, m, cus);
    GC_ARG(f->form != CgForm::kChip || chip.ty, "the grid does not fit on the chip");
    int &pause = g_chip_pause[dev];  // (the arena is for devices 0..63)
    bool solved = false;
    if (chip.ty && (f->form == CgForm::kChip || (f->form == CgForm::kAuto && pause == 0))) {
        rc = cg_chip_solve(chip, b, x, m, nx, ny, nz, max_iter, end_res, *f, h, ws, &solved, st);
        if (rc) return rc;
        pause = solved ? 0 : kChipPause;
    } else if (chip.ty && f->form == CgForm::kAuto) {
        --pause;
    }
    f->solved_by = solved ? CgForm::kChip : CgForm::kTwoLaunch;
    if (!solved) {
        const CgLayout l = cg_layout(n, m);
        CgArgs a;
        a.nx = nx;
        a.ny = ny;
        a.nz = nz;
        a.n = n;
        a.dnx = make_div32((uint32_t)nx);
        a.dplane = make_div32((uint32_t)nx * (uint32_t)ny);
        a.G = l.G;
        a.C = l.C;
        a.max_iter = max_iter;
        a.term = end_res * end_res;
        char *w = (char *)ws;
        a.phi = (float *)w;
        a.r = (float *)(w + l.slot);
        a.q = (float *)(w + 2 * l.slot);
        a.d0 = (float *)(w + 3 * l.slot);
        a.d1 = (float *)(w + 4 * l.slot);
        a.pq = (double *)(w + 5 * l.slot);
        a.prr = a.pq + (uint64_t)m * a.G;
        a.st = (CgState *)(a.prr + 2 * (uint64_t)m * a.G);
        const dim3 grid((unsigned)a.G, (unsigned)m);
        hipLaunchKernelGGL(cg_init_kernel, grid, dim3(kCgThreads), 0, st, b, a);
        GC_CHECK_LAUNCH();
        constexpr int kChunk = 16;
        for (int it0 = 0; it0 < max_iter; it0 += kChunk) {
            for (int it = it0; it < std::min(max_iter, it0 + kChunk); ++it) {
                hipLaunchKernelGGL(cg_a_kernel, grid, dim3(kCgThreads), 0, st, a, it);
                hipLaunchKernelGGL(cg_b_kernel, grid, dim3(kCgThreads), 0, st, a, it);
            }
            GC_CHECK_LAUNCH();
            GC_HIP(hipMemcpyAsync(h, a.st, m * sizeof(CgState), hipMemcpyDeviceToHost, st));
            GC_HIP(hipStreamSynchronize(st));
            bool all = true;
            for (int s = 0; s < m; ++s) all = all && h[s].done;
            if (all) break;
        }
        for (int s = 0; s < m; ++s)
            if (!h[s].done)
                return fail(GPUCAD_E_HIP, "internal: CG did not stop by iteration %d", max_iter);
        if (x != a.phi)
            GC_HIP(hipMemcpyAsync(x, a.phi, m * n * sizeof(float), hipMemcpyDeviceToDevice, st));
    }
    for (int s = 0; s < m; ++s) {
        if (iters) iters[s] = h[s].iters;
        if (res) res[s] = h[s].res;
    }
    return GPUCAD_OK;
}

// ---------------------------------------------------------------------------
// 2x upsampling of a coarse field as the reference's texture fetch does it
// (tex3D, unnormalised coordinates, texel centres at +0.5, linear filter,
// clamp at the far end: Gratings.cu:653-722, Interpolations.cu:57-107).
// Fine point f samples texel coordinate u = f * h; weights are the fraction
// of u quantised to 1/256 (the filter's 8 fraction bits); lerps run along
// x, then y, then z.
// ---------------------------------------------------------------------------
struct Tap {
    int64_t i0, i1;
    float w;
};

__device__ __forceinline__ Tap tap(int f, float h, int n) {
    const float u = (float)f * h;
    const float fl = floorf(u);
    float w = u - fl;
    w = rintf(w * 256.0f) * (1.0f / 256.0f);
    int64_t i0 = (int64_t)fl;
    if (w >= 1.0f) {
        i0 += 1;
        w = 0.0f;
    }
    Tap t;
    t.i0 = i0 < 0 ? 0 : (i0 > n - 1 ? n - 1 : i0);
    t.i1 = i0 + 1 > n - 1 ? n - 1 : (i0 + 1 < 0 ? 0 : i0 + 1);
    t.w = w;
    return t;
}

__device__ __forceinline__ float lerp1(float a, float b, float w) {
    return __builtin_fmaf(w, b, (1.0f - w) * a);
}

__device__ __forceinline__ float sample3(const float *c, const Tap &tx, const Tap &ty, const Tap &tz,
                                         int64_t row, int64_t plane) {
    const int64_t z0 = tz.i0 * plane, z1 = tz.i1 * plane, y0 = ty.i0 * row, y1 = ty.i1 * row;
    const float c00 = lerp1(c[z0 + y0 + tx.i0], c[z0 + y0 + tx.i1], tx.w);
    const float c10 = lerp1(c[z0 + y1 + tx.i0], c[z0 + y1 + tx.i1], tx.w);
    const float c01 = lerp1(c[z1 + y0 + tx.i0], c[z1 + y0 + tx.i1], tx.w);
    const float c11 = lerp1(c[z1 + y1 + tx.i0], c[z1 + y1 + tx.i1], tx.w);
    return lerp1(lerp1(c00, c10, ty.w), lerp1(c01, c11, ty.w), tz.w);
}

struct Up {
    int nx, ny, nz;     // coarse
    int fx, fy, fz;     // fine
    float hx, hy, hz;   // fine spacing in coarse texels
};

// mode 0: refine (the sample); 1: grating (cos, sin of the sample)
__global__ void upsample_kernel(const float *c, Up u, float *out, float2 *grating, int mode) {
    const uint64_t n = (uint64_t)u.fx * u.fy * u.fz;
    const int64_t row = u.nx, plane = (int64_t)u.nx * u.ny;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x) {
        int x, y, z;
        point_xyz(t, u.fx, u.fy, &x, &y, &z);
        const float v = sample3(c, tap(x, u.hx, u.nx), tap(y, u.hy, u.ny), tap(z, u.hz, u.nz), row,
                                plane);
        if (mode == 0) out[t] = v;
        else grating[t] = make_float2(cos_rad(v), sin_rad(v));
    }
}

// svl += Re(grating * c[index])  (svl_kernel, Gratings.cu:724-752)
__global__ void svl_acc_kernel(float *svl, const float2 *g, uint64_t n, const float2 *coeffs,
                               int index) {
    const float2 c = coeffs[index];
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x) {
        const float2 a = g[t];
        svl[t] = svl[t] + __builtin_fmaf(a.x, c.x, -(a.y * c.y));
    }
}

// ---------------------------------------------------------------------------
// native fused synthesis: svl[f] = sum over the first H harmonics (i, j, k)
// of Re(c_h e^{i (i Phi_x + j Phi_y + k Phi_z)(f)}), Phi upsampled as above;
// e^{i phi_h} = Ex^i Ey^j Ez^k from the three exponentials and their powers.
//
// Bound by FP32 VALU.  The sum is nested, k over j over i, and i and -i share
// their powers: c E^i + c' E^-i = (c + c') cos + i (c - c') sin, so a (j, k) pair costs
// 4 R + 4 multiply-adds instead of two complex products and a real part per
// harmonic.  A wave takes a row of the fine grid, four consecutive points per
// lane: the coefficients (LDS broadcasts) and the row's taps serve all four, and
// the rows' addresses are uniform.  240^3 from 120^3, 62 harmonics:
// 1081 -> 150 us.
// PACK: rows of up to 128 points, several of them in a wave, each on a power of
// two of its lanes; longer rows are split over gridDim.y.  Calls on 262144 rows
// of 8 points: 530 us with a row per wave, 81 so (250 with a thread per point);
// on 16 rows of 100000: 1640 us with a wave per row, 79 so.
// ---------------------------------------------------------------------------
constexpr int kMaxRange = 4;  // (2r+1)^3 <= 729 coefficients
constexpr int kSvlPoints = 4;  // fine points per lane

struct Cf {
    float re, im;
};
__device__ __forceinline__ Cf cmulf(Cf a, Cf b) {
    return Cf{__builtin_fmaf(a.re, b.re, -(a.im * b.im)), __builtin_fmaf(a.re, b.im, a.im * b.re)};
}

// LDS floats of one (j, k) pair: c_0, then c_i + c_-i and i (c_i - c_-i) for i = 1..R
constexpr int svl_pair_floats(int r) { return 2 + 4 * r; }

template <int R, bool PACK>
__global__ void __launch_bounds__(256) svl_field_kernel(const float *phix, const float *phiy,
                                                        const float *phiz, Up u,
                                                        const float2 *coeffs, int harmonics,
                                                        uint32_t row_lanes_log2, float *svl) {
    constexpr int kSide = 2 * R + 1, kPair = svl_pair_floats(R), P = kSvlPoints;
    __shared__ float s_c[kSide * kSide * kPair];
    auto coeff = [&](int i, int jk) {  // 0 past the harmonics
        const int h = (i + R) + kSide * jk;
        return h < harmonics ? coeffs[h] : make_float2(0.f, 0.f);
    };
    for (int t = threadIdx.x; t < kSide * kSide * (R + 1); t += 256) {
        const int jk = t / (R + 1), i = t - jk * (R + 1);
        float *c = s_c + jk * kPair;
        const float2 a = coeff(i, jk), b = coeff(-i, jk);
        if (i == 0) {
            c[0] = a.x;
            c[1] = a.y;
        } else {
            c[4 * i - 2] = a.x + b.x;
            c[4 * i - 1] = a.y + b.y;
            c[4 * i] = b.y - a.y;
            c[4 * i + 1] = a.x - b.x;
        }
    }
    __syncthreads();
    const int klim = (harmonics + kSide * kSide - 1) / (kSide * kSide);  // layers with coefficients
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t nrows = (uint32_t)u.fy * (uint32_t)u.fz;
    const int64_t crow = u.nx, cplane = (int64_t)u.nx * u.ny;
    const bool wide = (u.fx & 3) == 0 && ((uintptr_t)svl & 15u) == 0;
    // a wave's rows, the lane's one of them and its place in it
    const uint32_t wave_rows = PACK ? 64u >> row_lanes_log2 : 1u;
    const uint32_t lane_row = PACK ? lane >> row_lanes_log2 : 0u;
    const uint32_t row_lane = PACK ? lane & ((1u << row_lanes_log2) - 1u) : lane;
    for (int64_t x0 = (int64_t)blockIdx.y * 64 * P; x0 < u.fx; x0 += (int64_t)gridDim.y * 64 * P) {
        const int64_t x = x0 + (int64_t)row_lane * P;
        const int points = (int)min(max((int64_t)u.fx - x, (int64_t)0), (int64_t)P);
        uint32_t i0[P], i1[P];
        float w1[P], w0[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const Tap t = tap((int)min(x + p, (int64_t)u.fx - 1), u.hx, u.nx);
            i0[p] = (uint32_t)t.i0;
            i1[p] = (uint32_t)t.i1;
            w1[p] = t.w;
            w0[p] = 1.0f - t.w;
        }
        for (uint64_t first = (uint64_t)(blockIdx.x * 4 + wave) * wave_rows; first < nrows;
             first += (uint64_t)gridDim.x * 4 * wave_rows) {
            const bool in = !PACK || first + lane_row < nrows;
            const uint32_t row = (uint32_t)(in ? first + lane_row : first);
            const uint32_t fz = row / (uint32_t)u.fy, fy = row - fz * (uint32_t)u.fy;
            const Tap ty = tap((int)fy, u.hy, u.ny), tz = tap((int)fz, u.hz, u.nz);
            // Phi at the lane's points: lerps along x, then y, then z (sample3); a
            // row or plane of weight 0 is not read
            auto sample = [&](const float *phi, float (&v)[P]) {
                auto line = [&](int64_t iz, int64_t iy, float (&o)[P]) {
                    const float *c = phi + iz * cplane + iy * crow;
#pragma unroll
                    for (int p = 0; p < P; ++p)
                        o[p] = __builtin_fmaf(w1[p], c[i1[p]], w0[p] * c[i0[p]]);
                };
                auto plane = [&](int64_t iz, float (&o)[P]) {
                    line(iz, ty.i0, o);
                    if (ty.w != 0.0f) {
                        float q[P];
                        line(iz, ty.i1, q);
#pragma unroll
                        for (int p = 0; p < P; ++p) o[p] = lerp1(o[p], q[p], ty.w);
                    }
                };
                plane(tz.i0, v);
                if (tz.w != 0.0f) {
                    float q[P];
                    plane(tz.i1, q);
#pragma unroll
                    for (int p = 0; p < P; ++p) v[p] = lerp1(v[p], q[p], tz.w);
                }
            };
            // powers E^1..E^R per axis; negative powers are conjugates
            Cf ex[P][R + 1], ey[P][R + 1], ez[P][R + 1];
            auto powers = [&](const float *phi, Cf (&e)[P][R + 1]) {
                float v[P];
                sample(phi, v);
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    e[p][0] = Cf{1.0f, 0.0f};
                    if constexpr (R > 0) {
                        e[p][1] = Cf{cos_rad(v[p]), sin_rad(v[p])};
#pragma unroll
                        for (int q = 2; q <= R; ++q) e[p][q] = cmulf(e[p][q - 1], e[p][1]);
                    }
                }
            };
            powers(phix, ex);
            powers(phiy, ey);
            powers(phiz, ez);
            float acc[P] = {};
            for (int k = 0; k < klim; ++k) {
                Cf T[P] = {};
#pragma unroll
                for (int j = -R; j <= R; ++j) {
                    const float *c = s_c + (k * kSide + j + R) * kPair;
#pragma unroll
                    for (int p = 0; p < P; ++p) {
                        float re = c[0], im = c[1];
#pragma unroll
                        for (int i = 1; i <= R; ++i) {
                            re = __builtin_fmaf(c[4 * i - 2], ex[p][i].re, re);
                            im = __builtin_fmaf(c[4 * i - 1], ex[p][i].re, im);
                            re = __builtin_fmaf(c[4 * i], ex[p][i].im, re);
                            im = __builtin_fmaf(c[4 * i + 1], ex[p][i].im, im);
                        }
                        const int m = j < 0 ? -j : j;
                        const float er = ey[p][m].re, ei = j < 0 ? -ey[p][m].im : ey[p][m].im;
                        T[p].re = __builtin_fmaf(re, er, __builtin_fmaf(-im, ei, T[p].re));
                        T[p].im = __builtin_fmaf(re, ei, __builtin_fmaf(im, er, T[p].im));
                    }
                }
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    Cf e = ez[p][0];
#pragma unroll
                    for (int q = 1; q <= R; ++q) {
                        if (k - R == q) e = ez[p][q];
                        if (k - R == -q) e = Cf{ez[p][q].re, -ez[p][q].im};
                    }
                    acc[p] = __builtin_fmaf(T[p].re, e.re, __builtin_fmaf(-T[p].im, e.im, acc[p]));
                }
            }
            float *o = svl + (uint64_t)row * u.fx + x;
            if (wide && points && in) {
                *(float4 *)o = make_float4(acc[0], acc[1], acc[2], acc[3]);
            } else {
#pragma unroll
                for (int p = 0; p < P; ++p)
                    if (p < points && in) o[p] = acc[p];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// unit-cell Fourier coefficients by direct DFT: coefficient (i, j, k) =
// (1/N) sum f(x,y,z) e^{-2 pi i (i x/nx + j y/ny + k z/nz)}, the forward R2C
// transform scaled as fft_scalar does (Fft_lattice.cu) and picked as
// unit_lattice does (src/main.cu:3578-3711: loop k, j, i over [-r, r])
//
// Separable: the x sums of every row for i = 0..r (the cell is real, so -i is
// the conjugate), then one workgroup per (i >= 0, j, k) over the rows.  Sums
// and twiddles in FP64.  Bound by latency, the cell is small: 61^3,
// r = 2 took 290 us with a workgroup per coefficient over the whole cell, the
// two passes take 5.1 + 6.1 us.
// ---------------------------------------------------------------------------
// (cos, -sin)(2 pi num / n), num < n
__device__ __forceinline__ double2 twiddle(uint32_t num, uint32_t n) {
    double s, c;
    sincospi(2.0 * (double)num / (double)n, &s, &c);
    return make_double2(c, -s);
}
__device__ __forceinline__ double2 cmuld(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
constexpr int kDftRows = 4;  // rows per wave: a wave's twiddles serve all of them
// Rows whose sums are held at a time (16 bytes per row and i: at most 21 MB; a
// cell of 512^3 has this many).
constexpr uint32_t kDftPiece = 1u << 18;

// rows[i * nrows + row] = sum over x of f(x, row) e^{-2 pi i ix/nx}, i = 0..R
template <int R>
__global__ void __launch_bounds__(256) dft_rows_kernel(const float *cell, int nx, uint32_t nrows,
                                                       double2 *rows) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * kDftRows;
    if (row0 >= nrows) return;
    double2 acc[kDftRows][R + 1];
#pragma unroll
    for (int q = 0; q < kDftRows; ++q)
#pragma unroll
        for (int i = 0; i <= R; ++i) acc[q][i] = make_double2(0.0, 0.0);
    for (uint32_t x = lane; x < (uint32_t)nx; x += 64) {
        double2 e[R + 2];  // powers of e^{-2 pi i x/nx}
        e[0] = make_double2(1.0, 0.0);
        if constexpr (R > 0) e[1] = twiddle(x, (uint32_t)nx);
#pragma unroll
        for (int i = 2; i <= R; ++i) e[i] = cmuld(e[i - 1], e[1]);
#pragma unroll
        for (int q = 0; q < kDftRows; ++q) {
            const uint32_t row = row0 + q < nrows ? row0 + q : row0;
            const double f = cell[(uint64_t)row * nx + x];
#pragma unroll
            for (int i = 0; i <= R; ++i) {
                acc[q][i].x = fma(f, e[i].x, acc[q][i].x);
                acc[q][i].y = fma(f, e[i].y, acc[q][i].y);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < kDftRows; ++q)
#pragma unroll
        for (int i = 0; i <= R; ++i) {
            const double2 v = make_double2(wave_sum_d(acc[q][i].x), wave_sum_d(acc[q][i].y));
            if (lane == 0 && row0 + q < nrows) rows[(uint64_t)i * nrows + row0 + q] = v;
        }
}

// workgroup (i, j, k): the sums of rows first .. first + nrows over y and z,
// added to the earlier pieces' in sum; after the last piece it writes (i, j, k)
// and its mirror image (-i, -j, -k)
__global__ void __launch_bounds__(256) dft_planes_kernel(const double2 *rows, uint32_t first,
                                                         uint32_t nrows, bool last, int ny, int nz,
                                                         int range, double cells, double2 *sum,
                                                         float2 *out) {
    const int side = 2 * range + 1;
    const int j = (int)(blockIdx.x % side) - range, k = (int)(blockIdx.x / side) - range;
    const int i = (int)blockIdx.y;
    double re = 0.0, im = 0.0;
    for (uint32_t t = threadIdx.x; t < nrows; t += 256) {
        const uint32_t z = (first + t) / (uint32_t)ny, y = first + t - z * (uint32_t)ny;
        // the angle in periods (at most 2 range of them, so rounded to about 1e-15)
        const double a = (double)((int64_t)j * y) / (double)ny + (double)((int64_t)k * z) / (double)nz;
        double s, c;
        sincospi(2.0 * a, &s, &c);
        const double2 v = cmuld(rows[(uint64_t)i * nrows + t], make_double2(c, -s));
        re += v.x;
        im += v.y;
    }
    __shared__ double sr[4], si[4];
    re = wave_sum_d(re);
    im = wave_sum_d(im);
    if ((threadIdx.x & 63) == 0) {
        sr[threadIdx.x >> 6] = re;
        si[threadIdx.x >> 6] = im;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double2 v = make_double2((sr[0] + sr[1]) + (sr[2] + sr[3]),
                                 (si[0] + si[1]) + (si[2] + si[3]));
        double2 *before = sum + blockIdx.x + gridDim.x * blockIdx.y;
        if (first > 0) {
            v.x += before->x;
            v.y += before->y;
        }
        if (!last) {
            *before = v;
            return;
        }
        const float vr = (float)(v.x / cells);
        const float vi = (float)(v.y / cells);
        auto at = [=](int a, int b, int c) {
            return (a + range) + side * ((b + range) + side * (c + range));
        };
        out[at(i, j, k)] = make_float2(vr, vi);
        if (i > 0) out[at(-i, -j, -k)] = make_float2(vr, -vi);
    }
}

// fft_fill_kernel (Fft_lattice.cu): the half spectrum (nx/2+1 columns) into
// the full one with its conjugate mirror; the mirror indices use nx on every
// axis, as the reference's do
__global__ void fft_fill_kernel(const float2 *half, float2 *full, int nx, int ny, int nz) {
    const int nx2 = nx / 2 + 1;
    const uint64_t n = (uint64_t)nx2 * ny * nz;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x) {
        int x, y, z;
        point_xyz(t, nx2, ny, &x, &y, &z);
        if (t == 0) {
            full[0] = half[0];
            continue;
        }
        const int e = x == 0 ? 0 : nx - x, f = y == 0 ? 0 : nx - y, g = z == 0 ? 0 : nx - z;
        const float2 s = half[t];
        full[(uint64_t)x + (uint64_t)y * nx + (uint64_t)z * nx * ny] = s;
        full[(uint64_t)e + (uint64_t)f * nx + (uint64_t)g * nx * ny] = make_float2(s.x, -s.y);
    }
}

__global__ void fft_scale_kernel(float2 *d, float s, uint64_t n) {
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x) {
        float2 a = d[t];
        a.x /= s;
        a.y /= s;
        d[t] = a;
    }
}

// VecSMultAddKernel_lattice (Gratings.cu:73-94): v = a1 v + a2 w (fused)
__global__ void axpby_kernel(float *v, float a1, const float *w, float a2, uint64_t n) {
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x)
        v[t] = __builtin_fmaf(a2, w[t], a1 * v[t]);
}

// fillfrac_kernel (Gratings.cu:755-772): svl *= fillfrac
__global__ void fillfrac_kernel(float *svl, const float *frac, uint64_t n) {
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * blockDim.x)
        svl[t] = frac[t] * svl[t];
}

// GPUScalar_lattice (Gratings.cu:600-650, 22-70): a.b into result[0]
// (partial sums in double per block, one fixed-order final sum)
__global__ void dot_partial_kernel(const float *a, const float *b, uint64_t n, double *part) {
    double acc = 0.0;
    for (uint64_t t = (uint64_t)blockIdx.x * kCgThreads + threadIdx.x; t < n;
         t += (uint64_t)gridDim.x * kCgThreads)
        acc += (double)a[t] * (double)b[t];
    const double tot = block_sum(acc);
    if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

__global__ void dot_final_kernel(const double *part, int G, float *result) {
    const double tot = sum_partials(part, G);
    if (threadIdx.x == 0) result[0] = (float)tot;
}

dim3 stride_grid(uint64_t n) {
    return dim3((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((n + 255) / 256, 8192)));
}

int check_dims(int nx, int ny, int nz, int minimum) {
    GC_ARG(nx >= minimum && ny >= minimum && nz >= minimum, "grid sizes must be >= %d (got %d %d %d)",
           minimum, nx, ny, nz);
    GC_ARG((uint64_t)nx * ny * nz < (1ull << 32), "grid too large (2^32 points or more)");
    return GPUCAD_OK;
}

PhiArgs phi_args(const gc_svl_params *p, int i, int j, int k) {
    PhiArgs a;
    a.nx = p->nx;
    a.ny = p->ny;
    a.nz = p->nz;
    a.i = i;
    a.j = j;
    a.k = k;
    a.dx = p->dx;
    a.dy = p->dy;
    a.dz = p->dz;
    a.type = p->lattice_type;
    a.uniform_type = p->uniform_type;
    a.const_period = p->const_period;
    a.x_period = p->x_period;
    a.y_period = p->y_period;
    a.z_period = p->z_period;
    a.lcon = p->lcon;
    a.lcon_1 = p->lcon_1;
    a.sinewave_zaxis = p->sinewave_zaxis;
    return a;
}

int check_params(const gc_svl_params *p, const float *period) {
    GC_ARG(p, "params is NULL");
    int st = check_dims(p->nx, p->ny, p->nz, 4);
    if (st) return st;
    GC_ARG(p->lattice_type == 'n' || p->lattice_type == 'b' || p->lattice_type == 'r' ||
               p->lattice_type == 's',
           "lattice_type must be 'n', 'b', 'r' or 's'");
    GC_ARG(p->uniform_type >= 0 && p->uniform_type <= 2, "uniform_type must be 0, 1 or 2");
    GC_ARG(p->uniform_type != 2 || period, "uniform_type 2 needs a period field");
    return GPUCAD_OK;
}

}  // namespace
}  // namespace gc

using namespace gc;

extern "C" {

int gpucad_svl_period_data(float *d_period, int32_t nx, int32_t ny, int32_t nz, float dx, float dy,
                           float dz, float mean_x, float mean_y, float mean_z, char axis) {
    clear_error();
    GC_ARG(d_period, "NULL buffer");
    int st = check_dims(nx, ny, nz, 1);
    if (st) return st;
    const uint64_t n = (uint64_t)nx * ny * nz;
    hipLaunchKernelGGL(period_angle_kernel, stride_grid(n), dim3(256), 0, 0, d_period, nx, ny, nz,
                       dx, dy, dz, mean_x, mean_y, mean_z, (int)axis, 0);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_svl_angle_data(float *d_theta, int32_t nx, int32_t ny, int32_t nz, float dx, float dy,
                          float dz, float mean_x, float mean_y, float mean_z, char axis) {
    clear_error();
    GC_ARG(d_theta, "NULL buffer");
    int st = check_dims(nx, ny, nz, 1);
    if (st) return st;
    const uint64_t n = (uint64_t)nx * ny * nz;
    hipLaunchKernelGGL(period_angle_kernel, stride_grid(n), dim3(256), 0, 0, d_theta, nx, ny, nz,
                       dx, dy, dz, mean_x, mean_y, mean_z, (int)axis, 1);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

static int rescale(const float *in, float *out, uint64_t size, float a1, float b1, int affine) {
    clear_error();
    auto calls = lock_device_calls();  // shared scratch arena
    GC_ARG(in && out, "NULL buffer");
    GC_ARG(size > 0, "size must be positive");
    void *ws = nullptr;
    int st = scratch_arena(1024 * sizeof(float2), &ws);
    if (st) return st;
    float2 *part = (float2 *)ws;
    st = enqueue_minmax0(in, size, part, 0);
    if (st) return st;
    hipLaunchKernelGGL(rescale_kernel, stride_grid(size), dim3(256), 0, 0, in, out, size, part, a1,
                       b1, affine);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_normalise_three(const float *in, float *out, uint64_t size, float a1, float b1) {
    return rescale(in, out, size, a1, b1, 1);
}

int gpucad_normalise_buffer(const float *in, float *out, uint64_t size) {
    return rescale(in, out, size, 0.0f, 0.0f, 0);
}

int gpucad_svl_finding_phi(float *d_phi, const float *d_period, int32_t nx, int32_t ny, int32_t nz,
                           int32_t i, int32_t j, int32_t k, float dx, float dy, float dz,
                           char lattice_type, int32_t uniform_type, float const_period,
                           float x_period, float y_period, float z_period, float lcon,
                           float lcon_1, int32_t sinewave_zaxis) {
    clear_error();
    GC_ARG(d_phi, "NULL buffer");
    gc_svl_params p = {};
    p.nx = nx;
    p.ny = ny;
    p.nz = nz;
    p.dx = dx;
    p.dy = dy;
    p.dz = dz;
    p.lattice_type = lattice_type;
    p.uniform_type = uniform_type;
    p.const_period = const_period;
    p.x_period = x_period;
    p.y_period = y_period;
    p.z_period = z_period;
    p.lcon = lcon;
    p.lcon_1 = lcon_1;
    p.sinewave_zaxis = sinewave_zaxis;
    int st = check_params(&p, d_period);
    if (st) return st;
    const uint64_t n = (uint64_t)nx * ny * nz;
    hipLaunchKernelGGL(finding_phi_kernel, stride_grid(n), dim3(256), 0, 0, d_phi, d_period,
                       phi_args(&p, i, j, k));
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_svl_matvec(const float *d_d, float *d_q, int32_t nx, int32_t ny, int32_t nz) {
    clear_error();
    GC_ARG(d_d && d_q && d_d != d_q, "NULL or aliased buffer");
    int st = check_dims(nx, ny, nz, 4);
    if (st) return st;
    const uint64_t n = (uint64_t)nx * ny * nz;
    hipLaunchKernelGGL(matvec_kernel, stride_grid(n), dim3(256), 0, 0, d_d, d_q, nx, ny, nz);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

static int svl_cg(float *d_phi, int m, int nx, int ny, int nz, int iter, float end_res, CgForm *f,
                  int *final_iter, float *final_res) {
    clear_error();
    auto calls = lock_device_calls();  // shared scratch arena
    GC_ARG(d_phi, "NULL buffer");
    int st = check_dims(nx, ny, nz, 4);
    if (st) return st;
    GC_ARG(iter >= 1, "iter must be >= 1");
    void *ws = nullptr;
    if ((st = scratch_arena(cg_bytes(m, nx, ny, nz), &ws))) return st;
    st = cg_solve(d_phi, d_phi, m, nx, ny, nz, iter, end_res, f, final_iter, final_res, ws, 0);
    if (st) return st;
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_svl_cg(float *d_phi, int32_t nx, int32_t ny, int32_t nz, int32_t iter, float end_res,
                  int32_t *final_iter, float *final_res) {
    CgForm f;
    return svl_cg(d_phi, 1, nx, ny, nz, iter, end_res, &f, final_iter, final_res);
}

int gpucad_svl_cg_form(float *d_phi, int32_t m, int32_t nx, int32_t ny, int32_t nz, int32_t iter,
                       float end_res, int32_t form, float wait_first_ms, float wait_ms,
                       int32_t *final_iter, float *final_res, int32_t *how) {
    clear_error();
    GC_ARG(m >= 1 && m <= kMaxRhs, "m must be in [1, %d]", kMaxRhs);
    GC_ARG(form >= CgForm::kAuto && form <= CgForm::kChip, "unknown form %d", form);
    // (a longer wait than the default would hold the device's other work)
    const float most = (float)kChipWaitTicks / 1e5f;
    GC_ARG(wait_first_ms <= most && wait_ms <= most, "a wait is at most %g ms", (double)most);
    CgForm f;
    f.form = form;
    const auto ticks = [](float ms) { return ms < 0.f ? (int64_t)-1 : (int64_t)(ms * 1e5f); };
    if (wait_first_ms != 0.f) f.wait_first = ticks(wait_first_ms);
    if (wait_ms != 0.f) f.wait_others = ticks(wait_ms);
    int st = svl_cg(d_phi, m, nx, ny, nz, iter, end_res, &f, final_iter, final_res);
    if (st || !how) return st;
    int cus = 0;
    if ((st = cg_cus(&cus))) return st;
    const ChipPlan p = chip_plan(nx, ny, nz, m, cus);
    how[0] = f.solved_by;
    how[1] = p.ty;
    how[2] = p.tz;
    how[3] = p.ty ? ((nz + p.tz - 1) / p.tz + 3) / 4 * 4 : 0;
    how[4] = p.ty > 1 ? ((nz + p.tz - 1) / p.tz + p.threads / nx - 1) / (p.threads / nx) : 0;
    return GPUCAD_OK;
}

int gpucad_svl_axpby(float *d_v, float a1, const float *d_w, float a2, uint64_t n) {
    clear_error();
    GC_ARG(d_v && d_w, "NULL buffer");
    hipLaunchKernelGGL(axpby_kernel, stride_grid(n), dim3(256), 0, 0, d_v, a1, d_w, a2, n);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_svl_dot(float *d_result, const float *d_a, const float *d_b, uint64_t n) {
    clear_error();
    auto calls = lock_device_calls();  // shared scratch arena
    GC_ARG(d_result && d_a && d_b, "NULL buffer");
    const int G = (int)std::max<uint64_t>(1, std::min<uint64_t>((n + kCgThreads - 1) / kCgThreads,
                                                                kCgBlocks));
    void *ws = nullptr;
    int st = scratch_arena(G * sizeof(double), &ws);
    if (st) return st;
    hipLaunchKernelGGL(dot_partial_kernel, dim3(G), dim3(kCgThreads), 0, 0, d_a, d_b, n,
                       (double *)ws);
    hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(kCgThreads), 0, 0, (const double *)ws, G,
                       d_result);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_svl_fillfrac(float *d_svl, const float *d_fillfrac, int32_t nx, int32_t ny,
                        int32_t nz) {
    clear_error();
    GC_ARG(d_svl && d_fillfrac, "NULL buffer");
    int st = check_dims(nx, ny, nz, 1);
    if (st) return st;
    const uint64_t n = (uint64_t)nx * ny * nz;
    hipLaunchKernelGGL(fillfrac_kernel, stride_grid(n), dim3(256), 0, 0, d_svl, d_fillfrac, n);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_svl_refine(const float *d_coarse, int32_t nx, int32_t ny, int32_t nz, float *d_fine,
                      int32_t fx, int32_t fy, int32_t fz, float hx, float hy, float hz) {
    clear_error();
    GC_ARG(d_coarse && d_fine, "NULL buffer");
    int st = check_dims(nx, ny, nz, 1);
    if (!st) st = check_dims(fx, fy, fz, 1);
    if (st) return st;
    GC_ARG(hx >= 0.f && hy >= 0.f && hz >= 0.f, "spacings must be non-negative");
    const Up u = {nx, ny, nz, fx, fy, fz, hx, hy, hz};
    const uint64_t n = (uint64_t)fx * fy * fz;
    hipLaunchKernelGGL(upsample_kernel, stride_grid(n), dim3(256), 0, 0, d_coarse, u, d_fine,
                       (float2 *)nullptr, 0);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_svl_grating(const float *d_phi, int32_t nx, int32_t ny, int32_t nz, gc_float2 *d_grating,
                       int32_t fx, int32_t fy, int32_t fz, float hx, float hy, float hz) {
    clear_error();
    GC_ARG(d_phi && d_grating, "NULL buffer");
    int st = check_dims(nx, ny, nz, 1);
    if (!st) st = check_dims(fx, fy, fz, 1);
    if (st) return st;
    GC_ARG(hx >= 0.f && hy >= 0.f && hz >= 0.f, "spacings must be non-negative");
    const Up u = {nx, ny, nz, fx, fy, fz, hx, hy, hz};
    const uint64_t n = (uint64_t)fx * fy * fz;
    hipLaunchKernelGGL(upsample_kernel, stride_grid(n), dim3(256), 0, 0, d_phi, u, (float *)nullptr,
                       (float2 *)d_grating, 1);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_svl_accumulate(float *d_svl, const gc_float2 *d_grating, uint64_t n, int32_t index,
                          const gc_float2 *d_coeffs) {
    clear_error();
    GC_ARG(d_svl && d_grating && d_coeffs, "NULL buffer");
    GC_ARG(n > 0 && index >= 0, "n must be positive and index non-negative");
    hipLaunchKernelGGL(svl_acc_kernel, stride_grid(n), dim3(256), 0, 0, d_svl,
                       (const float2 *)d_grating, n, (const float2 *)d_coeffs, index);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_svl_field(const gc_svl_params *p, const float *d_period, const gc_float2 *d_coeffs,
                     float *d_svl, gc_svl_result *result, void *stream) {
    clear_error();
    auto calls = lock_device_calls();  // shared scratch arena
    int st = check_params(p, d_period);
    if (st) return st;
    GC_ARG(d_coeffs && d_svl, "NULL buffer");
    GC_ARG(p->range >= 0 && p->range <= kMaxRange, "range must be in [0, %d]", kMaxRange);
    const int side = 2 * p->range + 1;
    GC_ARG(p->harmonics >= 0 && p->harmonics <= side * side * side,
           "harmonics must be in [0, (2 range + 1)^3]");
    GC_ARG(p->cg_max_iter >= 1, "cg_max_iter must be >= 1");
    GC_ARG(p->cg_end_res > 0.f, "cg_end_res must be positive");
    st = check_dims(p->fx, p->fy, p->fz, 1);
    if (st) return st;
    hipStream_t s = (hipStream_t)stream;
    const uint64_t n = (uint64_t)p->nx * p->ny * p->nz;
    // the three unit right-hand sides, solved together; a harmonic's residual
    // is at most (|i| + |j| + |k|) times theirs, so they are solved to
    // cg_end_res / (3 range) to meet cg_end_res for every harmonic
    void *ws = nullptr;
    if ((st = scratch_arena(cg_bytes(3, p->nx, p->ny, p->nz), &ws))) return st;
    float *phi = (float *)ws, *b = cg_rhs(ws, n, 3);
    const int unit[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
    for (int a = 0; a < 3; ++a) {
        hipLaunchKernelGGL(finding_phi_kernel, stride_grid(n), dim3(256), 0, s, b + a * n,
                           d_period, phi_args(p, unit[a][0], unit[a][1], unit[a][2]));
        GC_CHECK_LAUNCH();
    }
    int iters[3] = {0, 0, 0};
    float res[3] = {0.f, 0.f, 0.f};
    const float tol = p->cg_end_res / (float)(3 * std::max(1, p->range));
    CgForm form;
    st = cg_solve(b, phi, 3, p->nx, p->ny, p->nz, p->cg_max_iter, tol, &form, iters, res, ws, s);
    if (st) {
        (void)hipStreamSynchronize(s);  // (the next call may have the arena on another stream)
        return st;
    }
    const Up u = {p->nx, p->ny, p->nz, p->fx, p->fy, p->fz, p->fine_dx, p->fine_dy, p->fine_dz};
    typedef void (*FieldKernel)(const float *, const float *, const float *, Up, const float2 *,
                                int, uint32_t, float *);
    static const FieldKernel kField[2][kMaxRange + 1] = {
        {svl_field_kernel<0, false>, svl_field_kernel<1, false>, svl_field_kernel<2, false>,
         svl_field_kernel<3, false>, svl_field_kernel<4, false>},
        {svl_field_kernel<0, true>, svl_field_kernel<1, true>, svl_field_kernel<2, true>,
         svl_field_kernel<3, true>, svl_field_kernel<4, true>}};
    // lanes of a row, workgroups along a row and over the rows (about 4096 in all)
    const uint64_t rows = (uint64_t)p->fy * p->fz;
    const uint64_t lanes = ((uint64_t)p->fx + kSvlPoints - 1) / kSvlPoints;
    const bool pack = lanes <= 32;
    uint32_t lanes_log2 = 0;
    while ((1ull << lanes_log2) < lanes) ++lanes_log2;
    const uint64_t along = (lanes + 63) / 64;
    const uint64_t wave_rows = pack ? 64 >> lanes_log2 : 1;
    const uint64_t over = (rows + 4 * wave_rows - 1) / (4 * wave_rows);
    const dim3 wgs((unsigned)std::min<uint64_t>(over, std::max<uint64_t>(1, 4096 / along)),
                   (unsigned)std::min<uint64_t>(along, 4096));
    hipLaunchKernelGGL(kField[pack][p->range], wgs, dim3(256), 0, s, phi, phi + n, phi + 2 * n, u,
                       (const float2 *)d_coeffs, p->harmonics, lanes_log2, d_svl);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(s));
    if (result) {
        for (int a = 0; a < 3; ++a) {
            result->cg_iters[a] = iters[a];
            result->cg_res[a] = res[a];
        }
    }
    return GPUCAD_OK;
}

int gpucad_unit_spectrum(const float *d_cell, int32_t nx, int32_t ny, int32_t nz, int32_t range,
                         gc_float2 *d_coeffs) {
    clear_error();
    auto calls = lock_device_calls();  // shared scratch arena
    GC_ARG(d_cell && d_coeffs, "NULL buffer");
    int st = check_dims(nx, ny, nz, 1);
    if (st) return st;
    GC_ARG(range >= 0 && range <= kMaxRange, "range must be in [0, %d]", kMaxRange);
    const int side = 2 * range + 1;
    const uint32_t nrows = (uint32_t)((uint64_t)ny * nz), piece = std::min(nrows, kDftPiece);
    const uint64_t nsums = (uint64_t)side * side * (range + 1);
    void *ws = nullptr;
    st = scratch_arena((nsums + (uint64_t)(range + 1) * piece) * sizeof(double2), &ws);
    if (st) return st;
    double2 *sums = (double2 *)ws, *rows = sums + nsums;
    typedef void (*RowsKernel)(const float *, int, uint32_t, double2 *);
    static const RowsKernel kRows[kMaxRange + 1] = {dft_rows_kernel<0>, dft_rows_kernel<1>,
                                                    dft_rows_kernel<2>, dft_rows_kernel<3>,
                                                    dft_rows_kernel<4>};
    for (uint64_t r = 0; r < nrows; r += piece) {
        const uint32_t first = (uint32_t)r, m = std::min(piece, nrows - first);
        hipLaunchKernelGGL(kRows[range], dim3((m - 1) / (4 * kDftRows) + 1), dim3(256), 0, 0,
                           d_cell + r * nx, nx, m, rows);
        GC_CHECK_LAUNCH();
        hipLaunchKernelGGL(dft_planes_kernel, dim3((unsigned)(side * side), (unsigned)(range + 1)),
                           dim3(256), 0, 0, rows, first, m, r + m == nrows, ny, nz, range,
                           (double)nx * ny * nz, sums, (float2 *)d_coeffs);
        GC_CHECK_LAUNCH();
    }
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_fft_fill(const gc_float2 *d_half, gc_float2 *d_full, int32_t nx, int32_t ny,
                    int32_t nz) {
    clear_error();
    GC_ARG(d_half && d_full, "NULL buffer");
    int st = check_dims(nx, ny, nz, 1);
    if (st) return st;
    GC_ARG(nx == ny && ny == nz, "the mirror indices assume a cubic grid");
    const uint64_t n = (uint64_t)(nx / 2 + 1) * ny * nz;
    hipLaunchKernelGGL(fft_fill_kernel, stride_grid(n), dim3(256), 0, 0, (const float2 *)d_half,
                       (float2 *)d_full, nx, ny, nz);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_fft_scale(gc_float2 *d_data, float scalar, uint64_t n) {
    clear_error();
    GC_ARG(d_data, "NULL buffer");
    hipLaunchKernelGGL(fft_scale_kernel, stride_grid(n), dim3(256), 0, 0, (float2 *)d_data, scalar,
                       n);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

}  // extern "C"
