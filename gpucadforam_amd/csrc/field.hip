// Field evaluation kernels.
//
//  * lattice_field_kernel: the native spatially varying TPMS lattice (see
//    gc_lattice_params in gpucad.h for the definition), one 64 x 4 x lz brick
//    per workgroup (lattice_body.hpp): each lane owns one (x, y) column and
//    walks `lz` z planes; each z step of a wave stores 64 consecutive floats
//    (256 B) and, if requested, the ballot of G < iso as one 64-bit sign word.
//
//  * drop-in kernels for the reference's field entry points:
//    Fft_lattice::create_lattice (src/lattice_files/Fft_lattice.cu:12-74),
//    the Modelling primitives (src/Modelling.cu:244-761),
//    Gratings::GPU_buffer_normalise_four (src/lattice_files/Gratings.cu:1089-1134,
//    1394-1495, 1579-1617) and Gratings::primitive_field
//    (src/lattice_files/Gratings.cu:1695-1734).
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>

#include "gc_common.hpp"
#include "gc_math.hpp"
#include "lattice_body.hpp"

namespace gc {
namespace {

// Rows per lane of the one-grid launch: a rotated lattice evaluates its z
// phase (and its cos) per lane and z, so four rows share it; without
// rotation the z terms come from the brick's table and one row per lane
// keeps small grids spread over more workgroups.
constexpr int rows_per_lane(bool rot) { return rot ? 4 : 1; }

// Bound by its vector instructions, near the field's write rate: 512^3 with
// every option 163 -> 158 us, 1024^3 bent 814 -> 762, a 203 x 149 x 181 part
// 49 -> 44 after its instructions were cut (constants in vector registers, the
// root by v_rsq and one correction, its range tested per column instead of
// per point, sign words by v_writelane).  Seven waves per SIMD: the rotated
// diamond's 74 registers hold six otherwise (512^3: 216 us, 208 so); with modes
// and a box that would take a scratch store per step.
template <bool ROT, int TPMS, bool THICK, int PRIM, int OP, bool XCD>
__global__ void __launch_bounds__(64 * kFieldWaves, !ROT ? 8 : (THICK && PRIM == GC_PRIM_BOX ? 6 : 7))
lattice_field_kernel(FieldConsts c, float *__restrict__ field, uint64_t *__restrict__ signs) {
    __shared__ float ztab[kMaxLZ * kZTab];
    constexpr int RY = rows_per_lane(ROT);
    // XCD: workgroup b runs on XCD b % 8, and the bricks of a row are 8
    // workgroups apart, in groups of 8 rows, so they share an L2 (rows_by_xcd)
    uint32_t bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    if (ROT && XCD) {
        // few rows of bricks: a last group takes what is left over all z runs
        const uint32_t nby = gridDim.y, b = bx + gridDim.x * (by + nby * bz);
        const uint32_t g = b / (8 * gridDim.x), in = b - g * 8 * gridDim.x;
        const uint32_t n = min(8u, nby * gridDim.z - 8 * g);
        bx = in / n;
        const uint32_t row = 8 * g + in % n;
        bz = row / nby;
        by = row - bz * nby;
    } else if (XCD) {
        // gridDim.x = 8 x bricks along x, no division; a last group of fewer
        // rows is dealt to other XCDs in every z run
        const uint32_t nby = ((uint32_t)c.ny + kFieldWaves - 1) / kFieldWaves;
        by = 8 * by + ((bx + (nby % 8 ? 3 * bz : 0)) & 7u);
        bx >>= 3;
        if (by >= nby) return;
    }
    lattice_brick<ROT, TPMS, THICK, 64, PRIM, OP, RY, !XCD>(
        c, field, signs, (int)bx * 64, (int)by * kFieldWaves * RY, (int)bz * c.lz, ztab);
}

typedef void (*FieldKernel)(FieldConsts, float *, uint64_t *);

// the primitive and the boolean are template parameters of the one-grid
// kernel: the per-point loop then carries no branch on them
template <bool XCD, bool ROT, int TPMS, bool THICK, int PRIM>
FieldKernel pick_op(int op) {
    switch (op) {
        case GC_OP_UNION: return lattice_field_kernel<ROT, TPMS, THICK, PRIM, GC_OP_UNION, XCD>;
        case GC_OP_SUBTRACT: return lattice_field_kernel<ROT, TPMS, THICK, PRIM, GC_OP_SUBTRACT, XCD>;
        case GC_OP_INTERSECT: return lattice_field_kernel<ROT, TPMS, THICK, PRIM, GC_OP_INTERSECT, XCD>;
        default: return lattice_field_kernel<ROT, TPMS, THICK, PRIM, GC_OP_NONE, XCD>;
    }
}

template <bool XCD, bool ROT, int TPMS, bool THICK>
FieldKernel pick_prim(int prim, int op) {
    switch (prim) {
        case GC_PRIM_SPHERE: return pick_op<XCD, ROT, TPMS, THICK, GC_PRIM_SPHERE>(op);
        case GC_PRIM_BOX: return pick_op<XCD, ROT, TPMS, THICK, GC_PRIM_BOX>(op);
        default: return lattice_field_kernel<ROT, TPMS, THICK, GC_PRIM_NONE, GC_OP_NONE, XCD>;
    }
}

template <bool XCD, bool ROT, int TPMS>
FieldKernel pick_thick(bool thick, int prim, int op) {
    return thick ? pick_prim<XCD, ROT, TPMS, true>(prim, op) : pick_prim<XCD, ROT, TPMS, false>(prim, op);
}

template <bool XCD, bool ROT>
FieldKernel pick_tpms(int tpms, bool thick, int prim, int op) {
    switch (tpms) {
        case GC_TPMS_GYROID: return pick_thick<XCD, ROT, GC_TPMS_GYROID>(thick, prim, op);
        case GC_TPMS_SCHWARZ_P: return pick_thick<XCD, ROT, GC_TPMS_SCHWARZ_P>(thick, prim, op);
        default: return pick_thick<XCD, ROT, GC_TPMS_DIAMOND>(thick, prim, op);
    }
}

}  // namespace

int validate_lattice(const gc_lattice_params *p) {
    GC_ARG(p, "params is NULL");
    GC_ARG(p->nx >= 2 && p->ny >= 2 && p->nz >= 2, "grid must have >= 2 points per axis");
    GC_ARG((uint64_t)p->nx * p->ny * p->nz < (1ull << 40), "grid too large");
    // the field kernels address a z plane with 32-bit byte offsets
    GC_ARG((uint64_t)p->nx * p->ny < (1ull << 30), "a z plane must hold fewer than 2^30 points");
    GC_ARG(p->tpms >= 0 && p->tpms <= 2, "unknown tpms %d", p->tpms);
    GC_ARG(p->period0 > 0.f && p->period1 > 0.f, "periods must be positive");
    GC_ARG(p->bend_radius >= 0.f, "bend radius must be >= 0");
    GC_ARG(!(p->bend_radius > 0.f && (p->rot0 != 0.f || p->rot1 != 0.f)),
           "rotation and bend are exclusive");
    GC_ARG(p->n_modes >= 0 && p->n_modes <= GC_MAX_MODES, "n_modes out of range");
    for (int m = 0; m < p->n_modes; ++m)
        for (int a = 0; a < 3; ++a)
            GC_ARG(p->mode_k[m][a] >= 0 && p->mode_k[m][a] <= 3, "mode wave numbers must be 0..3");
    GC_ARG(p->prim >= 0 && p->prim <= 2, "unknown primitive %d", p->prim);
    GC_ARG(p->op >= 0 && p->op <= 3, "unknown op %d", p->op);
    return GPUCAD_OK;
}

// z planes per workgroup of the one-grid launch.  A long run spreads the
// per-column work and the z table, a short one leaves more workgroups to fill
// the chip and its last wave.  With w = columns of bricks x planes the best run
// grew like sqrt(w) in sweeps from 33 x 47 x 61 to 1024^3 (rotated: 8 planes of
// 128^3, 10 of 203 x 149 x 181, 20 of 320 x 300 x 310; bent or with modes: 8 of
// 100^3, 20 of 200^3); 0.12 sqrt(w) is within 5 % of each, up to the longest run
// that pays (longest_z_run).  Large rotated grids, whose four rows per lane need
// more columns, are faster when five workgroups per CU take all of it at once,
// in runs of w / 1300 planes (512^3: 161 us in runs of 112, 173 of 47, 166 of 48:
// long runs are multiples of 16).  With an eighth of the planes (a fifth when
// rotated) and at least 16, as before: 40^3 5.0 us, now 3.1; rotated 128^3
// 31.9, now 17.5; 203 x 149 x 181 44.4, now 29.0; 320 x 300 x 310 76.9, now 60.
//
// Without rotation the longest run goes by what a column costs before its first
// point.  us at 512^3 in runs of 8, 16, 32, 64 and 96 (before: an eighth):
//   nothing            101  97.7  100  101  104 (102)
//   a primitive        125   109 96.2 99.4 99.2 (104)
//   bend, primitive    146   116  105  101 99.7 (110)
//   modes              225   158  125  110  104 (115)
// and with a row's bricks on one XCD, over 24 grids of 256^3 to 1024^3, against
// an eighth: nothing 0.88 in runs of 12, 0.90 of 16; bend 0.88 of 16, 0.95 of 12;
// primitive 0.93 of 24, 0.93 of 32, 0.98 of 16; bend and primitive 0.92 of 48,
// 0.93 of 64 (1024^3 827 and 785); modes 0.98 of 48 and 64, 1.06 of 32.  They
// differ by up to 10 % from one size to the next; edits, with their mesh, by 2 %.
// Past the 256 MB of the memory-side cache, rows that end inside a line need
// shorter runs: the parts of a line that two bricks share meet in the L2, which
// the active workgroups of an XCD, 1 KB each per plane, fill in 16 planes.  The
// more a plane costs the closer together they run.  us of 620^3 in runs of
// 12, 16, 24, 32 and 48 planes (before):
//   nothing            179  238  302  320  332 (477)
//   a primitive        211  201  180  309  330 (480)
//   bend, primitive    238  219  198  191  327 (483)
//   modes              323  289  247  221  325 (481)
//   all three          375  327  285  267  236 (487)
// and of 860^3 12 to 24 planes: 599 733 900; 548 514 824; 632 581 540.
int longest_z_run(const gc_lattice_params *p) {
    const bool bend = p->bend_radius > 0.f, prim = p->prim != GC_PRIM_NONE;
    const bool cut = p->nx % 32 != 0 && (uint64_t)p->nx * p->ny * p->nz >= (1u << 26);
    if (p->n_modes > 0) return cut && !prim ? 32 : (cut ? 48 : 64);
    if (prim && bend) return cut ? 24 : 64;
    if (prim) return cut ? 16 : 24;
    return bend && !cut ? 16 : 12;
}

int default_z_run(const gc_lattice_params *p, int bricks_x, int bricks_y) {
    const bool rot = p->rot0 != 0.f || p->rot1 != 0.f;
    const double w = (double)bricks_x * bricks_y * p->nz;
    const double best = std::max(0.12 * std::sqrt(w), rot ? w / 1300.0 : 0.0);
    int run = (int)std::min(std::max(best + 0.5, 4.0), (double)(rot ? kMaxLZ : longest_z_run(p)));
    run = std::max(run, (p->nz + 65534) / 65535);  // (a launch's third dimension)
    if (run > 40) return (run + 15) / 16 * 16;     // (the caller bounds it by kMaxLZ)
    const int chunks = (p->nz + run - 1) / run;
    return (p->nz + chunks - 1) / chunks;  // the planes evenly over the runs
}

// Whether a launch puts the bricks of a row on one XCD, where the lines and
// sign words that they share are merged in its L2: rows that end inside a line
// (500^3: 198 us plain and 228 rotated, 86 and 158 so), and without rotation
// whole lines as well, whose sign words share lines (edits: 1024^3 4.76 ms with
// the bricks over the XCDs, 4.67 so; 512^3 596 us, 582 so; 256 x 1024 x 1024 929,
// 886 so).  Not rotated grids of whole lines (the edit of 512^3 337 us, so 342).
// From 64 MB on: an edit of 128^3 took 22.1 us, so 22.4.  (Between them rows that
// end inside a line gain too: 203^3 17.3 us, so 12.1; 252^3 28.1, so 15.0; rotated
// 22.9 and 23.3, 34.1 and 29.2.)  The other launches store with the
// non-temporal hint always (field_nt_store).
bool rows_by_xcd(const gc_lattice_params *p, bool rot) {
    const uint64_t points = (uint64_t)p->nx * p->ny * p->nz;
    return points >= (1u << 24) && (!rot || p->nx % 32 != 0);
}

int launch_lattice_field(const gc_lattice_params *p, float *d_field, uint64_t *d_signs, float iso,
                         int lz, hipStream_t stream) {
    int st = validate_lattice(p);
    if (st) return st;
    GC_ARG(d_field, "field pointer is NULL");
    const bool rot = p->rot0 != 0.f || p->rot1 != 0.f;
    const int rows = rows_per_lane(rot);
    const int brick_y = kFieldWaves * rows;
    if (lz <= 0) lz = default_z_run(p, (p->nx + 63) / 64, (p->ny + brick_y - 1) / brick_y);
    if (lz > kMaxLZ) lz = kMaxLZ;
    const FieldConsts c = make_field_consts(p, iso, lz, (uint64_t)p->nx * p->ny * p->nz);
    const bool thick = p->n_modes > 0;
    dim3 grid((p->nx + 63) / 64, (p->ny + brick_y - 1) / brick_y, (p->nz + lz - 1) / lz);
    GC_ARG(grid.y <= 65535 && grid.z <= 65535, "grid too large for one launch");
    // (a launch holds fewer than 2^32 threads along x)
    const bool by_xcd =
        rows_by_xcd(p, rot) && (rot || (uint64_t)grid.x * 8 * 64 * kFieldWaves <= 0xffffffffull);
    const auto pick = by_xcd ? (rot ? pick_tpms<true, true> : pick_tpms<true, false>)
                             : (rot ? pick_tpms<false, true> : pick_tpms<false, false>);
    FieldKernel k = pick(p->tpms, thick, c.prim, c.op);
    if (!rot && by_xcd) {  // (lattice_field_kernel)
        grid.x *= 8;
        grid.y = (grid.y + 7) / 8;
    }
    hipLaunchKernelGGL(k, grid, dim3(64 * kFieldWaves), 0, stream, c, d_field, d_signs);
    GC_CHECK_LAUNCH();
    return GPUCAD_OK;
}

// ===========================================================================
// Drop-in field kernels
// ===========================================================================
namespace {

// Euler rotation rows exactly as the reference forms them in each primitive
// kernel (src/Modelling.cu:401-407), evaluated once on the host.
struct Rows {
    float3 x, y, z;
};

Rows euler_rows(gc_float3 a) {
    float cx = cosf(a.x), sx = sinf(a.x);
    float cy = cosf(a.y), sy = sinf(a.y);
    float cz = cosf(a.z), sz = sinf(a.z);
    Rows r;
    r.x = make_float3(cz * cy, cz * sy * sx - sz * cx, cz * sy * cx + sz * sx);
    r.y = make_float3(sz * cy, sz * sy * sx + cz * cx, sz * sy * cx - cz * sx);
    r.z = make_float3(-1.0f * sy, cy * sx, cy * cx);
    return r;
}

// Points are taken in runs of kRunPoints per workgroup: kRun per thread, 256
// apart.  The run's first point is decoded once (in 32 bits where they hold
// it), a thread's first from it, and the rest by steps with one carry per
// axis.
constexpr int kRun = 8;
constexpr uint32_t kRunPoints = 256 * kRun;

struct PointSteps {
    uint32_t nx, ny;
    uint32_t dx, dy, dz;  // `step` points as steps along x, y, z
};

PointSteps point_steps(int nx, int ny, uint32_t step) {
    PointSteps s;
    const uint64_t plane = (uint64_t)nx * ny;
    s.nx = (uint32_t)nx;
    s.ny = (uint32_t)ny;
    s.dz = (uint32_t)(step / plane);
    s.dy = (uint32_t)(step % plane / (uint64_t)nx);
    s.dx = (uint32_t)(step % plane % (uint64_t)nx);
    return s;
}

struct Point {
    uint32_t x, y, z;
    // point `first` + `ahead` (first: the same in every lane)
    __device__ __forceinline__ Point(const PointSteps &s, uint64_t first, uint32_t ahead) {
        const uint64_t plane = (uint64_t)s.nx * s.ny;
        if (((first | plane) >> 32) == 0) {
            z = (uint32_t)first / (uint32_t)plane;
            const uint32_t rem = (uint32_t)first - z * (uint32_t)plane;
            y = rem / s.nx;
            x = rem - y * s.nx;
        } else {
            const uint64_t zb = first / plane, rem = first - zb * plane, yb = rem / s.nx;
            z = (uint32_t)zb;
            y = (uint32_t)yb;
            x = (uint32_t)(rem - yb * s.nx);
        }
        // x, y < 2^31 and `ahead` is small: no sum wraps
        x += ahead;
        const uint32_t rows = x / s.nx;
        x -= rows * s.nx;
        y += rows;
        const uint32_t planes = y / s.ny;
        y -= planes * s.ny;
        z += planes;
    }
    __device__ __forceinline__ void advance(const PointSteps &s, uint32_t dx, uint32_t dy,
                                            uint32_t dz) {
        x += dx;
        y += dy;
        z += dz;
        if (x >= s.nx) {
            x -= s.nx;
            ++y;
        }
        if (y >= s.ny) {
            y -= s.ny;
            ++z;
        }
    }
};

struct Grid3 {
    int nx, ny, nz;
    float dx, dy, dz;
    float mx, my, mz;  // (N-1)/2.0
    PointSteps s;
};

Grid3 make_grid(int nx, int ny, int nz, float dx, float dy, float dz) {
    Grid3 g;
    g.nx = nx; g.ny = ny; g.nz = nz;
    g.dx = dx; g.dy = dy; g.dz = dz;
    g.mx = (float)((nx - 1) / 2.0);
    g.my = (float)((ny - 1) / 2.0);
    g.mz = (float)((nz - 1) / 2.0);
    g.s = point_steps(nx, ny, 256);
    return g;
}

// fn(i, x, y, z) for the points of this thread.  A primitive is bound by the
// 4 bytes that it writes per point once the point's coordinates cost little:
// cuboid on 211 x 193 x 229 25.2 us with a 64-bit division per point and axis,
// 18.0 so.
template <class F>
__device__ __forceinline__ void for_points(const Grid3 &g, F fn) {
    const uint64_t n = (uint64_t)g.nx * g.ny * g.nz, first = (uint64_t)blockIdx.x * kRunPoints;
    Point p(g.s, first, threadIdx.x);
    uint64_t i = first + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kRun; ++k) {
        if (i >= n) return;
        fn(i, (int)p.x, (int)p.y, (int)p.z);
        p.advance(g.s, g.s.dx, g.s.dy, g.s.dz);
        i += 256;
    }
}

__device__ __forceinline__ float3 centred(const Grid3 &g, int xx, int yy, int zz, float3 c) {
    return make_float3(((float)xx - g.mx) * g.dx - c.x, ((float)yy - g.my) * g.dy - c.y,
                       ((float)zz - g.mz) * g.dz - c.z);
}

__device__ __forceinline__ float dot_rows(float3 v, float3 r) {
    return v.x * r.x + v.y * r.y + v.z * r.z;
}

__global__ void sphere_kernel(Grid3 g, float *out, float3 c, float radius, float thick, int shell) {
    for_points(g, [&](uint64_t i, int xx, int yy, int zz) {
        float3 v = centred(g, xx, yy, zz, c);
        float t_diff = (float)(thick / 2.0);
        float r2 = v.x * v.x + v.y * v.y + v.z * v.z;
        if (shell) {
            float ri = radius - t_diff, ro = radius + t_diff;
            float f1 = r2 - ri * ri;
            float f2 = r2 - ro * ro;
            out[i] = (float)fmax((double)f1 * -1.0, (double)f2);
        } else {
            out[i] = r2 - radius * radius;
        }
    });
}

__global__ void cuboid_kernel(Grid3 g, float *out, float3 c, Rows R, float xw, float yw, float zw) {
    for_points(g, [&](uint64_t i, int xx, int yy, int zz) {
        float3 v = centred(g, xx, yy, zz, c);
        float f1 = fabsf(dot_rows(v, R.x)) - xw;
        float f2 = fabsf(dot_rows(v, R.y)) - yw;
        float f3 = fabsf(dot_rows(v, R.z)) - zw;
        out[i] = fmaxf(fmaxf(f1, f2), f3);
    });
}

__global__ void cuboid_shell_kernel(Grid3 g, float *out, float3 c, Rows R, float xw, float yw,
                                    float zw, float thick) {
    for_points(g, [&](uint64_t i, int xx, int yy, int zz) {
        float3 v = centred(g, xx, yy, zz, c);
        float f1 = dot_rows(v, R.x);
        float f11 = fabsf(f1) - xw;
        float f12 = fabsf(f1) - (xw - thick);
        float f2 = dot_rows(v, R.y);
        float f21 = fabsf(f2) - yw;
        float f22 = fabsf(f2) - (yw - thick);
        float f3 = fabsf(dot_rows(v, R.z)) - zw;
        double inner = (double)fmaxf(f12, f22) * -1.0;
        out[i] = (float)fmax(fmax((double)fmaxf(f11, f21), inner), (double)f3);
    });
}

__global__ void pyramid_kernel(Grid3 g, float *out, float3 c, Rows R, float xwb, float xwt,
                               float yh, float zwb, float zwt) {
    for_points(g, [&](uint64_t i, int xx, int yy, int zz) {
        float3 v = centred(g, xx, yy, zz, c);
        float f1 = dot_rows(v, R.x);
        float f2 = dot_rows(v, R.y);
        float f3 = dot_rows(v, R.z);
        float ratio = (yh - f2) / yh;
        float xw = ratio * (xwb - xwt) + xwt;
        f1 = fabsf(f1) - xw;
        f2 = fabsf(f2 - yh / 2) - yh / 2;
        float zw = ratio * (zwb - zwt) + zwt;
        f3 = fabsf(f3) - zw;
        out[i] = fmaxf(fmaxf(f1, f2), f3);
    });
}

__global__ void torus_kernel(Grid3 g, float *out, float3 c, Rows R, float tr, float cr) {
    for_points(g, [&](uint64_t i, int xx, int yy, int zz) {
        float3 v = centred(g, xx, yy, zz, c);
        float vx = dot_rows(v, R.x), vy = dot_rows(v, R.y), vz = dot_rows(v, R.z);
        float side = tr - __builtin_sqrtf(vx * vx + vy * vy);
        out[i] = vz * vz - cr * cr + side * side;
    });
}

__global__ void cone_kernel(Grid3 g, float *out, float3 c, Rows R, float br, float h) {
    for_points(g, [&](uint64_t i, int xx, int yy, int zz) {
        float3 v = centred(g, xx, yy, zz, c);
        float q = h / br;
        float f2 = q * q;
        float vx = dot_rows(v, R.x), vy = dot_rows(v, R.y), vz = dot_rows(v, R.z);
        float gg = (float)((double)vy - (double)h / 2.0);
        float hh = (float)fmax(((double)gg - (double)h / 2.0) * 100.0,
                               ((double)gg + (double)h / 2.0) * 100.0 * -1.0);
        float d = vy - h;
        float f1 = ((vx * vx + vz * vz) * f2) - d * d;
        out[i] = fmaxf(f1, hh);
    });
}

__global__ void cone_frustum_kernel(Grid3 g, float *out, float3 c, Rows R, float tr, float br,
                                    float h) {
    for_points(g, [&](uint64_t i, int xx, int yy, int zz) {
        float3 v = centred(g, xx, yy, zz, c);
        float vx = dot_rows(v, R.x), vy = dot_rows(v, R.y), vz = dot_rows(v, R.z);
        float r_diff = ((h - vy) / h) * (br - tr);
        float gg = (float)((double)vy - (double)h / 2.0);
        float hh = (float)fmax(((double)gg - (double)h / 2.0) * 100.0,
                               ((double)gg + (double)h / 2.0) * 100.0 * -1.0);
        double rr = (double)(r_diff + tr);
        float f1 = (float)((double)(vx * vx + vz * vz) - rr * rr);
        out[i] = fmaxf(f1, hh);
    });
}

__global__ void line_kernel(Grid3 g, float *out, float3 c, float3 axis, float radius, float t_diff,
                            float t_diff_ax, int cyl) {
    for_points(g, [&](uint64_t i, int xx, int yy, int zz) {
        float x1 = ((float)xx - g.mx) * g.dx;
        float y1 = ((float)yy - g.my) * g.dy;
        float z1 = ((float)zz - g.mz) * g.dz;
        float3 end = make_float3(axis.x + c.x, axis.y + c.y, axis.z + c.z);
        float3 w1 = make_float3(x1 - c.x, y1 - c.y, z1 - c.z);
        float3 w2 = make_float3(x1 - end.x, y1 - end.y, z1 - end.z);
        float3 w3 = make_float3(end.x - c.x, end.y - c.y, end.z - c.z);
        float3 d = make_float3(w1.y * w2.z - w1.z * w2.y, w1.z * w2.x - w1.x * w2.z,
                               w1.x * w2.y - w1.y * w2.x);
        float e = __builtin_sqrtf(d.x * d.x + d.y * d.y + d.z * d.z);
        float dis = __builtin_sqrtf(w3.x * w3.x + w3.y * w3.y + w3.z * w3.z);
        float f = e / dis;
        float gg = (x1 - c.x) * axis.x + (y1 - c.y) * axis.y + (z1 - c.z) * axis.z;
        float f1 = fmaxf(gg - t_diff_ax, (gg + t_diff_ax) * -1.0f);
        float f2;
        if (cyl)
            f2 = fmaxf(f - (radius + t_diff), (f - (radius - t_diff)) * -1.0f);
        else
            f2 = f - radius;
        out[i] = fmaxf(f1, f2);
    });
}

// Fft_lattice::create_lattice unit-cell forms (src/lattice_files/Fft_lattice.cu:12-66).
__global__ void unit_lattice_kernel(float *out, uint32_t nx, uint32_t ny, uint32_t nz,
                                    uint32_t type) {
    uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t y = blockIdx.y * blockDim.y + threadIdx.y;
    uint32_t z = blockIdx.z * blockDim.z + threadIdx.z;
    if (x >= nx || y >= ny || z >= nz) return;
    float xx = (float)((((double)x * 1.0) / (double)(nx - 1) - 0.5) / 0.5);
    float yy = (float)((((double)y * 1.0) / (double)(ny - 1) - 0.5) / 0.5);
    float zz = (float)((((double)z * 1.0) / (double)(nz - 1) - 0.5) / 0.5);
    float ax = (float)(3.14 * (double)xx), ay = (float)(3.14 * (double)yy),
          az = (float)(3.14 * (double)zz);
    float aa = 0.f;
    if (type == 0) {
        aa = cosf(ax) * sinf(ay) + cosf(ay) * sinf(az) + cosf(az) * sinf(ax);
    } else if (type == 1) {
        aa = cosf(ax) + cosf(ay) + cosf(az);
    } else if (type == 2) {
        aa = 4 * (cosf(xx) * cosf(yy) * cosf(zz)) -
             (cosf(2 * xx) * cosf(2 * yy) + cosf(2 * yy) * cosf(2 * zz) + cosf(2 * zz) * cosf(2 * xx));
    } else if (type == 3) {
        float bx = (float)(2 * 3.14 * (double)xx), by = (float)(2 * 3.14 * (double)yy),
              bz = (float)(2 * 3.14 * (double)zz);
        aa = 2 * (cosf(ax) * cosf(ay) + cosf(ay) * cosf(az) + cosf(az) * cosf(ax)) -
             (cosf(bx) + cosf(by) + cosf(bz));
    } else if (type == 4) {
        double X2 = (double)xx * (double)xx, Y2 = (double)yy * (double)yy,
               Z2 = (double)zz * (double)zz;
        double a = (double)(xx * xx) + Y2;
        aa = (float)fmin(fmin(a, Y2 + Z2), Z2 + X2);
    } else if (type == 5) {
        double t1 = cos(3.14 * (double)xx) * (double)cosf(ay) * (double)cosf(az);
        aa = (float)(t1 - (double)(sinf(ax) * sinf(ay) * sinf(az)));
    }
    out[(uint64_t)x + (uint64_t)y * nx + (uint64_t)z * nx * ny] = aa;
}

// ---- normalise_four: min/max (seeded with 0) then band indicator
// A workgroup's min and max into thread 0 (lo, hi: the thread's own).
__device__ __forceinline__ void block_minmax(float &lo, float &hi) {
    __shared__ float smin[4], smax[4];
    for (int d = 32; d > 0; d >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, d, 64));
        hi = fmaxf(hi, __shfl_xor(hi, d, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        smin[threadIdx.x >> 6] = lo;
        smax[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    lo = fminf(fminf(smin[0], smin[1]), fminf(smin[2], smin[3]));
    hi = fmaxf(fmaxf(smax[0], smax[1]), fmaxf(smax[2], smax[3]));
}

// Bound by the bytes read, with eight loads per thread under way (one load
// per iteration before: 240^3 19.5 us, now 11.2).
__global__ void __launch_bounds__(256) minmax_partial_kernel(const float *in, uint64_t n,
                                                             float2 *partial) {
    float lo = 0.f, hi = 0.f;  // the reference's second pass seeds with 0
    const uint64_t stride = (uint64_t)gridDim.x * 256;
    uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    for (; i + 7 * stride < n; i += 8 * stride) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = in[i + k * stride];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            lo = fminf(lo, v[k]);
            hi = fmaxf(hi, v[k]);
        }
    }
    for (; i < n; i += stride) {
        lo = fminf(lo, in[i]);
        hi = fmaxf(hi, in[i]);
    }
    block_minmax(lo, hi);
    if (threadIdx.x == 0) partial[blockIdx.x] = make_float2(lo, hi);
}

__global__ void __launch_bounds__(256) minmax_final_kernel(float2 *partial, int nparts) {
    float lo = 0.f, hi = 0.f;
    for (int i = threadIdx.x; i < nparts; i += 256) {
        lo = fminf(lo, partial[i].x);
        hi = fmaxf(hi, partial[i].y);
    }
    block_minmax(lo, hi);
    if (threadIdx.x == 0) partial[0] = make_float2(lo, hi);
}

// Points in fours, kBandFours per thread; VEC: the three arrays are 16-byte
// aligned.  Bound by the 12 bytes per point: 240^3 40.5 us with 64-bit
// divisions per point, 26.4 so.
constexpr int kBandFours = 4;
constexpr uint32_t kBandPoints = 1024 * kBandFours;

template <bool VEC>
__global__ void __launch_bounds__(256) band_kernel(const float *in, float *indicator,
                                                   float *normalised, const float2 *ab,
                                                   PointSteps s, uint32_t nz, float iso1,
                                                   float iso2) {
    const uint64_t size = (uint64_t)s.nx * s.ny * nz;
    const uint64_t first = (uint64_t)blockIdx.x * kBandPoints;
    const float a = ab->x, b = ab->y;
    Point p(s, first, 4 * threadIdx.x);
    uint64_t i = first + 4 * threadIdx.x;
    float v[kBandFours][4];
#pragma unroll
    for (int k = 0; k < kBandFours; ++k) {
        const uint64_t j = i + 1024 * k;
        if (VEC && j + 3 < size) {
            const float4 q = *(const float4 *)(in + j);
            v[k][0] = q.x;
            v[k][1] = q.y;
            v[k][2] = q.z;
            v[k][3] = q.w;
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) v[k][c] = j + c < size ? in[j + c] : 0.f;
        }
    }
#pragma unroll
    for (int k = 0; k < kBandFours; ++k) {
        const uint64_t j = i + 1024 * k;
        float m[4], t[4];
        Point q = p;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bool face = q.x == 0 || q.x == s.nx - 1 || q.y == 0 || q.y == s.ny - 1 ||
                              q.z == 0 || q.z == nz - 1;
            const float f = (v[k][c] - a) / (b - a);
            m[c] = !face && f >= iso1 && f <= iso2 ? 1.f : 0.f;
            t[c] = face ? 0.f : f;
            q.advance(s, 1, 0, 0);
        }
        p.advance(s, s.dx, s.dy, s.dz);
        if (VEC && j + 3 < size) {
            *(float4 *)(indicator + j) = make_float4(m[0], m[1], m[2], m[3]);
            *(float4 *)(normalised + j) = make_float4(t[0], t[1], t[2], t[3]);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (j + c < size) {
                    indicator[j + c] = m[c];
                    normalised[j + c] = t[c];
                }
        }
    }
}

__global__ void primitive_dynamic_kernel(const float *active, float *iso, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && active[i] >= 0.f) iso[i] = FLT_MAX;
}

// grid_points {int val; float t_x, t_y, t_z;}: only val is read
__global__ void primitive_fixed_kernel(const int4 *fixed, float *iso, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && fixed[i].x > -1) iso[i] = FLT_MAX;
}

int point_launch(int nx, int ny, int nz, dim3 *grid, uint32_t per_block = 256) {
    GC_ARG(nx >= 1 && ny >= 1 && nz >= 1, "grid sizes must be positive");
    uint64_t n = (uint64_t)nx * ny * nz;
    GC_ARG((n + 255) / 256 <= 0x7fffffffull, "grid too large");
    uint64_t blocks = (n + per_block - 1) / per_block;
    *grid = dim3((unsigned)blocks);
    return GPUCAD_OK;
}

}  // namespace
}  // namespace gc

using namespace gc;

namespace gc {
// min and max of in[0, n) seeded with 0 (the reference's reductions seed their
// second pass with 0) into part[0]; part holds 1024 float2
int enqueue_minmax0(const float *in, uint64_t n, float2 *part, hipStream_t st) {
    hipLaunchKernelGGL(minmax_partial_kernel, dim3(1024), dim3(256), 0, st, in, n, part);
    GC_CHECK_LAUNCH();
    hipLaunchKernelGGL(minmax_final_kernel, dim3(1), dim3(256), 0, st, part, 1024);
    GC_CHECK_LAUNCH();
    return GPUCAD_OK;
}
}  // namespace gc

extern "C" {

uint64_t gpucad_sign_words(int32_t nx, int32_t ny, int32_t nz) {
    if (nx <= 0 || ny <= 0 || nz <= 0) return 0;
    return (uint64_t)((nx + 63) / 64) * (uint64_t)ny * (uint64_t)nz;
}

int gpucad_lattice_field(const gc_lattice_params *p, float *d_field, uint64_t *d_signs, float iso,
                         void *stream) {
    clear_error();
    return launch_lattice_field(p, d_field, d_signs, iso, 0, as_stream(stream));
}

// Same launch with an explicit z-run length (autotuning hook).
int gpucad_lattice_field_lz(const gc_lattice_params *p, float *d_field, uint64_t *d_signs,
                            float iso, int32_t lz, void *stream) {
    clear_error();
    return launch_lattice_field(p, d_field, d_signs, iso, lz, as_stream(stream));
}

int gpucad_create_lattice(float *d, uint32_t nx, uint32_t ny, uint32_t nz, uint32_t size,
                          uint32_t type) {
    clear_error();
    GC_ARG(d, "output is NULL");
    GC_ARG(nx >= 2 && ny >= 2 && nz >= 2, "grid must have >= 2 points per axis");
    GC_ARG(type <= 5, "lattice type must be 0..5");
    (void)size;
    dim3 tids(16, 8, 8);
    dim3 grids((nx + 15) / 16, (ny + 7) / 8, (nz + 7) / 8);
    hipLaunchKernelGGL(unit_lattice_kernel, grids, tids, 0, 0, d, nx, ny, nz, type);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

#define GC_PRIM_PROLOGUE(ptr)                                   \
    clear_error();                                              \
    GC_ARG(ptr, "output is NULL");                              \
    dim3 grid;                                                  \
    {                                                           \
        int st_ = point_launch(nx, ny, nz, &grid, kRunPoints);  \
        if (st_) return st_;                                    \
    }                                                           \
    Grid3 g = make_grid(nx, ny, nz, dx, dy, dz);

#define GC_PRIM_EPILOGUE()            \
    GC_CHECK_LAUNCH();                \
    GC_HIP(hipStreamSynchronize(0)); \
    return GPUCAD_OK;

int gpucad_sphere_with_center(float *data, gc_float3 center, float radius, float thickness,
                              int32_t nx, int32_t ny, int32_t nz, float dx, float dy, float dz,
                              int32_t shell) {
    GC_PRIM_PROLOGUE(data)
    hipLaunchKernelGGL(sphere_kernel, grid, dim3(256), 0, 0, g, data,
                       make_float3(center.x, center.y, center.z), radius, thickness, shell);
    GC_PRIM_EPILOGUE()
}

int gpucad_cuboid(float *data, gc_float3 center, gc_float3 angles, float x_width, float y_width,
                  float z_width, int32_t nx, int32_t ny, int32_t nz, float dx, float dy,
                  float dz) {
    GC_PRIM_PROLOGUE(data)
    Rows R = euler_rows(angles);
    hipLaunchKernelGGL(cuboid_kernel, grid, dim3(256), 0, 0, g, data,
                       make_float3(center.x, center.y, center.z), R, (float)(x_width / 2.0),
                       (float)(y_width / 2.0), (float)(z_width / 2.0));
    GC_PRIM_EPILOGUE()
}

int gpucad_cuboid_shell(float *data, gc_float3 center, gc_float3 angles, float x_width,
                        float y_width, float z_width, float thickness, int32_t nx, int32_t ny,
                        int32_t nz, float dx, float dy, float dz) {
    GC_PRIM_PROLOGUE(data)
    Rows R = euler_rows(angles);
    hipLaunchKernelGGL(cuboid_shell_kernel, grid, dim3(256), 0, 0, g, data,
                       make_float3(center.x, center.y, center.z), R, (float)(x_width / 2.0),
                       (float)(y_width / 2.0), (float)(z_width / 2.0), thickness);
    GC_PRIM_EPILOGUE()
}

int gpucad_pyramid_frustum(float *data, gc_float3 center, gc_float3 angles, float x_width_base,
                           float x_width_top, float y_height, float z_width_base,
                           float z_width_top, int32_t nx, int32_t ny, int32_t nz, float dx,
                           float dy, float dz) {
    GC_PRIM_PROLOGUE(data)
    Rows R = euler_rows(angles);
    hipLaunchKernelGGL(pyramid_kernel, grid, dim3(256), 0, 0, g, data,
                       make_float3(center.x, center.y, center.z), R, (float)(x_width_base / 2.0),
                       (float)(x_width_top / 2.0), y_height, (float)(z_width_base / 2.0),
                       (float)(z_width_top / 2.0));
    GC_PRIM_EPILOGUE()
}

int gpucad_torus_with_center(float *data, gc_float3 center, gc_float3 angles, float torus_radius,
                             float circle_radius, int32_t nx, int32_t ny, int32_t nz, float dx,
                             float dy, float dz) {
    GC_PRIM_PROLOGUE(data)
    Rows R = euler_rows(angles);
    hipLaunchKernelGGL(torus_kernel, grid, dim3(256), 0, 0, g, data,
                       make_float3(center.x, center.y, center.z), R, torus_radius, circle_radius);
    GC_PRIM_EPILOGUE()
}

int gpucad_cone_with_base_radius_height(float *data, gc_float3 center, gc_float3 angles,
                                        float base_radius, float cone_height, int32_t nx,
                                        int32_t ny, int32_t nz, float dx, float dy, float dz) {
    GC_PRIM_PROLOGUE(data)
    Rows R = euler_rows(angles);
    hipLaunchKernelGGL(cone_kernel, grid, dim3(256), 0, 0, g, data,
                       make_float3(center.x, center.y, center.z), R, base_radius, cone_height);
    GC_PRIM_EPILOGUE()
}

int gpucad_cone_frustum(float *data, gc_float3 center, gc_float3 angles, float top_radius,
                        float bottom_radius, float height, int32_t nx, int32_t ny, int32_t nz,
                        float dx, float dy, float dz) {
    GC_PRIM_PROLOGUE(data)
    Rows R = euler_rows(angles);
    hipLaunchKernelGGL(cone_frustum_kernel, grid, dim3(256), 0, 0, g, data,
                       make_float3(center.x, center.y, center.z), R, top_radius, bottom_radius,
                       height);
    GC_PRIM_EPILOGUE()
}

int gpucad_distance_from_line(float *data, gc_float3 center, gc_float3 axis, float radius,
                              float thickness_radial, float thickness_axial, int32_t nx,
                              int32_t ny, int32_t nz, float dx, float dy, float dz,
                              int32_t cylinder_disc) {
    GC_PRIM_PROLOGUE(data)
    float mag = sqrtf(axis.x * axis.x + axis.y * axis.y + axis.z * axis.z);
    GC_ARG(mag > 0.f, "axis must be non-zero");
    float3 ax = make_float3(axis.x / mag, axis.y / mag, axis.z / mag);
    hipLaunchKernelGGL(line_kernel, grid, dim3(256), 0, 0, g, data,
                       make_float3(center.x, center.y, center.z), ax, radius,
                       (float)(thickness_radial / 2.0), (float)(thickness_axial / 2.0),
                       cylinder_disc);
    GC_PRIM_EPILOGUE()
}

int gpucad_normalise_four(const float *in, float *indicator, float *normalised, uint64_t size,
                          int32_t nx, int32_t ny, int32_t nz, float iso1, float iso2) {
    clear_error();
    auto calls = lock_device_calls();  // shared scratch arena
    GC_ARG(in && indicator && normalised, "NULL buffer");
    GC_ARG(nx >= 1 && ny >= 1 && nz >= 1, "grid sizes must be positive");
    GC_ARG(size == (uint64_t)nx * ny * nz, "size must equal nx*ny*nz");
    const int nparts = 1024;
    void *ws = nullptr;
    int st = scratch_arena(nparts * sizeof(float2), &ws);
    if (st) return st;
    float2 *part = (float2 *)ws;
    hipLaunchKernelGGL(minmax_partial_kernel, dim3(nparts), dim3(256), 0, 0, in, size, part);
    GC_CHECK_LAUNCH();
    hipLaunchKernelGGL(minmax_final_kernel, dim3(1), dim3(256), 0, 0, part, nparts);
    GC_CHECK_LAUNCH();
    const uint64_t blocks = (size + kBandPoints - 1) / kBandPoints;
    GC_ARG(blocks <= 0x7fffffffull, "grid too large");
    const bool vec = (((uintptr_t)in | (uintptr_t)indicator | (uintptr_t)normalised) & 15) == 0;
    hipLaunchKernelGGL(vec ? band_kernel<true> : band_kernel<false>, dim3((unsigned)blocks),
                       dim3(256), 0, 0, in, indicator, normalised, part,
                       point_steps(nx, ny, 1024), (uint32_t)nz, iso1, iso2);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_primitive_field_dynamic(const float *primitive_active, float *isosurf, int32_t nx,
                                   int32_t ny, int32_t nz) {
    clear_error();
    GC_ARG(primitive_active && isosurf, "NULL buffer");
    dim3 grid;
    int st = point_launch(nx, ny, nz, &grid);
    if (st) return st;
    hipLaunchKernelGGL(primitive_dynamic_kernel, grid, dim3(256), 0, 0, primitive_active, isosurf,
                       (uint64_t)nx * ny * nz);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

int gpucad_primitive_field_fixed(const void *primitive_fixed, float *isosurf, int32_t nx,
                                 int32_t ny, int32_t nz) {
    clear_error();
    GC_ARG(primitive_fixed && isosurf, "NULL buffer");
    dim3 grid;
    int st = point_launch(nx, ny, nz, &grid);
    if (st) return st;
    hipLaunchKernelGGL(primitive_fixed_kernel, grid, dim3(256), 0, 0,
                       (const int4 *)primitive_fixed, isosurf, (uint64_t)nx * ny * nz);
    GC_CHECK_LAUNCH();
    GC_HIP(hipStreamSynchronize(0));
    return GPUCAD_OK;
}

}  // extern "C"
