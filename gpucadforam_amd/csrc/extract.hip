// Native marching-cubes extraction with shared-edge vertex dedup.
//
// Classification follows the reference (cube bit k = [f(corner k) < iso],
// corner/edge numbering of src/MarchingCubes_kernel.cu:3449-3456, 3506-3517;
// triangle lists of src/tables.h).  The output is canonical:
//   vertex k   = k-th crossing grid edge in edge-id order 3*point + axis,
//                point = x + nx*(y + ny*z); each edge interpolated once from its
//                low end: t = (iso - f0)/(f1 - f0), v = fma(t, p1 - p0, p0);
//   triangle j = j-th triangle in cell order, triTable order inside a cell.
//
// The grid is seen through its sign words: bit b of word w of row r = y+ny*z
// is [f(64w+b, y, z) < iso].  A word (k = r*W + w) is the unit of
// bookkeeping: the lane that owns it (or half of it) derives the crossing
// edges of its points and the active cells with bit arithmetic.
//
// Launches (one stream, no host round trip, no inter-block waits):
//   signs : ballot of f < iso per 64 points; skipped when the field kernel
//           already produced the words
//   count : blocks of 256 words: vertex and triangle sums per block, each
//           word's first vertices and first triangle within its block, and
//           which groups of 8 words have something to emit
//   scan  : one workgroup scans the block sums (64-bit), writes the totals
//           and the vertex/triangle range of each grid; one grid of few
//           blocks needs no such launch, its emission sums them itself
//   emit  : a wave takes 8, 16 or 32 consecutive words, lists their cells (and
//           the points with an edge but no cell) in canonical order and runs
//           one lane per list entry: the 12 edge vertex numbers from popcounts
//           of the crossings of the four rows touching the cell, its triangles
//           and its own edges; then one lane per edge and one per triangle.
//           A wave's vertices and triangles are contiguous ranges whose starts
//           follow from count and scan.
//
// The kernels see grids as segments: a grid's words occupy a contiguous range
// of global blocks; the many-grid form (batched and served) finds each block's
// grid in a block -> grid table.  Both run the same code, so a grid's mesh
// does not depend on what it is launched with.
#include "extract_types.hpp"

namespace gc {
namespace {

struct ExtractLayout {
    uint64_t signs_off, base_off, live_off, bsum_off, ctl_off, res_off, bytes;
    uint64_t words, nb;
};

inline uint64_t align256(uint64_t v) { return (v + 255) & ~uint64_t(255); }

ExtractLayout layout(int nx, int ny, int nz) {
    ExtractLayout L;
    L.words = gpucad_sign_words(nx, ny, nz);
    L.nb = (L.words + kBlock - 1) / kBlock;
    uint64_t off = 0;
    L.signs_off = off;
    off = align256(off + L.words * 8);
    L.base_off = off;
    off = align256(off + L.nb * kBaseBytesPerBlock);
    L.live_off = off;
    off = align256(off + L.nb * kLiveBytesPerBlock);
    L.bsum_off = off;
    off = align256(off + L.nb * 16);
    L.ctl_off = off;  // [0] n_vertices [1] n_triangles [2] vertex numbers overflow 32 bits
    L.res_off = off + 64;
    off = align256(off + 64 + sizeof(SegResult));
    L.bytes = off;
    return L;
}

enum { CTL_NV = 0, CTL_NT = 1, CTL_OVF = 2 };

__device__ __forceinline__ uint64_t shift1(uint64_t cur, uint64_t next) {
    return (cur >> 1) | (next << 63);
}
__device__ __forceinline__ uint32_t popc64(uint64_t w) { return (uint32_t)__popcll(w); }
__device__ __forceinline__ uint32_t popc32(uint32_t w) { return (uint32_t)__popc(w); }
__device__ __forceinline__ uint64_t load_u64(const void *base, uint32_t off) {
    return *(const uint64_t *)((const char *)base + off);
}
__device__ __forceinline__ uint64_t mask_below(int64_t n) {
    if (n >= 64) return ~0ull;
    if (n <= 0) return 0ull;
    return (1ull << n) - 1ull;
}
__device__ __forceinline__ uint32_t gather32(uint32_t v, uint32_t src) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(src << 2), (int)v);
}
__device__ __forceinline__ uint32_t readlane32(uint32_t v, uint32_t l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}

// inclusive scan over the 64 lanes of a wave with DPP moves (no LDS): shifts
// by 1, 2, 4, 8 inside each row of 16 lanes, then the last lane of row 0 / 2
// is broadcast into rows 1 / 3 (row_bcast:15) and the last lane of row 1 into
// rows 2 and 3 (row_bcast:31).  Lanes without a source add the `old` operand, 0.
__device__ __forceinline__ uint32_t wave_scan_incl(uint32_t v) {
    int x = (int)v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return (uint32_t)x;
}

// 12-byte records with 4-byte alignment (stored as one dwordx3 where possible)
struct V3 {
    float x, y, z;
};
struct T3 {
    uint32_t a, b, c;
};

// The mesh is written once and not read back by this launch: its 12-byte
// records are stored with the non-temporal hint (one dwordx3 store each).
typedef float F3nt __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t U3nt __attribute__((ext_vector_type(3), aligned(4)));
__device__ __forceinline__ void store_nt(float *p, V3 v) {
    __builtin_nontemporal_store(F3nt{v.x, v.y, v.z}, (F3nt *)p);
}
__device__ __forceinline__ void store_nt(uint32_t *p, T3 t) {
    __builtin_nontemporal_store(U3nt{t.a, t.b, t.c}, (U3nt *)p);
}

__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv &f) {
    const uint32_t q = __umulhi(n, f.m);  // n / d or one less
    return q + (n - q * f.d >= f.d ? 1u : 0u);
}

struct WordPos {
    int y, z, w;
};
__device__ __forceinline__ WordPos word_pos(uint64_t k, const Grid &g) {
    const uint32_t kk = (uint32_t)k;
    const uint32_t r = fdiv(kk, g.divW);
    const uint32_t z = fdiv(r, g.divNy);
    WordPos p;
    p.w = (int)(kk - r * (uint32_t)g.W);
    p.z = (int)z;
    p.y = (int)(r - z * (uint32_t)g.ny);
    return p;
}

// ---------------------------------------------------------------------------
// grids and block scheduling
// ---------------------------------------------------------------------------
struct OneGrid {
    Seg s;
    __device__ __forceinline__ uint32_t seg_of(uint32_t) const { return 0; }
    __device__ __forceinline__ Seg get(uint32_t) const { return s; }
};

struct ManyGrids {
    const Seg *__restrict__ segs;
    const uint32_t *__restrict__ blk2seg;
    __device__ __forceinline__ uint32_t seg_of(uint32_t b) const {
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)blk2seg[b]);
    }
    __device__ __forceinline__ Seg get(uint32_t i) const { return segs[i]; }
};

// ---------------------------------------------------------------------------
// signs
// ---------------------------------------------------------------------------
// A wave makes the words of 64 points of kSignZ rows, one above the other in
// z.  Bound by the field's bytes; the rows' loads are all under way before
// the first comparison (one load, one wait and one 8-byte store per row
// before: 203 x 149 x 181, 22 MB, 12.6 us; 8.0 now).
constexpr int kSignZ = 8;

__global__ void __launch_bounds__(256)
signs_kernel(const float *__restrict__ field, uint64_t *__restrict__ signs, int nx, int ny, int nz,
             int W, float iso) {
    const uint32_t lane = threadIdx.x & 63;
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int x = blockIdx.x * 64 + lane;
    const int z0 = blockIdx.z * kSignZ;
    if (y >= ny) return;
    const bool xin = x < nx;
    const uint64_t plane = (uint64_t)nx * ny;
    const float *p = field + (uint64_t)z0 * plane + (uint64_t)y * nx + (xin ? x : nx - 1);
    const int n = min(kSignZ, nz - z0);
    float f[kSignZ];
#pragma unroll
    for (int i = 0; i < kSignZ; ++i) f[i] = p[(uint64_t)min(i, n - 1) * plane];
    __builtin_amdgcn_sched_barrier(0);
    uint64_t mine = 0;
#pragma unroll
    for (int i = 0; i < kSignZ; ++i) {
        const uint64_t m = __ballot(xin && f[i] < iso);
        mine = lane == (uint32_t)i ? m : mine;
    }
    if (lane < (uint32_t)n) signs[((uint64_t)(z0 + lane) * ny + y) * W + blockIdx.x] = mine;
}

// ---------------------------------------------------------------------------
// count
// ---------------------------------------------------------------------------
// Triangles the case table gives the active cells of one word, from the
// corner words k0..k7 (bit x of kc: corner c of cell x is inside, f < iso;
// corners 0 (x,y,z) 1 (x+1,y,z) 2 (x+1,y+1,z) 3 (x,y+1,z) 4 (x,y,z+1)
// 5 (x+1,y,z+1) 6 (x+1,y+1,z+1) 7 (x,y+1,z+1), the case table's numbering,
// bit c of the case index).  For every one of the table's 255 cases
// with an outside corner, a cell with inside-corner set S has
//   |S| - 2 (faces of the cube with all four corners in S)
//       - 4 [S = the cube minus both ends of a body diagonal]
// triangles: each crossing edge is a vertex of exactly one polygon of the
// case and a polygon of k vertices is cut into k - 2 triangles, so the count
// is (3|S| - 2 edges in S) - 2 polygons; the polygons are as many as the
// Euler characteristic |S| - edges + faces of S, except in the four
// body-diagonal cases, which have two (characteristic 0).  The identity is
// checked case by case against the table by the tests.  So a word's count is
// a weighted sum of popcounts over its 64 cells, with no per-cell lookup.
// The sums run over all cells of the word, not only the active ones: a cell
// with every corner outside adds 0 to each of them, and one with every corner
// inside adds 8 - 2 * 6 = -4, which the last term takes back.  Corner bits of
// cells past the end of the row must be 0 (the caller masks them).
__device__ __forceinline__ uint32_t word_triangles(uint64_t k0, uint64_t k1, uint64_t k2,
                                                   uint64_t k3, uint64_t k4, uint64_t k5,
                                                   uint64_t k6, uint64_t k7) {
    const uint32_t v = popc64(k0) + popc64(k1) + popc64(k2) + popc64(k3) + popc64(k4) +
                       popc64(k5) + popc64(k6) + popc64(k7);
    const uint64_t p01 = k0 & k1, p23 = k2 & k3, p45 = k4 & k5, p67 = k6 & k7;
    const uint64_t p12 = k1 & k2, p56 = k5 & k6, p03 = k0 & k3, p47 = k4 & k7;
    const uint64_t bottom = p01 & p23, top = p45 & p67;
    const uint32_t f = popc64(bottom) + popc64(top) + popc64(p01 & p45) + popc64(p23 & p67) +
                       popc64(p12 & p56) + popc64(p03 & p47);
    // body diagonals (0,6) (1,7) (2,4) (3,5): both ends outside, the rest inside
    const uint32_t d = popc64(~(k0 | k6) & p12 & p45 & k3 & k7) +
                       popc64(~(k1 | k7) & p03 & p56 & k2 & k4) +
                       popc64(~(k2 | k4) & p01 & p67 & k3 & k5) +
                       popc64(~(k3 | k5) & p12 & p67 & k0 & k4);
    const uint32_t inside = popc64(bottom & top);
    return v - 2 * f - 4 * d + 4 * inside;
}

// Block of workgroup b of n: workgroup b runs on XCD b % 8, and each XCD takes
// runs of 1 << lr consecutive blocks, so the rows and planes next to a block's
// own are in its L2.
__device__ __forceinline__ uint32_t run_order(uint32_t b, uint32_t n, uint32_t lr) {
    const uint32_t first = b >> (lr + 3) << (lr + 3);  // of the 8 runs
    if (n - first < (8u << lr)) return b;
    const uint32_t in = b - first;
    return first + ((in & 7u) << lr) + (in >> 3);
}

struct CountArgs {
    const uint64_t *signs;  // sign buffer base
    uint32_t *live;         // per block: bit i: its words 8i .. 8i + 7 have something to emit
    uint64_t *bsum;
    // per word: first vertex of its two half words (16 bits each) and its
    // first triangle, within the block (at most 49152 and 81920)
    uint2 *base;
    uint32_t lr;            // log2 of the blocks of a run
};

// Bound by the words that it reads four times, in rows and planes, and the 8
// bytes that it writes per word (1024^3: 134 MB each, 130 us).
template <class Src>
__global__ void __launch_bounds__(kBlock) count_kernel(Src src, CountArgs a) {
    __shared__ uint32_t s_sum[4][2];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    {
        const uint32_t gb = run_order(blockIdx.x, gridDim.x, a.lr);
        const Seg s = src.get(src.seg_of(gb));
        const Grid &g = s.g;
        const uint64_t *signs = a.signs + s.sign_off;
        const uint64_t k = (uint64_t)(gb - s.block_off) * kBlock + tid;
        uint32_t vc = 0, tc = 0, vlo = 0;
        if (k < g.words) {
            const WordPos p = word_pos(k, g);
            const bool has_y = p.y + 1 < g.ny, has_z = p.z + 1 < g.nz;
            // a row or word that does not exist stands for its predecessor: no
            // crossing between rows, and past the row's last word the masks
            // leave no bit that a next word would reach
            const uint32_t W8 = 8u * (uint32_t)g.W;
            const uint32_t dy = has_y ? W8 : 0u, dz = has_z ? (uint32_t)g.ny * W8 : 0u;
            const uint32_t dn = p.w + 1 < g.W ? 8u : 0u;
            const uint64_t *at = signs + (gb - s.block_off) * (uint64_t)kBlock;
            const uint32_t oa = 8u * tid, ob = oa + dy, oc = oa + dz, od = ob + dz;
            const uint64_t wa = load_u64(at, oa), an = load_u64(at, oa + dn);
            const uint64_t wb = load_u64(at, ob), bn = load_u64(at, ob + dn);
            const uint64_t wc = load_u64(at, oc), cn = load_u64(at, oc + dn);
            const uint64_t wd = load_u64(at, od), dn_ = load_u64(at, od + dn);
            // all eight loads issue before any of the arithmetic on them
            __builtin_amdgcn_sched_barrier(0);
            const uint64_t sa = shift1(wa, an), sb = shift1(wb, bn);
            const uint64_t sc = shift1(wc, cn), sd = shift1(wd, dn_);
            const uint64_t vpt = mask_below((int64_t)g.nx - 64 * p.w);
            const uint64_t ved = mask_below((int64_t)g.nx - 1 - 64 * p.w);
            const uint64_t any = (wa | sa | wb | sb | wc | sc | wd | sd) & vpt;
            const uint64_t all = wa & sa & wb & sb & wc & sc & wd & sd;
            // (a wave with all its signs equal, cells and own edges: nothing)
            if (__any((any & ~all) != 0)) {
                const uint64_t ex = (wa ^ sa) & ved;
                const uint64_t ey = (wa ^ wb) & vpt;
                const uint64_t ez = (wa ^ wc) & vpt;
                vlo = popc32((uint32_t)ex) + popc32((uint32_t)ey) + popc32((uint32_t)ez);
                vc = vlo + popc32((uint32_t)(ex >> 32)) + popc32((uint32_t)(ey >> 32)) +
                     popc32((uint32_t)(ez >> 32));
                if (has_y && has_z)
                    tc = word_triangles(wa & ved, sa & ved, sb & ved, wb & ved, wc & ved, sc & ved,
                                        sd & ved, wd & ved);
            }
        }
        const uint32_t vincl = wave_scan_incl(vc);
        const uint32_t vw = readlane32(vincl, 63);
        const uint32_t tincl = wave_scan_incl(tc);
        const uint32_t tw = readlane32(tincl, 63);
        const uint64_t used = __ballot((vc | tc) != 0);
        const uint64_t eights = __ballot(lane < 8 && ((used >> 8 * (lane & 7)) & 0xffu) != 0);
        if (lane == 0) {
            s_sum[wave][0] = vw;
            s_sum[wave][1] = tw;
            ((uint8_t *)a.live)[4 * (uint64_t)gb + wave] = (uint8_t)eights;
        }
        __syncthreads();
        if (k < g.words) {
            uint32_t v0 = vincl - vc, t0 = tincl - tc;
            for (uint32_t i = 0; i < 4; ++i) {
                v0 += i < wave ? s_sum[i][0] : 0u;
                t0 += i < wave ? s_sum[i][1] : 0u;
            }
            a.base[(uint64_t)gb * kBlock + tid] = make_uint2(v0 | (v0 + vlo) << 16, t0);
        }
        if (tid == 0) {
            a.bsum[2 * (uint64_t)gb] =
                (uint64_t)s_sum[0][0] + s_sum[1][0] + s_sum[2][0] + s_sum[3][0];
            a.bsum[2 * (uint64_t)gb + 1] =
                (uint64_t)s_sum[0][1] + s_sum[1][1] + s_sum[2][1] + s_sum[3][1];
        }
    }
}

// ---------------------------------------------------------------------------
// scan of the block sums (one workgroup); ctl = totals and the overflow flag;
// res = each grid's vertex and triangle range
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024)
scan_blocks_kernel(uint64_t *bsum, uint64_t nb, uint64_t *ctl, uint64_t *d_counts,
                   const Seg *segs, uint32_t nseg, SegResult *res) {
    // Wave w scans the contiguous entries [w*per, (w+1)*per) in steps of 64
    // (lane l takes entry 64*step + l: coalesced 16-byte loads and stores).
    // A block's sums (at most 256 words x 192 crossing edges, or 256 x 64
    // cells x 5 triangles) and a step's (64 of them) fit 32 bits, so each
    // step is a DPP wave scan of 32-bit values with 64-bit carries.  The
    // first kKeep steps stay in registers for the write-back (8192 blocks:
    // a 512^3 grid); steps past them are read again and scanned again.
    constexpr int kWaves = 16, kKeep = 8;
    static_assert((uint64_t)64 * kBlock * 64 * 5 < (1ull << 32), "a step's sums fit 32 bits");
    __shared__ uint64_t sw_v[kWaves], sw_t[kWaves];
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    ulonglong2 *io = (ulonglong2 *)bsum;
    const uint64_t per = (nb + kWaves * 64 - 1) / (kWaves * 64) * 64;
    const uint64_t w0 = min(nb, (uint64_t)wave * per), w1 = min(nb, w0 + per);
    const uint32_t nsteps = (uint32_t)((w1 - w0 + 63) / 64);
    uint32_t qv[kKeep], qt[kKeep];
#pragma unroll
    for (int u = 0; u < kKeep; ++u) {
        const uint64_t i = w0 + 64 * (uint64_t)u + lane;
        const ulonglong2 q = i < w1 ? io[i] : make_ulonglong2(0ull, 0ull);
        qv[u] = (uint32_t)q.x;
        qt[u] = (uint32_t)q.y;
    }
    uint32_t ev[kKeep], et[kKeep], tv[kKeep], tt[kKeep];  // exclusive scans, step totals
    uint64_t sv = 0, st = 0;                              // the wave's totals
#pragma unroll
    for (int u = 0; u < kKeep; ++u) {
        const uint32_t iv = wave_scan_incl(qv[u]), it = wave_scan_incl(qt[u]);
        ev[u] = iv - qv[u];
        et[u] = it - qt[u];
        tv[u] = readlane32(iv, 63);
        tt[u] = readlane32(it, 63);
        sv += tv[u];
        st += tt[u];
    }
    for (uint32_t u = kKeep; u < nsteps; ++u) {
        const uint64_t i = w0 + 64 * (uint64_t)u + lane;
        const ulonglong2 q = i < w1 ? io[i] : make_ulonglong2(0ull, 0ull);
        sv += readlane32(wave_scan_incl((uint32_t)q.x), 63);
        st += readlane32(wave_scan_incl((uint32_t)q.y), 63);
    }
    if (lane == 0) {
        sw_v[wave] = sv;
        sw_t[wave] = st;
    }
    __syncthreads();
    uint64_t rv = 0, rt = 0, carry_v = 0, carry_t = 0;
    for (uint32_t w = 0; w < kWaves; ++w) {
        if (w < wave) {
            rv += sw_v[w];
            rt += sw_t[w];
        }
        carry_v += sw_v[w];
        carry_t += sw_t[w];
    }
#pragma unroll
    for (int u = 0; u < kKeep; ++u) {
        const uint64_t i = w0 + 64 * (uint64_t)u + lane;
        if (i < w1) io[i] = make_ulonglong2(rv + ev[u], rt + et[u]);
        rv += tv[u];
        rt += tt[u];
    }
    for (uint32_t u = kKeep; u < nsteps; ++u) {
        const uint64_t i = w0 + 64 * (uint64_t)u + lane;
        const ulonglong2 q = i < w1 ? io[i] : make_ulonglong2(0ull, 0ull);
        const uint32_t iv = wave_scan_incl((uint32_t)q.x), it = wave_scan_incl((uint32_t)q.y);
        if (i < w1) io[i] = make_ulonglong2(rv + (iv - (uint32_t)q.x), rt + (it - (uint32_t)q.y));
        rv += readlane32(iv, 63);
        rt += readlane32(it, 63);
    }
    __syncthreads();
    // every thread holds the totals; the scanned sums are visible to the workgroup
    int any_ovf = 0;
    for (uint32_t i = t; i < nseg; i += 1024) {
        const uint64_t b0 = segs ? segs[i].block_off : 0;
        const uint64_t b1 = (segs && i + 1 < nseg) ? segs[i + 1].block_off : nb;
        // one grid: its first block's prefix is 0 (no read back)
        const uint64_t v0 = segs ? bsum[2 * b0] : 0ull, t0 = segs ? bsum[2 * b0 + 1] : 0ull;
        const uint64_t v1 = b1 < nb ? bsum[2 * b1] : carry_v;
        const uint64_t t1 = b1 < nb ? bsum[2 * b1 + 1] : carry_t;
        SegResult r;
        r.v_off = v0;
        r.nv = v1 - v0;
        r.t_off = t0;
        r.nt = t1 - t0;
        r.ovf = r.nv > 0xffffffffull ? 1u : 0u;
        r.pad = 0;
        res[i] = r;
        any_ovf |= (int)r.ovf;
    }
    any_ovf = __syncthreads_or(any_ovf);
    if (t == 0) {
        ctl[CTL_NV] = carry_v;
        ctl[CTL_NT] = carry_t;
        ctl[CTL_OVF] = any_ovf ? 1 : 0;
        if (d_counts) {
            d_counts[0] = carry_v;
            d_counts[1] = carry_t;
        }
    }
}

// ---------------------------------------------------------------------------
// emit: vertices and triangles
// ---------------------------------------------------------------------------
// Vertex on the edge from point (xf, yf, zf) along axis ax with end values f0,
// f1: t = (iso - f0)/(f1 - f0), p = fma(t, p1 - p0, p0) on that axis.  The
// three axes are interpolated and the edge's own one is kept (lanes of a wave
// hold edges of all three): selects cost twice an FMA.
struct Frame {
    float iso, ox, oy, oz, sx, sy, sz;
};
__device__ __forceinline__ V3 edge_vertex(const Frame &s, float xf, float yf, float zf, uint32_t ax,
                                          float f0, float f1) {
    const float t = (s.iso - f0) / (f1 - f0);
    const float px = __builtin_fmaf(xf, s.sx, s.ox);
    const float py = __builtin_fmaf(yf, s.sy, s.oy);
    const float pz = __builtin_fmaf(zf, s.sz, s.oz);
    const float ex = __builtin_fmaf(t, __builtin_fmaf(xf + 1.0f, s.sx, s.ox) - px, px);
    const float ey = __builtin_fmaf(t, __builtin_fmaf(yf + 1.0f, s.sy, s.oy) - py, py);
    const float ez = __builtin_fmaf(t, __builtin_fmaf(zf + 1.0f, s.sz, s.oz) - pz, pz);
    return V3{ax == 0 ? ex : px, ax == 1 ? ey : py, ax == 2 ? ez : pz};
}

constexpr int kEmitWaves = 4;          // waves per workgroup
constexpr int kCellCap = 512;          // cells of a wave listed at a time
constexpr int kRing = 256;             // edges waiting: at most 63 + a step's 192
constexpr int kIdStride = kEmitStride; // vertex numbers of an edge: 64 cells + 1 (banks)
// One grid of up to this many blocks needs no scan launch: every workgroup of
// the emission sums the counts (two per thread).  203 x 149 x 181, 422 blocks:
// 42.5 us for scan and emission (4.9 of them the scan, and its launch), 35.6 so.
constexpr int kSelfBlocks = 512;

constexpr uint32_t kMixed = ~0u;

struct EmitArgs {
    const float *field;     // field buffer base
    const uint64_t *signs;  // sign buffer base
    const uint2 *base;      // per word: block-local numbers (count_kernel)
    const uint32_t *live;   // per block: groups with something to emit
    const uint64_t *bsum;   // first vertex and triangle of each block (kSelf: their counts)
    const SegResult *res;
    const uint32_t *table;  // 5 x 256 triangle words (host_emit_table)
    float *vertices;
    uint64_t vcap;
    uint32_t *triangles;
    uint64_t tcap;
    uint32_t lw;            // log2 of the words per wave: 3, 4 or 5
    uint32_t lr;            // log2 of the workgroups of a run, or kMixed
    uint32_t nb;            // kSelf: blocks of the grid
    uint64_t *ctl, *d_counts;  // kSelf: written by the first workgroup
};

struct EmitWave {
    uint32_t vid[12 * kIdStride];  // vertex number of edge e of cell l at e * kIdStride + l
    uint32_t own[5 * 64 + 8];      // a step's triangles: byte offsets of their three numbers
    uint16_t list[kCellCap];       // cells: owner lane * 4 | x << 8
    uint16_t ring[kRing];          // edges: the cell's entry | axis
};

template <bool kSelf>
struct EmitShared {
    EmitWave w[kEmitWaves];
    uint64_t stride[3];  // bytes from a point to the next one along an axis
    uint32_t tab[5 * 256];  // words 0 and 1 in pairs, 2 and 3 in pairs, 4
    uint32_t pre[kSelf ? kSelfBlocks : 1];  // first vertex of each block
    uint2 sum[kSelf ? kEmitWaves : 1];      // the sums, wave by wave
    uint32_t first_tri;                     // first triangle of this block
};

// a wave's LDS accesses are in order: this only keeps the compiler from
// moving them across
__device__ __forceinline__ void wave_sync() { __builtin_amdgcn_wave_barrier(); }
// keeps a lane's LDS stores in program order, unmerged
__device__ __forceinline__ void in_order() { asm volatile("" ::: "memory"); }

__device__ __forceinline__ uint32_t below32(int n) {
    return n <= 0 ? 0u : (n >= 32 ? ~0u : (1u << n) - 1u);
}
__device__ __forceinline__ uint32_t load_u32(const void *base, uint32_t off) {
    return *(const uint32_t *)((const char *)base + off);
}

// Records of 12 bytes by which p lies past a 128-byte line boundary, modulo
// the 32 of three lines: 3 n = p / 4 mod 32, and 11 is the inverse of 3.
__device__ __forceinline__ uint32_t past_line(const void *p) {
    return (uint32_t)((uint64_t)p >> 2) * 11u & 31u;
}
// records [0, n) of a wave that fit below a capacity of `cap`, the wave's
// record `skip` being number `at`
__device__ __forceinline__ uint32_t record_limit(uint64_t cap, uint64_t at, uint32_t skip) {
    return cap > at ? (uint32_t)min(cap - at, (uint64_t)0x40000000u) + skip : 0u;
}

// The whole mesh of a chunk of 8, 16 or 32 words by one wave.
//
// Bound by the bytes it moves: at 1024^3 (222 M vertices, 445 M triangles) 14.6
// GB by the counters (6.2 read, 8.4 written), 2.8 ms at the rate of a large
// copy; at 512^3 0.73 GB, 140 us.  The vector units are busy 60 % and LDS 50 %
// of the time at 1024^3.
// One wave makes a chunk's vertices and triangles, so the signs are loaded and
// the crossings derived once and the edges come out of the cell steps as a
// ring, without a pass of their own (two kinds of workgroup before: 18 % of
// the vector instructions were second copies of this set-up, 30 % the edge
// lists).  Edge and triangle records leave 64 at a time on 128-byte line
// boundaries: non-temporal stores of 12-byte records move 3.9 TB/s when every
// store ends inside a line and 5.0 TB/s when only a wave's first and last do.
// 1024^3: 3231 -> 2665 us, 512^3: 186 -> 172 (143 in runs of a plane, run_order),
// 128^3: 25 -> 15, 40^3: 23 -> 10.
//
// Workgroups of four waves: they share the triangle table, and with eight a
// wave that is done waits for more of the others before its LDS is free
// (1024^3: 2860).  LDS (29 KB) and registers hold five workgroups per CU;
// owner data in LDS instead of cross-lane reads costs two of them (3225).
template <class Src, bool kSelf>
__global__ void __launch_bounds__(64 * kEmitWaves)
emit_kernel(Src src, EmitArgs a) {
    __shared__ EmitShared<kSelf> sh;
    constexpr uint32_t kThreads = 64 * kEmitWaves;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    // Few blocks: neighbours over the XCDs, mixed with the higher bits so that
    // no XCD has the same rows of every plane (run_log2).
    uint32_t bx = blockIdx.x;
    if (a.lr != kMixed)
        bx = run_order(bx, gridDim.x, a.lr);
    else if ((bx | 7u) < gridDim.x)
        bx ^= (bx >> 3 ^ bx >> 6 ^ bx >> 9 ^ bx >> 12 ^ bx >> 15) & 7u;
    // a workgroup takes 4 << lw words of a block of 256
    const uint32_t lw = a.lw, lparts = 6 - lw;
    const uint32_t gb = bx >> lparts, part = bx & ((1u << lparts) - 1u);
    const uint32_t w0 = (kEmitWaves * part + wave) << lw;  // the wave's first word in its block
    static_assert(kEmitWaves == 4 && kBlock == 256, "64 >> lw workgroups per block");
    uint64_t vblock, tblock;  // the block's first vertex and triangle
    ulonglong2 q0 = make_ulonglong2(0, 0), q1 = q0;
    if constexpr (kSelf) {
        static_assert(kSelfBlocks == 2 * kThreads, "two blocks per thread");
        if (2 * tid < a.nb) q0 = ((const ulonglong2 *)a.bsum)[2 * tid];
        if (2 * tid + 1 < a.nb) q1 = ((const ulonglong2 *)a.bsum)[2 * tid + 1];
    }
    const uint32_t live = a.live[gb];
    const uint32_t wg_groups = kEmitWaves << lw >> 3;  // groups of 8 words per workgroup
    const bool wg_live = (live >> (part * wg_groups)) & ((1u << wg_groups) - 1u);
    if (!wg_live && !(kSelf && gb == 0 && part == 0)) return;
    const uint32_t si = src.seg_of(gb);
    const Seg s = src.get(si);
    const Grid &g = s.g;
    // words of this wave: [k0, k0 + (1 << lw)); lane: one half word
    const uint32_t k0 = (gb - s.block_off) * kBlock + w0;
    const uint32_t h = lane & 1;
    const uint32_t kw = k0 + (lane >> 1);
    const bool mine = lane < (2u << lw) && kw < (uint32_t)g.words;
    const uint32_t kk = mine ? kw : k0;
    const bool wave_live = (live >> (w0 >> 3)) & ((1u << (1u << (lw - 3))) - 1u);
    uint32_t wa, wb, wc, wd, we, wf, wg, wh, na, nb, nc, nd, ne;
    uint32_t b1 = 0, b2 = 0, b3 = 0, vb1, vb2, vb3, todo = 0, cy = 0, off = 0, yz = 0, xh = 0, row0 = 0;
    constexpr int kTab = 5 * 256 / kThreads;
    static_assert(kTab * kThreads == 5 * 256, "the table is loaded whole");
    uint32_t tb[kTab];
#pragma unroll
    for (int i = 0; i < kTab; ++i) tb[i] = a.table[tid + i * kThreads];
    uint2 first = make_uint2(0, 0);
    if (wave_live) {
        const WordPos p = word_pos(kk, g);
        row0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(p.z * g.ny + p.y));
        xh = 64u * (uint32_t)p.w + 32u * h;
        off = ((uint32_t)(p.z * g.ny + p.y) - row0) * (uint32_t)g.nx + xh;
        yz = (uint32_t)p.y | (uint32_t)p.z << 16;
        const bool has_y = p.y + 1 < g.ny, has_z = p.z + 1 < g.nz;
        // a row that does not exist stands for its own predecessor (no
        // crossing between them), so no load needs a mask
        const uint32_t W8 = 8u * (uint32_t)g.W, RW8 = (uint32_t)g.ny * W8;
        const uint32_t dy = has_y ? W8 : 0u, dz = has_z ? RW8 : 0u;
        const uint32_t dy2 = p.y + 2 < g.ny ? W8 : 0u, dz2 = p.z + 2 < g.nz ? RW8 : 0u;
        const uint32_t dn = h == 0 || p.w + 1 < g.W ? 4u : 0u;  // the row's next half
        const uint64_t *sg = a.signs + s.sign_off + k0;
        const uint32_t oa = 8u * (kk - k0) + 4u * h;
        const uint32_t ob = oa + dy, oc = oa + dz, od = ob + dz, oe = ob + dy2;
        wa = load_u32(sg, oa);
        wb = load_u32(sg, ob);
        wc = load_u32(sg, oc);
        wd = load_u32(sg, od);
        we = load_u32(sg, oe);
        wf = load_u32(sg, oe + dz);
        wg = load_u32(sg, oc + dz2);
        wh = load_u32(sg, od + dz2);
        na = load_u32(sg, oa + dn);
        nb = load_u32(sg, ob + dn);
        nc = load_u32(sg, oc + dn);
        nd = load_u32(sg, od + dn);
        ne = load_u32(sg, oe + dn);
        // first vertex of the half within its block, and of the block
        const uint2 *bg = a.base + (uint64_t)s.block_off * kBlock + k0;
        first = bg[0];
        vb1 = *(const uint16_t *)((const char *)bg + (ob - 2u * h));
        vb2 = *(const uint16_t *)((const char *)bg + (oc - 2u * h));
        vb3 = *(const uint16_t *)((const char *)bg + (od - 2u * h));
        b1 = (k0 + (ob >> 3)) >> 8;
        b2 = (k0 + (oc >> 3)) >> 8;
        b3 = (k0 + (od >> 3)) >> 8;
        if constexpr (!kSelf) {
            const uint64_t *gs = a.bsum + 2 * (uint64_t)s.block_off;
            const uint32_t v_off = (uint32_t)a.res[si].v_off;
            vb1 += (uint32_t)gs[2 * (uint64_t)b1] - v_off;
            vb2 += (uint32_t)gs[2 * (uint64_t)b2] - v_off;
            vb3 += (uint32_t)gs[2 * (uint64_t)b3] - v_off;
        }
        __builtin_amdgcn_sched_barrier(0);
        // the sign past the row's last point repeats it (no crossing there)
        const int nv = g.nx - (int)xh;  // points from this half on
        const uint32_t mw = (uint32_t)nv < 32u ? 1u << nv : 0u;
        const uint32_t mn = nv == 32 ? 1u : (nv == 33 ? 2u : 0u);
        na = (na & ~mn) | (__builtin_amdgcn_alignbit(na, wa, 31) & mn);
        nb = (nb & ~mn) | (__builtin_amdgcn_alignbit(nb, wb, 31) & mn);
        nc = (nc & ~mn) | (__builtin_amdgcn_alignbit(nc, wc, 31) & mn);
        wa = (wa & ~mw) | ((wa + wa) & mw);
        wb = (wb & ~mw) | ((wb + wb) & mw);
        wc = (wc & ~mw) | ((wc + wc) & mw);
        const uint32_t sa = __builtin_amdgcn_alignbit(na, wa, 1);
        const uint32_t sb = __builtin_amdgcn_alignbit(nb, wb, 1);
        const uint32_t sc = __builtin_amdgcn_alignbit(nc, wc, 1);
        const uint32_t sd = __builtin_amdgcn_alignbit(nd, wd, 1);
        const uint32_t own = (wa ^ sa) | (wa ^ wb) | (wa ^ wc);  // points with an edge
        const uint32_t any = wa | sa | wb | sb | wc | sc | wd | sd;
        const uint32_t all = wa & sa & wb & sb & wc & sc & wd & sd;
        const uint32_t cells = has_y && has_z ? below32(nv - 1) : 0u;
        todo = mine ? (own & below32(nv)) | (any & ~all & cells) : 0u;
        cy = (na & 3u) | (nb & 3u) << 2 | (nc & 3u) << 4 | (nd & 1u) << 6 | (ne & 1u) << 7 |
             (uint32_t)__popc(cells) << 16;
    }
    if constexpr (kSelf) {
        // block sums -> first vertex of every block, this block's first
        // triangle; the first block's workgroup writes the totals (512 blocks
        // hold at most 512 x 81920 triangles: 32 bits)
        const uint32_t qv = (uint32_t)(q0.x + q1.x), qt = (uint32_t)(q0.y + q1.y);
        const uint32_t iv = wave_scan_incl(qv), it = wave_scan_incl(qt);
        if (lane == 63) sh.sum[wave] = make_uint2(iv, it);
        __syncthreads();
        uint32_t v = iv - qv, t = it - qt;
        for (uint32_t i = 0; i < kEmitWaves; ++i) {
            v += i < wave ? sh.sum[i].x : 0u;
            t += i < wave ? sh.sum[i].y : 0u;
        }
        sh.pre[2 * tid] = v;
        sh.pre[2 * tid + 1] = v + (uint32_t)q0.x;
        if (tid == gb >> 1) sh.first_tri = t + (gb & 1 ? (uint32_t)q0.y : 0u);
        if (gb == 0 && part == 0 && tid == kThreads - 1) {
            a.ctl[CTL_NV] = v + qv;
            a.ctl[CTL_NT] = t + qt;
            a.ctl[CTL_OVF] = 0;
            if (a.d_counts) {
                a.d_counts[0] = v + qv;
                a.d_counts[1] = t + qt;
            }
        }
        if (!wg_live) return;
        __syncthreads();
        if (wave_live) {
            vb1 += sh.pre[b1];
            vb2 += sh.pre[b2];
            vb3 += sh.pre[b3];
        }
        vblock = sh.pre[gb];
        tblock = sh.first_tri;
    } else {
        vblock = a.bsum[2 * (uint64_t)gb];
        tblock = a.bsum[2 * (uint64_t)gb + 1];
    }
#pragma unroll
    for (int i = 0; i < kTab; ++i) sh.tab[tid + i * kThreads] = tb[i];
    if (tid < 3)
        sh.stride[tid] = 4 * (tid == 0 ? 1ull : (uint64_t)g.nx * (tid == 2 ? (uint32_t)g.ny : 1u));
    __syncthreads();
    if (!wave_live) return;
    uint64_t v_off = 0;
    if constexpr (!kSelf) {
        // vertex numbers that do not fit 32 bits: nothing of the grid is written
        if (a.res[si].ovf) return;
        v_off = a.res[si].v_off;
    }
    first.x = (uint32_t)__builtin_amdgcn_readfirstlane((int)first.x);
    first.y = (uint32_t)__builtin_amdgcn_readfirstlane((int)first.y);
    const uint64_t vout = vblock + (first.x & 0xffffu);  // the wave's first vertex
    const uint64_t tout = tblock + first.y;              // and triangle
    // Vertices and triangles are stored 64 at a time on line boundaries: the
    // wave's records are counted from the boundary at or before its first
    // one, `vskip` and `tskip` records earlier.
    const uint32_t vskip = past_line(a.vertices + 3 * vout);
    const uint32_t tskip = past_line(a.triangles + 3 * tout);
    char *const vp = (char *)(a.vertices + 3 * vout) - 12 * vskip;
    char *tp = (char *)(a.triangles + 3 * tout) - 12 * tskip;
    const uint32_t vlimit = record_limit(a.vcap, vout, vskip);
    uint32_t tlimit = record_limit(a.tcap, tout, tskip);
    const uint32_t vid0 = (uint32_t)(vout - v_off) - vskip;  // number of record 0
    uint32_t vnext = vskip, vdone = 0;                       // vertices listed, fetched
    const float *field = a.field + s.field_off + (uint64_t)row0 * (uint32_t)g.nx;
    EmitWave &w = sh.w[wave];
    char *const vid = (char *)w.vid + 4 * lane;

    // in VGPRs: an instruction with a scalar operand takes twice as long
    Frame fr = {s.iso, s.ox, s.oy, s.oz, s.sx, s.sy, s.sz};
    asm volatile("" : "+v"(fr.iso), "+v"(fr.ox), "+v"(fr.oy), "+v"(fr.oz));
    asm volatile("" : "+v"(fr.sx), "+v"(fr.sy), "+v"(fr.sz));
    uint32_t lane12 = 12 * lane;
    asm volatile("" : "+v"(lane12));

    // 64 edges from record `from` on (some listed): ring entries, owner data
    // and field values; lanes without a listed edge repeat the nearest one
    struct Flight {
        uint32_t en, x, yz;
        float f0, f1;
    };
    const auto fetch = [&](uint32_t from) {
        Flight t;
        t.en = w.ring[max(min(from + lane, vnext - 1), vskip) % kRing];
        const int jj = (int)(t.en & 0xfcu);
        const uint64_t step = sh.stride[t.en & 3u];
        const uint32_t o = (uint32_t)__builtin_amdgcn_ds_bpermute(jj, (int)off) + (t.en >> 8);
        t.yz = (uint32_t)__builtin_amdgcn_ds_bpermute(jj, (int)yz);
        t.x = (uint32_t)__builtin_amdgcn_ds_bpermute(jj, (int)xh) + (t.en >> 8);
        const char *p = (const char *)(field + o);
        t.f0 = *(const float *)p;
        t.f1 = *(const float *)(p + step);
        return t;
    };
    const auto write = [&](const Flight &t, uint32_t from, uint32_t to) {
        const V3 v = edge_vertex(fr, (float)t.x, (float)(t.yz & 0xffffu), (float)(t.yz >> 16),
                                 t.en & 3u, t.f0, t.f1);
        const uint32_t i = from + lane;
        if (i >= vskip && i < min(to, vlimit)) store_nt((float *)(vp + (12 * from + lane12)), v);
    };

    // the cells (and points with an edge but no cell) in canonical order
    const uint32_t ntodo = (uint32_t)__popc(todo);
    const uint32_t incl = wave_scan_incl(ntodo);
    const uint32_t total = readlane32(incl, 63);
    uint32_t next = incl - ntodo;
    // triangles left over by the last step: records [0, kept) in the lanes
    T3 rec = {0, 0, 0};
    uint32_t kept = tskip, tlow = tskip;

    for (uint32_t e0 = 0; e0 < total; e0 += 64) {
        if (e0 % kCellCap == 0) {
            uint16_t *to = w.list + (next - e0);
            for (; todo && next < e0 + kCellCap; todo &= todo - 1, ++next)
                *to++ = (uint16_t)(4 * lane | (uint32_t)__builtin_ctz(todo) << 8);
            wave_sync();
        }
        const bool on = e0 + lane < total;
        const uint32_t ent = w.list[min(e0 + lane, total - 1) % kCellCap];
        const bool ready = vnext - vdone >= 64;
        Flight fl = {0, 0, 0, 0.f, 0.f};
        if (ready) fl = fetch(vdone);
        const int j = (int)(ent & 0xfcu);
        const uint32_t x = ent >> 8;
        const auto at = [&](uint32_t v) {
            return (uint32_t)__builtin_amdgcn_ds_bpermute(j, (int)v);
        };
        const uint32_t c = at(cy);
        const uint32_t ga = at(wa), gB = at(wb), gc_ = at(wc), gd = at(wd);
        const uint32_t ge = at(we), gf = at(wf), gg = at(wg), gh = at(wh);
        const uint32_t p1 = at(vb1), p2 = at(vb2), p3 = at(vb3);
        // signs at x, x+1 (and x+2) of the four rows, at x (and x+1) past them
        const uint32_t A = __builtin_amdgcn_alignbit(c, ga, x);
        const uint32_t B = __builtin_amdgcn_alignbit(c >> 2, gB, x);
        const uint32_t C = __builtin_amdgcn_alignbit(c >> 4, gc_, x);
        const uint32_t D = __builtin_amdgcn_alignbit(c >> 6, gd, x);
        const uint32_t E = __builtin_amdgcn_alignbit(c >> 7, ge, x);
        const uint32_t G = gg >> x;
        const uint32_t corners =
            (((D << 2 | (C & 3u)) << 2 | (B & 3u)) << 2 | (A & 3u)) & 0xffu;
        const bool cell = on && x < c >> 16;
        const uint2 t01 = *(const uint2 *)(sh.tab + 2 * corners);
        const uint32_t nt = cell ? (t01.x & 3u) | (t01.y & 3u) << 2 : 0u;
        // row (y, z): edges of points x and x+1
        const uint32_t xa = A ^ A >> 1, ya = A ^ B, za = A ^ C;
        const uint32_t x0 = on ? xa & 1u : 0u, y0 = on ? ya & 1u : 0u, z0 = on ? za & 1u : 0u;
        const uint32_t c0 = x0 + y0 + z0;
        const uint32_t mine2 = c0 | nt << 16;
        const uint32_t inc2 = wave_scan_incl(mine2), tot2 = readlane32(inc2, 63);
        const uint32_t ex2 = inc2 - mine2;
        const uint32_t ttot = tot2 >> 16;
        uint32_t tpos = ex2 >> 16;
        const uint32_t rel = vnext + (ex2 & 0xffffu);
        const auto id = [&](int e, uint32_t v) { *(uint32_t *)(vid + 4 * kIdStride * e) = v; };
        {
            const uint32_t p = vid0 + rel, px = p + x0, py = px + y0, q = py + z0;
            const uint32_t qx = q + (xa >> 1 & 1u);
            id(0, p);
            id(3, px);
            id(8, py);
            id(1, qx);
            id(9, qx + (ya >> 1 & 1u));
            if (c0) {
                // its edges in order; a lane writes three entries, the
                // last first, and what is not its own is overwritten by
                // the lane that it belongs to
                w.ring[(rel + 2) % kRing] = (uint16_t)(ent + 2);
                in_order();
                w.ring[(rel + 1) % kRing] = (uint16_t)(ent + 2 - (x0 & y0));
                in_order();
                w.ring[rel % kRing] = (uint16_t)(ent + ((2 - y0) & (x0 - 1)));
            }
        }
        const uint32_t low = (1u << x) - 1u;  // points before x in the half
        {                                     // row (y+1, z)
            const uint32_t xb = B ^ B >> 1, yb = B ^ E, zb = B ^ D;
            const uint32_t s_b = __builtin_amdgcn_alignbit(c >> 2, gB, 1);
            const uint32_t p = p1 + __popc((gB ^ s_b) & low) + __popc((gB ^ ge) & low) +
                               __popc((gB ^ gd) & low);
            const uint32_t q = p + (xb & 1u) + (yb & 1u);
            id(2, p);
            id(11, q);
            id(10, q + (zb & 1u) + (xb >> 1 & 1u) + (yb >> 1 & 1u));
        }
        {  // row (y, z+1)
            const uint32_t xc = C ^ C >> 1, yc = C ^ D, zc = C ^ G;
            const uint32_t s_c = __builtin_amdgcn_alignbit(c >> 4, gc_, 1);
            const uint32_t p = p2 + __popc((gc_ ^ s_c) & low) + __popc((gc_ ^ gd) & low) +
                               __popc((gc_ ^ gg) & low);
            const uint32_t q = p + (xc & 1u);
            id(4, p);
            id(7, q);
            id(5, q + (yc & 1u) + (zc & 1u) + (xc >> 1 & 1u));
        }
        {  // row (y+1, z+1)
            const uint32_t s_d = __builtin_amdgcn_alignbit(c >> 6, gd, 1);
            id(6, p3 + __popc((gd ^ s_d) & low) + __popc((gd ^ gf) & low) +
                      __popc((gd ^ gh) & low));
        }
        // the step's triangles in order, the same way
        const uint32_t me = lane * 0x00401004u;
        if (nt) {
            uint32_t *own = w.own + tpos;
            if (__any(nt > 2)) {
                const uint2 t23 = *(const uint2 *)(sh.tab + 512 + 2 * corners);
                if (__any(nt > 4)) own[4] = sh.tab[1024 + corners] + me;
                in_order();
                own[3] = t23.y + me;
                in_order();
                own[2] = t23.x + me;
                in_order();
            }
            own[1] = t01.y + me;
            in_order();
            own[0] = t01.x + me;
        }
        vnext += tot2 & 0xffffu;
        wave_sync();
        // the edges whose loads were issued at the top of the step, before
        // the triangles' stores (a wait for loads waits for stores as well)
        if (ready) {
            write(fl, vdone, vdone + 64);
            vdone += 64;
        }
        // triangles: kept ones and this step's, 64 records per store
        const uint32_t avail = kept + ttot;
        const char *ids = (const char *)w.vid;
        for (uint32_t at = 0;; at += 64) {
            const uint32_t i = at + lane;
            if (i >= kept && i < avail) {
                const uint32_t q = w.own[i - kept];
                rec.a = *(const uint32_t *)(ids + (q & 0xffcu));
                rec.b = *(const uint32_t *)(ids + (q >> 10 & 0xffcu));
                rec.c = *(const uint32_t *)(ids + (q >> 20 & 0xffcu));
            }
            if (at + 64 > avail) break;
            if (lane >= tlow && lane < tlimit) store_nt((uint32_t *)(tp + lane12), rec);
            tp += 768;
            tlimit -= min(tlimit, 64u);
            tlow = 0;
        }
        kept = avail % 64;
        while (vnext - vdone >= 128) {
            write(fetch(vdone), vdone, vdone + 64);
            vdone += 64;
        }
        wave_sync();
    }
    if (lane >= tlow && lane < min(kept, tlimit)) store_nt((uint32_t *)(tp + lane12), rec);
    // at most 127 edges are left: both fetches before the first store
    if (vnext - vdone > 64) {
        const Flight f = fetch(vdone), l = fetch(vdone + 64);
        write(f, vdone, vnext);
        write(l, vdone + 64, vnext);
    } else if (max(vdone, vskip) < vnext) {
        write(fetch(vdone), vdone, vnext);
    }
}

}  // namespace

namespace {
// Words per wave of the emission for a launch of nb blocks, as a logarithm.
// The chip holds 5120 waves of it: a launch gets that many, in shorter chunks
// (a wave works through its cells 64 at a time), before the chunks grow to 32
// words, which costs least per cell.
// 128 blocks (128^3): 16.1 us in chunks of 8 words, 17.3 of 16; 422 blocks:
// 37.6, 35.6, 35.6 (32 words); 1.7 k blocks (16 served grids): 119.5 of 16, 126 of 32.
uint32_t words_per_wave_log2(uint64_t nb) { return nb >= 4096 ? 5 : (nb >= 256 ? 4 : 3); }

// Blocks of a run (run_order), as a logarithm: about a plane, with at least 8
// runs per XCD.  512^3 with a sphere, count to emission: 177 us with the
// workgroups mixed over the XCDs, 148 in runs of a plane, 144 of two, 149 of
// four; 1024^3 full of surface 2883, 2904, 2947, 3028; 640^3 294, 292, 293, 300.
uint32_t run_log2(uint64_t nb, uint64_t plane_blocks) {
    uint32_t lr = 0;
    while (lr < 20 && (1ull << lr) < plane_blocks) ++lr;
    while (lr > 0 && (64ull << lr) > nb) --lr;
    return lr;
}

// The order of the emission's workgroups (EmitArgs::lr).  Small launches gain
// nothing from runs: over 40 grids of 128 to 5488 blocks the two orders were within
// 2 % of each other (most often within 1 %), but for grids whose surface leaves
// part of the planes empty: 272^3 less all but a sphere (1445 blocks) 47.7 us
// mixed and 51.2 in runs, 340^3 (2710 blocks) 94.9 and 75.3, 192^3 (432) 23.9 and 22.4.
// 1536 is a line between the first two; where exactly it lies matters little.
uint32_t emit_order(uint64_t nb, uint64_t plane_blocks, uint32_t lw) {
    return nb < 1536 ? kMixed : run_log2(nb, plane_blocks) + 6 - lw;
}

template <class Src, bool kSelf>
int launch_emit(const Src &src, const EmitArgs &a, uint64_t nb, hipStream_t stream) {
    const uint64_t wgs = nb << (6 - a.lw);
    GC_ARG(wgs <= 0xffffffffull, "grid too large");
    hipLaunchKernelGGL((emit_kernel<Src, kSelf>), dim3((unsigned)wgs), dim3(64 * kEmitWaves), 0,
                       stream, src, a);
    GC_CHECK_LAUNCH();
    return GPUCAD_OK;
}
}  // namespace

// Enqueues the whole one-grid extraction on `stream` given a workspace.
int enqueue_extract(const gc_extract_args *a, hipStream_t stream) {
    GC_ARG(a, "args is NULL");
    GC_ARG(a->field, "field is NULL");
    GC_ARG(a->nx >= 2 && a->ny >= 2 && a->nz >= 2, "grid must have >= 2 points per axis");
    GC_ARG(a->ny < 65536 && a->nz < 65536, "ny and nz must be < 65536");
    GC_ARG(a->normals == nullptr, "per-vertex normals are not supported by this build");
    GC_ARG(a->vertices || a->vert_capacity == 0, "vertices is NULL");
    GC_ARG(a->triangles || a->tri_capacity == 0, "triangles is NULL");
    const ExtractLayout L = layout(a->nx, a->ny, a->nz);
    GC_ARG(a->workspace && a->workspace_bytes >= L.bytes,
           "workspace too small (%llu < %llu bytes)", (unsigned long long)a->workspace_bytes,
           (unsigned long long)L.bytes);
    GC_ARG(L.words < 0xffffffffull && a->nx <= 65536, "grid too large");
    const DeviceTables *tabs = nullptr;
    int st = device_tables(&tabs);
    if (st) return st;
    char *ws = (char *)a->workspace;
    OneGrid one;
    Seg &s = one.s;
    std::memset(&s, 0, sizeof(s));
    s.g = make_grid(a->nx, a->ny, a->nz);
    s.iso = a->iso;
    s.ox = a->origin.x;
    s.oy = a->origin.y;
    s.oz = a->origin.z;
    s.sx = a->spacing.x;
    s.sy = a->spacing.y;
    s.sz = a->spacing.z;
    const uint64_t *signs = a->signs;
    if (!signs) {
        GC_ARG((a->nz + kSignZ - 1) / kSignZ <= 65535 && (a->ny + 3) / 4 <= 65535,
               "grid too large");
        uint64_t *sw = (uint64_t *)(ws + L.signs_off);
        dim3 grid(s.g.W, (a->ny + 3) / 4, (a->nz + kSignZ - 1) / kSignZ);
        hipLaunchKernelGGL(signs_kernel, grid, dim3(256), 0, stream, a->field, sw, a->nx, a->ny,
                           a->nz, s.g.W, a->iso);
        GC_CHECK_LAUNCH();
        signs = sw;
    }
    uint2 *base = (uint2 *)(ws + L.base_off);
    uint32_t *live = (uint32_t *)(ws + L.live_off);
    const uint64_t plane_blocks = ((uint64_t)s.g.W * a->ny + kBlock - 1) / kBlock;
    uint64_t *bsum = (uint64_t *)(ws + L.bsum_off);
    uint64_t *ctl = (uint64_t *)(ws + L.ctl_off);
    SegResult *res = (SegResult *)(ws + L.res_off);
    hipLaunchKernelGGL(count_kernel<OneGrid>, dim3((unsigned)L.nb), dim3(kBlock), 0, stream, one,
                       CountArgs{signs, live, bsum, base, run_log2(L.nb, plane_blocks)});
    GC_CHECK_LAUNCH();
    const bool self = L.nb <= (uint64_t)kSelfBlocks;
    if (!self) {
        hipLaunchKernelGGL(scan_blocks_kernel, dim3(1), dim3(1024), 0, stream, bsum, L.nb, ctl,
                           a->d_counts, (const Seg *)nullptr, 1u, res);
        GC_CHECK_LAUNCH();
    }
    const uint32_t lw = words_per_wave_log2(L.nb);
    const EmitArgs ea = {a->field, signs, base, live, bsum, res, tabs->emit, a->vertices,
                         a->vertices ? a->vert_capacity : 0, a->triangles,
                         a->triangles ? a->tri_capacity : 0, lw, emit_order(L.nb, plane_blocks, lw),
                         (uint32_t)L.nb, ctl, a->d_counts};
    if (a->emit_event) GC_HIP(hipEventRecord((hipEvent_t)a->emit_event, stream));
    return self ? launch_emit<OneGrid, true>(one, ea, L.nb, stream)
                : launch_emit<OneGrid, false>(one, ea, L.nb, stream);
}

int enqueue_extract_batch(const BatchExtract &b, int phases, hipStream_t stream) {
    GC_ARG(b.nseg > 0 && b.nb > 0 && b.segs && b.blk2seg, "empty batch");
    const uint32_t lw = words_per_wave_log2(b.nb);
    const DeviceTables *tabs = nullptr;
    int st = device_tables(&tabs);
    if (st) return st;
    const ManyGrids src = {b.segs, b.blk2seg};
    const uint64_t plane_blocks = 4;  // (a plane of 128..256 points; longer runs: no gain)
    if (phases & EXTRACT_COUNT) {
        hipLaunchKernelGGL(count_kernel<ManyGrids>, dim3(b.nb), dim3(kBlock), 0, stream, src,
                           CountArgs{b.signs, b.live, b.bsum, (uint2 *)b.base,
                                     run_log2(b.nb, plane_blocks)});
        GC_CHECK_LAUNCH();
        hipLaunchKernelGGL(scan_blocks_kernel, dim3(1), dim3(1024), 0, stream, b.bsum,
                           (uint64_t)b.nb, b.ctl, (uint64_t *)nullptr, b.segs, b.nseg, b.res);
        GC_CHECK_LAUNCH();
    }
    if (phases & EXTRACT_EMIT) {
        const EmitArgs ea = {b.fields, b.signs, (const uint2 *)b.base, b.live, b.bsum, b.res,
                             tabs->emit, b.vertices, b.vertices ? b.vcap : 0, b.triangles,
                             b.triangles ? b.tcap : 0, lw, emit_order(b.nb, plane_blocks, lw), b.nb,
                             nullptr, nullptr};
        if ((st = launch_emit<ManyGrids, false>(src, ea, b.nb, stream))) return st;
    }
    return GPUCAD_OK;
}

}  // namespace gc

extern "C" {

uint64_t gpucad_extract_workspace_bytes(int32_t nx, int32_t ny, int32_t nz) {
    if (nx < 2 || ny < 2 || nz < 2) return 0;
    return gc::layout(nx, ny, nz).bytes;
}

int gpucad_extract(const gc_extract_args *a, gc_mesh_counts *counts, void *stream) {
    gc::clear_error();
    hipStream_t s = gc::as_stream(stream);
    int st = gc::enqueue_extract(a, s);
    if (st) return st;
    if (!counts) return GPUCAD_OK;
    GC_HIP(hipStreamSynchronize(s));
    uint64_t ctl[3];
    const char *ws = (const char *)a->workspace;
    GC_HIP(hipMemcpy(ctl, ws + gc::layout(a->nx, a->ny, a->nz).ctl_off, sizeof(ctl),
                     hipMemcpyDeviceToHost));
    counts->n_vertices = ctl[gc::CTL_NV];
    counts->n_triangles = ctl[gc::CTL_NT];
    if (ctl[gc::CTL_OVF])
        return gc::fail(GPUCAD_E_OVERFLOW, "%llu vertices exceed 32-bit indices",
                        (unsigned long long)ctl[gc::CTL_NV]);
    if (ctl[gc::CTL_NV] > a->vert_capacity || ctl[gc::CTL_NT] > a->tri_capacity)
        return gc::fail(GPUCAD_E_OVERFLOW,
                        "mesh needs %llu vertices / %llu triangles, capacity %llu / %llu",
                        (unsigned long long)ctl[gc::CTL_NV], (unsigned long long)ctl[gc::CTL_NT],
                        (unsigned long long)a->vert_capacity, (unsigned long long)a->tri_capacity);
    return GPUCAD_OK;
}

}  // extern "C"
