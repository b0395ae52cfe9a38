// rvs_synth.hip -- triangle binning, tile rasterisation and blending for gfx950.
//
// Reference semantics: detail::transform_trianglesMethod (rvs/src/transform.cpp:148-181)
// visits source quads in raster order and folds every covered target pixel
// sequentially: a candidate (depth d, triangle validity v) replaces the state
// (D, V) when fl(fl(fl(r*r)*r)*V) < v with r = fl(d/D), strict, so ties keep the
// earlier triangle.  Mathematically that is the argmax of v/d^3 with the lowest
// traversal index on ties, but the float test is not transitive for
// near-equal scores.  This file computes it for a batch of target views that
// share one set of resident sources:
//   0. k_bin_cull: binning work items (view, source, 64x4 source quads) whose
//      source points all lie behind a perspective view or beyond one side of
//      its image are dropped (bounding boxes of the unprojected points come
//      from k_src_bounds and are tested with error margins); the rest form a
//      work list.
//   1. k_bin (counting pass, scan, fill pass): every surviving source quad
//      is appended to the 16x16 or 32x32 target tiles its triangles' narrowed
//      (reference-exact) bounding boxes touch; the counting pass keeps each
//      work item's vertex block and validities for the raster.
//   2. k_raster: one 256- or 1024-thread block per target tile, four sources per
//      phase (one phase, 8 waves per SIMD, for launch sets of up to four
//      sources).  Every covered pixel takes an LDS 64-bit atomicMax, key1 = max
//      of (score bits << 32 | candidate id), and a 32-bit one, key2 = max
//      score over the candidates that are not the maximum (the loser of each
//      key1 update).  A pixel whose runner-up scores within 2^-18 of the
//      winner, or that saw a candidate with non-finite or extreme values (key2
//      = all ones), is deferred; where cameras are aligned and ties are the
//      rule, a second pass settles those between candidates of the very same
//      depth and validity (k_raster's SETTLE).  Every other pixel
//      provably ends the sequential fold on the argmax (the float test errs
//      by less than 2^-21 relative), so its winner is re-evaluated -- from
//      the kept vertices and validity of the work item the coverage pass
//      left in LDS -- and blended.
//   3. k_fallback_src / k_fallback_blend / k_fallback: deferred pixels replay
//      the reference fold literally, in traversal order (per-pixel candidate
//      lists gathered in LDS, or a sort of the tile's bins when a list
//      overflows), each source of a tile in its own block and then blended,
//      or (beyond the workspace for that) a block per tile folding its
//      sources in turn.
// Blending across sources (BlendedViewSimple::blendBasicMode) runs per pixel in
// registers inside the same block, in InputCameraNames order.
#include <hip/hip_runtime.h>

#include <cstring>

#include "rvs_kernels.h"

namespace rvs_k {

using namespace rvs_dev;

// Descriptor uploads travel as kernel arguments, so a launch set stays
// stream-ordered and capturable in a graph (no host-side memcpy).  The same
// launch clears the set's counters: a small view is bound by its launches, 4-5
// us each, and three clears and two uploads were five of them.
constexpr uint32_t kBlobBytes = 3584;
struct Blob {
    uint32_t n;
    uint8_t bytes[kBlobBytes];
};

__global__ void __launch_bounds__(256) k_begin(Blob b, uint8_t* dst, uint32_t* zero, size_t words) {
    if (blockIdx.x == 0)
        for (uint32_t i = threadIdx.x; i < b.n; i += blockDim.x) dst[i] = b.bytes[i];
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += (size_t)gridDim.x * blockDim.x)
        zero[i] = 0u;
}

hipError_t launch_begin(const void* host, size_t bytes, void* dst, uint32_t* zero, size_t words, hipStream_t s) {
    const uint8_t* src = (const uint8_t*)host;
    for (size_t off = 0; off < bytes; off += kBlobBytes) {
        Blob b;
        b.n = (uint32_t)((bytes - off) < (size_t)kBlobBytes ? (bytes - off) : (size_t)kBlobBytes);
        std::memcpy(b.bytes, src + off, b.n);
        const size_t w = off == 0 ? words : 0, blocks = (w + 2047) / 2048;
        hipLaunchKernelGGL(k_begin, dim3((unsigned)(blocks < 1 ? 1 : blocks < 8192 ? blocks : 8192)), dim3(256), 0, s, b,
                           (uint8_t*)dst + off, zero, w);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// View owning global tile T (views are sorted by tile_base).
__device__ inline int find_view(const ViewDesc* views, int nviews, uint32_t T) {
    int lo = 0, hi = nviews - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (views[mid].tile_base <= T) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Tile index of block b: each XCD (blocks are dealt round-robin over 8 XCDs)
// gets a contiguous band of tiles, so neighbouring tiles share that XCD's L2.
__device__ inline uint32_t tile_of_block(uint32_t b, uint32_t ntiles) {
    const uint32_t per = (ntiles + 7) / 8;
    return (b % 8) * per + b / 8;
}

// Bin of source s in global tile t.  Bins of one source are adjacent along a
// tile row, so that the atomics of a quad across many tiles share cache lines.
__device__ inline size_t bin_index(const BatchDims& d, uint32_t t, uint32_t s) { return (size_t)s * d.ntiles + t; }

// ------------------------------------------------------------------ quads

// vertex() of the N corners (i + di, j + dj), bit k of ROWS / COLS being di /
// dj of corner k, one after the other (not unrolled: the evaluation is large
// and, where a kept window is the rule, rare).
template <int N, class G>
__device__ inline void eval_corners(const G& g, int i, int j, uint32_t rows, uint32_t cols, float3 (&v)[N], bool* und) {
#pragma unroll 1
    for (int k = 0; k < N; ++k) {
        const float3 x = vertex(g, i + (int)((rows >> k) & 1u), j + (int)((cols >> k) & 1u), und);
#pragma unroll
        for (int m = 0; m < N; ++m)
            if (m == k) v[m] = x;
    }
}

// The (up to four) triangles of source quad (i, j), with the reference's
// vertex gating (transform.cpp:161-176).  alive bit k set = colorize_triangle
// is called for slot k and gets past its early returns.
struct Quad {
    Tri t[4];
    uint32_t alive;
    uint32_t prol;      // bit k: prol flag of slot k (transform.cpp:121-123)
};

// All three finite: times 0 anything else gives a NaN (a plain sum of finite
// numbers can overflow).
__device__ inline bool finite3(float3 v) {
    return __builtin_fmaf(v.z, 0.f, __builtin_fmaf(v.y, 0.f, v.x * 0.f)) == 0.f;
}

__device__ inline void quad_add(Quad& Q, int slot, float3 a, float3 b, float3 c, int out_w, int out_h, float rescale,
                                bool validity) {
    Tri T;
    const bool ok = validity ? tri_setup(T, a, b, c, out_w, out_h, rescale) : tri_setup_geom(T, a, b, c, out_w, out_h);
    Q.t[slot] = T;
    if (!ok) return;
    Q.alive |= 1u << slot;
    if ((a.z > 0.f) || (b.z > 0.f) || (c.z > 0.f)) Q.prol |= 1u << slot;
}

// validity = false leaves t[k].tv at 0 (binning needs only which triangles
// survive and their bounding boxes).
template <class G, class VF>
__device__ inline void quad_build(Quad& Q, const G& g, int i, int j, VF vtx, int out_w, int out_h,
                                  bool validity = true) {
    Q.alive = 0; Q.prol = 0;
    Q.t[0].tv = 0.f; Q.t[1].tv = 0.f;
    const float3 v00 = vtx(i, j), v01 = vtx(i, j + 1), v10 = vtx(i + 1, j), v11 = vtx(i + 1, j + 1);
    if (!(v01.z > 0.f && v10.z > 0.f && v01.x > 0.f && v10.x > 0.f)) return;
    if (v00.z > 0.f && v00.x > 0.f) quad_add(Q, 0, v00, v01, v10, out_w, out_h, g.rescale, validity);
    if (v11.z > 0.f && v11.x > 0.f) quad_add(Q, 1, v11, v10, v01, out_w, out_h, g.rescale, validity);
    if (g.wrap && j == 0) {
        const float3 l0 = vtx(i, g.sw - 1), l1 = vtx(i + 1, g.sw - 1);
        quad_add(Q, 2, l0, v00, l1, out_w, out_h, g.rescale, validity);
        quad_add(Q, 3, v10, l1, v00, out_w, out_h, g.rescale, validity);
    }
}

// Tile range [tx0, tx1] x [ty0, ty1] of the bounding boxes, narrowed to the
// pixels each can cover (tri_tight), of the triangles of source quad (i, j)
// that survive the gating and colorize_triangle's early returns (the union
// quad_build + quad_tiles compute), one triangle at a time; with tv, also the
// validities of T1 and T2 (0 when not alive or left undecided by the fast
// path).  False when no triangle can cover a pixel.
template <class G>
__device__ inline bool quad_range_tv(const G& g, int i, int j, float3 v00, float3 v01, float3 v10, float3 v11, int out_w,
                                     int out_h, int shift, int& tx0, int& tx1, int& ty0, int& ty1, float2* tv) {
    if (tv) *tv = make_float2(0.f, 0.f);
    if (!(v01.z > 0.f && v10.z > 0.f && v01.x > 0.f && v10.x > 0.f)) return false;
    int xmin = INT_MAX, xmax = INT_MIN, ymin = INT_MAX, ymax = INT_MIN;
    auto one = [&](float3 a, float3 b, float3 c, float* tvo) {
        Tri T;
        tri_load(T, a, b, c);
        int xa, xb, ya, yb;
        // a triangle that can cover no pixel is never rasterised
        if (!tri_box(T, out_w, out_h, 0, out_w - 1, 0, out_h - 1, xa, xb, ya, yb)) return;
        xmin = min(xmin, xa); xmax = max(xmax, xb);
        ymin = min(ymin, ya); ymax = max(ymax, yb);
        // fast path only: an undecided validity stays 0 (unknown), and the
        // raster then defers the pixels that depend on it
        if (tvo && !tri_validity_fast(T, g.rescale, *tvo)) *tvo = 0.f;
    };
    if (v00.z > 0.f && v00.x > 0.f) one(v00, v01, v10, tv ? &tv->x : nullptr);
    if (v11.z > 0.f && v11.x > 0.f) one(v11, v10, v01, tv ? &tv->y : nullptr);
    if (g.wrap && j == 0) {
        float3 l[2];   // (i, sw - 1), (i + 1, sw - 1)
        eval_corners<2>(g, i, g.sw - 1, 2u, 0u, l, nullptr);
#pragma unroll 1
        for (int k = 0; k < 2; ++k) one(k ? v10 : l[0], k ? l[1] : v00, k ? v00 : l[1], nullptr);
    }
    if (xmin > xmax) return false;
    tx0 = xmin >> shift; tx1 = xmax >> shift; ty0 = ymin >> shift; ty1 = ymax >> shift;   // boxes start at >= 0
    return true;
}

// Calls fn(slot, triangle, prol) for every triangle of source quad (i, j)
// that gets past the vertex gating and colorize_triangle's early returns, in
// slot order (the quad_build gating, one triangle at a time); vertices come
// from vtx (exact), and the triangle's validity is left 0 for fn to evaluate
// (tri_validity) when it needs it.
template <class G, class VF, class F>
__device__ inline void quad_tris(const G& g, int i, int j, VF vtx, int out_w, int out_h, F fn) {
    const float3 v00 = vtx(i, j), v01 = vtx(i, j + 1), v10 = vtx(i + 1, j);
    const float3 v11 = vtx(i + 1, j + 1);
    if (!(v01.z > 0.f && v10.z > 0.f && v01.x > 0.f && v10.x > 0.f)) return;
    auto one = [&](int slot, float3 a, float3 b, float3 c) {
        Tri T;
        if (tri_setup_geom(T, a, b, c, out_w, out_h)) fn(slot, T, (a.z > 0.f) || (b.z > 0.f) || (c.z > 0.f));
    };
    if (v00.z > 0.f && v00.x > 0.f) one(0, v00, v01, v10);
    if (v11.z > 0.f && v11.x > 0.f) one(1, v11, v10, v01);
    if (g.wrap && j == 0) {
        const float3 l0 = vtx(i, g.sw - 1), l1 = vtx(i + 1, g.sw - 1);
        one(2, l0, v00, l1);
        one(3, v10, l1, v00);
    }
}

// Bins hold source quads as (row << 16) | column: ascending order of these
// codes is the reference's traversal order (rows, then columns).
__device__ inline void unpack_ij(uint32_t ij, int& i, int& j) {
    i = (int)(ij >> 16);
    j = (int)(ij & 0xffffu);
}

// ------------------------------------------------------------ culling

// Minimum (MIN) or maximum over the wave, in its last lane: moves between
// lanes as DPP operands instead of through LDS.
template <bool MIN, int CTRL, int ROWS>
__device__ inline float dpp_step(float v) {
    const int m = __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, ROWS, 0xf, false);
    return MIN ? min3f(v, v, __int_as_float(m)) : max3f(v, v, __int_as_float(m));
}
template <bool MIN>
__device__ inline float wave_last(float v) {
    v = dpp_step<MIN, 0x111, 0xf>(v);   // row_shr:1
    v = dpp_step<MIN, 0x112, 0xf>(v);   // row_shr:2
    v = dpp_step<MIN, 0x114, 0xf>(v);   // row_shr:4
    v = dpp_step<MIN, 0x118, 0xf>(v);   // row_shr:8
    v = dpp_step<MIN, 0x142, 0xa>(v);   // row_bcast:15 into rows 1, 3
    return dpp_step<MIN, 0x143, 0xc>(v);   // row_bcast:31 into rows 2, 3
}

// Culling table of one source: per binning block (kBinQY x kBinQX quads), the
// bounding box (source camera frame) of the finite unprojected points of its
// vertex window (kBinQY+1 rows x kBinQX+1 columns) as min x, y, z, max x, y, z;
// no finite point -> min +inf, max -inf.  One wave per block; bound by VALU
// issue: 4096x2048 equirectangular 36 -> 30 us with the points in
// pairs, the columns' tables loaded once and DPP reductions.
__global__ void __launch_bounds__(256) k_src_bounds(PairGeom g, int bins_x, int bins_y, float* out) {
    const int lane = threadIdx.x & 63;
    const int item = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (item >= bins_x * bins_y) return;   // whole wave
    const int i0 = (item / bins_x) * kBinQY, j0 = (item % bins_x) * kBinQX;
    const float inf = __builtin_inff();
    float lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf};
    // points in pairs; the minima pass over NaNs, and a point with any
    // non-finite coordinate becomes NaNs
    auto add = [&](float3 p, float3 q) {
        const float n = __builtin_nanf("");
        const bool a = finite3(p), b = finite3(q);
        const float ps[3] = {a ? p.x : n, a ? p.y : n, a ? p.z : n}, qs[3] = {b ? q.x : n, b ? q.y : n, b ? q.z : n};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            lo[c] = min3f(lo[c], ps[c], qs[c]);
            hi[c] = max3f(hi[c], ps[c], qs[c]);
        }
    };
    const float none = __builtin_nanf("");
    const float3 no_point = make_float3(none, none, none);
    // a lane per column, the rows' depths loaded together; then the last column
    const int j = j0 + lane;
    float3 p[kBinQY + 2];
#pragma unroll
    for (int r = 0; r < kBinQY + 2; ++r) p[r] = no_point;
    if (j < g.sw) {
        float d[kBinQY + 1];
#pragma unroll
        for (int r = 0; r <= kBinQY; ++r) d[r] = src_depth(g, min(i0 + r, g.sh - 1), j);
#pragma unroll
        for (int r = 0; r <= kBinQY; ++r) p[r] = unproject_depth(g, min(i0 + r, g.sh - 1), j, d[r]);   // a row twice: the same box
    }
    if (lane <= kBinQY && i0 + lane < g.sh && j0 + kBinQX < g.sw)
        p[kBinQY + 1] = unproject_src(g, i0 + lane, j0 + kBinQX);
    static_assert(kBinQY == 4, "three pairs");
    add(p[0], p[1]); add(p[2], p[3]); add(p[4], p[5]);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        lo[c] = wave_last<true>(lo[c]);
        hi[c] = wave_last<false>(hi[c]);
    }
    if (lane == 63) {
        float* o = out + (size_t)item * 6;
        o[0] = lo[0]; o[1] = lo[1]; o[2] = lo[2];
        o[3] = hi[0]; o[4] = hi[1]; o[5] = hi[2];
    }
}

hipError_t launch_src_bounds(const PairGeom& g, float* out, hipStream_t s) {
    const int bx = bin_blocks_x(g.sw), by = bin_blocks_y(g.sh);
    hipLaunchKernelGGL(k_src_bounds, dim3((unsigned)((bx * by + 3) / 4)), dim3(256), 0, s, g, bx, by, out);
    return hipGetLastError();
}

// True when no triangle built from points inside box b can be alive for a
// perspective target: every point is behind the camera (X < 0), or beyond one
// image side by more than two pixels.  For X > 0 the side tests are linear in
// the point, u < -m <=> f0*Y - (p0 + m)*X > 0 (u = -f0*Y/X + p0), so their
// minimum over the box is at a corner.  A triangle is alive only if all its
// vertices have X > 0 (vertex gating), and a vertex with u' < -1 everywhere
// (or > W) gives xmin > xmax in tri_setup.  The margins cover the float error
// of the corner evaluation here and of the vertex stage (both below 1e-6 of
// the magnitudes involved); overflow or NaN never culls.
__device__ inline bool box_outside(const PairGeom& g, const float* b, int out_w, int out_h) {
    if (!(b[0] <= b[3])) return true;   // no finite point: every vertex is gated
    float X[8], Y[8], Z[8];
    float mag = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float x = (k & 1) ? b[3] : b[0], y = (k & 2) ? b[4] : b[1], z = (k & 4) ? b[5] : b[2];
        X[k] = g.R[0] * x + g.R[1] * y + g.R[2] * z + g.t[0];
        Y[k] = g.R[3] * x + g.R[4] * y + g.R[5] * z + g.t[1];
        Z[k] = g.R[6] * x + g.R[7] * y + g.R[8] * z + g.t[2];
        mag = fmaxf(mag, fabsf(x) + fabsf(y) + fabsf(z));
    }
    mag += fabsf(g.t[0]) + fabsf(g.t[1]) + fabsf(g.t[2]);
    const float e = 1e-5f * mag;
    const float f0 = -g.df0n, f1 = -g.df1n, p0 = g.dp0, p1 = g.dp1;
    const float mu = 2.f / g.sx, mv = 2.f / g.sy;                       // two output pixels
    const float ur = ((float)out_w + 2.f) / g.sx, vr = ((float)out_h + 2.f) / g.sy;
    const float tl = e * (fabsf(f0) + fabsf(p0) + mu), tr = e * (fabsf(f0) + fabsf(p0) + ur);
    const float tt = e * (fabsf(f1) + fabsf(p1) + mv), tb = e * (fabsf(f1) + fabsf(p1) + vr);
    bool behind = true, left = true, right = true, top = true, bottom = true;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        behind = behind && (X[k] < -e);
        left = left && (f0 * Y[k] - (p0 + mu) * X[k] > tl);
        right = right && (-f0 * Y[k] - (ur - p0) * X[k] > tr);
        top = top && (f1 * Z[k] - (p1 + mv) * X[k] > tt);
        bottom = bottom && (-f1 * Z[k] - (vr - p1) * X[k] > tb);
    }
    return behind || left || right || top || bottom;
}

template <class G>
__device__ inline bool item_culled(const G&, int, int, int, int) { return false; }
template <>
__device__ inline bool item_culled<PairGeom>(const PairGeom& g, int bx, int by, int out_w, int out_h) {
    if (!g.bounds || g.dst_erp || g.wrap) return false;
    return box_outside(g, g.bounds + ((size_t)by * g.bounds_bx + bx) * 6, out_w, out_h);
}

// One thread per (view, source, item): append the items that may cover the view
// to the work list (code = (view * nsrc + source) * items + item).
// One block row per (view, source) pair (blockIdx.y, striding): the pair's
// descriptor is then uniform and read with scalar loads.  Survivors are
// appended to the work list with one atomic per 1024-thread block (the waves'
// counts are combined in LDS): the list's counter is a single address, and
// same-address device atomics are serialised at the memory side.
constexpr int kCullThreads = 1024;

template <class G>
__global__ void __launch_bounds__(kCullThreads) k_bin_cull(const G* __restrict__ geoms,
                                                           const ViewDesc* __restrict__ views, BatchDims d,
                                                           RasterWS ws) {
    __shared__ uint32_t s_cnt[kCullThreads / 64];
    __shared__ uint32_t s_base;
    const uint32_t per = d.bins_x * d.bins_y;
    const uint32_t item = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t npairs = (uint32_t)d.nsrc * (uint32_t)d.nviews;
    const int lane = __lane_id(), wave = threadIdx.x >> 6;
    for (uint32_t vs = blockIdx.y; vs < npairs; vs += gridDim.y) {
        const size_t gid = (size_t)vs * per + item;
        bool keep = false;
        if (item < per) {
            const int v = (int)(vs / (uint32_t)d.nsrc);
            const G& g = geoms[vs];
            const int bx = (int)(item % d.bins_x), by = (int)(item / d.bins_x);
            if (by * kBinQY < g.sh - 1 && bx * kBinQX < g.sw - 1) keep = !item_culled(g, bx, by, views[v].w, views[v].h);
        }
        const uint64_t m = __ballot(keep);
        if (lane == 0) s_cnt[wave] = (uint32_t)__popcll(m);
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t tot = 0;
            for (int w = 0; w < kCullThreads / 64; ++w) tot += s_cnt[w];
            s_base = tot ? atomicAdd(&ws.status[4], tot) : 0u;
        }
        __syncthreads();
        uint32_t base = s_base;
        for (int w = 0; w < wave; ++w) base += s_cnt[w];
        uint32_t wi = 0xffffffffu;
        if (keep) {
            const uint64_t lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
            const uint32_t pos = base + (uint32_t)__popcll(m & lt);
            ws.work[pos] = (uint32_t)gid;
            if (pos < d.range_cap) wi = pos;
        }
        if (item < per) ws.imap[gid] = wi;
        __syncthreads();   // s_cnt / s_base free for the next pair
    }
}

// ------------------------------------------------------------------ binning
//
// Bins are compact: a counting pass (k_bin<COUNT>) finds every surviving
// quad's tile range and counts the (quad, tile) entries per (tile, source)
// bin; an exclusive scan turns the counts into bin offsets; fill passes write
// the quad codes.  For the first range_cap work items the counting pass keeps
// each quad's tile range (and the item's vertex window and triangle
// validities, for the raster) and reserves the item's places in its bins, so
// their fill pass (k_fill_kept) needs neither vertex work nor atomics on
// memory; later items re-evaluate their vertices in their fill pass
// (k_bin<FILL>) and take places through one cursor per bin, behind the reserved
// ones.  The order of a bin's entries is free: the raster's keys commute and
// the in-order replay sorts them.  When the entries exceed the list capacity
// the fill passes and the raster are skipped and the needed capacity is
// reported.
//
// Blocks first gather their entries per bin in an LDS table (a few to a few
// dozen distinct tiles per 64x4 quad block), then take one global atomic per
// bin: device-scope atomics are performed at the memory side, so their number
// and the cache lines they touch cost the wide-range scenes most of their
// binning time.
//
// The counting pass is bound by VALU issue: 0.50-0.55 T wave instructions/s of the
// 0.72 that its mix can reach (see raster_tile), the rest being waits (its waves
// wait 0.58 of their time, eight of them side by side).  Of its
// 995 us for 16 mixed views before the validity's shorter form: vertices 290,
// validities 270, boxes 200, stores of the kept state 130, tile walk 123,
// count atomics 0 (builds that skip a part).

constexpr uint32_t kRangeNone = 0xffffffffu;   // no surviving triangle
constexpr uint32_t kRangeBig = 0xfffffffeu;    // range too wide to pack: re-evaluated

__device__ inline uint32_t pack_range(int tx0, int tx1, int ty0, int ty1) {
    const int ntx = tx1 - tx0, nty = ty1 - ty0;
    if (ntx > 14 || nty > 14) return kRangeBig;
    return (uint32_t)tx0 | ((uint32_t)ty0 << 12) | ((uint32_t)ntx << 24) | ((uint32_t)nty << 28);
}

__device__ inline void unpack_range(uint32_t r, int& tx0, int& tx1, int& ty0, int& ty1) {
    tx0 = (int)(r & 0xfffu);
    ty0 = (int)((r >> 12) & 0xfffu);
    tx1 = tx0 + (int)((r >> 24) & 0xfu);
    ty1 = ty0 + (int)(r >> 28);
}

__device__ inline float3 load3(const float* p) { return make_float3(p[0], p[1], p[2]); }

// Vertex window of kept work item wi (the counting pass evaluated it with
// vertex(); the bits are the same).
__device__ inline float* kept_window(const RasterWS& ws, uint32_t wi) {
    return ws.vbuf + (size_t)wi * kItemFloats + kItemTv;
}
__device__ inline float3 kept_vertex(const float* vb, int lr, int lc) {
    return load3(vb + 3 * (lr * (kBinQX + 1) + lc));
}

// Work index of the kept work item holding quad ij of pair vs, or ~0 (always
// ~0 when kept items store no vertex windows).  KEPT: every surviving item is
// kept.  Fewer than 2^32 items, 2^14 item rows, 2^10 item columns.
static_assert(kBinQX == 64 && kBinQY == 4 && kMaxSourceSide == 65536, "item of a quad code");
template <bool KEPT = false>
__device__ inline uint32_t kept_index(const RasterWS& ws, const BatchDims& d, uint32_t vs, uint32_t ij) {
    if (!KEPT && !d.kept_geom) return 0xffffffffu;
    return ws.imap[vs * (d.bins_x * d.bins_y) + __umul24(ij >> 18, d.bins_x) + ((ij >> 6) & 0x3ffu)];
}

// Place of quad ij in a kept item: its validities (T1, T2; the counting pass
// evaluated them exactly, only alive triangles' values are meaningful) and its
// upper left vertex.
struct KeptQuad {
    const float *tv, *v;
};
__device__ inline KeptQuad kept_quad(const RasterWS& ws, uint32_t wi, uint32_t ij) {
    const float* p = ws.vbuf + (size_t)wi * kItemFloats;
    const uint32_t lr = (ij >> 16) & 3u, q = (lr << 6) | (ij & 63u);
    return {p + 2u * q, p + kItemTv + __umul24(q + lr, 3u)};
}

// Vertex window of quad ij of pair vs when its work item was kept, else null.
__device__ inline const float* kept_block(const RasterWS& ws, const BatchDims& d, uint32_t vs, uint32_t ij) {
    const uint32_t wi = kept_index(ws, d, vs, ij);
    return wi == 0xffffffffu ? nullptr : kept_window(ws, wi);
}

// Corners a, b, c of slot 0 (v00 v01 v10) or 1 (v11 v10 v01) of a kept quad.
__device__ inline void kept_corners(const float* v, int slot, float3 (&c)[3]) {
    c[0] = load3(v + (slot ? 3 * (kBinQX + 2) : 0));
    c[1] = load3(v + (slot ? 3 * (kBinQX + 1) : 3));
    c[2] = load3(v + (slot ? 3 : 3 * (kBinQX + 1)));
}

// Vertices (i, sw - 1) and (i + 1, sw - 1) of pair vs, every item being kept:
// from the window of the last quad of the row.
__device__ inline void kept_seam(const RasterWS& ws, const BatchDims& d, uint32_t vs, int i, int sw, float3 (&l)[2]) {
    const uint32_t ij = ((uint32_t)i << 16) | (uint32_t)(sw - 2);
    const float* p = kept_quad(ws, kept_index<true>(ws, d, vs, ij), ij).v + 3;
    l[0] = load3(p);
    l[1] = load3(p + 3 * (kBinQX + 1));
}

constexpr uint32_t kTableEmpty = 0xffffffffu;

// Slot of global tile t in the block's LDS table, inserting it; -1 when the
// table is full of other tiles (keys are never removed while an item runs,
// so a tile refused once stays absent and find_slot agrees).
__device__ inline int table_slot(uint32_t* keys, uint32_t t) {
    uint32_t h = (t * 2654435761u) >> 25;
    for (int probe = 0; probe < kBinTable; ++probe) {
        const uint32_t k = keys[h];
        if (k == t) return (int)h;
        if (k == kTableEmpty) {
            const uint32_t old = atomicCAS(&keys[h], kTableEmpty, t);
            if (old == kTableEmpty || old == t) return (int)h;
        }
        h = (h + 1) & (kBinTable - 1);
    }
    return -1;
}

__device__ inline int find_slot(const uint32_t* keys, uint32_t t) {
    uint32_t h = (t * 2654435761u) >> 25;
    for (int probe = 0; probe < kBinTable; ++probe) {
        const uint32_t k = keys[h];
        if (k == t) return (int)h;
        if (k == kTableEmpty) return -1;
        h = (h + 1) & (kBinTable - 1);
    }
    return -1;
}

// Block-cooperative walk over the tiles of the threads' quad ranges: entry e
// of the block's concatenated ranges goes to thread e % 256, which finds the
// owning quad by a binary search of the block-wide inclusive scan of the
// ranges' tile counts.  One quad with a wide range (a stretched triangle
// across a depth edge, a quad near an equirectangular pole) then costs every
// lane of the block a few iterations instead of holding its wave.  Ranges of
// at most kLaneTiles tiles (nearly all) are walked by their own lane, and a
// block without a wider one skips the scan.
struct RangeWalk {
    uint32_t incl[256];   // inclusive prefix of the tile counts
    uint32_t org[256];    // tx0 | ty0 << 16
    uint32_t wid[256];    // tx1 - tx0 + 1
    uint32_t wsum[4];     // wave totals
};

constexpr uint32_t kLaneTiles = 4;   // ranges up to this many tiles stay with their own lane
// Ranges above this many tiles (quads across the seam or near a pole of an
// equirectangular target, up to a whole row of tiles or more) would fill the
// table and then probe it in vain: their entries take a place each from their
// bins' cursors, a lane per tile, neighbouring tiles in neighbouring lanes.
// Below it the table saves atomics where several quads of an item share tiles.
// Counting pass plus fill, with bins of one tile adjacent and every entry
// tried in the table -> now: a 1920x1080 view beside a pole of its sources 0.60
// -> 0.19 ms, an 8192x4096 panorama of eleven with close objects 10.9 -> 4.2 ms.
constexpr uint32_t kTableTiles = 64;

// Publishes this thread's range (n = 0: none); all 256 threads call it, and
// the walk may start after the __syncthreads() that follows.
__device__ inline void range_publish(RangeWalk& W, int tid, bool on, int tx0, int tx1, int ty0, int ty1) {
    const uint32_t n = on ? (uint32_t)(tx1 - tx0 + 1) * (uint32_t)(ty1 - ty0 + 1) : 0u;
    const int lane = tid & 63, wave = tid >> 6;
    uint32_t x = n;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) W.wsum[wave] = x;
    W.org[tid] = on ? ((uint32_t)tx0 | ((uint32_t)ty0 << 16)) : 0u;
    W.wid[tid] = on ? (uint32_t)(tx1 - tx0 + 1) : 1u;
    __syncthreads();
    for (int w = 0; w < wave; ++w) x += W.wsum[w];
    W.incl[tid] = x;
}

template <class F>
__device__ inline void range_walk(const RangeWalk& W, int tid, F fn) {
    const uint32_t total = W.incl[255];
    for (uint32_t e = (uint32_t)tid; e < total; e += 256u) {
        int lo = 0, hi = 255;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (W.incl[mid] > e) hi = mid; else lo = mid + 1;
        }
        const uint32_t l = e - (lo ? W.incl[lo - 1] : 0u);
        const uint32_t o = W.org[lo], w = W.wid[lo];
        fn(lo, (int)(o & 0xffffu) + (int)(l % w), (int)(o >> 16) + (int)(l / w),
           W.incl[lo] - (lo ? W.incl[lo - 1] : 0u) <= kTableTiles);
    }
}

// The counting pass strides over all work items, the fill pass over those
// after the kept ones.
template <class G, bool FILL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) k_bin(const G* __restrict__ geoms, const ViewDesc* __restrict__ views,
                                             BatchDims d, RasterWS ws) {
    __shared__ float3 V[kBinQY + 1][kBinQX + 1];
    __shared__ uint32_t t_key[kBinTable];
    __shared__ uint32_t t_n[kBinTable];      // entries per bin
    __shared__ uint32_t t_base[kBinTable];   // fill write cursor per bin (fill pass)
    __shared__ RangeWalk walk;
    __shared__ uint32_t t_used;              // used table slots (kept items)
    const int tid = threadIdx.x;
    const uint32_t per = d.bins_x * d.bins_y;
    if (FILL && ws.status[1]) return;   // list capacity exceeded: nothing to fill
    const uint32_t nwork = ws.status[4];
    const uint64_t step = gridDim.x;
    for (uint64_t wi64 = (FILL ? d.range_cap : 0u) + blockIdx.x; wi64 < nwork; wi64 += step) {
        const uint32_t wi = (uint32_t)wi64;
        const uint32_t code = ws.work[wi];
        const uint32_t item = code % per, vs = code / per;
        const int s = (int)(vs % (uint32_t)d.nsrc), v = (int)(vs / (uint32_t)d.nsrc);
        const G& g = geoms[vs];
        const ViewDesc& vd = views[v];
        const int i0 = (int)(item / d.bins_x) * kBinQY, j0 = (int)(item % d.bins_x) * kBinQX;
        const int i = i0 + tid / kBinQX, j = j0 + tid % kBinQX;
        const bool stored = !FILL && wi < d.range_cap;   // same for the whole block
        const bool stored_geom = stored && d.kept_geom;
        if (tid < kBinTable) {
            t_key[tid] = kTableEmpty;
            t_n[tid] = 0;
        }
        bool more = false;
        int tx0 = 0, tx1 = -1, ty0 = 0, ty1 = -1;
        // a kept item also records its vertices and its quads' triangle validities for the raster
        {
            float* vb = stored_geom ? kept_window(ws, wi) : nullptr;
#pragma unroll 1
            for (int k = tid; k < kBinVerts; k += 256) {
                const int rr = k / (kBinQX + 1), c = k % (kBinQX + 1);
                const int ii = i0 + rr, jj = j0 + c;
                if (ii < g.sh && jj < g.sw) {
                    const float3 x = vertex(g, ii, jj);
                    V[rr][c] = x;
                    if (vb) { vb[3 * k] = x.x; vb[3 * k + 1] = x.y; vb[3 * k + 2] = x.z; }
                }
            }
            __syncthreads();   // vertices loaded, table cleared
            float2 tv = make_float2(0.f, 0.f);
            if (i < g.sh - 1 && j < g.sw - 1) {
                const int r = tid / kBinQX, c = tid % kBinQX;
                more = quad_range_tv(g, i, j, V[r][c], V[r][c + 1], V[r + 1][c], V[r + 1][c + 1], vd.w, vd.h,
                                     d.tile_shift, tx0, tx1, ty0, ty1, stored_geom ? &tv : nullptr);
                if (stored_geom) {
                    float* t = ws.vbuf + (size_t)wi * kItemFloats + 2 * tid;
                    t[0] = tv.x; t[1] = tv.y;
                }
            }
        }
        auto tile_of = [&](int tx, int ty) { return vd.tile_base + (uint32_t)(ty * vd.tiles_x + tx); };
        auto bin_of = [&](uint32_t t) { return bin_index(d, t, (uint32_t)s); };
        // the range of a kept quad, for its fill pass
        if (!FILL && stored)
            ws.ranges[(size_t)wi * 256 + tid] = more ? pack_range(tx0, tx1, ty0, ty1) : kRangeNone;
        // entries: narrow ranges by their own lane, wide ones dealt to the block
        auto quad_of = [&](int lane) {
            return ((uint32_t)(i0 + lane / kBinQX) << 16) | (uint32_t)(j0 + lane % kBinQX);
        };
        const bool wide = more && (uint32_t)(tx1 - tx0 + 1) * (uint32_t)(ty1 - ty0 + 1) > kLaneTiles;
        const bool any_wide = __syncthreads_or(wide);
        if (any_wide) {
            range_publish(walk, tid, wide, tx0, tx1, ty0, ty1);
            __syncthreads();   // ranges scanned
        }
        auto each_tile = [&](auto fn) {
            if (more && !wide)
                for (int ty = ty0; ty <= ty1; ++ty)
                    for (int tx = tx0; tx <= tx1; ++tx) fn(tid, tx, ty, true);
            if (any_wide) range_walk(walk, tid, fn);
        };
        each_tile([&](int lane, int tx, int ty, bool table) {
            const uint32_t t = tile_of(tx, ty);
            const int k = table ? table_slot(t_key, t) : -1;
            if (k >= 0) {
                atomicAdd(&t_n[k], 1u);
            } else if (FILL) {   // not in the table: a place of its own
                const size_t bin = bin_of(t);
                ws.lists[(size_t)ws.offsets[bin] + atomicAdd(&ws.fill[bin], 1u)] = quad_of(lane);
            } else {
                atomicAdd(&ws.fill[bin_of(t)], 1u);
            }
        });
        __syncthreads();   // table complete
        uint32_t rank = 0u;
        if (tid < kBinTable && t_n[tid]) {
            const size_t bin = bin_of(t_key[tid]);
            if (FILL) t_base[tid] = ws.offsets[bin] + atomicAdd(&ws.fill[bin], t_n[tid]);
            else if (stored) rank = atomicAdd(&ws.counts[bin], t_n[tid]);
            else atomicAdd(&ws.fill[bin], t_n[tid]);
        }
        if (stored) {
            // the item's table for its fill pass: (rank, tile) of the used slots
            // in any order, their number first
            if (tid == 0) t_used = 0u;
            __syncthreads();
            uint2* kt = ws.ktab + (size_t)wi * (1 + kBinTable);
            if (tid < kBinTable && t_n[tid]) kt[1 + atomicAdd(&t_used, 1u)] = make_uint2(rank, t_key[tid]);
            __syncthreads();
            if (tid == 0) kt[0] = make_uint2(t_used, 0u);
        }
        if (FILL) {
            __syncthreads();   // bases known
            each_tile([&](int lane, int tx, int ty, bool table) {
                const int k = table ? find_slot(t_key, tile_of(tx, ty)) : -1;
                if (k >= 0) ws.lists[atomicAdd(&t_base[k], 1u)] = quad_of(lane);
            });
        }
        __syncthreads();   // LDS free for the next item
    }
}

// A quad of the fill pass with more than kLaneTiles tiles.
struct WideFill {
    uint32_t org;    // tx0 | ty0 << 16
    uint32_t dim;    // tiles per row | rows << 16; 0: not known yet
    uint32_t quad;
};

// Fill pass over the kept work items, a wave per item and four quads per lane:
// the item's bins and the places reserved in them by the counting pass go to
// an LDS table, from which every (quad, tile) entry takes its place.  Quads
// with wide ranges are shared by the block's waves, a wave each with a lane
// per tile (an item near a pole deals thousands of tiles).  A tile that found
// the table full while counting takes its place from the bin's cursor.
// Bound by latency: a chain of four dependent accesses per item and the LDS
// atomics of lanes at one tile's cursor, so items in flight matter most (waves
// wait 0.78 of their time, VALU and scalar units issue a quarter of their rates).
// Against a block per item with a returning cursor atomic
// per bin (six accesses in the chain, 8 items per CU instead of 32): 16 mixed
// views 455 -> 280 us, an 8192x4096 panorama of eleven 1.4 -> 1.2 ms.
template <class G>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) k_fill_kept(const G* __restrict__ geoms, const ViewDesc* __restrict__ views,
                                                   BatchDims d, RasterWS ws) {
    __shared__ uint32_t t_key[4][kBinTable];
    __shared__ uint32_t t_base[4][kBinTable];
    __shared__ WideFill wide[4][256];   // [wave whose item it is]
    __shared__ uint32_t nwide[4];
    __shared__ uint32_t w_vs[4];        // (view, source) of the waves' items
    if (ws.status[1]) return;   // list capacity exceeded: nothing to fill
    const uint64_t lim = min(ws.status[4], d.range_cap);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t per = d.bins_x * d.bins_y;
    auto place = [&](int w, uint32_t t, uint32_t s, uint32_t quad, bool table) {
        const int k = table ? find_slot(t_key[w], t) : -1;
        if (k >= 0) {
            ws.lists[atomicAdd(&t_base[w][k], 1u)] = quad;
        } else {
            const size_t bin = bin_index(d, t, s);
            ws.lists[(size_t)ws.offsets[bin] + atomicAdd(&ws.fill[bin], 1u)] = quad;
        }
    };
    // item of wave w in a block's round: neighbouring items (those near a pole
    // are all costly) go to different blocks
    for (uint64_t b0 = blockIdx.x; b0 < lim; b0 += (uint64_t)gridDim.x * 4u) {
        const uint64_t wi64 = b0 + (uint64_t)wave * gridDim.x;
        const uint32_t wi = (uint32_t)wi64;
        t_key[wave][lane] = kTableEmpty;
        t_key[wave][lane + 64] = kTableEmpty;
        if (lane == 0) nwide[wave] = 0u;
        __syncthreads();
        if (wi64 < lim) {   // the same for the wave
            const uint2* kt = ws.ktab + (size_t)wi * (1 + kBinTable);
            const uint2 e0 = kt[1 + lane];   // with the count: entries past it are not used
            uint32_t r[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) r[q] = ws.ranges[(size_t)wi * 256 + q * 64 + lane];
            const uint32_t nused = kt[0].x;
            const uint32_t code = ws.work[wi];
            const uint32_t item = code % per, vs = code / per;
            const uint32_t s = vs % (uint32_t)d.nsrc, v = vs / (uint32_t)d.nsrc;
            const ViewDesc& vd = views[v];
            const int i0 = (int)(item / d.bins_x) * kBinQY, j0 = (int)(item % d.bins_x) * kBinQX;
            if (lane == 0) w_vs[wave] = vs;
            auto take = [&](uint2 e) {
                const uint32_t base = ws.offsets[bin_index(d, e.y, s)] + e.x;
                t_base[wave][table_slot(t_key[wave], e.y)] = base;   // at most kBinTable tiles: never full
            };
            if (lane < (int)nused) take(e0);
            if (lane + 64 < (int)nused) take(kt[65 + lane]);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (r[q] == kRangeNone) continue;
                int tx0, tx1, ty0, ty1;
                unpack_range(r[q], tx0, tx1, ty0, ty1);
                const uint32_t quad = ((uint32_t)(i0 + q) << 16) | (uint32_t)(j0 + lane);
                const uint32_t nx = (uint32_t)(tx1 - tx0 + 1), ny = (uint32_t)(ty1 - ty0 + 1);
                if (r[q] == kRangeBig || nx * ny > kLaneTiles) {
                    WideFill& w = wide[wave][atomicAdd(&nwide[wave], 1u)];
                    w.org = (uint32_t)tx0 | ((uint32_t)ty0 << 16);
                    w.dim = r[q] == kRangeBig ? 0u : nx | (ny << 16);
                    w.quad = quad;
                    continue;
                }
                for (int ty = ty0; ty <= ty1; ++ty)
                    for (int tx = tx0; tx <= tx1; ++tx)
                        place(wave, vd.tile_base + (uint32_t)(ty * vd.tiles_x + tx), s, quad, true);
            }
        }
        __syncthreads();   // wide quads known
        for (int o = 0; o < 4; ++o) {
            const uint32_t nw = nwide[o];
            if (nw == 0u) continue;
            const uint32_t vs = __builtin_amdgcn_readfirstlane(w_vs[o]);
            const uint32_t s = vs % (uint32_t)d.nsrc;
            const ViewDesc& vd = views[vs / (uint32_t)d.nsrc];
            for (uint32_t k = (uint32_t)wave; k < nw; k += 4u) {
                const WideFill w = wide[o][k];
                int tx0 = (int)(w.org & 0xffffu), ty0 = (int)(w.org >> 16);
                uint32_t nx = w.dim & 0xffffu, ny = w.dim >> 16;
                if (w.dim == 0u) {   // too wide to pack: binned again
                    const G& g = geoms[vs];
                    int i, j, tx1, ty1;
                    unpack_ij(w.quad, i, j);
                    float3 c[4];
                    if (d.kept_geom) {
                        const float* p = kept_quad(ws, (uint32_t)b0 + (uint32_t)o * gridDim.x, w.quad).v;
                        c[0] = load3(p); c[1] = load3(p + 3);
                        c[2] = load3(p + 3 * (kBinQX + 1)); c[3] = load3(p + 3 * (kBinQX + 1) + 3);
                    } else {
                        eval_corners<4>(g, i, j, 0xcu, 0xau, c, nullptr);
                    }
                    if (!quad_range_tv(g, i, j, c[0], c[1], c[2], c[3], vd.w, vd.h, d.tile_shift, tx0, tx1, ty0, ty1,
                                       nullptr))
                        continue;
                    nx = (uint32_t)(tx1 - tx0 + 1);
                    ny = (uint32_t)(ty1 - ty0 + 1);
                }
                for (uint32_t e = (uint32_t)lane; e < nx * ny; e += 64u)
                    place(o, vd.tile_base + ((uint32_t)ty0 + e / nx) * (uint32_t)vd.tiles_x + (uint32_t)tx0 + e % nx, s,
                          w.quad, nx * ny <= kTableTiles);
            }
        }
        __syncthreads();   // LDS free for the next items
    }
}

// Bin offsets from the bin counts.  The bins' places in the list need not
// follow their order, so a block scans its own bins and takes their place with
// one atomic on the entry total (64 bits in status[8], status[9]); status[1] is
// set when the list capacity is exceeded.  Three launches (block scans, a scan
// of their sums, an addition) took 15 us of a 1920x1080 view, one takes 6.
// A bin's entries are those with a place (counts) and, behind them, those
// without (fill); counts becomes their sum and fill the cursor of the latter.
constexpr int kScanPer = 2048;   // bins per scan block (256 threads x 8)

__global__ void __launch_bounds__(256) k_bin_places(uint32_t* counts, uint32_t* fill, uint32_t* offsets, size_t n,
                                                    uint32_t cap, uint32_t* status) {
    __shared__ unsigned long long wsum[4], first;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t base = (size_t)blockIdx.x * kScanPer + (size_t)threadIdx.x * 8;
    uint32_t c[8];
    unsigned long long sum = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        c[k] = 0u;
        if (base + k < n) {
            const uint32_t placed = counts[base + k], loose = fill[base + k];
            c[k] = placed + loose;
            if (loose) counts[base + k] = c[k];
            fill[base + k] = placed;
        }
        sum += c[k];
    }
    unsigned long long x = sum;   // inclusive scan over the wave
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned long long y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long all = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
        first = all ? atomicAdd((unsigned long long*)(status + 8), all) : 0ull;
        if (first + all > (unsigned long long)cap) status[1] = 1u;
    }
    __syncthreads();
    unsigned long long run = first + x - sum;
    for (int w = 0; w < wave; ++w) run += wsum[w];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (base + k < n) offsets[base + k] = (uint32_t)run;
        run += c[k];
    }
}

template <class G>
hipError_t launch_bin(const G* geoms, const ViewDesc* views, const BatchDims& d, const RasterWS& ws, hipStream_t s) {
    const size_t total = (size_t)d.bins_x * d.bins_y * d.nsrc * d.nviews;
    const uint32_t npairs = (uint32_t)d.nsrc * (uint32_t)d.nviews;
    hipLaunchKernelGGL(k_bin_cull<G>,
                       dim3((d.bins_x * d.bins_y + kCullThreads - 1) / kCullThreads, npairs < 65535u ? npairs : 65535u),
                       dim3(kCullThreads), 0, s, geoms, views, d, ws);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const size_t blocks = total < (size_t)kBinBlocks ? total : (size_t)kBinBlocks;
    // kept items: persistent blocks striding over them (blocks past the
    // surviving items return at once).  A block's set-up, including the few
    // registers these kernels spill at occupancy 8, is paid once per block, so
    // a few items per block beat a block per item; fewer, longer-lived blocks
    // lose to the tail when items differ in cost (equirectangular targets:
    // items near a pole deal thousands of tiles), so the plan picks the count.
    // A counter that blocks take items from is slower still: every take is a
    // same-address atomic.
    const size_t fb = d.flat_blocks ? d.flat_blocks : (uint32_t)kFlatBlocks;
    const unsigned flat = (unsigned)(d.range_cap < fb ? d.range_cap : fb);
    // (the counting pass strides on through the items past the kept ones)
    hipLaunchKernelGGL((k_bin<G, false>), dim3(flat > blocks ? flat : (unsigned)blocks), dim3(256), 0, s, geoms, views, d,
                       ws);
    const size_t nbins = (size_t)d.ntiles * d.nsrc;
    hipLaunchKernelGGL(k_bin_places, dim3((unsigned)((nbins + kScanPer - 1) / kScanPer)), dim3(256), 0, s, ws.counts,
                       ws.fill, ws.offsets, nbins, d.cap, ws.status);
    if (d.range_cap)
        hipLaunchKernelGGL(k_fill_kept<G>, dim3((flat + 3) / 4), dim3(256), 0, s, geoms, views, d, ws);
    if (total > d.range_cap)
        hipLaunchKernelGGL((k_bin<G, true>), dim3((unsigned)blocks), dim3(256), 0, s, geoms, views, d, ws);
    return hipGetLastError();
}

// ------------------------------------------------------------ tile raster

// The lane's index in its wave, computed where it is called (not merged with
// other reads of it, so it need not stay live in a VGPR in between).
__device__ inline int lane_now() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

// Colours of the corners of slot `slot` of source quad (i, j) (slot_vertex).
template <class G>
__device__ __forceinline__ void slot_colors(const G& g, int slot, int i, int j, float3 (&col)[3]) {
    uint32_t idx[3];
    if (slot < 2) {
        const uint32_t p = (uint32_t)i * (uint32_t)g.sw + (uint32_t)j, down = (uint32_t)g.sw;
        idx[0] = p + (slot ? down + 1u : 0u);
        idx[1] = p + (slot ? down : 1u);
        idx[2] = p + (slot ? 1u : down);
    } else {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            int r, c;
            slot_vertex(slot, k, i, j, g.sw, r, c);
            idx[k] = (uint32_t)r * (uint32_t)g.sw + (uint32_t)c;
        }
    }
    color3(g, idx, col);
}

// Winner's colour, depth and validity at pixel (x, y) for slot `slot` of
// source quad (i, j): the state the fold holds after accepting that candidate.
// FAST: vertex radii and the validity take only their fast float-float paths,
// and the result is false when one of them is undecided (the caller defers the
// pixel; the coverage pass, which evaluated the same triangle, deferred it
// already); otherwise they are exact and the result is true.
template <bool FAST, class G>
__device__ __forceinline__ bool resolve(const G& g, int i, int j, int slot, int x, int y, float3& c, float& dep,
                               float& shape, int out_w, int out_h, const float* vb) {
    float3 v[3], col[3];
    bool und = false;
    slot_colors(g, slot, i, j, col);   // issued first: its loads overlap the vertices'
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
        int rk, ck;
        slot_vertex(slot, k, i, j, g.sw, rk, ck);
        const float3 x = (vb && slot < 2) ? kept_vertex(vb, i % kBinQY + (rk - i), j % kBinQX + (ck - j))
                                          : vertex(g, rk, ck, FAST ? &und : nullptr);
#pragma unroll
        for (int m = 0; m < 3; ++m)
            if (m == k) v[m] = x;
    }
    Tri T;
    if (FAST) {
        tri_setup_geom(T, v[0], v[1], v[2], out_w, out_h);
        if (!tri_validity_fast(T, g.rescale, T.tv) || und) return false;
    } else {
        tri_setup(T, v[0], v[1], v[2], out_w, out_h, g.rescale);
    }
    float l1, l2, l3;
    tri_bary(T, x, y, l1, l2, l3);
    dep = tri_depth(T, l1, l2, l3);
    shape = T.tv;
    c = tri_color(col[0], col[1], col[2], l1, l2, l3);
    return true;
}

// The same from the corner vertices and validity the counting pass kept
// (identical float operations, without re-evaluating vertices or norms).
template <class G>
__device__ __forceinline__ void resolve_cached(const G& g, int i, int j, int slot, float3 a, float3 b, float3 cv, float tv,
                                      int x, int y, float3& c, float& dep, float& shape) {
    float3 col[3];
    slot_colors(g, slot, i, j, col);
    Tri T;
    tri_load(T, a, b, cv);
    T.tv = tv;
    float l1, l2, l3;
    tri_bary(T, x, y, l1, l2, l3);
    dep = tri_depth(T, l1, l2, l3);
    shape = tv;
    c = tri_color(col[0], col[1], col[2], l1, l2, l3);
}

// key2 value of a pixel that must take the in-order replay (above every
// score: scores are finite positive floats).
constexpr uint32_t kDeferKey = 0xffffffffu;

// Pushes candidate `id` of triangle T for the tile's pixel p with centre (fx,
// fy): the exact coverage test, then the key updates.  r: recip(T.den).
// Sets *tie (if any) when it meets a candidate of the same score.
// TIES: the second pass, over tied pixels only (their shape in tie[p], 0 for the
// others; their depth's bits in key2[p]): see settle_ties.
template <bool TIES>
__device__ __forceinline__ void raster_push(const Tri& T, float r, bool special, uint32_t id, uint32_t ij, float fx,
                                            float fy, int p, unsigned long long* key1, uint32_t* key2, float* tie) {
    if (TIES && !(tie[p] > 0.f)) return;
    // tri_num at the pixel
    const float dx = fx - T.C0, dy = fy - T.C1;
    const float n1 = (T.B1 - T.C1) * dx + (T.C0 - T.B0) * dy, n2 = (T.C1 - T.A1) * dx + (T.A0 - T.C0) * dy;
    float l1, l2, l3;
    if (!tri_cover_r(T, r, n1, n2, l1, l2, l3)) return;
    const float dd = tri_depth(T, l1, l2, l3);
    // the score only orders candidates outside the ambiguity band:
    // v_rcp_f32 (1 ulp) keeps its error within 5 * 2^-24 relative
    const float f = T.tv * __builtin_amdgcn_rcpf(dd * dd * dd);
    if (TIES) {
        const float v = tie[p], w = u2f(key2[p]);
        if (!special && f2u(dd) == f2u(w) && T.tv == v) {
            atomicMin(&key1[p], ((unsigned long long)ij << 32) | ((unsigned long long)(id & 3u) << 30) | (id >> 2));
        } else {
            const float fw = v * __builtin_amdgcn_rcpf(w * w * w);
            if (special || !(f < fw - fw * RVS_AMBIGUITY)) atomicMin(&key1[p], 0ull);
        }
        return;
    }
    const bool defer = special || !depth_regular(dd);
    const unsigned long long k = defer ? 0ull : ((unsigned long long)f2u(f) << 32) | id;
    const unsigned long long old = atomicMax(&key1[p], k);
    if (tie && (uint32_t)(old >> 32) == f2u(f)) *tie = 1.f;
    // the candidate that is not (or no longer) the maximum goes to the runner-up slot
    atomicMax(&key2[p], defer ? kDeferKey : (uint32_t)((old < k ? old : k) >> 32));
}

// Ids of a phase's wide triangles, put off until its other triangles are done.
template <int CAP>
struct WideQueue {
    static constexpr uint32_t cap = CAP;
    uint32_t n;        // pushed (those beyond cap were done in place)
    uint32_t id[CAP];
};

// Pixels of the tile that triangle T may cover; false when there are none.
template <int TILE>
__device__ __forceinline__ bool tile_box(Tri& T, int tx0, int ty0, int out_w, int out_h, int& xa, int& xb, int& ya,
                                         int& yb) {
    return tri_box(T, out_w, out_h, tx0, min(out_w, tx0 + TILE) - 1, ty0, min(out_h, ty0 + TILE) - 1, xa, xb, ya, yb);
}

// T's validity: the one the counting pass kept (> 0; KNOWN: it was evaluated
// there whenever T has a pixel), else the fast path.  False when the fast path
// leaves it undecided: the pixels the triangle covers are then deferred (T.tv
// is at least 0 then too).
template <bool KNOWN>
__device__ __forceinline__ bool take_validity(Tri& T, float rescale, float tv_known) {
    T.tv = tv_known;
    return tv_known > 0.f || (!KNOWN && tri_validity_fast(T, rescale, T.tv));
}

// Pass over one triangle of a binned quad for the tile at (tx0, ty0): per
// covered pixel, push the candidate key (score bits << 32 | candidate id)
// into key1 and the displaced score into key2.  Candidates with non-finite
// inputs or extreme depths mark the pixel for the in-order replay instead.
// The validity is evaluated only when a pixel of the tile may be covered (the
// reference computes it before the bounding box test, but it never causes a
// return, and a triangle that covers no pixel is never a winner, so skipping
// it changes nothing).  A finite triangle with more than kWidePx pixels of the
// tile in its box is left to raster_wide while the queue Q (null: none) has
// room.
template <int TILE, bool KNOWN, bool TIES, class Queue>
__device__ __forceinline__ void raster_tri(float3 a, float3 b, float3 c, uint32_t id, uint32_t ij, bool prol_false_possible, int tx0,
                                   int ty0, int out_w, int out_h, float rescale, unsigned long long* key1,
                                   uint32_t* key2, bool undecided, float tv_known, Queue* Q, float* tie) {
    Tri T;
    tri_load(T, a, b, c);
    int xa, xb, ya, yb;
    if (!tile_box<TILE>(T, tx0, ty0, out_w, out_h, xa, xb, ya, yb)) return;   // no pixel of this tile can be covered
    const bool prol = (a.z > 0.f) || (b.z > 0.f) || (c.z > 0.f);
    // a finite den has finite image coordinates
    bool special = !is_finite(a.z + b.z + c.z) || !is_finite(T.den) || (prol_false_possible && !prol) || undecided;
    if (!cover_den(T.den)) {
        if (TIES) return;   // done in the first pass
        // degenerate, gigantic or non-finite: whatever it may cover is deferred
        for (int y = ya; y <= yb; ++y)
            for (int x = xa; x <= xb; ++x) {
                float n1, n2;
                tri_num(T, x, y, n1, n2);
                if (!tri_surely_outside(T, n1, n2)) atomicMax(&key2[(y - ty0) * TILE + (x - tx0)], kDeferKey);
            }
        return;
    }
    if (Q && !special && (int)__umul24(xb - xa + 1, yb - ya + 1) > kWidePx) {
        const uint32_t q = atomicAdd(&Q->n, 1u);
        if (q < Queue::cap) {
            Q->id[q] = id;
            return;
        }
    }
    const float r = recip(T.den);
    const float ex1 = T.B1 - T.C1, ey1 = T.C0 - T.B0, ex2 = T.C1 - T.A1, ey2 = T.A0 - T.C0;   // tri_num's
    T.tv = -1.f;   // not taken yet
    // 8 x 4 pixels at a time (most boxes are smaller), in two steps, so that
    // lanes with few candidates do not wait through the exact test of lanes
    // with large boxes: the rejection by approximate barycentrics marks the
    // candidates (a bit each), then only those take the exact coverage test and
    // the key updates.
    for (int y0 = ya; y0 <= yb; y0 += 4)
        for (int x0 = xa; x0 <= xb; x0 += 8) {
            const int nx = min(xb - x0, 7), ny = min(yb - y0, 3);
            const float fx0 = (float)x0 + 0.5f, fy0 = (float)y0 + 0.5f;
            float fy = fy0;
            uint32_t mask = 0u;
            for (int row = 0; row <= ny; ++row) {
                const float dy = fy - T.C1, m1 = ey1 * dy, m2 = ey2 * dy;
                float fx = fx0;
                uint32_t bits = 0u;
                for (uint32_t bit = 1u; bit <= 1u << nx; bit <<= 1) {
                    const float dx = fx - T.C0;
                    if (!tri_outside_r(r, ex1 * dx + m1, ex2 * dx + m2)) bits |= bit;
                    fx += 1.f;
                }
                mask |= bits << (row * 8);
                fy += 1.f;
            }
            if (!mask) continue;
            if (T.tv < 0.f && !take_validity<KNOWN>(T, rescale, tv_known)) special = true;
            const int p0 = (y0 - ty0) * TILE + (x0 - tx0);
            while (mask) {
                const int bit = __builtin_ctz(mask), col = bit & 7, row = bit >> 3;
                mask &= mask - 1u;
                raster_push<TIES>(T, r, special, id, ij, fx0 + (float)col, fy0 + (float)row, p0 + row * TILE + col, key1, key2, tie);
            }
        }
}

__device__ __forceinline__ float lane_f(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Bins of the sources of a phase, concatenated: source k's entries e lie in
// [end[k - 1], end[k]) and at lists[e + add[k]] (modulo 2^32).  Uniform: in SGPRs.
struct Phase {
    uint32_t end0, end1, end2, n;
    uint32_t add0, d1, d2, d3;   // add[0], and each later source's step (selects between the sums
                                 // themselves become loads from scratch)
    // Source of entry e < n and its quad code.
    __device__ int find(const RasterWS& ws, uint32_t e, uint32_t& code) const {
        const bool a = e >= end0, b = e >= end1, c = e >= end2;
        const uint32_t at = add0 + (a ? d1 : 0u) + (b ? d2 : 0u) + (c ? d3 : 0u);
        code = ws.lists[e + at];
        return (int)a + (int)b + (int)c;
    }
};
static_assert(kRasterGroup == 4, "a phase of four sources");

// The wave's share of a phase's queued triangles: each lane fetches and sets
// up one (a single chain of loads for all of them), then the wave takes them
// one after the other from the lanes' registers, a lane per pixel.  A lane
// walking a wide triangle by itself holds its wave (and, at the barrier, the
// block) for up to TILE^2 steps, and wide triangles are neighbours in the
// bins: stretched across a depth edge, magnified, or near a pole.
// Measured: two 3840x2160 views of 11 perspective sources, raster 4.03 -> 3.40
// ms; 8 views of 1920x1080 of four panoramas 1.80 -> 1.22 ms.
template <int TILE, int NT, bool KEPT, bool TIES, class G, class Queue>
__device__ __forceinline__ void raster_wide(const G* gv, const Phase& ph, uint32_t nwide, const Queue& Q, int wave, int tx0, int ty0, int out_w,
                                            int out_h, unsigned long long (*key1)[NT], uint32_t (*key2)[NT],
                                            const RasterWS& ws, const BatchDims& d, uint32_t vs0,
                                            float (*ties)[NT], float* tie) {
    constexpr uint32_t NW = NT / 64;
    for (uint32_t q0 = (uint32_t)wave; q0 < nwide; q0 += 64u * NW) {
        const uint32_t q = q0 + NW * (uint32_t)lane_now();
        Tri T;
        float tr = 0.f;
        int k = 0, xa = 0, xb = -1, ya = 0, yb = -1, sp = 0;
        uint32_t id = 0u, code = 0u;
        if (q < nwide) {
            id = Q.id[q];
            k = ph.find(ws, id >> 2, code);
            int i, j;
            unpack_ij(code, i, j);
            const G& g = gv[k];
            const uint32_t wi = kept_index<KEPT>(ws, d, vs0 + (uint32_t)k, code);
            // one evaluated here was decided by the fast path when the triangle was queued
            const int slot = (int)(id & 3u);
            bool und = false;
            float2 tvk = make_float2(0.f, 0.f);
            float3 c3[3];
            if (KEPT || wi != 0xffffffffu) {
                const KeptQuad kq = kept_quad(ws, wi, code);
                kept_corners(kq.v, slot, c3);
                tvk = make_float2(kq.tv[0], kq.tv[1]);
            } else {
                eval_corners<3>(g, i, j, slot ? 3u : 4u, slot ? 5u : 2u, c3, &und);
            }
            const float3 a = c3[0], b = c3[1], c = c3[2];
            tri_load(T, a, b, c);
            tile_box<TILE>(T, tx0, ty0, out_w, out_h, xa, xb, ya, yb);
            if (!take_validity<KEPT>(T, g.rescale, slot ? tvk.y : tvk.x)) sp = 0x100;
            tr = recip(T.den);
        }
        const int m = min(64, (int)((nwide - q0 + NW - 1u) / NW));
        for (int l = 0; l < m; ++l) {
            Tri W;
            W.A0 = lane_f(T.A0, l); W.A1 = lane_f(T.A1, l);
            W.B0 = lane_f(T.B0, l); W.B1 = lane_f(T.B1, l);
            W.C0 = lane_f(T.C0, l); W.C1 = lane_f(T.C1, l);
            W.dA = lane_f(T.dA, l); W.dB = lane_f(T.dB, l); W.dC = lane_f(T.dC, l);
            W.den = lane_f(T.den, l); W.tv = lane_f(T.tv, l);
            const int wx = __builtin_amdgcn_readlane(xa, l), wy = __builtin_amdgcn_readlane(ya, l);
            const int bw = __builtin_amdgcn_readlane(xb, l) - wx + 1;
            const int n = bw * (__builtin_amdgcn_readlane(yb, l) - wy + 1);
            const int sk = __builtin_amdgcn_readlane(k | sp, l);
            const uint32_t wij = TIES ? (uint32_t)__builtin_amdgcn_readlane((int)code, l) : 0u;
            const uint32_t wid = (uint32_t)__builtin_amdgcn_readlane((int)id, l);
            const float inv = __builtin_amdgcn_rcpf((float)bw), r = lane_f(tr, l);
            for (int i = lane_now(); i < n; i += 64) {
                // row i / bw: i + 1/2 is at least 1 / (2 bw) of a row away from the next one
                const int row = (int)(((float)i + 0.5f) * inv);
                const int x = wx + (i - row * bw), y = wy + row;
                float n1, n2;
                tri_num(W, x, y, n1, n2);
                if (!tri_outside_r(r, n1, n2))
                    raster_push<TIES>(W, r, sk >= 0x100, wid, wij, (float)x + 0.5f, (float)y + 0.5f,
                                (y - ty0) * TILE + (x - tx0), key1[sk & 0xff], key2[sk & 0xff],
                                      TIES ? ties[sk & 0xff] : tie);
            }
        }
    }
}

// Per-phase LDS copy of what the coverage pass looked up for each binned
// quad: the quad code and its kept work item (~0: none), so that the winners'
// corner vertices and validities are read from the kept blocks without the
// work-item map.
template <int CAP>
struct RasterCache {
    static constexpr int cap = CAP;
    uint32_t ij[CAP];
    uint32_t wi[CAP];
};

// Candidate ids: (entry << 2) | slot, entry = index of the quad in the phase's
// concatenated bins.  A non-deferred pixel's winner beats every other
// candidate by more than the float test's error, so any unique id works; equal
// scores are deferred to the in-order replay or settled by the second pass,
// which goes by quad and slot.
// gt: any descriptor of the view (target-side fields: the same for all its
// sources, so they are read once per wave).
template <int TILE, bool KEPT, bool TIES, class G, class Cache, class Queue>
__device__ __forceinline__ void raster_quad(const G& g, const G& gt, uint32_t ij, uint32_t e, int tx0, int ty0,
                                            int out_w, int out_h, unsigned long long* key1, uint32_t* key2, Cache* C,
                                            Queue* Q, const RasterWS& ws, const BatchDims& d, uint32_t vs,
                                            float* tie) {
    int i, j;
    unpack_ij(ij, i, j);
    const uint32_t wi = kept_index<KEPT>(ws, d, vs, ij);
    // vertices evaluated here take the fast radius path; an undecided one
    // defers the pixels of the quad's triangles (kept vertices are exact)
    bool und = false;
    float2 tvk = make_float2(0.f, 0.f);
    float3 v00, v01, v10, v11;
    if (KEPT || wi != 0xffffffffu) {
        const KeptQuad kq = kept_quad(ws, wi, ij);
        const float* p = kq.v;
        v00 = load3(p); v01 = load3(p + 3);
        v10 = load3(p + 3 * (kBinQX + 1)); v11 = load3(p + 3 * (kBinQX + 1) + 3);
        tvk = make_float2(kq.tv[0], kq.tv[1]);
    } else {
        float3 v[4];
        eval_corners<4>(g, i, j, 0xcu, 0xau, v, &und);
        v00 = v[0]; v01 = v[1]; v10 = v[2]; v11 = v[3];
    }
    const bool gate = v01.z > 0.f && v10.z > 0.f && v01.x > 0.f && v10.x > 0.f;
    const uint32_t s0 = e << 2;
    if (gate && v00.z > 0.f && v00.x > 0.f)
        raster_tri<TILE, KEPT, TIES>(v00, v01, v10, s0, ij, false, tx0, ty0, out_w, out_h, gt.rescale, key1, key2, und, tvk.x, Q,
                                     tie);
    if (gate && v11.z > 0.f && v11.x > 0.f)
        raster_tri<TILE, KEPT, TIES>(v11, v10, v01, s0 | 1u, ij, false, tx0, ty0, out_w, out_h, gt.rescale, key1, key2, und,
                               tvk.y, Q, tie);
    if (__builtin_expect(gate && gt.wrap && j == 0, 0)) {
        float3 l[2];
        if (KEPT) kept_seam(ws, d, vs, i, g.sw, l);
        else eval_corners<2>(g, i, g.sw - 1, 2u, 0u, l, &und);
#pragma unroll 1
        for (uint32_t k = 0; k < 2u; ++k) {
            const bool s3 = k != 0u;
            raster_tri<TILE, false, TIES>(s3 ? v10 : l[0], s3 ? l[1] : v00, s3 ? v00 : l[1], s0 | (2u + k), ij, true, tx0, ty0,
                                    out_w, out_h, gt.rescale, key1, key2, und, 0.f, (Queue*)nullptr, tie);
        }
    }
    if (C) {
        C->ij[e] = ij;
        C->wi[e] = wi;
    }
}

template <int MODE>
__device__ inline void write_pixel(const ViewDesc& vd, size_t o, const BlendState& st, float3 rc, float rd, float rs,
                                   bool color = true, bool quality = true) {
    if (MODE == MODE_RAW) {
        vd.color[3 * o] = rc.x; vd.color[3 * o + 1] = rc.y; vd.color[3 * o + 2] = rc.z;
        vd.depth[o] = rd;
        vd.validity[o] = rs;
    } else {
        if (color) { vd.color[3 * o] = st.c.x; vd.color[3 * o + 1] = st.c.y; vd.color[3 * o + 2] = st.c.z; }
        if (vd.depth) vd.depth[o] = st.d;
        if (quality) vd.quality[o] = st.q;
        if (vd.validity) vd.validity[o] = st.v;
    }
}

// write_color (image_writing.cpp:142-203) of one pixel of a tile, from the
// blended colour in registers: Y here, U and V by the top-left pixel of each
// 2x2 block from its wave neighbours (a tile row is at most half a wave, so
// the block's four pixels are lanes l, l+1, l+TILE, l+TILE+1 of one wave).  The
// same quantisation and chroma rule as k_encode_views; tiles start at even
// coordinates and encoded views have even sizes, so a block is inside or
// outside as a whole.
template <int TILE>
__device__ inline void encode_tile_pixel(const ViewDesc& vd, float3 c, int px, int py, bool inside, int lx, int ly) {
    const unsigned maxv = (1u << vd.bitdepth) - 1u;
    const bool u8 = vd.bitdepth <= 8;
    uint32_t qy = quantize_u32(c.x, maxv), qu = quantize_u32(c.y, maxv), qv = quantize_u32(c.z, maxv);
    // the plane's element type truncates, as (T) does in k_encode_views
    if (u8) { qy &= 0xffu; qu &= 0xffu; qv &= 0xffu; } else { qy &= 0xffffu; qu &= 0xffffu; qv &= 0xffffu; }
    static_assert(2 * TILE <= 64, "a 2x2 block's two rows must lie in one wave");
    const uint32_t su = qu + (uint32_t)__shfl_down((int)qu, 1) + (uint32_t)__shfl_down((int)qu, TILE) +
                        (uint32_t)__shfl_down((int)qu, TILE + 1);
    const uint32_t sv = qv + (uint32_t)__shfl_down((int)qv, 1) + (uint32_t)__shfl_down((int)qv, TILE) +
                        (uint32_t)__shfl_down((int)qv, TILE + 1);
    if (!inside) return;
    const size_t o = (size_t)py * vd.ew + px;
    const bool corner = ((lx | ly) & 1) == 0;
    const size_t oc = (size_t)(py >> 1) * (vd.ew >> 1) + (px >> 1);
    if (u8) {
        ((uint8_t*)vd.y)[o] = (uint8_t)qy;
        if (corner) { ((uint8_t*)vd.u)[oc] = (uint8_t)((su + 2) >> 2); ((uint8_t*)vd.v)[oc] = (uint8_t)((sv + 2) >> 2); }
    } else {
        ((uint16_t*)vd.y)[o] = (uint16_t)qy;
        if (corner) {
            ((uint16_t*)vd.u)[oc] = (uint16_t)((su + 2) >> 2);
            ((uint16_t*)vd.v)[oc] = (uint16_t)((sv + 2) >> 2);
        }
    }
}

// LDS of a k_raster block.
template <int TILE>
struct RasterLds {
    static constexpr int NT = TILE * TILE;
    static constexpr int AREA = NT / (kTile * kTile);
    static constexpr int GRP = kRasterGroup;   // sources per phase
    unsigned long long key1[GRP][NT];
    uint32_t key2[GRP][NT];
    int s_deferred;       // any pixel of the tile deferred
    int s_hole;           // any pixel of the tile a hole (quality not > 0)
    RasterCache<kRasterCache * AREA> cache;
    typedef WideQueue<kWideQueue * AREA> Queue;
    Queue wide;
    float s_tie;          // two candidates of one score met (0 / 1)
};

// One tile of k_raster.  Bound by the issue of VALU instructions: 0.67 T wave
// instructions/s with 16 x 16 tiles, 0.61 with 32 x 32, of about 0.74 for its
// mix (loops of one kind of instruction at 8 waves per SIMD reach 0.97 T/s with
// two operands, 0.59 with three and for compares, 0.30 for reciprocals; a good
// half of the code is of the first kind).  Raster ms with the box and the narrowing one
// after the other, the candidates marked by exact numerators and every
// barycentric divided out, vertex code in one body, 64-bit index arithmetic and
// branches in the candidate and blend loops -> now: 16 views of mixed sizes
// 3.13 -> 2.38, one 1920x1080 view 0.246 -> 0.177 (four 4096x2048 panoramas);
// 8192x4096 panorama of eleven 11.0 -> 7.3; two 3840x2160 views of 11
// perspective sources 3.42 -> 2.66.  Of 2.57 ms (16 views, builds that skip a
// part): resolve and blend 0.75, exact tests and keys 0.56, vertex fetch and
// denominators 0.41, candidate scan 0.34, wide triangles 0.13, boxes 0.07, the
// rest of a tile 0.37.  KEPT: every surviving work item keeps its vertex
// window and validities, so this code evaluates no vertex and no validity of
// slots 0 and 1: a third of the instructions of the general form, whose
// registers would otherwise spill around them.  The general form is for launch
// sets with items beyond the kept range: few sources and large targets never
// have any, small targets of large sources do (1280x720 from 11 perspective
// 2048x2048 sources keep 63 k of 110 k items).  It spills 30-45 registers, most
// of them around the vertex evaluation; against the single body before this one
// (2 spilled at most): that 1280x720 view 0.82 -> 0.64 ms, four of them 2.83 ->
// 2.40, 854x480 0.65 -> 0.50, 854x480 from four panoramas 0.52 -> 0.52, and
// 320x180 into a pole of them, one tile of 50 k quads, 1.0-1.3 -> 1.1-1.3.
// Out-of-line vertices (9-23 spilled) are slower, 0.50 -> 0.72 ms.
template <class G, int MODE, bool MULTI, int TILE, bool KEPT, bool SETTLE>
__device__ __forceinline__ void raster_tile(const G* __restrict__ geoms, const ViewDesc* __restrict__ views,
                                            const BatchDims& d, const RasterWS& ws, RasterLds<TILE>& L) {
    typedef RasterLds<TILE> Lds;
    typedef typename Lds::Queue Queue;
    constexpr int NT = Lds::NT, GRP = Lds::GRP;
    auto& key1 = L.key1;
    auto& key2 = L.key2;
    auto& cache = L.cache;
    Queue& wide = L.wide;
    int& s_deferred = L.s_deferred;
    int& s_hole = L.s_hole;
    float& s_tie = L.s_tie;
    const uint32_t T = tile_of_block(blockIdx.x, d.ntiles);
    if (T >= d.ntiles) return;
    const int v = find_view(views, d.nviews, T);
    const ViewDesc& vd = views[v];
    const int tile = (int)(T - vd.tile_base);
    const int tid = threadIdx.x;
    const int tx0 = (tile % vd.tiles_x) * TILE, ty0 = (tile / vd.tiles_x) * TILE;
    // The thread's index is re-derived after the coverage pass (wave base in
    // an SGPR + lane id) instead of being held in a VGPR through it.
    const int wave_base = __builtin_amdgcn_readfirstlane(tid & ~63);
    const G* gv = geoms + (size_t)v * d.nsrc;
    bool deferred = false;
    BlendState st;
    float3 rc = make_float3(0.f, 0.f, 0.f);
    float rd = __builtin_inff(), rs = 0.f;
    for (int s0 = 0; s0 < (MULTI ? d.nsrc : 1); s0 += GRP) {
        const int gs = min(GRP, d.nsrc - s0);
        for (int k = 0; k < gs; ++k) {
            key1[k][tid] = 0ull;
            key2[k][tid] = 0u;
        }
        if (tid == 0) {
            if (s0 == 0) { s_deferred = 0; s_hole = 0; }
            wide.n = 0u;
            if (SETTLE) s_tie = 0.f;
        }
        uint32_t end[GRP], add[GRP], acc = 0u;
#pragma unroll
        for (int k = 0; k < GRP; ++k) {
            const size_t b = bin_index(d, T, (uint32_t)(s0 + (k < gs ? k : 0)));
            const uint32_t cnt = ws.counts[b], off = ws.offsets[b];
            add[k] = off - acc;
            acc += k < gs ? cnt : 0u;
            end[k] = acc;
        }
        const Phase ph = {end[0], end[1], end[2], acc, add[0], add[1] - add[0], add[2] - add[1], add[3] - add[2]};
        __syncthreads();
        const uint32_t N = ph.n;
        bool cached = N <= (uint32_t)cache.cap;
        // a wave-uniform trip count; the entry index is re-derived each trip
        const uint32_t trips = (N + (uint32_t)NT - 1u) / (uint32_t)NT;
        for (uint32_t it = 0; it < trips; ++it) {
            const uint32_t e = it * (uint32_t)NT + (uint32_t)(wave_base + lane_now());
            if (e >= N) continue;
            uint32_t ij;
            const int k = ph.find(ws, e, ij);
            raster_quad<TILE, KEPT, false>(gv[s0 + k], gv[0], ij, e, tx0, ty0, vd.w, vd.h, key1[k], key2[k],
                                           cached ? &cache : nullptr, &wide, ws, d, (uint32_t)(v * d.nsrc + s0 + k),
                                           SETTLE ? &s_tie : (float*)nullptr);
        }
        __syncthreads();
        const uint32_t nwide = __builtin_amdgcn_readfirstlane(min(wide.n, Queue::cap));
        if (nwide) {   // the same in every wave
            raster_wide<TILE, NT, KEPT, false>(gv + s0, ph, nwide, wide, wave_base / 64, tx0, ty0, vd.w, vd.h, key1, key2,
                                               ws, d, (uint32_t)(v * d.nsrc + s0), (float(*)[NT])nullptr,
                                               SETTLE ? &s_tie : (float*)nullptr);
            __syncthreads();
        }
        if (SETTLE && __builtin_amdgcn_readfirstlane(f2u(s_tie)) != 0u) {
            // Settles exact ties (a plane seen from an aligned camera puts every
            // pixel on the edge between two quads): where all candidates within
            // the ambiguity of the best have its very depth and validity, the
            // fold keeps the first of them -- each later one meets a ratio of 1
            // and its own validity -- so a second pass takes the least
            // (quad, slot); any other candidate that near leaves the pixel
            // deferred.  The second pass replaces the replay of those pixels:
            // 640x480 pair 290 -> 245 us.
            auto ties = reinterpret_cast<float(*)[NT]>(&cache);   // the cache is given up
            static_assert(sizeof(cache) >= sizeof(float) * GRP * NT, "the ties' shapes fit the cache");
            const int t2 = wave_base + lane_now();
            const int px = tx0 + (t2 % TILE), py = ty0 + (t2 / TILE);
            float shape[GRP];
#pragma unroll
            for (int k = 0; k < GRP; ++k) {
                shape[k] = 0.f;
                if (k >= gs) continue;
                const unsigned long long kw = key1[k][t2];
                if (kw == 0ull || key2[k][t2] != (uint32_t)(kw >> 32) || ((uint32_t)kw & 2u)) continue;
                uint32_t ij;
                ph.find(ws, (uint32_t)kw >> 2, ij);
                const KeptQuad kq = kept_quad(ws, kept_index<true>(ws, d, (uint32_t)(v * d.nsrc + s0 + k), ij), ij);
                const int slot = (int)((uint32_t)kw & 1u);
                float3 c3[3];
                kept_corners(kq.v, slot, c3);
                Tri W;
                tri_load(W, c3[0], c3[1], c3[2]);
                float l1, l2, l3;
                tri_bary(W, px, py, l1, l2, l3);
                shape[k] = kq.tv[slot];
                key1[k][t2] = ~0ull;
                key2[k][t2] = f2u(tri_depth(W, l1, l2, l3));
            }
            if (t2 == 0) wide.n = 0u;
            __syncthreads();   // the cache and the queue are no longer read
#pragma unroll
            for (int k = 0; k < GRP; ++k) ties[k][t2] = shape[k];
            __syncthreads();
            for (uint32_t it = 0; it < trips; ++it) {
                const uint32_t e = it * (uint32_t)NT + (uint32_t)(wave_base + lane_now());
                if (e >= N) continue;
                uint32_t ij;
                const int k = ph.find(ws, e, ij);
                raster_quad<TILE, KEPT, true>(gv[s0 + k], gv[0], ij, e, tx0, ty0, vd.w, vd.h, key1[k], key2[k],
                                              (decltype(&cache))nullptr, &wide, ws, d,
                                              (uint32_t)(v * d.nsrc + s0 + k), ties[k]);
            }
            __syncthreads();
            const uint32_t nw = __builtin_amdgcn_readfirstlane(min(wide.n, Queue::cap));
            if (nw) {
                raster_wide<TILE, NT, KEPT, true>(gv + s0, ph, nw, wide, wave_base / 64, tx0, ty0, vd.w, vd.h, key1, key2,
                                                  ws, d, (uint32_t)(v * d.nsrc + s0), ties, &s_tie);
                __syncthreads();
            }
            const int t4 = wave_base + lane_now();
            for (int k = 0; k < gs; ++k) {
                if (!(ties[k][t4] > 0.f)) continue;
                const unsigned long long o = key1[k][t4];
                const uint32_t id = ((uint32_t)o << 2) | ((uint32_t)o >> 30);
                key1[k][t4] = (1ull << 32) | id;
                key2[k][t4] = o == 0ull || o == ~0ull ? kDeferKey : 0u;
            }
            cached = false;
        }
        const int t2 = wave_base + lane_now();
        const int px = tx0 + (t2 % TILE), py = ty0 + (t2 / TILE);
        const bool inside = px < vd.w && py < vd.h;
        if (inside) {
            for (int k = 0; k < gs; ++k) {
                const int s = s0 + k;
                if (deferred) break;
                const unsigned long long kw = key1[k][t2];
                const uint32_t k2 = key2[k][t2];
                bool amb = k2 == kDeferKey;
                if (!amb && kw != 0ull && k2 != 0u) {
                    const float fw = u2f((uint32_t)(kw >> 32)), f2 = u2f(k2);
                    amb = f2 >= fw - fw * RVS_AMBIGUITY;
                }
                if (amb) { deferred = true; break; }
                float3 c = make_float3(0.f, 0.f, 0.f);
                float dep = __builtin_inff(), shape = 0.f;
                if (kw != 0ull) {
                    const uint32_t id = (uint32_t)kw, e = id >> 2;
                    const int slot = (int)(id & 3u);
                    const G& g = gv[s];
                    const uint32_t vs = (uint32_t)(v * d.nsrc + s);
                    uint32_t ij;
                    if (cached) ij = cache.ij[e];
                    else ph.find(ws, e, ij);
                    int i, j;
                    unpack_ij(ij, i, j);
                    const uint32_t wk = cached ? cache.wi[e] : kept_index<KEPT>(ws, d, vs, ij);
                    bool ok = true;
                    if (slot < 2 && (KEPT || wk != 0xffffffffu)) {
                        // the validity the counting pass kept (the coverage pass used it)
                        const KeptQuad kq = kept_quad(ws, wk, ij);
                        float3 t[3];
                        kept_corners(kq.v, slot, t);
                        resolve_cached(g, i, j, slot, t[0], t[1], t[2], kq.tv[slot], px, py, c, dep, shape);
                    } else if (KEPT) {   // slot 2: l0 v00 l1, slot 3: v10 l1 v00
                        const float* p = kept_quad(ws, wk, ij).v;
                        const float3 v00 = load3(p), v10 = load3(p + 3 * (kBinQX + 1));
                        float3 l[2];
                        kept_seam(ws, d, vs, i, g.sw, l);
                        const float3 a = slot == 2 ? l[0] : v10, b = slot == 2 ? v00 : l[1], cc = slot == 2 ? l[1] : v00;
                        Tri T;
                        tri_load(T, a, b, cc);
                        ok = tri_validity_fast(T, g.rescale, T.tv);
                        resolve_cached(g, i, j, slot, a, b, cc, T.tv, px, py, c, dep, shape);
                    } else {
                        ok = resolve<true>(g, i, j, slot, px, py, c, dep, shape, vd.w, vd.h, kept_block(ws, d, vs, ij));
                    }
                    if (!ok) { deferred = true; break; }
                }
                if (MODE == MODE_RAW) {
                    rc = c; rd = dep; rs = shape;
                } else if (s == 0) {
                    blend_first(st, c, dep, shape);
                } else {
                    blend_step(st, c, dep, shape, vd.blend_exp, vd.blend_inv);
                }
            }
        }
        __syncthreads();
    }
    const int t3 = wave_base + lane_now();
    const int lx = t3 % TILE, ly = t3 / TILE;
    const int px = tx0 + lx, py = ty0 + ly;
    const bool inside = px < vd.w && py < vd.h;
    const size_t o = (size_t)py * vd.w + px;
    // a tile with a deferred pixel or a hole (quality not > 0: the inpainting
    // mask) is finished by the replay / inpainting and encoded after them;
    // any other tile of a view that wants planes is encoded here
    if (deferred) s_deferred = 1;
    if (MODE == MODE_BLEND && inside && !deferred && !(st.q > 0.f)) s_hole = 1;
    __syncthreads();
    const bool enc = MODE == MODE_BLEND && vd.enc_raster && !s_deferred && !s_hole;
    if (inside && !deferred) {
        // an internal colour map of a tile encoded here is read only on the
        // tile's border (by the inpainting of a neighbouring tile)
        const bool border = lx == 0 || ly == 0 || lx == TILE - 1 || ly == TILE - 1;
        write_pixel<MODE>(vd, o, st, rc, rd, rs, !(enc && vd.partial_color && !border),
                          !(vd.partial_quality && !s_hole && !s_deferred));
    }
    if (enc) encode_tile_pixel<TILE>(vd, st.c, px, py, inside, lx, ly);
    if (t3 == 0) ws.tile_enc[T] = (enc ? 1 : 0) | (MODE == MODE_BLEND && (s_hole || s_deferred) ? 2 : 0);
    // the replay reads the per-pixel flags of the listed tiles only
    if (s_deferred) {
        if (inside) ws.deferred[vd.px_base + o] = deferred ? 1 : 0;
        if (t3 == 0) {
            const uint32_t k = atomicAdd(&ws.status[0], 1u);
            ws.deferred_tiles[k] = T;
        }
    }
}

// MULTI: more sources than one phase holds (the phases loop, and the blend
// state lives across them); otherwise one phase, which keeps the coverage pass
// free of the blend state's registers.
// TILE: the tile edge; a block has a thread per pixel (256 or 1024 threads),
// and the caches scale with the tile's area.
// SETTLE: exact ties are settled here (BatchDims::settle; one phase only).  Where
// ties are chance, meeting them costs the candidate loop more than their replay.
template <class G, int MODE, bool MULTI, int TILE, bool SETTLE>
__global__ void __launch_bounds__(TILE * TILE) __attribute__((amdgpu_waves_per_eu(MULTI ? (TILE > kTile ? 4 : 7) : 8)))
k_raster(const G* __restrict__ geoms, const ViewDesc* __restrict__ views, BatchDims d, RasterWS ws) {
    __shared__ RasterLds<TILE> lds;
    if (ws.status[1]) return;   // bins not filled: capacity reported to the host
    if (d.kept_geom && ws.status[4] <= d.range_cap)   // the same for the whole launch
        raster_tile<G, MODE, MULTI, TILE, true, SETTLE>(geoms, views, d, ws, lds);
    else
        raster_tile<G, MODE, MULTI, TILE, false, false>(geoms, views, d, ws, lds);
}

// ------------------------------------------------------ in-order replay

struct ReplayEntry {
    Tri t[4];
    uint32_t alive, prol, q;   // q: quad code (row << 16 | column)
};

// A candidate (triangle covering a deferred pixel) recorded for the in-order
// fold: quad code, slot | prol | next-in-list, depth, validity.
struct Cand {
    uint32_t ij;
    uint32_t meta;   // bits 0-15: next record (0xffff = end), 16-17: slot, 18: prol
    float d, tv;
};
constexpr int kCandPool = kFallbackSortCap * 4 / (int)sizeof(Cand);   // records sharing the sort buffer
static_assert(kCandPool < 0xffff, "candidate links are 16-bit");

// Sorts L[0, n) ascending in place, one block: a bitonic network in its
// all-ascending form (the first step of each merge compares e with its mirror
// e ^ (k - 1), the later ones with e ^ jj, always putting the smaller value at
// the lower index), so the positions from n up to the next power of two act
// as +inf and their comparisons are skipped.  Global memory written by the
// block's threads is read back by other threads of the block after each
// barrier.
__device__ void block_sort_global(uint32_t* L, uint32_t n) {
    uint32_t np2 = 1;
    while (np2 < n) np2 <<= 1;
    for (uint32_t k = 2; k <= np2; k <<= 1)
        for (uint32_t jj = k >> 1; jj > 0; jj >>= 1) {
            const uint32_t mate = jj == (k >> 1) ? k - 1 : jj;
            for (uint32_t e = threadIdx.x; e < n; e += blockDim.x) {
                const uint32_t p = e ^ mate;
                if (p > e && p < n) {
                    const uint32_t a = L[e], b = L[p];
                    if (a > b) { L[e] = b; L[p] = a; }
                }
            }
            __syncthreads();
        }
}

// Deferred pixels of one tile and source, in the reference's traversal order.
// Fast path: the block rasterises the source's bin in parallel and appends
// every candidate covering a deferred pixel of the current pixel range to
// that pixel's list in LDS; each pixel then folds its own candidates in
// ascending (quad, slot) order.  When a range's lists overflow the pool, the
// range is split (down to a single pixel); only a single pixel with more
// candidates than the pool falls back to sorting the bin (in LDS, or in place
// in the entry list when it is longer than the LDS buffer; only this block
// reads this bin after the raster) and scanning it in order.
template <class G>
__device__ void replay_source(const G& g, uint32_t* L, uint32_t n, int tx0, int ty0, int out_w, int out_h,
                              bool mine, int px, int py, const uint8_t* dmask, uint32_t* sorted, ReplayEntry* rec,
                              uint32_t* pool_n, FoldState& fs, const RasterWS& ws, const BatchDims& d, uint32_t vs) {
    const int tid = threadIdx.x;
    // vertex (ii, jj) of the neighbourhood of a quad whose work item keeps
    // the vertex window vb (null: none) starting at row r0, column c0: from
    // the window (the same bits as vertex()), else evaluated
    auto kept_or_eval = [&](const float* vb, int r0, int c0, int ii, int jj) -> float3 {
        const int rr = ii - r0, cc = jj - c0;
        if (vb && rr >= 0 && rr <= kBinQY && cc >= 0 && cc <= kBinQX) return kept_vertex(vb, rr, cc);
        return vertex(g, ii, jj);
    };
    Cand* pool = reinterpret_cast<Cand*>(sorted);
    int* head = reinterpret_cast<int*>(rec);
    const int pme = (py - ty0) * kTile + (px - tx0);
    fold_init(fs);
    int lo = 0, span = kTile * kTile;
    bool scan_all = false;
    while (lo < kTile * kTile) {
        const int hi = min(lo + span, kTile * kTile);
        head[tid] = -1;
        if (tid == 0) *pool_n = 0u;
        __syncthreads();
        for (uint32_t e = tid; e < n; e += 256) {
            const uint32_t q = L[e];
            int i, j;
            unpack_ij(q, i, j);
            const float* vb = kept_block(ws, d, vs, q);
            const int r0 = i - i % kBinQY, c0 = j - j % kBinQX;
            auto vtx = [&](int ii, int jj) { return kept_or_eval(vb, r0, c0, ii, jj); };
            quad_tris(g, i, j, vtx, out_w, out_h, [&](int k, Tri& Tr, bool prol) {
                bool have_tv = false;   // the validity, evaluated for the first candidate
                int xa = max(Tr.xmin, tx0), xb = min(Tr.xmax, tx0 + kTile - 1);
                int ya = max(Tr.ymin, ty0), yb = min(Tr.ymax, ty0 + kTile - 1);
                if (is_finite(Tr.A0) && is_finite(Tr.A1) && is_finite(Tr.B0) && is_finite(Tr.B1) &&
                    is_finite(Tr.C0) && is_finite(Tr.C1) && is_finite(Tr.den))
                    tri_tight(Tr, xa, xb, ya, yb);
                for (int y = ya; y <= yb; ++y)
                    for (int x = xa; x <= xb; ++x) {
                        const int p = (y - ty0) * kTile + (x - tx0);
                        if (p < lo || p >= hi || !dmask[p]) continue;
                        float n1, n2;
                        tri_num(Tr, x, y, n1, n2);
                        if (tri_surely_outside(Tr, n1, n2)) continue;
                        float l1, l2, l3;
                        if (!tri_cover(Tr, n1, n2, l1, l2, l3)) continue;
                        if (!have_tv) {
                            Tr.tv = tri_validity(Tr, g.rescale);
                            have_tv = true;
                        }
                        const uint32_t r = atomicAdd(pool_n, 1u);
                        if (r >= (uint32_t)kCandPool) continue;
                        const int nx = atomicExch(&head[p], (int)r);
                        Cand& C = pool[r];
                        C.ij = q;
                        C.meta = (uint32_t)(nx < 0 ? 0xffff : nx) | ((uint32_t)k << 16) | ((prol ? 1u : 0u) << 18);
                        C.d = tri_depth(Tr, l1, l2, l3);
                        C.tv = Tr.tv;
                    }
            });
        }
        __syncthreads();
        const bool overflow = *pool_n > (uint32_t)kCandPool;
        __syncthreads();
        if (overflow) {
            if (span > 1) {
                span = max(1, span / 4);   // retry this range in smaller pieces
                continue;
            }
            scan_all = true;               // one pixel with more candidates than the pool
            break;
        }
        if (mine && pme >= lo && pme < hi) {
            bool first = true;
            uint64_t last = 0;
            while (true) {
                uint64_t best = ~0ull;
                int bi = -1;
                for (int r = head[pme]; r >= 0;) {
                    const Cand& C = pool[r];
                    const uint64_t key = ((uint64_t)C.ij << 2) | ((C.meta >> 16) & 3u);
                    if ((first || key > last) && key < best) { best = key; bi = r; }
                    const uint32_t nx = C.meta & 0xffffu;
                    r = nx == 0xffffu ? -1 : (int)nx;
                }
                if (bi < 0) break;
                const Cand& C = pool[bi];
                fold_step(fs, C.d, C.tv, (C.meta >> 18) & 1u, C.ij, (int)((C.meta >> 16) & 3u));
                last = best;
                first = false;
            }
        }
        __syncthreads();
        lo = hi;
        span = min(span * 2, kTile * kTile);
    }
    if (!scan_all) return;
    // the remaining deferred pixels (from lo on) scan the whole bin in order
    mine = mine && pme >= lo;
    if (mine) fold_init(fs);
    // overflow: sort the bin (bitonic, ascending quad code = traversal order) and scan it
    const uint32_t* S = sorted;
    if (n <= (uint32_t)kFallbackSortCap) {
        uint32_t np2 = 1;
        while (np2 < n) np2 <<= 1;
        for (uint32_t e = tid; e < np2; e += 256) sorted[e] = e < n ? L[e] : 0xffffffffu;
        __syncthreads();
        for (uint32_t k = 2; k <= np2; k <<= 1)
            for (uint32_t jj = k >> 1; jj > 0; jj >>= 1) {
                for (uint32_t e = tid; e < np2; e += 256) {
                    const uint32_t p = e ^ jj;
                    if (p > e) {
                        const uint32_t a = sorted[e], b = sorted[p];
                        const bool asc = (e & k) == 0;
                        if ((a > b) == asc) { sorted[e] = b; sorted[p] = a; }
                    }
                }
                __syncthreads();
            }
    } else {
        block_sort_global(L, n);
        S = L;
    }
    for (uint32_t b = 0; b < n; b += kFallbackChunk) {
        if (tid < kFallbackChunk && b + tid < n) {
            const uint32_t q = S[b + tid];
            int i, j;
            unpack_ij(q, i, j);
            Quad Q;
            const float* vb = kept_block(ws, d, vs, q);
            const int r0 = i - i % kBinQY, c0 = j - j % kBinQX;
            auto vtx = [&](int ii, int jj) { return kept_or_eval(vb, r0, c0, ii, jj); };
            quad_build(Q, g, i, j, vtx, out_w, out_h);
            ReplayEntry& R = rec[tid];
            for (int k = 0; k < 4; ++k) R.t[k] = Q.t[k];
            R.alive = Q.alive; R.prol = Q.prol; R.q = q;
        }
        __syncthreads();
        if (mine) {
            const uint32_t m = min((uint32_t)kFallbackChunk, n - b);
            for (uint32_t e = 0; e < m; ++e) {
                const ReplayEntry& R = rec[e];
                for (int k = 0; k < 4; ++k) {
                    if (!(R.alive & (1u << k))) continue;
                    const Tri& Tr = R.t[k];
                    if (px < Tr.xmin || px > Tr.xmax || py < Tr.ymin || py > Tr.ymax) continue;
                    float l1, l2, l3;
                    if (!tri_pixel(Tr, px, py, l1, l2, l3)) continue;
                    fold_step(fs, tri_depth(Tr, l1, l2, l3), Tr.tv, (R.prol >> k) & 1u, R.q, k);
                }
            }
        }
        __syncthreads();
    }
}

// Deferred tiles [first, n_deferred): one block per tile folds every source
// in order and blends (the tiles before `first` take the per-source pair of
// kernels below).
template <class G, int MODE>
__global__ void __launch_bounds__(256) k_fallback(const G* __restrict__ geoms, const ViewDesc* __restrict__ views,
                                                  BatchDims d, RasterWS ws, uint32_t first) {
    __shared__ uint32_t sorted[kFallbackSortCap];
    __shared__ ReplayEntry rec[kFallbackChunk];
    __shared__ uint8_t dmask[kTile * kTile];
    __shared__ uint32_t pool_n[1];   // candidate records
    const int tid = threadIdx.x;
    const uint32_t ndef = ws.status[1] ? 0u : ws.status[0];
    for (uint32_t ti = first + blockIdx.x; ti < ndef; ti += gridDim.x) {
        const uint32_t T = ws.deferred_tiles[ti];
        const int v = find_view(views, d.nviews, T);
        const ViewDesc& vd = views[v];
        const G* gv = geoms + (size_t)v * d.nsrc;
        const int tile = (int)(T - vd.tile_base);
        const int edge = 1 << d.tile_shift;
        // the tile in sub-tiles of kTile x kTile pixels, a thread per pixel
        // (each folds the whole bin of the tile, clipped to its sub-tile)
        const int nsub = edge / kTile;
        for (int sub = 0; sub < nsub * nsub; ++sub) {
        const int tx0 = (tile % vd.tiles_x) * edge + (sub % nsub) * kTile;
        const int ty0 = (tile / vd.tiles_x) * edge + (sub / nsub) * kTile;
        const int px = tx0 + (tid % kTile), py = ty0 + (tid / kTile);
        const bool inside = px < vd.w && py < vd.h;
        const size_t o = inside ? (size_t)py * vd.w + px : 0;
        const bool mine = inside && ws.deferred[vd.px_base + o];
        dmask[tid] = mine ? 1 : 0;
        // a sub-tile of a larger tile may hold no deferred pixel (the barrier
        // also publishes dmask)
        if (!__syncthreads_or(mine ? 1 : 0)) continue;
        BlendState st;
        float3 rc = make_float3(0.f, 0.f, 0.f);
        float rd = __builtin_inff(), rs = 0.f;
        for (int s = 0; s < d.nsrc; ++s) {
            const G& g = gv[s];
            const size_t bin = bin_index(d, T, (uint32_t)s);
            const uint32_t n = ws.counts[bin];
            FoldState fs;
            replay_source(g, ws.lists + ws.offsets[bin], n, tx0, ty0, vd.w, vd.h, mine, px, py, dmask, sorted, rec,
                          pool_n, fs, ws, d, (uint32_t)(v * d.nsrc + s));
            __syncthreads();
            if (mine) {
                float3 c = make_float3(0.f, 0.f, 0.f);
                float dep = __builtin_inff(), shape = 0.f;
                if (fs.slot >= 0) {
                    float dd, sh;
                    int i, j;
                    unpack_ij(fs.ij, i, j);
                    resolve<false>(g, i, j, fs.slot, px, py, c, dd, sh, vd.w, vd.h, nullptr);
                    dep = fs.new_d;
                    shape = fs.shape;
                }
                if (MODE == MODE_RAW) {
                    rc = c; rd = dep; rs = shape;
                } else if (s == 0) {
                    blend_first(st, c, dep, shape);
                } else {
                    blend_step(st, c, dep, shape, vd.blend_exp, vd.blend_inv);
                }
            }
        }
        if (mine) write_pixel<MODE>(vd, o, st, rc, rd, rs);
        __syncthreads();
        }
    }
}

// The first d.rbuf_tiles deferred tiles, sources in parallel: a block per
// (tile, source) folds that source's bin for the tile's deferred pixels (the
// same replay_source and resolve as k_fallback) and stores each pixel's
// colour, depth and validity in ws.rbuf; k_fallback_blend then blends them in
// source order.  A tile's chain of sources is the replay's critical path when
// few tiles are deferred.
template <class G>
__global__ void __launch_bounds__(256) k_fallback_src(const G* __restrict__ geoms,
                                                      const ViewDesc* __restrict__ views, BatchDims d, RasterWS ws) {
    __shared__ uint32_t sorted[kFallbackSortCap];
    __shared__ ReplayEntry rec[kFallbackChunk];
    __shared__ uint8_t dmask[kTile * kTile];
    __shared__ uint32_t pool_n[1];
    const int tid = threadIdx.x;
    const uint32_t ndef = ws.status[1] ? 0u : min(ws.status[0], d.rbuf_tiles);
    const int edge = 1 << d.tile_shift;
    const int nsub = edge / kTile;
    for (uint32_t job = blockIdx.x; job < ndef * (uint32_t)d.nsrc; job += gridDim.x) {
        const uint32_t ti = job / (uint32_t)d.nsrc;
        const int s = (int)(job % (uint32_t)d.nsrc);
        const uint32_t T = ws.deferred_tiles[ti];
        const int v = find_view(views, d.nviews, T);
        const ViewDesc& vd = views[v];
        const G& g = geoms[(size_t)v * d.nsrc + s];
        const int tile = (int)(T - vd.tile_base);
        float* out = ws.rbuf + ((size_t)ti * d.nsrc + s) * ((size_t)edge * edge) * 5;
        for (int sub = 0; sub < nsub * nsub; ++sub) {
            const int tx0 = (tile % vd.tiles_x) * edge + (sub % nsub) * kTile;
            const int ty0 = (tile / vd.tiles_x) * edge + (sub / nsub) * kTile;
            const int px = tx0 + (tid % kTile), py = ty0 + (tid / kTile);
            const bool inside = px < vd.w && py < vd.h;
            const size_t o = inside ? (size_t)py * vd.w + px : 0;
            const bool mine = inside && ws.deferred[vd.px_base + o];
            dmask[tid] = mine ? 1 : 0;
            if (!__syncthreads_or(mine ? 1 : 0)) continue;
            const size_t bin = bin_index(d, T, (uint32_t)s);
            FoldState fs;
            replay_source(g, ws.lists + ws.offsets[bin], ws.counts[bin], tx0, ty0, vd.w, vd.h, mine, px, py, dmask,
                          sorted, rec, pool_n, fs, ws, d, (uint32_t)(v * d.nsrc + s));
            if (mine) {
                float3 c = make_float3(0.f, 0.f, 0.f);
                float dep = __builtin_inff(), shape = 0.f;
                if (fs.slot >= 0) {
                    float dd, sh;
                    int i, j;
                    unpack_ij(fs.ij, i, j);
                    resolve<false>(g, i, j, fs.slot, px, py, c, dd, sh, vd.w, vd.h, nullptr);
                    dep = fs.new_d;
                    shape = fs.shape;
                }
                float* r = out + (size_t)(sub * kTile * kTile + tid) * 5;
                r[0] = c.x; r[1] = c.y; r[2] = c.z; r[3] = dep; r[4] = shape;
            }
            __syncthreads();
        }
    }
}

template <class G>
__global__ void __launch_bounds__(256) k_fallback_blend(const ViewDesc* __restrict__ views, BatchDims d,
                                                        RasterWS ws) {
    const int tid = threadIdx.x;
    const uint32_t ndef = ws.status[1] ? 0u : min(ws.status[0], d.rbuf_tiles);
    const int edge = 1 << d.tile_shift;
    const int nsub = edge / kTile;
    for (uint32_t ti = blockIdx.x; ti < ndef; ti += gridDim.x) {
        const uint32_t T = ws.deferred_tiles[ti];
        const int v = find_view(views, d.nviews, T);
        const ViewDesc& vd = views[v];
        const int tile = (int)(T - vd.tile_base);
        for (int sub = 0; sub < nsub * nsub; ++sub) {
            const int px = (tile % vd.tiles_x) * edge + (sub % nsub) * kTile + (tid % kTile);
            const int py = (tile / vd.tiles_x) * edge + (sub / nsub) * kTile + (tid / kTile);
            if (px >= vd.w || py >= vd.h) continue;
            const size_t o = (size_t)py * vd.w + px;
            if (!ws.deferred[vd.px_base + o]) continue;
            BlendState st;
            for (int s = 0; s < d.nsrc; ++s) {
                const float* r = ws.rbuf + (((size_t)ti * d.nsrc + s) * ((size_t)edge * edge) +
                                            (size_t)(sub * kTile * kTile + tid)) * 5;
                const float3 c = make_float3(r[0], r[1], r[2]);
                if (s == 0) blend_first(st, c, r[3], r[4]);
                else blend_step(st, c, r[3], r[4], vd.blend_exp, vd.blend_inv);
            }
            write_pixel<MODE_BLEND>(vd, o, st, make_float3(0.f, 0.f, 0.f), 0.f, 0.f);
        }
    }
}

template <class G, int MODE>
hipError_t launch_raster(const G* geoms, const ViewDesc* views, const BatchDims& d, const RasterWS& ws,
                         hipStream_t s) {
    const dim3 blocks(8u * ((d.ntiles + 7u) / 8u)), nb(kTileBig * kTileBig), nt(kTile * kTile);
    const bool big = d.tile_shift == 5;
    if (d.nsrc > kRasterGroup) {
        if (big) hipLaunchKernelGGL((k_raster<G, MODE, true, kTileBig, false>), blocks, nb, 0, s, geoms, views, d, ws);
        else hipLaunchKernelGGL((k_raster<G, MODE, true, kTile, false>), blocks, nt, 0, s, geoms, views, d, ws);
    } else if (MODE == MODE_BLEND && d.settle) {
        constexpr bool SETTLE = MODE == MODE_BLEND;   // a raw launch set never settles
        if (big) hipLaunchKernelGGL((k_raster<G, MODE, false, kTileBig, SETTLE>), blocks, nb, 0, s, geoms, views, d, ws);
        else hipLaunchKernelGGL((k_raster<G, MODE, false, kTile, SETTLE>), blocks, nt, 0, s, geoms, views, d, ws);
    } else {
        if (big) hipLaunchKernelGGL((k_raster<G, MODE, false, kTileBig, false>), blocks, nb, 0, s, geoms, views, d, ws);
        else hipLaunchKernelGGL((k_raster<G, MODE, false, kTile, false>), blocks, nt, 0, s, geoms, views, d, ws);
    }
    return hipGetLastError();
}

template <class G, int MODE>
hipError_t launch_replay(const G* geoms, const ViewDesc* views, const BatchDims& d, const RasterWS& ws,
                         hipStream_t s) {
    const unsigned fb_blocks = d.ntiles < (uint32_t)kFallbackBlocks ? d.ntiles : (uint32_t)kFallbackBlocks;
    uint32_t first = 0;
    if (MODE == MODE_BLEND && d.nsrc > 1 && d.rbuf_tiles > 0) {
        // the first rbuf_tiles deferred tiles: sources in parallel, then the blend
        const uint64_t jobs = (uint64_t)d.rbuf_tiles * (uint64_t)d.nsrc;
        const unsigned sb = (unsigned)(jobs < (uint64_t)kFallbackBlocks * 4 ? jobs : (uint64_t)kFallbackBlocks * 4);
        hipLaunchKernelGGL((k_fallback_src<G>), dim3(sb), dim3(256), 0, s, geoms, views, d, ws);
        const unsigned bb = d.rbuf_tiles < (uint32_t)kFallbackBlocks ? d.rbuf_tiles : (uint32_t)kFallbackBlocks;
        hipLaunchKernelGGL((k_fallback_blend<G>), dim3(bb), dim3(256), 0, s, views, d, ws);
        first = d.rbuf_tiles;
    }
    hipLaunchKernelGGL((k_fallback<G, MODE>), dim3(fb_blocks), dim3(256), 0, s, geoms, views, d, ws, first);
    return hipGetLastError();
}

template hipError_t launch_bin<PairGeom>(const PairGeom*, const ViewDesc*, const BatchDims&, const RasterWS&,
                                         hipStream_t);
template hipError_t launch_bin<ArrayGeom>(const ArrayGeom*, const ViewDesc*, const BatchDims&, const RasterWS&,
                                          hipStream_t);
template hipError_t launch_raster<PairGeom, MODE_BLEND>(const PairGeom*, const ViewDesc*, const BatchDims&,
                                                        const RasterWS&, hipStream_t);
template hipError_t launch_raster<ArrayGeom, MODE_RAW>(const ArrayGeom*, const ViewDesc*, const BatchDims&,
                                                       const RasterWS&, hipStream_t);
template hipError_t launch_replay<PairGeom, MODE_BLEND>(const PairGeom*, const ViewDesc*, const BatchDims&,
                                                        const RasterWS&, hipStream_t);
template hipError_t launch_replay<ArrayGeom, MODE_RAW>(const ArrayGeom*, const ViewDesc*, const BatchDims&,
                                                       const RasterWS&, hipStream_t);

}  // namespace rvs_k
