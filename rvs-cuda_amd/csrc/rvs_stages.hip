// rvs_stages.hip -- element-wise stages: decode, reproject, blend step, encode.
#include <hip/hip_runtime.h>

#include "rvs_stages.h"

namespace rvs_k {

using namespace rvs_dev;

// Writers of four horizontally adjacent decoded pixels (Y, U, V before the
// colour scale): the float colour map, the resident plane of 16-bit integers
// (exact for even sizes and codes below 2^14, whose upsampled chroma is a
// multiple of 1/4), or the resident plane of floats.
struct ColorOut {
    float* p;
    float cs;
    __device__ void put(size_t o, float y, float u, float v) const {
        p[3 * o] = y * cs; p[3 * o + 1] = u * cs; p[3 * o + 2] = v * cs;
    }
    __device__ void put4(size_t o, const float (&y)[4], const float (&u)[4], const float (&v)[4]) const {
        float t[12];
#pragma unroll
        for (int k = 0; k < 4; ++k) { t[3 * k] = y[k] * cs; t[3 * k + 1] = u[k] * cs; t[3 * k + 2] = v[k] * cs; }
        __builtin_memcpy(p + 3 * o, t, sizeof t);
    }
};
struct PackedOut {
    ushort4* p;
    __device__ void put(size_t o, float y, float u, float v) const {
        p[o] = make_ushort4((unsigned short)y, (unsigned short)(u * 4.f), (unsigned short)(v * 4.f), 0);
    }
    __device__ void put4(size_t o, const float (&y)[4], const float (&u)[4], const float (&v)[4]) const {
#pragma unroll
        for (int k = 0; k < 4; ++k) put(o + k, y[k], u[k], v[k]);
    }
};
struct FloatOut {
    float4* p;
    __device__ void put(size_t o, float y, float u, float v) const { p[o] = make_float4(y, u, v, 0.f); }
    __device__ void put4(size_t o, const float (&y)[4], const float (&u)[4], const float (&v)[4]) const {
#pragma unroll
        for (int k = 0; k < 4; ++k) put(o + k, y[k], u[k], v[k]);
    }
};

// read_color_YUV -> resizeImage + mergeFrame (image_loading.cpp:74-145), any
// size: a thread per pixel.
template <class Out>
__global__ void k_color(const void* y, const void* u, const void* v, int u8, int w, int h, Out out) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int r = blockIdx.y;
    if (x >= w || r >= h) return;
    PairGeom g;
    g.sw = w; g.sh = h; g.py = y; g.pu = u; g.pv = v; g.color_u8 = u8; g.col = nullptr; g.colq = nullptr;
    const float3 c = color_raw(g, r, x);
    out.put((size_t)r * w + x, c.x, c.y, c.z);
}

// The same for even sizes: a thread takes four pixels of two rows, whose chroma
// needs three samples of two rows of each plane (color_raw's even form: the
// sums and halves are exact, so the order does not matter).  Bound by HBM: 3 B
// read and 8 (packed) or 12 B written per pixel.  A thread per pixel took up to
// nine 1- or 2-byte loads each: 4096x2048 10-bit to the packed plane 61 -> 29 us,
// 2048x2048 to the float map 25.7 -> 17.1 us.
template <typename T, class Out>
__global__ void __launch_bounds__(256) k_color_even(const T* __restrict__ Y, const T* __restrict__ U,
                                                    const T* __restrict__ V, int w, int h, Out out) {
    const int x = 4 * (int)(blockIdx.x * 64 + (threadIdx.x & 63));
    const int r = 2 * (int)(blockIdx.y * 4 + (threadIdx.x >> 6));
    if (x >= w || r >= h) return;
    const int cw = w / 2, ch = h / 2, cx = x / 2, cy = r / 2;
    const int x1 = min(cx + 1, cw - 1), x2 = min(cx + 2, cw - 1);
    const size_t r0 = (size_t)cy * cw, r1 = (size_t)min(cy + 1, ch - 1) * cw;
    // chroma of the upper row (even: its own samples) and the lower one (the
    // mean with the next), at columns x .. x + 3
    float c[2][2][4];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const T* P = p ? V : U;
        const float a0 = (float)P[r0 + cx], a1 = (float)P[r0 + x1], a2 = (float)P[r0 + x2];
        const float b0 = (float)P[r1 + cx], b1 = (float)P[r1 + x1], b2 = (float)P[r1 + x2];
        const float up[4] = {a0, (a0 + a1) * 0.5f, a1, (a1 + a2) * 0.5f};
        const float lo[4] = {b0, (b0 + b1) * 0.5f, b1, (b1 + b2) * 0.5f};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            c[p][0][k] = up[k];
            c[p][1][k] = (up[k] + lo[k]) * 0.5f;
        }
    }
#pragma unroll
    for (int row = 0; row < 2; ++row) {
        const size_t o = (size_t)(r + row) * w + x;
        if (x + 4 <= w) {
            T q[4];
            __builtin_memcpy(q, Y + o, sizeof q);
            const float l[4] = {(float)q[0], (float)q[1], (float)q[2], (float)q[3]};
            out.put4(o, l, c[0][row], c[1][row]);
        } else {   // the last two columns
            out.put(o, (float)Y[o], c[0][row][0], c[1][row][0]);
            out.put(o + 1, (float)Y[o + 1], c[0][row][1], c[1][row][1]);
        }
    }
}

template <class Out>
hipError_t launch_color(const void* y, const void* u, const void* v, int u8, int w, int h, Out out, hipStream_t s) {
    if (((w | h) & 1) == 0) {
        const dim3 grid((w + 255) / 256, (h + 7) / 8);
        if (u8)
            hipLaunchKernelGGL((k_color_even<uint8_t, Out>), grid, dim3(256), 0, s, (const uint8_t*)y,
                               (const uint8_t*)u, (const uint8_t*)v, w, h, out);
        else
            hipLaunchKernelGGL((k_color_even<uint16_t, Out>), grid, dim3(256), 0, s, (const uint16_t*)y,
                               (const uint16_t*)u, (const uint16_t*)v, w, h, out);
    } else {
        hipLaunchKernelGGL(k_color<Out>, dim3((w + 255) / 256, h), dim3(256), 0, s, y, u, v, u8, w, h, out);
    }
    return hipGetLastError();
}

// read_depth_YUV -> formatDepth (image_loading.cpp:147-213).
__global__ void k_decode_depth(const void* raw, int u8, size_t n, float scale, float znear, float zfar,
                               int has_invalid, float* __restrict__ out) {
    const size_t i = 4 * ((size_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n) return;
    if (i + 4 <= n) {
        uint32_t q[4];
        if (u8) {
            uint8_t t[4];
            __builtin_memcpy(t, (const uint8_t*)raw + i, sizeof t);
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = t[k];
        } else {
            uint16_t t[4];
            __builtin_memcpy(t, (const uint16_t*)raw + i, sizeof t);
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = t[k];
        }
        float d[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) d[k] = decode_depth_raw(q[k], scale, znear, zfar, has_invalid);
        __builtin_memcpy(out + i, d, sizeof d);
        return;
    }
    for (size_t k = i; k < n; ++k) out[k] = decode_depth_raw(load_plane(raw, u8, k), scale, znear, zfar, has_invalid);
}

// SynthesizedView::computeBasicMode stage (a) (SynthesizedView.cpp:315-331).
__global__ void k_reproject(PairGeom g, float* __restrict__ uv, float* __restrict__ vd) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = blockIdx.y;
    if (j >= g.sw || i >= g.sh) return;
    const float3 r = vertex(g, i, j);
    const size_t o = (size_t)i * g.sw + j;
    uv[2 * o] = r.x; uv[2 * o + 1] = r.y;
    vd[o] = r.z;
}

// BlendedViewSimple::blendBasicMode on whole maps.
__global__ void k_blend_step(float* acc_c, float* acc_q, float* acc_d, float* acc_v, uint8_t* acc_m,
                             const float* __restrict__ c, const float* __restrict__ d,
                             const float* __restrict__ shape, size_t n, float a, float a_inv, int first) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float3 cv = make_float3(c[3 * i], c[3 * i + 1], c[3 * i + 2]);
    BlendState s;
    if (first) {
        blend_first(s, cv, d[i], shape[i]);
        s.mask = s.mask ? 255 : 0;
    } else {
        s.c = make_float3(acc_c[3 * i], acc_c[3 * i + 1], acc_c[3 * i + 2]);
        s.q = acc_q[i]; s.d = acc_d[i]; s.v = acc_v[i]; s.mask = acc_m[i];
        blend_step(s, cv, d[i], shape[i], a, a_inv);
    }
    acc_c[3 * i] = s.c.x; acc_c[3 * i + 1] = s.c.y; acc_c[3 * i + 2] = s.c.z;
    acc_q[i] = s.q; acc_d[i] = s.d; acc_v[i] = s.v;
    acc_m[i] = (uint8_t)(s.mask ? (s.mask == 1 ? 1 : 255) : 0);
}

// write_color (image_writing.cpp:142-203) for the 2x2 block (bx, by).
template <typename T>
__device__ inline void encode_block(const float* __restrict__ color, int w, int bx, int by, unsigned maxv,
                                    T* __restrict__ Y, T* __restrict__ U, T* __restrict__ V) {
    const int hw = w / 2;
    uint32_t su = 0, sv = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int x = 2 * bx + (k & 1), y = 2 * by + (k >> 1);
        const size_t o = (size_t)y * w + x;
        const float* c = color + 3 * o;
        Y[o] = (T)quantize_u32(c[0], maxv);
        su += (uint32_t)(T)quantize_u32(c[1], maxv);
        sv += (uint32_t)(T)quantize_u32(c[2], maxv);
    }
    U[(size_t)by * hw + bx] = (T)((su + 2) >> 2);
    V[(size_t)by * hw + bx] = (T)((sv + 2) >> 2);
}

// One thread per 2x2 block.
template <typename T>
__global__ void k_encode(const float* __restrict__ color, int w, int h, unsigned maxv, T* __restrict__ Y,
                         T* __restrict__ U, T* __restrict__ V) {
    const int bx = blockIdx.x * blockDim.x + threadIdx.x;
    const int by = blockIdx.y;
    if (bx >= w / 2 || by >= h / 2) return;
    encode_block(color, w, bx, by, maxv, Y, U, V);
}

// Batch of views (grid.z = view); views without output planes are skipped.
// The planes encode ecol at the view's size (ew x eh).
__global__ void k_encode_views(const ViewDesc* __restrict__ views, const uint8_t* __restrict__ tile_enc) {
    const ViewDesc& vd = views[blockIdx.z];
    const int bx = blockIdx.x * blockDim.x + threadIdx.x;
    const int by = blockIdx.y;
    if (!vd.y || bx >= vd.ew / 2 || by >= vd.eh / 2) return;
    // tiles without holes or deferred pixels were encoded by the raster pass
    if (tile_enc && vd.enc_raster &&
        (tile_enc[vd.tile_base + (uint32_t)(((2 * by) >> vd.tile_shift) * vd.tiles_x + ((2 * bx) >> vd.tile_shift))] & 1))
        return;
    const unsigned maxv = (1u << vd.bitdepth) - 1u;
    if (vd.bitdepth <= 8)
        encode_block(vd.ecol, vd.ew, bx, by, maxv, (uint8_t*)vd.y, (uint8_t*)vd.u, (uint8_t*)vd.v);
    else
        encode_block(vd.ecol, vd.ew, bx, by, maxv, (uint16_t*)vd.y, (uint16_t*)vd.u, (uint16_t*)vd.v);
}

// Oversampled views: colour (w x h) resized to the view's size (ew x eh).
__global__ void k_resize_views(const ViewDesc* __restrict__ views) {
    const ViewDesc& vd = views[blockIdx.z];
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
    if (vd.ecol == vd.color || x >= vd.ew || y >= vd.eh) return;
    const float3 c = resize_linear_px(vd.color, vd.w, vd.h, vd.ew, vd.eh, x, y, vd.rtab, vd.rtab + vd.ew);
    float* o = vd.ecol + 3 * ((size_t)y * vd.ew + x);
    o[0] = c.x; o[1] = c.y; o[2] = c.z;
}

// The same for one colour image (the stage entry point; taps: dw column
// entries, then dh row entries).
__global__ void k_resize_color(const float* __restrict__ src, int sw, int sh, float* __restrict__ dst, int dw,
                               int dh, const int2* __restrict__ taps) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
    if (x >= dw || y >= dh) return;
    const float3 c = resize_linear_px(src, sw, sh, dw, dh, x, y, taps, taps + dw);
    float* o = dst + 3 * ((size_t)y * dw + x);
    o[0] = c.x; o[1] = c.y; o[2] = c.z;
}

hipError_t launch_resize_views(const ViewDesc* views, int nviews, int max_ew, int max_eh, hipStream_t s) {
    hipLaunchKernelGGL(k_resize_views, dim3((max_ew + 255) / 256, max_eh, nviews), dim3(256), 0, s, views);
    return hipGetLastError();
}

hipError_t launch_resize_color(const float* src, int sw, int sh, float* dst, int dw, int dh, const int2* taps,
                               hipStream_t s) {
    hipLaunchKernelGGL(k_resize_color, dim3((dw + 255) / 256, dh), dim3(256), 0, s, src, sw, sh, dst, dw, dh, taps);
    return hipGetLastError();
}

hipError_t launch_decode_color(const void* y, const void* u, const void* v, int u8, int w, int h, float cs,
                               float* out, hipStream_t s) {
    return launch_color(y, u, v, u8, w, h, ColorOut{out, cs}, s);
}

hipError_t launch_prep_color(const void* y, const void* u, const void* v, int u8, int w, int h, int packed,
                             void* out, hipStream_t s) {
    if (packed) return launch_color(y, u, v, u8, w, h, PackedOut{(ushort4*)out}, s);
    return launch_color(y, u, v, u8, w, h, FloatOut{(float4*)out}, s);
}

hipError_t launch_decode_depth(const void* raw, int u8, size_t n, float scale, float znear, float zfar,
                               int has_invalid, float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_decode_depth, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, s, raw, u8, n, scale, znear,
                       zfar, has_invalid, out);
    return hipGetLastError();
}

hipError_t launch_reproject(const PairGeom& g, float* uv, float* vd, hipStream_t s) {
    hipLaunchKernelGGL(k_reproject, dim3((g.sw + 255) / 256, g.sh), dim3(256), 0, s, g, uv, vd);
    return hipGetLastError();
}

hipError_t launch_blend_step(float* acc_c, float* acc_q, float* acc_d, float* acc_v, uint8_t* acc_m, const float* c,
                             const float* d, const float* shape, size_t n, float a, int first, hipStream_t s) {
    const float a_inv = 1.0f / a;
    hipLaunchKernelGGL(k_blend_step, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, acc_c, acc_q, acc_d, acc_v,
                       acc_m, c, d, shape, n, a, a_inv, first);
    return hipGetLastError();
}

hipError_t launch_encode(const float* color, int w, int h, int bitdepth, void* y, void* u, void* v, hipStream_t s) {
    const unsigned maxv = (1u << bitdepth) - 1u;
    const dim3 grid((w / 2 + 255) / 256, h / 2);
    if (bitdepth <= 8)
        hipLaunchKernelGGL(k_encode<uint8_t>, grid, dim3(256), 0, s, color, w, h, maxv, (uint8_t*)y, (uint8_t*)u,
                           (uint8_t*)v);
    else
        hipLaunchKernelGGL(k_encode<uint16_t>, grid, dim3(256), 0, s, color, w, h, maxv, (uint16_t*)y, (uint16_t*)u,
                           (uint16_t*)v);
    return hipGetLastError();
}

hipError_t launch_encode_views(const ViewDesc* views, int nviews, int max_w, int max_h, const uint8_t* tile_enc,
                               hipStream_t s) {
    const dim3 grid((max_w / 2 + 255) / 256, max_h / 2, nviews);
    hipLaunchKernelGGL(k_encode_views, grid, dim3(256), 0, s, views, tile_enc);
    return hipGetLastError();
}

}  // namespace rvs_k
