// vs_pre.hip — input pre-steps around the filter: reprojection of a depth
// frame into another camera (z_tdrcc) and the crop of depths outside the
// object volume (god). One thread per pixel; both are memory-bound streams.
#include "vs_device.hpp"
#include "vs_launch.hpp"

namespace vs {

// z_tdrcc_Transform_Depth_to_Rgb_Camera_Coordinates (z_yooji_object_scanner.cpp:2429-2476)
// with convert_pixel_coord (z_yooji_matrix_rgbd.cpp:101-118): back-project the
// source pixel (CKvYooji_Intrinsics::back_project, z_yooji_camera_parameters.cpp:104-108),
// transform into the destination camera (CKvYooji_Extrinsics::transform, :678-685),
// project (:89-96), ROUNDF, and keep the nearest source depth per destination
// pixel. The value written is the source depth itself, so the operator is
// exact on integer millimetres; the nearest one is an atomic minimum on its
// bit pattern (non-negative values order like their bits), which makes the
// result independent of the order of the writes.
template <class T>
__device__ __forceinline__ float depth_value(T v);
template <>
__device__ __forceinline__ float depth_value<uint16_t>(uint16_t v) { return depth_m(v); }
template <>
__device__ __forceinline__ float depth_value<float>(float v) { return v; }
__device__ __forceinline__ uint32_t depth_key(uint16_t v) { return v; }
__device__ __forceinline__ uint32_t depth_key(float v) { return __float_as_uint(v); }

// One workgroup per 64x16 source tile, four rows a wave. The tile's pixels
// land in a small window of the destination (its source scale plus the
// parallax of its depths), so their minima are taken in LDS first and only one
// atomic per destination pixel and tile goes to memory: those atomics, not the
// arithmetic, bound the launch (1920x1080 into 1280x720: one per source pixel
// 32 us, per tile and destination pixel 11). An upright pair's window is wide
// and flat; one of more than kWinUpright pixels goes to memory directly (its
// scale keeps the pixels apart, and a wave's lie in one row: 640x480 into
// 1280x960 8.8 us, 10.9 through the window). A rolled pair's is as high as wide,
// or a column, and a wave's pixels lie in as many rows: it is taken in up to
// kWinBands bands of rows of kWin pixels (640x480 rolled by 90 degrees into
// equal scale 17.4 us to memory directly and 8.5 so, by 45 into 960x960 19.3 and
// 13.4, by 45 into 1280x1280 20.0 and 16.4).
constexpr int kRepW = 64, kRepH = 16, kRepRows = 4;  // 256 threads
constexpr int kWin = 4096, kWinBands = 4, kWinUpright = 3072;
template <class T>
__global__ __launch_bounds__(256) void k_depth_reproject(const T *__restrict__ src, int sw, int sh, Mat16f Ks4,
                                                         Mat16f Tds, uint32_t *key, int dw, int dh) {
    __shared__ uint32_t win[kWin];
    __shared__ int box[4][4];  // per wave: min x, min y, -max x, -max y
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int x0 = blockIdx.x * kRepW + lane, y0 = blockIdx.y * kRepH + wave * kRepRows;
    const float *Ks = Ks4.m, *Kd = Ks4.m + 4, *M = Tds.m;
    T raw[kRepRows];
    int tx[kRepRows], ty[kRepRows];
#pragma unroll
    for (int r = 0; r < kRepRows; ++r) {
        const int y = y0 + r;
        raw[r] = x0 < sw && y < sh ? ldg(src, (size_t)y * sw + x0) : T(0);
    }
    int b[4] = {0x7FFFFFFF, 0x7FFFFFFF, 0x7FFFFFFF, 0x7FFFFFFF};
#pragma unroll
    for (int r = 0; r < kRepRows; ++r) {
        const float td = depth_value<T>(raw[r]);
        tx[r] = -1;
        ty[r] = 0;
        if (td > 0.0f) {
            const float x = (float)x0, y = (float)(y0 + r);
            const f3 p = {td * (x - Ks[2]) / Ks[0], td * (y - Ks[3]) / Ks[1], td};
            const f3 q = transform(M, p);
            const float u = Kd[0] * q.x / q.z + Kd[2], v = Kd[1] * q.y / q.z + Kd[3];
            int ix, iy;
            if (roundf_ref(u, ix) && roundf_ref(v, iy) && ix >= 0 && ix <= dw - 1 && iy >= 0 && iy <= dh - 1) {
                tx[r] = ix;
                ty[r] = iy;
                b[0] = min(b[0], ix);
                b[1] = min(b[1], iy);
                b[2] = min(b[2], -ix);
                b[3] = min(b[3], -iy);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) b[k] = min(b[k], __shfl_xor(b[k], off, 64));
        if (lane == 0) box[wave][k] = b[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) b[k] = min(min(box[0][k], box[1][k]), min(box[2][k], box[3][k]));
    if (b[0] == 0x7FFFFFFF) return;  // no pixel of the tile lands
    const int w = -b[2] - b[0] + 1, h = -b[3] - b[1] + 1;
    const bool rolled = 2 * h > w;
    if (w * h > (rolled ? kWinBands * kWin : kWinUpright)) {  // w and h at most 8192
#pragma unroll
        for (int r = 0; r < kRepRows; ++r)
            if (tx[r] >= 0) atomicMin(key + (size_t)ty[r] * dw + tx[r], depth_key(raw[r]));
        return;
    }
    const int rows = min(h, kWin / w);  // per band; a tall window's w is below kWin
    for (int y0 = b[1]; y0 < b[1] + h; y0 += rows) {
        const int n = w * min(rows, b[1] + h - y0);
        for (int i = threadIdx.x; i < n; i += 256) win[i] = 0xFFFFFFFFu;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRepRows; ++r) {
            const int i = (ty[r] - y0) * w + tx[r] - b[0];
            if (tx[r] >= 0 && i >= 0 && i < n) atomicMin(&win[i], depth_key(raw[r]));
        }
        __syncthreads();
        const auto flush = [&](int x, int y, uint32_t k) {
            if (k != 0xFFFFFFFFu) atomicMin(key + (size_t)(y0 + y) * dw + b[0] + x, k);
        };
        if (rolled)  // rows of few pixels
            for (int i = threadIdx.x; i < n; i += 256) flush(i % w, i / w, win[i]);
        else
            for (int y = wave; y < n / w; y += 4)
                for (int x = lane; x < w; x += 64) flush(x, y, win[y * w + x]);
        __syncthreads();
    }
}

__device__ __forceinline__ void key_to_depth(uint32_t k, uint16_t &out) { out = k == 0xFFFFFFFFu ? 0 : (uint16_t)k; }
__device__ __forceinline__ void key_to_depth(uint32_t k, float &out) {
    out = k == 0xFFFFFFFFu ? 0.0f : __uint_as_float(k);
}
template <class T>
__global__ void k_depth_key_finish(uint32_t *key, T *dst, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const uint32_t k = ldg(key, i);
        T v;
        key_to_depth(k, v);
        stg(dst, i, v);
        if (k != 0xFFFFFFFFu) stg(key, i, 0xFFFFFFFFu);  // empty for the next frame
    }
}

template <class T>
static void reproject_t(const void *src, int sw, int sh, const float Ks[4], const float Kd[4], const float M[16],
                        uint32_t *key, void *dst, int dw, int dh, hipStream_t s) {
    Mat16f k{}, m{};
    for (int i = 0; i < 4; ++i) {
        k.m[i] = Ks[i];
        k.m[4 + i] = Kd[i];
    }
    for (int i = 0; i < 16; ++i) m.m[i] = M[i];
    const size_t nd = (size_t)dw * dh;
    hipLaunchKernelGGL(k_depth_reproject<T>, dim3((unsigned)((sw + kRepW - 1) / kRepW), (unsigned)((sh + kRepH - 1) / kRepH)),
                       dim3(256), 0, s, (const T *)src, sw, sh, k, m, key, dw, dh);
    hipLaunchKernelGGL(k_depth_key_finish<T>, dim3((unsigned)std::min<size_t>((nd + 255) / 256, 4096)), dim3(256), 0, s,
                       key, (T *)dst, nd);
}
void launch_depth_reproject(int is_float, const void *src, int sw, int sh, const float Ks[4], const float Kd[4],
                            const float T[16], uint32_t *key, void *dst, int dw, int dh, hipStream_t s) {
    if (is_float)
        reproject_t<float>(src, sw, sh, Ks, Kd, T, key, dst, dw, dh, s);
    else
        reproject_t<uint16_t>(src, sw, sh, Ks, Kd, T, key, dst, dw, dh, s);
}

// god_Get_Object_Depth (z_yooji_object_extractor.cpp:357-410), its cube test:
// back-project the integer pixel with its depth, map it to the world with
// the camera-to-world transform (CKvYooji_Extrinsics::transform_inv,
// z_yooji_camera_parameters.cpp:687-694) and zero the depth when the point
// leaves [origin, origin + size] on any axis. T_cg is the session's FP32
// pose inverse unless one is given.
template <class T>
__global__ void k_depth_crop(const SessParams *__restrict__ SP, T *depth, int w, int h, Mat16f K4, Mat16f Tcg,
                             int use_session_pose) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= w * h) return;
    const SessParams &P = SP[0];
    const float td = depth_value<T>(depth[i]);
    const float *K = K4.m;
    const float *M = use_session_pose ? P.st->T_cg_f : Tcg.m;
    const f3 p = {td * ((float)(i % w) - K[2]) / K[0], td * ((float)(i / w) - K[3]) / K[1], td};
    const f3 g = transform(M, p);
    // size_cube = dim * voxel (z_yooji_object_extractor.cpp:388), per axis
    const float sx = (float)P.vdim[0] * P.voxel, sy = (float)P.vdim[1] * P.voxel, sz = (float)P.vdim[2] * P.voxel;
    if (g.x < P.origin[0] || g.x > P.origin[0] + sx || g.y < P.origin[1] || g.y > P.origin[1] + sy ||
        g.z < P.origin[2] || g.z > P.origin[2] + sz)
        depth[i] = T(0);
}
void launch_depth_crop(const SessParams *P, int is_float, void *depth, int w, int h, const float K[4],
                       const float *Tcg, hipStream_t s) {
    Mat16f k{}, m{};
    for (int i = 0; i < 4; ++i) k.m[i] = K[i];
    if (Tcg)
        for (int i = 0; i < 16; ++i) m.m[i] = Tcg[i];
    const unsigned blocks = (unsigned)(((size_t)w * h + 255) / 256);
    if (is_float)
        hipLaunchKernelGGL(k_depth_crop<float>, dim3(blocks), dim3(256), 0, s, P, (float *)depth, w, h, k, m,
                           Tcg ? 0 : 1);
    else
        hipLaunchKernelGGL(k_depth_crop<uint16_t>, dim3(blocks), dim3(256), 0, s, P, (uint16_t *)depth, w, h, k, m,
                           Tcg ? 0 : 1);
}

}  // namespace vs
