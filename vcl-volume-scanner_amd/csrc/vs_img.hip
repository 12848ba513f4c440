// vs_img.hip — image stages of the fusion step: bilateral depth filter (A2-A3),
// depth pyramid (A4) and the vertex/normal-map operator (A6-A7).
//
// Launch shape: one 256-thread workgroup (4 wave64) per 32 x 8 output tile,
// tiles of every session of a batch concatenated in one work list, so a
// single launch serves the whole batch. Rows of 32 pixels keep global loads
// and stores coalesced (a wave covers two 128-byte rows of a float image).
#include "vs_device.hpp"
#include "vs_launch.hpp"

namespace vs {

constexpr int kHalo = 3;  // largest bilateral radius supported

// The 2R+1 x 2R+1 window of one pixel (tile coordinates of the centre): sum
// of w and of w (d - c), and whether a tap is 0 (raw_depth is never below, and
// bit patterns of such values order as the values do: one three-operand
// minimum per two taps instead of a compare and a mask operation each: radius 3
// at 1280x720 with the rest of the frame's preparation 35.5 -> 33.3 us, 64
// sessions at radius 2 6.13 -> 6.10 ms a step). The radius is a
// compile-time constant (1, 2 or 3, the radii a session accepts), so the
// loops unroll. The spatial products g[i] g[j] come from the session
// parameters (uniform, in scalar registers) and the range weight is one
// hardware base-2 exponential of the pre-scaled squared difference.
template <int R, int TW>
__device__ __forceinline__ void bil_window(const float (*tile)[TW], int cy, int cx, const float *wij, float c,
                                           float nk, float &s, float &t, bool &zero) {
    constexpr int r = R, n = 2 * R + 1;
    uint32_t least = 0xFFFFFFFFu;
#pragma unroll
    for (int i = -r; i <= r; ++i) {
#pragma unroll
        for (int j = -r; j <= r; ++j) {
            const float p = tile[cy + i][cx + j];
            least = min(least, __float_as_uint(p));
            const float d = p - c;
            const float w = wij[(i + r) * n + (j + r)] * __builtin_amdgcn_exp2f((d * d) * nk);
            t = fmaf(w, d, t);
            s += w;
        }
    }
    zero = least == 0u;
}

// Bilateral filter of the raw uint16 mm frame into pyramid level 0 (metres).
// Reference: d_bilateral_filter (z_yooji_cuda_img_proc.cu:103-141): weight
// g[i] g[j] exp(-(d - c)^2 / (2 sigma_r^2)), output 0 if any tap <= 0. Taps are
// point samples with clamp-to-edge addressing; the sum is accumulated about
// the centre value (c + sum w (d - c) / sum w), which is the same weighted mean
// with a smaller rounding error.
__global__ __launch_bounds__(kTileThreads) void k_bilateral(const SessParams *__restrict__ SP,
                                                            const WorkItem *__restrict__ work, int force,
                                                            float *out) {
    __shared__ float tile[kTileH + 2 * kHalo][kTileW + 2 * kHalo];
    const WorkItem wi = work[blockIdx.x];
    const SessParams &P = SP[wi.sess];
    const LevelDesc &L = P.lev[0];
    if (tile_out(L, wi.tile) || !(force || P.st->active)) return;
    const int W = L.W, H = L.H;
    const int x0 = (wi.tile % L.tiles_x) * kTileW, y0 = (wi.tile / L.tiles_x) * kTileH;
    const int R = P.bil_radius;
    constexpr int TW = kTileW + 2 * kHalo, TH = kTileH + 2 * kHalo;
    for (int i = threadIdx.x; i < TW * TH; i += kTileThreads) {
        int ly = i / TW, lx = i - ly * TW;
        int gx = min(max(x0 + lx - kHalo, 0), W - 1);
        int gy = min(max(y0 + ly - kHalo, 0), H - 1);
        tile[ly][lx] = raw_depth(P, (size_t)gy * W + gx);
    }
    __syncthreads();
    const int lx = threadIdx.x % kTileW, ly = threadIdx.x / kTileW;
    const int x = x0 + lx, y = y0 + ly;
    if (x >= W || y >= H) return;
    const float c = tile[ly + kHalo][lx + kHalo];
    float s = 0.0f, t = 0.0f;
    bool zero = false;
    const float nk = P.bil_nk;
    const int cy = ly + kHalo, cx = lx + kHalo;
    const auto store = [&](float v) {
        stg(P.filt[0], (size_t)y * W + x, v);
        if (out) stg(out, (size_t)y * W + x, v);
    };
    // session creation accepts radii 1..3 only; each radius has its own
    // complete path to the store
    switch (R) {
    case 1:
        bil_window<1, TW>(tile, cy, cx, P.bil_w, c, nk, s, t, zero);
        store(zero ? 0.0f : c + t / s);
        break;
    case 2:
        bil_window<2, TW>(tile, cy, cx, P.bil_w, c, nk, s, t, zero);
        store(zero ? 0.0f : c + t / s);
        break;
    case 3:
        bil_window<3, TW>(tile, cy, cx, P.bil_w, c, nk, s, t, zero);
        store(zero ? 0.0f : c + t / s);
        break;
    }
}

// One pyramid step, level l-1 -> l: the separable [1 4 6 4 1]^2/256 blur of
// level l-1 sampled at (2i+1, 2j+1), 0 where the 5x5 window leaves the image.
// Reference: cpdd_Construct_Pyramids_Down_Depth + sdg5 + ddh
// (z_yooji_image_processor.cpp:368-407, 857-940, 567-596). Only the decimated
// pixels are computed.
__global__ __launch_bounds__(kTileThreads) void k_pyr_down(const SessParams *__restrict__ SP,
                                                           const WorkItem *__restrict__ work, int l, int force) {
    const WorkItem wi = work[blockIdx.x];
    const SessParams &P = SP[wi.sess];
    const LevelDesc &L = P.lev[l];
    if (l >= P.levels || tile_out(L, wi.tile) || !(force || P.st->active)) return;
    const int Wi = P.lev[l - 1].W, Hi = P.lev[l - 1].H;
    const int x = (wi.tile % L.tiles_x) * kTileW + threadIdx.x % kTileW;
    const int y = (wi.tile / L.tiles_x) * kTileH + threadIdx.x / kTileW;
    if (x >= L.W || y >= L.H) return;
    const int i = 2 * x + 1, j = 2 * y + 1;
    float v = 0.0f;
    if (i >= 2 && i <= Wi - 3 && j >= 2 && j <= Hi - 3) {
        const float *in = P.filt[l - 1];
        float h[5];
#pragma unroll
        for (int r = 0; r < 5; ++r) {
            const size_t row = (size_t)(j + r - 2) * Wi;
            h[r] = 1.0f * ldg(in, row + i - 2) + 1.0f * ldg(in, row + i + 2) + 4.0f * ldg(in, row + i - 1) +
                   4.0f * ldg(in, row + i + 1) + 6.0f * ldg(in, row + i);
        }
        v = (1.0f * h[0] + 1.0f * h[4] + 4.0f * h[1] + 4.0f * h[3] + 6.0f * h[2]) / (16.0f * 16.0f);
    }
    stg(P.filt[l], (size_t)y * L.W + x, v);
}

// Levels 1 and 2 in one launch: a workgroup computes the level-1 pixels around
// its 32x8 level-2 tile in LDS (the row sums of the blur first, each used by up
// to three level-1 rows), writes the 64x16 of them that are its own, and
// decimates them once more. Values as k_pyr_down's, operation for operation.
// The halo repeats a quarter of level 1; a launch and its gap go (640x480 scan
// 419 -> 416 us; with 4 waves a tile, walking its rows one after another, 419).
constexpr int kP1W = 2 * kTileW + 3, kP1H = 2 * kTileH + 3;  // level-1 region: 67 x 19
constexpr int kP0H = 2 * kP1H + 3;                           // level-0 rows of the row sums: 41
template <int THREADS>
__global__ __launch_bounds__(THREADS) void k_pyr_down2(const SessParams *__restrict__ SP,
                                                            const WorkItem *__restrict__ work, int force) {
    __shared__ float rows[kP0H][kP1W], l1[kP1H][kP1W];
    const WorkItem wi = work[blockIdx.x];
    const SessParams &P = SP[wi.sess];
    const LevelDesc &L = P.lev[2];
    if (P.levels < 3 || tile_out(L, wi.tile) || !(force || P.st->active)) return;
    const int W0 = P.lev[0].W, H0 = P.lev[0].H, W1 = P.lev[1].W, H1 = P.lev[1].H;
    const int tx = wi.tile % L.tiles_x, ty = wi.tile / L.tiles_x;
    const int x1 = 2 * tx * kTileW - 1, y1 = 2 * ty * kTileH - 1;  // level-1 region's corner
    const int y0 = 2 * y1 - 1;                                     // first level-0 row: 2 y1 + 1 - 2
    const float *in = P.filt[0];
#pragma unroll
    for (int k0 = 0; k0 < kP0H * kP1W; k0 += THREADS) {
        const int k = k0 + threadIdx.x;
        if (k >= kP0H * kP1W) break;
        const int r = k / kP1W, c = k - r * kP1W;
        const int i = 2 * (x1 + c) + 1, y = y0 + r;
        float h = 0.0f;
        if (i >= 2 && i <= W0 - 3 && y >= 0 && y < H0) {
            const size_t row = (size_t)y * W0;
            h = 1.0f * ldg(in, row + i - 2) + 1.0f * ldg(in, row + i + 2) + 4.0f * ldg(in, row + i - 1) +
                4.0f * ldg(in, row + i + 1) + 6.0f * ldg(in, row + i);
        }
        rows[r][c] = h;
    }
    __syncthreads();
    // the last tile of a row or column also owns the odd column or row of level 1
    const int xe = tx == L.tiles_x - 1 ? W1 : min(W1, 2 * (tx + 1) * kTileW);
    const int ye = ty == L.tiles_y - 1 ? H1 : min(H1, 2 * (ty + 1) * kTileH);
#pragma unroll
    for (int k0 = 0; k0 < kP1H * kP1W; k0 += THREADS) {
        const int k = k0 + threadIdx.x;
        if (k >= kP1H * kP1W) break;
        const int r = k / kP1W, c = k - r * kP1W;
        const int x = x1 + c, y = y1 + r, i = 2 * x + 1, j = 2 * y + 1;
        float v = 0.0f;
        if (i >= 2 && i <= W0 - 3 && j >= 2 && j <= H0 - 3) {
            const float *h = &rows[2 * r][c];  // level-0 row j - 2
            v = (1.0f * h[0] + 1.0f * h[4 * kP1W] + 4.0f * h[kP1W] + 4.0f * h[3 * kP1W] + 6.0f * h[2 * kP1W]) /
                (16.0f * 16.0f);
        }
        l1[r][c] = v;
        if (r >= 1 && c >= 1 && x < xe && y < ye) stg(P.filt[1], (size_t)y * W1 + x, v);
    }
    __syncthreads();
    const int lx = threadIdx.x % kTileW, ly = threadIdx.x / kTileW;
    const int x = tx * kTileW + lx, y = ty * kTileH + ly;
    if (ly >= kTileH || x >= L.W || y >= L.H) return;
    const int i = 2 * x + 1, j = 2 * y + 1;
    float v = 0.0f;
    if (i >= 2 && i <= W1 - 3 && j >= 2 && j <= H1 - 3) {
        float h[5];
#pragma unroll
        for (int r = 0; r < 5; ++r) {
            const float *q = l1[2 * ly + r] + 2 * lx;  // level-1 row j + r - 2, columns i - 2 .. i + 2
            h[r] = 1.0f * q[0] + 1.0f * q[4] + 4.0f * q[1] + 4.0f * q[3] + 6.0f * q[2];
        }
        v = (1.0f * h[0] + 1.0f * h[4] + 4.0f * h[1] + 4.0f * h[3] + 6.0f * h[2]) / (16.0f * 16.0f);
    }
    stg(P.filt[2], (size_t)y * L.W + x, v);
}

// Vertex and normal maps of pyramid level l (AoS float3, -100 invalid).
// Reference: cpm_Compute_Point_Map / enm_Estimate_Normal_Map
// (z_yooji_image_processor.cpp:119-227): n = normalize(dz/dx, dz/dy, -1) from
// central differences, 1-pixel border skipped, |dx| or |dy| < 1e-7 rejected,
// and grazing normals (-n_z <= cos 60 deg) invalidate vertex and normal.
struct VnPixel {
    f3 c, n;                       // vertex; normal (when `normal`)
    bool valid, normal, grazing;   // depth > 0; accepted normal; rejected as grazing
};
__device__ __forceinline__ VnPixel vn_pixel(const float *D, const float *K, int W, int H, int x, int y) {
    auto vert = [&](int xx, int yy, f3 &v) -> bool {
        float d = ldg(D, (size_t)yy * W + xx);
        if (d <= 0.0f) return false;
        v = {d * ((float)xx - K[2]) / K[0], d * ((float)yy - K[3]) / K[1], d};
        return true;
    };
    VnPixel r;
    r.normal = r.grazing = false;
    r.valid = vert(x, y, r.c);
    if (r.valid && x >= 1 && x < W - 1 && y >= 1 && y < H - 1) {
        f3 x1, x2, y1, y2;
        if (vert(x - 1, y, x1) && vert(x + 1, y, x2) && vert(x, y - 1, y1) && vert(x, y + 1, y2)) {
            float dx = x2.x - x1.x, dy = y2.y - y1.y;
            if (fabsf(dx) >= 1.0e-7f && fabsf(dy) >= 1.0e-7f) {
                float gx = (x2.z - x1.z) / dx, gy = (y2.z - y1.z) / dy;
                float nn = sqrtf(gx * gx + gy * gy + 1.0f);
                r.n = {gx / nn, gy / nn, -1.0f / nn};
                r.grazing = -r.n.z <= 0.5f;
                r.normal = !r.grazing;
            }
        }
    }
    return r;
}
// Pixel t of the caller's maps: the vertex unless it is gone, the normal if
// there is one.
__device__ __forceinline__ void put_vn(const VnPixel &r, bool gone, float *vtx, float *nrm, size_t t) {
    const bool v = r.valid && !gone;
    stg(vtx, 3 * t + 0, v ? r.c.x : -100.f);
    stg(vtx, 3 * t + 1, v ? r.c.y : -100.f);
    stg(vtx, 3 * t + 2, v ? r.c.z : -100.f);
    stg(nrm, 3 * t + 0, r.normal ? r.n.x : -100.f);
    stg(nrm, 3 * t + 1, r.normal ? r.n.y : -100.f);
    stg(nrm, 3 * t + 2, r.normal ? r.n.z : -100.f);
}
// Without `inv`: every pixel evaluated on the input vertex map (the
// order-independent form). With it (the reference loop's in-place order,
// below): one bit per pixel, rows of `nw` 64-bit words, set where the loop
// invalidates the vertex.
__global__ __launch_bounds__(kTileThreads) void k_vnmap(const SessParams *__restrict__ SP,
                                                        const WorkItem *__restrict__ work, int l, float *vtx,
                                                        float *nrm, const unsigned long long *inv, int nw) {
    const WorkItem wi = work[blockIdx.x];
    const SessParams &P = SP[wi.sess];
    const LevelDesc &L = P.lev[l];
    const int W = L.W, H = L.H;
    const int x = (wi.tile % L.tiles_x) * kTileW + threadIdx.x % kTileW;
    const int y = (wi.tile / L.tiles_x) * kTileH + threadIdx.x / kTileW;
    if (x >= W || y >= H) return;
    VnPixel r = vn_pixel(P.filt[l], L.K, W, H, x, y);
    bool gone = r.grazing;
    if (inv) {
        auto bit = [&](int xx, int yy) -> bool {
            return xx >= 0 && yy >= 0 && ((ldg(inv, (size_t)yy * nw + (xx >> 6)) >> (xx & 63)) & 1ull);
        };
        gone = bit(x, y);
        r.normal &= !(bit(x - 1, y) || bit(x, y - 1));
    }
    put_vn(r, gone, vtx, nrm, (size_t)y * W + x);
}

// The reference CPU loop's in-place order (enm_Estimate_Normal_Map,
// z_yooji_image_processor.cpp:155-227, which writes the grazing invalidation
// into the vertex map it is still reading): pixels after a grazing pixel in
// raster order see its vertex as -100. A grazing pixel is invalidated only
// when neither its left nor its upper neighbour was:
//     inv(i, j) = c(i, j) & !inv(i, j-1) & !inv(i-1, j)
// where c marks the grazing pixels of the order-independent form. A grazing
// pixel that is not invalidated keeps its vertex (its normal was never
// computed), and a pixel whose left or upper neighbour is invalidated loses
// its normal. Three launches: the bits of c, the recurrence on bits, the maps.
// Only the recurrence is serial, one row after another, so it is kept to one
// wave working on bits alone. (With that wave also reading the maps back and
// resolving each row's runs one at a time in one lane it had taken 3.2 ms a
// level: frame preparation and the maps of three levels of a 640x480 frame,
// alone, 9.31 -> 0.19 ms.)
//
// Where the bits are, a row's vn_words(W) words of 64 pixels, bit 0 the leftmost:
//   calls on the session's own stream, which follow one another: in a scratch
//   of the session's, where the ordered bits of a row replace its bits of c;
//   calls on a caller's stream, of which several may run at once (MAP): in the
//   caller's vertex map, until the last launch writes it. Row y's 12 W bytes
//   begin with its bits of c, followed by the ordered bits of row y - 1; the
//   last launch's workgroup for a row finds both in the row that it alone
//   overwrites, and takes the recurrence's step for its row once more. (640x480
//   frame preparation 54.0 us with the scratch, 55.0 so.) A map is aligned to
//   4 bytes, hence the half words.
template <bool MAP>
struct VnBits {
    static __device__ __forceinline__ uint32_t *row(uint32_t *bits, int nw, int W, int y) {
        return bits + (size_t)y * (MAP ? 3 * W : 2 * nw);
    }
};
__device__ __forceinline__ unsigned long long ld_word(const uint32_t *row, int k) {
    return (unsigned long long)ldg(row, 2 * k) | (unsigned long long)ldg(row, 2 * k + 1) << 32;
}
__device__ __forceinline__ void st_word(uint32_t *row, int k, unsigned long long v) {
    stg(row, 2 * k, (uint32_t)v);
    stg(row, 2 * k + 1, (uint32_t)(v >> 32));
}

// One wave per 64 pixels of a row: word k of row y = bits of c.
template <bool MAP>
__global__ __launch_bounds__(kTileThreads) void k_vn_graze(const SessParams *__restrict__ SP, int l, uint32_t *bits,
                                                           int nw) {
    const SessParams &P = SP[0];
    const LevelDesc &L = P.lev[l];
    const int item = blockIdx.x * (kTileThreads / 64) + (threadIdx.x >> 6);
    const int y = item / nw, k = item - y * nw;
    if (y >= L.H) return;
    const int x = k * 64 + (threadIdx.x & 63);
    const bool c = x < L.W && vn_pixel(P.filt[l], L.K, L.W, L.H, x, y).grazing;
    const unsigned long long m = __ballot(c);
    if ((threadIdx.x & 63) == 0) st_word(VnBits<MAP>::row(bits, nw, L.W, y), k, m);
}

// One step of the recurrence by one wave, lane k holding words k * N .. k * N +
// N - 1 of a row: up, the ordered bits of the row above, becomes this row's.
// Along a row, a run of r = c & ~inv(row above) is invalidated at every other
// pixel from its first: adding the first bits of the runs that start at even
// columns to r (one addition over the whole row) clears exactly those runs,
// which tells the runs' parities apart. The addition's carries cross lanes by
// the generate / propagate masks of the wave.
template <int N>
__device__ __forceinline__ void vn_order_row(const unsigned long long *c, unsigned long long *up, int lane) {
    unsigned long long r[N], sum[N];
#pragma unroll
    for (int q = 0; q < N; ++q) r[q] = c[q] & ~up[q];
    // last bit of the previous lane's words
    unsigned prev = __shfl_up((unsigned)(r[N - 1] >> 63), 1, 64);
    if (lane == 0) prev = 0u;
    bool carry = false, prop = true;
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const unsigned long long first = r[q] & ~((r[q] << 1) | prev);
        const unsigned long long s = r[q] + (first & 0x5555555555555555ull);
        sum[q] = s + (carry ? 1ull : 0ull);
        carry = s < r[q] || sum[q] < s;
        prop &= sum[q] == ~0ull;
        prev = (unsigned)(r[q] >> 63);
    }
    const unsigned long long G = __ballot(carry), Pr = __ballot(prop);
    bool in = ((((G << 1) + Pr) ^ Pr) >> lane) & 1ull;  // carry into this lane's first word
#pragma unroll
    for (int q = 0; q < N; ++q) {
        sum[q] += in ? 1ull : 0ull;
        in = in && sum[q] == 0ull;
        up[q] = r[q] & ((~sum[q] & 0x5555555555555555ull) | (sum[q] & 0xAAAAAAAAAAAAAAAAull));
    }
}

// The recurrence over all rows by one wave: a row's ordered bits in place, or
// (MAP) those of the row above behind its bits of c. Bound: a chain of ~25
// dependent instructions per row; the rows' bits are loaded kAhead rows ahead
// of their use.
template <int N, bool MAP>
__global__ __launch_bounds__(64) void k_vn_order(uint32_t *bits, int nw, int W, int H) {
    constexpr int kAhead = 16;
    const int lane = threadIdx.x;
    unsigned long long up[N], nxt[kAhead][N];
#pragma unroll
    for (int q = 0; q < N; ++q) up[q] = 0ull;
    auto fetch = [&](int row0) {
#pragma unroll
        for (int a = 0; a < kAhead; ++a)
#pragma unroll
            for (int q = 0; q < N; ++q) {
                const int k = lane * N + q;
                nxt[a][q] = (k < nw && row0 + a < H) ? ld_word(VnBits<MAP>::row(bits, nw, W, row0 + a), k) : 0ull;
            }
    };
    fetch(0);
    for (int row0 = 0; row0 < H; row0 += kAhead) {
        unsigned long long cur[kAhead][N];
#pragma unroll
        for (int a = 0; a < kAhead; ++a)
#pragma unroll
            for (int q = 0; q < N; ++q) cur[a][q] = nxt[a][q];
        fetch(row0 + kAhead);
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            if (!MAP) vn_order_row<N>(cur[a], up, lane);
#pragma unroll
            for (int q = 0; q < N; ++q) {
                const int k = lane * N + q;
                if (k < nw && row0 + a < H)
                    st_word(VnBits<MAP>::row(bits, nw, W, row0 + a), MAP ? nw + k : k, up[q]);
            }
            if (MAP) vn_order_row<N>(cur[a], up, lane);
        }
    }
}

// The maps from bits in the vertex map, one workgroup per row: its ordered bits and the row above's into
// LDS by the first wave, then the row's pixels over what they were read from.
// A thread per pixel of the row while the workgroup holds them.
template <int N>
__global__ __launch_bounds__(1024) void k_vnmap_rows(const SessParams *__restrict__ SP, int l, float *vtx,
                                                              float *nrm, int nw) {
    __shared__ unsigned long long here[64 * N], above[64 * N];
    const SessParams &P = SP[0];
    const LevelDesc &L = P.lev[l];
    const int W = L.W, y = blockIdx.x;
    unsigned long long c[N], up[N];
    if (threadIdx.x < 64) {
        const uint32_t *row = VnBits<true>::row((uint32_t *)vtx, nw, W, y);
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const int k = threadIdx.x * N + q;
            c[q] = k < nw ? ld_word(row, k) : 0ull;
            up[q] = k < nw ? ld_word(row, nw + k) : 0ull;
        }
    }
    int x = threadIdx.x;
    VnPixel r{};
    if (x < W) r = vn_pixel(P.filt[l], L.K, W, L.H, x, y);  // its loads in flight with the bits
    if (threadIdx.x < 64) {
#pragma unroll
        for (int q = 0; q < N; ++q) above[threadIdx.x * N + q] = up[q];
        vn_order_row<N>(c, up, threadIdx.x);
#pragma unroll
        for (int q = 0; q < N; ++q) here[threadIdx.x * N + q] = up[q];
    }
    __syncthreads();
    const auto bit = [](const unsigned long long *b, int i) -> bool { return i >= 0 && ((b[i >> 6] >> (i & 63)) & 1ull); };
    while (x < W) {
        r.normal &= !(bit(here, x - 1) || bit(above, x));
        put_vn(r, bit(here, x), vtx, nrm, (size_t)y * W + x);
        x += blockDim.x;
        if (x < W) r = vn_pixel(P.filt[l], L.K, W, L.H, x, y);
    }
}

// Copies the caller's device-resident frames into the sessions' raw-frame
// buffers (in each session's depth units, copied as 16-bit halves): one
// launch for a whole batch (blockIdx.y = session of the chunk), 16-byte
// vector loads/stores where the frame size allows.
__global__ __launch_bounds__(256) void k_gather_depth(const SessParams *__restrict__ SP, DepthChunk ch) {
    const int s = blockIdx.y;
    if (s >= ch.n) return;
    const SessParams &P = SP[ch.slot[s]];
    const size_t npx = (size_t)P.lev[0].W * P.lev[0].H * (P.raw_f32 ? 2 : 1);
    const uint16_t *src = ch.src[s];
    uint16_t *dst = (uint16_t *)const_cast<void *>(P.raw);
    const bool vec = ((npx & 7) == 0) && ((((uintptr_t)src) & 15) == 0);
    if (vec) {
        const uint4 *s4 = reinterpret_cast<const uint4 *>(src);
        uint4 *d4 = reinterpret_cast<uint4 *>(dst);
        for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < npx / 8; i += (size_t)gridDim.x * blockDim.x)
            d4[i] = s4[i];
    } else {
        for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < npx; i += (size_t)gridDim.x * blockDim.x)
            dst[i] = src[i];
    }
}

// Image buffers of a new session: empty pyramid, images and textures, model
// maps at the -100 sentinel, the reprojection's keys empty, in one launch (a
// fill per buffer had cost an open ~12 launches). Every buffer is 256-byte
// aligned and padded.
__global__ __launch_bounds__(256) void k_session_init(const SessParams *__restrict__ SP, uint32_t *keys) {
    const SessParams &P = SP[0];
    const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
    const auto fill = [&](void *p, size_t bytes, uint32_t v) {
        for (size_t i = i0; i < (bytes + 15) / 16; i += step) stg((vs_u4 *)p, i, vs_u4{v, v, v, v});
    };
    fill(keys, (size_t)P.lev[0].W * P.lev[0].H * 4, 0xFFFFFFFFu);
    for (int l = 0; l < kMaxLevels; ++l) {
        const size_t n = (size_t)P.lev[l].W * P.lev[l].H;
        fill(P.filt[l], n * 4, 0u);
        fill(P.mvn[l], (n + 1) * 2 * sizeof(MapXYZ), 0xC2C80000u);  // -100.0f
        fill(P.mimg[l], n, 0u);
        if (P.mtex[l]) fill(P.mtex[l], n * 3, 0u);
    }
}
void launch_session_init(const SessParams *P, size_t npx, uint32_t *keys, hipStream_t s) {
    const size_t blocks = std::min<size_t>((npx + 255) / 256, 2048);
    hipLaunchKernelGGL(k_session_init, dim3((unsigned)blocks), dim3(256), 0, s, P, keys);
}

void launch_gather_depth(const SessParams *P, const DepthChunk &ch, hipStream_t s) {
    if (ch.n > 0) hipLaunchKernelGGL(k_gather_depth, dim3(64, ch.n), dim3(256), 0, s, P, ch);
}

void launch_bilateral(const SessParams *P, const WorkItem *work, int n, int force, float *out, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_bilateral, dim3(n), dim3(kTileThreads), 0, s, P, work, force, out);
}
void launch_pyramid(const SessParams *P, const WorkItem *const work[kMaxLevels], const int n[kMaxLevels], int levels,
                    bool pair, int force, hipStream_t s) {
    if (levels == 3 && pair) {
        if (n[2] <= 0) return;
        // 16 waves a tile against 4, us in a step: 75 tiles 7.5 / 11.0, 300 8.4 / 11.4,
        // 600 11.8 / 12.5, 975 13.9 / 13.2, 1200 16.7 / 13.7, 4800 44.1 / 35.6
        if (n[2] <= 768)
            hipLaunchKernelGGL(k_pyr_down2<1024>, dim3(n[2]), dim3(1024), 0, s, P, work[2], force);
        else
            hipLaunchKernelGGL(k_pyr_down2<kTileThreads>, dim3(n[2]), dim3(kTileThreads), 0, s, P, work[2], force);
        return;
    }
    for (int l = 1; l < levels; ++l)
        if (n[l] > 0) hipLaunchKernelGGL(k_pyr_down, dim3(n[l]), dim3(kTileThreads), 0, s, P, work[l], l, force);
}
void launch_vnmap(const SessParams *P, const WorkItem *work, int n, int l, float *vtx, float *nrm, hipStream_t s) {
    if (n > 0)
        hipLaunchKernelGGL(k_vnmap, dim3(n), dim3(kTileThreads), 0, s, P, work, l, vtx, nrm,
                           (const unsigned long long *)nullptr, 0);
}
void launch_vnmap_inplace(const SessParams *P, const WorkItem *work, int n, int l, int W, int H, void *scratch,
                          float *vtx, float *nrm, hipStream_t s) {
    if (n <= 0) return;
    const int nw = vn_words(W);  // at most 128 (frames are at most 8192 wide)
    const size_t per = kTileThreads / 64, grid = ((size_t)nw * H + per - 1) / per;
    uint32_t *bits = (uint32_t *)(scratch ? scratch : vtx);
    if (scratch) {
        hipLaunchKernelGGL(k_vn_graze<false>, dim3((unsigned)grid), dim3(kTileThreads), 0, s, P, l, bits, nw);
        if (nw <= 64)
            hipLaunchKernelGGL((k_vn_order<1, false>), dim3(1), dim3(64), 0, s, bits, nw, W, H);
        else
            hipLaunchKernelGGL((k_vn_order<2, false>), dim3(1), dim3(64), 0, s, bits, nw, W, H);
        hipLaunchKernelGGL(k_vnmap, dim3(n), dim3(kTileThreads), 0, s, P, work, l, vtx, nrm,
                           (const unsigned long long *)scratch, nw);
        return;
    }
    const dim3 row(std::min(nw * 64, 1024));
    hipLaunchKernelGGL(k_vn_graze<true>, dim3((unsigned)grid), dim3(kTileThreads), 0, s, P, l, bits, nw);
    if (nw <= 64) {
        hipLaunchKernelGGL((k_vn_order<1, true>), dim3(1), dim3(64), 0, s, bits, nw, W, H);
        hipLaunchKernelGGL(k_vnmap_rows<1>, dim3(H), row, 0, s, P, l, vtx, nrm, nw);
    } else {
        hipLaunchKernelGGL((k_vn_order<2, true>), dim3(1), dim3(64), 0, s, bits, nw, W, H);
        hipLaunchKernelGGL(k_vnmap_rows<2>, dim3(H), row, 0, s, P, l, vtx, nrm, nw);
    }
}

}  // namespace vs
