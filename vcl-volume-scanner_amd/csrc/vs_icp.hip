// vs_icp.hip — projective point-to-plane ICP with the Gauss-Newton loop on
// the device (A8-A12).
//
// Reference: LGKvPoseTracker::tp_Track_Pose (z_yooji_cuda_pose_tracker.cu:790-1042)
// launches one summand+reduction kernel per iteration, copies ~200 KB of
// block partials to the host, sums them in FP32, solves on the host and copies
// the pose back. Here each iteration is two launches: k_icp_iter writes one
// FP64 partial of the 29 sums per group of tiles, then k_icp_solve (one
// workgroup per session) sums them in FP64 in a fixed order, solves the 6x6
// system (Cholesky, FP64), applies the SE(3) update and publishes the FP32
// pose the next iteration reads. Small launches take one launch per iteration,
// in which every workgroup solves the last one's system before its sums
// (k_icp_step, the same results). Convergence (|x|_inf < 5e-7) and failure are
// flags the following launches test, so the host enqueues a fixed launch
// sequence that can be captured in a graph.
#include "vs_device.hpp"
#include "vs_launch.hpp"

namespace vs {

struct Mat16d {
    double m[16];
};

// ---------------------------------------------------------------------------
// FP64 pose algebra (one thread)
// ---------------------------------------------------------------------------
__device__ void matmul4d(const double *A, const double *B, double *C) {
    double t[16];
    for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 4; ++c) {
            double s = 0.0;
            for (int k = 0; k < 4; ++k) s = fma(A[r * 4 + k], B[k * 4 + c], s);
            t[r * 4 + c] = s;
        }
    for (int k = 0; k < 16; ++k) C[k] = t[k];
}
// Inverse of a rigid transform: [R^T, -R^T t]. Equals the reference's general
// 4x4 inverse (d_im_Inverse_Matrix_4x4, _yooji_math_inlines.h:404-465) on
// rigid inputs.
__device__ void rigid_inverse(const double *T, double *Ti) {
    double o[16];
    for (int r = 0; r < 3; ++r) {
        for (int c = 0; c < 3; ++c) o[r * 4 + c] = T[c * 4 + r];
        o[r * 4 + 3] = -(T[0 * 4 + r] * T[3] + T[1 * 4 + r] * T[7] + T[2 * 4 + r] * T[11]);
    }
    o[12] = o[13] = o[14] = 0.0;
    o[15] = 1.0;
    for (int k = 0; k < 16; ++k) Ti[k] = o[k];
}
__device__ void publish_T21(SessState *st) {
    rigid_inverse(st->T_12, st->T_21);
    for (int k = 0; k < 16; ++k) st->T_21_f[k] = (float)st->T_21[k];
}

// ---------------------------------------------------------------------------
// per-pixel summand (d_cssfp_Compute_Single_Summand_with_Forward_Params,
// pose_tracker.cu:279-395; bilinear taps d_giv/d_gin, _yooji_cuda_math.h:365-481)
// ---------------------------------------------------------------------------
// The 2x2 neighbourhood of (u, v) in a model map. A tap takes part only when
// its weight is positive (rx > 0 for the right column, ry > 0 for the lower
// row); a participating tap at -100 rejects the pixel. The maps interleave
// vertex and normal records, so a row's two pixels x0, x0 + 1 are 48
// contiguous bytes (vertex, normal, vertex, normal), read as three 16-byte
// loads: an unused right column (rx == 0) is read and ignored (x0 + 1 <= W,
// and the padding pixel after the last covers the last row), an unused
// lower row re-reads the upper one. Every address is inside the buffer, so
// all taps are loaded together, before any test.
struct Quad {
    MapXYZ a, b, c, d;
};
typedef vs_f4 vs_f4_a4 __attribute__((aligned(4)));  // 24-byte records: 8-byte aligned
struct Row {
    vs_f4 q0, q1, q2;  // vertex x0 | normal x0 | vertex x0 + 1 | normal x0 + 1, 3 floats each
};
__device__ __forceinline__ Row load_row(const MapXYZ *mvn, size_t i) {
    const VS_GLOBAL vs_f4_a4 *p = (const VS_GLOBAL vs_f4_a4 *)(mvn + 2 * i);
    return {p[0], p[1], p[2]};
}
__device__ __forceinline__ Quad vertex_quad(const Row &r0, const Row &r1) {
    return {{r0.q0.x, r0.q0.y, r0.q0.z}, {r0.q1.z, r0.q1.w, r0.q2.x}, {r1.q0.x, r1.q0.y, r1.q0.z},
            {r1.q1.z, r1.q1.w, r1.q2.x}};
}
__device__ __forceinline__ Quad normal_quad(const Row &r0, const Row &r1) {
    return {{r0.q0.w, r0.q1.x, r0.q1.y}, {r0.q2.y, r0.q2.z, r0.q2.w}, {r1.q0.w, r1.q1.x, r1.q1.y},
            {r1.q2.y, r1.q2.z, r1.q2.w}};
}
// Taps are picked by selects, not branches, so that no tap's load is sunk
// into a branch of its own (and waited for alone).
__device__ __forceinline__ bool bilerp(const Quad &q, float rx, float ry, f3 &out) {
    const bool ux = rx > 0.0f, uy = ry > 0.0f, uxy = ux & uy;
    const bool ok = (q.a.x != -100.0f) & (!ux | (q.b.x != -100.0f)) & (!uy | (q.c.x != -100.0f)) &
                    (!uxy | (q.d.x != -100.0f));
    const f3 t1 = {q.a.x, q.a.y, q.a.z};
    const f3 t2 = {ux ? q.b.x : 0.0f, ux ? q.b.y : 0.0f, ux ? q.b.z : 0.0f};
    const f3 t3 = {uy ? q.c.x : 0.0f, uy ? q.c.y : 0.0f, uy ? q.c.z : 0.0f};
    const f3 t4 = {uxy ? q.d.x : 0.0f, uxy ? q.d.y : 0.0f, uxy ? q.d.z : 0.0f};
    const float ix = 1.0f - rx, iy = 1.0f - ry;
    out = add(scale(iy, add(scale(ix, t1), scale(rx, t2))), scale(ry, add(scale(ix, t3), scale(rx, t4))));
    return ok;
}

// The summand of pixel (x, y) as a branch-free sequence: every test of the
// reference is evaluated (same FP32 expressions, so the same decisions) and
// folded into `ok`; the model taps use coordinates clamped into the map, so
// every load is in range whatever the tests say, and a rejected pixel's
// Jacobian and residual are zero. In two halves, so that a caller can issue
// the next pixel's model taps (icp_pre) before it evaluates this pixel's
// (icp_post); the operations are the same either way.
struct IcpPre {
    f3 p;            // the pixel's vertex in the model's frame
    float rx, ry;    // bilinear weights of the taps
    bool ok;         // depth valid, projection inside the map
    Row r0, r1;      // model vertex and normal taps of the two rows (loads in flight)
};
// td1: the filtered depth at (x, y), loaded by the caller
__device__ __forceinline__ IcpPre icp_pre(const SessParams &P, int l, int x, int y, float td1, const float *T21) {
    const LevelDesc &L = P.lev[l];
    const int W = L.W, H = L.H;
    IcpPre r;
    // back_project and project by shared divisors (640x480 level 0: the pixels
    // are 8000 of an iteration's 23500 cycles, vector issue)
    r.p = transform(T21, f3{quotient(td1 * ((float)x - L.K[2]), divisor(L.K[0])),
                            quotient(td1 * ((float)y - L.K[3]), divisor(L.K[1])), td1});
    float u, v;
    project_finite(r.p, L.K, u, v);
    const bool inside = u >= 0.0f && u <= float(W - 1) && v >= 0.0f && v <= float(H - 1);
    r.ok = !(td1 < 1.0e-6f) && inside;
    const float uc = inside ? u : 0.0f, vc = inside ? v : 0.0f;
    const int x0 = (int)uc, y0 = (int)vc;
    r.rx = uc - (float)x0;
    r.ry = vc - (float)y0;
    const size_t i0 = (size_t)y0 * W + x0, dj = r.ry > 0.0f ? (size_t)W : 0;
    r.r0 = load_row(P.mvn[l], i0);
    r.r1 = load_row(P.mvn[l], i0 + dj);
    return r;
}
__device__ __forceinline__ bool icp_post(const SessParams &P, const IcpPre &r, float A[6], float &b) {
    const f3 p = r.p;
    bool ok = r.ok;
    f3 v0, n;
    ok &= bilerp(vertex_quad(r.r0, r.r1), r.rx, r.ry, v0);
    const float dx = v0.x - p.x, dy = v0.y - p.y, dz = v0.z - p.z;
    ok &= !(dx * dx + dy * dy + dz * dz > P.icp_dist2);
    ok &= bilerp(normal_quad(r.r0, r.r1), r.rx, r.ry, n);
    {
        const Divisor len = divisor(sqrtf(dot(n, n)));
        n = scale(quotient(1.0f, len), n);
    }
    A[0] = ok ? p.z * n.y + (-p.y) * n.z : 0.0f;
    A[1] = ok ? (-p.z) * n.x + p.x * n.z : 0.0f;
    A[2] = ok ? p.y * n.x + (-p.x) * n.y : 0.0f;
    A[3] = ok ? -n.x : 0.0f;
    A[4] = ok ? -n.y : 0.0f;
    A[5] = ok ? -n.z : 0.0f;
    b = ok ? n.x * dx + n.y * dy + n.z * dz : 0.0f;
    return ok;
}
__device__ __forceinline__ bool icp_summand_d(const SessParams &P, int l, int x, int y, float td1, const float *T21,
                                              float A[6], float &b) {
    return icp_post(P, icp_pre(P, l, x, y, td1, T21), A, b);
}
__device__ __forceinline__ bool icp_summand(const SessParams &P, int l, int x, int y, const float *T21, float A[6],
                                            float &b) {
    return icp_summand_d(P, l, x, y, ldg(P.filt[l], (size_t)y * P.lev[l].W + x), T21, A, b);
}

// Adds one pixel's 29 terms (JtJ upper triangle, Jtr, count, r^2) to the
// thread's FP32 sums; a rejected pixel has A = 0, b = 0 and adds zeros.
__device__ __forceinline__ void add_terms(bool ok, const float A[6], float b, float acc[kIcpVals]) {
    int k = 0;
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = i; j < 6; ++j, ++k) acc[k] = fmaf(A[i], A[j], acc[k]);
#pragma unroll
    for (int i = 0; i < 6; ++i, ++k) acc[k] = fmaf(A[i], b, acc[k]);
    acc[k++] += ok ? 1.0f : 0.0f;
    acc[k] = fmaf(b, b, acc[k]);
}

// Block sum of the 29 terms through LDS: every thread stores its 29 FP32
// sums (term-major rows of 257 words, so that the stores of a wave and the
// reads below spread over the LDS banks), 8 threads per term each add a fixed
// chunk of 32 threads' values in FP32 (in a fixed order), and the 8 chunk sums
// of a term are added in FP64 in chunk order. Result in red64 (shared), valid
// after the call for all threads. (29 wave-wide DPP trees cost ~11 VALU
// instructions per term and wave; this costs ~4 per term and thread.)
constexpr int kTermRow = kTileThreads + 1;
constexpr int kChunks = 8, kChunk = kTileThreads / kChunks;
__device__ __forceinline__ void block_terms(float v[kIcpVals], double *red64) {
    __shared__ float rows[kIcpVals * kTermRow];
    __shared__ double part[kIcpVals][kChunks];
    const int t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < kIcpVals; ++k) rows[k * kTermRow + t] = v[k];
    __syncthreads();
    if (t < kIcpVals * kChunks) {
        const int k = t / kChunks, c = t % kChunks;
        const float *row = rows + k * kTermRow + c * kChunk;
        float s = 0.0f;
#pragma unroll 8
        for (int i = 0; i < kChunk; ++i) s += row[(i + 4 * c) & (kChunk - 1)];
        part[k][c] = (double)s;
    }
    __syncthreads();
    if (t < kIcpVals) {
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < kChunks; ++c) s += part[t][c];
        red64[t] = s;
    }
    __syncthreads();
}

// VS_ICP_MFMA (1 in the default build; build.py --variant icp_lds builds the
// per-thread FMA sums and LDS chunk sums instead): the block's 29 sums from
// the matrix cores. For each tile of the group, each pixel's row
// x = [A (6), b, ok] goes to LDS (2 KB per wave) and the wave runs
// v_mfma_f32_16x16x4f32 over its 64 rows, 8 pixels per instruction:
// the 16x16 product packs two 8x8 Gram blocks (two sets of 4 pixels) on its
// diagonal, with x read as both operands (lane l supplies feature l % 8 of
// pixel 4 * ((l % 16) / 8) + l / 16 of the instruction's 8), so
// G = sum x x^T holds J^T J, J^T r, sum r^2 and the count. The two diagonal
// blocks are added across lanes (lane l and l + 40 hold matching entries),
// and the 4 waves' blocks are added in FP64 in wave order. Without the 29
// per-thread accumulators and the 30 KB of LDS rows the kernel holds 64
// registers and 9 KB of LDS, so 8 waves per SIMD are resident instead of 5:
// the iteration waits on its dependent gathers (depth, then the model taps),
// and the extra waves hide them (ICP stage 2.61 -> 2.22 ms per 64-session
// step, with the same VALU work and bytes fetched).
#ifndef VS_ICP_MFMA
#define VS_ICP_MFMA 1
#endif
#if VS_ICP_MFMA
typedef float vs_f4x __attribute__((ext_vector_type(4)));
// entry (i, j) of the 8x8 Gram block that holds term k of the 29
__device__ __forceinline__ void term_ij(int k, int &i, int &j) {
    if (k < 21) {
        int r = 0, n = 6;
        while (k >= n) {
            k -= n;
            ++r;
            --n;
        }
        i = r;
        j = r + k;
    } else if (k < 27) {
        i = k - 21;
        j = 6;
    } else if (k == 27) {
        i = j = 7;
    } else {
        i = j = 6;
    }
}
#endif

__device__ __forceinline__ bool icp_skip(const SessParams &P, const SessState *st, int level, int iter) {
    return !ldg(&st->do_track, 0) || ldg(&st->icp_failed, 0) || ldg(&st->conv_level, 0) == level ||
           iter >= P.iters[level] || (ldg(&st->force_single, 0) && level != 0);
}

// The group's depths (independent loads; a pixel outside the frame re-reads
// pixel 0 and is skipped).
template <int G>
struct GroupPixels {
    int xs[G], ys[G];
    bool in[G];
    float td[G];
    __device__ __forceinline__ void load(const SessParams &P, int level, int t0) {
        const LevelDesc &L = P.lev[level];
        const int ntiles = L.tiles_x * L.tiles_y;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int tile = t0 + g;
            xs[g] = (tile % L.tiles_x) * kTileW + threadIdx.x % kTileW;
            ys[g] = (tile / L.tiles_x) * kTileH + threadIdx.x / kTileW;
            in[g] = tile < ntiles && xs[g] < L.W && ys[g] < L.H;
            td[g] = ldg(P.filt[level], in[g] ? (size_t)ys[g] * L.W + xs[g] : (size_t)0);
        }
    }
};

// The 29 sums of one group (G = icp_group(level) consecutive 32x8 tiles) at
// the pose T21s (LDS), one FP64 partial into out, summed on the matrix cores
// (above) or, with VS_ICP_MFMA=0, by per-thread FP32 accumulation over the
// group's tiles and one block reduction (block_terms).
template <int G>
__device__ __forceinline__ void group_sums(const SessParams &P, int level, const GroupPixels<G> &px_, const float *T21s,
                                           double *out) {
    const int *xs = px_.xs, *ys = px_.ys;
    const bool *in = px_.in;
    const float *td = px_.td;
#if VS_ICP_MFMA
    __shared__ float feat[kTileThreads / 64][64][8];
    __shared__ float gw[kTileThreads / 64][8][8];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int px = ((lane & 15) >> 3) * 4 + (lane >> 4), fi = lane & 7;
    vs_f4x g4 = {0.0f, 0.0f, 0.0f, 0.0f};
    // one pixel ahead: the next tile's model taps are in flight while this
    // tile's summand is evaluated (a pixel outside the frame has depth 0 and
    // adds zeros)
    IcpPre nxt = icp_pre(P, level, xs[0], ys[0], in[0] ? td[0] : 0.0f, T21s);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        float A[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, b = 0.0f;
        const IcpPre cur = nxt;
        if (g + 1 < G) nxt = icp_pre(P, level, xs[g + 1], ys[g + 1], in[g + 1] ? td[g + 1] : 0.0f, T21s);
        const bool ok = icp_post(P, cur, A, b);
        // the wave's 64 rows of this tile. A wave reads only its own rows, and
        // the LDS performs one wave's accesses in the order they are issued,
        // so no workgroup barrier is needed between the writes and the reads
        // (nor before the next tile's writes); the compiler keeps their order
        // (the rows may alias) and wave_barrier keeps it from moving them.
        __builtin_amdgcn_wave_barrier();
        float *f = feat[wv][lane];
#pragma unroll
        for (int k = 0; k < 6; ++k) f[k] = A[k];
        f[6] = b;
        f[7] = ok ? 1.0f : 0.0f;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const float a = feat[wv][8 * m + px][fi];
            g4 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, a, g4, 0, 0, 0);
        }
    }
    // lane l holds D[4 (l / 16) + r][l % 16]; the second block's entry
    // D[i + 8][j + 8] of the first block's D[i][j] sits in lane l + 40
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float other = __shfl_down(g4[r], 40, 64);
        if ((lane >> 4) < 2 && (lane & 15) < 8) gw[wv][4 * (lane >> 4) + r][lane & 15] = g4[r] + other;
    }
    __syncthreads();
    if (threadIdx.x < kIcpVals) {
        int i, j;
        term_ij(threadIdx.x, i, j);
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kTileThreads / 64; ++w) s += (double)gw[w][i][j];
        stg(out, threadIdx.x, s);
    }
#else
    __shared__ double red64[kIcpVals];
    float acc[kIcpVals];
#pragma unroll
    for (int k = 0; k < kIcpVals; ++k) acc[k] = 0.0f;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        if (in[g]) {
            float A[6], b;
            const bool ok = icp_summand_d(P, level, xs[g], ys[g], td[g], T21s, A, b);
            add_terms(ok, A, b, acc);
        }
    }
    block_terms(acc, red64);
    if (threadIdx.x < kIcpVals) stg(out, threadIdx.x, red64[threadIdx.x]);
#endif
}

// One Gauss-Newton iteration at `level`, first half of the two-launch form:
// the partial of every group of every session of the work list (items are
// (session, group)). No cross-workgroup synchronisation here: on a
// multi-XCD device an agent-scope release per workgroup would write back L2
// each time, so the reduction and the solve are the next launch
// (k_icp_solve).
template <int G>
__global__ __launch_bounds__(kTileThreads) void k_icp_iter(const SessParams *__restrict__ SP,
                                                           const WorkItem *__restrict__ work, int level, int iter) {
    __shared__ float T21s[16];
    const WorkItem wi = work[blockIdx.x];
    const SessParams &P = SP[wi.sess];
    const SessState *st = P.st;
    if (level >= P.levels || icp_skip(P, st, level, iter)) return;
    const LevelDesc &L = P.lev[level];
    const int t0 = wi.tile * G;
    if (t0 >= L.tiles_x * L.tiles_y) return;
    if (threadIdx.x < 16) T21s[threadIdx.x] = ldg(st->T_21_f, threadIdx.x);
    __syncthreads();
    GroupPixels<G> px;
    px.load(P, level, t0);
    group_sums<G>(P, level, px, T21s, P.icp_part + (size_t)wi.tile * kIcpVals);
}

// The 29 totals of ng group partials in FP64, in a fixed order that depends
// on the group count alone: chunk c adds groups c, c + 64, ..., then the 64
// chunk sums of a term are added as a tree of halves. A thread takes chunks c
// and c + 32 of a term, the tree's first pair, so neighbouring threads read
// neighbouring terms and a load covers whole lines. In two halves, so that a
// kernel can have the first loads in flight together with the state it needs
// before it knows whether there is anything to sum.
constexpr int kSumChunks = 64, kSumPairs = kSumChunks / 2;
template <int THREADS>
struct PartialSums {
    static constexpr int N = (kSumPairs * kIcpVals + THREADS - 1) / THREADS;  // pairs per thread
    static constexpr int U = N == 1 ? 5 : 3;                                  // groups per chunk and round
    double v[N][2][U];
    // groups g0 + c, g0 + c + 64, ... of the thread's chunks (0 beyond the
    // last group: a running sum that began at 0.0 is never -0.0, so adding it
    // changes nothing)
    __device__ __forceinline__ void load(const double *part, int ng, int g0) {
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const int p = n * THREADS + (int)threadIdx.x, c = p / kIcpVals, k = p - c * kIcpVals;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int g = g0 + c + h * kSumPairs + u * kSumChunks;
                    v[n][h][u] = 0.0;
                    if (p < kSumPairs * kIcpVals && g < ng) v[n][h][u] = ldg(part, (size_t)g * kIcpVals + k);
                }
        }
    }
    // after load(part, ng, 0); tot (LDS) is visible to the first wave only
    __device__ __forceinline__ void finish(const double *part, int ng, double (*pair)[kIcpVals], double *tot) {
        double s[N][2];
#pragma unroll
        for (int n = 0; n < N; ++n)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                s[n][h] = 0.0;
#pragma unroll
                for (int u = 0; u < U; ++u) s[n][h] += v[n][h][u];
            }
        for (int g0 = U * kSumChunks; g0 < ng; g0 += U * kSumChunks) {
            load(part, ng, g0);
#pragma unroll
            for (int n = 0; n < N; ++n)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int u = 0; u < U; ++u) s[n][h] += v[n][h][u];
        }
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const int p = n * THREADS + (int)threadIdx.x, c = p / kIcpVals, k = p - c * kIcpVals;
            if (p < kSumPairs * kIcpVals) pair[c][k] = s[n][0] + s[n][1];
        }
        __syncthreads();
        // two threads per term, each half of the next level's pairs
        const int t = threadIdx.x;
        if (t < 2 * 32) {
            const int k = t & 31, side = t >> 5;
            if (k < kIcpVals) {
                double w[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int c = q + 8 * side;
                    w[q] = pair[c][k] + pair[c + 16][k];
                }
#pragma unroll
                for (int q = 0; q < 8; ++q) w[q] += __shfl_xor(w[q], 32, 64);
#pragma unroll
                for (int h = 4; h >= 1; h >>= 1)
#pragma unroll
                    for (int q = 0; q < h; ++q) w[q] += w[q + h];
                if (side == 0) tot[k] = w[0];
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
};

// Value of a double in a given lane (all lanes active), and in lane Q of each
// quad of lanes.
__device__ __forceinline__ double lane_of(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
template <int Q>
__device__ __forceinline__ double quad_of(double v) {
    constexpr int ctrl = Q * 0x55;
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), ctrl, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), ctrl, 0xf, 0xf, true));
}
// position of entry (p, q), p <= q, of a 6x6 upper triangle stored by rows
__device__ __forceinline__ constexpr int tri6(int p, int q) { return p * (11 - p) / 2 + q; }

// One solve and SE(3) update from the 29 totals (LDS), by one wave; all of its
// lanes are active. The outcome is the same in every lane, t12 is entry
// lane % 16 of the updated increment.
struct SolveResult {
    bool updated, converged;
    int failed;
    double t12;
};
// Cholesky and triangular solves with the reference's pivot rule
// (d_lld_LL_Decomposition / d_sls_Solve_Linear_System_using_LLD,
// _yooji_cuda_math.h:489-592): entries below a pivot < 1e-8 are zeroed and the
// solve fails (status 4) if any pivot is below 1e-8 (or not a number). With
// rel > 0 it also fails (status 8) when a squared pivot L_jj^2 is below
// rel * A_jj: column j of J is then nearly a combination of the columns
// before it (a plane leaves 3 of the 6 motions unconstrained), a near-rank
// deficiency the absolute test cannot see at FP32 scales. The ratio is
// invariant to the units of the rotation and translation columns. Each
// below-diagonal entry and substitution step is scaled by the column's
// reciprocal pivot (6 FP64 divisions instead of 33).
// The update T12 <- exp(x) T12 takes x = [w; v] as a twist
// (z_uitme_Update_Incremental_Tracking_with_Matrix_Exponential,
// pose_tracker.cu:50-149), with a series branch for small |w| (the reference
// divides by |w|).
// Lane i holds row i of the factor and lane 4r + c entry (r, c) of the 4x4
// matrices; every operation and its order are those of one lane doing it all,
// which took 7000 cycles of a workgroup's 27000 in an iteration (640x480,
// level 0), many of them the issue of independent FP64 operations; it is 5500
// now, and an iteration 23500 with StepLoads (fused frame with preview: 412 ->
// 408 us, 320x240 358 -> 354, 64 sessions 6.52 -> 6.45 ms).
__device__ __forceinline__ SolveResult solve_wave(const SessParams &P, const double *tot, const double *T12) {
    const int lane = threadIdx.x & 63;
    SolveResult r{false, false, 0, 0.0};
    const double cnt = tot[21 + 6];
    if (P.icp_min_valid > 0 && cnt < (double)P.icp_min_valid) {
        r.failed = 7;
        return r;
    }
    const int i = min(lane, 5), er = (lane >> 2) & 3, ec = lane & 3;
    double a[6], l[6], t12c[4];
#pragma unroll
    for (int j = 0; j < 6; ++j) a[j] = tot[tri6(min(i, j), max(i, j))];
    const double b = tot[21 + i];
#pragma unroll
    for (int k = 0; k < 4; ++k) t12c[k] = T12[k * 4 + ec];
    double U[6][6], D[6], inv[6];  // the factor and its diagonal's reciprocals, in every lane
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < j; ++k) {
            U[j][k] = lane_of(l[k], j);
            t += l[k] * U[j][k];
        }
        const double d = a[j] - t;
        D[j] = sqrt(lane_of(d, j));
        inv[j] = 1.0 / D[j];
        l[j] = fabs(D[j]) >= 1e-8 ? d * inv[j] : 0.0;
    }
    bool pivots = true, guard = false;
    const double rel = (double)P.icp_rel_pivot;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        pivots &= fabs(D[j]) >= 1e-8;
        guard |= D[j] * D[j] < rel * tot[tri6(j, j)];
    }
    r.failed = !pivots ? 4 : (rel > 0.0 && guard) ? 8 : 0;
    if (r.failed != 0) return r;
    double y[6], x[6], s = 0.0;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        y[k] = lane_of((b - s) * inv[k], k);
        s += l[k] * y[k];
    }
#pragma unroll
    for (int j = 5; j >= 0; --j) {
        double q = 0.0;
#pragma unroll
        for (int k = j + 1; k < 6; ++k) q += U[k][j] * x[k];
        x[j] = (y[j] - q) * inv[j];
    }
    double ninf = 0.0;
#pragma unroll
    for (int k = 0; k < 6; ++k) ninf = fmax(ninf, fabs(x[k]));
    if (ninf < 5.0e-7) {
        r.converged = true;
        return r;
    }
    const double w0 = x[0], w1 = x[1], w2 = x[2];
    const double th2 = w0 * w0 + w1 * w1 + w2 * w2, th = sqrt(th2);
    double A, B, C;
    if (th < 1e-4) {
        A = 1.0 - th2 / 6.0 + th2 * th2 / 120.0;
        B = 0.5 - th2 / 24.0 + th2 * th2 / 720.0;
        C = 1.0 / 6.0 - th2 / 120.0 + th2 * th2 / 5040.0;
    } else {
        A = sin(th) / th;
        B = (1.0 - cos(th)) / th2;
        C = (th - sin(th)) / (th2 * th);
    }
    // W = [0 -w2 w1; w2 0 -w0; -w1 w0 0]: row er, column ec, and their product
    const double Wr0 = er == 1 ? w2 : er == 2 ? -w1 : 0.0, Wr1 = er == 0 ? -w2 : er == 2 ? w0 : 0.0,
                 Wr2 = er == 0 ? w1 : er == 1 ? -w0 : 0.0;
    const double W0c = ec == 1 ? -w2 : ec == 2 ? w1 : 0.0, W1c = ec == 0 ? w2 : ec == 2 ? -w0 : 0.0,
                 W2c = ec == 0 ? -w1 : ec == 1 ? w0 : 0.0;
    const double W = ec == 0 ? Wr0 : ec == 1 ? Wr1 : Wr2, xv = ec == 0 ? x[3] : ec == 1 ? x[4] : x[5];
    const double WW = Wr0 * W0c + Wr1 * W1c + Wr2 * W2c, I = er == ec ? 1.0 : 0.0;
    const double rot = I + A * W + B * WW, vx = (I + B * W + C * WW) * xv;
    double tr = 0.0;
    tr += quad_of<0>(vx);
    tr += quad_of<1>(vx);
    tr += quad_of<2>(vx);
    const double E = er == 3 ? (ec == 3 ? 1.0 : 0.0) : (ec == 3 ? tr : rot);
    double m = 0.0;
    m = fma(quad_of<0>(E), t12c[0], m);
    m = fma(quad_of<1>(E), t12c[1], m);
    m = fma(quad_of<2>(E), t12c[2], m);
    m = fma(quad_of<3>(E), t12c[3], m);
    r.t12 = m;
    r.updated = true;
    return r;
}
// Entry lane % 16 of the inverse of a rigid transform in LDS (rigid_inverse's
// operations).
__device__ __forceinline__ double rigid_inverse_lane(const double *T) {
    const int er = (threadIdx.x >> 2) & 3, ec = threadIdx.x & 3;
    const double rot = er < 3 && ec < 3 ? T[ec * 4 + er] : (er == ec ? 1.0 : 0.0);
    const int c = min(er, 2);
    const double t = -(T[c] * T[3] + T[4 + c] * T[7] + T[8 + c] * T[11]);
    return er < 3 && ec == 3 ? t : rot;
}

// Second half of the two-launch form: one workgroup per session sums the
// group partials, solves the 6x6 system and applies the SE(3) update. THREADS
// changes how many of the sums run at once, not their order.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void k_icp_solve(const SessParams *__restrict__ SP, int nsess, int level,
                                                            int iter) {
    __shared__ double pair[kSumPairs][kIcpVals], tot[kIcpVals], T12[16];
    const int s = blockIdx.x;
    if (s >= nsess) return;
    const SessParams &P = SP[s];
    SessState *st = P.st;
    if (level >= P.levels) return;
    const int ng = icp_groups(P.lev[level].tiles_x * P.lev[level].tiles_y, level);
    PartialSums<THREADS> sums;
    sums.load(P.icp_part, ng, 0);  // in flight during the tests
    const double t12 = ldg(st->T_12, threadIdx.x & 15);
    const int solves = ldg(&st->solves, 0);
    if (icp_skip(P, st, level, iter)) return;
    if (threadIdx.x < 16) T12[threadIdx.x] = t12;
    sums.finish(P.icp_part, ng, pair, tot);
    if (threadIdx.x >= 64) return;
    const SolveResult r = solve_wave(P, tot, T12);
    if (threadIdx.x == 0) {
        stg(&st->solves, 0, solves + 1);
        if (r.failed) stg(&st->icp_failed, 0, r.failed);
        else if (r.converged) stg(&st->conv_level, 0, level);
    }
    if (!r.updated) return;
    if (threadIdx.x < 16) T12[threadIdx.x] = r.t12;
    __builtin_amdgcn_wave_barrier();  // one wave's LDS accesses are in order
    const double t21 = rigid_inverse_lane(T12);
    if (threadIdx.x < 16) {
        stg(st->T_12, threadIdx.x, r.t12);
        stg(st->T_21, threadIdx.x, t21);
        stg(st->T_21_f, threadIdx.x, (float)t21);
    }
}

// The one-launch form of an iteration: every workgroup of a session first
// solves the previous iteration's system, each for itself from the same
// partials in the same order, and then sums its group at the new pose. It
// costs the solve (~2 us of one wave) in every workgroup and saves a launch
// and its gap per iteration; which form is faster depends on how many
// workgroups share a CU (kIcpStepGroups). The kernel boundary orders the
// partials; workgroup 0 of a session records where the loop stands for the
// next launch, in the record and the half of icp_part that this launch's
// workgroups do not read.
constexpr int kStepThreads = 1024;
struct StepShared {
    double pair[kSumPairs][kIcpVals], tot[kIcpVals];
    double T12[16];
    float T21f[16];
    int failed, conv_level, solves;
};
// What a launch needs before it can go on, all loads in flight together: both
// records, the tracker's flags, and the partials it expects to find pending,
// those of the launch before (level prev, -1: none) in the half that alternates
// with seq. (Flags, then records, then partials, each waited for: a workgroup
// began its solve after 7000 cycles of its 27000.)
struct StepLoads {
    vs_u4 a0, a1;  // seq, pending, failed, conv_level
    int n0, n1;    // solves
    double t0, t1;
    int track, single;
    PartialSums<kStepThreads> sums;
    // part, ng: the expected partials (ng 0: none)
    __device__ __forceinline__ void load(const SessState *st, const double *part, int ng) {
        a0 = ldg((const vs_u4 *)&st->step[0].seq, 0);
        a1 = ldg((const vs_u4 *)&st->step[1].seq, 0);
        n0 = ldg(&st->step[0].solves, 0);
        n1 = ldg(&st->step[1].solves, 0);
        t0 = ldg(st->step[0].T_12, threadIdx.x & 15);
        t1 = ldg(st->step[1].T_12, threadIdx.x & 15);
        track = ldg(&st->do_track, 0);
        single = ldg(&st->force_single, 0);
        sums.load(part, ng, 0);
    }
};
// Brings the loop up to date into sh (all threads); returns the record it
// started from. seq: only records of earlier launches count.
__device__ __forceinline__ int step_resume(const SessParams &P, StepLoads &ld, int seq, int prev, StepShared &sh) {
    const int s0 = (int)ld.a0.x, s1 = (int)ld.a1.x;
    const int cur = (int)(s1 < seq) & ((int)(s0 >= seq) | (int)(s1 > s0));
    const vs_u4 S = cur ? ld.a1 : ld.a0;
    const int pending = (int)S.y;
    if (threadIdx.x < 16) sh.T12[threadIdx.x] = cur ? ld.t1 : ld.t0;
    if (threadIdx.x == 16) {
        sh.failed = (int)S.z;
        sh.conv_level = (int)S.w;
        sh.solves = cur ? ld.n1 : ld.n0;
    }
    if (pending >= 0) {
        const double *part = P.icp_part + (size_t)cur * P.icp_half;
        const int ng = icp_groups(P.lev[pending].tiles_x * P.lev[pending].tiles_y, pending);
        // not where they were expected: a session with fewer levels than the batch
        if (pending != prev || cur != ((seq - 1) & 1)) ld.sums.load(part, ng, 0);
        ld.sums.finish(part, ng, sh.pair, sh.tot);
    } else {
        __syncthreads();
    }
    if (threadIdx.x < 64) {
        if (pending >= 0) {
            const SolveResult r = solve_wave(P, sh.tot, sh.T12);
            if (threadIdx.x == 0) {
                sh.solves += 1;
                if (r.failed) sh.failed = r.failed;
                else if (r.converged) sh.conv_level = pending;
            }
            if (r.updated && threadIdx.x < 16) sh.T12[threadIdx.x] = r.t12;
        }
        __builtin_amdgcn_wave_barrier();  // one wave's LDS accesses are in order
        const double t21 = rigid_inverse_lane(sh.T12);
        if (threadIdx.x < 16) sh.T21f[threadIdx.x] = (float)t21;
    }
    __syncthreads();
    return cur;
}

// The same sums as group_sums by 16 waves: wave (c, q), c = wave % 4, evaluates
// the pixels that wave c of group_sums has in the group's tiles q * G / 4,
// ..., all loads at once, and leaves their rows in LDS; then wave (c, 0) runs
// c's chain of matrix instructions over the group's rows in the same order,
// so the sums are the same bits. A 150-group launch leaves 106 CUs idle
// anyway; with 4 waves a workgroup walked its 8 tiles one after another
// (640x480, level 0: 7.2 us of the iteration's 13.1; the launch-to-launch time
// of an iteration is now 11.3).
#if VS_ICP_MFMA
template <int G>
struct WidePixels {
    static constexpr int N = G / 4;  // tiles per wave
    int xs[N], ys[N];
    float td[N];
    __device__ __forceinline__ void load(const LevelDesc &L, const float *filt, int t0) {
        const int ntiles = L.tiles_x * L.tiles_y;
        const int wave = threadIdx.x >> 6, tt = (wave & 3) * 64 + (threadIdx.x & 63);  // thread of the tile
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const int tile = t0 + (wave >> 2) * N + j;
            xs[j] = (tile % L.tiles_x) * kTileW + tt % kTileW;
            ys[j] = (tile / L.tiles_x) * kTileH + tt / kTileW;
            const bool in = tile < ntiles && xs[j] < L.W && ys[j] < L.H;
            const float d = ldg(filt, in ? (size_t)ys[j] * L.W + xs[j] : (size_t)0);
            td[j] = in ? d : 0.0f;
        }
    }
};
template <int G>
__device__ __forceinline__ void group_sums_wide(const SessParams &P, int level, const WidePixels<G> &px,
                                                const float *T21s, double *out, int ti, int tj) {
    constexpr int N = WidePixels<G>::N;
    __shared__ __align__(16) float feat[4][G][64][8];
    __shared__ float gw[4][8][8];
    const int wave = threadIdx.x >> 6, c = wave & 3, q = wave >> 2, lane = threadIdx.x & 63;
    IcpPre pre[N];
#pragma unroll
    for (int j = 0; j < N; ++j) pre[j] = icp_pre(P, level, px.xs[j], px.ys[j], px.td[j], T21s);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        float A[6], b;
        const bool ok = icp_post(P, pre[j], A, b);
        float *f = feat[c][q * N + j][lane];
#pragma unroll
        for (int k = 0; k < 6; ++k) f[k] = A[k];
        f[6] = b;
        f[7] = ok ? 1.0f : 0.0f;
    }
    __syncthreads();
    if (q == 0) {
        const int row = ((lane & 15) >> 3) * 4 + (lane >> 4), fi = lane & 7;
        vs_f4x g4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const float a = feat[c][g][8 * m + row][fi];
                g4 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, a, g4, 0, 0, 0);
            }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float other = __shfl_down(g4[r], 40, 64);
            if ((lane >> 4) < 2 && (lane & 15) < 8) gw[c][4 * (lane >> 4) + r][lane & 15] = g4[r] + other;
        }
    }
    __syncthreads();
    if (threadIdx.x < kIcpVals) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < 4; ++w) s += (double)gw[w][ti][tj];
        stg(out, threadIdx.x, s);
    }
}

// prev: level of launch seq - 1 (-1: none)
template <int G>
__global__ __launch_bounds__(kStepThreads) void k_icp_step(const SessParams *__restrict__ SP,
                                                           const WorkItem *__restrict__ work, int level, int iter,
                                                           int seq, int prev) {
    __shared__ StepShared sh;
    const WorkItem wi = work ? work[blockIdx.x] : WorkItem{0, (int)blockIdx.x};
    const SessParams &P = SP[__builtin_amdgcn_readfirstlane(wi.sess)];
    // read now, with the sizes tested below, not in a round of its own after them
    SessState *st = P.st;
    double *part = P.icp_part;
    const float *filt = P.filt[level];
    int half = P.icp_half, nprev = prev < 0 ? 0 : P.lev[prev].tiles_x * P.lev[prev].tiles_y;
    asm volatile("" : "+s"(st), "+s"(part), "+s"(filt), "+s"(half), "+s"(nprev));
    const LevelDesc &L = P.lev[level];
    const int t0 = wi.tile * G;
    if ((int)(level >= P.levels) | (int)(t0 >= L.tiles_x * L.tiles_y)) return;
    StepLoads ld;
    ld.load(st, part + (size_t)((seq - 1) & 1) * half, icp_groups(nprev, prev));
    WidePixels<G> px;
    px.load(L, filt, t0);  // in flight during the solve
    int ti, tj;
    term_ij(threadIdx.x < kIcpVals ? threadIdx.x : 0, ti, tj);
    if (!ld.track) return;
    const int out = step_resume(P, ld, seq, prev, sh) ^ 1;
    const bool skip = sh.failed || sh.conv_level == level || iter >= P.iters[level] || (ld.single && level != 0);
    if (wi.tile == 0) {
        IcpStep *S = &st->step[out];
        if (threadIdx.x < 16) stg(S->T_12, threadIdx.x, sh.T12[threadIdx.x]);
        if (threadIdx.x == 16) {
            stg(&S->seq, 0, seq);
            stg(&S->pending, 0, skip ? -1 : level);
            stg(&S->failed, 0, sh.failed);
            stg(&S->conv_level, 0, sh.conv_level);
            stg(&S->solves, 0, sh.solves);
        }
    }
    if (skip) return;
    group_sums_wide<G>(P, level, px, sh.T21f, P.icp_part + (size_t)out * P.icp_half + (size_t)wi.tile * kIcpVals, ti, tj);
}
#endif

// Per-frame / per-track reset of the tracker state (one thread per session).
// `active` (nullable: all active) marks the sessions of a slot table that have
// a frame in this step; the others keep their state untouched by the step.
__global__ void k_track_setup(const SessParams *__restrict__ SP, int nsess, Mat16d Tinit, int has_init,
                              int force_track, const int *__restrict__ active) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsess) return;
    SessState *st = SP[s].st;
    st->active = active ? active[s] : 1;
    if (!st->active) {
        st->do_track = 0;
        st->fuse_ok = 0;
        return;
    }
    st->do_track = force_track ? 1 : (st->frames > 0);
    st->icp_failed = 0;
    st->conv_level = -1;
    st->solves = 0;
    st->force_single = has_init;
    for (int k = 0; k < 16; ++k) {
        const double v = has_init ? Tinit.m[k] : ((k % 5) == 0 ? 1.0 : 0.0);
        st->T_12[k] = v;
        st->step[0].T_12[k] = v;
    }
    publish_T21(st);
    st->step[0].seq = 0;
    st->step[0].pending = -1;
    st->step[0].failed = 0;
    st->step[0].conv_level = -1;
    st->step[0].solves = 0;
    st->step[1].seq = -1;
}

__device__ void set_pose_derived(const SessParams &P, SessState *st) {
    rigid_inverse(st->T_gc, st->T_cg);
    for (int k = 0; k < 16; ++k) {
        st->T_gc_f[k] = (float)st->T_gc[k];
        st->T_cg_f[k] = (float)st->T_cg[k];
    }
    // raycast constants from the FP32 pose (d_gcc_Get_Camera_Center and
    // rmi_Render_Maps_for_ICP, tsdf_renderer.cu:1667-1675)
    const float *T = st->T_gc_f;
    const float tx = T[3], ty = T[7], tz = T[11];
    const f3 cam = {-T[0] * tx - T[4] * ty - T[8] * tz, -T[1] * tx - T[5] * ty - T[9] * tz,
                    -T[2] * tx - T[6] * ty - T[10] * tz};
    const f3 vcc = sub({P.cube_cen[0], P.cube_cen[1], P.cube_cen[2]}, cam);
    const f3 ncc = normalised(vcc);
    const float d = sqrtf(dot(vcc, vcc));
    const float s = P.r_cube / d;
    st->cam[0] = cam.x; st->cam[1] = cam.y; st->cam[2] = cam.z;
    st->ncc[0] = ncc.x; st->ncc[1] = ncc.y; st->ncc[2] = ncc.z;
    st->dist_cc = d;
    st->cos_max = (s < 1.0f) ? sqrtf(1.0f - s * s) : -2.0f;
}

// The session's record in host memory (HostState), by one thread; visible to
// the host once it has waited for the stream. A pose read back by a 128-byte
// device-to-host copy cost ~20 us of the host's time (64-session step with the
// poses read back 7.90 -> 6.67 ms, 640x480 scan with preview 463 -> 440 us,
// 8 of 24 server slots 1.34 -> 1.21 ms).
__device__ __forceinline__ void publish_host(const SessParams &P, const SessState *st) {
    HostState *h = P.host;
    if (!h) return;
#pragma unroll
    for (int k = 0; k < 16; ++k) stg(h->T_gc, k, st->T_gc[k]);
    stg(&h->last_status, 0, st->last_status);
    stg(&h->frames, 0, st->frames);
    stg(&h->solves, 0, st->solves);
}

__device__ double rotation_deg(const double *T) {
    double c = (T[0] + T[5] + T[10] - 1.0) * 0.5;
    c = fmax(-1.0, fmin(1.0, c));
    return acos(c) * 57.295779513082320876798;
}

// Apply the tracked increment (T_gc <- T_12 T_gc, pose_tracker.cu:992-998) or
// record the failure; decides whether the frame is integrated.
__device__ __forceinline__ void track_finalize(const SessParams &P, SessState *st) {
    int status = 0;
    if (st->do_track) {
        if (st->icp_failed) {
            status = st->icp_failed;
        } else {
            const double *T = st->T_12;
            const double tn = sqrt(T[3] * T[3] + T[7] * T[7] + T[11] * T[11]);
            if ((P.max_motion_m > 0.0f && tn > P.max_motion_m) ||
                (P.max_motion_deg > 0.0f && rotation_deg(T) > P.max_motion_deg)) {
                status = 5;
            } else {
                matmul4d(st->T_12, st->T_gc, st->T_gc);
                set_pose_derived(P, st);
            }
        }
    }
    st->last_status = status;
    st->fuse_ok = (status == 0);
    if (status == 0) st->frames += 1;
    publish_host(P, st);
}
// What the step's integration counts from zero: the batch's brick list (by the
// launch's first thread), a session's visible bricks and updated voxels, and
// whether it gained a band superbrick (every kernel that reads that flag runs
// after the integration that sets it and before the next reset). A track of
// its own (bricks null) has no integration behind it and leaves them alone:
// the counts are the last integration's until the next one.
__device__ __forceinline__ void integrate_begin(SessState *st) {
    st->vis_count = 0u;
    st->upd_count = 0ull;
    st->sdist_dirty = 0;
}
__global__ void k_integrate_begin(const SessParams *__restrict__ SP, unsigned *bricks) {
    if (threadIdx.x != 0) return;
    *bricks = 0u;
    SP[0].st->active = 1;
    integrate_begin(SP[0].st);
}
__global__ void k_track_finalize(const SessParams *__restrict__ SP, int nsess, unsigned *bricks) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0 && bricks) *bricks = 0u;
    if (s >= nsess) return;
    const SessParams &P = SP[s];
    SessState *st = P.st;
    if (!st->active) {
        st->fuse_ok = 0;
        return;
    }
    if (bricks) integrate_begin(st);
    track_finalize(P, st);
}
// The same after the one-launch iterations: one workgroup per session solves
// the last one first.
__global__ __launch_bounds__(kStepThreads) void k_icp_finish(const SessParams *__restrict__ SP, unsigned *bricks,
                                                             int seq, int prev) {
    __shared__ StepShared sh;
    if (blockIdx.x == 0 && threadIdx.x == 0 && bricks) *bricks = 0u;
    const SessParams &P = SP[blockIdx.x];
    SessState *st = P.st;
    if (!st->active) {
        if (threadIdx.x == 0) st->fuse_ok = 0;
        return;
    }
    StepLoads ld;
    ld.load(st, P.icp_part + (size_t)((seq - 1) & 1) * P.icp_half,
            prev < 0 ? 0 : icp_groups(P.lev[prev].tiles_x * P.lev[prev].tiles_y, prev));
    if (ld.track) {
        step_resume(P, ld, seq, prev, sh);
        if (threadIdx.x == 0) {
            for (int i = 0; i < 16; ++i) st->T_12[i] = sh.T12[i];
            st->icp_failed = sh.failed;
            st->conv_level = sh.conv_level;
            st->solves = sh.solves;
        }
    }
    if (threadIdx.x == 0) {
        if (bricks) integrate_begin(st);
        track_finalize(P, st);
    }
}

// Pose set from the host, with its derived copies; reset: every other field of
// the state as for a new session first; set_frames: the frame count too.
__global__ __launch_bounds__(64) void k_set_pose(const SessParams *__restrict__ SP, Mat16d T, int reset, int set_frames,
                                                 int frames) {
    SessState *st = SP[0].st;
    if (reset) {
        static_assert(sizeof(SessState) % 4 == 0, "cleared by words");
        for (unsigned i = threadIdx.x; i < sizeof(SessState) / 4; i += 64) stg((uint32_t *)st, i, 0u);
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int k = 0; k < 16; ++k) st->T_gc[k] = T.m[k];
    if (reset) {
        st->conv_level = -1;
        st->active = 1;
    }
    if (set_frames) st->frames = frames;
    set_pose_derived(SP[0], st);
    publish_host(SP[0], st);
}

// Normal equations of one iteration without a solve (diagnostics/parity).
__global__ __launch_bounds__(kTileThreads) void k_icp_system(const SessParams *__restrict__ SP,
                                                             const WorkItem *__restrict__ work, int level, Mat16f T21,
                                                             double *out_part, uint8_t *mask) {
    __shared__ double red64[kIcpVals];
    const WorkItem wi = work[blockIdx.x];
    const SessParams &P = SP[wi.sess];
    const LevelDesc &L = P.lev[level];
    const int x = (wi.tile % L.tiles_x) * kTileW + threadIdx.x % kTileW;
    const int y = (wi.tile / L.tiles_x) * kTileH + threadIdx.x / kTileW;
    float A[6] = {0, 0, 0, 0, 0, 0}, b = 0.0f;
    bool ok = false;
    if (x < L.W && y < L.H) {
        ok = icp_summand(P, level, x, y, T21.m, A, b);
        if (mask) mask[(size_t)y * L.W + x] = ok ? 1 : 0;
    }
    float v[kIcpVals];
#pragma unroll
    for (int k = 0; k < kIcpVals; ++k) v[k] = 0.0f;
    add_terms(ok, A, b, v);
    block_terms(v, red64);
    if (threadIdx.x < kIcpVals) out_part[(size_t)wi.tile * kIcpVals + threadIdx.x] = red64[threadIdx.x];
}

void launch_track_setup(const SessParams *P, int nsess, const double *T_init, hipStream_t s) {
    Mat16d m{};
    int has = T_init != nullptr;
    if (has)
        for (int k = 0; k < 16; ++k) m.m[k] = T_init[k];
    // force_track: an explicit T_init call (vs_track) always tracks
    hipLaunchKernelGGL(k_track_setup, dim3((nsess + 63) / 64), dim3(64), 0, s, P, nsess, m, has, 0,
                       (const int *)nullptr);
}
void launch_track_setup_forced(const SessParams *P, int nsess, const double *T_init, hipStream_t s) {
    Mat16d m{};
    int has = T_init != nullptr;
    if (has)
        for (int k = 0; k < 16; ++k) m.m[k] = T_init[k];
    hipLaunchKernelGGL(k_track_setup, dim3((nsess + 63) / 64), dim3(64), 0, s, P, nsess, m, has, 1,
                       (const int *)nullptr);
}
void launch_track_setup_active(const SessParams *P, int nsess, const int *active, hipStream_t s) {
    Mat16d m{};
    hipLaunchKernelGGL(k_track_setup, dim3((nsess + 63) / 64), dim3(64), 0, s, P, nsess, m, 0, 0, active);
}

// Writes a slot table's active flags from a bit mask passed by value, so a
// captured step reads them from device memory.
struct ActiveMask {
    uint32_t bits[kMaxSlots / 32];
};
__global__ void k_set_active(int *active, int nslots, ActiveMask m) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nslots) active[s] = (m.bits[s >> 5] >> (s & 31)) & 1u;
}
void launch_set_active(int *active, int nslots, const uint32_t bits[kMaxSlots / 32], hipStream_t s) {
    ActiveMask m;
    for (int k = 0; k < kMaxSlots / 32; ++k) m.bits[k] = bits[k];
    hipLaunchKernelGGL(k_set_active, dim3((nslots + 255) / 256), dim3(256), 0, s, active, nslots, m);
}
void launch_icp_iter(const SessParams *P, const WorkItem *work, int n, int nsess, int level, int iter,
                     hipStream_t s) {
    if (n <= 0) return;
    static_assert(kMaxLevels == 3, "one launch case per level");
    // one instantiation per distinct group size in use
    if (level == 0)
        hipLaunchKernelGGL(k_icp_iter<icp_group(0)>, dim3(n), dim3(kTileThreads), 0, s, P, work, level, iter);
    else if (level == 1)
        hipLaunchKernelGGL(k_icp_iter<icp_group(1)>, dim3(n), dim3(kTileThreads), 0, s, P, work, level, iter);
    else
        hipLaunchKernelGGL(k_icp_iter<icp_group(2)>, dim3(n), dim3(kTileThreads), 0, s, P, work, level, iter);
    // 16 waves read a 1280x960 frame's 600 partials fastest when the chip is
    // otherwise idle (fused frame with preview 1177 us with 4 waves, 1125 with
    // 16), but have to wait for a CU with room for all of them while the other
    // parts of a large batch fill it (64 sessions: 6.27 ms a step with 2 or 4
    // waves, 6.35 with 8, 6.30 with 1; 24-slot server 889 us with 4 and 958
    // with 1)
    if (nsess <= 4)
        hipLaunchKernelGGL(k_icp_solve<kStepThreads>, dim3(nsess), dim3(kStepThreads), 0, s, P, nsess, level, iter);
    else
        hipLaunchKernelGGL(k_icp_solve<kTileThreads>, dim3(nsess), dim3(kTileThreads), 0, s, P, nsess, level, iter);
}
void launch_icp_step(const SessParams *P, const WorkItem *work, int n, int level, int iter, int seq, int prev,
                     hipStream_t s) {
    if (n <= 0) return;
#if VS_ICP_MFMA
    if (level == 0)
        hipLaunchKernelGGL(k_icp_step<icp_group(0)>, dim3(n), dim3(kStepThreads), 0, s, P, work, level, iter, seq,
                           prev);
    else if (level == 1)
        hipLaunchKernelGGL(k_icp_step<icp_group(1)>, dim3(n), dim3(kStepThreads), 0, s, P, work, level, iter, seq,
                           prev);
    else
        hipLaunchKernelGGL(k_icp_step<icp_group(2)>, dim3(n), dim3(kStepThreads), 0, s, P, work, level, iter, seq,
                           prev);
#endif
}
void launch_icp_finish(const SessParams *P, int nsess, unsigned *bricks, int seq, int prev, hipStream_t s) {
    hipLaunchKernelGGL(k_icp_finish, dim3(nsess), dim3(kStepThreads), 0, s, P, bricks, seq, prev);
}
void launch_track_finalize(const SessParams *P, int nsess, unsigned *bricks, hipStream_t s) {
    hipLaunchKernelGGL(k_track_finalize, dim3((nsess + 63) / 64), dim3(64), 0, s, P, nsess, bricks);
}
void launch_integrate_begin(const SessParams *P, unsigned *bricks, hipStream_t s) {
    hipLaunchKernelGGL(k_integrate_begin, dim3(1), dim3(64), 0, s, P, bricks);
}
void launch_set_pose(const SessParams *P, const double *T, int reset, const int *frames, hipStream_t s) {
    Mat16d m;
    for (int k = 0; k < 16; ++k) m.m[k] = T ? T[k] : ((k % 5) == 0 ? 1.0 : 0.0);
    hipLaunchKernelGGL(k_set_pose, dim3(1), dim3(64), 0, s, P, m, reset, frames != nullptr, frames ? *frames : 0);
}
// Sum of one ICP system's tile partials in tile order: thread k adds term k
// of tiles 0, 1, ..., nt-1 in FP64, the order of vs_icp_system's host loop,
// so both give the same bits.
__global__ void k_icp_sum_tiles(const double *__restrict__ part, int nt, double *__restrict__ out) {
    const int k = threadIdx.x;
    if (k >= kIcpVals) return;
    double s = 0.0;
    for (int t = 0; t < nt; ++t) s += ldg(part, (size_t)t * kIcpVals + k);
    stg(out, k, s);
}
void launch_icp_sum_tiles(const double *part, int nt, double *out, hipStream_t s) {
    hipLaunchKernelGGL(k_icp_sum_tiles, dim3(1), dim3(64), 0, s, part, nt, out);
}
void launch_icp_system(const SessParams *P, const WorkItem *work, int n, int level, const float *T21,
                       double *out_part, uint8_t *mask, hipStream_t s) {
    Mat16f m;
    for (int k = 0; k < 16; ++k) m.m[k] = T21[k];
    if (n > 0)
        hipLaunchKernelGGL(k_icp_system, dim3(n), dim3(kTileThreads), 0, s, P, work, level, m, out_part, mask);
}

}  // namespace vs
