// vs_launch.hpp — host-side launchers of the fusion kernels. Every launcher
// takes the device array of session parameters and a work list; n is the
// number of work items (one workgroup each) unless stated otherwise.
#pragma once

#include "vs_device.hpp"

#ifndef VS_ICP_STEP_GROUPS
#define VS_ICP_STEP_GROUPS 256  // (0 with VS_ICP_MFMA=0: the form exists for the matrix-core sums only)
#endif
namespace vs {

// image stages (vs_img.hip)
constexpr int kDepthChunk = 64;
struct DepthChunk {  // passed by value: device frame pointers and the batch slots they go to
    const uint16_t *src[kDepthChunk];
    int slot[kDepthChunk];
    int n;
};
void launch_gather_depth(const SessParams *P, const DepthChunk &ch, hipStream_t s);
// image buffers of a new session (P[0]; npx level-0 pixels; keys: launch_depth_reproject's)
void launch_session_init(const SessParams *P, size_t npx, uint32_t *keys, hipStream_t s);
// force (here and below): run also for sessions whose state does not have a
// frame in a step (the single operators)
// out (nullable, single session): the filtered frame also goes there
void launch_bilateral(const SessParams *P, const WorkItem *work, int n, int force, float *out, hipStream_t s);
// levels 1 .. levels - 1 from level 0; pair: no session has exactly two levels
void launch_pyramid(const SessParams *P, const WorkItem *const work[kMaxLevels], const int n[kMaxLevels], int levels,
                    bool pair, int force, hipStream_t s);
void launch_vnmap(const SessParams *P, const WorkItem *work, int n, int level, float *vtx, float *nrm, hipStream_t s);
// single session (P[0]), the reference loop's in-place order of a W x H level;
// scratch: vn_words(W) * H 64-bit words that no other call uses meanwhile, null:
// the vertex map serves
constexpr int vn_words(int W) { return (W + 63) / 64; }
void launch_vnmap_inplace(const SessParams *P, const WorkItem *work, int n, int level, int W, int H, void *scratch,
                          float *vtx, float *nrm, hipStream_t s);

// tracker (vs_icp.hip); nsess = sessions in the batch
void launch_track_setup(const SessParams *P, int nsess, const double *T_init, hipStream_t s);
// slot-table form: active[s] != 0 selects the slots that fuse this step
constexpr int kMaxSlots = 256;
void launch_track_setup_active(const SessParams *P, int nsess, const int *active, hipStream_t s);
void launch_set_active(int *active, int nslots, const uint32_t bits[kMaxSlots / 32], hipStream_t s);
void launch_icp_iter(const SessParams *P, const WorkItem *work, int n, int nsess, int level, int iter,
                     hipStream_t s);
// bricks: the step's brick counter, which this launch and launch_icp_finish
// then reset with the sessions' integrate counters (integrate_begin); null: no
// integration follows, the counters stay
void launch_track_finalize(const SessParams *P, int nsess, unsigned *bricks, hipStream_t s);
// The one-launch form of an iteration, for launches of up to kIcpStepGroups
// level-0 groups, a CU each for their 16-wave workgroups. Fused frame with
// preview, two launches / one: 38 groups (320x240) 443 / 398 us, 150
// (640x480) 509 / 463, 136 with colour 550 / 506; beyond it, 600 groups
// (1280x960) 1125 / 1246 and a 24-slot server's 2291 1295 / 1359 (these two
// with a shorter solve on both sides).
constexpr int kIcpStepGroups = VS_ICP_STEP_GROUPS;
// seq: 1, 2, ... over the launches of one track; prev: the level of launch seq - 1
// (-1: none); work null: a single session's groups 0..n-1
void launch_icp_step(const SessParams *P, const WorkItem *work, int n, int level, int iter, int seq, int prev,
                     hipStream_t s);
// the last iteration's solve, then launch_track_finalize's work
void launch_icp_finish(const SessParams *P, int nsess, unsigned *bricks, int seq, int prev, hipStream_t s);
// integrate_begin alone, for an integration without a track (single session)
void launch_integrate_begin(const SessParams *P, unsigned *bricks, hipStream_t s);
// one system, no solve: writes 29 doubles (+ optional mask) for diagnostics
void launch_icp_system(const SessParams *P, const WorkItem *work, int n, int level, const float *T21,
                       double *out_part, uint8_t *mask, hipStream_t s);
// the 29 sums of nt tile partials, in tile order, into out (one workgroup)
void launch_icp_sum_tiles(const double *part, int nt, double *out, hipStream_t s);

// volume stages (vs_vol.hip)
struct BrickList {
    int2 *items;        // (session, brick)
    unsigned *count;    // device counter
    unsigned capacity;
};
// marks the visible bricks' bits, then compacts every session's bits into
// the brick list (max_words: the longest bitmap of the nsess sessions)
void launch_vis_mark(const SessParams *P, const WorkItem *work, int n, int nsess, uint32_t max_words, BrickList bl,
                     int force, hipStream_t s);
// sd_slices: the most superbricks along z of any session (distance field)
void launch_integrate(const SessParams *P, int nsess, BrickList bl, int tsdf_type, int weight_type, int grid,
                      int sd_slices, hipStream_t s);
// How the raycast addresses the sessions of a launch: 32-bit offsets when
// every session's voxel records are below 4 GB, and then a compile-time
// superbrick size when every session has the one of grids up to 512^3 (whose
// records are at most 1 GB). The form for mixed and large grids reads the
// superbrick size per session.
enum VoxAddr { kAddrSmall = 0, kAddr32 = 1, kAddr64 = 2 };
// Caller buffers of a single session's maps at one level (each nullable):
// depth, vertex and normal (3 floats per pixel), image.
struct MapsOut {
    float *depth, *vtx, *nrm;
    uint8_t *img;
};
void launch_raycast(const SessParams *P, const WorkItem *work, int n, int level, int tsdf_type, int weight_type,
                    int addr, const MapsOut *out, hipStream_t s);
// Several pyramid levels in one launch: segment k of the grid is level
// level[k]'s work list (passed by value).
struct LevelWork {
    const WorkItem *w[kMaxLevels];
    int n[kMaxLevels];
    int level[kMaxLevels];
    int nseg;
    int force;
    int blocks() const {
        int t = 0;
        for (int k = 0; k < nseg; ++k) t += n[k];
        return t;
    }
};
LevelWork level_work(const WorkItem *const work[kMaxLevels], const int n[kMaxLevels], int levels);
// superbrick distance field of sessions P[0..nsess) (only those that gained
// a band superbrick unless force); sd_slices >= every session's sdim[2]
void launch_sdist(const SessParams *P, int nsess, int sd_slices, int force, hipStream_t s);
// Ray block of one wave in the raycast kernels (same results for each).
enum RayBlock { kRay8x8 = 0, kRay16x4 = 1, kRay32x2 = 2 };
// groups: the workgroups that decide the march's form (0: the launch's own);
// addr: VoxAddr
void launch_raycast_march(const SessParams *P, const LevelWork &lw, int tsdf_type, int weight_type,
                          unsigned long long *stats, int ray_block, int groups, int addr, hipStream_t s);
// waves: the waves per SIMD its registers aim for (4 or 5); addr: VoxAddr
void launch_raycast_shade(const SessParams *P, const LevelWork &lw, int tsdf_type, int weight_type,
                          unsigned long long *stats, int ray_block, int waves, int addr, hipStream_t s);
// volume maintenance (single session, P points at its parameters)
void launch_volume_init(const SessParams *P, size_t nvox, int tsdf_type, int weight_type, uint32_t nwords,
                        hipStream_t s);
void launch_volume_to_linear(const SessParams *P, size_t nvox, int tsdf_type, int weight_type, float *F, float *Wt,
                             hipStream_t s);
void launch_volume_from_linear(const SessParams *P, size_t nvox, int tsdf_type, int weight_type, const float *F,
                               const float *Wt, hipStream_t s);
// idx (nullable): only these nbricks bricks, of a volume whose other bricks are
// as launch_volume_init leaves them
void launch_occupancy_rebuild(const SessParams *P, const uint32_t *idx, uint32_t nbricks, int tsdf_type,
                              int weight_type, int sd_slices, hipStream_t s);
void launch_color_to_linear(const SessParams *P, size_t nvox, uint8_t *rgb, hipStream_t s);
// input pre-steps (vs_pre.hip); is_float selects float metres, else uint16 mm;
// key: dw * dh words, all ones before and after a call
void launch_depth_reproject(int is_float, const void *src, int sw, int sh, const float Ks[4], const float Kd[4],
                            const float T[16], uint32_t *key, void *dst, int dw, int dh, hipStream_t s);
void launch_depth_crop(const SessParams *P, int is_float, void *depth, int w, int h, const float K[4],
                       const float *Tcg, hipStream_t s);
// g_uvv carving: reset visible bricks with no valid voxel; *carved += their count
void launch_carve(const SessParams *P, int tsdf_type, int weight_type, const uint8_t *valid, unsigned *carved,
                  hipStream_t s);
// snapshots: copy the listed bricks into (unpack = 0) or out of (1) a packed buffer
void launch_brick_pack(const SessParams *P, const uint32_t *idx, unsigned n, int value_bytes, int weight_bytes,
                       int color_bytes, uint8_t *buf, int unpack, hipStream_t s);

}  // namespace vs
