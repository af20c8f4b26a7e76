// gps_kernels.h — launch interface of the gfx950 kernels (gps_kernels.hip).
#pragma once

#include "gps_internal.h"

namespace gps {

struct PreprocessArgs {
    DevScene scene;
    FrameConsts f;
    uint32_t* maskA;
    uint32_t* maskB;
    const uint32_t* iteration;
    uint32_t* weights;
    SplatRecord* recs;
    uint32_t* tile_sum;
    uint32_t* tile_cnt;
    CullView cull;
    HiZView hiz;
    const uint8_t* gocc = nullptr;  // occluded-group bytes of this pass (group cull), or null
    // one byte per workgroup, 0 when the block cull culled its block (and
    // zeroed its mask words), or null; needs gaussians_per_block a multiple of 256
    const uint8_t* wg_live = nullptr;
    uint2* bounds = nullptr;      // the records' bounds again, for the binned splat's lists, or null
    uint32_t* rejects = nullptr;  // 2 x 9 reject-reason counters + 2 group checks (diagnostic), or null
};

struct BinnedArgs;
struct DistributeArgs {
    const BinnedArgs* bin = nullptr;  // the pass may be binned: count its regions' points too
    uint32_t* tile_sum;
    uint32_t* tile_cnt;
    uint32_t ntiles;
    uint32_t* tile_off;
    uint32_t* tile_voff;
    PassCounters* ctr;
    uint32_t budget;
    const uint32_t* weights;
    uint32_t* cidx;
    uint32_t* coff;
    uint32_t* chunk_start;
    uint32_t* iteration;
    CullView cull;
    int32_t hier;
    uint32_t N;
};

// The tile sums of a pass without a scan launch, for the splat kernel to clear
// (n = 0: the pass had one, distribute_kernel has cleared them).
struct TileSums {
    uint32_t *sum, *cnt;
    uint32_t n;
    uint32_t* iteration;
};

// (entry, start) items of the Gaussians too large to bin (big_items): the first
// slices, one per Gaussian, then slice_cap further ones from items[slice0] on.
struct BigList {
    uint2* items;
    uint32_t slice0, slice_cap;
};

struct SplatArgs {
    const SplatRecord* recs;
    const uint32_t* cidx;
    const uint32_t* coff;
    const uint32_t* chunk_start;
    const PassCounters* ctr;
    uint64_t* fb;
    uint32_t* atomics_count;
    int32_t spp, K, up_w, unbiased;
    uint32_t frame_seed;
    uint32_t grid;   // multiple of xcds
    int32_t xcds;    // accelerator complex dies (workgroups round-robin over them)
    // a pass that may be binned: when the binned splat did not stand down
    // (bin_state[3] == 0) only its big slices are splatted
    const uint32_t* bin_state = nullptr;
    BigList big{};
    TileSums sums{};
};

// Ordered point-parallel splat (dense passes, GPS_ORD_BINS): the splat
// arguments plus the ordering buffers.
struct OrderedArgs {
    SplatArgs s;
    int32_t up_w, up_h;       // framebuffer pixels of this frame
    int32_t forced;           // order whatever the density
    int32_t pre_test;         // the framebuffer holds an earlier pass: phase 0 tests too
    uint16_t* bucket;         // per chunk
    uint32_t* hist;           // GPS_ORD_BINS, zero between passes
    uint32_t* lim;            // GPS_ORD_PHASES
    uint32_t* tmax;           // per 16x16 tile of the framebuffer
    uint32_t ntiles;          // 16x16 tiles of this frame's framebuffer
    int32_t tw64;             // 64x64 tiles per framebuffer row
    uint32_t cus;
    uint32_t* skipped_count;  // points skipped (diagnostic; may be null)
};
void launch_ordered_splat(const OrderedArgs& a, hipStream_t st);

// Splat constants shared by the point-parallel and the binned splat.
struct SplatConsts {
    int32_t spp, K, up_w, unbiased;
    uint32_t frame_seed;
    int32_t xcds;
};

struct BinnedArgs {
    const SplatRecord* recs;
    const uint32_t* cidx;
    const uint32_t* coff;
    const PassCounters* ctr;
    BinGeom g;
    SplatConsts sc;
    uint64_t background;
    uint64_t* fb;
    int32_t fresh;        // the frame's first pass: the framebuffer holds only the background
    uint64_t clear_words; // framebuffer words that the lists' kernel still has to clear (0: cleared)
    const uint2* bounds;  // (bmin, bmax) per record (PreprocessArgs::bounds)
    unsigned long long* reg_pts;  // points per region, zero between passes
    uint32_t *reg_ptot, *reg_poff, *reg_cursor;
    uint32_t *job_reg, *job_p0;
    uint2* list;          // (record, point) of every point and region, region by region
    BigList big;
    uint32_t* state;      // 8 words: (entry, region) pairs, jobs, points per job, stand-down, job cursor, unused,
                          // big Gaussians and further slices (one 64-bit counter)
    uint32_t list_cap, job_cap;
    uint32_t cus;
    uint32_t dense_points;  // more points than this: the binned kernels stand down (state[3] = 2)
    uint32_t sparse_points; // fewer: likewise (state[3] = 3)
    uint32_t* atomics_count;
};
bool binned_geometry(int up_w, int up_h, int spp, BinGeom* g);
// Whether the automatic choice may bin a frame of N Gaussians, and the points
// above which such a frame is too dense to bin, tested on the device; `views`: of a
// batch, 0 for a single frame
// (GPS_BIN_AUTO_SAMPLES, GPS_BIN_DENSE_SAMPLES; a point writes K * spp samples
// into up_w * up_h * spp words).
bool binned_auto(int up_w, int up_h, int spp, int K, uint64_t N, bool occl, int views);
uint32_t binned_dense_points(int up_w, int up_h, int spp, int K, bool batch);
uint32_t binned_sparse_points(int up_w, int up_h, int spp, int K);  // too few (single frames)
void launch_binned_splat(const BinnedArgs& a, hipStream_t st);

// Binned splat buffers of a batch: entries are the batch's compacted entries,
// regions those of all binned views (view v owns [rbase, rbase + nregions)).
struct BatchBinArgs {
    int32_t any;                // at least one view is binned
    uint32_t views;             // views with binned regions
    uint32_t nregions;          // regions of all binned views
    uint32_t max_view_regions;  // largest view's regions (LDS histogram size)
    uint2* bounds;
    BigList big;
    unsigned long long* reg_pts;
    uint32_t *reg_ptot, *reg_poff, *reg_cursor;
    uint32_t *job_reg, *job_p0;
    uint2* list;                // as BinnedArgs::list
    uint32_t* state;            // as BinnedArgs::state
    uint32_t list_cap, job_cap;
    uint32_t cus;
};

// Multi-view batch (see the batch kernels): all arrays are concatenated per view.
struct BatchArgs {
    DevScene scene;
    BatchView* views;        // device table, nviews entries
    int32_t nviews;
    uint32_t npad;           // per-view stride of weights / records (multiple of the tile)
    uint32_t tiles_per_view;
    uint32_t* weights;
    SplatRecord* recs;
    uint32_t *tile_sum, *tile_cnt, *tile_off, *tile_voff;
    uint32_t *cidx, *coff;
    uint8_t* cview;
    uint32_t* chunk_start;
    PassCounters* ctr;
    uint32_t* iteration;     // scratch word (the scan flips it)
    CullView cull;           // mask = first view's mask
    uint32_t mask_stride;
    int32_t hier;
    uint64_t* fb;            // pool; views address it by fb_offset
    uint64_t max_fb_words;   // largest view
    int32_t fb_key32;        // every word of the batch's views has a 32-bit index (below 2^32 - 1)
    uint32_t grid;
    int32_t xcds;
    int32_t threads, ppt;    // splat variant
    int32_t pre_views;       // views one preprocess workgroup evaluates (0: all)
    uint32_t* atomics;
    BatchBinArgs bin;
};
extern const int kBatchSplatVariants[][2];
extern const int kNumBatchSplatVariants;
extern const int kBatchPreViews[];
extern const int kNumBatchPreViews;
void launch_batch_clear(const BatchArgs& a, hipStream_t st);
void launch_batch_cull(const BatchArgs& a, hipStream_t st);
void launch_batch_preprocess(const BatchArgs& a, hipStream_t st);
void launch_batch_distribute(const BatchArgs& a, hipStream_t st);
bool launch_batch_splat(const BatchArgs& a, hipStream_t st);
void launch_batch_binned(const BatchArgs& a, hipStream_t st);
void launch_batch_bin_big(const BatchArgs& a, hipStream_t st);

// Fills the framebuffer with `value`; also zeroes n0 words at z0 and n1 at z1.
void launch_clear(uint64_t* fb, uint64_t words, uint64_t value, hipStream_t st, uint32_t* z0 = nullptr,
                  uint32_t n0 = 0, uint32_t* z1 = nullptr, uint32_t n1 = 0);
// `live` (or null): the unculled blocks are listed there, their count in
// *live_count (zeroed by the frame's clear).  `wg_live` (or null): one byte
// per 256-Gaussian preprocess workgroup, 0 when its block is culled (blocks
// must be whole workgroups), and the culled blocks' valid-mask words zeroed
// in the preprocess's current mask (maskA / maskB by *iteration).
void launch_cull(const CullView& cv, const float planes[24], const Mat4& vp, const HiZView& h, int occl,
                 uint32_t* culled_count, uint32_t* live, uint32_t* live_count, uint32_t* maskA, uint32_t* maskB,
                 const uint32_t* iteration, uint8_t* wg_live, uint32_t N, hipStream_t st);
void launch_preprocess(const PreprocessArgs& a, hipStream_t st);
void launch_distribute(const DistributeArgs& a, hipStream_t st);
void launch_splat(const SplatArgs& a, hipStream_t st);
void launch_combine(const uint64_t* fb, float* color, float* depth, int W, int H, int ss, int spp, float near_plane,
                    float far_plane, int depth_only, hipStream_t st);
void launch_hiz_build(const HiZView& h, const float* depth, int kmin, uint32_t* ticket, hipStream_t st);
void launch_zero_u32(uint32_t* p, uint32_t n, hipStream_t st);
void launch_fill_f32(float* p, uint32_t n, float v, hipStream_t st);
void launch_build_nodes(const DevScene& s, uint32_t gpb, uint32_t nb, CullNode* nodes, hipStream_t st);
// Bounds of every group of GPS_GROUP Gaussians (once per pass), and the
// per-pass conservative group occlusion test against the pass's Hi-Z chain.
void launch_group_boxes(const DevScene& s, GroupBox* boxes, uint32_t count, hipStream_t st);
void launch_group_cull(const GroupView& gv, const FrameConsts& f, const HiZView& h, uint32_t* culled_count,
                       hipStream_t st);
void launch_group_cull_live(const GroupView& gv, const CullView& cv, const uint32_t* live, const uint32_t* live_count,
                            uint32_t N, const FrameConsts& f, const HiZView& h, uint32_t grid,
                            uint32_t* culled_count, hipStream_t st);
void launch_taa(const float* cur, const float* cur_depth, const float* prev, const Mat4& M, float blend, int W, int H,
                int frame_number, float* out, uint8_t* rgb8, hipStream_t st);
void launch_progressive(float* color, float* accum, int W, int H, int n, uint8_t* rgb8, hipStream_t st);
void launch_materialize_indices(const uint32_t* cidx, const uint32_t* coff, const PassCounters* ctr, uint32_t* out,
                                uint32_t max_points, hipStream_t st);

}  // namespace gps
