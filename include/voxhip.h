/*
 * voxhip.h -- C ABI of the voxurf_amd HIP library (libvoxhip.so, gfx950).
 *
 * Every entry point takes plain device pointers, element counts, scalars and the
 * hipStream_t to launch on (passed as void*, NULL = the null stream), and returns a
 * status code (VX_OK = 0).  On failure vx_last_error() returns a thread-local message.
 * Nothing here allocates or frees caller-visible memory: outputs and workspaces are
 * provided by the caller.  Index outputs are int64, matching the reference's tensors.
 *
 * `dtype` selects the floating type of the float arrays: VX_F32 or VX_F64 (the
 * reference dispatches both through AT_DISPATCH_FLOATING_TYPES).
 *
 * Each declaration cites the reference interface it replaces (paths relative to the
 * Voxurf repository).
 */
#ifndef VOXHIP_H
#define VOXHIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum { VX_OK = 0, VX_ERR_ARG = 1, VX_ERR_LAUNCH = 2, VX_ERR_SIZE = 3, VX_ERR_DTYPE = 4 };
enum { VX_F32 = 0, VX_F64 = 1 };

const char* vx_last_error(void);
int vx_version(void);
/* Hash of this header the library was built against (bindings refuse a mismatch). */
const char* vx_abi_hash(void);

/* ---- render_utils: ray sampling ------------------------------------------------ */

/* lib/cuda/render_utils.cpp:50-58 infer_t_minmax (kernel render_utils_kernel.cu:12-35). */
int vx_infer_t_minmax(int dtype, const void* rays_o, const void* rays_d, const void* xyz_min,
                      const void* xyz_max, float near_, float far_, int64_t n_rays,
                      void* t_min, void* t_max, void* stream);

/* lib/cuda/render_utils.cpp:60-65 infer_n_samples (render_utils_kernel.cu:38-55). */
int vx_infer_n_samples(int dtype, const void* rays_d, const void* t_min, const void* t_max,
                       float stepdist, int64_t n_rays, int64_t* n_samples, void* stream);

/* lib/cuda/render_utils.cpp:67-72 infer_ray_start_dir (render_utils_kernel.cu:58-79). */
int vx_infer_ray_start_dir(int dtype, const void* rays_o, const void* rays_d, const void* t_min,
                           int64_t n_rays, void* rays_start, void* rays_dir, void* stream);

/* lib/cuda/render_utils.cpp:74-85 sample_pts_on_rays, phase 1 of 2
 * (render_utils_kernel.cu:196-212: t_min/t_max, N_steps, N_steps.cumsum, total).
 * Writes t_min/t_max [n_rays], n_steps [n_rays], n_steps_cumsum [n_rays] (inclusive)
 * and total [1] (device).  `scan_ws` is a device workspace of
 * vx_scan_workspace_elems(n_rays) int64 elements. */
int vx_sample_pts_count(int dtype, const void* rays_o, const void* rays_d, const void* xyz_min,
                        const void* xyz_max, float near_, float far_, float stepdist,
                        int64_t n_rays, void* t_min, void* t_max, int64_t* n_steps,
                        int64_t* n_steps_cumsum, int64_t* total, int64_t* scan_ws,
                        void* stream);

/* No counterpart in the reference: vx_sample_pts_count without the `scan_ws` workspace,
 * for callers that cannot allocate device memory (code under HIP graph capture, serving
 * loops and harnesses that forbid hipMalloc).  Same arguments, outputs and errors as
 * vx_sample_pts_count; the scan's scratch is a fixed 64 KiB device array per GPU, so
 * n_rays is limited to 8,388,608 (larger returns VX_ERR_ARG before any launch).  The
 * array is shared by every call on a GPU: calls that overlap on one GPU race.  The
 * stream must belong to the current device.  Allocates nothing. */
int vx_sample_pts_count_noalloc(int dtype, const void* rays_o, const void* rays_d,
                                const void* xyz_min, const void* xyz_max, float near_,
                                float far_, float stepdist, int64_t n_rays, void* t_min,
                                void* t_max, int64_t* n_steps, int64_t* n_steps_cumsum,
                                int64_t* total, void* stream);

/* Phase 2 (render_utils_kernel.cu:213-241): fills rays_pts [M,3], mask_outbbox [M]
 * (bool, 1 byte), ray_id [M], step_id [M] for M = n_steps_cumsum[n_rays-1]. */
int vx_sample_pts_fill(int dtype, const void* rays_o, const void* rays_d, const void* xyz_min,
                       const void* xyz_max, const void* t_min, float stepdist, int64_t n_rays,
                       const int64_t* n_steps_cumsum, int64_t total, void* rays_pts,
                       uint8_t* mask_outbbox, int64_t* ray_id, int64_t* step_id, void* stream);

/* Scratch size (int64 elements) the inclusive scan of vx_sample_pts_count needs. */
int64_t vx_scan_workspace_elems(int64_t n);

/* Inclusive prefix sum of n int64 values (used by sample_pts_on_rays and segment
 * offsets); `ws` as for vx_sample_pts_count. */
int vx_inclusive_scan_i64(const int64_t* in, int64_t* out, int64_t n, int64_t* ws, void* stream);

/* lib/cuda/render_utils.cpp:87-98 sample_ndc_pts_on_rays (render_utils_kernel.cu:244-293).
 * rays_pts [n_rays,N_samples,3], mask_outbbox [n_rays,N_samples]. */
int vx_sample_ndc_pts_on_rays(int dtype, const void* rays_o, const void* rays_d,
                              const void* xyz_min, const void* xyz_max, int n_samples,
                              int64_t n_rays, void* rays_pts, uint8_t* mask_outbbox,
                              void* stream);

/* lib/cuda/render_utils.cpp:100-107 sample_bg_pts_on_rays (render_utils_kernel.cu:300-360). */
int vx_sample_bg_pts_on_rays(int dtype, const void* rays_o, const void* rays_d,
                             const void* t_max, float bg_preserve, int n_samples,
                             int64_t n_rays, void* rays_pts, void* stream);

/* lib/cuda/render_utils.cpp:109-118 maskcache_lookup (render_utils_kernel.cu:367-424).
 * world [sz_i,sz_j,sz_k] bool bytes; out [n_pts] bool bytes (fully written). */
int vx_maskcache_lookup(int dtype, const uint8_t* world, const void* xyz, const void* scale,
                        const void* shift, int sz_i, int sz_j, int sz_k, int64_t n_pts,
                        uint8_t* out, void* stream);

/* lib/cuda/ub360_utils.cpp:16-19 cumdist_thres (ub360_utils_kernel.cu:12-47): dist
 * [n_rays, n_pts] (contiguous) -> mask [n_rays, n_pts] bool bytes (fully written): per
 * ray, a float running sum of dist restarting after every point where it exceeds thres. */
int vx_cumdist_thres(int dtype, const void* dist, float thres, int64_t n_rays, int64_t n_pts,
                     uint8_t* mask, void* stream);

/* ---- render_utils: alpha and transmittance ------------------------------------- */

/* lib/cuda/render_utils.cpp:120-124 raw2alpha (render_utils_kernel.cu:431-481). */
int vx_raw2alpha(int dtype, const void* density, float shift, float interval, int64_t n_pts,
                 void* exp_d, void* alpha, void* stream);
/* lib/cuda/render_utils.cpp:125-129 raw2alpha_nonuni (render_utils_kernel.cu:446-504). */
int vx_raw2alpha_nonuni(int dtype, const void* density, float shift, const void* interval,
                        int64_t n_pts, void* exp_d, void* alpha, void* stream);
/* lib/cuda/render_utils.cpp:131-135 raw2alpha_backward (render_utils_kernel.cu:507-552). */
int vx_raw2alpha_backward(int dtype, const void* exp_d, const void* grad_back, float interval,
                          int64_t n_pts, void* grad, void* stream);
/* lib/cuda/render_utils.cpp:136-140 raw2alpha_nonuni_backward (render_utils_kernel.cu:520-574). */
int vx_raw2alpha_nonuni_backward(int dtype, const void* exp_d, const void* grad_back,
                                 const void* interval, int64_t n_pts, void* grad, void* stream);

/* lib/cuda/render_utils.cpp:142-149 alpha2weight (render_utils_kernel.cu:577-651).
 * Outputs weight [n_pts], T [n_pts], alphainv_last [n_rays], i_start/i_end [n_rays];
 * the function initialises all of them itself (weight=0, T=1, alphainv_last=1,
 * i_start=i_end=0 before the scan) and needs no host synchronisation. */
int vx_alpha2weight(int dtype, const void* alpha, const int64_t* ray_id, int64_t n_pts,
                    int64_t n_rays, void* weight, void* T, void* alphainv_last,
                    int64_t* i_start, int64_t* i_end, void* stream);

/* lib/cuda/render_utils.cpp:151-167 alpha2weight_backward (render_utils_kernel.cu:654-707).
 * grad [n_pts] is fully written (zero outside every ray's [i_start, i_end)). */
int vx_alpha2weight_backward(int dtype, const void* alpha, const void* weight, const void* T,
                             const void* alphainv_last, const int64_t* i_start,
                             const int64_t* i_end, int64_t n_pts, int64_t n_rays,
                             const void* grad_weights, const void* grad_last, void* grad,
                             void* stream);

/* ---- dense grids --------------------------------------------------------------- */
/* A grid is described by geom[8] = {C, X, Y, Z, stride_c, stride_x, stride_y, stride_z}
 * (element strides): the reference's contiguous [1,C,X,Y,Z] tensor and the
 * channels-last layout are both accepted.  xyz_min/xyz_max are [3] device arrays. */

/* lib/grid.py:47-58 DenseGrid.forward (F.grid_sample, bilinear, align_corners=True,
 * zero padding): out [n, C]. */
int vx_grid_sample_fwd(int dtype, const void* grid, const int64_t* geom, const void* xyz,
                       const void* xyz_min, const void* xyz_max, int64_t n, void* out,
                       void* stream);
/* Adjoint of vx_grid_sample_fwd w.r.t. the grid (the grid_sample backward autograd
 * runs for lib/grid.py:54): grad += scatter of gout [n, C] (atomic adds). */
int vx_grid_sample_bwd(int dtype, void* grad, const int64_t* geom, const void* xyz,
                       const void* xyz_min, const void* xyz_max, int64_t n, const void* gout,
                       void* stream);

/* lib/voxurf_fine.py:537-577 Voxurf.sample_sdfs: feat [n, 6*nd], grad [n, 3*nd] (zyx
 * component order, as the reference), disp [nd] device array of displacements. */
int vx_sample_sdfs_fwd(int dtype, const void* grid, const int64_t* geom, const void* xyz,
                       const void* xyz_min, const void* xyz_max, const void* disp, int nd,
                       double voxel_size, int use_grad_norm, int64_t n, void* feat, void* grad,
                       void* stream);
/* Adjoint of vx_sample_sdfs_fwd: ggrid += d(feat, grad)/d(grid)^T (gfeat, ggrad);
 * either gradient may be NULL. */
int vx_sample_sdfs_bwd(int dtype, void* ggrid, const void* grid, const int64_t* geom,
                       const void* xyz, const void* xyz_min, const void* xyz_max,
                       const void* disp, int nd, double voxel_size, int use_grad_norm, int64_t n,
                       const void* gfeat, const void* ggrad, void* stream);

/* lib/voxurf_fine.py:502-534 Voxurf.grid_sampler(xyz, sdf_grid, sample_ret=True,
 * sample_grad=True): sdf [n], gradient [n,3] (xyz order), feat [n,6] (may be NULL). */
int vx_sdf_grad_fwd(int dtype, const void* grid, const int64_t* geom, const void* xyz,
                    const void* xyz_min, const void* xyz_max, double voxel_size, int64_t n,
                    void* sdf, void* grad, void* feat, void* stream);
/* Adjoint of vx_sdf_grad_fwd; gsdf / ggrad / gfeat may be NULL. */
int vx_sdf_grad_bwd(int dtype, void* ggrid, const int64_t* geom, const void* xyz,
                    const void* xyz_min, const void* xyz_max, double voxel_size, int64_t n,
                    const void* gsdf, const void* ggrad, const void* gfeat, void* stream);

/* lib/voxurf_fine.py:440-450 neus_sdf_gradient(mode='interpolate'): sdf [X,Y,Z] ->
 * out [3,X,Y,Z]; and its adjoint (gsdf += ...). */
int vx_dense_sdf_gradient_fwd(int dtype, const void* sdf, int X, int Y, int Z, double voxel_size,
                              void* out, void* stream);
int vx_dense_sdf_gradient_bwd(int dtype, const void* gout, int X, int Y, int Z,
                              double voxel_size, void* gsdf, void* stream);

/* lib/cuda/total_variation.cpp:16-20 total_variation_add_grad
 * (total_variation_kernel.cu:13-35, 68-98): grad += TV gradient, in place. */
int vx_total_variation_add_grad(int dtype, const void* param, void* grad, const int64_t* geom,
                                float wx, float wy, float wz, int dense_mode, void* stream);
/* lib/cuda/total_variation.cpp:22-27 total_variation_add_grad_new
 * (total_variation_kernel.cu:38-66, 101-133); mask has the grid's layout. */
int vx_total_variation_add_grad_new(int dtype, const void* param, void* grad, const void* mask,
                                    const int64_t* geom, float wx, float wy, float wz,
                                    int dense_mode, void* stream);

/* lib/voxurf_fine.py:930-942 MaskCache.forward (also lib/dvgo_ori.py:440-473): out [n]
 * = 1 - exp(-softplus(density(xyz) + act_shift) * voxel_size_ratio) >= thres, with the
 * density looked up trilinearly (nearest = 0) or at the nearest lattice point. */
int vx_maskcache_alpha(int dtype, const void* density, const int64_t* geom, const void* xyz,
                       const void* xyz_min, const void* xyz_max, double act_shift,
                       double voxel_size_ratio, double thres, int nearest, int64_t n,
                       uint8_t* out, void* stream);

/* ---- camera rays and the MaskCache ray pre-filter --------------------------------
 * cam: 26 floats in host memory, {H, W, K[0][0], K[1][1], K[0][2], K[1][2], c2w[:3,:3]
 * row-major (9), c2w[:3,3] (3), pixel offset (0.5 'center' / 0 'lefttop'), inverse_y,
 * flip_x, flip_y, ndc, -1/(W/(2 focal)), -1/(H/(2 focal)), ndc near}. */

/* lib/voxurf_fine.py:1062-1068 get_rays_of_a_view (with get_rays :1001-1029 and
 * ndc_rays :1042-1059): rays_o, rays_d, viewdirs [H*W, 3] float32, row-major pixels. */
int vx_camera_rays(const float* cam, float* rays_o, float* rays_d, float* viewdirs, void* stream);

/* lib/voxurf_fine.py:1042-1059 ndc_rays on n rays; c0 = -1/(W/(2 focal)),
 * c1 = -1/(H/(2 focal)). */
int vx_ndc_rays(int64_t n, float c0, float c1, float near_, const float* rays_o,
                const float* rays_d, float* o_out, float* d_out, void* stream);

/* lib/voxurf_fine.py:579-591 Voxurf.hit_coarse_geo: does any in-box sample of the ray
 * (sample_pts_on_rays with far = 1e9) pass the MaskCache?  box = {xyz_min, xyz_max},
 * params = {stepdist, near} (host); mc / mc_geom / mc_params as vx_fused_fine_fwd.
 * Outputs: hit [n] bytes and/or flag [n] int64 (either may be NULL). */
int vx_hit_coarse_geo(const float* rays_o, const float* rays_d, int64_t n_rays, const float* box,
                      const float* params, const float* mc, const int64_t* mc_geom,
                      const float* mc_params, uint8_t* hit, int64_t* flag, void* stream);

/* hit_coarse_geo on the rays of one view (lib/voxurf_fine.py:1145-1149), the rays made
 * in the kernel: flag [H*W] int64. */
int vx_view_hit_coarse_geo(const float* cam, const float* box, const float* params,
                           const float* mc, const int64_t* mc_geom, const float* mc_params,
                           int64_t* flag, void* stream);

/* SDF and unit normal grad / (|grad| + 1e-5) of the 6-neighbour gradient at the tile^3 points
 * -1 + 2 (origin + i) / (res - 1) of a res^3 lattice (lib/dvgo_ori.py:679-693 with
 * lib/voxurf_fine.py:502-534); box = {xyz_min, xyz_max} and origin[3] in host memory; out
 * [tile^3], normal [tile^3, 3], z fastest. */
int vx_sdf_query(const float* sdf, const int64_t* geom, const float* box, float voxel_size,
                 float res, const float* origin, int tile, float* out, float* normal, void* stream);

/* Occupancy of a MaskCache: which bricks and blocks of its grid hold a sample that could pass
 * (vx_maskcache_occupancy_bytes bytes, 8-byte aligned; -1: bad geometry).  The _occ forms of
 * the two entries above take it (or NULL, as the two entries above: a wavefront a ray that
 * looks every sample up) and give the same flags, a thread a ray jumping over what is clear;
 * it must be that of the same mc, mc_geom and mc_params. */
int64_t vx_maskcache_occupancy_bytes(const int64_t* mc_geom);
int vx_maskcache_occupancy(const float* mc, const int64_t* mc_geom, const float* mc_params,
                           void* occ, void* stream);
int vx_hit_coarse_geo_occ(const float* rays_o, const float* rays_d, int64_t n_rays,
                          const float* box, const float* params, const float* mc,
                          const int64_t* mc_geom, const float* mc_params, const void* occ,
                          uint8_t* hit, int64_t* flag, void* stream);
int vx_view_hit_coarse_geo_occ(const float* cam, const float* box, const float* params,
                               const float* mc, const int64_t* mc_geom, const float* mc_params,
                               const void* occ, int64_t* flag, void* stream);

/* lib/voxurf_fine.py:1150-1155 (img[mask], rays_o[mask], ...): incl = inclusive scan of
 * the view's flags; kept pixels are written in pixel order to rows incl[p] - 1 of
 * rgb_out, o_out, d_out, v_out [*, 3] (rgb [H*W, 3] float32). */
int vx_view_compact_rays(const float* cam, const float* rgb, const int64_t* incl, float* rgb_out,
                         float* o_out, float* d_out, float* v_out, void* stream);

/* ---- dense per-step grid operators ---------------------------------------------- */

/* Number of per-block partial sums vx_smooth_grad_tv writes for an X*Y*Z grid. */
int64_t vx_smooth_grad_tv_partials(int64_t X, int64_t Y, int64_t Z);

/* lib/voxurf_fine.py:412-421 density_total_variation(smooth_grad_tv=weight) on the
 * 'interpolate' gradient grid (:440-450) with tv_smooth_conv (:204-240, replicate
 * padding): loss = weight * mean over masked entries of (S(G) - G)^2, S detached.
 * taps[3] (host): the 1-D factors of the 3x3x3 smoothing kernel.  mask [X,Y,Z] bytes or
 * NULL (all voxels); mask_count = number of selected voxels.  Writes dgrad [3,X,Y,Z]
 * (dloss/dG), partials [vx_smooth_grad_tv_partials], loss [1] (if not NULL) and adds
 * dloss/dsdf into sdf_grad [X,Y,Z] (if not NULL). */
int vx_smooth_grad_tv(int dtype, const void* sdf, int X, int Y, int Z, double voxel_size,
                      const double* taps, const uint8_t* mask, int64_t mask_count, double weight,
                      void* dgrad, void* partials, void* loss, void* sdf_grad, void* stream);

/* lib/voxurf_fine.py:246-258 _gaussian_3dconv applied to [C,X,Y,Z] (each channel):
 * conv3d with replicate padding by the separable kernel taps (x) taps (x) taps (k odd,
 * <= 9; host array), or its adjoint (transpose = 1).  tmp: scratch of the input's size. */
int vx_smooth3d(int dtype, const void* in, void* out, void* tmp, int C, int X, int Y, int Z,
                const double* taps, int k, int transpose, void* stream);

/* lib/grid.py:60-65 DenseGrid.scale_volume_grid / lib/voxurf_fine.py:280-283:
 * F.interpolate(..., mode='trilinear', align_corners=True) of [C,X,Y,Z] to [C,X2,Y2,Z2]. */
int vx_resample_trilinear(int dtype, const void* in, int C, int X, int Y, int Z, void* out, int X2,
                          int Y2, int Z2, void* stream);

/* ---- mesh extraction (lib/voxurf_fine.py:894-910, lib/dvgo_ori.py:679-703) --------- */

/* lib/dvgo_ori.py:679-693 extract_fields with Voxurf.grid_sampler as query: u[i,j,k] =
 * scale * trilinear(sdf) at (linspace(bmin, bmax, n)[i], ...) (float32 linspace).  box =
 * {grid xyz_min, xyz_max}, bounds = {bmin, bmax} (host); u [n0, n1, n2] float32. */
int vx_extract_fields(const float* sdf, const int64_t* geom, const float* box, const float* bounds,
                      int n0, int n1, int n2, float scale, float* u, void* stream);

/* Marching-cubes tables (host memory): count [256] triangles per corner configuration
 * (bit c set when corner c = (c&1, c>>1&1, c>>2&1) is below the threshold), edges
 * [256 * 3 * vx_mc_max_tris()] lattice-edge ids of each triangle.  No counterpart in the
 * reference (which calls PyMCubes, lib/dvgo_ori.py:698); generated, not stored. */
int vx_mc_tables(int8_t* count, int8_t* edges);
int vx_mc_max_tris(void);

/* lib/dvgo_ori.py:698 mcubes.marching_cubes(u, iso), pass 1: per lattice point, vcnt =
 * crossing lattice edges it owns (+x, +y, +z), tcnt = triangles of the cube at it
 * (count/edges: device copies of vx_mc_tables). */
int vx_mc_count(const float* u, int nx, int ny, int nz, float iso, const int8_t* count,
                const int8_t* edges, int64_t* vcnt, int64_t* tcnt, void* stream);

/* Pass 2: vincl/tincl = inclusive scans of vcnt/tcnt; verts [V, 3] float64 (index space,
 * or world space v / (n - 1) * (bmax - bmin) + bmin when bounds = {bmin, bmax} host
 * doubles is given, as lib/dvgo_ori.py:699-702), faces [F, 3] int64. */
int vx_mc_emit(const float* u, int nx, int ny, int nz, float iso, const int8_t* count,
               const int8_t* edges, const int64_t* vincl, const int64_t* tincl,
               const double* bounds, double* verts, int64_t* faces, void* stream);

/* Marching cubes of the whole field in two calls: vx_mc_classify fills the workspace `ws`
 * (vx_mc_workspace_bytes, 16-byte aligned; -1: sizes out of range) and totals = {vertices,
 * triangles} (device); vx_mc_write, with those totals, the mesh vx_mc_emit writes (same
 * vertices, triangles and order).  u, iso and ws must be the classify call's. */
int64_t vx_mc_workspace_bytes(int nx, int ny, int nz);
int vx_mc_classify(const float* u, int nx, int ny, int nz, float iso, const int8_t* count,
                   void* ws, int64_t* totals, void* stream);
int vx_mc_write(const float* u, int nx, int ny, int nz, float iso, const int8_t* count,
                const int8_t* edges, void* ws, int64_t n_verts, int64_t n_faces,
                const double* bounds, double* verts, int64_t* faces, void* stream);

/* Zero n elements (a fill kernel, safe inside captured graphs). */
int vx_zero(int dtype, void* p, int64_t n, void* stream);

/* ---- optimisers ---------------------------------------------------------------- */

/* lib/cuda/adam_upd.cpp:36-86 adam_upd / masked_adam_upd / adam_upd_with_perlr
 * (adam_upd_kernel.cu:8-132): masked != 0 skips grad == 0; perlr may be NULL. */
int vx_adam_upd(int dtype, void* param, const void* grad, void* exp_avg, void* exp_avg_sq,
                const void* perlr, int64_t n, int step, float beta1, float beta2, float lr,
                float eps, int masked, void* stream);

/* lib/utils.py:154-199 adam() for one parameter (the optimiser the training step
 * runs): step is the 1-based step count after increment; per_lr may be NULL;
 * clear_grad != 0 zeroes grad after use.  pages (may be NULL; float32 with clear_grad
 * only): one flag per page of grad (vx_adam_page_elems() elements), nonzero where
 * anything was added to that page since the last step; pages flagged zero are all-zero
 * gradient and are neither read nor cleared; the flags are reset to zero. */
int vx_adam_step(int dtype, void* param, void* grad, void* exp_avg, void* exp_avg_sq,
                 const void* per_lr, int64_t n, int step, double lr, double beta1, double beta2,
                 double eps, int clear_grad, uint32_t* pages, void* stream);
/* Elements per gradient page (the page flags of vx_adam_step, vx_adam_step_split and
 * the fused forward; the touched words of vx_adam_step_touched): 64.  No counterpart in
 * the reference, which updates every element. */
int64_t vx_adam_page_elems(void);
/* lib/utils.py:169-199 utils.Adam on one float32 parameter (clear_grad = 1, 16-byte
 * aligned buffers), skipping pages whose update is the identity: touched word zero
 * (moments still zero) and an all-zero gradient this step.  A page with a nonzero
 * gradient is marked touched.  touched: ceil(n / vx_adam_page_elems()) words,
 * zero-initialised with the moments (all ones after loading moments from elsewhere). */
int vx_adam_step_touched(float* param, float* grad, float* exp_avg, float* exp_avg_sq,
                         const float* per_lr, int64_t n, int step, double lr, double beta1,
                         double beta2, double eps, uint32_t* touched, void* stream);
/* vx_adam_step (float32, clear_grad = 1, 16-byte aligned buffers) split in two passes
 * over disjoint element sets, for overlap with other work.  pages holds 2 * P + 1 words
 * (P = ceil(n / vx_adam_page_elems())): the page flags, a count and a page list (count
 * and list zero-initialised once).  Phase 1 updates the pages flagged zero (all-zero gradient, so
 * it may run as soon as the flags are final, before the gradient is) from one block per
 * CU, and lists the flagged pages; phase 2 updates the listed pages, clears their
 * gradient and resets flags and count.  Phase 1 then phase 2 with the same step equal
 * one vx_adam_step.  touched (one word per page, or NULL): nonzero for every page whose
 * moments may be nonzero; phase 1 skips pages with a zero flag and a zero touched word
 * (their p, m and v are left exactly as utils.Adam leaves them: m = v = g = 0 makes the
 * update an identity) and phase 2 marks the pages it updates.  Zero-initialise it with
 * the moments; set it to all ones after loading moments from elsewhere. */
int vx_adam_step_split(int phase, float* param, float* grad, float* exp_avg, float* exp_avg_sq,
                       const float* per_lr, int64_t n, int step, double lr, double beta1,
                       double beta2, double eps, uint32_t* pages, uint32_t* touched, void* stream);

/* ---- per-sample ops ------------------------------------------------------------ */

/* lib/voxurf_fine.py:463-500 neus_alpha_from_sdf_scatter (use_mid=True): alpha [n]. */
int vx_neus_alpha_fwd(int dtype, const void* viewdirs, const int64_t* ray_id, const void* sdf,
                      const void* gradient, int64_t n, double dist, double inv_s, void* alpha,
                      void* stream);
/* Its adjoint: gsdf [n], ggradient [n,3]. */
int vx_neus_alpha_bwd(int dtype, const void* viewdirs, const int64_t* ray_id, const void* sdf,
                      const void* gradient, int64_t n, double dist, double inv_s,
                      const void* galpha, void* gsdf, void* ggradient, void* stream);

/* Row selection by a boolean mask [n] (one byte each; 1 <= n < 2^31): offsets
 * [vx_select_blocks(n)] and total [1] (device) of the selected elements, then up to eight
 * arrays (host arrays of device addresses, words: 32-bit words a row) copied under them:
 * dst [total] = src[mask]; transpose = 1: dst [n] = src at the selected rows, zero elsewhere. */
int64_t vx_select_blocks(int64_t n);
int vx_select_count(const uint8_t* mask, int64_t n, int* offsets, int64_t* total, void* stream);
int vx_select_rows(const uint8_t* mask, int64_t n, const int* offsets, int count,
                   const int64_t* src, const int64_t* dst, const int* words, int transpose,
                   void* stream);
/* torch_scatter.segment_coo(src, index, out, reduce='sum') as called at
 * lib/voxurf_fine.py:753-777: out [n_out, C] += segment sums of src [n, C] over the
 * sorted index [n]. */
int vx_segment_sum(int dtype, const void* src, const int64_t* index, int64_t n, int C,
                   int64_t n_out, void* out, void* stream);
/* Its adjoint: gsrc [n, C] = gout[index]. */
int vx_segment_gather(int dtype, const void* gout, const int64_t* index, int64_t n, int C,
                      int64_t n_out, void* gsrc, void* stream);

/* ---- fused fine step (per-ray kernels) ------------------------------------------ */
/* These fuse the per-sample stages of lib/voxurf_fine.py:620-802 (sample_ray,
 * grid_sampler with sample_grad, neus_alpha_from_sdf_scatter, the two fast_color_thres
 * compactions and Alphas2Weights) into one pass per ray, and their adjoints
 * (Alphas2Weights.backward -> render_utils_kernel.cu:654-677, the NeuS and grid_sample
 * adjoints that autograd runs) into a per-ray backward over the stored walk range.
 * Host-side arrays: sdf_geom/k0_geom as for the grid ops; box[6] = {xyz_min, xyz_max};
 * params[6] = {stepdist, voxel_size, inv_s, fast_color_thres, near, far}.
 * Per-ray slots hold `cap` walk-range samples (alpha > thres, up to the terminating
 * one) of two float4 each: s4 = (x, y, z, transmittance before the sample),
 * g4 = (SDF gradient xyz, SDF value); stats[3 r + 1] is the number of slots used.
 * mc (may be NULL): the MaskCache density grid (device, one channel, geometry mc_geom)
 * with mc_params[10] = {act_shift, voxel_size_ratio, thres, nearest, xyz_min[3],
 * xyz_max[3]}; samples it rejects are dropped like out-of-box ones
 * (lib/voxurf_fine.py:631-636).  k0_pages (may be NULL, then k0_geom may be too): set the
 * page flag (vx_adam_step) of every k0_grad page the feature scatter of the survivors
 * can write, as soon as they are known.  sdf_pages (may be NULL): the same for every
 * SDF-gradient page the stencil scatter of vx_fused_fine_bwd can write (walk-range
 * samples), and with hier_reach > 0 every page within hier_reach voxels of a survivor's
 * cell (the sample_sdfs stencils of vx_voxurf_feat_bwd; 0 for the plain fine step).
 * walk_total (may be NULL): a device word the walk adds every ray's number of used slots
 * to (the caller clears it), to size the backward's workspace.
 * skip_bounds (may be NULL): vx_sdf_skip_bounds of this SDF grid, current for its
 * values; samples these bounds prove to have alpha <= thres skip their lookups (every
 * output is the same with and without them). */
int vx_fused_fine_fwd(const float* sdf, const int64_t* sdf_geom, const float* box,
                      const float* params, const float* mc, const int64_t* mc_geom,
                      const float* mc_params, const float* rays_o, const float* rays_d,
                      const float* viewdirs, int64_t n_rays, int cap, void* s4, void* g4,
                      int64_t* cnt, float* last, int* stats, int count_all, int* overflow,
                      int64_t* walk_total, const int64_t* k0_geom, uint32_t* k0_pages,
                      uint32_t* sdf_pages, int hier_reach, const void* skip_bounds,
                      void* stream);
/* Empty-space bounds of an SDF grid (no counterpart in the reference, which evaluates
 * every in-box sample): per brick of 8^3 cells, float4 (lower bound of the SDF, upper
 * bound of the length of its 6-neighbour central-difference gradient, 0, 0) over every
 * voxel the 7-point lookup of a sample in the brick reads.  bounds and ws: device
 * arrays of vx_sdf_skip_bricks(sdf_geom) float4 each.  margin >= 0: the bounds also hold
 * for any grid within margin of this one voxel by voxel (e.g. after an optimiser step
 * whose update is bounded by margin); 0 for this grid only.  Recompute them after every
 * change of the grid beyond that. */
int64_t vx_sdf_skip_bricks(const int64_t* sdf_geom);
int vx_sdf_skip_bounds(const float* sdf, const int64_t* sdf_geom, float voxel_size,
                       float margin, void* bounds, void* ws, void* stream);
/* Keeps the survivors (weight > thres) of each ray's slots at rows
 * off_incl[r]-cnt[r] .. off_incl[r]-1 and builds the rgbnet input rows
 * X [M, xstride] = [k0 | normal | view PE | 0] (lib/voxurf_fine.py:678-716; xstride a
 * multiple of 4, at most 64); P4 [M] = (x, y, z, weight), G4 [M] = (gradient, sdf),
 * rid [M] int32 ray ids; rows at or past max_rows (the buffers' capacity) are not
 * written, so the call may be issued before M is known on the host and repeated with
 * larger buffers when M exceeds the capacity.  k0_pages (may be NULL): set the page flag
 * (vx_adam_step) of every k0_grad page the feature scatter of these rows can write, so
 * that the k0 Adam pass over the other pages can start before the backward. */
int vx_fused_fine_gather(const float* k0, const int64_t* k0_geom, const int64_t* sdf_geom,
                         const float* box, const float* params, const float* viewdirs,
                         int64_t n_rays, int cap, int n_freq, const void* s4, const void* g4,
                         const int* stats, const int64_t* cnt, const int64_t* off_incl,
                         int xstride, int64_t max_rows, float* X, void* P4, void* G4, int* rid,
                         uint32_t* k0_pages, void* stream);
/* segment_coo compositing (lib/voxurf_fine.py:753-763), MSE loss per ray (run.py:604)
 * and the colour-side adjoints: dlogit [M,3], gw [M] (d loss / d weight), glast [N],
 * S [N] (sum of gw*w per ray), loss_r [N] (sum of squared errors).  With target NULL
 * only rgb [N,3] is written (rendering; the adjoint pointers may be NULL).  Rays whose
 * rows reach past max_rows (the row buffers' capacity) are left out. */
int vx_fused_fine_composite(int64_t n_rays, const int64_t* cnt, const int64_t* off_incl,
                            const float* logits, int lstride, const void* P4, const float* last,
                            const float* target, float bg, float* rgb, float* dlogit, float* gw,
                            float* glast, float* S, float* loss_r, int64_t max_rows,
                            void* stream);
/* Adjoint of the feature rows: k0_grad += trilinear scatter of dX[:, :C]; dgf [M,3] =
 * d loss / d gradient through the normalised normal dX[:, C:C+3].  k0_pages (may be
 * NULL): the page flags of k0_grad for vx_adam_step, set for every page written.  m_dev
 * (may be NULL): device row count, min(*m_dev, m) rows are processed. */
int vx_fused_fine_feat_bwd(const int64_t* k0_geom, const int64_t* sdf_geom, const float* box,
                           const float* params, int64_t m, const float* dX, int dxs,
                           const void* P4, const void* G4, float* k0_grad, float* dgf,
                           uint32_t* k0_pages, const int64_t* m_dev, void* stream);
/* Backward of the SDF side over each ray's stored walk range: sdf_grad += adjoint of
 * (7-point SDF lookup -> NeuS alpha -> transmittance walk), with dgf [M,3] added to the
 * survivors' gradient adjoint and dsf [M] (may be NULL) to their centre-SDF adjoint.
 * The stencil scatter is binned by 16^3-voxel brick and staged in LDS; g4 is
 * overwritten with each walk-range sample's stencil adjoints (gd_z, gd_y, gd_x, gsdf)
 * and s4's w (the transmittance) with the sample's bricks.  ws: device scratch of
 * vx_fused_bwd_workspace_bytes() bytes.  Rays whose rows reach past max_rows are left
 * out, as in the composite. */
int vx_fused_fine_bwd(const float* sdf, const int64_t* sdf_geom, const float* box,
                      const float* params, const float* viewdirs, int64_t n_rays, int cap,
                      void* s4, void* g4, const int* stats, const int64_t* cnt,
                      const int64_t* off_incl, const float* last, const float* gw,
                      const float* glast, const float* S, const float* dgf, const float* dsf,
                      float* sdf_grad, int64_t max_rows, void* ws, int64_t ws_bytes,
                      void* stream);
/* The two phases of vx_fused_fine_bwd (its steps in order, for callers that run the
 * first beside the rgbnet backward): _alpha needs only the compositing's adjoints (gw,
 * glast, S) and bins the walk-range samples by brick (g4 then holds each sample's alpha
 * adjoints, s4's w its bricks and a survivor bit); _grid adds dgf / dsf and scatters into
 * sdf_grad.  Both take the same n_rays, cap, max_rows and workspace. */
int vx_fused_fine_bwd_alpha(const float* sdf, const int64_t* sdf_geom, const float* box,
                            const float* params, const float* viewdirs, int64_t n_rays, int cap,
                            void* s4, void* g4, const int* stats, const int64_t* cnt,
                            const int64_t* off_incl, const float* last, const float* gw,
                            const float* glast, const float* S, int64_t max_rows, void* ws,
                            int64_t ws_bytes, void* stream);
int vx_fused_fine_bwd_grid(const float* sdf, const int64_t* sdf_geom, const float* box,
                           const float* params, int64_t n_rays, int cap, const void* s4, void* g4,
                           const int* stats, const int64_t* cnt, const int64_t* off_incl,
                           const float* dgf, const float* dsf, float* sdf_grad, int64_t max_rows,
                           void* ws, int64_t ws_bytes, void* stream);
/* Scratch bytes of vx_fused_fine_bwd on an X x Y x Z SDF grid for a walk whose rays hold
 * walk_total walk-range samples in all (the sum of stats[3 r + 1], which
 * vx_fused_fine_fwd also adds into its walk_total word).  With a smaller workspace the
 * samples of the bricks whose slot lists do not fit are left out of the gradient (nothing
 * is written outside the workspace); word 1 of the workspace holds the number of list
 * entries the walk needed. */
int64_t vx_fused_bwd_workspace_bytes(int64_t walk_total, int X, int Y, int Z);
/* ---- rgbnet on the matrix cores ---------------------------------------------------
 * The colour MLP of lib/voxurf_fine.py:132-149 (nn.Linear/ReLU layers of width 192,
 * which the reference runs as cuBLAS GEMMs plus elementwise kernels).  prec selects
 * the arithmetic:
 *   0: FP32 MFMAs, float32 activations;
 *   1: BF16 MFMAs with FP32 accumulation, bfloat16 activations;
 *   2: FP32 accuracy from BF16 MFMAs: both operands of every product are split into three
 *      bfloat16 parts (x = x0 + x1 + x2 exactly) and the six part products with
 *      i + j <= 2 accumulate in FP32, within 2^-23 relative of the exact product;
 *      float32 activations (the weight-gradient GEMMs run as with prec 0).
 * Weights are packed per call into the MFMA operand order; activation rows are
 * [M, 192] (element type per prec), inputs [M, 32*kt] zero padded.  M_dev (may be NULL):
 * a device int64 row count; when given the calls process min(*M_dev, M) rows, M being
 * the buffers' capacity, so they can be queued before the count is known on the host. */

/* Pack W [n_out, k_in] (row-major, float32) as the A operand of a layer with kt input
 * tiles of 32 (reduction) and nto output tiles; transpose = 1 packs W^T (backward). */
int vx_mlp_pack(int prec, const float* W, int n_out, int k_in, int kt, int nto, int transpose,
                void* out, void* stream);
/* Element count of a packed operand (float32 for prec 0, bfloat16 for prec 1; prec 2
 * packs three times as many bfloat16 elements). */
int64_t vx_mlp_pack_elems(int kt, int nto);
/* All packed operands of an rgbnet in one launch: w_ptrs is a host array of the
 * n_hidden hidden layers' device weight pointers (layer 0 [192, k_in0], the others
 * [192, 192]).  For each layer li in order, the forward operand (kt = 2 or 3 for layer
 * 0 -- k_in0 <= 64 or <= 96 -- else 6; nto = 6) then the transposed backward operand
 * (kt = 6, nto = the forward kt), concatenated. */
int64_t vx_mlp_pack_net_elems(int n_hidden, int k_in0);
int vx_mlp_pack_net(int prec, int n_hidden, const int64_t* w_ptrs, int k_in0, void* out,
                    void* stream);
/* One hidden layer: out = relu(W in + b); with last = 1 also logits [M,3] = W3 out + b3.
 * mask_bits (prec 2 only, may be NULL): also writes the ReLU mask as bits, six uint32
 * words per row (bit k of word w: out column 32 w + k positive), for vx_mlp_layer_bwd.
 * k_in: the layer's real input width (0: all 32 kt; the packed weights are zero past
 * it): with prec 2 and k_in <= 32 kt - 16 the last 16 input columns, whose products are
 * zero, are not multiplied. */
int vx_mlp_layer_fwd(int prec, int kt, int k_in, int last, const void* in, int in_stride,
                     int64_t M, const void* wpk, const float* bias, void* out, int out_stride,
                     const float* w3, const float* b3, float* logits, const int64_t* M_dev,
                     uint32_t* mask_bits, void* stream);
/* The whole network in one launch without keeping activations: the logits [M, 3] that
 * vx_mlp_layer_fwd and vx_mlp_logits give with prec 2, bit for bit, for X [M, xs] (float32 rows
 * padded to 64 columns for k_in0 <= 64, else 96; finite past k_in0), 1..4 hidden layers of
 * width 192 and input width k_in0 <= 96; packed: vx_mlp_pack_net's output for prec 2; biases:
 * host array of n_hidden device addresses. */
int vx_mlp_net_fwd(int n_hidden, int k_in0, const float* X, int xs, int64_t M, const void* packed,
                   const int64_t* biases, const float* w3, const float* b3, float* logits,
                   const int64_t* M_dev, void* stream);
/* The 3-output layer alone: logits [M, 3] = W3 H + b3 from the last hidden activations
 * H [M, hs] (the last = 1 part of vx_mlp_layer_fwd). */
int vx_mlp_logits(int prec, const void* H, int hs, int64_t M, const float* w3, const float* b3,
                  float* logits, const int64_t* M_dev, void* stream);
/* Data gradient through a layer: dx = (W^T dy) * [mask > 0] (mask NULL: no ReLU).
 * mask_bits (prec 2, nto 6, may be NULL): the mask as written by vx_mlp_layer_fwd, read
 * instead of the float rows (mask must still be given).  nto = 1 (prec 2, no mask):
 * only dx's first 32 columns, from an operand packed for nto = 2 (for callers that need
 * the gradient of the first input columns only). */
int vx_mlp_layer_bwd(int prec, int nto, const float* dy, int dy_stride, int64_t M,
                     const void* wpk_t, const void* mask, int mask_stride, float* dx,
                     int dx_stride, const int64_t* M_dev, const uint32_t* mask_bits,
                     void* stream);
/* Floats the `part` / `partb` workspaces of vx_mlp_wgrad and vx_mlp_last_bwd need for
 * M rows (row-block partial sums plus the reduction's group sums). */
int64_t vx_mlp_wgrad_part_elems(int64_t M);
int64_t vx_mlp_wgrad_partb_elems(int64_t M);
/* dW [192, k_real] = dY^T X, db [192] = column sums of dY (split over row blocks, then
 * a deterministic two-pass reduction).  max_blocks: 0 for one row block per CU (the
 * fastest alone), or fewer, to leave CUs to kernels running beside it on other
 * streams (the result does not depend on it beyond FP32 summation order). */
int vx_mlp_wgrad(int prec, int kt, int k_real, const float* dY, int dys, const void* X, int xs,
                 int64_t M, float* part, float* partb, float* dW, float* db, const int64_t* M_dev,
                 int max_blocks, void* stream);
/* The two halves of vx_mlp_wgrad (no counterpart in the reference; for callers that time
 * or schedule the row-block pass apart from the reduction): the row-block partial sums
 * into part / partb, then their reduction into dW / db.  Both calls take the same M, kt
 * and max_blocks (they fix the number of row blocks); the reduction also writes its
 * group sums into the workspaces' tails.  stamps (prec 2 only; may be NULL): two device
 * words that receive the pass's duration on the device wall clock, stamps[0] = min
 * (first workgroup start), stamps[1] = max (last workgroup end); the caller sets them to
 * UINT64_MAX / INT64_MAX and 0 beforehand. */
int vx_mlp_wgrad_partials(int prec, int kt, const float* dY, int dys, const void* X, int xs,
                          int64_t M, float* part, float* partb, const int64_t* M_dev,
                          int max_blocks, uint64_t* stamps, void* stream);
/* Rate of the device wall clock that the stamps above count, in kHz (-1 on error). */
int64_t vx_wall_clock_khz(void);
int vx_mlp_wgrad_reduce(int kt, int k_real, int64_t M, float* part, float* partb,
                        float* dW, float* db, int max_blocks, void* stream);
/* Backward through the 3-output layer in one pass over H: dH = (dlogit W3) * [H > 0],
 * dW3 [3, 192] = dlogit^T H, db3 [3] = column sums of dlogit. */
int vx_mlp_last_bwd(int prec, const float* dlogit, const void* H, int hs, int64_t M,
                    const float* w3, float* dH, int dhs, float* part, float* partb, float* dW3,
                    float* db3, const int64_t* M_dev, void* stream);
/* The two halves of vx_mlp_last_bwd, for callers that run them on different streams:
 * the data gradient dH = (dlogit W3) * mask from the last hidden layer's mask bits as
 * written by vx_mlp_layer_fwd (prec 2; H itself is not read), and dW3, db3 (the pass
 * over H). */
int vx_mlp_last_dgrad(const float* dlogit, const uint32_t* mask_bits, int64_t M, const float* w3,
                      float* dH, int dhs, const int64_t* M_dev, void* stream);
int vx_mlp_last_wgrad(int prec, const float* dlogit, const void* H, int hs, int64_t M,
                      float* part, float* partb, float* dW3, float* db3, const int64_t* M_dev,
                      void* stream);
/* y = bfloat16(x), n elements. */
int vx_f32_to_bf16(const float* x, int64_t n, void* y, void* stream);

/* *out = scale * (sum of x[0..n)) (float32, device scalar; fixed summation order). */
int vx_sum_f32(const float* x, int64_t n, float scale, float* out, void* stream);

/* ---- the reference fine model's colour side, fused -----------------------------------
 * lib/voxurf_fine.py:678-763 with configs/dtu_e2e/fine.py (rgbnet + the residual
 * k_rgbnet), on the survivors of vx_fused_fine_fwd.  row_cfg = {pos_pe, view_pe,
 * k_view_pe, nd, xstride, kstride} (host array), disp [nd] (host array): the grad_feat
 * displacements.  Row layouts:
 *   X  [M, xstride]: xyz PE (3 + 6 pos_pe) | view PE (3 + 6 view_pe) | sdf | sample_sdfs
 *                    feat (6 nd, [offset][displacement]) | normalised grad (3 nd) | 0
 *   XK [M, kstride]: k0 (C) | xyz PE | k view PE (3 + 6 k_view_pe) | gradient (3, xyz,
 *                    raw) | rgb logit (3, written by vx_voxurf_logit_cols) | 0 */

/* Survivor rows (lib/voxurf_fine.py:678-740): P4/G4/rid as vx_fused_fine_gather, X and
 * XK (k_rgbnet's logit columns are left 0). */
int vx_voxurf_gather(const float* sdf, const int64_t* sdf_geom, const float* k0,
                     const int64_t* k0_geom, const float* box, const float* params,
                     const int* row_cfg, const float* disp, const float* viewdirs,
                     int64_t n_rays, int cap, const void* s4, const void* g4, const int* stats,
                     const int64_t* cnt, const int64_t* off_incl, int64_t max_rows, float* X,
                     float* XK, void* P4, void* G4, int* rid, void* stream);
/* XK[:, col .. col+3) = logits [m, 3] (the rgb_logit.detach() input of k_rgbnet,
 * lib/voxurf_fine.py:736-739); m_dev (may be NULL): device row count. */
int vx_voxurf_logit_cols(int64_t m, const int64_t* m_dev, const float* logits, float* XK,
                         int kstride, int col, void* stream);
/* Compositing and loss of the fine model (lib/voxurf_fine.py:741-763, run.py:604-633):
 * rgb [N,3] = clamp(seg(w sigmoid(logits + k_logits)) + last bg, 0, 1), rgb0 [N,3] =
 * seg(w sigmoid(logits)) + last bg; with target given: loss_r [N] (w_main |rgb - t|^2 +
 * w_rgb0 |rgb0 - t|^2, plus the last ray's entropy term, all to be scaled by 1/(3N)),
 * dlogit0 / dlogitk [M,3] (the two MLPs' output gradients), gw [M], glast [N], S [N] as
 * vx_fused_fine_composite. */
int vx_voxurf_composite(int64_t n_rays, const int64_t* cnt, const int64_t* off_incl,
                        const float* logits, const float* k_logits, const void* P4,
                        const float* last, const float* target, float bg, float w_main,
                        float w_rgb0, float w_ent, float* rgb, float* rgb0, float* dlogit0,
                        float* dlogitk, float* gw, float* glast, float* S, float* loss_r,
                        int64_t max_rows, void* stream);
/* Adjoint of the rows: k0_grad += trilinear scatter of dXK[:, :C]; sdf_grad += the
 * adjoint of sample_sdfs (lib/voxurf_fine.py:537-577) from dX's feat and grad columns;
 * dgf [M,3] = dXK's gradient columns and dsf [M] = dX's sdf column (added at the
 * survivor's sample by vx_fused_fine_bwd).  m_dev as above. */
int vx_voxurf_feat_bwd(const float* sdf, const int64_t* sdf_geom, const int64_t* k0_geom,
                       const float* box, const float* params, const int* row_cfg,
                       const float* disp, int64_t m, const int64_t* m_dev, const float* dX,
                       const float* dXK, const void* P4, float* k0_grad, float* sdf_grad,
                       float* dgf, float* dsf, void* stream);

/* lib/voxurf_fine.py:765-777 (render_grad / render_depth, run.py:1052-1054) on the
 * survivor rows of either fine model: normal [N,3] = seg(w g / (|g| + 1e-6)) of the raw
 * SDF gradient, depth [N] = seg(w step_id dist); either output may be NULL.  box and
 * params as vx_fused_fine_fwd's; rays_o / rays_d are the rays of the forward (the step
 * ids are recovered from the rows' points). */
int vx_fused_render_extras(const float* box, const float* params, int64_t n_rays,
                           const int64_t* cnt, const int64_t* off_incl, const void* P4,
                           const void* G4, const float* rays_o, const float* rays_d,
                           float* normal, float* depth, int64_t max_rows, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* VOXHIP_H */
