// Internal declarations shared by the HIP sources of libkevernals_amd.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <functional>
#include <string>
#include <vector>

#include "kevernals_amd.h"

// Geometry as the kernels see it: passed by value as a kernel argument.
// Per-view arrays live in device memory (det/src: np*3 floats each).
struct KvGeom {
    int nx, ny, nz;
    int nu, nv, np;
    float sx, sy, sz;
    float pu, pv;
    const float *det;
    const float *src;
    // Ray constants in FP32, evaluated by kv_set_geometry as the forward
    // kernels would: rc[KV_RC*p + 0..6] = source x, y, z over the spacing,
    // dz (detector z / sz - source z / sz), the z-face alphas
    // (-nz/2 - sz_p) / dz and (nz/2 - sz_p) / dz and 1 / dz (the last three
    // 0 when |dz| <= 1e-6); for the backprojectors rc[KV_RC*p + 8, 9] =
    // detector corner x over sx and the far detector edge
    // (det x + nu * pu) / sx (Projector.cu:473-492); rc[KV_RC*p + 10] = the
    // rounding of x plane positions relative to the source in the mode-R
    // walk, in voxels (0 when source and half size are exact), [11] and [12] =
    // the interval of detector columns whose rays cross no x face inside the
    // z slab (ints); then per view and
    // detector column, at rc + KV_RC*np, four floats: the pixel-centre
    // coordinate qx = (det x + (u + 0.5) pu) / sx, the x-face alphas
    // (-nx/2 - sx_p) / dx and (nx/2 - sx_p) / dx (0 unless |dx| > 1e-6,
    // dx = qx - sx_p) and 1 / dx (0 when dx = 0); then the same per view
    // and detector row for y.
    const float *rc;
    // Mode-A forward walk of a detector row: the (y, z) segments its rays
    // share (KvSeg lists of seg_stride entries per view and row, built on the
    // first forward pass), and per list its alpha range and count.  Null before
    // that, when the lists would exceed KV_SEG_MAX_BYTES, and when memory is
    // short: the rays are then walked voxel by voxel.
    const struct KvSeg *seg_a;
    const struct KvSegHead *seg_a_head;
    int seg_stride;
    // The same for the mode-R walk (kv_fp.hip, "mode R, row by row"): null
    // also where too few rays could take it (row_r_ok).  seg_delta is the
    // largest alpha distance from a segment's ends within which a lane may
    // have to look up an x crossing's voxels one by one.
    const struct KvSegR *seg_r;
    const struct KvSegHeadR *seg_r_head;
    float seg_delta;
    // widest over the views: the interval of columns that run row by row
    // (rc[KV_RC*p + 11, 12]), and the other columns together
    int row_cols, edge_cols;
    int walk_fast;  // forward walk may use end thresholds and 24-bit indices (see kv_fp.hip)
    float bp_shift; // largest shift of a voxel edge's shadow over one slice, in detector columns (0: unbounded)
    int bp_beside;  // many backprojection bricks lie beside views' detector rows (see kv_bp.hip)
    int bp_posz;    // every view's z planes at alpha >= 1e-6: clamped backprojection weights (see kv_bp.hip)
};

constexpr int KV_RC = 16;

// One segment of a detector row's rays between two (y, z) plane crossings:
// it ends at alpha b and lies in the volume row that starts `row` bytes into
// the volume.  A list ends in KV_SEG_PAD empty segments, which a walk may
// read past its last one.
struct KvSeg {
    float b;
    unsigned row;
};
struct KvSegHead {
    float a, end;   // first segment's start and last one's end
    float longest;  // longest segment
    int segs;
};
// Mode R: besides b and row (bit 0: look the segment's voxels up one by one),
// an x crossing c splits the segment into two that both lie in that volume
// row if |c - m| <= r.
struct KvSegR {
    float b;
    unsigned row;
    float m, r;
};
struct KvSegHeadR {
    float a, end;      // first and last (y, z) crossing of the list
    float amin, amax;  // the row's alpha range, x faces left out
    float longest;
    int segs;          // -1: walk the row's rays one by one
    int filler;        // the list ends in entries of 1.0
    int empty;         // no ray of the row meets the volume
};
constexpr int KV_SEG_PAD = 16;
// The lists of one mode take at most KV_SEG_MAX_BYTES, and only where they
// leave KV_SEG_SPARE_BYTES free.
constexpr size_t KV_SEG_MAX_BYTES = size_t(1) << 30;
constexpr size_t KV_SEG_SPARE_BYTES = size_t(1) << 30;

// Unsigned division by a divisor fixed for a launch: n / d =
// (umulhi(n, m) + n) >> l for every n < 2^31, with l = ceil(log2 d) and
// m = floor(2^32 (2^l - d) / d) + 1 (the round-up method of Granlund and
// Montgomery, "Division by invariant integers using multiplication", 1994;
// the 33-bit sum cannot overflow for n < 2^31).
struct KvUDiv {
    unsigned m, l;
};
inline KvUDiv kv_udiv(unsigned d)
{
    if (d < 1)
        d = 1;  // no divisor of a valid launch is 0; keep the host arithmetic defined
    unsigned l = 0;
    while (l < 31 && (1ull << l) < d)
        ++l;
    const unsigned long long m = ((1ull << 32) * ((1ull << l) - d)) / d + 1;
    return KvUDiv{(unsigned)m, l};
}

// Mapping of a one-dimensional forward launch onto tiles (kv_fp.hip
// fp_xcd_tile): tile layout, stripe width in tiles, stripes per tile row and
// tile rows per view with their divisors, first view of the launch; ntx, if
// not 0: a view is one row, of the detector's rows of ntx tiles.
struct KvFpMap {
    int layout, chunk, nch, gy, p0, ntx;
    KvUDiv dchunk, dnch, dgy, dntx;
};

// Per-view plane-crossing tables.  For mode R an entry is the reference's
// alpha1/alpha2 of Projector.cu:653-669 for plane k of a pixel's ray:
//   x[p][k][u] = (|rx| > 1e-24) ? ((k - nx/2) - sx) / rx : 0
// For mode A it is the mode-A plane crossing ((k - n/2) - s) * (1/d), with
// +-INF encoding of rays parallel to the planes, plus the squared mm
// components of each ray (lx2[p][u], ly2[p][v], lz2[p]).
struct KvTables {
    float *x = nullptr;   // [np][nx+1][nu]
    float *y = nullptr;   // [np][ny+1][nv], then 16 bytes of padding (read, never used)
    float *z = nullptr;   // [np][nz+1]
    float *lx2 = nullptr; // mode A: [np][nu]
    float *ly2 = nullptr; // mode A: [np][nv]
    float *lz2 = nullptr; // mode A: [np]
    // Per view and z-plane l = 0..nz, KV_ZS floats (both modes):
    //  [0] T  = (qz - sz) / ((l - nz/2) - sz), the lateral scale of plane l's
    //          shadow on the detector (Projector.cu:473-480 form)
    //  [1] AZ = the same ratio at the slice centre l + 0.5 (0 if singular)
    //  [2] Kx1, [3] Kx0: detector column (pixel-centre units) of lateral x
    //          coordinate c on plane l, u ~= Kx0 + c * Kx1 (bounds only)
    //  [4] Ky1, [5] Ky0: the same for detector rows
    float *zs = nullptr;
    // Per view, y row j and z slice l (index (p * ny + j) * nz + l: the
    // slices of one row are adjacent, as a brick reads them), KV_YZ
    // words, the backprojectors' terms shared by the voxels of one (y, z)
    // row: [0] first and [1] last detector row of the voxel box's shadow
    // (intersected with the +-5 window around the voxel centre's row in mode
    // R; empty, first > last, when mode R's centre row lies off the widened
    // detector), [2] 1 if the shadow is defined (both planes in front of the
    // source), as ints; [4], [5] = entries 2 and 3 of the zs table's plane
    // l + 1, [3] = entry 3 plus 1 less the shadow's padding (the floor of
    // column + 1 - padding is the shadow's first column); [6] lz = max(0, min
    // z-plane alpha) and [7] uz = min(1, max z-plane alpha); [8 + 2 r], [9 + 2 r]
    // the alpha interval in which the rays of detector row [0] + r are inside
    // the voxel row's y and z planes (empty: both ends equal), for the
    // KV_YZ_ROWS first rows.  One entry more may be read past the end.
    float *yz = nullptr;
};
constexpr int KV_BP_TY = 4;  // voxel rows of a backprojection brick
constexpr int KV_ZS = 8;
constexpr int KV_YZ = 16;
constexpr int KV_YZ_ROWS = 4;

// Epilogues of the projection kernels: plain result, fused MLEM ratio/update,
// fused SART residual/update, or the count of accepted (ray, voxel) pairs.
enum KvEpilogue { KV_EP_PLAIN = 0, KV_EP_MLEM = 1, KV_EP_SART = 2, KV_EP_COUNT = 3 };

// What a batch descriptor's forward tiles are: the whole detector in tiles of
// fp_layout, the columns (or the whole detector, mode A) that run row by row,
// or mode R's other columns.  A mode-R reconstruction with segment lists has
// two descriptors, the second without bricks.
enum KvFpPart { KV_FP_WHOLE = 0, KV_FP_ROWS = 1, KV_FP_EDGES = 2 };

// One reconstruction of a batch, as the batch kernels read it (device
// memory, wave-uniform loads).  Work items are numbered consecutively over
// the batch.  Forward tiles sit in KV_XCDS lists, one per XCD (stripes of
// fp_chunk tile columns, stripe i in list i % KV_XCDS, as fp_xcd_tile): this
// reconstruction holds items [fp_first, fp_first + views*fp_nch*fp_chunk)
// of every list, each view being padded to whole rounds of stripes.
// Backprojection bricks: [bp_first, bp_first + bp_bx*bp_by*bp_bz).
struct KvProblem {
    KvGeom g;
    KvTables t;
    float *vol;
    const float *data;
    float *ratio;
    const float *sens;         // mode A: sensitivity A^T 1
    int iters;                 // MLEM iterations for this reconstruction
    int fp_layout;             // forward tile layout: 1, 2, 4 or 8 rows per wavefront
    int fp_part;               // KvFpPart
    int owner;                 // index of the reconstruction (its own, or its first descriptor's)
    int fp_tx, fp_ty;          // forward tiles per view (fp_tx padded to whole rounds of stripes where it has one)
    int fp_chunk;              // tiles per XCD stripe
    int fp_nch;                // stripes per view in one list
    KvUDiv fp_dchunk, fp_dnch, fp_dtx;  // divisors fp_chunk, fp_nch, fp_tx
    long long fp_first;
    int bp_zt;                 // backprojection brick depth: 4 or 8 slices
    int bp_bx, bp_by, bp_bz;   // bricks per axis
    long long bp_first;
};

struct kv_context {
    int device = 0;
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    bool has_geom = false;
    KvGeom g{};
    float *d_det = nullptr;
    float *d_src = nullptr;
    float *d_rc = nullptr;     // KvGeom::rc
    KvSeg *d_seg_a = nullptr;  // KvGeom::seg_a
    KvSegHead *d_seg_a_head = nullptr;
    KvSegR *d_seg_r = nullptr;  // KvGeom::seg_r
    KvSegHeadR *d_seg_r_head = nullptr;
    bool lists_ok[2] = {false, false};  // mode's lists not built yet, and worth it for the geometry
    bool lists_held = false;            // their addresses are kept elsewhere (a batch, a captured graph)
    KvTables tab_r{};
    bool tab_r_ok = false;
    KvTables tab_a{};
    bool tab_a_ok = false;
    float *d_ratio = nullptr;  // projection-sized work buffer of fused iterations
    float *d_sens = nullptr;   // mode-A sensitivity A^T 1
    bool sens_ok = false;
    double *d_red = nullptr;   // partial sums of deterministic reductions
    size_t red_cap = 0;        // doubles in d_red
    float *d_ll = nullptr;     // projections of the further volumes of kv_log_likelihoods
    float *d_pack = nullptr;   // kv_log_likelihoods' volumes interleaved per voxel (4 floats per voxel)
};

// Reconstruction count and operator mode of a batch (0 / -1 for null).
int kv_internal_batch_size(const kv_batch *b);
int kv_internal_batch_mode(const kv_batch *b);

// Thread-local error message.
void kv_set_error(const char *fmt, ...);

// Builds the crossing tables of `mode` for the context's geometry (once).
kv_status kv_internal_ensure_tables(kv_context *ctx, int mode);
// Computes the mode-A sensitivity A^T 1 (once).
kv_status kv_internal_ensure_sens(kv_context *ctx);
// Device memory that a call cannot do without (hipMalloc): the context's
// segment lists make room for it, unless they are held.
kv_status kv_internal_alloc(kv_context *ctx, void **p, size_t bytes);
// Builds a mode's segment lists where the geometry has them, for a caller
// that copies KvGeom: the context keeps them as long as its geometry.
kv_status kv_internal_hold_lists(kv_context *ctx, int mode);
// Frees the segment lists; the geometry's later passes go without.  Not for
// a context whose lists are held.
kv_status kv_internal_drop_lists(kv_context *ctx);
// The same for every reconstruction of a batch.
kv_status kv_internal_batch_drop_lists(kv_batch *b);

#define KV_TRY_HIP(expr)                                                                        \
    do {                                                                                        \
        hipError_t kv_e_ = (expr);                                                              \
        if (kv_e_ != hipSuccess) {                                                              \
            kv_set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(kv_e_), __FILE__, \
                         __LINE__);                                                             \
            return KV_ERR_DEVICE;                                                               \
        }                                                                                       \
    } while (0)

// a * b with 0 * anything = +-0, also for INF and NaN (v_mul_legacy_f32); the
// IEEE product when neither operand is zero.  A sum s + kv_mul_legacy(0, x)
// is s bit for bit unless s is -0.
__device__ __forceinline__ float kv_mul_legacy(float a, float b)
{
    float r;
    asm("v_mul_legacy_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// AlmostEqualRelative(a, 0.F) of commons/Maths.h:25-34: the projection
// values MLEM leaves unchanged (Reconstructors.h:207-213).
__device__ __forceinline__ bool almost_equal_zero(float a)
{
    const float diff = fabsf(a - 0.f);
    const float A = fabsf(a), B = 0.f;
    const float m = (A < B) ? B : A;  // std::max
    return diff <= __FLT_EPSILON__ * m;
}

inline int64_t kv_nvox(const KvGeom &g) { return (int64_t)g.nx * g.ny * g.nz; }
inline int64_t kv_nray(const KvGeom &g) { return (int64_t)g.np * g.nv * g.nu; }

// ---- launchers (kv_fp.hip, kv_bp.hip, kv_misc.hip) ----------------------
// Forward tiling (fp_tile_pixel: rows per wavefront; fp_xcd_tile and the
// batch kernels' per-XCD lists: detector columns per XCD stripe).  Measured
// at 1024x1024x64 with a 2048^2 detector and 25 views: 8x8 rays per
// wavefront in 32-column stripes, mode R forward 10.9 -> 8.8 ms and mode A
// 10.0 -> 8.3 ms against 64x1 rays per wavefront round-robin.  The batch
// kernels' default layouts: mode R 8, mode A 4 (eight full-size mode-A
// reconstructions, 100 batched iterations: 9.56 s against 10.45 s in 8x8);
// the autotuner may choose others.
// The multi-volume likelihood walk takes its layout by volume count: one
// gather per step, of one volume or of a record holding two or three
// (interleaved first by pack_kernel).  Measured at the size above (walk,
// reductions and packing per call): 6.9 / 7.7 / 10.1 ms for one / two /
// three volumes in 8x8 / 16x4 / 16x4 rays per wavefront; before the current
// mode-A walk, two and three volumes took 9.4 / 11.7 ms in these layouts,
// 10.3 / 13.4 ms in 8x8, three 13.6 ms in 32x2, and one gather per volume
// and step 12.5 / 21.5 ms.
constexpr int KV_XCDS = 8;
constexpr int KV_FP_LAYOUT = 8;
constexpr int KV_FP_LAYOUT_MULTI[KV_LL_MAX] = {8, 4, 4};
constexpr int KV_FP_STRIPE = 32;
// Row-by-row walks: a stripe's chunk is KV_ROW_CY tiles of 64 columns by 4
// rows on one XCD (fp_row_pixel).  Neighbouring rows read nearly the same
// volume rows: with one tile per chunk the rotation of stripes over the XCDs
// sent them to different L2s (1024x1024x64 / 25 views: 3.3 ms; 4, 8 or 16
// tiles, one or two columns wide, 3.0-3.1 ms).  4 keeps small volumes
// balanced (256x256x32 / 15 views: 48 us; two columns by 8 tiles 51 us).
constexpr int KV_ROW_CY = 4;
constexpr int KV_FP_BATCH_LAYOUT_R = 8;
constexpr int KV_FP_BATCH_LAYOUT_A = 4;

// Tiles of the row-by-row walks along tx and ty.
inline int kv_row_tiles_x(int nu) { return (nu + 63) / 64 * KV_ROW_CY; }
inline int kv_row_tiles_y(int nv) { return (nv + 4 * KV_ROW_CY - 1) / (4 * KV_ROW_CY); }
// Tiles of 8 columns by 32 rows over mode R's other columns.
constexpr int KV_FP_TILE = 64 / KV_FP_LAYOUT;
inline int kv_edge_tiles_x(int cols) { return (cols + KV_FP_TILE - 1) / KV_FP_TILE; }
inline int kv_edge_tiles_y(int nv) { return (nv + 4 * KV_FP_LAYOUT - 1) / (4 * KV_FP_LAYOUT); }

hipError_t kv_launch_fp_r(const KvGeom &g, const float *vol, float *out, int epilogue, const float *data,
                          float relax, hipStream_t s);
// Mode-A forward pass.  KV_EP_MLEM writes the MLEM ratio data/Ax
// premultiplied by the ray's length factor from the mode-A tables t (the
// input the mode-A backprojector expects); the other epilogues ignore t.
// Mode-A forward projections of n <= KV_LL_MAX volumes in one walk per ray.
// Without segment lists (KvGeom::seg_a null), n >= 2 volumes are first
// interleaved into pack (4 floats per voxel), so that one gather per step
// reads every volume; pack is unused (may be null) with them.
hipError_t kv_launch_fp_a_multi(const KvGeom &g, int n, const float *const *vols, float *pack, float *const *outs,
                                hipStream_t s);
hipError_t kv_launch_fp_a(const KvGeom &g, const KvTables &t, const float *vol, float *out, int epilogue,
                          const float *data, hipStream_t s);
// Fills KvGeom::seg_a and its heads (lists of g.seg_stride entries).
hipError_t kv_launch_seg_a(const KvGeom &g, KvSeg *seg, KvSegHead *head, hipStream_t s);
// Fills KvGeom::seg_r and its heads.
hipError_t kv_launch_seg_r(const KvGeom &g, KvSegR *seg, KvSegHeadR *head, hipStream_t s);
hipError_t kv_launch_trace(const KvGeom &g, int mode, int nrays, const int32_t *rays, int cap, int64_t *idx,
                           float *w, int32_t *counts, hipStream_t s);
hipError_t kv_launch_tables_r(const KvGeom &g, const KvTables &t, hipStream_t s);
hipError_t kv_launch_tables_a(const KvGeom &g, const KvTables &t, hipStream_t s);
hipError_t kv_launch_bp_r(const KvGeom &g, const KvTables &t, const float *proj, float *vol, int epilogue,
                          hipStream_t s);
// Mode-A backprojection of projections already multiplied by each ray's
// length factor (kv_launch_scale_a, or the forward pass's MLEM epilogue);
// unit_input backprojects the length factors themselves (sensitivity).
hipError_t kv_launch_bp_a(const KvGeom &g, const KvTables &t, const float *proj, float *vol, int epilogue,
                          const float *sens, bool unit_input, hipStream_t s);
// out = proj * length factor of each ray (mode-A tables), np*nv*nu values.
hipError_t kv_launch_scale_a(const KvGeom &g, const KvTables &t, const float *proj, float *out, hipStream_t s);
// Batched passes (MLEM epilogues, mode R or A), a workgroup of 256 threads per
// work item and no more than KV_BATCH_GRID workgroups, which then take several:
// the forward pass over KV_XCDS lists of `total` items, the backprojection over
// one.  posz: every reconstruction has KvGeom::bp_posz.
constexpr long long KV_BATCH_GRID = 1ll << 22;  // a multiple of KV_XCDS
hipError_t kv_launch_fp_batch(int mode, const KvProblem *probs, int nprob, long long total, int iteration, float relax,
                              hipStream_t s);
hipError_t kv_launch_bp_batch(int mode, const KvProblem *probs, int nprob, long long total, int iteration, bool posz,
                              hipStream_t s);
// Per-device address of the no-allocation shift-and-add staging array
// (kv_misc.hip): _init resolves it once per device, with that device current;
// kv_internal_scratch returns it (nullptr before _init).  Word layout:
// [src_y: KV_SAA_NOALLOC_MAX_VIEWS][plane_z: KV_SAA_NOALLOC_MAX_PLANES]
// [shifts: KV_SAA_NOALLOC_MAX_SHIFTS + KV_SAA_PAD].
hipError_t kv_internal_scratch_init(int device);
int32_t *kv_internal_scratch(int device);
hipError_t kv_launch_saa_shifts(int np, int nplanes, float sid, float mF, float voxel_dy, const float *src_y,
                                const float *plane_z, int32_t *shifts, hipStream_t s);
// The shift table of a shift-and-add: the planes' row shifts view by view
// (shift of plane k, view p at [p * nplanes + k]), and KV_SAA_PAD more words
// that may be read.
constexpr int KV_SAA_PAD = 8;
// Planes per chunk of the shift-and-add kernel for these shifts (shift(k, p)
// = row shift of plane k, view p), the largest of 8, 4, 2 whose staged rows
// fit the kernel's LDS, else 1; and the staged rows, 32 or 64.
struct KvSaaPlan {
    int kc, rows;
};
KvSaaPlan kv_saa_plan(int nplanes, int np, const std::function<int(int, int)> &shift);
hipError_t kv_launch_saa(int nu, int nv, int np, const float *proj, const int32_t *shifts, int nplanes,
                         const KvSaaPlan &plan, float *out, hipStream_t s);
hipError_t kv_launch_sum(int64_t n, const float *x, double *partials, int nblocks, hipStream_t s);
hipError_t kv_launch_loglik(const KvGeom &g, const float *data, const float *ax, double *partials, int nblocks,
                            hipStream_t s);

// ---- data path (kv_misc.hip) --------------------------------------------
// px/py/pz: the voxels' grid points per axis (device); paves/spheres: device
// copies of the shape lists.
hipError_t kv_launch_phantom(int nx, int ny, int nz, const float *px, const float *py, const float *pz,
                             float background, const kv_pave *paves, int npaves, const kv_sphere *spheres,
                             int nspheres, float *out, hipStream_t s);
hipError_t kv_launch_correct(int64_t n, int loop, float relax, const float *data, float *proj, hipStream_t s);
hipError_t kv_launch_update(int64_t n, int loop, float *vol, const float *bp, hipStream_t s);
hipError_t kv_launch_log_scale(int64_t n, const float *in, float *out, double c, hipStream_t s);

// ---- trajectory extrapolation (kv_traj.hip) ------------------------------
struct KvTraj {
    const float *x[KV_TRAJ_MAX + 1];  // iterates, oldest first
};
struct KvTrajCoef {
    double c[KV_TRAJ_MAX];
};
// Workgroups of the Gram pass (fixed for a volume size) and the number of
// 4x4 blocks of the upper triangle it writes per workgroup (16 doubles each).
int kv_traj_gram_blocks(int64_t n);
int kv_traj_pairs(int h);
hipError_t kv_launch_traj_gram(const KvTraj &tr, int h, int64_t n, const float *sens, double *partials,
                               hipStream_t s);
hipError_t kv_launch_traj_combine(const KvTraj &tr, const KvTrajCoef &cf, int h, int64_t n, float *out,
                                  hipStream_t s);
