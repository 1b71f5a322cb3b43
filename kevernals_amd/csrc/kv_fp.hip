// Forward projectors for gfx950.
//
// One ray per lane.  Mode A runs row by row where a geometry's segment lists
// exist ("mode A, row by row" below).  Otherwise a 256-thread workgroup is
// four wavefronts, each covering
// a (64/L) x L tile of detector pixels (8 x 8 for the plain walk; 16 x 4 and
// 32 x 2 for the walks that gather two and three volumes per step), so the
// rays of a wavefront stay close in u and v and their voxel gathers at each
// step fall on nearby lines of the x-fastest volume.  Workgroup tiles are
// launched in a one-dimensional order that puts stripes of 32 detector
// columns on the eight XCDs in turn (stripe i on XCD i % 8, each XCD walking
// its stripes column-first), so every XCD's L2 holds one band of the volume.
//
// Mode R reproduces CudaPerformProjection (KevLoq/Kevernals
// source/modules/reconstruction/Projector.cu:227-372) bit for bit.  The
// reference fills a per-thread 2000-float array with 1.0, writes three
// arithmetic runs of plane crossings into it and selection-sorts it
// (FindProjectionAlphas_d, Projector.cu:45-223).  Each run is non-decreasing
// (a[i] = a[i-1] + |1/d| in FP32), so the sorted list is exactly the merge of
// the x run, the y run, the (truncated) z run and the leftover 1.0 fillers:
// here the four runs are merged on the fly in registers, with no scratch
// array and O(n) work instead of O(n^2).
//
// All arithmetic that decides voxel indices is evaluated as the reference
// writes it, with contraction off.
#pragma clang fp contract(off)

#include <algorithm>

#include "kv_internal.h"

// The structured-buffer load intrinsic (no clang builtin spells it):
// rsrc, record index, byte offset within the record, scalar offset, cache
// policy.
typedef int KvRsrc __attribute__((ext_vector_type(4)));
typedef float KvF32x2 __attribute__((ext_vector_type(2)));
typedef float KvF32x4 __attribute__((ext_vector_type(4)));
__device__ float kv_struct_load_f32(KvRsrc rsrc, int vindex, int voffset, int soffset, int aux) __asm(
    "llvm.amdgcn.struct.buffer.load.f32");
__device__ KvF32x2 kv_struct_load_f32x2(KvRsrc rsrc, int vindex, int voffset, int soffset, int aux) __asm(
    "llvm.amdgcn.struct.buffer.load.v2f32");
__device__ KvF32x4 kv_struct_load_f32x4(KvRsrc rsrc, int vindex, int voffset, int soffset, int aux) __asm(
    "llvm.amdgcn.struct.buffer.load.v4f32");

namespace {

constexpr float kInf = __builtin_inff();

// Projector.cu:22-42
__device__ __forceinline__ bool feq(float a, float b, float t)
{
    if (t < 0)
        return (a - b) < -t && (a - b) > t;
    return (a - b) < t && (a - b) > -t;
}
__device__ __forceinline__ bool fsupeq(float a, float b, float t) { return a > b || feq(a, b, t); }

struct RayF {
    float sx, sy, sz;    // source, floating-voxel units
    float dx, dy, dz;    // source -> pixel centre
    float hx, hy, hz;    // half sizes
    float a1x, aNx, ivx; // x-face alphas (0 when |dx| <= 1e-6) and 1/dx (0 when dx = 0)
    float a1y, aNy, ivy; // the same for y
    float a1z, aNz, stz; // z-face alphas and 1/dz (0 when |dz| <= 1e-6)
};

// Projector.cu:303-323.  The terms that depend on the view alone, and those
// of the pixel's detector column and row (its centre coordinate, the face
// alphas and the reciprocal of the direction along that axis), come from the
// geometry's ray constants: the same FP32 operations evaluated once on the
// host.
__device__ __forceinline__ void ray_setup(const KvGeom &g, int p, int u, int v, RayF &r)
{
    const float *C = g.rc + KV_RC * p;
    r.sx = C[0];
    r.sy = C[1];
    r.sz = C[2];
    const float4 cx = *(const float4 *)(g.rc + (size_t)g.np * KV_RC + ((size_t)p * g.nu + u) * 4);
    const float4 cy = *(const float4 *)(g.rc + (size_t)g.np * (KV_RC + 4 * g.nu) + ((size_t)p * g.nv + v) * 4);
    r.dx = cx.x - r.sx;
    r.dy = cy.x - r.sy;
    r.a1x = cx.y;
    r.aNx = cx.z;
    r.ivx = cx.w;
    r.a1y = cy.y;
    r.aNy = cy.z;
    r.ivy = cy.w;
    r.dz = C[3];
    r.hx = (float)g.nx / 2.f;
    r.hy = (float)g.ny / 2.f;
    r.hz = (float)g.nz / 2.f;
    r.a1z = C[4];
    r.aNz = C[5];
    r.stz = C[6];
}

// Projector.cu:88-120
__device__ __forceinline__ void axis_range(float d, float s, float h, int n, float amin, float amax, int &lo, int &hi)
{
    int mx, mn;
    if (d > 0) {
        mx = max(0, min(n - 1, (int)(h + s + amax * d)));
        mn = max(0, min(mx, n - (int)(h - s - amin * d)));
    } else {
        mx = max(0, min(n - 1, (int)(h + s + amin * d)));
        mn = max(0, min(mx, n - (int)(h - s - amax * d)));
    }
    lo = mn;
    hi = mx;
}

// a * b + c on the low 24 bits of a and b, one instruction (the compiler
// would otherwise form two products and a three-way add); b is
// wavefront-uniform (a scalar operand).
__device__ __forceinline__ unsigned mad_u24(unsigned a, unsigned b, unsigned c)
{
    unsigned r;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
}

// a in the lanes whose bit of mask is set, else b: one v_cndmask with a
// scalar mask.  (Not inline assembly: the compiler does not see the wait
// states that a mask fresh from a vector compare needs before one.)
__device__ __forceinline__ float selm(unsigned long long mask, float a, float b)
{
    return __builtin_amdgcn_inverse_ballot_w64(mask) ? a : b;
}

// Distance in alpha from an x face within which the rounding of positions
// (some ulps of the coordinates, in voxels) may matter.
__device__ __forceinline__ float x_face_room(float h, float s, int n, float inc)
{
    return (h + fabsf(s) + (float)n) * 2.4e-7f * inc + 1e-6f;
}

// A wavefront-uniform value in a scalar register.
__device__ __forceinline__ double uniform(double a)
{
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(a)),
                            __builtin_amdgcn_readfirstlane(__double2loint(a)));
}

// min(1, a) as one instruction (a is never NaN where it is used).
__device__ __forceinline__ float min1(float a)
{
    float r;
    asm("v_min_f32 %0, 1.0, %1" : "=v"(r) : "v"(a));
    return r;
}

// min(a, b) as one instruction (operands never NaN where it is used); b may
// be wavefront-uniform.
__device__ __forceinline__ float minf(float a, float b)
{
    float r;
    asm("v_min_f32 %0, %2, %1" : "=v"(r) : "v"(a), "s"(b));
    return r;
}

// Minimum of three run heads as one v_min3_f32.  The heads are finite or
// +INF (never NaN), so the IEEE-mode operand canonicalisation the compiler
// would add for fminf is not needed.
__device__ __forceinline__ float min3f(float a, float b, float c)
{
    float m;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
    return m;
}

// Volume gathers by voxel index: a structured buffer of 4-byte records,
// bounds-checked by index (an index at or past the voxel count reads 0), so
// the gather takes the linear index with no byte-offset shift.
__device__ __forceinline__ KvRsrc voxel_rsrc(const KvGeom &g, const float *vol, unsigned stride = 4)
{
    const unsigned long long a = (unsigned long long)vol;
    KvRsrc r;
    r.x = (int)(unsigned)a;
    r.y = (int)(((unsigned)(a >> 32) & 0xFFFFu) | (stride << 16));  // record stride in bytes
    r.z = g.nx * g.ny * g.nz;                                        // records (at most 2^30)
    r.w = 0x00020000;
    return r;
}

// Mode-R walk of one ray.  visit(ok, voxel_index, weight) is called for every
// segment of the sorted list in order; ok marks the segments the reference
// accepts (Projector.cu:356-366).
// FAST (the geometry's walk_fast flag, set by kv_set_geometry): nx * ny <
// 2^24, so an accepted segment's index vz*(nx*ny) + vy*nx + vx uses full-rate
// 24-bit multiplies (a rejected segment's index is never dereferenced
// outside a bounds-checked buffer access); and for every axis
// (n + 2) * (max|source| + n/2 + 2) < 2^22 in voxel units.  A run's values are
// a0 + j*inc accumulated in FP32 with |a| <= (|s| + n/2) * inc, so after j <= n+1
// additions the accumulated rounding error stays below inc/4: the value
// T = a0 + (c - 1/2) * inc (rounded once to FP32) then lies strictly
// between the run's last value and the one after it, and "exhausted" is one
// comparison with T instead of a count.  Without FAST each run counts down.
template <bool FAST, class Visit>
__device__ __forceinline__ void walk_r(const KvGeom &g, const RayF &r, Visit &&visit)
{
    const float tol = 1e-6f;
    const bool okx = fabsf(r.dx) > tol, oky = fabsf(r.dy) > tol, okz = fabsf(r.dz) > tol;
    // okx ? (-hx - sx) / dx : 0 and the like, from the ray constants
    const float a1x = r.a1x, a1y = r.a1y, a1z = r.a1z;
    const float aNx = r.aNx, aNy = r.aNy, aNz = r.aNz;
    const float amin = fmaxf(fmaxf(0.f, fminf(a1x, aNx)), fmaxf(fminf(a1y, aNy), fminf(a1z, aNz)));
    const float amax = fminf(fminf(1.f, fmaxf(a1x, aNx)), fminf(fmaxf(a1y, aNy), fmaxf(a1z, aNz)));
    if (fsupeq(amin, amax, 1e-7f))
        return;  // the reference's early exit (Projector.cu:79-85): empty list

    int lox, hix, loy, hiy, loz, hiz;
    axis_range(r.dx, r.sx, r.hx, g.nx, amin, amax, lox, hix);
    axis_range(r.dy, r.sy, r.hy, g.ny, amin, amax, loy, hiy);
    axis_range(r.dz, r.sz, r.hz, g.nz, amin, amax, loz, hiz);
    const int n = (hix - lox) + (hiy - loy) + (hiz - loz) + 3;

    // Run heads, lengths and increments (Projector.cu:139-201).  A run whose
    // axis fails |d| > tol leaves its slots at the 1.0 filler.
    int cx = 0, cy = 0, cz = 0;
    float ax = 0.f, ay = 0.f, az = 0.f, ix = 0.f, iy = 0.f, iz = 0.f;
    if (okx) {
        const float st = r.ivx;  // 1 / dx
        ax = st * (-r.hx - r.sx + (float)(r.dx > 0 ? lox : hix));
        ix = fabsf(st);
        cx = hix - lox + 1;
    }
    if (oky) {
        const float st = r.ivy;  // 1 / dy
        ay = st * (-r.hy - r.sy + (float)(r.dy > 0 ? loy : hiy));
        iy = fabsf(st);
        cy = hiy - loy + 1;
    }
    if (okz) {
        // z run written over (hiz-loz)-1 slots, at least its first entry
        // (Projector.cu:181-201).
        const float st = r.stz;  // 1 / dz
        az = st * (-r.hz - r.sz + (float)(r.dz > 0 ? loz : hiz));
        iz = fabsf(st);
        const int dzr = hiz - loz;
        cz = dzr >= 2 ? dzr - 1 : 1;
    }
    const int cf = n - cx - cy - cz;  // 1.0 fillers left unsorted-over
    // T = a0 + (c - 1/2) * inc rounded once to FP32 (one fma: c - 1/2 is
    // exact): |T| < 2^22 / (n + 2) * inc under FAST, so the rounding moves T
    // by less than inc / (4 (n + 2)), far inside the inc / 4 margins above
    // (any T in the band separates the same run values).
    const float tx = FAST ? __builtin_fmaf((float)cx - 0.5f, ix, ax) : 0.f;
    const float ty = FAST ? __builtin_fmaf((float)cy - 0.5f, iy, ay) : 0.f;
    const float tz = FAST ? __builtin_fmaf((float)cz - 0.5f, iz, az) : 0.f;

    // A run's head holds +INF once the run is exhausted, so the next list
    // entry is the plain minimum of the heads.  All heads equal to the
    // minimum are consumed together: equal entries of the sorted list only
    // bound zero-width segments, which Projector.cu:358-359 rejects (w must
    // exceed 1e-6), so the accepted segments and their order are those of
    // the full list.  The 1.0 fillers form one entry for the same reason,
    // merged in between two loops over the runs (values below 1.0, then the
    // rare values above it).
    if (cx == 0) ax = kInf;
    if (cy == 0) ay = kInf;
    if (cz == 0) az = kInf;
    // Steps of the main loops, where m is the minimum head (FAST): only the
    // first run in x, y, z order whose head equals m advances.  A tie
    // between runs is then consumed over several steps, each extra step a
    // zero-width segment that Projector.cu:358-359 rejects, so the accepted
    // segments are unchanged and one run's increment and end threshold are
    // selected instead of stepping all three.
    auto advance1 = [&](float m) {
        // Two vector compares of bit patterns give the lane masks of "x
        // holds m" and "y holds m"; the scalar unit combines them into the
        // three run masks and the selects take them directly (left to
        // itself the compiler negates a mask with a third vector compare).
        // m is one of the three heads, so its bits equal those of the first
        // run that holds it; heads that equal m as floats with other bits
        // (+0 and -0) only order the consumption of equal list entries,
        // which bound zero-width segments.
        const unsigned mb = __float_as_uint(m);
        const unsigned long long mx = __builtin_amdgcn_ballot_w64(__float_as_uint(ax) == mb);
        const unsigned long long my = __builtin_amdgcn_ballot_w64(__float_as_uint(ay) == mb);
        const unsigned long long mpy = my & ~mx, mpz = ~(mx | my);
        const float inc = selm(mx, ix, selm(my, iy, iz));
        const float thr = selm(mx, tx, selm(my, ty, tz));
        float nv = m + inc;
        nv = nv > thr ? kInf : nv;
        ax = selm(mx, nv, ax);
        ay = selm(mpy, nv, ay);
        az = selm(mpz, nv, az);
    };
    // a[i] = a[i-1] + |1/d| in FP32 (Projector.cu:156,177,199)
    auto advance = [&](float m) {
        const bool px = ax == m, py = ay == m, pz = az == m;
        if (FAST) {
            const float nx_ = ax + ix, ny_ = ay + iy, nz_ = az + iz;
            ax = px ? (nx_ > tx ? kInf : nx_) : ax;
            ay = py ? (ny_ > ty ? kInf : ny_) : ay;
            az = pz ? (nz_ > tz ? kInf : nz_) : az;
        } else {
            cx -= px;
            cy -= py;
            cz -= pz;
            ax = px ? (cx == 0 ? kInf : ax + ix) : ax;
            ay = py ? (cy == 0 ? kInf : ay + iy) : ay;
            az = pz ? (cz == 0 ? kInf : az + iz) : az;
        }
    };

    // Segment (prev, cur), Projector.cu:348-367.  The midpoint is the FP32
    // sum divided by 2.0 in FP64.  (double)float * (double)float is exact,
    // and so is the halving, so each index expression equals one FP64 fma of
    // the FP32 sum with the halved direction.  visit(ok, k, w): ok marks an
    // accepted segment; k is its voxel index when ok and meaningless
    // (possibly out of range) otherwise.
    const double bx = (double)(r.hx + r.sx);
    const double by = (double)(r.hy + r.sy);
    const double bz = (double)(r.hz + r.sz);
    const double hdx = 0.5 * (double)r.dx, hdy = 0.5 * (double)r.dy, hdz = 0.5 * (double)r.dz;
    const unsigned nx = (unsigned)g.nx, ny = (unsigned)g.ny, nz = (unsigned)g.nz, nxy = nx * ny;
    auto segment = [&](float prev, float cur) {
        const float w = cur - prev;
        const double sum = (double)(cur + prev);
        const int vx = (int)__builtin_fma(sum, hdx, bx);
        const int vy = (int)__builtin_fma(sum, hdy, by);
        const int vz = (int)__builtin_fma(sum, hdz, bz);
        const bool ok = (unsigned)vx < nx && (unsigned)vy < ny && (unsigned)vz < nz && w > tol;
        const unsigned k = FAST ? mad_u24((unsigned)vz, nxy, mad_u24((unsigned)vy, nx, (unsigned)vx))
                                : ((unsigned)vz * ny + (unsigned)vy) * nx + (unsigned)vx;
        visit(ok, k, w);
    };

    const float fill = cf > 0 ? 1.0f : kInf;
    // first entry
    float prev = min3f(ax, ay, az);
    bool filler_left = cf > 0;
    if (fill <= prev) {
        prev = fill;
        filler_left = false;
    }
    // entries below the fillers' value (all of them when there is no filler);
    // two entries per turn, so that the previous entry needs no copy
    const float lim = filler_left ? fill : kInf;
    // The entries below lim are known in advance when every run of two or
    // more entries ends below lim (its values lie below its end threshold):
    // a run of one entry contributes it if it lies below lim.  Each step of
    // advance1 then takes exactly one of them, so the loop below runs a fixed
    // count of steps: those entries, less the ones the first entry takes
    // (every run head equal to it).  Run entries at or above lim stay for
    // the part after the fillers.
    auto ends_below = [&](int c, float t) { return c <= 1 || t < lim; };
    auto below = [&](int c, float a) { return c == 1 ? (int)(a < lim) : c; };
    const bool counted = FAST && ends_below(cx, tx) && ends_below(cy, ty) && ends_below(cz, tz);
    const int left = (below(cx, ax) + below(cy, ay) + below(cz, az)) - ((ax == prev) + (ay == prev) + (az == prev));
    advance(prev);
    if (counted) {
        // pairs of steps under a wavefront-uniform turn counter (the
        // per-lane count only masks lanes), then the odd step
        const int pairs = left >> 1;
        for (int it = 0;; ++it) {
            const bool act = it < pairs;
            if (!__any(act))
                break;
            if (act) {
                const float c1 = min3f(ax, ay, az);
                advance1(c1);
                segment(prev, c1);
                const float c2 = min3f(ax, ay, az);
                advance1(c2);
                segment(c1, c2);
                prev = c2;
            }
        }
        if (left & 1) {
            const float c1 = min3f(ax, ay, az);
            advance1(c1);
            segment(prev, c1);
            prev = c1;
        }
    } else if (FAST) {
        for (;;) {
            const float c1 = min3f(ax, ay, az);
            if (!(c1 < lim))
                break;
            advance1(c1);
            segment(prev, c1);
            const float c2 = min3f(ax, ay, az);
            if (!(c2 < lim)) {
                prev = c1;
                break;
            }
            advance1(c2);
            segment(c1, c2);
            prev = c2;
        }
    } else {
        for (;;) {
            const float cur = min3f(ax, ay, az);
            if (!(cur < lim))
                break;
            advance(cur);
            segment(prev, cur);
            prev = cur;
        }
    }
    if (filler_left) {
        // the 1.0 entry (run values equal to it are the same entry), then
        // run values above it
        advance(fill);
        segment(prev, fill);
        prev = fill;
        for (;;) {
            const float cur = min3f(ax, ay, az);
            if (cur == kInf)
                break;
            advance(cur);
            segment(prev, cur);
            prev = cur;
        }
    }
}

// Epilogue of the mode-R forward pass for the value fp of ray o.
template <int EP>
__device__ __forceinline__ void fp_r_store(float fp, float *__restrict__ out, const float *__restrict__ data,
                                           float relax, size_t o)
{
    if (EP == KV_EP_PLAIN) {
        out[o] = fp;
    } else if (EP == KV_EP_MLEM) {
        // Reconstructors.h:207-213: the ratio overwrites the projection
        // unless it is (almost) zero, where the projection value stays.
        out[o] = almost_equal_zero(fp) ? fp : relax * (data[o] / fp);
    } else {
        // Reconstructors.h:90-93
        out[o] = relax * (data[o] - fp);
    }
}

// One ray of the mode-R forward pass with its epilogue.
template <int EP>
__device__ __forceinline__ void fp_r_ray(const KvGeom &g, const float *__restrict__ vol, float *__restrict__ out,
                                         const float *__restrict__ data, float relax, int p, int u, int v)
{
    RayF r;
    ray_setup(g, p, u, v, r);
    const size_t o = ((size_t)p * g.nv + v) * g.nu + u;
    if (EP == KV_EP_COUNT) {
        int c = 0;
        walk_r<false>(g, r, [&](bool ok, unsigned, float) { c += ok; });
        out[o] = (float)c;
        return;
    }
    float tot = 0.f, tw = 0.f;
    // Branch-free accumulation: every segment gathers through a
    // bounds-checked buffer resource over the volume (an offset outside it
    // reads 0; a rejected segment's index may lie outside it).  Each segment is added one step after its gather is issued, so the
    // load is in flight while the next segment is walked; the sums take
    // the segments in the same order.  A rejected segment carries weight +0
    // and adds +0 to tw and kv_mul_legacy(+0, value) = +-0 to tot (for any
    // value, INF and NaN included); neither sum is ever -0 (they start at
    // +0 and x + (-x) rounds to +0), so both are left bit-identical.
    const KvRsrc vrs = voxel_rsrc(g, vol);
    float pw = 0.f, pv = 0.f;
    auto acc = [&](bool ok, unsigned k, float w) {
        const float val = kv_struct_load_f32(vrs, (int)k, 0, 0, 0);
        tw = tw + pw;
        tot = tot + kv_mul_legacy(pw, pv);
        pw = ok ? w : 0.f;
        pv = val;
    };
    if (g.walk_fast)
        walk_r<true>(g, r, acc);
    else
        walk_r<false>(g, r, acc);
    tw = tw + pw;
    tot = tot + kv_mul_legacy(pw, pv);
    fp_r_store<EP>(tw > 1e-6f ? tot / tw : 0.f, out, data, relax, o);
}

// Pixel of lane `tid` in forward tile (tx, ty) for tile layout L (1, 2, 4 or
// 8): each wavefront covers 64/L consecutive detector columns of L rows, the
// four wavefronts of a workgroup are stacked along v; a tile is (64/L) x 4L
// pixels.  64/L is a power of two: the lane splits by mask and shift.
__device__ __forceinline__ void fp_tile_pixel(int layout, int tx, int ty, int tid, int &u, int &v)
{
    const int lane = tid & 63, wv = tid >> 6;
    const int wu = 64 / layout;  // uniform
    const int lw = __builtin_ctz((unsigned)wu);
    u = tx * wu + (lane & (wu - 1));
    v = ty * (4 * layout) + wv * layout + (lane >> lw);
}

// n / d for n < 2^31 with the divisor's precomputed multiplier (KvUDiv); on
// wavefront-uniform operands it runs on the scalar unit.
__device__ __forceinline__ unsigned udiv(unsigned n, KvUDiv d) { return (__umulhi(n, d.m) + n) >> d.l; }

// Forward tile of workgroup w in an XCD-aware order.  Workgroups are
// handed to the eight XCDs round-robin by linear id.  The launch is
// one-dimensional over gxp x gy x np tiles; tile columns are grouped in
// stripes of `chunk` tiles, and each XCD walks its stripes column-fastest,
// then rows, then views.  In tile row r (rows and views counted together)
// stripe i goes to XCD (i - r) mod 8.  A stripe keeps an XCD's L2 on a few
// neighbouring detector columns (round-robin single tiles of an 8-column
// layout made every L2 fetch the same volume lines, 43.5 GB per full-size
// launch), and the interleaving balances the eight XCDs' shares of the
// uneven ray lengths (one contiguous band per XCD left the outer bands
// idle: 11.4 ms against 8.8 ms).  Rotating the assignment by one stripe per
// tile row gives every XCD every stripe equally often: with a fixed
// i mod 8 two XCDs carried 7 % more than the mean at full size, as the
// detector's columns hold ray lengths in a V profile cut off at the edges
// of the volume's shadow.  gxp = tile columns rounded up to a multiple of
// 8 x chunk; tiles of padding columns (u past the detector) exit at the
// kernel's bounds test.  A launch covers views p0, p0 + 1, ...  The
// divisions by chunk, the stripe count and gy use precomputed multipliers
// (they were a tenth of the vector instructions a wavefront issues before
// its walk).
__device__ __forceinline__ void fp_xcd_tile(const KvFpMap &fm, unsigned w, int &tx, int &ty, int &p)
{
    constexpr unsigned X = KV_XCDS;
    const unsigned j = w / X;
    const unsigned jc = udiv(j, fm.dchunk), t = j - jc * (unsigned)fm.chunk;
    const unsigned r = udiv(jc, fm.dnch), ci = jc - r * (unsigned)fm.nch;
    tx = (int)((ci * X + (w + r) % X) * (unsigned)fm.chunk + t);
    const unsigned q = udiv(r, fm.dgy);
    ty = (int)(r - q * (unsigned)fm.gy);
    p = fm.p0 + (int)q;
    if (fm.ntx) {
        // a view as one row of tiles, cut into the detector's rows (the
        // padding lies past the last one)
        const unsigned y = udiv((unsigned)tx, fm.dntx);
        ty = (int)y;
        tx -= (int)(y * (unsigned)fm.ntx);
    }
}

template <int EP>
__global__ __launch_bounds__(256) void fp_r_kernel(KvGeom g, const float *__restrict__ vol, float *__restrict__ out,
                                                   const float *__restrict__ data, float relax, KvFpMap fm)
{
    int tx, ty, p, u, v;
    fp_xcd_tile(fm, blockIdx.x, tx, ty, p);
    fp_tile_pixel(fm.layout, tx, ty, threadIdx.x, u, v);
    if (u >= g.nu || v >= g.nv)
        return;
    fp_r_ray<EP>(g, vol, out, data, relax, p, u, v);
}

// Forward pass over a batch of reconstructions.  The tiles sit in KV_XCDS
// lists (KvProblem), list k holding the stripes an XCD-ordered launch gives
// XCD k (fp_xcd_tile), `total` items per list; the launch deals a workgroup per
// item round the lists, as a one-dimensional launch deals workgroups round the
// XCDs (the placement only decides the caches' locality).  Workgroups that
// stay and claim tiles from a counter per list were slower: claims are atomics
// on one word, some 70 ns each.  An iteration of six reconstructions of
// 384x320x48 voxels and less (18 000 tiles a list) took 1.67 / 1.65 ms in mode
// R / A with one tile per claim, 0.96 / 0.84 with eight; it takes 0.75 / 0.72.
// Problems whose iteration count is reached skip their tiles; padding columns
// (u past the detector) are skipped at the bounds test.
template <typename Tile>
__device__ __forceinline__ void fp_batch_tiles(const KvProblem *__restrict__ probs, int nprob, long long total,
                                               int iteration, Tile &&tile)
{
    const int k = (int)(blockIdx.x % (unsigned)KV_XCDS);  // (the grid is a multiple of KV_XCDS)
    for (long long item = blockIdx.x / (unsigned)KV_XCDS; item < total; item += gridDim.x / (unsigned)KV_XCDS) {
        // the last descriptor whose items begin at or before this one (by
        // halves: each step waits for a load)
        int pi = 0;
        for (int n = nprob; n > 1; n -= n / 2)
            if (probs[pi + n / 2].fp_first <= item)
                pi += n / 2;
        const KvProblem &P = probs[pi];
        if (iteration >= P.iters)
            continue;
        // item indices within a reconstruction stay far below 2^31 (it
        // has fewer than 2^31 rays, 256 per tile): 32-bit divisions by
        // the precomputed multipliers
        const unsigned local = (unsigned)(item - P.fp_first);
        const unsigned ch = (unsigned)P.fp_chunk, nch = (unsigned)P.fp_nch;
        const unsigned jc = udiv(local, P.fp_dchunk), r = udiv(jc, P.fp_dnch);
        const unsigned lin = ((jc - r * nch) * KV_XCDS + (unsigned)k) * ch + (local - jc * ch);
        const unsigned q = udiv(lin, P.fp_dtx);
        const int ty = (int)q, tx = (int)(lin - q * (unsigned)P.fp_tx), p = (int)r;
        if (ty >= P.fp_ty)
            continue;  // padding of the view's last stripes
        tile(P, p, tx, ty);
    }
}

// ---------------------------------------------------------------- mode A --
struct RayA {
    float s[3], d[3], inv[3], h[3];
    int n[3];
    int fixed[3];
    float L;
};

__device__ __forceinline__ void ray_setup_a(const KvGeom &g, int p, int u, int v, RayA &r)
{
    RayF f;
    ray_setup(g, p, u, v, f);
    r.s[0] = f.sx; r.s[1] = f.sy; r.s[2] = f.sz;
    r.d[0] = f.dx; r.d[1] = f.dy; r.d[2] = f.dz;
    r.h[0] = f.hx; r.h[1] = f.hy; r.h[2] = f.hz;
    r.n[0] = g.nx; r.n[1] = g.ny; r.n[2] = g.nz;
    r.inv[0] = f.ivx;
    r.inv[1] = f.ivy;
    r.inv[2] = r.d[2] != 0.f ? 1.f / r.d[2] : 0.f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        r.fixed[c] = 0;
        if (r.d[c] == 0.f) {
            const float pos = r.s[c] + r.h[c];
            r.fixed[c] = (pos > 0.f && pos < (float)r.n[c]) ? (int)floorf(pos) : -1;
        }
    }
    const float lx = r.d[0] * g.sx, ly = r.d[1] * g.sy, lz = r.d[2] * g.sz;
    r.L = sqrtf(lx * lx + ly * ly + lz * lz);
}

__device__ __forceinline__ float plane_a(const RayA &r, int c, int k)
{
    return (((float)k - r.h[c]) - r.s[c]) * r.inv[c];
}

// Maximum of three values as one v_max3_f32 (operands finite or -INF, never
// NaN: no canonicalisation needed).
__device__ __forceinline__ float max3f(float a, float b, float c)
{
    float m;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
    return m;
}

// Mode-A Siddon walk: visit(ok, voxel, len) for every voxel the ray's
// parameter interval [ain, aout] passes through, ok = len > 0 (voxel is the
// linear index; in range for every call).
// Each axis keeps the crossing of its next plane, hi = ((k - N/2) - s) / d
// evaluated as plane_a does, with k - N/2 carried as an exact float (an
// integer or half-integer far below 2^24), the crossing of the last plane
// passed (lo) and the voxel index folded into one linear index.  The axis
// that exits first (first minimum on ties, as the oracle) is found from the
// minimum of the three heads; an axis without motion holds hi = +INF.  The
// walk ends when the nearest exit reaches aout: the exit through an axis's
// boundary plane is that plane's crossing, which is where aout comes from,
// so no index is ever stepped outside the volume.
template <class Visit>
__device__ __forceinline__ void walk_a(const RayA &r, Visit &&visit)
{
    float ain = 0.f, aout = 1.f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (r.d[c] == 0.f) {
            if (r.fixed[c] < 0)
                return;
            continue;
        }
        const float a0 = plane_a(r, c, 0), aN = plane_a(r, c, r.n[c]);
        ain = fmaxf(ain, fminf(a0, aN));
        aout = fminf(aout, fmaxf(a0, aN));
    }
    if (!(ain < aout))
        return;
    int ii[3];
    float lo[3], hi[3], kf[3], st[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (r.d[c] == 0.f) {
            ii[c] = r.fixed[c];
            lo[c] = -kInf;
            hi[c] = kInf;
            kf[c] = 0.f;
            st[c] = 0.f;
            continue;
        }
        const float pos = r.s[c] + r.h[c] + ain * r.d[c];
        int i = (int)floorf(pos);
        i = max(0, min(r.n[c] - 1, i));
        const int stp = r.d[c] > 0.f ? 1 : -1;
        // lo/hi of voxel i on axis c
        auto lohi = [&](int k, float &l, float &h) {
            const float a0 = plane_a(r, c, k), a1 = plane_a(r, c, k + 1);
            l = fminf(a0, a1);
            h = fmaxf(a0, a1);
        };
        float l, h;
        for (;;) {
            lohi(i, l, h);
            const int j = i - stp;
            if (l > ain && j >= 0 && j < r.n[c]) i = j; else break;
        }
        for (;;) {
            lohi(i, l, h);
            const int j = i + stp;
            if (h <= ain && j >= 0 && j < r.n[c]) i = j; else break;
        }
        ii[c] = i;
        lo[c] = l;
        hi[c] = h;
        // the plane whose crossing is hi: k = i + 1 going up, i going down
        kf[c] = (float)(stp > 0 ? i + 1 : i) - r.h[c];
        st[c] = (float)stp;
    }
    const int nx = r.n[0], nxy = r.n[0] * r.n[1];
    const int sx = (int)st[0], sy = (int)st[1] * nx, sz = (int)st[2] * nxy;
    unsigned idx = (unsigned)(ii[2] * nxy + ii[1] * nx + ii[0]);
    const int guard = r.n[0] + r.n[1] + r.n[2] + 3;
    // max(0, lo[0], lo[1], lo[2]) of the current voxel.  The exiting axis's
    // lo becomes its old hi, which is the step's minimum head and at least
    // its old lo, so the new maximum is max(old maximum, that minimum): one
    // running max, the same value as the maximum over the three axes (IEEE
    // max of non-NaN values is associative).
    float ent = fmaxf(0.f, max3f(lo[0], lo[1], lo[2]));
    // One step: visit the segment through the current voxel, then true at
    // the walk's end, else move to the next voxel.  The exit axis's lane
    // masks come from two vector compares (the scalar unit forms the first-
    // minimum masks), and the selects take them directly.  Two steps per
    // turn of the guard loop: the guard only bounds the walk (a ray crosses
    // fewer planes than it counts), so one test per two steps will do.
    auto step = [&]() {
        const float best = min3f(hi[0], hi[1], hi[2]);
        const float len = min1(best) - ent;
        visit(len > 0.f, idx, len);
        if (best >= aout)
            return true;
        ent = max3f(ent, best, best);
        const unsigned long long m0 = __builtin_amdgcn_ballot_w64(hi[0] == best);
        const unsigned long long m1 = __builtin_amdgcn_ballot_w64(hi[1] == best);
        const unsigned long long p1 = m1 & ~m0, p2 = ~(m0 | m1);
        idx += (unsigned)__float_as_int(
            selm(m0, __int_as_float(sx), selm(p1, __int_as_float(sy), __int_as_float(sz))));
        // the exiting axis: its next plane (same operation sequence as plane_a)
        const float k0 = kf[0] + st[0], k1 = kf[1] + st[1], k2 = kf[2] + st[2];
        hi[0] = selm(m0, (k0 - r.s[0]) * r.inv[0], hi[0]);
        hi[1] = selm(p1, (k1 - r.s[1]) * r.inv[1], hi[1]);
        hi[2] = selm(p2, (k2 - r.s[2]) * r.inv[2], hi[2]);
        kf[0] = selm(m0, k0, kf[0]);
        kf[1] = selm(p1, k1, kf[1]);
        kf[2] = selm(p2, k2, kf[2]);
        return false;
    };
    for (int n = 0; n < guard; n += 2) {
        if (step())
            break;
        if (step())
            break;
    }
}

// Sum over a mode-A walk of len * vol[voxel] for the accepted segments, the
// value of acc = ok ? acc + len * v : acc, with no branch around the load:
// every step gathers its voxel (the walk's indices are always in range) and
// a rejected segment carries weight +0, whose legacy product is +-0 for any
// voxel value (INF and NaN included) and leaves acc unchanged (acc starts
// at +0 and never becomes -0); an accepted weight is positive, where the
// legacy product is the IEEE one.  Each product is added one step later, so
// that the load is in flight while the next step is walked.
struct AccA {
    KvRsrc rs;
    float acc = 0.f, pw = 0.f, pv = 0.f;
    __device__ __forceinline__ void init(const KvGeom &g, const float *vol) { rs = voxel_rsrc(g, vol); }
    __device__ __forceinline__ void visit(bool ok, unsigned k, float len)
    {
        const float v = kv_struct_load_f32(rs, (int)k, 0, 0, 0);
        acc = acc + kv_mul_legacy(pw, pv);
        pw = ok ? len : 0.f;
        pv = v;
    }
    __device__ __forceinline__ float sum() const { return acc + kv_mul_legacy(pw, pv); }
};

// ------------------------------------------------- mode A, row by row ----
// The y and z plane crossings of a ray depend only on its view and detector
// row, so the 64 rays of a wavefront that covers 64 columns of one row share
// the sequence of (y, z) segments: alpha interval and volume row.  That
// sequence is a list built once per geometry (seg_a_kernel) and read by
// scalar loads; each lane only follows its x crossings inside the segments.
// The crossings, voxel order, lengths and sums are those of walk_a, so the
// result is bit-identical to it.
//
// walk_a was bound by instruction issue and by the L1's tag lookups (29.5
// vector instructions and one gather of ~34 cache lines per voxel step,
// because the lanes of an 8x8 tile drift apart in y and z).  A segment holds
// 1.25 voxel steps on average and costs 13 vector instructions and one load
// of neighbouring voxels in seg_sums_row, 20 and two loads in seg_sums.

// The x crossings of one lane: the plane its voxel ends at, as f = k - nx/2
// (an integer or half-integer below 2^24: exact), its step and its crossing
// hx = (f - s) * inv as plane_a evaluates it, and the voxel's x index j (k - 1
// going up, k going down).  Voxels off the volume in x (j < 0 or j >= nx)
// read 0 through the bounds-checked row loads, and all of those ahead of the
// ray's entry count as one, whose exit is the entry plane.  A lane whose ray
// never enters the segments' part of the volume rests outside: hx = +INF.
struct LaneX {
    float hx, f, st, s, inv, d;
    int j;
    bool live;
};

__device__ __forceinline__ LaneX lane_x(const KvGeom &g, int p, int u, float a, float end)
{
    LaneX l;
    const float4 c = *(const float4 *)(g.rc + (size_t)g.np * KV_RC + ((size_t)p * g.nu + u) * 4);
    const int n = g.nx;
    const float h = (float)n / 2.f;
    l.s = g.rc[KV_RC * p];
    l.inv = c.w;
    l.d = c.x - l.s;
    l.st = l.d > 0.f ? 1.f : -1.f;
    const float pos = l.s + h;
    const int up = l.d > 0.f ? 1 : 0;
    auto exit_of = [&](int i) { return (((float)(i + up) - h) - l.s) * c.w; };
    if (l.d == 0.f) {
        l.j = (pos > 0.f && pos < (float)n) ? (int)floorf(pos) : -1;
        l.live = l.j >= 0;
    } else {
        // the voxel with entry <= a < exit, or the outside voxel ahead of
        // the entry plane; past the far face the ray has left
        const int st = up ? 1 : -1;
        int i = (int)fminf(fmaxf(floorf(pos + a * l.d), -1.f), (float)n);
#pragma clang loop unroll(disable)
        while ((up ? i >= 0 : i < n) && exit_of(i - st) > a)
            i -= st;
#pragma clang loop unroll(disable)
        while ((up ? i < n : i >= 0) && exit_of(i) <= a)
            i += st;
        l.j = i;
        l.hx = exit_of(i);
        l.live = (up ? i < n : i >= 0) && ((unsigned)i < (unsigned)n || l.hx < end);
    }
    l.f = (float)(l.j + up) - h;
    if (l.d == 0.f || !l.live) {
        // nothing is crossed: (f - s) * inv stays +INF
        l.j = l.live ? l.j : -1;
        l.f = l.live ? (float)l.j - h : -1.f - h;
        l.s = -kInf;
        l.inv = 1.f;
        l.hx = kInf;
        l.st = 0.f;
    }
    return l;
}

// Segments per block: a block's loads are in flight while the block before it
// is walked.  With one segment at a time the loads' latency lay open: 70 % of
// the wavefronts' time was spent waiting (1024x1024x64 forward pass, 25 views
// of 2048^2: 5.4 ms against 4.2 ms, both with the gathers of seg_sums).
constexpr int SEG_DEPTH = 4;
static_assert(4 * SEG_DEPTH <= KV_SEG_PAD, "seg_sums_row reads at most 4 blocks past its last segment's");

typedef const __attribute__((address_space(4))) KvSegHead KvSegHeadC;
typedef const __attribute__((address_space(4))) KvSeg KvSegC;
// A block of segments as one scalar load: b and row of segment k are words
// 2 k and 2 k + 1.
typedef unsigned KvSegBlock __attribute__((ext_vector_type(2 * SEG_DEPTH)));
typedef const __attribute__((address_space(4), aligned(8))) KvSegBlock KvSegBlockC;

// The sums of NV volumes over a row's segments for any rays: two gathers of
// one volume row per segment and volume, and further turns on a segment with
// more than one x plane of some lane.
template <int NV>
__device__ __forceinline__ void seg_sums(const KvRsrc (&rs)[NV], int nx, KvSegC *sp, int segs, float a, LaneX &l,
                                         float *sum)
{
    // The products of a segment are added SEG_DEPTH segments later.  Weights
    // start at 0: a legacy product by 0 is +-0 whatever the voxel, and the
    // sums are never -0.  Likewise a lane that crosses no plane has w2 = 0
    // and leaves v2 as it was.
    float w1[SEG_DEPTH], w2[SEG_DEPTH], v1[NV][SEG_DEPTH], v2[NV][SEG_DEPTH];
#pragma unroll
    for (int k = 0; k < SEG_DEPTH; ++k) {
        w1[k] = w2[k] = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i)
            v1[i][k] = v2[i][k] = 0.f;
    }
    auto add = [&](int k) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            sum[i] = sum[i] + kv_mul_legacy(w1[k], v1[i][k]);
            sum[i] = sum[i] + kv_mul_legacy(w2[k], v2[i][k]);
        }
    };
    float x = a;
    float b = sp[0].b, nb = sp[1].b;
    unsigned row = sp[0].row, nrow = sp[1].row;
    const int dj = (int)l.st;
    for (int n = 0; n < segs;) {
#pragma unroll
        for (int k = 0; k < SEG_DEPTH; ++k) {
            add(k);
#pragma unroll
            for (int i = 0; i < NV; ++i)
                v1[i][k] = kv_struct_load_f32(rs[i], l.j, 0, (int)row, 0);
            const bool cross = l.hx < b;
            const float x1 = minf(l.hx, b);
            w1[k] = x1 - x;
            l.j += cross ? dj : 0;
            l.f += cross ? l.st : 0.f;
            l.hx = (l.f - l.s) * l.inv;
            if (cross)
#pragma unroll
                for (int i = 0; i < NV; ++i)
                    v2[i][k] = kv_struct_load_f32(rs[i], l.j, 0, (int)row, 0);
            x = minf(l.hx, b);
            w2[k] = x - x1;
            // another turn on this segment as long as some lane with a plane
            // ahead in it is inside the volume (the others read 0 whatever
            // their weights), so at most nx turns
            if ((__builtin_amdgcn_ballot_w64(l.hx < b) & __builtin_amdgcn_ballot_w64((unsigned)l.j < (unsigned)nx)) == 0) {
                ++n;
                b = nb;
                row = nrow;
                nb = sp[n + 1].b;
                nrow = sp[n + 1].row;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < SEG_DEPTH; ++k)
        add(k);
}

// The same for rays that cross at most one x plane per segment and stay
// within 64 voxels of each other (row_sums decides).  A volume row is then
// one load of neighbouring voxels, voxel i in lane i % 64, from which each
// lane takes its two voxels by a lane permute (which selects by index modulo
// 64 itself).  The gathers were bound by the L1 (10 cycles per load and CU:
// 4.0 ms at the size above, 8.0 / 11.9 ms for two / three volumes); this form
// takes 3.0 ms, bound by instruction issue, and 6.3 / 9.2 ms, bound by the
// L1's row loads (texture addressers 83 % busy).
//
// Rows are loaded one block ahead.  A window placed when block n starts holds
// every voxel of blocks n and n + 1: the lanes' range now, plus `below` /
// `above` voxels the lanes may move in two blocks and one of slack on each
// side (lanes are ordered in x up to the rounding of their crossings).
template <int NV>
__device__ __forceinline__ void seg_sums_row(const KvRsrc (&rs)[NV], float h, KvSegC *sp, int segs, float a,
                                             LaneX &l, unsigned long long live, int below, int above, float *sum)
{
    // f + MAGIC has an ulp of 1/4: the bits of the sum count quarters of a
    // voxel, i.e. they are a permute's byte address (64 lanes x 4 bytes) up
    // to a constant, for |f| < 2^20.
    constexpr float MAGIC = 3145728.f;  // 1.5 * 2^21
    const int lane = (int)(threadIdx.x & 63);
    const int first = __builtin_ctzll(live), last = 63 - __builtin_clzll(live);
    // bits of (voxel index + fc) + MAGIC: j = k - 1 or k, f = k - h
    const float up = l.st > 0.f ? 1.f : 0.f;
    const float ac = MAGIC + (h - up);  // f + ac = j + MAGIC, exact
    constexpr int MAGIC_BITS = 0x4A400000;
    int at = __float_as_int(l.f + ac);
    KvSegBlock q, nq, mq;
    auto read = [&](KvSegBlock &d) {
        d = *(KvSegBlockC *)sp;
        sp += SEG_DEPTH;
    };
    // Ends the time a block may be in flight: its words are in scalar
    // registers from here on (loads of constant memory would otherwise be
    // moved to, or issued again at, their first use, and waited for there).
    auto arrived = [](KvSegBlock &d) { asm volatile("" : "+s"(d)); };
    float ra[NV][SEG_DEPTH], rb[NV][SEG_DEPTH];
    auto rows = [&](const KvSegBlock &d, float (&r)[NV][SEG_DEPTH]) {
        const int j0 = (__builtin_amdgcn_readlane(at, first) - MAGIC_BITS) >> 2,
                  j1 = (__builtin_amdgcn_readlane(at, last) - MAGIC_BITS) >> 2;
        const int base = min(j0, j1) - 1 - below, width = max(j0, j1) + 2 + above - base;
        const int o = (lane - base) & 63;
        const int i = o < width ? base + o : -1;
#pragma unroll
        for (int k = 0; k < SEG_DEPTH; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v)
                r[v][k] = kv_struct_load_f32(rs[v], i, 0, (int)d[2 * k + 1], 0);
    };
    auto walk = [&](const KvSegBlock &d, const float (&r)[NV][SEG_DEPTH]) {
        float w1[SEG_DEPTH], w2[SEG_DEPTH], v1[NV][SEG_DEPTH], v2[NV][SEG_DEPTH];
#pragma unroll
        for (int k = 0; k < SEG_DEPTH; ++k) {
            const float b = __uint_as_float(d[2 * k]);
#pragma unroll
            for (int v = 0; v < NV; ++v)
                v1[v][k] = __int_as_float(__builtin_amdgcn_ds_bpermute(at, __float_as_int(r[v][k])));
            const float x1 = minf(l.hx, b);
            w1[k] = x1 - a;
            w2[k] = b - x1;
            l.f += l.hx < b ? l.st : 0.f;
            l.hx = (l.f - l.s) * l.inv;
            at = __float_as_int(l.f + ac);
#pragma unroll
            for (int v = 0; v < NV; ++v)
                v2[v][k] = __int_as_float(__builtin_amdgcn_ds_bpermute(at, __float_as_int(r[v][k])));
            a = b;
        }
        __builtin_amdgcn_sched_barrier(0);  // every permute issued before the first is waited for
#pragma unroll
        for (int k = 0; k < SEG_DEPTH; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                sum[v] = sum[v] + kv_mul_legacy(w1[k], v1[v][k]);
                sum[v] = sum[v] + kv_mul_legacy(w2[k], v2[v][k]);
            }
    };
    read(q);
    read(nq);
    arrived(q);
    arrived(nq);
    rows(q, ra);
    for (int n = 0; n < segs; n += 2 * SEG_DEPTH) {
        rows(nq, rb);
        read(mq);
        __builtin_amdgcn_sched_barrier(0);
        walk(q, ra);
        __builtin_amdgcn_sched_barrier(0);
        arrived(mq);
        if (n + SEG_DEPTH >= segs)
            break;
        rows(mq, ra);
        read(q);
        __builtin_amdgcn_sched_barrier(0);
        walk(nq, rb);
        __builtin_amdgcn_sched_barrier(0);
        arrived(q);
        nq = q;
        q = mq;
    }
    // the other lanes permuted some lane's voxels with weights of their own
#pragma unroll
    for (int v = 0; v < NV; ++v)
        sum[v] = l.live ? sum[v] : 0.f;
}

// Line sums (alpha length x voxel, not yet times the ray length) of NV
// volumes along the ray of view p, column u, row v; v and p are
// wavefront-uniform.  vol[i] must hold g.nx * g.ny * g.nz floats.
template <int NV>
__device__ __forceinline__ void row_sums(const KvGeom &g, const float *const *vol, int p, int u, int v, float *sum)
{
    const size_t id = (size_t)p * g.nv + v;
    KvSegHeadC *hp = (KvSegHeadC *)(size_t)(g.seg_a_head + id);
    KvSegC *sp = (KvSegC *)(size_t)(g.seg_a + id * (size_t)g.seg_stride);
    const int segs = hp->segs;
#pragma unroll
    for (int i = 0; i < NV; ++i)
        sum[i] = 0.f;
    if (segs == 0)
        return;
    KvRsrc rs[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        // records = the voxels of one row: the row itself is the scalar
        // offset, which the bounds check leaves out
        const unsigned long long at = (unsigned long long)vol[i];
        rs[i].x = (int)(unsigned)at;
        rs[i].y = (int)(((unsigned)(at >> 32) & 0xFFFFu) | (4u << 16));
        rs[i].z = g.nx;
        rs[i].w = 0x00020000;
    }
    const float a = hp->a, longest = hp->longest, end = hp->end;
    {
        // none of the columns' rays between the x faces while in the
        // segments (by the reference's face alphas, good to a few ulps)
        const float4 c = *(const float4 *)(g.rc + (size_t)g.np * KV_RC + ((size_t)p * g.nu + u) * 4);
        if (!__any(c.y == c.z || (fminf(c.y, c.z) < end + 1e-5f && fmaxf(c.y, c.z) > a - 1e-5f)))
            return;
    }
    LaneX l = lane_x(g, p, u, a, end);
    const unsigned long long live = __builtin_amdgcn_ballot_w64(l.live);
    if (live == 0)
        return;
    // Steepness and distance of the rays in x: |d| planes per unit of alpha,
    // largest at an end of the wavefront's live columns; the lanes' distance
    // grows along the rays.  With coordinates below 2^16 voxels FP32
    // positions are good to a fraction of a voxel.
    const float df = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l.d), __builtin_ctzll(live))),
                dl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l.d), 63 - __builtin_clzll(live)));
    const float steep = fmaxf(fabsf(df), fabsf(dl)) * longest;
    const int ahead = (int)fminf(steep * (2.f * SEG_DEPTH), 64.f) + 2;
    const int below = __any(l.live && l.st < 0.f) ? ahead : 0, above = __any(l.live && l.st > 0.f) ? ahead : 0;
    // One plane per segment at most: crossings lie 1 / |d| apart up to their
    // FP32 rounding (below 4e-7 in alpha for the two; 1e-6 taken).
    const bool single = steep + (fabsf(df) + fabsf(dl)) * 1e-6f < 1.f;
    const float range = end * fabsf(dl - df) + 4.f + (float)(below + above);
    if (single && range <= 63.f && fmaxf(fabsf(df), fabsf(dl)) < 65536.f && fabsf(g.rc[KV_RC * p]) < 65536.f &&
        g.nx < 65536)
        seg_sums_row<NV>(rs, (float)g.nx / 2.f, sp, segs, a, l, live, __builtin_amdgcn_readfirstlane(below),
                         __builtin_amdgcn_readfirstlane(above), sum);
    else
        seg_sums<NV>(rs, g.nx, sp, segs, a, l, sum);
}

// The mode-A segment list of one (view, detector row) per thread: walk_a
// restricted to y and z.
__global__ __launch_bounds__(64) void seg_a_kernel(KvGeom g, KvSeg *__restrict__ seg, KvSegHead *__restrict__ head)
{
    const int id = blockIdx.x * 64 + threadIdx.x;
    if (id >= g.np * g.nv)
        return;
    const int p = id / g.nv, v = id - p * g.nv;
    const float *C = g.rc + KV_RC * p;
    const float4 cy = *(const float4 *)(g.rc + (size_t)g.np * (KV_RC + 4 * g.nu) + ((size_t)p * g.nv + v) * 4);
    const float s[2] = {C[1], C[2]}, d[2] = {cy.x - C[1], C[3]}, h[2] = {(float)g.ny / 2.f, (float)g.nz / 2.f};
    const float inv[2] = {cy.w, C[3] != 0.f ? 1.f / C[3] : 0.f};
    const int n[2] = {g.ny, g.nz};
    auto plane = [&](int c, int k) { return (((float)k - h[c]) - s[c]) * inv[c]; };
    head[id] = KvSegHead{0.f, 0.f, 0.f, 0};
    float ain = 0.f, aout = 1.f;
    int ii[2], stp[2];
    float hi[2];
    for (int c = 0; c < 2; ++c) {
        if (d[c] == 0.f) {
            const float pos = s[c] + h[c];
            if (!(pos > 0.f && pos < (float)n[c]))
                return;
            continue;
        }
        const float a0 = plane(c, 0), aN = plane(c, n[c]);
        ain = fmaxf(ain, fminf(a0, aN));
        aout = fminf(aout, fmaxf(a0, aN));
    }
    if (!(ain < aout))
        return;
    for (int c = 0; c < 2; ++c) {
        if (d[c] == 0.f) {
            ii[c] = (int)floorf(s[c] + h[c]);
            hi[c] = kInf;
            stp[c] = 0;
            continue;
        }
        int i = max(0, min(n[c] - 1, (int)floorf(s[c] + h[c] + ain * d[c])));
        const int st = d[c] > 0.f ? 1 : -1;
        // entry and exit crossings of voxel i
        auto lo_of = [&](int k) { return st > 0 ? plane(c, k) : plane(c, k + 1); };
        auto hi_of = [&](int k) { return st > 0 ? plane(c, k + 1) : plane(c, k); };
        while (lo_of(i) > ain && i - st >= 0 && i - st < n[c])
            i -= st;
        while (hi_of(i) <= ain && i + st >= 0 && i + st < n[c])
            i += st;
        ii[c] = i;
        hi[c] = hi_of(i);
        stp[c] = st;
    }
    KvSeg *out = seg + (size_t)id * g.seg_stride;
    const int cap = g.seg_stride - KV_SEG_PAD;
    float a = ain, longest = 0.f;
    unsigned row = 0;
    int m = 0;
    while (m < cap) {
        const float best = fminf(hi[0], hi[1]);
        const float b = fminf(1.f, best);
        if (b > a) {
            row = (((unsigned)ii[1] * (unsigned)g.ny + (unsigned)ii[0]) * (unsigned)g.nx) * 4u;
            out[m++] = KvSeg{b, row};
            longest = fmaxf(longest, b - a);
            a = b;
        }
        if (best >= aout)
            break;
        const int c = hi[0] == best ? 0 : 1;
        ii[c] += stp[c];
        hi[c] = stp[c] > 0 ? plane(c, ii[c] + 1) : plane(c, ii[c]);
    }
    head[id] = KvSegHead{ain, a, longest, m};
    for (int k = 0; k < KV_SEG_PAD; ++k)
        out[m + k] = KvSeg{a, row};
}

// ------------------------------------------------- mode R, row by row ----
// As in mode A, the 64 rays of a wavefront on one detector row share the y
// and z planes.  The reference's runs depend on the ray's alpha range: a run
// starts at the first plane after alpha_min and sums its increment in FP32.
// Where the y and z faces set the range, the y run and the z run are the same
// values for the whole row; their merge is a list built once per geometry
// (seg_r_kernel), and a lane merges in only its own x run.  The columns whose
// rays cross no x face inside the z slab are one interval per view (rc[KV_RC p
// + 11, 12]); the others are walked voxel by voxel in 8x8 tiles by the same
// launch (a tenth of the rays that meet a 1024x1024x64 volume).
//
// A segment [a, b] of the list and at most one x crossing c in it give the
// reference's segments [a, b], or [a, c] and [c, b].  The reference finds
// each one's voxel from its midpoint in FP64.  That voxel is the one that
// stepping from plane to plane gives unless the midpoint lies closer to a
// plane than the rounding of the run values (about 1e-6 in alpha against a
// mean segment of 5e-4):
//  * y and z: the builder finds, in FP64, the sums of two list values
//    between which the midpoint's row is the segment's own.  It flags
//    segments whose own midpoint fails, or which the reference rejects, and
//    turns the bounds into an interval of c (m, r).
//  * x: a run value differs from the plane's crossing, as the FP64 midpoint
//    formula has it, by at most E = P/|d| + 2^-24 (3 + n/2) after n
//    additions of values below 1: P the rounding of the plane's position
//    (rc[KV_RC p + 10], voxels), 2^-25 per addition, 1/d's rounding in the
//    first value (2^-24) and in n increments (2^-24 in all), the first
//    product's and the midpoint sum's (2^-25 each).  A segment longer than
//    delta = 2 E therefore has its midpoint between the planes that bound
//    it; delta also covers the acceptance w > 1e-6.
// Lanes whose c lies within delta of an end of the interval look up the x
// index in FP64 (one segment in ten of a wavefront), lanes outside it and
// flagged segments take the reference's whole arithmetic (one in 50).
// Likewise the x entries before the list's first value and everything after
// its last one.  Within 4e-5 of the row's alpha range's ends a segment is
// flagged, so that the ends of the x run (which planes the FP32 positions of
// Projector.cu:88-120 include) need no thought elsewhere: a run value past
// the run's end lies beyond alpha_max less that margin.
//
// A step of walk_r takes 32.5 vector instructions; a segment, 1.25 steps on
// average, takes 18 here and one row load instead of gathers.  Forward pass of
// 1024x1024x64 / 25 views of 2048^2 6.45 -> 4.43 ms, 512x512x48 / 21 views of
// 1024^2 0.79 -> 0.55, 256x256x32 / 15 views of 512^2 0.087 -> 0.071, 128x128x32
// / 15 views of 256^2 0.026 -> 0.022 (bound by the latency of a wavefront).

typedef const __attribute__((address_space(4))) KvSegHeadR KvSegHeadRC;
typedef const __attribute__((address_space(4))) KvSegR KvSegRC;
typedef unsigned KvSegBlockR __attribute__((ext_vector_type(4 * SEG_DEPTH)));
typedef const __attribute__((address_space(4), aligned(16))) KvSegBlockR KvSegBlockRC;

// One lane's x run: head, increment, end threshold (walk_r), x index in bytes
// of a row, and twice the bound E.
struct LaneR {
    float hx, inc, tx, delta;
    int at, dat;
};

// Ray sums (tot, tw) of the lanes in mask `in` along a row's segment list.
__device__ __forceinline__ void seg_sums_r(const KvGeom &g, const float *__restrict__ vol, const RayF &r,
                                           KvSegHeadRC *hp, KvSegRC *sp, unsigned long long in, int below, int above,
                                           LaneR &l, float &tot, float &tw)
{
    // (the y and z terms are uniform: scalar registers)
    const double bx = uniform((double)(r.hx + r.sx)), by = uniform((double)(r.hy + r.sy)),
                 bz = uniform((double)(r.hz + r.sz));
    const double hdx = 0.5 * (double)r.dx, hdy = uniform(0.5 * (double)r.dy), hdz = uniform(0.5 * (double)r.dz);
    const unsigned nx = (unsigned)g.nx, ny = (unsigned)g.ny, nz = (unsigned)g.nz, nxy = nx * ny;
    const KvRsrc vrs = voxel_rsrc(g, vol);
    // the reference's segment (prev, cur): its weight, 0 if rejected, and
    // its voxel
    auto exact = [&](float prev, float cur, float &w, float &val) {
        const double sum = (double)(cur + prev);
        const int vx = (int)__builtin_fma(sum, hdx, bx);
        const int vy = (int)__builtin_fma(sum, hdy, by);
        const int vz = (int)__builtin_fma(sum, hdz, bz);
        const float d = cur - prev;
        const bool ok = (unsigned)vx < nx && (unsigned)vy < ny && (unsigned)vz < nz && d > 1e-6f;
        const unsigned k = mad_u24((unsigned)vz, nxy, mad_u24((unsigned)vy, nx, (unsigned)vx));
        val = kv_struct_load_f32(vrs, (int)k, 0, 0, 0);
        w = ok ? d : 0.f;
    };
    auto add = [&](float w, float val) {
        tw = tw + w;
        tot = tot + kv_mul_legacy(w, val);
    };
    auto one = [&](float prev, float cur) {
        float w, val;
        exact(prev, cur, w, val);
        add(w, val);
    };
    auto pass = [&](bool c) {
        const float nv = l.hx + l.inc;
        l.hx = c ? (nv > l.tx ? kInf : nv) : l.hx;
        l.at += c ? l.dat : 0;
    };
    // entries of the x run below `lim`, from the entry prev on
    auto entries = [&](float &prev, float lim) {
        while (__any(l.hx < lim)) {
            const bool c = l.hx < lim;
            const float cur = c ? l.hx : prev;
            one(prev, cur);
            prev = cur;
            pass(c);
        }
    };
    const int segs = hp->segs;
    float a = hp->a;
    if (__any(l.hx < a)) {
        // ahead of the list: the x run's head is the first entry
        float prev = minf(l.hx, a);
        pass(l.hx < a);
        entries(prev, a);
        one(prev, a);
    }
    const int lane = (int)(threadIdx.x & 63);
    const int first = __builtin_ctzll(in), last = 63 - __builtin_clzll(in);
    KvRsrc rs = vrs;
    rs.z = g.nx;  // one row's voxels: the row is the scalar offset
    KvSegBlockR q, nq, mq;
    auto read = [&](KvSegBlockR &d) {
        d = *(KvSegBlockRC *)sp;
        sp += SEG_DEPTH;
    };
    auto arrived = [](KvSegBlockR &d) { asm volatile("" : "+s"(d)); };
    float ra[SEG_DEPTH], rb[SEG_DEPTH];
    auto rows = [&](const KvSegBlockR &d, float (&row)[SEG_DEPTH]) {
        const int j0 = __builtin_amdgcn_readlane(l.at, first) >> 2, j1 = __builtin_amdgcn_readlane(l.at, last) >> 2;
        const int base = min(j0, j1) - 1 - below, width = max(j0, j1) + 2 + above - base;
        const int of = (lane - base) & 63;
        const int i = of < width ? base + of : -1;
#pragma unroll
        for (int k = 0; k < SEG_DEPTH; ++k)
            row[k] = kv_struct_load_f32(rs, i, 0, (int)(d[4 * k + 1] & ~1u), 0);
    };
    auto walk = [&](const KvSegBlockR &d, const float (&row)[SEG_DEPTH]) {
        float w1[SEG_DEPTH], w2[SEG_DEPTH], v1[SEG_DEPTH], v2[SEG_DEPTH];
#pragma unroll
        for (int k = 0; k < SEG_DEPTH; ++k) {
            const float b = __uint_as_float(d[4 * k]), off = fabsf(l.hx - __uint_as_float(d[4 * k + 2])),
                        r = __uint_as_float(d[4 * k + 3]);
            const unsigned long long flag = d[4 * k + 1] & 1u;
            // (one ballot per compare: the masks combine on the scalar unit)
            const unsigned long long cross = __builtin_amdgcn_ballot_w64(l.hx < b);
            const unsigned long long close = cross & __builtin_amdgcn_ballot_w64(off > r - l.delta);
            const float h0 = l.hx, x1 = minf(h0, b);
            v1[k] = __int_as_float(__builtin_amdgcn_ds_bpermute(l.at, __float_as_int(row[k])));
            w1[k] = x1 - a;
            w2[k] = b - x1;
            const int at0 = l.at;
            l.hx = selm(cross, h0 + l.inc, h0);
            l.at = at0 + __float_as_int(selm(cross, __int_as_float(l.dat), 0.f));
            v2[k] = __int_as_float(__builtin_amdgcn_ds_bpermute(l.at, __float_as_int(row[k])));
            if (close | flag) {
                // a crossing close to a plane, or a flagged segment
                const float h = h0 > l.tx ? kInf : h0;
                const unsigned long long c = __builtin_amdgcn_ballot_w64(h < b);
                const float y1 = minf(h, b);
                l.hx = selm(c, h + l.inc, h);
                l.at = at0 + __float_as_int(selm(c, __int_as_float(l.dat), 0.f));
                float e1, e2, u1, u2;
                if ((c & __builtin_amdgcn_ballot_w64(off > r)) | flag) {
                    // flagged, or close to a y or z plane.  The gathers are
                    // waited for here: left in flight, they would make the
                    // common path wait too, for the row loads behind them.
                    exact(a, y1, e1, u1);
                    exact(y1, b, e2, u2);
                    asm volatile("" : "+v"(u1), "+v"(u2));
                } else {
                    // close to an x plane: the row is the segment's
                    const int i1 = (int)__builtin_fma((double)(y1 + a), hdx, bx),
                              i2 = (int)__builtin_fma((double)(b + y1), hdx, bx);
                    u1 = __int_as_float(__builtin_amdgcn_ds_bpermute(i1 << 2, __float_as_int(row[k])));
                    u2 = __int_as_float(__builtin_amdgcn_ds_bpermute(i2 << 2, __float_as_int(row[k])));
                    const float d1 = y1 - a, d2 = b - y1;
                    e1 = d1 > 1e-6f ? d1 : 0.f;
                    e2 = d2 > 1e-6f ? d2 : 0.f;
                }
                v1[k] = u1;
                v2[k] = u2;
                w1[k] = e1;
                w2[k] = e2;
            }
            a = b;
        }
#pragma unroll
        for (int k = 0; k < SEG_DEPTH; ++k) {
            add(w1[k], v1[k]);
            add(w2[k], v2[k]);
        }
    };
    read(q);
    read(nq);
    arrived(q);
    arrived(nq);
    rows(q, ra);
    for (int i = 0; i < segs; i += 2 * SEG_DEPTH) {
        rows(nq, rb);
        read(mq);
        __builtin_amdgcn_sched_barrier(0);
        walk(q, ra);
        __builtin_amdgcn_sched_barrier(0);
        arrived(mq);
        if (i + SEG_DEPTH >= segs)
            break;
        rows(mq, ra);
        read(q);
        __builtin_amdgcn_sched_barrier(0);
        walk(nq, rb);
        __builtin_amdgcn_sched_barrier(0);
        arrived(q);
        nq = q;
        q = mq;
    }
    // the rest of the x run, with the fillers' 1.0 in its place
    l.hx = l.hx > l.tx ? kInf : l.hx;
    float prev = hp->end;
    if (hp->filler) {
        entries(prev, 1.f);
        pass(l.hx == 1.f);
        one(prev, 1.f);
        prev = 1.f;
    }
    entries(prev, kInf);
}

// Column u of a row whose p and v are wavefront-uniform, with its epilogue;
// lanes with u >= end are idle.
template <int EP>
__device__ __forceinline__ void fp_r_row(const KvGeom &g, const float *__restrict__ vol, float *__restrict__ out,
                                         const float *__restrict__ data, float relax, int p, int u, int v, int end)
{
    const size_t id = (size_t)p * g.nv + v;
    KvSegHeadRC *hp = (KvSegHeadRC *)(size_t)(g.seg_r_head + id);
    KvSegRC *sp = (KvSegRC *)(size_t)(g.seg_r + id * (size_t)g.seg_stride);
    const bool inside = u < end;
    const size_t o = id * g.nu + u;
    u = inside ? u : end - 1;
    if (hp->empty) {
        if (inside)
            fp_r_store<EP>(0.f, out, data, relax, o);
        return;
    }
    RayF r;
    ray_setup(g, p, u, v, r);
    const float xlo = fminf(r.a1x, r.aNx), xhi = fmaxf(r.a1x, r.aNx);
    const float amin = hp->amin, amax = hp->amax;
    // the reference's early exit: the ray's value is 0
    const bool live = inside && !fsupeq(fmaxf(amin, xlo), fminf(amax, xhi), 1e-7f);
    LaneR l;
    l.inc = fabsf(r.ivx);
    int lox, hix;
    axis_range(r.dx, r.sx, r.hx, g.nx, amin, amax, lox, hix);
    const int cx = hix - lox + 1;
    l.delta = fmaxf(2.f * (g.rc[KV_RC * p + 10] * l.inc + 6.e-8f * (3.2f + 0.5f * (float)cx)), 1.2e-6f);
    // the lanes that can follow the list: no x face in the row's alpha range
    // (x_face_room), x planes farther apart than the segments' ends, and a
    // rounding bound within the builder's
    const float room = x_face_room(r.hx, r.sx, g.nx, l.inc);
    const bool mine = live && xlo + room <= amin && xhi - room >= amax && l.inc > hp->longest + 2.f * l.delta &&
                      l.delta <= g.seg_delta && hp->segs >= 0;
    const unsigned long long in = __builtin_amdgcn_ballot_w64(mine);
    float tot = 0.f, tw = 0.f;
    bool done = !live;
    if (in != 0) {
        // distance of the lanes in voxels, as in row_sums
        const float df = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.dx), __builtin_ctzll(in))),
                    dl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.dx), 63 - __builtin_clzll(in)));
        const float most = fmaxf(fabsf(df), fabsf(dl));
        const int ahead = (int)fminf(most * hp->longest * (2.f * SEG_DEPTH), 64.f) + 2;
        const int below = __builtin_amdgcn_readfirstlane(__any(mine && r.dx < 0.f) ? ahead : 0),
                  above = __builtin_amdgcn_readfirstlane(__any(mine && r.dx > 0.f) ? ahead : 0);
        if (hp->end * fabsf(dl - df) + 4.f + (float)(below + above) <= 63.f && most + fabsf(r.sx) < 65536.f) {
            l.hx = mine ? r.ivx * (-r.hx - r.sx + (float)(r.dx > 0 ? lox : hix)) : kInf;
            l.tx = __builtin_fmaf((float)cx - 0.5f, l.inc, l.hx);
            l.at = (r.dx > 0 ? lox - 1 : hix) * 4;
            l.dat = r.dx > 0 ? 4 : -4;
            seg_sums_r(g, vol, r, hp, sp, in, below, above, l, tot, tw);
            done = done || mine;
        }
    }
    if (inside && done)
        fp_r_store<EP>(mine && tw > 1e-6f ? tot / tw : 0.f, out, data, relax, o);
    if (inside && !done)
        fp_r_ray<EP>(g, vol, out, data, relax, p, u, v);
}

// The mode-R segment list of one (view, detector row) per thread: the merge
// of walk_r's y and z runs for rays whose alpha range the x faces leave
// alone.
__global__ __launch_bounds__(64) void seg_r_kernel(KvGeom g, KvSegR *__restrict__ seg, KvSegHeadR *__restrict__ head)
{
    const int id = blockIdx.x * 64 + threadIdx.x;
    if (id >= g.np * g.nv)
        return;
    const int p = id / g.nv, v = id - p * g.nv;
    RayF r;
    ray_setup(g, p, 0, v, r);
    KvSegHeadR H{};
    const float amin = fmaxf(0.f, fmaxf(fminf(r.a1y, r.aNy), fminf(r.a1z, r.aNz)));
    const float amax = fminf(1.f, fminf(fmaxf(r.a1y, r.aNy), fmaxf(r.a1z, r.aNz)));
    H.amin = amin;
    H.amax = amax;
    // taking the x faces in only raises amin and lowers amax
    H.empty = fsupeq(amin, amax, 1e-7f) ? 1 : 0;
    if (H.empty) {
        head[id] = H;
        return;
    }
    int loy, hiy, loz, hiz;
    axis_range(r.dy, r.sy, r.hy, g.ny, amin, amax, loy, hiy);
    axis_range(r.dz, r.sz, r.hz, g.nz, amin, amax, loz, hiz);
    // |d| > 1e-6 on both axes: else the face alphas are 0 and the row empty
    float ay = r.ivy * (-r.hy - r.sy + (float)(r.dy > 0 ? loy : hiy));
    float az = r.stz * (-r.hz - r.sz + (float)(r.dz > 0 ? loz : hiz));
    const float iy = fabsf(r.ivy), iz = fabsf(r.stz);
    const int dzr = hiz - loz;
    int cy = hiy - loy + 1, cz = dzr >= 2 ? dzr - 1 : 1;
    H.filler = dzr + 1 - cz > 0 ? 1 : 0;
    const double by = (double)(r.hy + r.sy), bz = (double)(r.hz + r.sz);
    const double hdy = 0.5 * (double)r.dy, hdz = 0.5 * (double)r.dz;
    const float delta = g.seg_delta;
    KvSegR *out = seg + (size_t)id * g.seg_stride;
    const int cap = g.seg_stride - KV_SEG_PAD;
    float a = fminf(ay, az), longest = 0.f;
    H.a = a;
    unsigned row = 0;
    int m = 0;
    bool whole = true;
    auto next = [&](float cur) {
        if (cy > 0 && ay == cur) {
            --cy;
            ay = cy > 0 ? ay + iy : kInf;
        }
        if (cz > 0 && az == cur) {
            --cz;
            az = cz > 0 ? az + iz : kInf;
        }
    };
    next(a);
    while (cy > 0 || cz > 0) {
        const float b = fminf(ay, az);
        if (m >= cap) {
            whole = false;
            break;
        }
        const double sum = (double)(b + a);
        const double py = __builtin_fma(sum, hdy, by), pz = __builtin_fma(sum, hdz, bz);
        const int vy = (int)py, vz = (int)pz;
        const float w = b - a;
        const double mid = 0.5 * sum, margin = 4e-5;
        const bool good = (unsigned)vy < (unsigned)g.ny && (unsigned)vz < (unsigned)g.nz && w > 1e-6f && w > delta &&
                          py >= 0.0 && pz >= 0.0 && mid >= (double)amin + margin && mid <= (double)amax - margin;
        KvSegR e{b, row | 1u, 0.f, -kInf};
        if (good) {
            row = (((unsigned)vz * (unsigned)g.ny + (unsigned)vy) * (unsigned)g.nx) * 4u;
            // sums between which the midpoint stays in row (vy, vz), in from
            // the FP32 rounding of a sum below 2
            const double y0 = ((double)vy - by) / hdy, y1 = ((double)(vy + 1) - by) / hdy;
            const double z0 = ((double)vz - bz) / hdz, z1 = ((double)(vz + 1) - bz) / hdz;
            const double lo = fmax(fmin(y0, y1), fmin(z0, z1)) + 2e-7, hi = fmin(fmax(y0, y1), fmax(z0, z1)) - 2e-7;
            // a crossing within 1e-6 of a or b cuts off a segment that is
            // rejected wherever it lies
            double A = fmax(fmax((double)a, (double)amin + margin), lo - (double)a);
            double B = fmin(fmin((double)b, (double)amax - margin), hi - (double)b);
            A = A - (double)a <= 9.9e-7 ? (double)a : A;
            B = (double)b - B <= 9.9e-7 ? (double)b : B;
            e.row = row;
            e.m = (float)(0.5 * (A + B));
            e.r = (float)(0.5 * (B - A) - 2e-7);
        }
        out[m++] = e;
        longest = fmaxf(longest, w);
        a = b;
        next(b);
    }
    // entries at or above the fillers' 1.0 are left to walk_r
    if (!(a < 0.999f) || !(H.a > 0.f))
        whole = false;
    H.end = a;
    H.longest = longest;
    H.segs = whole ? m : -1;
    // empty segments: a crossing x run entry is impossible (c < a), flagged
    // or not
    for (int k = 0; whole && k < KV_SEG_PAD; ++k)
        out[m + k] = KvSegR{a, row, 0.f, kInf};
    head[id] = H;
}

// Length in mm of a ray from the source to its pixel, as ray_setup_a.
__device__ __forceinline__ float ray_length(const KvGeom &g, int p, int u, int v)
{
    RayF f;
    ray_setup(g, p, u, v, f);
    const float lx = f.dx * g.sx, ly = f.dy * g.sy, lz = f.dz * g.sz;
    return sqrtf(lx * lx + ly * ly + lz * lz);
}

// Epilogue of the mode-A forward pass for the line integral ax of a ray.
template <int EP>
__device__ __forceinline__ void fp_a_store(const KvGeom &g, const KvTables &t, float ax, float *__restrict__ out,
                                           const float *__restrict__ data, int p, int u, int v)
{
    const size_t o = ((size_t)p * g.nv + v) * g.nu + u;
    if (EP == KV_EP_PLAIN) {
        out[o] = ax;
    } else {
        // MLEM ratio on line-integral data, stored premultiplied by the
        // ray's length factor as the mode-A backprojector weighs it (its
        // tables' sqrt((lx2 + ly2) + lz2), the same FP32 product it would
        // form per pixel)
        const float L = sqrtf((t.lx2[(size_t)p * g.nu + u] + t.ly2[(size_t)p * g.nv + v]) + t.lz2[p]);
        out[o] = ax > 0.f ? L * (data[o] / ax) : 0.f;
    }
}

// One ray of the mode-A forward pass with its epilogue.
template <int EP>
__device__ __forceinline__ void fp_a_ray(const KvGeom &g, const KvTables &t, const float *__restrict__ vol,
                                         float *__restrict__ out, const float *__restrict__ data, int p, int u, int v)
{
    RayA r;
    ray_setup_a(g, p, u, v, r);
    const size_t o = ((size_t)p * g.nv + v) * g.nu + u;
    if (EP == KV_EP_COUNT) {
        int c = 0;
        walk_a(r, [&](bool ok, unsigned, float) { c += ok; });
        out[o] = (float)c;
        return;
    }
    AccA a;
    a.init(g, vol);
    walk_a(r, [&](bool ok, unsigned k, float len) { a.visit(ok, k, len); });
    fp_a_store<EP>(g, t, r.L * a.sum(), out, data, p, u, v);
}

// The same for column u of a row whose p and v are wavefront-uniform, along
// the row's segment list.
template <int EP>
__device__ __forceinline__ void fp_a_row(const KvGeom &g, const KvTables &t, const float *__restrict__ vol,
                                         float *__restrict__ out, const float *__restrict__ data, int p, int u, int v)
{
    const bool live = u < g.nu;
    u = live ? u : g.nu - 1;
    float sum;
    const float *vols[1] = {vol};
    row_sums<1>(g, vols, p, u, v, &sum);
    if (live)
        fp_a_store<EP>(g, t, ray_length(g, p, u, v) * sum, out, data, p, u, v);
}

template <int EP>
__global__ __launch_bounds__(256) void fp_a_kernel(KvGeom g, KvTables t, const float *__restrict__ vol,
                                                   float *__restrict__ out, const float *__restrict__ data, KvFpMap fm)
{
    int tx, ty, p, u, v;
    fp_xcd_tile(fm, blockIdx.x, tx, ty, p);
    fp_tile_pixel(fm.layout, tx, ty, threadIdx.x, u, v);
    if (u >= g.nu || v >= g.nv)
        return;
    fp_a_ray<EP>(g, t, vol, out, data, p, u, v);
}

// Pixel of this lane in the row-by-row walks, whose tiles are 64 columns by 4
// rows, one row per wavefront: the row is wavefront-uniform (a scalar).  The
// launch order's tx counts KV_ROW_CY tiles of consecutive rows per column, so
// that a chunk's workgroups follow each other on one XCD.
__device__ __forceinline__ void fp_row_pixel(int tx, int ty, int &u, int &v)
{
    u = tx / KV_ROW_CY * 64 + (int)(threadIdx.x & 63);
    v = (ty * KV_ROW_CY + tx % KV_ROW_CY) * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

template <int EP>
__global__ __launch_bounds__(256) void fp_a_row_kernel(KvGeom g, KvTables t, const float *__restrict__ vol,
                                                       float *__restrict__ out, const float *__restrict__ data,
                                                       KvFpMap fm)
{
    int tx, ty, p, u, v;
    fp_xcd_tile(fm, blockIdx.x, tx, ty, p);
    fp_row_pixel(tx, ty, u, v);
    if (v < g.nv && __any(u < g.nu))
        fp_a_row<EP>(g, t, vol, out, data, p, u, v);
}

// Columns of view p whose rays run row by row: [first, end).
__device__ __forceinline__ void row_columns(const KvGeom &g, int p, int &first, int &end)
{
    const float *c = g.rc + KV_RC * p;
    first = __float_as_int(c[11]);
    end = __float_as_int(c[12]);
}

// Pixel of this lane in tile (tx, ty) of the other columns, in 8x8 tiles as
// fp_tile_pixel's: those left of the interval, then those right of it;
// u >= g.nu where there is none.
__device__ __forceinline__ void fp_edge_pixel(const KvGeom &g, int tx, int ty, int p, int &u, int &v)
{
    int first, end;
    row_columns(g, p, first, end);
    fp_tile_pixel(KV_FP_LAYOUT, tx, ty, threadIdx.x, u, v);
    u = u < first ? u : end + (u - first);
}

// The first `row_blocks` workgroups take the row-by-row tiles (map rm), the
// others the tiles of the remaining columns (map em).
template <int EP>
__global__ __launch_bounds__(256, 7) void fp_r_row_kernel(KvGeom g, const float *__restrict__ vol,
                                                          float *__restrict__ out, const float *__restrict__ data,
                                                          float relax, KvFpMap rm, KvFpMap em, unsigned row_blocks)
{
    int tx, ty, p, u, v;
    if (blockIdx.x < row_blocks) {
        int first, end;
        fp_xcd_tile(rm, blockIdx.x, tx, ty, p);
        fp_row_pixel(tx, ty, u, v);
        row_columns(g, p, first, end);
        u += first;
        if (v < g.nv && __any(u < end))
            fp_r_row<EP>(g, vol, out, data, relax, p, u, v, end);
        return;
    }
    fp_xcd_tile(em, blockIdx.x - row_blocks, tx, ty, p);
    fp_edge_pixel(g, tx, ty, p, u, v);
    if (u < g.nu && v < g.nv)
        fp_r_ray<EP>(g, vol, out, data, relax, p, u, v);
}

// Mode-A forward projections of NV <= 3 volumes in one walk per ray: one
// volume gathered as fp_a_ray does, two or three interleaved per voxel
// (pack_kernel: records of 2 or 4 floats) so that one gather per step reads
// them all.  Each volume's sum takes the same products and additions in the
// same order as fp_a_ray, so every projection is bit-identical to a
// single-volume pass.
struct KvMulti {
    const float *vol[KV_LL_MAX];
    float *out[KV_LL_MAX];
};

// The sums of a walk over NV = 2 or 3 interleaved volumes, as AccA's.
template <int NV>
struct AccPack {
    static constexpr int W = NV == 2 ? 2 : 4;  // floats per record
    KvRsrc rs;
    float acc[NV], pv[NV];
    float pw = 0.f;
    __device__ __forceinline__ void init(const KvGeom &g, const float *pack)
    {
        rs = voxel_rsrc(g, pack, 4 * W);
#pragma unroll
        for (int i = 0; i < NV; ++i)
            acc[i] = pv[i] = 0.f;
    }
    __device__ __forceinline__ void visit(bool ok, unsigned k, float len)
    {
        float v[NV];
        if constexpr (NV == 2) {
            const KvF32x2 r = kv_struct_load_f32x2(rs, (int)k, 0, 0, 0);
            v[0] = r.x, v[1] = r.y;
        } else {
            const KvF32x4 r = kv_struct_load_f32x4(rs, (int)k, 0, 0, 0);
            v[0] = r.x, v[1] = r.y, v[2] = r.z;
        }
#pragma unroll
        for (int i = 0; i < NV; ++i)
            acc[i] = acc[i] + kv_mul_legacy(pw, pv[i]);
        pw = ok ? len : 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i)
            pv[i] = v[i];
    }
    __device__ __forceinline__ float sum(int i) const { return acc[i] + kv_mul_legacy(pw, pv[i]); }
};

// Volumes m.vol[0..NV) interleaved per voxel: float2 records for two, float4
// records (fourth float 0) for three.
template <int NV>
__global__ __launch_bounds__(256) void pack_kernel(KvMulti m, int64_t n, float *__restrict__ pack)
{
    for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
        if constexpr (NV == 2) {
            const float2 r = make_float2(m.vol[0][v], m.vol[1][v]);
            reinterpret_cast<float2 *>(pack)[v] = r;
        } else {
            const float4 r = make_float4(m.vol[0][v], m.vol[1][v], m.vol[2][v], 0.f);
            reinterpret_cast<float4 *>(pack)[v] = r;
        }
    }
}

template <int NV>
__global__ __launch_bounds__(256) void fp_a_multi_kernel(KvGeom g, const float *__restrict__ pack, KvMulti m,
                                                         KvFpMap fm)
{
    int tx, ty, p, u, v;
    fp_xcd_tile(fm, blockIdx.x, tx, ty, p);
    fp_tile_pixel(fm.layout, tx, ty, threadIdx.x, u, v);
    if (u >= g.nu || v >= g.nv)
        return;
    RayA r;
    ray_setup_a(g, p, u, v, r);
    const size_t o = ((size_t)p * g.nv + v) * g.nu + u;
    if constexpr (NV == 1) {
        AccA a;
        a.init(g, m.vol[0]);
        walk_a(r, [&](bool ok, unsigned k, float len) { a.visit(ok, k, len); });
        m.out[0][o] = r.L * a.sum();
    } else {
        AccPack<NV> a;
        a.init(g, pack);
        walk_a(r, [&](bool ok, unsigned k, float len) { a.visit(ok, k, len); });
#pragma unroll
        for (int i = 0; i < NV; ++i)
            m.out[i][o] = r.L * a.sum(i);
    }
}

// The same along the rows' segment lists: each volume's rows are read as
// they lie (neighbouring voxels of one row are neighbouring lanes), so
// several volumes need no interleaved copy.
template <int NV>
__global__ __launch_bounds__(256) void fp_a_row_multi_kernel(KvGeom g, KvMulti m, KvFpMap fm)
{
    int tx, ty, p, u, v;
    fp_xcd_tile(fm, blockIdx.x, tx, ty, p);
    fp_row_pixel(tx, ty, u, v);
    if (v >= g.nv || !__any(u < g.nu))
        return;
    const bool live = u < g.nu;
    u = live ? u : g.nu - 1;
    float sum[NV];
    row_sums<NV>(g, m.vol, p, u, v, sum);
    if (!live)
        return;
    const float L = ray_length(g, p, u, v);
    const size_t o = ((size_t)p * g.nv + v) * g.nu + u;
#pragma unroll
    for (int i = 0; i < NV; ++i)
        m.out[i][o] = L * sum[i];
}

template <int EP>
__global__ __launch_bounds__(256) void fp_r_batch_kernel(const KvProblem *__restrict__ probs, int nprob,
                                                         long long total, int iteration, float relax)
{
    fp_batch_tiles(probs, nprob, total, iteration, [&](const KvProblem &P, int p, int tx, int ty) {
        int u, v;
        if (P.fp_part == KV_FP_ROWS) {
            int first, end;
            fp_row_pixel(tx, ty, u, v);
            row_columns(P.g, p, first, end);
            u += first;
            if (v < P.g.nv && __any(u < end))
                fp_r_row<EP>(P.g, P.vol, P.ratio, P.data, relax, p, u, v, end);
            return;
        }
        if (P.fp_part == KV_FP_EDGES)
            fp_edge_pixel(P.g, tx, ty, p, u, v);
        else
            fp_tile_pixel(P.fp_layout, tx, ty, threadIdx.x, u, v);
        if (u < P.g.nu && v < P.g.nv)
            fp_r_ray<EP>(P.g, P.vol, P.ratio, P.data, relax, p, u, v);
    });
}

// Mode-A forward pass (MLEM ratio) over a batch, as
// fp_r_batch_kernel; reconstructions with segment lists run row by row.
__global__ __launch_bounds__(256) void fp_a_batch_kernel(const KvProblem *__restrict__ probs, int nprob,
                                                         long long total, int iteration)
{
    fp_batch_tiles(probs, nprob, total, iteration, [&](const KvProblem &P, int p, int tx, int ty) {
        int u, v;
        if (P.fp_part == KV_FP_ROWS) {
            fp_row_pixel(tx, ty, u, v);
            if (v < P.g.nv && __any(u < P.g.nu))
                fp_a_row<KV_EP_MLEM>(P.g, P.t, P.vol, P.ratio, P.data, p, u, v);
            return;
        }
        fp_tile_pixel(P.fp_layout, tx, ty, threadIdx.x, u, v);
        if (u < P.g.nu && v < P.g.nv)
            fp_a_ray<KV_EP_MLEM>(P.g, P.t, P.vol, P.ratio, P.data, p, u, v);
    });
}

// Records the accepted pairs of sampled rays through the same walks.
__global__ void trace_kernel(KvGeom g, int mode, int nrays, const int32_t *__restrict__ rays, int cap,
                             int64_t *__restrict__ idx, float *__restrict__ w, int32_t *__restrict__ counts)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nrays)
        return;
    const int id = rays[t];
    const int per = g.nu * g.nv;
    const int p = id / per, rem = id - p * per, v = rem / g.nu, u = rem - v * g.nu;
    int c = 0;
    auto rec = [&](bool ok, unsigned k, float wt) {
        if (!ok)
            return;
        if (c < cap) {
            idx[(size_t)t * cap + c] = (int64_t)k;
            w[(size_t)t * cap + c] = wt;
        }
        ++c;
    };
    if (mode == KV_MODE_R) {
        RayF r;
        ray_setup(g, p, u, v, r);
        walk_r<false>(g, r, rec);
    } else {
        RayA r;
        ray_setup_a(g, p, u, v, r);
        walk_a(r, rec);
    }
    counts[t] = c;
}

}  // namespace

// One-dimensional launches of the single-reconstruction forward kernels over
// gxp x gy tiles per view (fp_xcd_tile), as many views per launch as keep a
// launch within 2^32 threads.
struct FpGrid {
    int gxp, gy, chunk, views;
    KvFpMap fm{};
    // gx x ty tiles of the detector, in stripes of chunk tiles dealt to the
    // XCDs.  Rows of a round of stripes and more are padded to whole rounds;
    // the tiles of shorter ones follow each other in one row per view, since
    // empty workgroups are not free (mode R, 128x128x32 voxels, 15 views of
    // 256x256: 25.0 us padded, 22.3 not; detectors of 127 to 224 columns by
    // 221 to 411: 5 to 25 % of the time).
    FpGrid(int gx, int ty, int chunk_, int np) : chunk(chunk_)
    {
        const int span = KV_XCDS * chunk;
        const long long n = (long long)gx * ty;
        if (gx >= span || n > INT32_MAX - span) {
            gxp = (int)(((long long)gx + span - 1) / span * span);
            gy = ty;
        } else {
            gxp = (int)((n + span - 1) / span * span);
            gy = 1;
            fm.ntx = gx;
            fm.dntx = kv_udiv(gx);
        }
        const unsigned long long per_view = std::max(1ull, (unsigned long long)gxp * (unsigned long long)gy * 256ull);
        views = (int)std::min<unsigned long long>((unsigned long long)np, 0xFFFFFFFFull / per_view);
        fm.chunk = chunk;
        fm.nch = gxp / span;
        fm.gy = gy;
        fm.dchunk = kv_udiv(chunk);
        fm.dnch = kv_udiv(fm.nch);
        fm.dgy = kv_udiv(gy);
    }
    // tiles of a layout over the whole detector
    FpGrid(const KvGeom &g, int layout)
        : FpGrid((g.nu + 64 / layout - 1) / (64 / layout), (g.nv + 4 * layout - 1) / (4 * layout), stripe(64 / layout), g.np)
    {
        fm.layout = layout;
    }
    // the row-by-row walk over the whole detector
    static FpGrid rows(const KvGeom &g)
    {
        return FpGrid(kv_row_tiles_x(g.nu), kv_row_tiles_y(g.nv), KV_ROW_CY, g.np);
    }
    static int stripe(int wu) { return std::max(1, KV_FP_STRIPE / wu); }
    KvFpMap map(int p0) const
    {
        KvFpMap m = fm;
        m.p0 = p0;
        return m;
    }
    // Runs launch(blocks, p0) for each range of views; a view too large for
    // one launch is an invalid configuration.
    template <typename F>
    hipError_t run(const KvGeom &g, F &&launch) const
    {
        if (views < 1)
            return hipErrorInvalidConfiguration;
        for (int p0 = 0; p0 < g.np; p0 += views) {
            const int nv = std::min(views, g.np - p0);
            launch((unsigned)gxp * (unsigned)gy * (unsigned)nv, p0);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess)
                return e;
        }
        return hipSuccess;
    }
};

hipError_t kv_launch_fp_r(const KvGeom &g, const float *vol, float *out, int epilogue, const float *data, float relax,
                          hipStream_t s)
{
    if (g.seg_r && epilogue != KV_EP_COUNT) {
        const FpGrid rg(kv_row_tiles_x(g.row_cols), kv_row_tiles_y(g.nv), KV_ROW_CY, g.np),
            eg(kv_edge_tiles_x(g.edge_cols), kv_edge_tiles_y(g.nv), KV_FP_STRIPE / KV_FP_TILE, g.np);
        // as many views per launch as keep it within 2^32 threads
        const unsigned long long per_view =
            256ull * ((unsigned long long)rg.gxp * (unsigned long long)rg.gy +
                      (unsigned long long)eg.gxp * (unsigned long long)eg.gy);
        const int views = (int)std::min<unsigned long long>((unsigned long long)g.np, 0xFFFFFFFFull / per_view);
        if (views < 1)
            return hipErrorInvalidConfiguration;
        for (int p0 = 0; p0 < g.np; p0 += views) {
            const unsigned n = (unsigned)std::min(views, g.np - p0), rb = (unsigned)rg.gxp * (unsigned)rg.gy * n,
                           nb = rb + (unsigned)eg.gxp * (unsigned)eg.gy * n;
            switch (epilogue) {
            case KV_EP_PLAIN:
                fp_r_row_kernel<KV_EP_PLAIN><<<nb, 256, 0, s>>>(g, vol, out, data, relax, rg.map(p0), eg.map(p0), rb);
                break;
            case KV_EP_MLEM:
                fp_r_row_kernel<KV_EP_MLEM><<<nb, 256, 0, s>>>(g, vol, out, data, relax, rg.map(p0), eg.map(p0), rb);
                break;
            default:
                fp_r_row_kernel<KV_EP_SART><<<nb, 256, 0, s>>>(g, vol, out, data, relax, rg.map(p0), eg.map(p0), rb);
                break;
            }
            if (const hipError_t e = hipGetLastError())
                return e;
        }
        return hipSuccess;
    }
    const int L = KV_FP_LAYOUT;
    const FpGrid fg(g, L);
    return fg.run(g, [&](unsigned nb, int p0) {
        switch (epilogue) {
        case KV_EP_PLAIN:
            fp_r_kernel<KV_EP_PLAIN><<<nb, 256, 0, s>>>(g, vol, out, data, relax, fg.map(p0));
            break;
        case KV_EP_MLEM:
            fp_r_kernel<KV_EP_MLEM><<<nb, 256, 0, s>>>(g, vol, out, data, relax, fg.map(p0));
            break;
        case KV_EP_COUNT:
            fp_r_kernel<KV_EP_COUNT><<<nb, 256, 0, s>>>(g, vol, out, data, relax, fg.map(p0));
            break;
        default:
            fp_r_kernel<KV_EP_SART><<<nb, 256, 0, s>>>(g, vol, out, data, relax, fg.map(p0));
            break;
        }
    });
}

hipError_t kv_launch_fp_a_multi(const KvGeom &g, int n, const float *const *vols, float *pack, float *const *outs,
                                hipStream_t s)
{
    KvMulti m{};
    for (int i = 0; i < n; ++i)
        m.vol[i] = vols[i], m.out[i] = outs[i];
    if (g.seg_a) {
        const FpGrid fg = FpGrid::rows(g);
        return fg.run(g, [&](unsigned nb, int p0) {
            switch (n) {
            case 1: fp_a_row_multi_kernel<1><<<nb, 256, 0, s>>>(g, m, fg.map(p0)); break;
            case 2: fp_a_row_multi_kernel<2><<<nb, 256, 0, s>>>(g, m, fg.map(p0)); break;
            default: fp_a_row_multi_kernel<3><<<nb, 256, 0, s>>>(g, m, fg.map(p0)); break;
            }
        });
    }
    if (n >= 2) {
        const int64_t nvox = (int64_t)g.nx * g.ny * g.nz;
        const unsigned nb = (unsigned)std::max<int64_t>(1, std::min<int64_t>(8192, (nvox + 255) / 256));
        if (n == 2)
            pack_kernel<2><<<nb, 256, 0, s>>>(m, nvox, pack);
        else
            pack_kernel<3><<<nb, 256, 0, s>>>(m, nvox, pack);
        if (hipError_t e = hipGetLastError())
            return e;
    }
    const int L = KV_FP_LAYOUT_MULTI[std::min(std::max(n, 1), KV_LL_MAX) - 1];
    const FpGrid fg(g, L);
    return fg.run(g, [&](unsigned nb, int p0) {
        switch (n) {
        case 1: fp_a_multi_kernel<1><<<nb, 256, 0, s>>>(g, pack, m, fg.map(p0)); break;
        case 2: fp_a_multi_kernel<2><<<nb, 256, 0, s>>>(g, pack, m, fg.map(p0)); break;
        default: fp_a_multi_kernel<3><<<nb, 256, 0, s>>>(g, pack, m, fg.map(p0)); break;
        }
    });
}

hipError_t kv_launch_fp_a(const KvGeom &g, const KvTables &t, const float *vol, float *out, int epilogue,
                          const float *data, hipStream_t s)
{
    if (g.seg_a && epilogue != KV_EP_COUNT) {
        const FpGrid fg = FpGrid::rows(g);
        return fg.run(g, [&](unsigned nb, int p0) {
            if (epilogue == KV_EP_PLAIN)
                fp_a_row_kernel<KV_EP_PLAIN><<<nb, 256, 0, s>>>(g, t, vol, out, data, fg.map(p0));
            else
                fp_a_row_kernel<KV_EP_MLEM><<<nb, 256, 0, s>>>(g, t, vol, out, data, fg.map(p0));
        });
    }
    const int L = KV_FP_LAYOUT;
    const FpGrid fg(g, L);
    return fg.run(g, [&](unsigned nb, int p0) {
        if (epilogue == KV_EP_PLAIN)
            fp_a_kernel<KV_EP_PLAIN><<<nb, 256, 0, s>>>(g, t, vol, out, data, fg.map(p0));
        else if (epilogue == KV_EP_COUNT)
            fp_a_kernel<KV_EP_COUNT><<<nb, 256, 0, s>>>(g, t, vol, out, data, fg.map(p0));
        else
            fp_a_kernel<KV_EP_MLEM><<<nb, 256, 0, s>>>(g, t, vol, out, data, fg.map(p0));
    });
}

hipError_t kv_launch_seg_a(const KvGeom &g, KvSeg *seg, KvSegHead *head, hipStream_t s)
{
    seg_a_kernel<<<(unsigned)(((int64_t)g.np * g.nv + 63) / 64), 64, 0, s>>>(g, seg, head);
    return hipGetLastError();
}

hipError_t kv_launch_seg_r(const KvGeom &g, KvSegR *seg, KvSegHeadR *head, hipStream_t s)
{
    seg_r_kernel<<<(unsigned)(((int64_t)g.np * g.nv + 63) / 64), 64, 0, s>>>(g, seg, head);
    return hipGetLastError();
}

hipError_t kv_launch_trace(const KvGeom &g, int mode, int nrays, const int32_t *rays, int cap, int64_t *idx, float *w,
                           int32_t *counts, hipStream_t s)
{
    trace_kernel<<<(nrays + 63) / 64, 64, 0, s>>>(g, mode, nrays, rays, cap, idx, w, counts);
    return hipGetLastError();
}

hipError_t kv_launch_fp_batch(int mode, const KvProblem *probs, int nprob, long long total, int iteration, float relax,
                              hipStream_t s)
{
    const int grid = (int)std::min<long long>(KV_BATCH_GRID, total * KV_XCDS);
    if (mode == KV_MODE_A)
        fp_a_batch_kernel<<<grid, 256, 0, s>>>(probs, nprob, total, iteration);
    else
        fp_r_batch_kernel<KV_EP_MLEM><<<grid, 256, 0, s>>>(probs, nprob, total, iteration, relax);
    return hipGetLastError();
}
