// Beam-staged forward projectors for gfx950.
//
// A 1024-thread workgroup traces the rays of a detector tile in up to four views that share a principal axis P (the
// horizontal axis, x or y, along which their rays advance fastest) and its direction.  A wavefront takes 16 x 4
// pixels of one view; the tile (BeamShape) is 32 x 8 pixels (Siddon) or 16 x 16 (interpolated) in four views, 32 x 16
// in two or one, 32 x 32 in one (build_forward_records chooses).  Wavefronts without a view, half of them where a
// 32 x 16 tile has one view, only copy.
// The rays form a thin beam.  The workgroup sweeps the volume along P in slabs of a few planes; for
// each slab it copies the box of voxels the beam crosses into LDS (16-byte
// loads of rows of a re-laid-out copy of the volume), and every ray walks its
// voxels inside the slab from LDS.  The gathers of
// the walk thus never reach the texture/L1 path, which bounds a gather-driven
// walk; the slab copies are coalesced and are shared by the 1024 rays.
//
// The staging copy ("stage") of the volume is [p][z][a], a = the other
// horizontal axis fastest, with a zero border: p in -1 .. nP + 1, z in -1 ..
// nz, a in -4 .. round_up(nA, 4) + 3.  Every voxel a walk can reach (indices
// -1 .. n) therefore exists, rows start on 16-byte boundaries, and so does the
// upper interpolation tap of a sample clamped to the far face (index n + 1:
// row nz + 1 of plane p is row -1 of plane p + 1, and the extra zero plane
// nP + 1 ends the copy), as do the whole rows of the last plane a slab box
// copies.
//
// Planning: every wavefront evaluates the 16 corner rays of the tile (four
// corners in each view) and computes the box origins of a share of the slabs (Siddon skips the slabs
// before and after the volume);
// the box extents, maxed over the slabs, are the same for the whole sweep, so
// a ray's LDS offset carries from one slab to the next by a uniform shift.
// Slabs are double-buffered: slab s + 1 streams into LDS by direct
// global-to-LDS loads while the rays walk slab s, and one barrier ends each
// slab.  A tile whose box does not fit the LDS buffer even with one plane per
// slab walks the staging copy in global memory instead (same arithmetic).
#include <cmath>

#include "common.hpp"
#include "ray.hpp"

namespace tigre {

namespace {

constexpr int kBeamThreads = 1024;
constexpr int kSlabCap = 9216;      // floats per LDS slab buffer (two per workgroup)
constexpr int kSlabPlanesMax = 8;   // principal planes per slab, at most (the tunable limit is <= this)

// Minimum / maximum over lanes 0..15 (the 16 corner rays; the other rows of
// the wavefront hold copies), by four DPP row shifts, returned as a uniform.
template <int kCtrl>
__device__ __forceinline__ float row_shr(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(x), __float_as_int(x), kCtrl, 0xF, 0xF, false));
}
__device__ __forceinline__ float corner_min(float x) {
    x = fminf(x, row_shr<0x111>(x));
    x = fminf(x, row_shr<0x112>(x));
    x = fminf(x, row_shr<0x114>(x));
    x = fminf(x, row_shr<0x118>(x));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 15));
}
__device__ __forceinline__ float corner_max(float x) {
    x = fmaxf(x, row_shr<0x111>(x));
    x = fmaxf(x, row_shr<0x112>(x));
    x = fmaxf(x, row_shr<0x114>(x));
    x = fmaxf(x, row_shr<0x118>(x));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 15));
}

// Extent of the beam over principal planes lo .. hi: the beam's lines are
// A(p) = cA + kA p, z(p) = cz + kz p (corner ray c in lane c; the other rows of
// the wavefront hold copies), the voxels of the planes span P coordinates
// [lo, hi + 1], and a margin of one voxel covers rounding; `tap` = 1 adds the
// upper interpolation tap.  Clipped to -1 .. n + tap (no walk or tap leaves
// it: a sample clamped to the face n reads the zero tap n + 1 with weight 0);
// a0 is aligned down to 4 for 16-byte rows.
// `rim`: a line may leave the volume in the planes; `out`: all of them stay outside it (a 64th of a voxel
// covers the rounding of the lines).
struct BoxExtent {
    int a0, a1, z0, z1;
    bool rim, out;
};
__device__ inline BoxExtent beam_extent(int lo, int hi, float cA, float kA, float cz, float kz, int nA, int nz,
                                        int tap) {
    const float p0 = (float)lo, p1 = (float)(hi + 1);
    const float A0 = fmaf(kA, p0, cA), A1 = fmaf(kA, p1, cA);
    const float Z0 = fmaf(kz, p0, cz), Z1 = fmaf(kz, p1, cz);
    float amin = corner_min(fminf(A0, A1)), amax = corner_max(fmaxf(A0, A1));
    float zmin = corner_min(fminf(Z0, Z1)), zmax = corner_max(fmaxf(Z0, Z1));
    constexpr float kTol = 1.0f / 64.0f;
    BoxExtent e;
    e.rim = amin < kTol || amax > (float)nA - kTol || zmin < kTol || zmax > (float)nz - kTol;
    e.out = amax < -kTol || amin > (float)nA + kTol || zmax < -kTol || zmin > (float)nz + kTol;
    amin = fminf(fmaxf(amin, -2.0f), (float)nA + 1.0f);
    amax = fminf(fmaxf(amax, -2.0f), (float)nA + 1.0f);
    zmin = fminf(fmaxf(zmin, -2.0f), (float)nz + 1.0f);
    zmax = fminf(fmaxf(zmax, -2.0f), (float)nz + 1.0f);
    e.a0 = max((int)floorf(amin) - 1, -1) & ~3;
    e.a1 = min((int)floorf(amax) + 1 + tap, nA + tap);
    e.z0 = max((int)floorf(zmin) - 1, -1);
    e.z1 = min((int)floorf(zmax) + 1 + tap, nz + tap);
    return e;
}

// Slab s of a sweep with `planes` planes per slab along direction dir over
// principal indices -1 .. nP.
__device__ __forceinline__ void slab_range(int s, int planes, int dir, int nP, int& lo, int& hi) {
    if (dir > 0) {
        lo = -1 + s * planes;
        hi = min(lo + planes - 1, nP);
    } else {
        hi = nP - s * planes;
        lo = max(hi - planes + 1, -1);
    }
}

struct StageGeom {
    int NZ, NA;  // bordered extents of the staging copy (z, a)
};

__device__ __forceinline__ unsigned long long stage_index(const StageGeom& s, int p, int z, int a) {
    return ((unsigned long long)(p + 1) * (unsigned)s.NZ + (unsigned)(z + 1)) * (unsigned)s.NA + (unsigned)(a + 4);
}

// Per-ray Siddon state (Siddon_projection.cu:110-268 restated: exact path
// through the voxel grid, crossings taken in increasing parameter order).
// The crossing counts k per axis give the next crossing on each axis,
// t0 + k dt (recomputed exactly, never accumulated).
struct RayWalk {
    float tx, ty, tz, t0x, t0y, t0z, dtx, dty, dtz;
    float kx, ky, kz;      // crossings so far per axis (exact small integers)
    unsigned off;          // voxel offset in the current source (LDS box or staging copy)
    unsigned dX, dY, dZ;   // offset steps of one crossing on each axis
    int kexit;             // principal crossing count at which the ray leaves the slab
    float T, tc, sum;
};

// Walks crossings until the ray leaves the volume (returns true) or its
// principal crossing count reaches kexit (returns false).  Voxel reads are
// at offset (off + slot) from `base`, in bytes for the LDS slabs (base is the
// shared buffer, a constant address folded into the load; slot selects the
// half of the double buffer) and in elements for the staging copy in global
// memory.  The axis of each crossing is selected without branches, the
// principal axis P first on ties, then the other horizontal axis A, then z;
// every step reads one voxel, issued one step before its value is needed;
// the steps are unrolled four to a guard count.
// Leaving the slab and leaving the volume are one test, tm >= Te with
// Te = min(T, time of the slab's last principal crossing): that time is the
// same fma as the crossing's own, and P wins ties, so the test can only
// pass on the principal crossing itself (or at the volume's exit).  Segments
// end at the crossing times themselves: at a slab's exit the crossing time is
// Te exactly, and the volume's exit T is itself a crossing, whose computed
// time differs from T by rounding only (a ray that stops short of it reads
// the zero border for its next segment), so no segment is clamped to Te.
template <int kP, bool kLds>
__device__ inline bool walk(RayWalk& r, const float* __restrict__ base, unsigned slot, int guard) {
    // locals only, named by role (P principal, A other horizontal, z): a
    // conditional between struct members would be compiled as a select of
    // their addresses and force the struct into scratch memory
    float tp = kP == 0 ? r.tx : r.ty, ta = kP == 0 ? r.ty : r.tx, tz = r.tz;
    float kp = kP == 0 ? r.kx : r.ky, ka = kP == 0 ? r.ky : r.kx, kz = r.kz;
    const float t0p = kP == 0 ? r.t0x : r.t0y, t0a = kP == 0 ? r.t0y : r.t0x, t0z = r.t0z;
    const float dtp = kP == 0 ? r.dtx : r.dty, dta = kP == 0 ? r.dty : r.dtx, dtz = r.dtz;
    // LDS: byte offsets; global staging copy: element offsets (its byte offsets can pass 2^32)
    constexpr int kSh = kLds ? 2 : 0;
    const unsigned dP = (kP == 0 ? r.dX : r.dY) << kSh, dA = (kP == 0 ? r.dY : r.dX) << kSh, dZ = r.dZ << kSh;
    unsigned off = (r.off + slot) << kSh;
    float tc = r.tc, sum = r.sum;
    const float T = r.T;
    const float Te = r.kexit >= 1 ? fminf(T, fmaf((float)(r.kexit - 1), dtp, t0p)) : T;
    auto read = [&](unsigned o) {
        return kLds ? *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + o) : base[o];
    };
    float tm = tc;
    float va = read(off), vb = 0.0f;
#define TIGRE_BEAM_STEP(CUR, NEXT)                                       \
    {                                                                    \
        tm = fminf(tp, fminf(ta, tz));                                   \
        sum = fmaf(tm - tc, CUR, sum);                                   \
        tc = tm;                                                         \
        const bool bp = tp == tm, ba = ta == tm;                         \
        kp += bp ? 1.0f : 0.0f;                                          \
        ka += (ba && !bp) ? 1.0f : 0.0f;                                 \
        kz += (bp || ba) ? 0.0f : 1.0f;                                  \
        off += bp ? dP : (ba ? dA : dZ);                                 \
        tp = fmaf(kp, dtp, t0p);                                         \
        ta = fmaf(ka, dta, t0a);                                         \
        tz = fmaf(kz, dtz, t0z);                                         \
        if (tm >= Te) break;                                             \
        NEXT = read(off);                                                \
    }
    for (; guard > 0; --guard) {
        TIGRE_BEAM_STEP(va, vb)
        TIGRE_BEAM_STEP(vb, va)
        TIGRE_BEAM_STEP(va, vb)
        TIGRE_BEAM_STEP(vb, va)
    }
#undef TIGRE_BEAM_STEP
    r.tx = kP == 0 ? tp : ta;
    r.ty = kP == 0 ? ta : tp;
    r.tz = tz;
    r.kx = kP == 0 ? kp : ka;
    r.ky = kP == 0 ? ka : kp;
    r.kz = kz;
    r.off = (off >> kSh) - slot;
    r.tc = tc;
    r.sum = sum;
    return tm >= T;
}

// Plane walk of the Siddon projector: one principal cell (one plane of voxels) per step.
//
// Along the sweep a ray advances one voxel in P per step and at most one voxel in A and in z (slopes
// below 1), so a cell holds at most two crossings and three segments.  A and z are taken in mirrored
// indices that increase along the sweep and in fixed point with 32 fraction bits, A(s) = A0 + s kA, s counted in
// cells from cell -1.  In the cell the ray enters at fraction f of an A voxel it crosses the next A plane
// at the fraction tA = min((1 - f) / kA, 1) of the cell, and likewise in z; 1 - f is what the cell carries (rounded to
// FP32 near 1, f would lose a crossing that is near: 2^-24 voxel, a whole cell at a slope of 6e-8).  With t1 <= t2 the two
// sorted, the cell adds
//     t1 v0 + (t2 - t1) v1 + (1 - t2) v2,
// v0 the entry voxel, v1 the one past the first crossing, v2 the exit voxel.  Whether an axis crosses is the
// borrow of the rest's subtraction, so voxel and position cannot part, a voxel that is not crossed is
// not read.  The cells of each eight are summed by themselves first: adding the same voxel value again and again
// rounds the same way each time, and one sum over 1024 cells was off by 2.6e-6 on a phantom of constant regions
// (rel-L2 at 1024^3; 3.7e-7 in eights).  Slabs have 8, 4, 2 or 1 cells and start at multiples of that, so the sums do not
// depend on how a sweep is cut.  The slope in 32 bits puts a ray
// at most 2^-33 voxel a cell off its line (1e-7 after 1024 cells), which moves a crossing by that over the slope; an FP32
// crossing time is off by 3e-5 cells there.  Rays with a smaller slope than flat_slope() on an axis that they move on
// therefore take the crossing walk.  Off by, here and there (rms over rays that cross one plane, random voxels): 64
// cells, slope 2^-12: 1.5e-7, 1.7e-7; 256, 2^-13: 2.7e-7, 3.0e-7; 1024, 2^-14: 5.4e-7, 7.1e-7; 64, 2^-14: 5.9e-7, 1.8e-7.
//
// The step has no branch and no division, about 20 VALU instructions and (planes at a constant LDS stride, so
// the plane is an immediate of the read) three LDS reads, all lanes in step; the crossing walk above takes
// one crossing per step, about 17 instructions each, 1.6 times a cell on average, and its lanes leave a slab
// at different steps.  It stays for rays with a slope of 1 or more (detector tiles that look across the 45
// degree diagonal, about 4 % of them at a fan angle of 15 degrees) and for the flat ones (a pixel row or column about
// the central one, where pixels are smaller than about 2^-12 of the source's distance).
//
// Measured at 512^3 voxels, 512^2 pixels, 360 views: 25.8 ms, 36.5 ms with the crossing walk alone; 23.5 VALU
// instructions per ray and plane (33.8 before), 3.4 cycles each (most pairs of an FMA and another operation
// issue together), and 5.7 TB/s of copies.  The second walk for infinite voxels and the flat rays' walk are 2 %
// of it.  What is scalar or serial in the slab loop counts as much: with the slabs' addresses formed in the loop
// instead of read from a table the same walk took 30.5 ms.  Two rays per lane with half the wavefronts moved 40 %
// less and were slower (33 ms).
struct PlaneRay {
    unsigned long long A0, z0;  // mirrored A and z at the start of cell -1, 2^-32 voxel
    unsigned kA, kz;            // slopes, 2^-32 voxel
    float iA, iz;               // their reciprocals, in cells per 2^-32 voxel
    int dA, dZ;                 // offset step of one (mirrored) index on A (1 or -1) and on z (row steps)
    unsigned off;               // voxel offset in the current source, as in RayWalk
    float sum, part;            // of the whole eights of cells so far, of the cells since
};

// Smallest slope of the plane walk over nP planes: where it is as exact as the crossing walk, whose times round to
// nP 2^-24 cells.
__device__ __forceinline__ float flat_slope(int nP) { return fmaxf(0x1p-9f / sqrtf((float)nP), 0x1p-6f / (float)nP); }

// Mirrored position and slope on one axis of the line s0 + r a, from the start of cell -1, which the
// sweep enters at parameter a0 and leaves da later; a ray parallel to the axis stays inside its voxel,
// or on the border that it is next to (the other one need not lie in the box).
__device__ __forceinline__ void plane_axis(double s0, double r, double a0, double da, int n, unsigned long long& x0,
                                           unsigned& k, float& ik, int& step) {
    double x = s0 + r * a0, slope = r * da;
    step = 1;
    if (r == 0.0) x = s0 <= 0.0 ? -1.0 : s0 >= (double)n ? (double)n : floor(s0) + 0.5;
    if (slope < 0.0) {
        x = (double)n - x;
        slope = -slope;
        step = -1;
    }
    const double f = floor(x);
    x0 = ((unsigned long long)(long long)f << 32) + (unsigned long long)((x - f) * 4294967296.0);
    k = (unsigned)rint(slope * 4294967296.0);
    ik = k != 0u ? (float)(0x1p-32 / slope) : 1e20f;
}

// Offset of the voxel of a ray at the start of cell `first`, in a box of origin (a0, z0) and row length na;
// positions outside the volume are taken on the border (-1 or n).
__device__ __forceinline__ unsigned plane_offset(const PlaneRay& r, int first, int a0, int z0, int na, int nA, int nz) {
    const int iA = min(max((int)((r.A0 + (unsigned long long)r.kA * (unsigned)first) >> 32), -1), nA);
    const int iz = min(max((int)((r.z0 + (unsigned long long)r.kz * (unsigned)first) >> 32), -1), nz);
    const int a = r.dA > 0 ? iA : nA - 1 - iA, z = r.dZ > 0 ? iz : nz - 1 - iz;
    return (unsigned)((z - z0) * na + (a - a0));
}

// Whether a ray is in the volume in cells first .. first + count - 1: 0 outside in all of them, 2 never
// further out than the border, 1 else.
__device__ __forceinline__ int plane_range(const PlaneRay& r, int first, int count, int nA, int nz) {
    const unsigned long long xA = r.A0 + (unsigned long long)r.kA * (unsigned)first;
    const unsigned long long xz = r.z0 + (unsigned long long)r.kz * (unsigned)first;
    const int sA = (int)(xA >> 32), eA = (int)((xA + (unsigned long long)r.kA * (unsigned)count) >> 32);
    const int sz = (int)(xz >> 32), ez = (int)((xz + (unsigned long long)r.kz * (unsigned)count) >> 32);
    if (eA < 0 || sA >= nA || ez < 0 || sz >= nz) return 0;
    return sA >= -1 && eA <= nA && sz >= -1 && ez <= nz ? 2 : 1;
}

// Cells first .. first + count - 1 of the sweep (at most eight); the ray's voxel is at r.off + slot of
// `base`, planes PS apart (kPS > 0: this constant).  kRim: a ray of the tile may lie outside the volume
// here; outside, it stays on the border, whose voxels are 0, and enters with the index that the border is next to.
// kLds: from LDS, where a term of no length is added as 0 v; else from the staging copy, where it is left out (an
// infinite or undefined voxel makes the one NaN, not the other).
template <bool kLds, int kPS, bool kRim>
__device__ __forceinline__ void plane_cells(PlaneRay& r, const float* __restrict__ base, unsigned slot, unsigned PS,
                                            int nA, int nz, int first, int count) {
    constexpr int kSh = kLds ? 2 : 0;  // byte offsets in LDS, element offsets in the staging copy
    const unsigned long long xA = r.A0 + (unsigned long long)r.kA * (unsigned)first;
    const unsigned long long xz = r.z0 + (unsigned long long)r.kz * (unsigned)first;
    unsigned A = ~(unsigned)xA, z = ~(unsigned)xz;  // what is left to the next plane
    int iA = (int)(xA >> 32), iz = (int)(xz >> 32);
    const unsigned dA = (unsigned)r.dA << kSh, dZ = (unsigned)r.dZ << kSh;
    unsigned off = (r.off + slot) << kSh;
    float sum = kPS > 0 ? 0.0f : r.part;  // a constant stride: eight cells
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if (j >= count) break;  // uniform
        auto read = [&](unsigned o) {
            return kLds ? *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + (o + (kPS > 0 ? 4 * kPS * j : 0)))
                        : base[o];
        };
        const float tA = __builtin_amdgcn_fmed3f((float)A * r.iA, 0.0f, 1.0f);
        const float tz = __builtin_amdgcn_fmed3f((float)z * r.iz, 0.0f, 1.0f);
        bool cA = __builtin_sub_overflow(A, r.kA, &A), cz = __builtin_sub_overflow(z, r.kz, &z);
        if (kRim) {
            const bool inA = (unsigned)(iA + 1) <= (unsigned)nA, inz = (unsigned)(iz + 1) <= (unsigned)nz;
            iA += cA ? 1 : 0;
            iz += cz ? 1 : 0;
            cA = cA && inA;
            cz = cz && inz;
        }
        const unsigned stepA = cA ? dA : 0u, stepz = cz ? dZ : 0u;
        const unsigned mid = off + (tA < tz ? stepA : stepz), end = off + stepA + stepz;
        const float t1 = fminf(tA, tz), t2 = fmaxf(tA, tz);
        auto add = [&](float t, unsigned o) {
            if (kLds || t != 0.0f) sum = fmaf(t, read(o), sum);
        };
        add(t1, off);
        add(t2 - t1, mid);
        add(1.0f - t2, end);
        off = kPS > 0 ? end : end + (PS << kSh);
    }
    r.off = (off >> kSh) - slot;
    if (kPS > 0 || ((first + count) & 7) == 0) {
        r.sum += sum;
        r.part = 0.0f;
    } else {
        r.part = sum;
    }
}

// Workgroup table entry: views [first, first + count) of the ordered view
// records share principal axis `principal` and direction `dir`.
struct BeamGroup {
    int first, count, principal, dir;
};

constexpr int kMaxSlabs = 272;

// What the sweep needs of a slab, uniform: the byte offset of its box's lowest corner in the staging copy, the
// box's origin and whether a ray may lie outside the volume there (rim).
struct SlabBox {
    long long src;
    int a0, z0;  // Siddon: a0 holds the origin's offset a0 + z0 na, z0 the rim flag
};
__device__ __forceinline__ SlabBox slab_box(const int4* box, int s) {
    const int4 v = box[s];
    SlabBox b;
    b.src = (long long)(((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane(v.y) << 32) |
                        (unsigned)__builtin_amdgcn_readfirstlane(v.x));
    b.a0 = __builtin_amdgcn_readfirstlane(v.z);
    b.z0 = __builtin_amdgcn_readfirstlane(v.w);
    return b;
}
constexpr int kPlaneStride = kSlabCap / kSlabPlanesMax;  // LDS plane stride of an eight-plane Siddon slab

struct SweepShared {
    float buf[2 * kSlabCap];
    int4 box[kMaxSlabs];     // per slab, see SlabBox (during planning: a0, z0, rim)
    int ext[2];              // box extents na (multiple of 4) and nzb, maxed over the slabs
    int live[2];             // first and last slab whose box meets the volume (Siddon)
    int again[4];            // staging copy's rows and columns, direction, planes: for the rays that are walked again
};

// Per-ray state of the interpolated projector (ray_interpolated_projection.cu
// :117-206 restated): samples m = 0 .. count - 1 at q + m f (voxel-centre index
// frame), already clipped to the ones inside the zero-bordered volume.
struct RaySamples {
    float qP, qA, qz, fP, fA, fz;
    int m, count;
    float sum;
};

// Product of a box-relative index and a stride: both below 2^24 in an LDS box; a plane of the staging copy can be larger.
template <bool kLds>
__device__ __forceinline__ unsigned stride_mul(unsigned i, unsigned stride) {
    return kLds ? __umul24(i, stride) : i * stride;
}

// Trilinear (kMode 1) or nearest (kMode 2) sample of a box whose fastest axis
// is A: `src` holds planes P, rows z, columns A with strides SP and SZ; (pc, zc,
// ac) is the lower tap relative to the box origin.
template <int kMode, bool kLds>
__device__ __forceinline__ float box_sample(const float* __restrict__ src, int SP, int SZ, float P, float A, float Z,
                                            int P0, int Z0, int A0) {
    // tap indices relative to the box origin are >= 0
    if (kMode == 2) {
        const unsigned pc = (unsigned)((int)floorf(P + 0.5f) - P0), zc = (unsigned)((int)floorf(Z + 0.5f) - Z0),
                       ac = (unsigned)((int)floorf(A + 0.5f) - A0);
        return src[stride_mul<kLds>(pc, (unsigned)SP) + stride_mul<kLds>(zc, (unsigned)SZ) + ac];
    }
    const float flP = floorf(P), flA = floorf(A), flZ = floorf(Z);
    const float wP = P - flP, wA = A - flA, wZ = Z - flZ;
    const unsigned o = stride_mul<kLds>((unsigned)((int)flP - P0), (unsigned)SP) +
                       stride_mul<kLds>((unsigned)((int)flZ - Z0), (unsigned)SZ) + (unsigned)((int)flA - A0);
    const float c00 = fmaf(wA, src[o + 1] - src[o], src[o]);
    const float c10 = fmaf(wA, src[o + SZ + 1] - src[o + SZ], src[o + SZ]);
    const float c01 = fmaf(wA, src[o + SP + 1] - src[o + SP], src[o + SP]);
    const float c11 = fmaf(wA, src[o + SP + SZ + 1] - src[o + SP + SZ], src[o + SP + SZ]);
    const float c0 = fmaf(wZ, c10 - c00, c00), c1 = fmaf(wZ, c11 - c01, c01);
    return fmaf(wP, c1 - c0, c0);
}

// Samples of one slab (cells lo .. hi along P, box origin (a0, z0), LDS or
// global `src`); stops at the first sample whose cell lies beyond the slab.
// Returns true when the ray has no samples left.  The samples of the slab are
// counted once (P advances monotonically with the sample index), so the loop
// tests one bound per sample.  kLds: offsets inside a box are below the slab
// capacity (far below 2^24) and are formed from box-relative cell indices in
// float arithmetic, exactly; the staging copy in global memory needs the
// integer form.
template <int kMode, bool kLds>
__device__ inline bool sample_slab(RaySamples& r, const float* __restrict__ base, unsigned slot, int SP, int SZ,
                                   int P0, int Z0, int A0, int lo, int hi, int dir, float hP, float hA, float hz) {
    int m = r.m;
    const int count = r.count;
    const float qP = r.qP, qA = r.qA, qz = r.qz, fP = r.fP, fA = r.fA, fz = r.fz;
    float sum = r.sum;
    // positions stay in [-1, n] (rounding at the clipped ends), so the taps
    // stay in the zero-bordered range
    auto posP = [&](int k) { return __builtin_amdgcn_fmed3f(fmaf((float)k, fP, qP), -1.0f, hP); };
    auto cell = [&](int k) { return (int)floorf(kMode == 2 ? posP(k) + 0.5f : posP(k)); };
    auto inside = [&](int k) { return dir > 0 ? cell(k) <= hi : cell(k) >= lo; };
    // A sample clamped to the far face P = nP lies in cell nP, beyond every
    // slab (both its taps are on the zero border, so it contributes exactly
    // 0).  A sweep towards +P meets it last and stops before it; a sweep
    // towards -P meets it first, and would take it into the first slab with
    // its upper tap outside the box: skip it.
    if (dir < 0)
        while (m < count && cell(m) > hi) ++m;
    // first sample beyond the slab: an estimate, then corrected with the
    // per-sample test itself
    int me = count;
    if (fP != 0.0f) {
        const float lim = (dir > 0 ? (float)hi + 1.0f : (float)lo) - (kMode == 2 ? 0.5f : 0.0f);
        const float est = ceilf((lim - qP) / fP);
        me = est < (float)m ? m : (est > (float)count ? count : (int)est);
        while (me > m && !inside(me - 1)) --me;
        while (me < count && inside(me)) ++me;
    }
    const bool done = me >= count;
    // trilinear: the 8 taps of the last cell and their four differences along
    // A stay in registers; consecutive samples (half a voxel apart at the
    // default accuracy) mostly share a cell, so only the lanes that moved to a
    // new cell read again.  The sample index runs as an exact float.
    const float fP0 = (float)P0, fSP = (float)SP, fSZ = (float)SZ;
    // A0 + Z0 SZ - slot, so that fma(flZ, SZ, flA - cza) = (flZ - Z0) SZ + flA - A0 + slot
    // (exact: every term is an integer of magnitude below 2^24)
    const float cza = (float)(A0 + Z0 * SZ - (int)slot);
    unsigned cached = 0xffffffffu;
    float c000 = 0.f, c010 = 0.f, c100 = 0.f, c110 = 0.f, d00 = 0.f, d10 = 0.f, d01 = 0.f, d11 = 0.f;
    const float fme = (float)me;
    float fm = (float)m;
    for (; fm < fme; fm += 1.0f) {
        const float P = __builtin_amdgcn_fmed3f(fmaf(fm, fP, qP), -1.0f, hP);
        const float A = __builtin_amdgcn_fmed3f(fmaf(fm, fA, qA), -1.0f, hA);
        const float Z = __builtin_amdgcn_fmed3f(fmaf(fm, fz, qz), -1.0f, hz);
        if (kMode == 2) {
            sum += box_sample<kMode, kLds>(base + slot, SP, SZ, P, A, Z, P0, Z0, A0);
        } else {
            const float flP = floorf(P), flA = floorf(A), flZ = floorf(Z);
            const float wP = P - flP, wA = A - flA, wZ = Z - flZ;
            const unsigned o =
                kLds ? (unsigned)fmaf(flP - fP0, fSP, fmaf(flZ, fSZ, flA - cza))
                     : stride_mul<kLds>((unsigned)((int)flP - P0), (unsigned)SP) +
                           stride_mul<kLds>((unsigned)((int)flZ - Z0), (unsigned)SZ) + (unsigned)((int)flA - A0);
            if (o != cached) {
                const float* t = base + o;
                c000 = t[0];
                c010 = t[SZ];
                c100 = t[SP];
                c110 = t[SP + SZ];
                d00 = t[1] - c000;
                d10 = t[SZ + 1] - c010;
                d01 = t[SP + 1] - c100;
                d11 = t[SP + SZ + 1] - c110;
                cached = o;
            }
            // the arithmetic of box_sample, tap for tap
            const float a00 = fmaf(wA, d00, c000);
            const float a10 = fmaf(wA, d10, c010);
            const float a01 = fmaf(wA, d01, c100);
            const float a11 = fmaf(wA, d11, c110);
            const float b0 = fmaf(wZ, a10 - a00, a00), b1 = fmaf(wZ, a11 - a01, a01);
            sum += fmaf(wP, b1 - b0, b0);
        }
    }
    r.m = (int)fm;
    r.sum = sum;
    return done;
}

// One workgroup: the rays of a detector tile in the views of a group.  The tile is cut into units of 16 x 4
// pixels of one view, one wavefront each, one lane per pixel (see BeamShape).
// kMode 0: Siddon; 1: trilinear interpolation; 2: nearest-voxel sampling.
template <int kP, int kMode>
__device__ inline void beam_sweep(const float* __restrict__ stage, const StageGeom& sg, int nx, int ny, int nz,
                                  const FwdView* __restrict__ views, const BeamGroup& grp, int tile_u, int tile_v,
                                  BeamShape shape, int nU, int nV, long long su, long long sv, long long sview,
                                  float* __restrict__ out, double acc, double dvx, double dvy, double dvz,
                                  int max_planes, SweepShared& sh) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nP = kP == 0 ? nx : ny, nA = kP == 0 ? ny : nx;
    const int dir = grp.dir;
    // Siddon visits principal voxels -1 .. nP; samples have lower taps in cells
    // -1 .. nP - 1 and upper taps one plane further
    const int last_cell = kMode == 0 ? nP : nP - 1;
    const int tap = kMode == 0 ? 0 : 1;

    // ---- this lane's pixel ----
    const int upv = shape.units_u * shape.units_v;  // units per view
    const int edge_u = 16 * shape.units_u, edge_v = 4 * shape.units_v;
    const int vi = wave / upv, k = wave % upv;
    const int u = tile_u * edge_u + 16 * (k % shape.units_u) + (lane & 15);
    const int v = tile_v * edge_v + 4 * (k / shape.units_u) + (lane >> 4);
    const bool active = vi < grp.count && u < nU && v < nV;
    const FwdView& w = views[grp.first + min(vi, grp.count - 1)];

    // ---- corner rays of the tile (lanes 0..15 of every wavefront, four per view) ----
    float cA, kA, cz, kz;
    {
        const int c = lane & 15;
        const FwdView& cw = views[grp.first + min(c >> 2, grp.count - 1)];
        const int cu = min(tile_u * edge_u + ((c & 1) ? edge_u - 1 : 0), nU - 1);
        const int cvv = min(tile_v * edge_v + ((c & 2) ? edge_v - 1 : 0), nV - 1);
        const double pv = (double)(nV - 1 - cvv);
        double csrc[3];
        ray_source(cw, cu, pv, csrc);
        const double dP = cw.org[kP] + cu * cw.du[kP] + pv * cw.dv[kP] - csrc[kP];
        const double dA = cw.org[1 - kP] + cu * cw.du[1 - kP] + pv * cw.dv[1 - kP] - csrc[1 - kP];
        const double dZ = cw.org[2] + cu * cw.du[2] + pv * cw.dv[2] - csrc[2];
        const double ka = dA / dP, kzz = dZ / dP;
        kA = (float)ka;
        cA = (float)(csrc[1 - kP] - csrc[kP] * ka);
        kz = (float)kzz;
        cz = (float)(csrc[2] - csrc[kP] * kzz);
    }

    // ---- plan: box origins of every slab (in parallel over the wavefronts)
    // and the extents shared by all of them; fewer planes per slab until the
    // box fits an LDS buffer ----
    int planes = 0, first_slab = 0, nslabs = 0, na = 0, nzb = 0;
    bool staged = false;
    if (kMode == 0 && tid == 0) sh.again[0] = sg.NZ, sh.again[1] = sg.NA, sh.again[2] = dir, sh.again[3] = nP;
    for (int attempt = 0; attempt < 5 && !staged; ++attempt) {
        int pl_try = attempt == 0 ? max_planes
                                  : min(max_planes, attempt == 1 ? 6 : (attempt == 2 ? 4 : (attempt == 3 ? 2 : 1)));
        // Siddon: a constant plane stride, or a power of two of planes
        if (kMode == 0) pl_try = pl_try >= 8 ? 8 : (pl_try >= 4 ? 4 : (pl_try >= 2 ? 2 : 1));
        const int ns = (last_cell + 2 + pl_try - 1) / pl_try;
        if (ns > kMaxSlabs) continue;
        if (tid == 0) {
            sh.ext[0] = sh.ext[1] = 0;
            sh.live[0] = ns;
            sh.live[1] = -1;
        }
        __syncthreads();
        for (int s = wave; s < ns; s += kBeamThreads / 64) {
            int lo, hi;
            slab_range(s, pl_try, dir, last_cell, lo, hi);
            const BoxExtent e = beam_extent(lo, hi, cA, kA, cz, kz, nA, nz, tap);
            if (lane == 0) {
                sh.box[s] = make_int4(e.a0, e.z0, e.rim ? 1 : 0, 0);
                // (a slab outside the volume can lie between two that meet it: the beams of several views part)
                atomicMax(&sh.ext[0], (e.a1 - e.a0 + 4) & ~3);
                atomicMax(&sh.ext[1], e.z1 - e.z0 + 1);
                if (kMode != 0 || !e.out) {
                    atomicMin(&sh.live[0], s);
                    atomicMax(&sh.live[1], s);
                }
            }
        }
        __syncthreads();
        na = __builtin_amdgcn_readfirstlane(sh.ext[0]);
        nzb = __builtin_amdgcn_readfirstlane(sh.ext[1]);
        if (na * nzb * (pl_try + tap) <= kSlabCap && slab_offsets_fit(pl_try + tap, nzb, sg.NZ, sg.NA)) {
            staged = true;
            planes = pl_try;
            first_slab = __builtin_amdgcn_readfirstlane(sh.live[0]);
            nslabs = __builtin_amdgcn_readfirstlane(sh.live[1]) + 1;
        }
        __syncthreads();  // ext is reset by the next attempt
    }

    // ---- copies: Siddon planes lie in sweep order at a fixed stride, samples' planes in increasing
    // order and close ----
    const int SP = kMode == 0 ? kSlabCap / max(planes, 1) : nzb * na;
    const bool down = kMode == 0 && dir < 0;  // the first LDS plane is the highest
    // this thread's quads of a box: row (plane, z) and 4-float column, as a byte offset from the box's lowest
    // corner (32 bits: slab_offsets_fit); quads in the pad between planes and after the last copy the corner
    const int nq4 = max(na >> 2, 1), prow = max(kMode == 0 ? SP >> 2 : nzb * nq4, 1);  // row and plane in quads
    const int nq = (planes + tap) * prow;                                             // of a full slab
    constexpr int kLoads = (kSlabCap / 4 + kBeamThreads - 1) / kBeamThreads;
    unsigned qoff[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
        const int q = tid + j * kBeamThreads;
        const int pl = q / prow, rest = q - pl * prow;
        const int zr = rest / nq4, aq = rest - zr * nq4;
        const bool in = pl < planes + tap && zr < nzb;
        const unsigned row = (unsigned)(down ? planes - 1 - pl : pl) * (unsigned)sg.NZ + (unsigned)zr;
        qoff[j] = in ? 4u * (row * (unsigned)sg.NA + 4u * (unsigned)aq) : 0u;
    }
    // the slabs' table, one slab per lane (a short last slab's lowest corner is where a full one's would be)
    const int cells_total = last_cell + 2;
    if (staged && tid < nslabs) {
        int lo, hi;
        slab_range(tid, planes, dir, last_cell, lo, hi);
        const int4 e = sh.box[tid];
        const long long src = ((long long)((down ? hi - planes + 1 : lo) + 1) * sg.NZ + (e.y + 1)) * sg.NA + (e.x + 4);
        sh.box[tid] = make_int4((int)(4 * src), (int)((4 * src) >> 32), kMode == 0 ? e.y * na + e.x : e.x,
                                kMode == 0 ? e.z : e.y);
    }
    __syncthreads();
    const int wave_first = wave * 64;
    const char* stage_bytes = reinterpret_cast<const char*>(stage);
    // Direct global-to-LDS copies (16 bytes per lane) of slab s: quad q lands
    // at buf[4 q]; the LDS base of each instruction is uniform per wavefront.
    auto fetch = [&](int s, long long from) {
        float* dst = sh.buf + (s & 1) * kSlabCap + 4 * wave_first;
        const char* src = stage_bytes + from;
        const int count = cells_total - s * planes;
        if (count >= planes) {
#pragma unroll
            for (int j = 0; j < kLoads; ++j)
                if (wave_first + j * kBeamThreads < nq)  // uniform
                    __builtin_amdgcn_global_load_lds(src + qoff[j], dst + 4 * j * kBeamThreads, 16, 0, 0);
        } else {
            // a short last slab: its own planes alone
            const int nqs = (count + tap) * prow;
#pragma unroll
            for (int j = 0; j < kLoads; ++j)
                if (wave_first + j * kBeamThreads < nqs && tid + j * kBeamThreads < nqs && (qoff[j] != 0u || tid + j == 0))
                    __builtin_amdgcn_global_load_lds(src + qoff[j], dst + 4 * j * kBeamThreads, 16, 0, 0);
        }
    };
    // The slabs one after the other: `cells(s, box, slot)` walks the box of slab s, staged at buf[slot].  The
    // table is read two slabs ahead, so that the copies of the next slab start at once.
    auto sweep = [&](auto cells) {
        SlabBox cur{}, next{};
        if (first_slab < nslabs) {
            cur = slab_box(sh.box, first_slab);
            next = slab_box(sh.box, min(first_slab + 1, nslabs - 1));
            fetch(first_slab, cur.src);
        }
        __builtin_amdgcn_s_waitcnt(0);  // the direct LDS loads have landed
        __syncthreads();
        for (int s = first_slab; s < nslabs; ++s) {
            if (s + 1 < nslabs) fetch(s + 1, next.src);
            cells(s, cur, (unsigned)((s & 1) * kSlabCap));
            cur = next;
            next = slab_box(sh.box, min(s + 2, nslabs - 1));
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
        }
    };
    auto store = [&](double value) {
        if (active) out[(long long)w.pad[0] * sview + (long long)u * su + (long long)v * sv] = (float)value;
    };

    // ---- the lane's ray (FP64 set-up) and its walk ----
    const double pv = (double)(nV - 1 - v);  // detector row flip, Siddon_projection.cu:141
    double sp[3];
    ray_source(w, u, pv, sp);
    double rx = ray_dir(w, u, pv, 0);
    double ry = ray_dir(w, u, pv, 1);
    double rz = ray_dir(w, u, pv, 2);
    if (kMode == 0) {
        // The plane walk, unless a ray of the 16 x 16 pixels around this unit has a slope of 1 or more in
        // its view (their corner rays hold the extremes: the slopes are linear-fractional in the pixel), or one of the
        // unit's own a slope below flat_slope().
        // This depends on the pixel and the view alone, so a ray's sum does not depend on the group.
        const int cu = min((u & ~15) + ((lane & 1) ? 15 : 0), nU - 1);
        const double cv = (double)(nV - 1 - min((v & ~15) + ((lane & 2) ? 15 : 0), nV - 1));
        const double dP = 0.999 * fabs(ray_dir(w, cu, cv, kP));
        const bool steep = !(fabs(ray_dir(w, cu, cv, 1 - kP)) < dP && fabs(ray_dir(w, cu, cv, 2)) < dP);
        if (w.pad[1] != 0.0) parallel_siddon_height(sp, rx, ry, rz, nx, ny);
        // components below 1e-3 voxel are treated as exactly zero (:155-159)
        if (fabs(rx) < 1e-3) rx = 0.0;
        if (fabs(ry) < 1e-3) ry = 0.0;
        if (fabs(rz) < 1e-3) rz = 0.0;
        const float flat = flat_slope(nP) * fabsf((float)(kP == 0 ? rx : ry));
        const float ra = fabsf((float)(kP == 0 ? ry : rx)), rh = fabsf((float)rz);
        const bool crossings = __ballot(steep || (active && ((ra > 0.0f && ra < flat) || (rh > 0.0f && rh < flat)))) != 0;
        const double len = sqrt(rx * rx * dvx * dvx + ry * ry * dvy * dvy + rz * rz * dvz * dvz);  // mm (:241, :267)
        if (!crossings) {  // uniform per wavefront; both branches pass the same barriers
            const double rp = kP == 0 ? rx : ry;
            const double da = 1.0 / fabs(rp), a0 = ((dir > 0 ? -1.0 : (double)nP + 1.0) - sp[kP]) / rp;
            PlaneRay r;
            r.sum = r.part = 0.0f;
            plane_axis(sp[1 - kP], kP == 0 ? ry : rx, a0, da, nA, r.A0, r.kA, r.iA, r.dA);
            plane_axis(sp[2], rz, a0, da, nz, r.z0, r.kz, r.iz, r.dZ);
            if (staged) {
                r.dZ *= na;
                int at0 = 0;         // origin offset of the box that r.off refers to
                bool carry = false;  // r.off is the ray's voxel
                sweep([&](int s, const SlabBox& box, unsigned at) {
                    const int first = planes * s, count = min(planes, cells_total - first);
                    const bool was = carry;
                    bool rim = box.z0 != 0;
                    if (rim || count < 8) {
                        // what matters is whether this wavefront's rays leave the volume
                        const int e = plane_range(r, first, count, nA, nz);
                        const bool out = __ballot(active && e != 0) == 0;  // all stay outside: nothing to add
                        rim = __ballot(active && e != 2) != 0;
                        carry = false;
                        if (out) return;
                    }
                    if (was)
                        r.off -= (unsigned)(box.a0 - at0);  // from box to box by a uniform shift
                    else
                        r.off = plane_offset(r, first, box.a0, 0, na, nA, nz);
                    carry = !rim && count == 8;
                    at0 = box.a0;
                    if (!active) return;
                    if (count < 8)
                        plane_cells<true, 0, true>(r, sh.buf, at, (unsigned)SP, nA, nz, first, count);
                    else if (rim)
                        plane_cells<true, kPlaneStride, true>(r, sh.buf, at, 0u, nA, nz, first, 8);
                    else
                        plane_cells<true, kPlaneStride, false>(r, sh.buf, at, 0u, nA, nz, first, 8);
                });
            }
            // A beam whose box does not fit an LDS buffer reads the staging copy; so does a ray whose sum is not a
            // number, once more, without the terms of no length.
            const float swept = r.sum + r.part;
            if (active && (!staged || swept != swept)) {
                // from LDS: uniform values kept for this through the sweep cost it 1 % (they spilled)
                const StageGeom g2{sh.again[0], sh.again[1]};
                const int dir2 = sh.again[2], nP2 = sh.again[3];
                r.sum = r.part = 0.0f;
                r.dZ = r.dZ > 0 ? g2.NA : -g2.NA;
                r.off = plane_offset(r, 0, 0, 0, g2.NA, nA, nz) + (unsigned)stage_index(g2, dir2 > 0 ? -1 : nP2, 0, 0);
                for (int c = 0; c < nP2 + 2; c += 8)
                    plane_cells<false, 0, true>(r, stage, 0u, (unsigned)(dir2 * g2.NZ * g2.NA), nA, nz, c,
                                                min(8, nP2 + 2 - c));
            }
            store((double)(r.sum + r.part) * (len * da));  // the sum is in cells
            return;
        }
        RayWalk r;
        r.sum = 0.0f;
        int state = 0;  // 0: no ray or finished, 1: waiting for the slab of its entry, 2: walking
        int ip0 = 0, ia0 = 0, iz0 = 0, sx = 0, sy = 0, sz = 0;
        double am = -INFINITY, aM = INFINITY;
        bool hit = active && slab(sp[0], rx, nx, am, aM);
        hit = hit && slab(sp[1], ry, ny, am, aM);
        hit = hit && slab(sp[2], rz, nz, am, aM);
        if (hit && am < aM) {  // a ray that misses the volume projects to 0 (:179-180)
            const Axis ax = axis_setup(sp[0], rx, am);
            const Axis ay = axis_setup(sp[1], ry, am);
            const Axis az = axis_setup(sp[2], rz, am);
            r.tx = r.t0x = ax.t0;
            r.ty = r.t0y = ay.t0;
            r.tz = r.t0z = az.t0;
            r.dtx = ax.dt;
            r.dty = ay.dt;
            r.dtz = az.dt;
            r.kx = r.ky = r.kz = 0.0f;
            r.T = (float)(aM - am);
            r.tc = 0.0f;
            ip0 = kP == 0 ? ax.idx : ay.idx;
            ia0 = kP == 0 ? ay.idx : ax.idx;
            iz0 = az.idx;
            sx = ax.step;
            sy = ay.step;
            sz = az.step;
            state = 1;
        }
        if (!staged) {
            if (state == 1) {
                r.off = (unsigned)stage_index(sg, ip0, iz0, ia0);
                r.dX = (unsigned)(sx * (kP == 0 ? sg.NZ * sg.NA : 1));
                r.dY = (unsigned)(sy * (kP == 1 ? sg.NZ * sg.NA : 1));
                r.dZ = (unsigned)(sz * sg.NA);
                r.kexit = -1;  // never reached
                walk<kP, false>(r, stage, 0u, (nx + ny + nz + 10) / 4);
            }
        } else {
            // offset steps inside a box
            r.dX = (unsigned)(kP == 0 ? SP : sx);
            r.dY = (unsigned)(kP == 1 ? SP : sy);
            r.dZ = (unsigned)(sz * na);
            int at0 = 0;
            sweep([&](int s, const SlabBox& box, unsigned at) {
                int lo, hi;
                slab_range(s, planes, dir, last_cell, lo, hi);
                if (state == 2) {
                    // paused at the first plane of this slab: re-base the offset
                    r.off -= (unsigned)(planes * SP + box.a0 - at0);
                    r.kexit += planes;
                } else if (state == 1 && ip0 >= lo && ip0 <= hi) {
                    const int pl = dir > 0 ? ip0 - lo : hi - ip0;
                    r.off = (unsigned)(pl * SP + iz0 * na + ia0 - box.a0);
                    r.kexit = hi - lo + 1 - pl;
                    state = 2;
                }
                if (state == 2) {
                    // crossings inside one slab: its planes plus the box's a and z planes
                    if (walk<kP, true>(r, sh.buf, at, (planes + na + nzb + 7) / 4)) state = 0;
                }
                at0 = box.a0;
            });
        }
        store((double)r.sum * len);
    } else {
        RaySamples rs;
        rs.sum = 0.0f;
        bool on = false;
        double len = 0.0;
        // samples per ray and step (ray_interpolated_projection.cu:164-169)
        const double n = sample_count(w, sqrt(rx * rx + ry * ry + rz * rz), acc);
        if (active && n >= 1.0 && n < 1e9) {  // else: degenerate ray (pixel at the source), 0
            const double st[3] = {rx / n, ry / n, rz / n};
            // sample range [first, last] of the reference (:182-193), clipped to
            // the samples strictly inside (-1, n) on every axis (the others are
            // exactly zero)
            const double last = (w.cap < n) ? ceil(w.cap) : n;
            double lo = -INFINITY, hi = INFINITY;
            const int nn[3] = {nx, ny, nz};
            bool empty = false;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                if (st[a] == 0.0) {
                    if (!(sp[a] > -1.0 && sp[a] < (double)nn[a])) empty = true;
                } else {
                    const double a0 = (-1.0 - sp[a]) / st[a], a1 = ((double)nn[a] - sp[a]) / st[a];
                    lo = fmax(lo, fmin(a0, a1));
                    hi = fmin(hi, fmax(a0, a1));
                }
            }
            const double i0 = fmax(w.first, floor(lo));
            const double i1 = fmin(last, ceil(hi));
            len = sqrt(st[0] * dvx * st[0] * dvx + st[1] * dvy * st[1] * dvy + st[2] * dvz * st[2] * dvz);
            if (!empty && i0 <= i1) {
                // positions relative to the first sample keep the FP32 loop accurate
                rs.qP = (float)(sp[kP] + i0 * st[kP]);
                rs.qA = (float)(sp[1 - kP] + i0 * st[1 - kP]);
                rs.qz = (float)(sp[2] + i0 * st[2]);
                rs.fP = (float)st[kP];
                rs.fA = (float)st[1 - kP];
                rs.fz = (float)st[2];
                rs.m = 0;
                rs.count = (int)(i1 - i0) + 1;
                on = true;
            }
        }
        if (!staged) {
            // box origin (-1, -1, -4): the bordered staging copy itself
            if (on)
                sample_slab<kMode, false>(rs, stage, 0u, sg.NZ * sg.NA, sg.NA, -1, -1, -4, -1, last_cell, dir,
                                          (float)nP, (float)nA, (float)nz);
        } else {
            sweep([&](int s, const SlabBox& box, unsigned at) {
                int lo, hi;
                slab_range(s, planes, dir, last_cell, lo, hi);
                if (on && sample_slab<kMode, true>(rs, sh.buf, at, SP, na, lo, box.z0, box.a0, lo, hi, dir, (float)nP,
                                                   (float)nA, (float)nz))
                    on = false;
            });
        }
        store((double)rs.sum * len);
    }
}

// Logical block of hardware block b: runs of kRun consecutive ones on each XCD (blocks are dealt round-robin to
// the eight XCDs), all XCDs near the same place.
__device__ __forceinline__ int beam_logical_block(int b, int nblk) {
    constexpr int kRun = 64;
    const int seg = b / (8 * kRun), r = b - seg * 8 * kRun;
    return (seg + 1) * 8 * kRun <= nblk ? seg * 8 * kRun + (r & 7) * kRun + (r >> 3) : b;
}

// Workgroup L of one projection: tile rows slowest, then the groups, then the tiles of a row, so that the
// launch works through the volume in bands of z, which stay in the Infinity Cache over the groups (512^3,
// 360 views: 30.5 ms against 32.4 with the groups slowest).
template <int kMode>
__device__ __forceinline__ void beam_block(const float* __restrict__ stage_x, const float* __restrict__ stage_y,
                                           int nx, int ny, int nz, int na_x, int na_y,
                                           const FwdView* __restrict__ views, const BeamGroup* __restrict__ groups,
                                           int ngroups, int nU, int nV, long long su, long long sv, long long sview,
                                           float* __restrict__ out, double acc, double dvx, double dvy, double dvz,
                                           int max_planes, BeamShape shape, int L, SweepShared& sh) {
    const int edge_u = 16 * shape.units_u, edge_v = 4 * shape.units_v;
    const int tilesU = (nU + edge_u - 1) / edge_u, tilesV = (nV + edge_v - 1) / edge_v;
    const int row = ngroups * tilesU;
    const int tile_v = L / row, gi = (L - tile_v * row) / tilesU, tile_u = L - tile_v * row - gi * tilesU;
    if (tile_v >= tilesV) return;  // uniform per workgroup
    const BeamGroup grp = groups[gi];
    StageGeom sg;
    sg.NZ = nz + 2;
    if (grp.principal == 0) {
        sg.NA = na_x + 8;
        beam_sweep<0, kMode>(stage_x, sg, nx, ny, nz, views, grp, tile_u, tile_v, shape, nU, nV, su, sv,
                             sview, out, acc, dvx, dvy, dvz, max_planes, sh);
    } else {
        sg.NA = na_y + 8;
        beam_sweep<1, kMode>(stage_y, sg, nx, ny, nz, views, grp, tile_u, tile_v, shape, nU, nV, su, sv,
                             sview, out, acc, dvx, dvy, dvz, max_planes, sh);
    }
}

// Two workgroups per CU (8 wavefronts per SIMD): the register budget is held
// to that occupancy, which the slab barriers need to keep the SIMDs busy.
template <int kMode>
__global__ __launch_bounds__(kBeamThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void ax_beam_kernel(
    const float* __restrict__ stage_x, const float* __restrict__ stage_y, int nx, int ny, int nz, int na_x, int na_y,
    const FwdView* __restrict__ views, const BeamGroup* __restrict__ groups, int ngroups, int nU, int nV,
    long long su, long long sv, long long sview, float* __restrict__ out, double acc, double dvx, double dvy,
    double dvz, int max_planes, BeamShape shape) {
    __shared__ SweepShared sh;
    beam_block<kMode>(stage_x, stage_y, nx, ny, nz, na_x, na_y, views, groups, ngroups, nU, nV, su, sv, sview, out,
                      acc, dvx, dvy, dvz, max_planes, shape, beam_logical_block(blockIdx.x, gridDim.x), sh);
}

// Siddon projections of many independent problems (Python detector layout) in
// one launch; the XCD-ordered block index runs over the whole grid, so the
// consecutive workgroups of one group still share an XCD.
__global__ __launch_bounds__(kBeamThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void ax_beam_multi_kernel(
    const BeamJob* __restrict__ jobs, int njobs) {
    __shared__ SweepShared sh;
    const int L = beam_logical_block(blockIdx.x, gridDim.x);
    const int j = find_job(jobs, njobs, L);
    const BeamJob& J = jobs[j];
    beam_block<0>(J.stage_x, J.stage_y, J.nx, J.ny, J.nz, J.na_x, J.na_y, J.views,
                  reinterpret_cast<const BeamGroup*>(J.groups), J.ngroups, J.nU, J.nV, 1, J.nU,
                  (long long)J.nU * J.nV, J.out, J.acc, J.dvx, J.dvy, J.dvz, J.max_planes, J.shape, L - J.begin, sh);
}

// Staging copies of an x-fastest volume, for principal axis x (out_x: planes p = x, columns a = y) and y (out_y: p = y,
// a = x), or one of them: out[p][z][a] over the bordered ranges p -1 .. nP + 1, z -1 .. nz, a -4 .. na_pad + 3, zero
// outside the volume.  A workgroup reads 64 x 32 voxels (x, y) of a slice once for both, all its loads together;
// out_y is written as it was read, out_x through LDS, so reads and writes are coalesced.
//
// What bounds it: memory.  170 x 230 x 201, both copies: 26 us, 46 with a launch and a read for each and the loads one
// at a time; 512^3: 0.51 ms (1.6 GB, 3.2 TB/s); 64^3: 7 us, 16 before.
constexpr int kStageX = 64, kStageY = 32;
__device__ __forceinline__ void stage_volume_block(const void* __restrict__ vol, int dtype, int nx, int ny, int nz,
                                                   float* __restrict__ out_x, float* __restrict__ out_y, int bx, int by,
                                                   int bz) {
    __shared__ float tile[kStageX][kStageY + 1];
    constexpr int kPer = kStageX * kStageY / 256;
    const int ax = ((nx + 3) & ~3) + 8, ay = ((ny + 3) & ~3) + 8, NZ = nz + 2;  // column counts where x / y is a
    const int x0 = bx * kStageX - 4, y0 = by * kStageY - 4, z = bz - 1;
    {
        const int tx = threadIdx.x & (kStageX - 1), ty = threadIdx.x / kStageX, x = x0 + tx;
        float v[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int y = y0 + ty + k * (256 / kStageX);
            v[k] = x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz
                       ? load_storage(vol, ((long long)z * ny + y) * nx + x, dtype)
                       : 0.0f;
        }
        if (out_y) {
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                const int y = y0 + ty + k * (256 / kStageX);
                if (y >= -1 && y <= ny + 1 && x + 4 < ax) out_y[((long long)(y + 1) * NZ + (z + 1)) * ax + (x + 4)] = v[k];
            }
        }
        if (!out_x) return;  // uniform
#pragma unroll
        for (int k = 0; k < kPer; ++k) tile[tx][ty + k * (256 / kStageX)] = v[k];
    }
    __syncthreads();
    const int tx = threadIdx.x & (kStageY - 1), ty = threadIdx.x / kStageY, y = y0 + tx;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const int r = ty + k * (256 / kStageY), x = x0 + r;
        if (x >= -1 && x <= nx + 1 && y + 4 < ay) out_x[((long long)(x + 1) * NZ + (z + 1)) * ay + (y + 4)] = tile[r][tx];
    }
}

__global__ __launch_bounds__(256) void stage_volume_kernel(const void* __restrict__ vol, int dtype, int nx, int ny,
                                                           int nz, int gx, float* __restrict__ out_x,
                                                           float* __restrict__ out_y) {
    stage_volume_block(vol, dtype, nx, ny, nz, out_x, out_y, (int)(blockIdx.x % (unsigned)gx),
                       (int)(blockIdx.x / (unsigned)gx), blockIdx.z);
}

// Staging copies of many FP32 volumes in one launch.
__global__ __launch_bounds__(256) void stage_volume_multi_kernel(const StageJob* __restrict__ jobs, int njobs) {
    const int b = blockIdx.x;
    const int j = find_job(jobs, njobs, b);
    const StageJob& J = jobs[j];
    const int l = b - J.begin;
    stage_volume_block(J.vol, TIGRE_DTYPE_F32, J.nx, J.ny, J.nz, J.out_x, J.out_y, l % J.gx, (l / J.gx) % J.gy,
                       l / (J.gx * J.gy));
}

}  // namespace

int stage_pad(int n) { return (n + 3) & ~3; }

long long stage_elements(const HostGeometry& g, int principal) {
    const int nP = principal == 0 ? g.nVoxel[0] : g.nVoxel[1];
    const int nA = principal == 0 ? g.nVoxel[1] : g.nVoxel[0];
    // planes -1 .. nP + 1 written, plus one unwritten plane of slack: the
    // last rows a slab box copies may run past the copy by less than a plane
    return (long long)(nP + 4) * (g.nVoxel[2] + 2) * (stage_pad(nA) + 8);
}

int stage_job_blocks(const HostGeometry& g, int* gx, int* gy) {
    *gx = (stage_pad(g.nVoxel[0]) + 8 + kStageX - 1) / kStageX;
    *gy = (stage_pad(g.nVoxel[1]) + 8 + kStageY - 1) / kStageY;
    return *gx * *gy * (g.nVoxel[2] + 2);
}

long long beam_job_blocks(const HostGeometry& g, int ngroups, const BeamShape& shape) {
    const int edge_u = 16 * shape.units_u, edge_v = 4 * shape.units_v;
    const long long tiles = (long long)((g.nDetec[0] + edge_u - 1) / edge_u) * ((g.nDetec[1] + edge_v - 1) / edge_v);
    return tiles * ngroups;
}

int launch_stage_multi(const StageJob* d_jobs, int njobs, long long blocks, hipStream_t stream) {
    TIGRE_REQUIRE(njobs > 0 && blocks > 0 && blocks < (1LL << 31), "bad multi-job launch");
    KernelTimerScope timer(TIGRE_KERNEL_RELAYOUT, stream);
    hipLaunchKernelGGL(stage_volume_multi_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, d_jobs, njobs);
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

int launch_ax_beam_multi(const BeamJob* d_jobs, int njobs, long long blocks, hipStream_t stream) {
    TIGRE_REQUIRE(njobs > 0 && blocks > 0 && blocks < (1LL << 31), "bad multi-job launch");
    KernelTimerScope timer(TIGRE_KERNEL_AX_SIDDON, stream);
    hipLaunchKernelGGL(ax_beam_multi_kernel, dim3((unsigned)blocks), dim3(kBeamThreads), 0, stream, d_jobs, njobs);
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

int launch_stage_volume(const void* vol, int dtype, const HostGeometry& g, float* const* stage, hipStream_t stream) {
    int gx, gy;
    stage_job_blocks(g, &gx, &gy);
    TIGRE_REQUIRE((long long)gx * gy < (1LL << 31) && g.nVoxel[2] + 2 <= 65535, "volume too large for the staging copy");
    KernelTimerScope timer(TIGRE_KERNEL_RELAYOUT, stream);
    hipLaunchKernelGGL(stage_volume_kernel, dim3((unsigned)(gx * gy), 1, (unsigned)(g.nVoxel[2] + 2)), dim3(256), 0,
                       stream, vol, dtype, g.nVoxel[0], g.nVoxel[1], g.nVoxel[2], gx, stage[0], stage[1]);
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

int launch_ax_beam(const float* stage_x, const float* stage_y, const HostGeometry& g, const FwdView* d_views,
                   const int* d_groups, int ngroups, const BeamShape& shape, int projection_type, int layout, float* proj,
                   int max_planes, hipStream_t stream) {
    TIGRE_REQUIRE(max_planes >= 1 && max_planes <= kSlabPlanesMax, "slab planes out of range");
    const long long nU = g.nDetec[0], nV = g.nDetec[1];
    long long su = 1, sv = nU;
    if (layout == TIGRE_LAYOUT_MATLAB) {
        su = nV;
        sv = 1;
    }
    const long long blocks = beam_job_blocks(g, ngroups, shape);
    TIGRE_REQUIRE(blocks < (1LL << 31), "too many detector tiles for one launch");
    // LDS offsets are 32-bit; global element offsets of the staging copy too
    TIGRE_REQUIRE(stage_elements(g, 0) < (1LL << 32) && stage_elements(g, 1) < (1LL << 32),
                  "volume too large for 32-bit staging offsets");
    const bool interp = projection_type == TIGRE_PROJ_INTERPOLATED;
    // point filtering when accuracy > 1 (ray_interpolated_projection.cu:589-595)
    auto kern = !interp ? ax_beam_kernel<0> : (g.accuracy > 1.0 ? ax_beam_kernel<2> : ax_beam_kernel<1>);
    KernelTimerScope timer(interp ? TIGRE_KERNEL_AX_INTERPOLATED : TIGRE_KERNEL_AX_SIDDON, stream);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kBeamThreads), 0, stream, stage_x, stage_y, g.nVoxel[0],
                       g.nVoxel[1], g.nVoxel[2], stage_pad(g.nVoxel[1]), stage_pad(g.nVoxel[0]), d_views,
                       reinterpret_cast<const BeamGroup*>(d_groups), ngroups, g.nDetec[0], g.nDetec[1], su, sv,
                       nU * nV, proj, g.accuracy, g.dVoxel[0], g.dVoxel[1], g.dVoxel[2], max_planes, shape);
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

}  // namespace tigre
