// Cone-beam voxel-driven backprojectors for gfx950 ('FDK' and 'matched').
//
// A 256-thread workgroup owns a 16 x 16 column block of the volume and kZ
// consecutive slices; each lane keeps its kZ voxels in registers across all
// views, so the volume is read once and written once per call.  The four
// 64-lane wavefronts each cover an 8 x 8 column patch: neighbouring lanes read
// the same or the next detector pixels.  Per-view parameters are uniform
// across the workgroup and are fetched with scalar loads.
//
// Projections are read from a "quad" copy: with the four taps a = p(u,v),
// b = p(u+1,v), c = p(u,v+1), d = p(u+1,v+1) (zero outside the detector),
// element (u, v) holds (a, b - a, c - a, (d - c) - (b - a)) for tap origins
// u in [-1, nU], v in [-1, nV], stored at index (u + 1, v + 1).  One 16-byte
// load per voxel update replaces four scattered taps, the zero border
// replaces the border-addressed linear texture of the reference without
// bounds checks, and the bilinear sample is three fused multiply-adds
// (bilerp below): the differences are formed once per detector pixel instead
// of once per voxel update.  Detector coordinates are carried in
// that storage frame (pixel index + 1, the offset folded into the per-view
// records), clamped with one med3 to [0, n + 1]: the tap origin is then the
// truncating conversion and the weight the hardware fraction.
//
// When no view tilts the rotation axis (dZ has no x/y component, the case of
// every planar orbit without detector pitch/yaw) a column projects to one
// detector column, so the u interpolation weights, the 1/x division and the
// FDK weight are computed once per column and only v steps with z: those views
// take the staged kernel (atb_lds_block), all others the gather kernel.
#include <algorithm>
#include <cmath>

#include "common.hpp"

namespace tigre {

namespace {
// 1/x with the hardware reciprocal (1 ulp), instead of a correctly rounded division.
__device__ inline float rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// Waves per SIMD the gather kernel is compiled for: the register budget that
// keeps the kZ gathers of a column in flight (the compiler otherwise trades
// them for occupancy and serialises the loads).  The matched weight with 16
// slices needs more than the 168 registers of three waves (it spilled), so it
// gets two.
constexpr int atb_waves(int kW, int kZ) {
    return kZ >= 16 ? (kW == 1 ? 2 : 4) : kZ == 8 ? (kW == 1 ? 5 : 6) : 8;
}

// Matched weight l2^(3/2) / s2 from the DSD-normalised squares l2 (source to
// detector point, about 1) and s2 (source to voxel, about (DSO/DSD)^2): one
// reciprocal square root, l2^2 / sqrt(l2 s2^2), instead of a square root and a
// reciprocal.  The normalised operands keep every product near 1, whatever
// the length unit of the geometry.
__device__ __forceinline__ float matched_weight(float l2, float s2) {
    return (l2 * l2) * __builtin_amdgcn_rsqf(l2 * s2 * s2);
}

// Bilinear sample from a quad (a, b - a, c - a, (d - c) - (b - a)) at weights
// (wu, wv): s = a0 + wv (a1 - a0) with a0 = a + wu (b - a) and
// a1 - a0 = (c - a) + wu ((d - c) - (b - a)).
__device__ __forceinline__ float bilerp(const float4& q, float wu, float wv) {
    const float a0 = fmaf(wu, q.y, q.x);
    return fmaf(wv, fmaf(wu, q.w, q.z), a0);
}
}

// Writes a lane's kZ accumulated voxels: the plain result acc * scale or,
// with ep.x set, the SART update x + inv_v * (acc * scale) (clamped at 0 when
// ep.noneg) with the rounding steps of that tensor expression.
template <int kZ>
__device__ __forceinline__ void store_column(const float (&acc)[kZ], float* vol, int ix, int iy, int z0, int nx,
                                             int ny, int nz, float scale, const AtbUpdate& ep) {
    const long long plane = (long long)nx * ny;
    const long long at = (long long)z0 * plane + (long long)iy * nx + ix;
    float* out = vol + at;
    if (ep.x == nullptr) {
#pragma unroll
        for (int k = 0; k < kZ; ++k)
            if (z0 + k < nz) out[(long long)k * plane] = acc[k] * scale;
    } else {
        // three roundings, no fused multiply-add (contraction is off in this block)
#pragma clang fp contract(off)
        const float inv = ep.inv_v[(long long)iy * nx + ix];
        const float* xin = ep.x + at;
#pragma unroll
        for (int k = 0; k < kZ; ++k) {
            if (z0 + k < nz) {
                const float b = acc[k] * scale;
                const float t = inv * b;
                float v = xin[(long long)k * plane] + t;
                if (ep.noneg) v = fmaxf(v, 0.0f);
                out[(long long)k * plane] = v;
            }
        }
    }
}

// kZ: slices per lane (4, 8 or 16; fewer gives more workgroups on small
// volumes).  With ep.x set, the result is not stored but applied as the SART
// update x + inv_v[iy, ix] * result, clamped at 0 when ep.noneg, written to
// vol (which may alias ep.x: each voxel is read and written by one lane).
// kW: 0 FDK weight (voxel_backprojection.cu:241-249), 1 matched weight
// (voxel_backprojection2.cu:201-279), 2 parallel beam: the voxel projects
// orthogonally, u = y + nU/2 - 0.5, v = z + nV/2 - 0.5, weight 1
// (voxel_backprojection_parallel.cu:221-251).
template <int kW, int kZ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(atb_waves(kW, kZ), atb_waves(kW, kZ)))) void atb_kernel(const float* __restrict__ proj, int nU, int nV, int nviews,
                                                  const BwdView* __restrict__ views, float* vol, int nx,
                                                  int ny, int nz, float scale, AtbUpdate ep) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ix = blockIdx.x * 16 + (wave & 1) * 8 + (lane & 7);
    const int iy = blockIdx.y * 16 + (wave >> 1) * 8 + (lane >> 3);
    const int z0 = blockIdx.z * kZ;
    if (ix >= nx || iy >= ny) return;

    const long long QU = quad_det(nU);
    const long long QP = QU * quad_det(nV);
    const float4* __restrict__ quads = reinterpret_cast<const float4*>(proj);
    const unsigned rowb = (unsigned)QU * 16u;  // bytes per quad row (< 2^24, checked by the launcher)
    const float hu = (float)(nU + 1), hv = (float)(nV + 1);  // storage-frame clamp bounds
    const float fx = (float)ix, fy = (float)iy;

    float acc[kZ];
#pragma unroll
    for (int k = 0; k < kZ; ++k) acc[k] = 0.0f;

    // one voxel update from a storage-frame detector position (u, v) already
    // clamped to [0, n + 1]: bilinear sample of the quad copy.  Offsets are
    // 32-bit bytes from the view's (uniform) base, formed with one 24-bit
    // multiply-add.
    auto sample = [&](const char* pjb, unsigned colb, float wu, float pv) {
        const float wv = __builtin_amdgcn_fractf(pv);
        const float4 q = *reinterpret_cast<const float4*>(pjb + (__umul24((unsigned)pv, rowb) + colb));
        return bilerp(q, wu, wv);
    };

    for (int p = 0; p < nviews; ++p) {
        const BwdView& w = views[p];
        const char* pjb = reinterpret_cast<const char*>(quads + (long long)p * QP);
        // source -> voxel (ix, iy, z0) vector, frame of computeDeltasCube
        const float bx = fmaf(fy, w.dY[0], fmaf(fx, w.dX[0], w.org[0]));
        const float by = fmaf(fy, w.dY[1], fmaf(fx, w.dX[1], w.org[1]));
        const float bz = fmaf(fy, w.dY[2], fmaf(fx, w.dX[2], w.org[2]));
        constexpr bool kMatched = kW == 1, kParallel = kW == 2;
        // FDK distance weight, constant along the column (voxel_backprojection.cu:241-249)
        float wfdk = 1.0f;
        if (kW == 0) {
            const float ww = fmaf(fy, w.wfdk[2], fmaf(fx, w.wfdk[1], w.wfdk[0]));
            wfdk = rcp(ww * ww);
        }
        // matched weight: squared in-plane source-voxel distance / DSD^2, constant along z
        float Axy = 0.0f;
        if (kMatched) {
            const float ex = w.mS[0] - fmaf(fx, w.mdv[0], w.mrv0[0]);
            const float ey = w.mS[1] - fmaf(fy, w.mdv[1], w.mrv0[1]);
            Axy = ex * ex + ey * ey;
        }
#pragma unroll
        for (int k = 0; k < kZ; ++k) {
            const float fz = (float)(z0 + k);
            const float vx = fmaf(fz, w.dZ[0], bx), vy = fmaf(fz, w.dZ[1], by), vz = fmaf(fz, w.dZ[2], bz);
            const float t = kParallel ? 1.0f : w.tnum * rcp(vx);
            const float pu_raw = fmaf(vy, t, w.uoff), pv_raw = fmaf(vz, t, w.voff);
            const float pu = __builtin_amdgcn_fmed3f(pu_raw, 0.0f, hu);
            const float s = sample(pjb, (unsigned)pu * 16u, __builtin_amdgcn_fractf(pu),
                                   __builtin_amdgcn_fmed3f(pv_raw, 0.0f, hv));
            if (kMatched) {
                const float Day = fmaf(pu_raw, w.mdet[0], w.mdet[2]);
                const float Dz = fmaf(pv_raw, w.mdet[1], w.mdet[3]);
                const float rvz = fmaf(fz, w.mdv[2], w.mrv0[2]);
                acc[k] = fmaf(s, matched_weight(fmaf(Dz, Dz, fmaf(Day, Day, 1.0f)), fmaf(rvz, rvz, Axy)),
                              acc[k]);
            } else {
                acc[k] = fmaf(s, wfdk, acc[k]);
            }
        }
    }
    store_column<kZ>(acc, vol, ix, iy, z0, nx, ny, nz, scale, ep);
}

// LDS-staged kernel for axial views, all three weights.
//
// Gathered from memory, every voxel update moves 16 bytes through the
// texture-address path (about 64 bytes per clock per CU), which bounds it.
// Here the workgroup copies the detector window its 16 x 16 x kZ patch
// projects to (at most kWinRows x kWinCols quads, about 25 x 36 at unit
// magnification) into LDS with direct global-to-LDS loads, and gathers from
// there.  Two windows are kept: the copy of view p + 1 is issued at the start
// of view p, into the window of view p - 1, so it overlaps the updates; one
// barrier a view both publishes a window and frees the other.
//
// What bounds it: vector issue (9.3 instructions an update, 8.8 of them in the
// slice loop: row, conversion, fraction, address, three for the sample, one for
// the sum, and 0.8 for the column) next to LDS reads (one ds_read_b128 an update, 5.4 clocks with
// conflicts).  A window per wavefront (8 x 8 columns) copied 2.2 times the
// quads, and L2 could not feed them: 15.3 to 17.5 ms at 512^3, 360 views,
// depending on how many wavefronts shared a cache.  512^3: 17.2 -> 10.9 ms;
// 256^3, 180 views: 1.28 -> 0.79 ms; matched weight, 237 x 256 x 191, 180
// views: 1.15 -> 1.05 ms (18.7 instructions an update, one of them a reciprocal
// root).
//
// The window is the projection of the patch's corners: u and v are
// linear-fractional in the voxel position, so over a patch on one side of the
// source their extremes lie at corners (a patch on both sides, where the
// source is among the voxels, counts as one that does not fit); kWinMargin (or
// four roundings of the coordinate, on detectors beyond 32768) covers the
// rounding of the other lanes.  A view whose window does not fit is gathered
// from global memory; both paths read the same quads with the same
// arithmetic, so the results differ only in the roundings of a row position
// counted from the window.
namespace {
constexpr int kWinCols = 32;  // quads per staged row: 512 bytes of LDS
constexpr int kWinRows = 40;  // two windows are 40 KiB: four workgroups a CU
constexpr float kWinMargin = 0.125f;
// Quads a lane reads before it uses them.  More in flight cost registers and
// so wavefronts (32 slices: 86 registers with 4, 106 with 8, 146 with 16;
// 512^3: 10.4, 10.4, 11.3 ms, matched 128^3: 291, 296, 308 us a call).
constexpr int kBatch = 4;
// Columns of workgroups that one XCD's share of a layer walks through: its
// workgroups cover a compact piece of the layer, all XCDs the same slices, so
// that the views' rows are shared in L2 and in the last-level cache (512^3:
// 11.75 ms a call against 12.0 with plain block order, 11.9 with 16).
constexpr int kStrip = 8;
}  // namespace

// kN quads of one column at row positions pv + z dpv, z = z0, z0 + 1, ..., and
// their v weights, from a staged window (LDS) or from the quad copy in global
// memory.  The positions are rounded once each: added up slice by slice, 31
// roundings at a row number of 1000 are 1e-4 pixel.  kClamp: the
// column may leave the detector's rows.  The LDS pointer is
// restrict-qualified: its reads then carry alias-scope information, and the
// compiler does not make them wait for the direct LDS loads of the next view
// (into the other window) that are still in flight.
template <int kN, bool kClamp>
__device__ __forceinline__ void read_lds(const char* __restrict__ lds, int lb, float pv, float dpv, float z0, float lo,
                                         float hi, float4 (&q)[kN], float (&wv)[kN]) {
#pragma unroll
    for (int k = 0; k < kN; ++k) {
        const float row = fmaf(z0 + (float)k, dpv, pv);
        const float at = kClamp ? __builtin_amdgcn_fmed3f(row, lo, hi) : row;
        wv[k] = __builtin_amdgcn_fractf(at);
        q[k] = *reinterpret_cast<const float4*>(lds + ((int)((unsigned)at << 9) + lb));
    }
}

template <int kN>
__device__ __forceinline__ void read_global(const char* pjb, unsigned rowb, unsigned colb, float pv, float dpv,
                                            float z0, float hv, float4 (&q)[kN], float (&wv)[kN]) {
#pragma unroll
    for (int k = 0; k < kN; ++k) {
        const float at = __builtin_amdgcn_fmed3f(fmaf(z0 + (float)k, dpv, pv), 0.0f, hv);
        wv[k] = __builtin_amdgcn_fractf(at);
        q[k] = *reinterpret_cast<const float4*>(pjb + (__umul24((unsigned)at, rowb) + colb));
    }
}

// An order point for the compiler: the sum has been formed.
__device__ __forceinline__ void settled(float& a) { asm volatile("" : "+v"(a)); }

// What a column's updates need of a view, uniform over the workgroup.
struct ViewParams {
    float org[3], dX[3], dY[3], dZ2, tnum, uoff, voff, wfdk[3];
    float mdet[4], mS[2], mrv0[3], mdv[3];  // matched weight
};
__device__ __forceinline__ ViewParams view_params(const BwdView& w) {
    ViewParams v;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        v.org[c] = w.org[c];
        v.dX[c] = w.dX[c];
        v.dY[c] = w.dY[c];
        v.wfdk[c] = w.wfdk[c];
    }
    v.dZ2 = w.dZ[2];
    v.tnum = w.tnum;
    v.uoff = w.uoff;
    v.voff = w.voff;
#pragma unroll
    for (int c = 0; c < 4; ++c) v.mdet[c] = w.mdet[c];
    v.mS[0] = w.mS[0];
    v.mS[1] = w.mS[1];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        v.mrv0[c] = w.mrv0[c];
        v.mdv[c] = w.mdv[c];
    }
    return v;
}

// The workgroup of block coordinates (bx, by, bz): columns 16 bx .. + 15,
// rows 16 by .. + 15, slices kZ bz .. + kZ - 1.  With fewer than 16 slices the
// window and the row positions are those of the 16 slices they belong to, so
// 4, 8 and 16 slices give the same bits.
template <int kW, int kZ>
__device__ __forceinline__ void atb_lds_block(const float* __restrict__ proj, int nU, int nV, int nviews,
                                              const BwdView* __restrict__ views, float* vol, int nx, int ny, int nz,
                                              float scale, const AtbUpdate& ep, int bx, int by, int bz) {
    constexpr int kN = kZ < kBatch ? kZ : kBatch;
    constexpr int kG = kZ < 16 ? 16 : kZ;  // slices of a window
    __shared__ float4 win[2][kWinRows * kWinCols];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: LDS bases stay scalar
    const int px = bx * 16, py = by * 16;  // the workgroup's patch
    const int ix = px + (wave & 1) * 8 + (lane & 7);
    const int iy = py + (wave >> 1) * 8 + (lane >> 3);
    const int z0 = bz * kZ, za = z0 / kG * kG;
    // no early exit: every lane takes part in the copies, the windows and the
    // barriers; lanes outside the volume only skip the store

    const unsigned rowb = (unsigned)quad_det(nU) * 16u;
    const long long viewb = (long long)rowb * (nV + 2);
    const char* qbase = reinterpret_cast<const char*>(proj);
    const float hu = (float)(nU + 1), hv = (float)(nV + 1);
    const float fx = (float)ix, fy = (float)iy, fz = (float)za;
    // this lane's quad in each 2 x 32 block of a copy: row lane / 32, column lane % 32
    const unsigned laneoff = (unsigned)(lane >> 5) * rowb + (unsigned)(lane & 31) * 16u;
    const char* lds = reinterpret_cast<const char*>(&win[0][0]);

    // A column of the patch in a view: u, and v at slice za and its step.
    auto project = [&](const ViewParams& w, float x, float y, float& u, float& pv0, float& dpv) {
        const float vx = fmaf(y, w.dY[0], fmaf(x, w.dX[0], w.org[0]));
        const float vy = fmaf(y, w.dY[1], fmaf(x, w.dX[1], w.org[1]));
        const float vz = fmaf(y, w.dY[2], fmaf(x, w.dX[2], w.org[2]));
        const float t = kW == 2 ? 1.0f : w.tnum * rcp(vx);
        u = fmaf(vy, t, w.uoff);
        dpv = w.dZ2 * t;
        pv0 = fmaf(fmaf(fz, w.dZ2, vz), t, w.voff);
    };
    // The windows of 64 views at a time, one view per lane, from the patch's corner columns (in the view loop a
    // window is then four lane reads, not a serial chain of projections and minima): byte offset of the window's
    // first quad in its view's copy, LDS byte offset of column 0 before it, its first row, and its 2-row blocks
    // (0: it does not fit; + 32: no slice of the patch projects beyond the detector's rows).
    unsigned wsrc = 0;
    int wlds = 0, wblocks = 0;
    float wrow = 0.0f;
    auto windows = [&](int first) {
        const ViewParams w = view_params(views[min(first + lane, nviews - 1)]);
        float vlo = __builtin_inff(), vhi = -vlo, ulo = hu, uhi = 0.0f, dlo = vlo, dhi = vhi;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float pu, pv0, dpv;
            project(w, (float)(px + (j & 1) * 15), (float)(py + (j >> 1) * 15), pu, pv0, dpv);
            // rows of the first and last slice (v is monotonic along the column)
            const float pv1 = fmaf((float)(kG - 1), dpv, pv0);
            vlo = fminf(vlo, fminf(pv0, pv1));
            vhi = fmaxf(vhi, fmaxf(pv0, pv1));
            dlo = fminf(dlo, dpv);
            dhi = fmaxf(dhi, dpv);
            pu = __builtin_amdgcn_fmed3f(pu, 0.0f, hu);
            ulo = fminf(ulo, pu);
            uhi = fmaxf(uhi, pu);
        }
        const float mu = fmaxf(kWinMargin, hu * 0x1p-18f), mv = fmaxf(kWinMargin, hv * 0x1p-18f);
        const int r0 = (int)__builtin_amdgcn_fmed3f(vlo - mv, 0.0f, hv);
        const int r1 = (int)__builtin_amdgcn_fmed3f(vhi + mv, 0.0f, hv);
        const int c0 = (int)fmaxf(ulo - mu, 0.0f), c1 = (int)fminf(uhi + mu, hu);
        wsrc = (unsigned)r0 * rowb + (unsigned)c0 * 16u;
        wlds = -c0 * 16;
        wrow = (float)r0;
        // (steps of one sign: the patch lies on one side of the source)
        const bool fits = r1 - r0 < kWinRows && c1 - c0 < kWinCols && dlo * dhi > 0.0f && dhi - dlo < __builtin_inff();
        wblocks = fits ? (r1 - r0 + 2) >> 1 : 0;
        if (wblocks > 0 && vlo >= mv && vhi <= hv - mv) wblocks += 32;
    };
    // Issues the copy of view p's window, the 2 x 32 blocks shared out over the wavefronts (the quads past the
    // window belong to the next row or view or to the slack after the copy, and are never read).
    auto fetch = [&](int p, int& offset, int& blocks, float& row) {
        const int l = p & 63;
        blocks = __builtin_amdgcn_readlane(wblocks, l);
        offset = __builtin_amdgcn_readlane(wlds, l) + (p & 1) * (kWinRows * kWinCols * 16);
        row = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wrow), l));
        const char* src = qbase + (long long)p * viewb + (unsigned)__builtin_amdgcn_readlane((int)wsrc, l);
        const int n = p < nviews ? blocks & 31 : 0;
        float4* dst = &win[p & 1][0];
#pragma unroll 1  // unrolled, the copy's branches split the view's code and its registers spill
        for (int j = wave; j < n; j += 4)
            __builtin_amdgcn_global_load_lds(src + (long long)(2 * j) * rowb + laneoff, dst + 64 * j, 16, 0, 0);
    };
    // per view and column: u weight, quad column (bytes), v at slice za and its step, distance weight
    struct Col {
        float wu, pv0, dpv, wt;
        unsigned colb;
        // matched weight: detector and voxel height at slice za with their steps, and the in-plane squares
        float dz, ddz, rz, drz, Day2, Axy;
    };
    auto column = [&](const ViewParams& w, Col& c) {
        float u;
        project(w, fx, fy, u, c.pv0, c.dpv);
        const float pu = __builtin_amdgcn_fmed3f(u, 0.0f, hu);
        c.wt = 1.0f;
        if (kW == 0) {  // voxel_backprojection.cu:241-249
            const float ww = fmaf(fy, w.wfdk[2], fmaf(fx, w.wfdk[1], w.wfdk[0]));
            c.wt = rcp(ww * ww);
        }
        if (kW == 1) {  // voxel_backprojection2.cu:201-279, squares over DSD^2
            const float Day = fmaf(u, w.mdet[0], w.mdet[2]);
            c.Day2 = fmaf(Day, Day, 1.0f);
            const float ex = w.mS[0] - fmaf(fx, w.mdv[0], w.mrv0[0]);
            const float ey = w.mS[1] - fmaf(fy, w.mdv[1], w.mrv0[1]);
            c.Axy = ex * ex + ey * ey;
            c.dz = fmaf(c.pv0, w.mdet[1], w.mdet[3]);
            c.ddz = c.dpv * w.mdet[1];
            c.rz = fmaf(fz, w.mdv[2], w.mrv0[2]);
            c.drz = w.mdv[2];
        }
        c.wu = __builtin_amdgcn_fractf(pu);
        c.colb = (unsigned)pu * 16u;
    };

    float acc[kZ];
#pragma unroll
    for (int k = 0; k < kZ; ++k) acc[k] = 0.0f;

    if (nviews > 0) {
        int offset, blocks;
        float row;
        windows(0);
        fetch(0, offset, blocks, row);
        Col c;
        column(view_params(views[0]), c);
        ViewParams next = view_params(views[min(1, nviews - 1)]);
        int p = 0;
        // one view; read: fills a batch of quads and v weights from the row position
        auto view = [&](auto&& read) {
            const int lb = (int)c.colb + offset, nb = blocks;
            const float r0 = row;
            // this view's window has landed, and every wavefront is done with the other one
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (((p + 1) & 63) == 0) windows(p + 1);
            fetch(p + 1, offset, blocks, row);
            const ViewParams v = next;
            next = view_params(views[min(p + 2, nviews - 1)]);
            const float pv = nb > 0 ? c.pv0 - r0 : c.pv0;
#pragma unroll
            for (int k = 0; k < kZ; k += kN) {
                float4 q[kN];
                float wv[kN];
                read(lb, r0, pv, (float)(z0 - za + k), q, wv);
                __builtin_amdgcn_sched_barrier(0);
                float wt[kN];
#pragma unroll
                for (int i = 0; i < kN; ++i) {
                    wt[i] = c.wt;
                    if (kW == 1) {
                        const float z = (float)(z0 - za + k + i);
                        const float dz = fmaf(z, c.ddz, c.dz), rz = fmaf(z, c.drz, c.rz);
                        wt[i] = matched_weight(fmaf(dz, dz, c.Day2), fmaf(rz, rz, c.Axy));
                    }
                }
#pragma unroll
                for (int i = 0; i < kN; ++i) acc[k + i] = fmaf(bilerp(q[i], c.wu, wv[i]), wt[i], acc[k + i]);
                if (k + kN < kZ) {
                    // the batch is used up before the next is read (or the quads of both need registers)
#pragma unroll
                    for (int i = 0; i < kN; ++i) settled(acc[k + i]);
                }
            }
            column(v, c);
            ++p;
        };
        // runs of views of one kind: a branch within the view loop would move the sums between registers
        while (p < nviews) {
            while (p < nviews && blocks >= 32)
                view([&](int lb, float, float pv, float z, float4 (&q)[kN], float (&wv)[kN]) {
                    read_lds<kN, false>(lds, lb, pv, c.dpv, z, 0.0f, 0.0f, q, wv);
                });
            while (p < nviews && blocks > 0 && blocks < 32)
                view([&](int lb, float r0, float pv, float z, float4 (&q)[kN], float (&wv)[kN]) {
                    read_lds<kN, true>(lds, lb, pv, c.dpv, z, -r0, hv - r0, q, wv);
                });
            while (p < nviews && blocks == 0)
                view([&](int, float, float pv, float z, float4 (&q)[kN], float (&wv)[kN]) {
                    read_global<kN>(qbase + (long long)p * viewb, rowb, c.colb, pv, c.dpv, z, hv, q, wv);
                });
        }
    }
    if (ix < nx && iy < ny) store_column<kZ>(acc, vol, ix, iy, z0, nx, ny, nz, scale, ep);
}

template <int kW, int kZ>
__global__ __launch_bounds__(256, 3) void atb_lds_kernel(const float* __restrict__ proj, int nU, int nV, int nviews,
                                                      const BwdView* __restrict__ views, float* vol, int nx,
                                                      int ny, int nz, float scale, AtbUpdate ep) {
    // workgroups go to the XCDs in turn
    const int gx = (nx + 15) / 16, gy = (ny + 15) / 16;
    const int per = (gx * gy + 7) / 8;  // blocks of an XCD in one layer of slices
    const int i = (int)blockIdx.x >> 3, bz = i / per, b = ((int)blockIdx.x & 7) * per + i - bz * per;
    if (b >= gx * gy) return;
    const int strip = b / (kStrip * gy), r = b - strip * kStrip * gy, w = min(kStrip, gx - strip * kStrip);
    const int by = r / w, bx = strip * kStrip + r - by * w;
    atb_lds_block<kW, kZ>(proj, nU, nV, nviews, views, vol, nx, ny, nz, scale, ep, bx, by, bz);
}

// Many independent FDK backprojections with the SART update epilogue in one
// launch: job j owns blocks [begin, begin + gx gy gz) of the grid.
template <int kZ>
__global__ __launch_bounds__(256, 3) void atb_lds_multi_kernel(const AtbJob* __restrict__ jobs, int njobs) {
    const int b = (int)blockIdx.x;
    const int j = find_job(jobs, njobs, b);
    const AtbJob& J = jobs[j];
    const int l = b - J.begin;
    AtbUpdate ep;
    ep.x = J.x;
    ep.inv_v = J.inv_v;
    ep.noneg = J.noneg;
    atb_lds_block<0, kZ>(J.quads, J.nU, J.nV, J.nviews, J.views, J.vol, J.nx, J.ny, J.nz, J.scale, ep, l % J.gx,
                         (l / J.gx) % J.gy, l / (J.gx * J.gy));
}

// Quad copy of the projections (see above), view-major, rows of quad_det(nU)
// elements.  Reads either detector layout.  A wavefront writes kQuadRows rows
// of 64 quads, each from its upper neighbour's lower taps; units first,
// first + stride, ...
constexpr int kQuadRows = 4;
__device__ __forceinline__ void quad_projections_range(const void* __restrict__ proj, int dtype, int nU, int nV,
                                                       int nviews, int layout, float4* __restrict__ quads,
                                                       long long first, long long stride) {
    const int QU = nU + 2, QV = nV + 2, lane = threadIdx.x & 63;
    const int nx = (QU + 63) / 64, ny = (QV + kQuadRows - 1) / kQuadRows;
    const long long units = (long long)nx * ny * nviews;
    for (long long w = first; w < units; w += stride) {
        const int bx = (int)(w % nx), by = (int)(w / nx % ny);
        const long long p = w / ((long long)nx * ny);
        const int u = bx * 64 + lane - 1, v = by * kQuadRows - 1;
        if (u > nU) continue;
        const long long base = p * (long long)nU * nV;
        auto at = [&](int uu, int vv) {
            if (uu < 0 || uu >= nU || vv < 0 || vv >= nV) return 0.0f;
            return load_storage(proj, layout == TIGRE_LAYOUT_MATLAB ? base + (long long)uu * nV + vv : base + (long long)vv * nU + uu,
                                dtype);
        };
        float a[kQuadRows + 1], b[kQuadRows + 1];
#pragma unroll
        for (int k = 0; k <= kQuadRows; ++k) {
            a[k] = at(u, v + k);
            b[k] = at(u + 1, v + k);
        }
        float4* out = quads + (p * QV + v + 1) * QU + u + 1;
#pragma unroll
        for (int k = 0; k < kQuadRows; ++k) {
            const float du0 = b[k] - a[k], du1 = b[k + 1] - a[k + 1];
            if (v + k <= nV) out[(long long)k * QU] = make_float4(a[k], du0, a[k + 1] - a[k], du1 - du0);
        }
    }
}

__global__ __launch_bounds__(256) void quad_projections_kernel(const void* __restrict__ proj, int dtype, int nU,
                                                               int nV, int nviews, int layout,
                                                               float4* __restrict__ quads) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    quad_projections_range(proj, dtype, nU, nV, nviews, layout, quads, (long long)blockIdx.x * 4 + wave,
                           (long long)gridDim.x * 4);
}

// Pair or quad copies of many FP32 projection sets (Python layout) in one launch.
__global__ __launch_bounds__(256) void quad_projections_multi_kernel(const QuadJob* __restrict__ jobs, int njobs) {
    const int b = blockIdx.x;
    const int j = find_job(jobs, njobs, b);
    const QuadJob& J = jobs[j];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    quad_projections_range(J.proj, TIGRE_DTYPE_F32, J.nU, J.nV, J.nviews, TIGRE_LAYOUT_PYTHON,
                           reinterpret_cast<float4*>(J.quads), (long long)(b - J.begin) * 4 + wave,
                           (long long)J.blocks * 4);
}

int quad_job_blocks(int nU, int nV, int nviews) {
    const long long units = (quad_det(nU) + 63) / 64 * ((quad_det(nV) + kQuadRows - 1) / kQuadRows) * nviews;
    long long blocks = (units + 3) / 4;
    if (blocks > 65536) blocks = 65536;
    return (int)(blocks < 1 ? 1 : blocks);
}

int launch_quad_multi(const QuadJob* d_jobs, int njobs, long long blocks, hipStream_t stream) {
    TIGRE_REQUIRE(njobs > 0 && blocks > 0 && blocks < (1LL << 31), "bad multi-job launch");
    KernelTimerScope timer(TIGRE_KERNEL_RELAYOUT, stream);
    hipLaunchKernelGGL(quad_projections_multi_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, d_jobs, njobs);
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

int launch_atb_multi(const AtbJob* d_jobs, int njobs, long long blocks, int zper, hipStream_t stream) {
    TIGRE_REQUIRE(njobs > 0 && blocks > 0 && blocks < (1LL << 31), "bad multi-job launch");
    TIGRE_REQUIRE(zper == 4 || zper == 8 || zper == 16 || zper == 32, "slices per lane must be 4, 8, 16 or 32");
    KernelTimerScope timer(TIGRE_KERNEL_ATB_FDK, stream);
    if (zper == 32)
        hipLaunchKernelGGL(atb_lds_multi_kernel<32>, dim3((unsigned)blocks), dim3(256), 0, stream, d_jobs, njobs);
    else if (zper == 16)
        hipLaunchKernelGGL(atb_lds_multi_kernel<16>, dim3((unsigned)blocks), dim3(256), 0, stream, d_jobs, njobs);
    else if (zper == 8)
        hipLaunchKernelGGL(atb_lds_multi_kernel<8>, dim3((unsigned)blocks), dim3(256), 0, stream, d_jobs, njobs);
    else
        hipLaunchKernelGGL(atb_lds_multi_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, stream, d_jobs, njobs);
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

int launch_quad_projections(const void* proj, int dtype, int nU, int nV, int nviews, int layout, float* quads,
                            hipStream_t stream) {
    KernelTimerScope timer(TIGRE_KERNEL_RELAYOUT, stream);
    hipLaunchKernelGGL(quad_projections_kernel, dim3((unsigned)quad_job_blocks(nU, nV, nviews)), dim3(256), 0, stream,
                       proj, dtype, nU, nV, nviews, layout, reinterpret_cast<float4*>(quads));
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

// Slices per lane of the staged kernel for the default of 16: twice as many share a column's and a window's work
// (whole calls, 512^3, 360 views: 11.2 ms with 32, 12.5 with 16; 256^3, 180 views: 1.69 and 1.81 ms) where that
// leaves two full rounds of the chip's 1024 workgroups (below, 237 x 256 x 191 with 1440: 1.27 ms with 32, 1.21
// with 16).  32 slices also have to fit the window's rows (192^3 on 200 rows, where many did not: 660 us with 32,
// 454 with 16), estimated where the circle inscribed in the volume comes closest to the source; the corners beyond
// it may still miss and are gathered.  Eight or four slices give a small volume more workgroups (64^3, 100 views: 171
// us a call with 8, 198 with 16; 128^3, 180 views: 216 with 8 and 1024 workgroups, 221 with 16 and 512); in a batch
// the other jobs fill the chip.  Never twice the volume's slices: a lane computes all of its own (one slice of 1024 x
// 1024, 720 views: 2.5 ms matched and 1.9 FDK with 4, 9.9 and 4.9 with 32).
int staged_slices(const HostGeometry& g, int zper, bool batched) {
    if (zper != 16) return zper;
    const long long columns = (long long)((g.nVoxel[0] + 15) / 16) * ((g.nVoxel[1] + 15) / 16);
    const double radius = std::max(g.sVoxel[0], g.sVoxel[1]) / 2, depth = 15 * std::hypot(g.dVoxel[0], g.dVoxel[1]);
    bool fits = true;
    for (int i = 0; i < g.nangles && fits; ++i) {
        const double near = g.DSO[i] - radius;
        const double m1 = g.parallel ? 1.0 : g.DSD[i] / near, m2 = g.parallel ? 1.0 : g.DSD[i] / (near + depth);
        const double rows = (31 * g.dVoxel[2] * m1 + g.sVoxel[2] / 2 * (m1 - m2)) / g.dDetec[1];
        fits = (g.parallel || near > 0) && rows + 2 * kWinMargin + 2 <= kWinRows;
    }
    auto blocks = [&](int z) { return columns * ((g.nVoxel[2] + z - 1) / z); };
    const int nz = g.nVoxel[2];
    if (nz > 16 && fits && blocks(32) >= 2048) return 32;
    if (nz > 8 && (batched || blocks(16) >= 512)) return 16;
    return nz > 4 && (batched || blocks(8) >= 512) ? 8 : 4;
}

int launch_atb(const float* quads, const HostGeometry& g, const BwdView* d_views, bool matched, bool axial,
               float* vol, int zper, const AtbUpdate& ep, hipStream_t stream) {
    // the parallel-beam backprojector serves both 'FDK' and 'matched' (_Atb.pyx:56-76)
    const int kind = g.parallel ? 2 : (matched ? 1 : 0);
    TIGRE_REQUIRE(zper == 4 || zper == 8 || zper == 16, "slices per lane must be 4, 8 or 16");
    // per-view byte offsets are 32-bit and the row stride enters a 24-bit multiply
    TIGRE_REQUIRE(quad_det(g.nDetec[0]) * 16 < (1LL << 24) &&
                      quad_det(g.nDetec[0]) * quad_det(g.nDetec[1]) * 16 < (1LL << 32),
                  "detector too large for one backprojection launch");
    const int nx = g.nVoxel[0], ny = g.nVoxel[1], nz = g.nVoxel[2];
    dim3 grid((nx + 15) / 16, (ny + 15) / 16, (nz + zper - 1) / zper);
    TIGRE_REQUIRE(grid.z <= 65535u && grid.y <= 65535u, "volume too large for one launch");
    if (axial) zper = staged_slices(g, zper, false);
    const long long blocks = ((long long)grid.x * grid.y + 7) / 8 * 8 * ((nz + zper - 1) / zper);
    TIGRE_REQUIRE(!axial || blocks < (1LL << 31), "volume too large for one launch");
    // matched: final scaling by dVx dVy dVz / (dU dV) (voxel_backprojection2.cu:585)
    const float scale =
        kind == 1 ? (float)(g.dVoxel[0] * g.dVoxel[1] * g.dVoxel[2] / (g.dDetec[0] * g.dDetec[1])) : 1.0f;
    KernelTimerScope timer(kind == 1 ? TIGRE_KERNEL_ATB_MATCHED : TIGRE_KERNEL_ATB_FDK, stream);
#define TIGRE_ATB_LAUNCH(M, Z)                                                                                 \
    do {                                                                                                       \
        if (axial)                                                                                             \
            hipLaunchKernelGGL((atb_lds_kernel<M, Z>), dim3((unsigned)blocks), dim3(256), 0, stream, quads,    \
                               g.nDetec[0], g.nDetec[1], g.nangles, d_views, vol, nx, ny, nz, scale, ep);      \
        else                                                                                                   \
            hipLaunchKernelGGL((atb_kernel<M, (Z <= 16 ? Z : 16)>), grid, dim3(256), 0, stream, quads, g.nDetec[0],             \
                               g.nDetec[1], g.nangles, d_views, vol, nx, ny, nz, scale, ep);                   \
    } while (0)
#define TIGRE_ATB_Z(M)                                \
    do {                                              \
        if (zper == 32) TIGRE_ATB_LAUNCH(M, 32);      \
        else if (zper == 16) TIGRE_ATB_LAUNCH(M, 16); \
        else if (zper == 8) TIGRE_ATB_LAUNCH(M, 8);   \
        else TIGRE_ATB_LAUNCH(M, 4);                  \
    } while (0)
    if (kind == 0) TIGRE_ATB_Z(0);
    else if (kind == 1) TIGRE_ATB_Z(1);
    else TIGRE_ATB_Z(2);
#undef TIGRE_ATB_Z
#undef TIGRE_ATB_LAUNCH
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

}  // namespace tigre
