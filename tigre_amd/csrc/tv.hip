// TV steps for gfx950: POCS-TV steepest descent (minimizeTV) and the ROF
// primal-dual denoiser.
//
// POCS-TV, GD_TV.cu:489-597 (and its adaptive-weighted and PICCS variants,
// GD_AwTV.cu, PICCS.cu).  The TV sub-gradient of GD_TV.cu:117-143 at voxel v
// is the divergence of the normalised backward-difference field
//     n_c(v) = w_c d_c(v) / (sqrt(sum_k w_k d_k(v)^2) + eps),
//     g(v)   = n_x(v) + n_y(v) + n_z(v) - n_x(v + x) - n_y(v + y) - n_z(v + z),
// (w = 1 for TV, exp(-(d / delta)^2) per component for AwTV, with the fast
// exponential as the reference's __expf), so each n is
// computed once per voxel instead of four times.  An iteration needs the norm
// of the whole g before it can step, f' = f - alpha / sqrt(sum g^2 + norm_eps)
// g.  Three forms, chosen by a rule on the sizes (run_tv_descent):
//   one pass   makes f' from f and also sums g^2 of f' for the next step (FP32
//              over eight voxels, FP64 beyond); the next pass adds up the
//              workgroups' sums in a fixed order at its start, every wavefront for
//              itself.  A first pass only sums, the last only steps: maxiter + 1
//              launches, 8 bytes of traffic per voxel and iteration;
//   two passes a pass for the norm and one for the step: 2 maxiter launches, 12
//              bytes;
//   LDS tiles  (tv_tiles.hip) two passes and a reduction: 3 maxiter launches, 12
//              bytes.
// None has a host round trip for the norm.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "ray.hpp"  // xcd_logical_block

namespace tigre {

namespace {
constexpr int kTvThreads = 256, kTvWaves = kTvThreads / 64;  // wavefronts work on tiles of their own
constexpr int kTvColumns = 60;                               // columns of a tile, but for the volume's edges
template <int k>
using Int = std::integral_constant<int, k>;
constexpr int kTvBatch = 6;                                  // rows whose chains are interleaved
constexpr int kTvBlocks = 1024;                              // workgroups of a pass, at most

// Workgroup sum of one double per lane (wavefront shuffles, then LDS), in every thread.
__device__ inline double block_sum(double v) {
    __shared__ double part[kTvWaves];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int i = 0; i < kTvWaves; ++i) s += part[i];
    return s;
}

// Value of the lane before / after this one (0 in lane 0 / 63).
__device__ __forceinline__ float lane_before(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xF, 0xF, true));
}
__device__ __forceinline__ float lane_after(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xF, 0xF, true));
}
// An order point for the compiler: the value is formed before the branches that follow, not after them with all that
// it is formed from kept in registers.
__device__ __forceinline__ void formed(float& v) { asm volatile("" : "+v"(v)); }

// The normalised difference field at kB voxels from their values c, the values below them (z - 1) and their
// neighbours at x - 1 and y - 1 (GD_TV.cu:104-140: a missing neighbour's difference is 0, and beyond the high edges n
// is 0 in its axis).  No masks: beyond the edges the rows and columns hold copies of the edge voxels, so those
// differences are exactly 0, and the zero slices (planes -1 and nz) hold 0.  z: whether PICCS has the z difference.
// In stages over the voxels, kept apart: left to itself the compiler finishes one voxel's chain of square root,
// reciprocal and products after the other's, and three wavefronts a SIMD do not hide that.  n: the numerator in z, the
// field in y and x; s: what the numerator is to be multiplied with.
template <int kKind, int kB>
__device__ __forceinline__ void n_field(const float (&c)[kB], const float (&below)[kB], const float (&cy)[kB], bool z,
                                        const TvParams& tp, float (&n)[kB][3], float (&s)[kB]) {
    constexpr float eps = kKind == 2 ? 1e-6f : 1e-8f;
    float d[kB][3], w[kB][3];
#pragma unroll
    for (int i = 0; i < kB; ++i) {
        d[i][0] = kKind == 2 ? (z ? c[i] - below[i] : 0.0f) : c[i] - below[i];
        d[i][1] = c[i] - cy[i];
        d[i][2] = c[i] - lane_before(c[i]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (kKind == 1) {
#pragma unroll
        for (int i = 0; i < kB; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float a = d[i][k] * tp.inv_delta;
                w[i][k] = __expf(-a * a);
            }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < kB; ++i) {
        const float(&e)[3] = d[i];
        if (kKind == 0) s[i] = fmaf(e[2], e[2], fmaf(e[0], e[0], e[1] * e[1]));
        if (kKind == 1) s[i] = fmaf(e[2], w[i][2] * e[2], fmaf(e[0], w[i][0] * e[0], e[1] * (w[i][1] * e[1])));
        if (kKind == 2) s[i] = fmaf(e[2], e[2], fmaf(e[1], e[1], e[0] * e[0]));
    }
    __builtin_amdgcn_sched_barrier(0);
    // hardware square root and reciprocal (1 ulp each)
#pragma unroll
    for (int i = 0; i < kB; ++i) s[i] = __builtin_amdgcn_sqrtf(s[i]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kB; ++i) s[i] = __builtin_amdgcn_rcpf(s[i] + eps);
    __builtin_amdgcn_sched_barrier(0);
    // rounded products: g takes an n once as a voxel's own and once as its neighbour's, and where the two should cancel
    // they have to be the same number (what is left of them is normalised in the next iteration)
    {
#pragma clang fp contract(off)
#pragma unroll
        for (int i = 0; i < kB; ++i) {
            n[i][0] = kKind == 1 ? w[i][0] * d[i][0] : d[i][0];
#pragma unroll
            for (int k = 1; k < 3; ++k) n[i][k] = (kKind == 1 ? w[i][k] * d[i][k] : d[i][k]) * s[i];
        }
    }
}
}  // namespace

// kKind 0: TV (GD_TV; the image sits between zero slices, so z always has a
// neighbour, GD_TV.cu:367-368,456-465), 1: adaptive-weighted TV (GD_AwTV,
// same padding), 2: PICCS, (1 - ratio) g(f) + ratio g(f - prior) with the z
// term dropped at the edges like x and y (PICCS.cu:109-157,322-347).  At the
// low x / y edge the difference is 0; beyond the high edge n is 0
// (GD_TV.cu:104-114).
//
// A wavefront works alone, without LDS or barriers: a tile of 64 columns (one a lane) and kCore + 4 rows (in
// registers) marches along z through a chunk of planes.  In step p it reads f of plane p, completes g of plane p - 1
// and steps it (kUpdate), then completes g' of plane p - 2 from the stepped planes (kNorm); x neighbours come by
// wavefront shifts.  Both stages need one voxel more on either side, so 60 of the columns and kCore rows are stored.
// The volume's own edges need no halo: there, loads give copies of the edge voxels, and after the step the copies are
// made again, under branches that are uniform in the tile.  Loads run two planes ahead through buffer descriptors
// (planes outside the volume read 0).
//
// What bounds it: vector issue, 20 evaluations of n (a square root and a reciprocal each) for 8 stored rows a plane
// with 3 wavefronts a SIMD; the halo costs 1.5 to 1.9 times the voxels.  20 iterations, two passes and a one-workgroup
// sum an iteration with barriers and LDS before and this: 40 x 36 x 42 486 -> 151 us, 128^3 521 -> 361, 200^3 768 -> 578,
// 256^3 975 -> 940 (its 256 columns fill 5 tiles of 60 badly), 400^3 4514 -> 3069, 512^3 7474 -> 6297; AwTV 240^3
// 1164 -> 1092; PICCS 300^3 3216 -> 2396.
template <int kKind, int kCore, bool kUpdate, bool kNorm>
__global__ __launch_bounds__(kTvThreads, kKind == 2 ? 2 : 3) void tv_kernel(const float* __restrict__ f, float* __restrict__ out,
                                                        TvParams tp, int nx, int ny, int nz, int ntx, int nty,
                                                        int chunk, int ntiles, float alpha, double norm_eps,
                                                        const double* __restrict__ partial_in, int npartial,
                                                        double* __restrict__ partial_out) {
    constexpr int kR = kCore + 4;               // rows with the halo
    constexpr int NF = kKind == 2 ? 2 : 1;      // fields: f, and f - prior
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned plane_bytes = (unsigned)nx * (unsigned)ny * 4u;
    const long long plane = (long long)nx * ny;
    auto rsrc = [&](const float* base, int z) {  // a plane; planes outside the volume read 0 and drop stores
        const bool in = z >= 0 && z < nz;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base + (in ? z : 0) * plane), (short)0,
                                                 in ? (int)plane_bytes : 0, 0x00020000);
    };
    // alpha / sqrt(sum of the partials + norm_eps), in the same order and so with the same bits in every wavefront
    float scale = 0.0f;
    auto read_scale = [&]() {
        double part[kTvBlocks / 64], sum = 0.0;
#pragma unroll
        for (int k = 0; k < kTvBlocks / 64; ++k) part[k] = k * 64 + lane < npartial ? partial_in[k * 64 + lane] : 0.0;
#pragma unroll
        for (int k = 0; k < kTvBlocks / 64; ++k) sum += part[k];
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
        scale = (float)((double)alpha / sqrt(sum + norm_eps));
    };
    double total = 0.0;
    const int first = xcd_logical_block((int)blockIdx.x, (int)gridDim.x) * kTvWaves + wave;
    for (int tile = first; tile < ntiles; tile += (int)gridDim.x * kTvWaves) {
        const int tx = tile % ntx, ty = tile / ntx % nty, tz = tile / (ntx * nty);
        const int z0 = tz * chunk, z1 = min(z0 + chunk, nz);
        // columns x0 - 1 .. x0 + 62, of which 60 are stored, but for the volume's edges; rows y0 .. y0 + kR - 1
        const int x = tx * kTvColumns + lane - 1, y0 = ty * kCore - 2;
        const bool low_x = tx == 0, high_x = (tx + 1) * kTvColumns + 3 >= nx, low_y = ty == 0, high_y = y0 + kR > ny;
        const bool core = x >= 0 && x < nx && (lane >= 2 || low_x) && (lane < 62 || high_x);
        const unsigned xofs = (unsigned)min(max(x, 0), nx - 1) * 4u;
        unsigned rowofs[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) rowofs[r] = (unsigned)min(max(y0 + r, 0), ny - 1) * (unsigned)nx * 4u;

        // per row: f and prior one plane back, prior two back, the z-free part of g of the plane before; the same of
        // the updated image one plane further back
        float fp[kR], pp[kR], ppp[kR], sp[kR], up[kR], tpv[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) fp[r] = pp[r] = ppp[r] = sp[r] = up[r] = tpv[r] = 0.0f;
        float ring[2][NF][kR];
        auto fetch = [&](int z, float (&v)[NF][kR]) {
#pragma unroll
            for (int k = 0; k < NF; ++k) {
                const __amdgpu_buffer_rsrc_t b = rsrc(k == 0 ? f : tp.prior, z);
#pragma unroll
                for (int r = 0; r < kR; ++r)
                    v[k][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, xofs + rowofs[r], 0, 0));
            }
        };
        // n of plane z at rows lo .. hi from the plane's values c (and prior c2) and those below; n_z = value * by goes
        // to done(r, value, by, false), which completes g of the plane before, and the z-free part of g, n_z + n_y +
        // n_x - n_y(y + 1) - n_x(x + 1), to done(r, value, 1, true) for rows lo .. hi - 1
        auto differences = [&](int z, auto lo_, auto hi_, const float (&c)[kR], const float (&c2)[kR],
                               const float (&below)[kR], const float (&below2)[kR], auto&& done) {
            constexpr int lo = decltype(lo_)::value, hi = decltype(hi_)::value, kB = kTvBatch < hi - lo + 1 ? kTvBatch : hi - lo + 1;
            const bool has_z = z >= 1 && z < nz;
            float keep = 0.0f;
#pragma unroll
            for (int r0 = lo; r0 <= hi; r0 += kB) {
                float n[kB][3], s[kB];
#pragma unroll
                for (int k = 0; k < NF; ++k) {
                    float v[kB], b[kB], u[kB], t[kB][3];
#pragma unroll
                    for (int i = 0; i < kB; ++i) {
                        const int r = r0 + i <= hi ? r0 + i : hi;
                        v[i] = k == 0 ? c[r] : c[r] - c2[r];
                        b[i] = k == 0 ? below[r] : below[r] - below2[r];
                        u[i] = k == 0 ? c[r - 1] : c[r - 1] - c2[r - 1];
                    }
                    n_field<kKind>(v, b, u, has_z, tp, t, s);
#pragma unroll
                    for (int i = 0; i < kB; ++i)
#pragma unroll
                        for (int q = 0; q < 3; ++q) {
                            const float m = NF == 2 && q == 0 ? t[i][0] * s[i] : t[i][q];
                            n[i][q] = NF == 1   ? m
                                      : k == 0 ? (1.0f - tp.ratio) * m
                                               : fmaf(tp.ratio, m, n[i][q]);
                        }
                }
                // n_z + n_y.  n is discontinuous where all differences vanish, so another rounding of g than the one results
                // have always had moves single voxels by 1e-3 of the range after some iterations: here that is the
                // rounded product, and in every sixteenth plane the fused one.  (No more exact than one form in all planes,
                // and the bits depend on where the image starts in z: the rounded product throughout moved one of 25
                // images of 256^3 by 1.6e-3, the same n_z for the voxel and its neighbour 19 of 80 images by up to 9.4e-3.)
                float zy[kB];
                if (NF == 1 && (z & 15) == 0) {
#pragma unroll
                    for (int i = 0; i < kB; ++i) zy[i] = fmaf(n[i][0], s[i], n[i][1]);
                } else {
#pragma clang fp contract(off)
#pragma unroll
                    for (int i = 0; i < kB; ++i) zy[i] = (NF == 1 ? n[i][0] * s[i] : n[i][0]) + n[i][1];
                }
#pragma unroll
                for (int i = 0; i < kB; ++i) {
                    const int r = r0 + i;
                    if (r > hi) break;
                    if (r > lo) done(r - 1, keep - n[i][1], 1.0f, true);
                    done(r, n[i][0], NF == 1 ? s[i] : 1.0f, false);
                    keep = zy[i] + n[i][2] - lane_after(n[i][2]);
                }
            }
        };
        // the passes' planes: p reads f, p - 1 is updated, p - 2 adds to the norm
        constexpr int kLead = kUpdate && kNorm ? 1 : 0;
        constexpr int kLow = kNorm ? 1 : 2;  // rows from which the updated image is formed
        const int begin = z0 - kLead, end = z1 + kLead;
        auto step = [&](int p, float (&v)[NF][kR]) {
            float u[kR];  // the image whose norm is taken, plane q
            float cu[kR], cu2[kR];
#pragma unroll
            for (int r = 0; r < kR; ++r) {
                cu[r] = v[0][r];
                cu2[r] = NF == 2 ? v[NF - 1][r] : 0.0f;
            }
            if (kUpdate) {
                const float alpha_p = p >= 1 && p <= nz ? scale : 0.0f;  // the zero slices stay 0
                differences(p, Int<kLow>{}, Int<kR - kLow>{}, cu, cu2, fp, pp, [&](int r, float val, float by, bool rest) {
                    if (rest) {
                        sp[r] = val;
                    } else {
                        u[r] = fmaf(-alpha_p, fmaf(-val, by, sp[r]), fp[r]);
                    }
                });
#pragma unroll
                for (int r = kLow; r < kR - kLow; ++r) formed(sp[r]);
                if (kNorm) {  // copies of the edge voxels beyond the edges, as the loads give them
                    if (low_y) u[1] = u[2];
                    if (high_y) {
#pragma unroll
                        for (int r = 2; r < kR; ++r)
                            if (y0 + r >= ny) u[r] = u[r - 1];
                    }
                    if (low_x) {
#pragma unroll
                        for (int r = 1; r < kR; ++r) {
                            const float next = lane_after(u[r]);
                            u[r] = x < 0 ? next : u[r];
                        }
                    }
                    if (high_x) {
#pragma unroll
                        for (int r = 1; r < kR; ++r) {
                            const float before = lane_before(u[r]);
                            u[r] = x == nx ? before : u[r];
                        }
                    }
                }
                if (p > z0 && p <= z1) {
                    const __amdgpu_buffer_rsrc_t b = rsrc(out, p - 1);
                    if (core) {
#pragma unroll
                        for (int r = 2; r < kR - 2; ++r)
                            if (y0 + r < ny)
                                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(u[r]), b, xofs + rowofs[r], 0, 0);
                    }
                }
            }
            if (kNorm) {
                const int q = kUpdate ? p - 1 : p;
                const bool counts = q > z0 && q <= z1;
                if (!kUpdate) {
#pragma unroll
                    for (int r = 0; r < kR; ++r) u[r] = cu[r];
                }
                float c2[kR];
#pragma unroll
                for (int r = 0; r < kR; ++r) c2[r] = kUpdate ? pp[r] : cu2[r];
                float g[kR];
                differences(q, Int<2>{}, Int<kR - 2>{}, u, c2, up, ppp, [&](int r, float val, float by, bool rest) {
                    if (rest) {
                        tpv[r] = val;
                    } else if (r < kR - 2) {
                        g[r] = fmaf(-val, by, tpv[r]);
                    }
                });
                if (high_y) {
#pragma unroll
                    for (int r = 3; r < kR - 2; ++r)
                        if (y0 + r >= ny) g[r] = 0.0f;
                }
                float sum = g[2] * g[2];
#pragma unroll
                for (int r = 3; r < kR - 2; ++r) sum = fmaf(g[r], g[r], sum);
                if (counts) total += core ? (double)sum : 0.0;
#pragma unroll
                for (int r = 0; r < kR; ++r) {
                    up[r] = u[r];
                    ppp[r] = c2[r];
                }
            }
#pragma unroll
            for (int r = 0; r < kR; ++r) {
                fp[r] = cu[r];
                pp[r] = cu2[r];
            }
            fetch(min(p + 2, end), v);
        };
        {
            float v[NF][kR];
            fetch(begin - 1, v);
            fetch(begin, ring[0]);
            fetch(min(begin + 1, end), ring[1]);
            if (kUpdate && tile == first) read_scale();
#pragma unroll
            for (int r = 0; r < kR; ++r) {
                fp[r] = v[0][r];
                pp[r] = v[NF - 1][r];
                if (!kUpdate) {
                    up[r] = fp[r];
                    ppp[r] = pp[r];
                }
            }
        }
        for (int p = begin; p <= end; p += 2) {
            step(p, ring[0]);
            if (p + 1 <= end) step(p + 1, ring[1]);
        }
    }
    if (kNorm) {
        const double sum = block_sum(total);
        if (threadIdx.x == 0) partial_out[blockIdx.x] = sum;
    }
}

namespace {
long long ceil_div(long long a, long long b) { return (a + b - 1) / b; }

// Planes of a chunk for `column` tiles a chunk of planes, each with `halo` planes beyond its own.  A CU takes one
// workgroup of four tiles after another, and up to four at a time in about that multiple of the time of one (one or two
// leave it waiting for its own loads and chains: 1.4 and 1.08); the chunks that cost a CU the least
// are taken.  Measured, us for 20 iterations (tiles): 320^3 1654 (2880), 1672 (1920), 1808 (2400), 1917 (3120); 400^3
// 3121 (2800), 3387 (1750), 3789 (3150); 512^3 6315 (4032), 6422 (2880), 6908 (1728), 9767 (4608).
int tv_chunk(long long column, long long nz, int halo) {
    int chunk = (int)nz;
    double best = INFINITY;
    for (int most = 1; most <= 64; most += most < 4 ? 1 : 4) {  // workgroups a CU: as many chunks as that allows
        const long long chunks = std::max(1LL, std::min(256LL * kTvWaves * most / column, nz / 4));
        const long long planes = ceil_div(nz, chunks), groups = ceil_div(column * ceil_div(nz, planes), kTvWaves);
        const long long each = groups <= kTvBlocks ? ceil_div(groups, 256) : 4 * ceil_div(groups, kTvBlocks);
        const double cost = (double)(each * (planes + halo)) * (each == 1 ? 1.4 : (each == 2 ? 1.08 : 1.0));
        if (cost < best) {
            best = cost;
            chunk = (int)planes;
        }
    }
    return chunk;
}

template <int kKind>
int run_tv_descent(const float* img, float* dst, float alpha, const TvParams& tp, double norm_eps, long nx, long ny,
                   long nz, int maxiter, hipStream_t stream) {
    TIGRE_REQUIRE(nx > 0 && ny > 0 && nz > 0, "empty image");
    // 32-bit byte offsets within a plane
    TIGRE_REQUIRE(nx * ny * nz < (1LL << 40) && nx * ny < (1LL << 30), "image too large");
    const size_t n = (size_t)nx * ny * nz;
    if (maxiter <= 0) {
        if (dst != img) TIGRE_HIP_TRY(hipMemcpyAsync(dst, img, n * sizeof(float), hipMemcpyDeviceToDevice, stream));
        return TIGRE_OK;
    }
    const long long ntx = nx <= 63 ? 1 : (nx - 63 + kTvColumns - 1) / kTvColumns + 1;
    // 8 rows a tile cost the least halo; 2 rows and chunks from 2 planes give a small volume more wavefronts and
    // shorter ones (20 iterations: 40 x 36 x 42 151 us, 240 with 8 rows; 64^3 180 and 237; 128^3, 1536 tiles of 8
    // rows, 383 and 363).
    const bool small = ntx * ((ny + 7) / 8) * ((nz + 3) / 4) < 1024;
    const int rows = small ? 2 : 8;
    const long long nty = (ny + rows - 1) / rows, column = ntx * nty;
    // Three forms.  A pass that takes the norm too evaluates n on 20 rows for 8 and 4 planes more a chunk, a pass for each
    // on 18 and 2, and moves 8 bytes a voxel instead of 12: one pass pays where the Infinity Cache no longer serves two
    // and the chunks are not mostly halo (us an iteration, one and two passes: TV 250^3 47.3 and 45.0, 320^3 80.2 and 80.4,
    // 512^3 315 and 406, 8 x 2048^2 108 and 95, 16 x 2048^2 206 and 225; PICCS 250^3 88 and 80, 300^3 125 and 120, 384^3
    // 251 and 285), and never for AwTV, which spends most on the weights' exponentials (240 x 230 x 250 69 and 55).
    // LDS tiles (tv_tiles.hip) take 1.2 to 1.5 times a wavefront tile's time for a column and plane, but have no halo to
    // speak of: they serve AwTV where wavefront tiles fill the columns badly (LDS tiles and two passes: 250^3 59 and 68,
    // 256^3 60 and 68, 384^3 192 and 198, 64 x 1024^2 226 and 248; 280^3 100 and 80, 320^3 123 and 111, 400^3 254 and 228),
    // and the others on slabs of few planes (LDS tiles and the better of the rest: TV 16 x 1024^2 46 and 50, 16 x 2048^2
    // 189 and 206, 8 x 2048^2 96 and 95; PICCS 8 x 1024^2 50 and 52, 16 x 2048^2 326 and 383, 4 x 1024^2 35 and 33).
    const bool fused = small || (kKind == 0 && n > (1u << 24) && nz > 8) || (kKind == 2 && n > (1u << 25));
    const int chunk = small ? (int)std::max(2LL, ceil_div(nz, std::max(1LL, 3072 / column)))
                            : tv_chunk(column, nz, fused ? 4 : 2);
    bool tiles = false;
    if (!small) {
        // evaluations of n an iteration, by LDS tiles and by two passes
        const double by_tiles = 16.0 * (double)(ceil_div(nx, 128) * 128 * nty) * (double)(nz + ceil_div(nz, 16));
        const double by_passes = 18.0 * (double)(64 * column) * (double)(nz + 2 * ceil_div(nz, tv_chunk(column, nz, 2)));
        const bool cheap = tv_tile_count(nx, ny, nz) >= 960 && by_tiles < 0.8 * by_passes;
        tiles = cheap && (kKind == 0 ? nz > 8 && nz <= 32 && n >= (1u << 24) : kKind == 1 ? nz >= 2 : nz >= 8 && nz <= 32);
    }
    const long long ntiles = column * ((nz + chunk - 1) / chunk);
    TIGRE_REQUIRE(ntiles < (1LL << 30), "image too large");
    const int nblocks = (int)std::min((long long)kTvBlocks, (ntiles + kTvWaves - 1) / kTvWaves);
    const size_t npartial = tiles ? (size_t)tv_tile_count(nx, ny, nz) + 1 : 2 * kTvBlocks;
    StreamScratch scratch(stream);
    float* buf[2] = {nullptr, nullptr};
    double* partial[2] = {nullptr, nullptr};
    TIGRE_CHECK(scratch.alloc(&buf[0], n * sizeof(float)));
    TIGRE_CHECK(scratch.alloc(&buf[1], n * sizeof(float)));
    TIGRE_CHECK(scratch.alloc(&partial[0], npartial * sizeof(double)));
    partial[1] = partial[0] + kTvBlocks;
    const float* src = img;
    int cur = 0;
    for (int it = 0; it < maxiter; ++it) {
        const bool last = it == maxiter - 1;
        float* o = (last && dst != img) ? dst : buf[cur];
        KernelTimerScope timer(TIGRE_KERNEL_POCS_TV, stream);
        if (tiles) {
            TIGRE_CHECK(launch_tv_tile_iteration(kKind, src, o, tp, (int)nx, (int)ny, (int)nz, alpha, norm_eps, partial[0],
                                                 reinterpret_cast<float*>(partial[0] + npartial - 1), stream));
            src = o;
            cur ^= 1;
            continue;
        }
#define TIGRE_TV(C, U, N)                                                                                          \
    hipLaunchKernelGGL((tv_kernel<kKind, C, U, N>), dim3((unsigned)nblocks), dim3(kTvThreads), 0, stream, src, o, tp, \
                       (int)nx, (int)ny, (int)nz, (int)ntx, (int)nty, chunk, (int)ntiles, alpha, norm_eps,          \
                       partial[cur], nblocks, partial[(U) ? cur ^ 1 : cur])
#define TIGRE_TV_ROWS(U, N)             \
    do {                                \
        if (rows == 8) TIGRE_TV(8, U, N); \
        else TIGRE_TV(2, U, N);         \
    } while (0)
        if (it == 0 || !fused) TIGRE_TV_ROWS(false, true);
        if (last || !fused) TIGRE_TV_ROWS(true, false);
        else TIGRE_TV_ROWS(true, true);
#undef TIGRE_TV_ROWS
#undef TIGRE_TV
        TIGRE_HIP_TRY(hipGetLastError());
        src = o;
        cur ^= 1;
    }
    if (src != dst) TIGRE_HIP_TRY(hipMemcpyAsync(dst, src, n * sizeof(float), hipMemcpyDeviceToDevice, stream));
    return TIGRE_OK;
}
}  // namespace

int run_pocs_tv(const float* img, float* dst, float alpha, long nx, long ny, long nz, int maxiter,
                hipStream_t stream) {
    return run_tv_descent<0>(img, dst, alpha, TvParams{nullptr, 0.0f, 0.0f}, 1e-7, nx, ny, nz, maxiter, stream);
}

int run_aw_pocs_tv(const float* img, float* dst, float alpha, float delta, long nx, long ny, long nz, int maxiter,
                   hipStream_t stream) {
    TIGRE_REQUIRE(delta != 0.0f, "delta must be nonzero");
    return run_tv_descent<1>(img, dst, alpha, TvParams{nullptr, 1.0f / delta, 0.0f}, 1e-7, nx, ny, nz, maxiter,
                             stream);
}

int run_piccs_tv(const float* img, const float* prior, float* dst, float alpha, float ratio, long nx, long ny, long nz,
                 int maxiter, hipStream_t stream) {
    return run_tv_descent<2>(img, dst, alpha, TvParams{prior, 0.0f, ratio}, 0.0, nx, ny, nz, maxiter, stream);
}

// ---------------------------------------------------------------------------
// ROF primal-dual denoise, tv_proximal.cu:81-181 (kernels) and :436-502 (loop).
// Domain: nz + 2 slices; slice 0 mirrors image slice 1, slices 1..nz hold the
// image, slice nz + 1 is zero (the single-device layout of cpy_from_host,
// tv_proximal.cu:672-693).  All slices evolve; slices 1..nz are returned.
// ---------------------------------------------------------------------------
//
// A pass runs kT iterations.  A workgroup of eight wavefronts holds a tile of 64 columns (one per lane) by
// 8 kRows rows, a halo of kT on every side, and marches along z; a pass reads the image and the
// state (u, px, py, pz in one float4) once and writes the state once, 36 bytes a voxel for kT iterations and not
// 52 for each.  Iteration k of the pass computes u_k at plane z_k = s - 2 (k - 1) in step s, and p_k one
// plane below, so that all it needs was computed in earlier steps: p_{k-1}(z_k) in the step before,
// u_{k-1}(z_k) two before.  The two last generations stay in registers, x neighbours come by wavefront
// shifts, y neighbours from the lane's own rows or, between wavefronts, from LDS rows that are written at the end of a
// step and read in the next: one barrier a step.  Columns and rows within k of the tile's edge are
// wrong after k iterations and are not stored; the volume's own edges drop terms where the reference does.
// The first pass starts from u = f, p = 0 without reading a state; the last one writes u to the result and
// computes no last p.
//
// Measured at 150 x 181 x 170, 50 iterations: 684 us, 2.60 ms with one kernel for u and one for p an
// iteration (13 array passes at 4.2 TB/s; their index arithmetic divided by nx and ny in 64 bits).  A pass of
// three iterations takes 40 us, about 28 of them VALU time with the halo's share (1.9 times the voxels).
// 2 x 8, 3 x 8 rows, 2 or 4 iterations a pass: 0.69 to 1.2 ms.
namespace {
constexpr int kRofWaves = 8;

template <int kT>
struct RofSteps {
    float tau1[kT], tau2[kT];
};

struct RofP {
    float x, y, z;
};
}  // namespace

template <int kT, int kRows, bool kFirst, bool kLast>
__global__ __launch_bounds__(64 * kRofWaves) void rof_kernel(const float* __restrict__ src, const float4* __restrict__ in,
                                                            float4* __restrict__ out, float* __restrict__ dst, int nx,
                                                            int ny, int nz, int chunk, RofSteps<kT> tau,
                                                            float inv_lambda, float idx, float idy, float idz) {
    constexpr int kY = kRofWaves * kRows;
    // rows that cross a wavefront's edge: last row of p_{k-1}.y (for u_k) and first row of u_k (for p_k)
    __shared__ float rows[2][kT][2][kRofWaves][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int D = nz + 2;
    const int tilesX = (nx + 64 - 2 * kT - 1) / (64 - 2 * kT), tilesY = (ny + kY - 2 * kT - 1) / (kY - 2 * kT);
    const int L = xcd_logical_block((int)blockIdx.x, (int)gridDim.x);
    const int x = (L % tilesX) * (64 - 2 * kT) - kT + lane;
    const int y0 = ((L / tilesX) % tilesY) * (kY - 2 * kT) - kT + wave * kRows;
    const int z0 = (L / (tilesX * tilesY)) * chunk, z1 = min(z0 + chunk, D);
    const long long plane = (long long)nx * ny;
    const bool x_first = x == 0, x_last = x == nx - 1;
    const float sx = x_first ? 1.0f : idx;
    // stored columns and rows
    const bool x_mine = lane >= kT && lane < 64 - kT && x < nx;
    unsigned at[kRows];  // offset in a plane, clamped into it
    bool mine[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int y = y0 + r, row = wave * kRows + r;
        at[r] = (unsigned)min(max(y, 0), ny - 1) * (unsigned)nx + (unsigned)min(max(x, 0), nx - 1);
        mine[r] = x_mine && row >= kT && row < kY - kT && y < ny;
    }

    // image at plane z of the extended domain, and the state
    auto load_f = [&](int z, float (&v)[kRows]) {
        z = min(max(z, 0), D - 1);
        // slice 0 mirrors image slice 1 (0 in an image of one slice), slice nz + 1 is 0
        const int zi = z == 0 ? 1 : z - 1;
        const float* f = src + (long long)min(zi, nz - 1) * plane;
#pragma unroll
        for (int r = 0; r < kRows; ++r) v[r] = zi < nz ? f[at[r]] : 0.0f;
    };
    auto load_state = [&](int z, float4 (&v)[kRows]) {
        const float4* q = in + (long long)min(max(z, 0), D - 1) * plane;
#pragma unroll
        for (int r = 0; r < kRows; ++r) v[r] = q[at[r]];
    };

    // The last two generations by the parity of the step, so that none is moved: in a step of parity q,
    // P[k][r][q] was computed one step ago and P[k][r][!q] two (k = 0: planes s and s - 1), U[k][r] likewise
    // for u_k, k >= 1.  F[q][j][r]: the image 2 j planes back.
    RofP P[kT][kRows][2];
    float U[kT + 1][kRows][2], F[2][kT][kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
#pragma unroll
            for (int k = 0; k < kT; ++k) {
                P[k][r][g] = RofP{0.0f, 0.0f, 0.0f};
                F[g][k][r] = 0.0f;
            }
#pragma unroll
            for (int k = 0; k <= kT; ++k) U[k][r][g] = 0.0f;
        }
    const int s0 = max(z0 - kT, 0), s1 = z1 + 2 * kT - 2;
    float nf[kRows];   // loaded ahead: image and state of the next plane
    float4 nq[kRows];
    load_f(s0, nf);
    if (!kFirst) load_state(s0, nq);
    const bool y_edge = y0 < 1 || y0 + kRows >= ny;

    // Step s of parity kQ; kEdge: a row or plane may lie on or outside the volume's y or z faces.
    auto step = [&](int s, auto parity, auto edge) {
        constexpr int kQ = decltype(parity)::value;
        constexpr bool kEdge = decltype(edge)::value;
        // the loaded plane
        float u0[kRows];
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            if (!kFirst) P[0][r][kQ] = RofP{nq[r].y, nq[r].z, nq[r].w};
#pragma unroll
            for (int j = kT - 1; j > 0; --j) F[kQ][j][r] = F[kQ][j - 1][r];
            F[kQ][0][r] = nf[r];
            u0[r] = kFirst ? nf[r] : nq[r].x;
        }
        if (s < s1) {  // past the domain the last plane again
            load_f(s + 1, nf);
            if (!kFirst) load_state(s + 1, nq);
        }
        // the last iteration first: each uses its predecessor's results of earlier steps
#pragma unroll
        for (int k = kT; k >= 1; --k) {
            const int z = s - 2 * (k - 1);
            const float t1 = tau.tau1[k - 1], t2 = tau.tau2[k - 1];
            const float py_edge = rows[kQ][k - 1][0][max(wave - 1, 0)][lane];
            const float u_edge = rows[kQ][k - 1][1][min(wave + 1, kRofWaves - 1)][lane];
            float un[kRows];
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                const int y = y0 + r;
                const RofP& p = P[k - 1][r][kQ];
                const float pyl = r > 0 ? P[k - 1][r > 0 ? r - 1 : 0][kQ].y : py_edge, pzl = P[k - 1][r][kQ ^ 1].z;
                const float dx = p.x - lane_before(p.x);
                float dv = !kEdge || z >= 1 ? (p.z - pzl) * idz : p.z;
                dv = !kEdge || y >= 1 ? fmaf(p.y - pyl, idy, dv) : dv + p.y;
                dv = fmaf(x_first ? p.x : dx, sx, dv);
                const float ui = k == 1 ? u0[r] : U[k - 1][r][kQ ^ 1];
                // t1 is negative in the first iterations: the larger term is the one that is not rounded first
                un[r] = fmaf(ui, 1.0f - t1, t1 * fmaf(inv_lambda, dv, F[kQ][k - 1][r]));
            }
            const bool store = z - 1 >= z0 && z - 1 < z1;  // uniform
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                const int y = y0 + r;
                const float u = U[k][r][kQ];  // u_k at plane z - 1
                RofP q{0.0f, 0.0f, 0.0f};
                if (!(kLast && k == kT)) {
                    const float uy = r < kRows - 1 ? U[k][r < kRows - 1 ? r + 1 : r][kQ] : u_edge;
                    const float dx = lane_after(u) - u;
                    const RofP& p = P[k - 1][r][kQ ^ 1];
                    q.z = fmaf(t2 * idz, !kEdge || z < D ? un[r] - u : 0.0f, p.z);
                    q.y = fmaf(t2 * idy, !kEdge || y + 1 < ny ? uy - u : 0.0f, p.y);
                    q.x = fmaf(t2 * idx, x_last ? 0.0f : dx, p.x);
                    // 1 / max(1, |q|); q = 0 gives 1.  Errors from FP64 as with a square root and divisions, geometric means
                    // over 24 cases a spacing: 1.0924e-7 and 1.0943e-7 (spacing 1), 1.5549e-7 and 1.5562e-7 (0.3 to 0.9);
                    // 150 x 181 x 170, 50 iterations: 669 and 1249 us.
                    const float inv = fminf(1.0f, __builtin_amdgcn_rsqf(fmaf(q.z, q.z, fmaf(q.y, q.y, q.x * q.x))));
                    q.z *= inv;
                    q.y *= inv;
                    q.x *= inv;
                }
                if (k == kT) {
                    if (store && mine[r]) {
                        if (!kLast)
                            out[(long long)(z - 1) * plane + at[r]] = make_float4(u, q.x, q.y, q.z);
                        else if (z - 1 >= 1 && z - 1 <= nz)
                            dst[(long long)(z - 2) * plane + at[r]] = u;
                    }
                } else {
                    P[k < kT ? k : 0][r][kQ ^ 1] = q;
                }
            }
#pragma unroll
            for (int r = 0; r < kRows; ++r) U[k][r][kQ ^ 1] = un[r];
        }
        // rows of the next step
#pragma unroll
        for (int k = 0; k < kT; ++k) {
            rows[kQ ^ 1][k][0][wave][lane] = k == 0 ? (kFirst ? 0.0f : nq[kRows - 1].z) : P[k][kRows - 1][kQ ^ 1].y;
            rows[kQ ^ 1][k][1][wave][lane] = U[k + 1][0][kQ ^ 1];
        }
        __syncthreads();
    };
    // the rows that the first step reads
#pragma unroll
    for (int k = 0; k < kT; ++k) {
        rows[0][k][0][wave][lane] = k == 0 && !kFirst ? nq[kRows - 1].z : 0.0f;
        rows[0][k][1][wave][lane] = 0.0f;
    }
    __syncthreads();
    auto any_step = [&](int s, auto parity) {
        if (y_edge || s < 2 * kT - 1 || s >= D)  // uniform per wavefront; both branches pass the same barrier
            step(s, parity, std::true_type{});
        else
            step(s, parity, std::false_type{});
    };
    for (int s = s0; s <= s1; s += 2) {
        any_step(s, std::integral_constant<int, 0>{});
        if (s + 1 <= s1) any_step(s + 1, std::integral_constant<int, 1>{});
    }
}

namespace {
constexpr int kRofT = 3, kRofRows = 2, kRofSlots = 512;  // two workgroups fit a CU

// Step sizes of iterations it, it + 1, .. (tv_proximal.cu:478-479), evaluated in float as there.
template <int kT>
RofSteps<kT> rof_steps(int it) {
    RofSteps<kT> tau;
    for (int k = 0; k < kT; ++k) {
        tau.tau2[k] = 0.3f + 0.02f * (float)(it + k);
        tau.tau1[k] = (1.f / tau.tau2[k]) * ((1.f / 6.f) - (5.f / (15.f + (float)(it + k))));
    }
    return tau;
}

// One pass of kT iterations from iteration `it` on.
template <int kT>
int rof_pass(const float* src, const float4* in, float4* out, float* dst, float inv_lambda, const float* spacing, int nx,
             int ny, int nz, int it, bool first, bool last, hipStream_t stream) {
    const RofSteps<kT> tau = rof_steps<kT>(it);
    constexpr int kX = 64 - 2 * kT, kY = kRofWaves * kRofRows - 2 * kT;
    const long long tiles = (long long)((nx + kX - 1) / kX) * ((ny + kY - 1) / kY);
    const int D = nz + 2;
    // Planes per workgroup: a workgroup of c planes runs c + 3 kT - 1 steps, and kRofSlots workgroups run at
    // once; the smallest number of rounds times steps, of the most chunks that each number of rounds allows (50
    // iterations against multiples of four planes: 256^3 2.76 and 2.88 ms, 37 and 24 planes; 100^3 345 and 404 us, 5
    // and 8).  No more than 128 planes: the last workgroups of a single round hold up the pass (512^3, 514 and 104
    // planes: 8.04 and 7.88 ms, 20 iterations).
    int chunk = D;
    long long cost = -1;
    for (int most = 1; most <= 16; ++most) {
        const long long chunks =
            std::max(ceil_div(D, 128), std::min((long long)most * kRofSlots / tiles, (long long)(D + 3) / 4));
        const int c = (int)ceil_div(D, chunks);
        const long long rounds = ceil_div(tiles * ceil_div(D, c), kRofSlots);
        const long long t = rounds * (c + 3 * kT - 1);
        if (cost < 0 || t < cost) {
            cost = t;
            chunk = c;
        }
    }
    const long long blocks = tiles * ((D + chunk - 1) / chunk);
    TIGRE_REQUIRE(blocks < (1LL << 31), "image too large");
    const dim3 grid((unsigned)blocks), threads(64 * kRofWaves);
    const float ix = 1.0f / spacing[0], iy = 1.0f / spacing[1], iz = 1.0f / spacing[2];
    KernelTimerScope timer(TIGRE_KERNEL_TVDENOISE, stream);
#define TIGRE_ROF(F, E)                                                                                            \
    hipLaunchKernelGGL((rof_kernel<kT, kRofRows, F, E>), grid, threads, 0, stream, src, in, out, dst, nx, ny, nz, \
                       chunk, tau, inv_lambda, ix, iy, iz)
    if (last) {
        if (first) TIGRE_ROF(true, true);
        else TIGRE_ROF(false, true);
    } else if constexpr (kT == kRofT) {  // only the last pass runs fewer iterations
        if (first) TIGRE_ROF(true, false);
        else TIGRE_ROF(false, false);
    }
#undef TIGRE_ROF
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

// One iteration on a single state, u and then p in place, with the operations of rof_kernel in its order and so with its
// bits.  It serves volumes whose two states do not fit into memory (20 bytes a voxel with the image's copy of a call in
// place, 36 with two states): 150 x 181 x 170, 50 iterations 3.9 ms a call, 0.86 with two states.
constexpr int kRofPlainBlocks = 16384;
template <bool kFirst>
__global__ __launch_bounds__(256) void rof_u_kernel(const float* __restrict__ src, float4* __restrict__ state, int nx,
                                                    int ny, int nz, float t1, float inv_lambda, float idx, float idy,
                                                    float idz) {
    const long long plane = (long long)nx * ny, n = plane * (nz + 2);
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < n; q += (long long)gridDim.x * 256) {
        const int z = (int)(q / plane);
        const long long r = q - z * plane;
        const int y = (int)(r / nx), x = (int)(r - (long long)y * nx);
        const int zi = z == 0 ? 1 : z - 1;  // slice 0 mirrors image slice 1, slice nz + 1 is 0
        const float f = zi < nz ? src[zi * plane + r] : 0.0f;
        float px = 0.0f, py = 0.0f, pz = 0.0f, pxl = 0.0f, pyl = 0.0f, pzl = 0.0f;
        if (!kFirst) {
            px = state[q].y, py = state[q].z, pz = state[q].w;
            if (x >= 1) pxl = state[q - 1].y;
            if (y >= 1) pyl = state[q - nx].z;
            if (z >= 1) pzl = state[q - plane].w;
        }
        float dv = z >= 1 ? (pz - pzl) * idz : pz;
        dv = y >= 1 ? fmaf(py - pyl, idy, dv) : dv + py;
        dv = fmaf(x >= 1 ? px - pxl : px, x >= 1 ? idx : 1.0f, dv);
        state[q].x = fmaf(kFirst ? f : state[q].x, 1.0f - t1, t1 * fmaf(inv_lambda, dv, f));
    }
}

template <bool kFirst>
__global__ __launch_bounds__(256) void rof_p_kernel(float4* __restrict__ state, int nx, int ny, int nz, float t2, float idx,
                                                    float idy, float idz) {
    const long long plane = (long long)nx * ny, n = plane * (nz + 2);
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < n; q += (long long)gridDim.x * 256) {
        const int z = (int)(q / plane);
        const long long r = q - z * plane;
        const int y = (int)(r / nx), x = (int)(r - (long long)y * nx);
        const float u = state[q].x;
        RofP p{0.0f, 0.0f, 0.0f};
        if (!kFirst) p = RofP{state[q].y, state[q].z, state[q].w};
        p.z = fmaf(t2 * idz, z + 1 < nz + 2 ? state[q + plane].x - u : 0.0f, p.z);
        p.y = fmaf(t2 * idy, y + 1 < ny ? state[q + nx].x - u : 0.0f, p.y);
        p.x = fmaf(t2 * idx, x + 1 < nx ? state[q + 1].x - u : 0.0f, p.x);
        const float inv = fminf(1.0f, __builtin_amdgcn_rsqf(fmaf(p.z, p.z, fmaf(p.y, p.y, p.x * p.x))));
        state[q].y = p.x * inv;
        state[q].z = p.y * inv;
        state[q].w = p.z * inv;
    }
}

__global__ __launch_bounds__(256) void rof_u_out_kernel(const float4* __restrict__ state, float* __restrict__ dst, long long n) {
    for (long long q = (long long)blockIdx.x * 256 + threadIdx.x; q < n; q += (long long)gridDim.x * 256) dst[q] = state[q].x;
}

// All iterations on one state; src and dst may overlap if `overlap`.
int run_tvdenoise_plain(const float* src, float* dst, float inv_lambda, const float* spacing, int nx, int ny, int nz,
                        int maxiter, bool overlap, StreamScratch& scratch, hipStream_t stream) {
    const size_t plane = (size_t)nx * ny, n = plane * (nz + 2);
    float4* state = nullptr;
    if (!scratch.try_alloc(&state, n * sizeof(float4))) {  // a block that work still uses can be had once it is done
        TIGRE_HIP_TRY(hipStreamSynchronize(stream));
        TIGRE_CHECK(scratch.alloc(&state, n * sizeof(float4)));
    }
    if (overlap) {  // every iteration reads the image; the result is written once, after the last
        float* image = nullptr;
        TIGRE_CHECK(scratch.alloc(&image, plane * nz * sizeof(float)));
        TIGRE_HIP_TRY(hipMemcpyAsync(image, src, plane * nz * sizeof(float), hipMemcpyDeviceToDevice, stream));
        src = image;
    }
    const dim3 grid((unsigned)std::min<size_t>((n + 255) / 256, kRofPlainBlocks)), threads(256);
    const float ix = 1.0f / spacing[0], iy = 1.0f / spacing[1], iz = 1.0f / spacing[2];
    for (int it = 0; it < maxiter; ++it) {
        const RofSteps<1> tau = rof_steps<1>(it);
        KernelTimerScope timer(TIGRE_KERNEL_TVDENOISE, stream);
#define TIGRE_ROF_PLAIN(F)                                                                                          \
    do {                                                                                                            \
        hipLaunchKernelGGL(rof_u_kernel<F>, grid, threads, 0, stream, src, state, nx, ny, nz, tau.tau1[0],           \
                           inv_lambda, ix, iy, iz);                                                                 \
        if (it + 1 < maxiter)                                                                                       \
            hipLaunchKernelGGL(rof_p_kernel<F>, grid, threads, 0, stream, state, nx, ny, nz, tau.tau2[0], ix, iy, iz); \
    } while (0)
        if (it == 0) TIGRE_ROF_PLAIN(true);
        else TIGRE_ROF_PLAIN(false);
#undef TIGRE_ROF_PLAIN
    }
    hipLaunchKernelGGL(rof_u_out_kernel, grid, threads, 0, stream, state + plane, dst, (long long)(plane * nz));
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}
}  // namespace

int run_tvdenoise(const float* src, float* dst, float lambda, const float* spacing, long nx, long ny, long nz,
                  int maxiter, hipStream_t stream) {
    TIGRE_REQUIRE(nx > 0 && ny > 0 && nz > 0, "empty image");
    TIGRE_REQUIRE(nx < (1LL << 31) && ny < (1LL << 31) && nx * ny < (1LL << 32) && nz < (1LL << 31) - 128, "image too large");
    const size_t out_bytes = (size_t)nz * ny * nx * sizeof(float);
    if (maxiter <= 0) {
        if (dst != src) TIGRE_HIP_TRY(hipMemcpyAsync(dst, src, out_bytes, hipMemcpyDeviceToDevice, stream));
        return TIGRE_OK;
    }
    const size_t n = (size_t)(nz + 2) * nx * ny;
    StreamScratch scratch(stream);
    const int passes = (maxiter + kRofT - 1) / kRofT;
    float4* state[2] = {nullptr, nullptr};
    // every pass reads the image: a result that overlaps it goes through scratch
    float* to = dst;
    const char *sb = reinterpret_cast<const char*>(src), *db = reinterpret_cast<const char*>(dst);
    const bool overlap = sb < db + out_bytes && db < sb + out_bytes;
    const float inv_lambda = 1.0f / lambda;
    bool fits = true;
    for (int k = 0; k < 2 && k < passes - 1; ++k) fits = fits && scratch.try_alloc(&state[k], n * sizeof(float4));
    if (overlap) fits = fits && scratch.try_alloc(&to, out_bytes);
    if (!fits) {
        scratch.release();
        return run_tvdenoise_plain(src, dst, inv_lambda, spacing, (int)nx, (int)ny, (int)nz, maxiter, overlap, scratch, stream);
    }
    for (int p = 0, it = 0; p < passes; ++p) {
        const int t = std::min(kRofT, maxiter - it);
        const float4* in = p > 0 ? state[(p - 1) & 1] : nullptr;
        float4* out = p < passes - 1 ? state[p & 1] : nullptr;
        const bool first = p == 0, last = p == passes - 1;
        const int X = (int)nx, Y = (int)ny, Z = (int)nz;
        if (t == 1) TIGRE_CHECK(rof_pass<1>(src, in, out, to, inv_lambda, spacing, X, Y, Z, it, first, last, stream));
        else if (t == 2) TIGRE_CHECK(rof_pass<2>(src, in, out, to, inv_lambda, spacing, X, Y, Z, it, first, last, stream));
        else TIGRE_CHECK(rof_pass<3>(src, in, out, to, inv_lambda, spacing, X, Y, Z, it, first, last, stream));
        it += t;
    }
    if (overlap) TIGRE_HIP_TRY(hipMemcpyAsync(dst, to, out_bytes, hipMemcpyDeviceToDevice, stream));
    return TIGRE_OK;
}

}  // namespace tigre
