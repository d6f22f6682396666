// 3D convolutions of the learned proximal network, BF16 MFMA on gfx950.
//
// The network (a residual CNN that stands in for the TV step of ASD-POCS) is
// six 3x3x3 'same' convolutions with 32 channels between them.  All of them,
// forward and backward, run as implicit GEMMs on v_mfma_f32_16x16x32_bf16
// (A: 16 rows x 32 k, B: 32 k x 16 columns, FP32 accumulate; lane l holds
// row / column l % 16 and k = 8 (l / 16) .. + 7, and result register r of lane
// l is row 4 (l / 16) + r, column l % 16):
//
//  * conv_zm_kernel (32 -> 32 channels): rows 16 output channels, columns 16
//    voxels along x, k one tap's 32 input channels; the weights in registers,
//    input planes staged in LDS once each while the workgroup marches along z.
//  * conv_taps_kernel (one FP32 channel -> 32): k is the tap instead, so one
//    MFMA covers all 27 taps of 16 voxels.
//  * conv_out_kernel (32 -> one FP32 channel added to a residual input): the
//    taps are the columns instead, P[u][tap] for every input voxel, then
//    in-plane tap sums in LDS.
//  * conv_kernel: the plain gather form (one 16-byte load per lane per tap is
//    an A fragment), for the single-channel input with the residual epilogue.
//  * wgrad_kernel: dw[tap][o][i] = sum_v x[v + tap][i] dy[v][o], GEMM k =
//    32 voxels of an x-row, read from LDS with the transposing eight-byte
//    reads; all taps in one workgroup.  Tap 27 is the bias: x replaced by 1
//    in channel 0, so dw[27][o][0] = sum_v dy[v][o].
//
// Volumes are N x D x H x W (x fastest); taps index (dz, dy, dx) in
// {-1, 0, 1}^3 as 9 (dz + 1) + 3 (dy + 1) + (dx + 1); outside the volume the
// input is zero.
#include <mutex>
#include <type_traits>

#include "common.hpp"

namespace tigre {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kC = 32;            // channels between layers
constexpr int kTilesPerWave = 4;  // 16-voxel tiles per wavefront (64 voxels along x)

// Round to nearest even; infinities keep their bits and NaNs stay NaN (quiet
// bit set when the dropped half of the significand was not zero).  Both
// results are computed and one selected, so a store loop has no branches.
__device__ __forceinline__ unsigned short bf16_bits(float f) {
    const unsigned u = __float_as_uint(f);
    const unsigned special = (u >> 16) | ((u & 0xffffu) ? 0x40u : 0u);
    const unsigned rounded = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
    return (unsigned short)((u & 0x7f800000u) == 0x7f800000u ? special : rounded);
}

// A fragment of 8 channels (8 q .. 8 q + 7) of voxel `vox`, or zeros.
template <int kIn>
__device__ __forceinline__ bf16x8 load_frag(const void* __restrict__ src, long long vox, int q, bool ok) {
    bf16x8 f;
    if (kIn == TIGRE_CNN_IN_BF16X32) {
        uint4 raw = make_uint4(0u, 0u, 0u, 0u);
        if (ok) raw = *reinterpret_cast<const uint4*>(static_cast<const unsigned short*>(src) + vox * kC + 8 * q);
        f = __builtin_bit_cast(bf16x8, raw);
    } else {
        float v = 0.0f;
        if (ok && q == 0) v = static_cast<const float*>(src)[vox];
        uint4 raw = make_uint4((unsigned)bf16_bits(v), 0u, 0u, 0u);
        f = __builtin_bit_cast(bf16x8, raw);
    }
    return f;
}

template <int kIn, int kEpi>
__global__ __launch_bounds__(256) void conv_kernel(const void* __restrict__ x, const unsigned short* __restrict__ w,
                                                   const float* __restrict__ bias, const void* __restrict__ aux,
                                                   void* __restrict__ y, int N, int D, int H, int W) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, q = lane >> 4;
    const long long row = (long long)blockIdx.y * 4 + wave;  // (n, z, y) row of the wavefront
    const long long rows = (long long)N * D * H;
    if (row >= rows) return;  // uniform per wavefront
    const int yy0 = (int)(row % H), zz0 = (int)((row / H) % D);
    const long long n = row / ((long long)H * D);
    const int x0 = blockIdx.x * (16 * kTilesPerWave);

    f32x4 acc[kTilesPerWave][2];
#pragma unroll
    for (int t = 0; t < kTilesPerWave; ++t) acc[t][0] = acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int tap = 0; tap < 27; ++tap) {
        const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
        const int zz = zz0 + dz, yy = yy0 + dy;
        const bool row_ok = zz >= 0 && zz < D && yy >= 0 && yy < H;
        const long long base = ((n * D + zz) * H + yy) * (long long)W;
        const unsigned short* wt = w + (long long)tap * kC * kC;
        const bf16x8 b0 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(wt + m * kC + 8 * q));
        const bf16x8 b1 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(wt + (16 + m) * kC + 8 * q));
#pragma unroll
        for (int t = 0; t < kTilesPerWave; ++t) {
            const int xx = x0 + 16 * t + m + dx;
            const bf16x8 a = load_frag<kIn>(x, base + xx, q, row_ok && xx >= 0 && xx < W);
            acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b0, acc[t][0], 0, 0, 0);
            acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b1, acc[t][1], 0, 0, 0);
        }
    }

    const long long obase = row * (long long)W;
#pragma unroll
    for (int t = 0; t < kTilesPerWave; ++t) {
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            const int o = hb * 16 + m;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int xo = x0 + 16 * t + 4 * q + r;
                if (xo >= W) continue;
                const long long vox = obase + xo;
                float v = acc[t][hb][r];
                if (kEpi == TIGRE_CNN_EPI_BIAS_RELU) {
                    v += bias[o];
                    v = v > 0.0f ? v : 0.0f;
                    static_cast<unsigned short*>(y)[vox * kC + o] = bf16_bits(v);
                } else if (kEpi == TIGRE_CNN_EPI_RELU_MASK) {
                    const unsigned short a = static_cast<const unsigned short*>(aux)[vox * kC + o];
                    v = (a != 0 && (a & 0x8000u) == 0) ? v : 0.0f;  // activation > 0
                    static_cast<unsigned short*>(y)[vox * kC + o] = bf16_bits(v);
                } else {  // residual output: channel 0 only, FP32
                    if (o == 0) static_cast<float*>(y)[vox] = static_cast<const float*>(aux)[vox] + (v + bias[0]);
                }
            }
        }
    }
}

// Staged input blocks.  A workgroup computes 4 output rows; the 6-row block
// of an input plane its taps read (with one halo voxel on either side along x)
// is copied into LDS, voxels outside the volume as zeros.
constexpr int kLdsTiles = 8;                    // 16-voxel tiles per workgroup row (single channel)
constexpr int kLdsBX = 16 * kLdsTiles + 2;      // staged voxels along x (with the halo)
constexpr int kLdsRows = 4 + 2;                 // staged rows: the workgroup's 4 and the halo

__device__ uint4 g_zero_chunk[4];  // zero-initialised, never written: the source of the zero halo

// The 32 -> 32 channel convolution (forward with bias and ReLU; data gradient
// with the ReLU mask), implicit GEMM on v_mfma_f32_16x16x32_bf16: rows = 16
// output channels (one half of the 32, fixed per wavefront), columns = 16
// voxels along x, k = one tap's 32 input channels.  The A fragments of all 27
// taps for the wavefront's half (108 VGPRs) are loaded once, so LDS carries
// only the staged activations: a B fragment is one 16-byte read of 8 channels
// of one voxel, with the channel groups stored in the order q ^ ((x >> 2) & 3)
// (conflict free).  Result register r of lane (m, q) is output channel
// 16 hb + 4 q + r of voxel m: four consecutive channels, stored as one 8-byte
// write.  A workgroup owns a 4 x (16 kZmTiles) voxel tile for a chunk of
// `chunk` output planes and marches through its input planes z0 - 1 ..
// z0 + chunk once: each input plane is staged once (direct global-to-LDS
// loads, the zero halo from a zero chunk), into one of two LDS buffers while
// the previous plane is computed, and feeds the accumulators of the three
// output planes it contributes to (z + 1 through its dz = -1 taps, z through
// dz = 0, z - 1 through dz = +1); the output plane that has received all three
// is written.  The staged row sr feeds output row sr - dy for each dy, so one
// fragment read serves up to 3 dz x 3 dy MFMAs.  The wavefronts are the
// kZmTiles x-tiles times the two channel halves; the two halves of a tile
// read the same staged fragments.  The two buffers are separate arrays, so
// the compiler can tell the copies into one from the reads of the other and
// does not wait for the copies before the reads.  Every output voxel sums its
// taps in the order dz = -1, 0, +1, then dx, then dy.  (With the weights
// staged in LDS as well and 32 output channels per wavefront, every plane
// read 72 fragments per 216 MFMAs instead of 18 per 108: 0.88 ms per 256^3
// layer against 0.77 ms here; staging the three input planes of each output
// plane in turn, with a full wait between copy and use, 1.39 ms.)
constexpr int kZmTiles = 2;                        // 16-voxel x-tiles per workgroup
constexpr int kZmChunk = 32;                       // output planes per workgroup, at most
constexpr int kZmBX = 16 * kZmTiles + 2;           // staged voxels along x (with the halo)
constexpr int kZmChunks = kLdsRows * kZmBX * 4;    // 16-byte chunks of one staged plane
constexpr int kZmThreads = 128 * kZmTiles;

// Output plane `plane` (pointer offsets of 32-bit lane parts from a uniform
// plane base): row orow of the tile at lane offset loff + orow W kC.
template <int kEpi, bool full>
__device__ __forceinline__ void zm_store(const f32x4 (&acc)[4], const float (&bias)[4], const void* __restrict__ aux,
                                         void* __restrict__ y, long long plane, int H, int W, int y0, int xv,
                                         int loff) {
    const unsigned short* ap = static_cast<const unsigned short*>(aux) + plane;
    unsigned short* yp = static_cast<unsigned short*>(y) + plane;
#pragma unroll
    for (int orow = 0; orow < 4; ++orow) {
        if (y0 + orow >= H) break;
        if (!full && xv >= W) continue;
        const int off = loff + orow * W * kC;
        float v[4] = {acc[orow][0], acc[orow][1], acc[orow][2], acc[orow][3]};
        if (kEpi == TIGRE_CNN_EPI_BIAS_RELU) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] += bias[r];
                v[r] = v[r] > 0.0f ? v[r] : 0.0f;
            }
        } else {
            const uint2 a = *reinterpret_cast<const uint2*>(ap + off);
            const unsigned ah[4] = {a.x & 0xffffu, a.x >> 16, a.y & 0xffffu, a.y >> 16};
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = (ah[r] != 0 && (ah[r] & 0x8000u) == 0) ? v[r] : 0.0f;  // activation > 0
        }
        const uint2 out = make_uint2((unsigned)bf16_bits(v[0]) | ((unsigned)bf16_bits(v[1]) << 16),
                                     (unsigned)bf16_bits(v[2]) | ((unsigned)bf16_bits(v[3]) << 16));
        *reinterpret_cast<uint2*>(yp + off) = out;
    }
}

template <int kEpi>
__global__ __launch_bounds__(kZmThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void conv_zm_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, const float* __restrict__ bias,
    const void* __restrict__ aux, void* __restrict__ y, int N, int D, int H, int W, int chunk) {
    __shared__ uint4 plane_a[kZmChunks], plane_b[kZmChunks];  // [row][voxel][channel group, swizzled]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, q = lane >> 4;
    const int tile = wave % kZmTiles, hb = wave / kZmTiles;
    const int x0 = blockIdx.x * (16 * kZmTiles), y0 = blockIdx.y * 4;
    const int nchunk = (D + chunk - 1) / chunk;
    const int zc = (int)(blockIdx.z % (unsigned)nchunk);
    const long long n = blockIdx.z / (unsigned)nchunk;
    const int z_lo = zc * chunk, z_hi = min(z_lo + chunk, D);  // output planes z_lo .. z_hi - 1
    const int xv = x0 + 16 * tile + m;                                // this lane's output voxel along x
    const int och = 16 * hb + 4 * q;                                  // its first output channel

    // A fragments: row = output channel 16 hb + m, k = input channels 8 q .. 8 q + 7, per tap
    bf16x8 wf[27];
#pragma unroll
    for (int t = 0; t < 27; ++t)
        wf[t] = __builtin_bit_cast(bf16x8,
                                   *reinterpret_cast<const uint4*>(w + ((long long)(t * kC + 16 * hb + m) * kC + 8 * q)));
    float bias_lane[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (kEpi == TIGRE_CNN_EPI_BIAS_RELU) {
#pragma unroll
        for (int r = 0; r < 4; ++r) bias_lane[r] = bias[och + r];
    }
    unsigned boff[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int xi = 16 * tile + m + d;
        boff[d] = (unsigned)((xi * 4 + (q ^ ((xi >> 2) & 3))) * 16);
    }

    // the chunks this thread copies of every staged plane: element offsets inside the plane, or -1
    // for the zero halo (a plane has fewer than 2^31 elements)
    constexpr int kStageIters = (kZmChunks + kZmThreads - 1) / kZmThreads;
    int soff[kStageIters];
#pragma unroll
    for (int it = 0; it < kStageIters; ++it) {
        const int i = it * kZmThreads + tid;
        const int yi = i / (4 * kZmBX), r = i - yi * 4 * kZmBX, xi = r >> 2, sg = r & 3;
        const int gy = y0 - 1 + yi, gx = x0 - 1 + xi;
        soff[it] = (gy >= 0 && gy < H && gx >= 0 && gx < W) ? (gy * W + gx) * kC + 8 * (sg ^ ((xi >> 2) & 3)) : -1;
    }
    const long long plane_elems = (long long)H * W * kC;
    auto stage = [&](int zi, auto buf) {  // issue the copies of input plane zi into buffer buf
        const unsigned short* xp = x + (n * D + zi) * plane_elems;
        uint4* dst = decltype(buf)::value ? plane_b : plane_a;
#pragma unroll
        for (int it = 0; it < kStageIters; ++it) {
            if (it * kZmThreads + tid < kZmChunks) {
                const void* src = soff[it] >= 0 ? static_cast<const void*>(xp + soff[it]) : g_zero_chunk;
                __builtin_amdgcn_global_load_lds(src, &dst[it * kZmThreads + wave * 64], 16, 0, 0);
            }
        }
    };
    const int loff = (y0 * W + xv) * kC + och;  // this lane's output offset in row y0 of a plane

    f32x4 acc[3][4];
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[s][r] = f32x4{0.f, 0.f, 0.f, 0.f};

    if (z_lo - 1 >= 0) stage(z_lo - 1, std::integral_constant<int, 0>{});
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    // one input plane, staged in buffer kB: the accumulator slots of output planes zi + 1, zi, zi - 1
    // are kN, kC0, kP
    auto plane_step = [&](int zi, auto sn, auto sc, auto sp, auto sb) {
        constexpr int kN = decltype(sn)::value, kC0 = decltype(sc)::value, kP = decltype(sp)::value;
        constexpr int kB = decltype(sb)::value;
        // addresses are formed from the plane index afresh in every step (a scalar base plus the
        // lane's 32-bit offset), instead of 64-bit pointers per unrolled step held in VGPRs
        asm volatile("" : "+s"(zi));
        if (zi + 1 <= z_hi && zi + 1 < D) stage(zi + 1, std::integral_constant<int, 1 - kB>{});
        if (zi >= 0 && zi < D) {  // uniform per workgroup
            const char* lds = reinterpret_cast<const char*>(kB ? plane_b : plane_a);
            const bool on[3] = {zi + 1 < z_hi, zi >= z_lo && zi < z_hi, zi - 1 >= z_lo};
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                bf16x8 b[kLdsRows];
#pragma unroll
                for (int sr = 0; sr < kLdsRows; ++sr)
                    b[sr] = __builtin_bit_cast(bf16x8,
                                               *reinterpret_cast<const uint4*>(lds + boff[d] + sr * (kZmBX * 64)));
#pragma unroll
                for (int dz = 0; dz < 3; ++dz) {
                    if (!on[dz]) continue;
                    f32x4(&A)[4] = acc[dz == 0 ? kN : (dz == 1 ? kC0 : kP)];
#pragma unroll
                    for (int sr = 0; sr < kLdsRows; ++sr)
#pragma unroll
                        for (int dy = 0; dy < 3; ++dy) {
                            const int orow = sr - dy;
                            if (orow < 0 || orow > 3) continue;  // resolved at compile time
                            A[orow] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[dz * 9 + dy * 3 + d], b[sr], A[orow],
                                                                             0, 0, 0);
                        }
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // the next plane is in LDS; this plane's buffer may be overwritten
        const int zo = zi - 1;  // complete: it has received its dz = -1, 0 and +1 taps
        if (zo >= z_lo && zo < z_hi) {
            const long long plane = (n * D + zo) * plane_elems;
            if (x0 + 16 * kZmTiles <= W)
                zm_store<kEpi, true>(acc[kP], bias_lane, aux, y, plane, H, W, y0, xv, loff);
            else
                zm_store<kEpi, false>(acc[kP], bias_lane, aux, y, plane, H, W, y0, xv, loff);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[kP][r] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    for (int zi = z_lo - 1; zi <= z_hi; zi += 6) {
        plane_step(zi, I0{}, I1{}, I2{}, I0{});
        if (zi + 1 > z_hi) break;
        plane_step(zi + 1, I2{}, I0{}, I1{}, I1{});
        if (zi + 2 > z_hi) break;
        plane_step(zi + 2, I1{}, I2{}, I0{}, I0{});
        if (zi + 3 > z_hi) break;
        plane_step(zi + 3, I0{}, I1{}, I2{}, I1{});
        if (zi + 4 > z_hi) break;
        plane_step(zi + 4, I2{}, I0{}, I1{}, I0{});
        if (zi + 5 > z_hi) break;
        plane_step(zi + 5, I1{}, I2{}, I0{}, I1{});
    }
}

// The residual output layer (32 bf16 channels -> one FP32 channel added to
// aux) with the taps as the GEMM columns.  P[u][tap] = sum_i x[u][i] w[tap][0][i]
// for every input voxel u is one MFMA pair per 16 voxels (columns = taps
// 0..31, 27 used), and y[v] = aux[v] + (sum_tap P[v + tap][tap] + bias[0]).
// The 32 -> 32 kernel would spend 27 MFMAs per 16 outputs on this layer with 15 of its
// 16 columns idle; here it is 2 per 16 input voxels.  A workgroup owns a
// 64 x 8 tile of outputs and a chunk of planes, and marches through the
// input planes z0 - 1 .. z0 + chunk: for each it computes P over the 66 x 10
// halo'd tile into LDS; then every lane (one output column) adds the 9-tap
// in-plane sum of each dz group to the accumulator of the output plane that
// group feeds (input plane z feeds z + 1 with the dz = -1 taps, z with dz = 0,
// z - 1 with dz = +1), and writes the output plane that has received all three.
// Every output sums its groups in the order dz = -1, 0, +1 and each group in
// (dy, dx) order: the result does not depend on the launch shape.  The next
// plane's A fragments are loaded while the current plane is summed.
//
// What bounds it: reading the 64 bytes a voxel, 1.29 times with the halo of 8
// rows.  128^3: 40 us, 56 with tiles of 4 rows (1.55 times) and four-byte LDS
// writes; 8 x 32^3: 14 us.
constexpr int kOutTX = 64, kOutTY = 8, kOutZ = 16;  // kOutZ: planes per workgroup, at most
constexpr int kOutHX = kOutTX + 2, kOutHY = kOutTY + 2;
constexpr int kOutU = kOutHX * kOutHY;           // halo'd voxels per plane (660)
constexpr int kOutBlocks = (kOutU + 15) / 16;     // MFMA row blocks per plane (42)
constexpr int kOutPerWave = (kOutBlocks + kOutTY - 1) / kOutTY;  // row blocks per wavefront (one a tile row), at most (6)
// LDS row stride of one tap: an odd number of 16-byte pieces, so the 16 lanes of a write meet all banks
constexpr int kOutStride = kOutBlocks * 16 + 4;
static_assert(kOutStride / 4 % 2 == 1, "conflict-free writes");

__global__ __launch_bounds__(64 * kOutTY) void conv_out_kernel(const unsigned short* __restrict__ x,
                                                       const unsigned short* __restrict__ w,
                                                       const float* __restrict__ bias, const float* __restrict__ aux,
                                                       float* __restrict__ y, int N, int D, int H, int W, int chunk) {
    __shared__ __align__(16) float P[27 * kOutStride];  // [tap][halo'd voxel]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, q = lane >> 4;
    const int x0 = blockIdx.x * kOutTX, y0 = blockIdx.y * kOutTY;
    const int nchunk = (D + chunk - 1) / chunk;
    const int zc = (int)(blockIdx.z % (unsigned)nchunk);
    const long long n = blockIdx.z / (unsigned)nchunk;
    const int z0 = zc * chunk, z1 = min(z0 + chunk, D);  // output planes z0 .. z1 - 1

    // B fragments: column 16 hb + m is the tap, k = 8 q .. 8 q + 7 the input channel
    bf16x8 b[2];
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
        const int tap = 16 * hb + m;
        uint4 raw = make_uint4(0u, 0u, 0u, 0u);
        if (tap < 27) raw = *reinterpret_cast<const uint4*>(w + (long long)tap * kC * kC + 8 * q);
        b[hb] = __builtin_bit_cast(bf16x8, raw);
    }
    // A fragments of plane z: row block wave + kOutTY k, voxel 16 (wave + kOutTY k) + m, channels 8 q ..
    auto load_plane = [&](int z, bf16x8* a) {
#pragma unroll
        for (int k = 0; k < kOutPerWave; ++k) {
            const int u = 16 * (wave + kOutTY * k) + m;
            const int ux = u % kOutHX, uy = u / kOutHX;
            const int gx = x0 - 1 + ux, gy = y0 - 1 + uy;
            const bool ok = u < kOutU && gx >= 0 && gx < W && gy >= 0 && gy < H && z >= 0 && z < D;
            const long long vox = ((n * D + z) * H + gy) * (long long)W + gx;
            a[k] = load_frag<TIGRE_CNN_IN_BF16X32>(x, vox, q, ok);
        }
    };
    bf16x8 a[kOutPerWave];
    load_plane(z0 - 1, a);

    const int ox = x0 + lane, oy = y0 + wave;
    const bool out_ok = ox < W && oy < H;
    // accumulators of output planes zi - 1, zi, zi + 1 while input plane zi is processed
    float a_prev = 0.0f, a_cur = 0.0f, a_next = 0.0f;
    for (int zi = z0 - 1; zi <= z1; ++zi) {
        if (zi >= 0 && zi < D) {  // uniform per workgroup
#pragma unroll
            for (int k = 0; k < kOutPerWave; ++k) {
                const int blk = wave + kOutTY * k;
                if (blk >= kOutBlocks) break;  // uniform per wavefront
                const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                const f32x4 r0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k], b[0], zero, 0, 0, 0);
                const f32x4 r1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k], b[1], zero, 0, 0, 0);
                const int u = 16 * blk + 4 * q;
                *reinterpret_cast<f32x4*>(&P[m * kOutStride + u]) = r0;
                if (16 + m < 27) *reinterpret_cast<f32x4*>(&P[(16 + m) * kOutStride + u]) = r1;
            }
            __syncthreads();  // P complete
            if (zi + 1 <= z1) load_plane(zi + 1, a);
            float s[3];
            const int c = (wave + 1) * kOutHX + lane + 1;  // this lane's voxel in the halo'd tile
#pragma unroll
            for (int g = 0; g < 3; ++g) {
                float t = 0.0f;
#pragma unroll
                for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
                    for (int dx = -1; dx <= 1; ++dx) {
                        const int tap = 9 * g + 3 * (dy + 1) + (dx + 1);
                        t += P[tap * kOutStride + c + dy * kOutHX + dx];
                    }
                s[g] = t;
            }
            a_next += s[0];  // dz = -1: output plane zi + 1
            a_cur += s[1];   // dz = 0:  output plane zi
            a_prev += s[2];  // dz = +1: output plane zi - 1
            __syncthreads();  // P is read before the next plane overwrites it
        } else if (zi + 1 <= z1) {
            load_plane(zi + 1, a);
        }
        const int zo = zi - 1;  // complete: it has its dz = -1, 0 and +1 groups
        if (zo >= z0 && zo < z1 && out_ok) {
            const long long vox = ((n * D + zo) * H + oy) * (long long)W + ox;
            y[vox] = aux[vox] + (a_prev + bias[0]);
        }
        a_prev = a_cur;
        a_cur = a_next;
        a_next = 0.0f;
    }
}

// Convolution of a single FP32 channel (the image, or the loss gradient) into
// 32 channels.  With one input channel the GEMM k dimension of conv_kernel
// holds 1 useful channel of 32; here k is the tap instead: A[o][k] =
// w[k][o][0] (k < 27, zero above), B[k][v] = x[v + tap k], so one MFMA covers
// all taps of 16 voxels and 16 output channels, and with the channels as rows a
// lane ends with eight consecutive channels of a voxel: one 16-byte store.  A
// workgroup owns 128 x 4 outputs and marches along z through a chunk of planes:
// the weights' scattered two-byte loads are paid once a chunk, and three planes
// of the input (6 x 130, zero outside the volume) stay in an LDS ring, from
// which every lane gathers its 8 taps of each tile.
//
// What bounds it: the 64 bytes a voxel it writes.  128^3: 43 us (58 with a
// workgroup a plane and two-byte stores; the stores alone 53), 8 x 32^3: 17 us
// (24; with the mask 19, was 25).
template <int kEpi>
__global__ __launch_bounds__(256) void conv_taps_kernel(const float* __restrict__ x,
                                                        const unsigned short* __restrict__ w,
                                                        const float* __restrict__ bias, const void* __restrict__ aux,
                                                        void* __restrict__ y, int N, int D, int H, int W, int chunk, bool wide) {
    constexpr int kPlane = kLdsRows * kLdsBX, kStage = (kPlane + 255) / 256;
    // [plane % 3][row][voxel], rounded to bf16 once when staged; then zeros for the taps past the 27
    __shared__ unsigned short blk[3 * kPlane + 16 * kLdsTiles];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, q = lane >> 4;
    const int x0 = blockIdx.x * (16 * kLdsTiles), y0 = blockIdx.y * 4;
    const int nchunk = (D + chunk - 1) / chunk;
    const int z0 = (int)(blockIdx.z % (unsigned)nchunk) * chunk, z1 = min(z0 + chunk, D);
    const long long n = blockIdx.z / (unsigned)nchunk;
    const int yo = y0 + wave;

    // plane z of the block: this lane's entries, into registers and then into its LDS slot
    unsigned from[kStage];
#pragma unroll
    for (int k = 0; k < kStage; ++k) {
        const int i = tid + 256 * k, yi = i / kLdsBX, xi = i - yi * kLdsBX;
        const int gy = y0 - 1 + yi, gx = x0 - 1 + xi;
        from[k] = i < kPlane && gy >= 0 && gy < H && gx >= 0 && gx < W ? (unsigned)gy * (unsigned)W + (unsigned)gx : ~0u;
    }
    auto load = [&](int z, float (&v)[kStage]) {
        const float* src = x + (n * D + z) * ((long long)H * W);
#pragma unroll
        for (int k = 0; k < kStage; ++k) v[k] = z >= 0 && z < D && from[k] != ~0u ? src[from[k]] : 0.0f;
    };
    auto keep = [&](int slot, const float (&v)[kStage]) {
#pragma unroll
        for (int k = 0; k < kStage; ++k)
            if (tid + 256 * k < kPlane) blk[slot * kPlane + tid + 256 * k] = bf16_bits(v[k]);
    };
    float next[kStage];
#pragma unroll
    for (int p = 0; p < 3; ++p) {  // planes z0 - 1 .. z0 + 1 into slots 0 .. 2
        load(z0 - 1 + p, next);
        keep(p, next);
    }
    if (tid < 16 * kLdsTiles) blk[3 * kPlane + tid] = 0;
    // this lane's output channels 8 q .. 8 q + 7
    float bias_lane[8];
#pragma unroll
    for (int o = 0; o < 8; ++o) bias_lane[o] = kEpi == TIGRE_CNN_EPI_BIAS_RELU ? bias[8 * q + o] : 0.0f;
    // A fragments: k = 8 q + j is the tap, row m of product hb the channel 8 (m / 4) + 4 hb + m % 4, so that the two
    // products leave a lane with eight consecutive channels of one voxel
    bf16x8 b[2];
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
        unsigned short bits[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int tap = 8 * q + j;
            bits[j] = tap < 27 ? w[((long long)tap * kC + 8 * (m >> 2) + 4 * hb + (m & 3)) * kC] : (unsigned short)0;
        }
        const uint4 raw = make_uint4(bits[0] | ((unsigned)bits[1] << 16), bits[2] | ((unsigned)bits[3] << 16),
                                     bits[4] | ((unsigned)bits[5] << 16), bits[6] | ((unsigned)bits[7] << 16));
        b[hb] = __builtin_bit_cast(bf16x8, raw);
    }
    // this lane's taps: offsets in the block relative to (row wave, voxel m) of tile 0, for the first output plane;
    // a plane further, its input planes are one slot further in the ring
    int toff[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int tap = 8 * q + j;
        const int dz = tap / 9, dy = (tap / 3) % 3, dx = tap % 3;  // each + 1
        toff[j] = tap < 27 ? (dz * kLdsRows + wave + dy) * kLdsBX + m + dx : 3 * kPlane + m;
    }
    for (int z = z0; z < z1; ++z) {
        __syncthreads();  // the planes of z are in LDS
        if (z + 1 < z1) load(z + 2, next);
        const long long obase = ((n * D + z) * H + yo) * (long long)W;
        // one tile at a time (its MFMA pair, then its store), so few registers are live and several workgroups share a CU
#pragma unroll
        for (int t = 0; t < kLdsTiles; ++t) {
            if (x0 + 16 * t >= W || yo >= H) break;
            unsigned short bits[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) bits[j] = blk[toff[j] + 16 * t];
            const uint4 raw = make_uint4(bits[0] | ((unsigned)bits[1] << 16), bits[2] | ((unsigned)bits[3] << 16),
                                         bits[4] | ((unsigned)bits[5] << 16), bits[6] | ((unsigned)bits[7] << 16));
            const bf16x8 a = __builtin_bit_cast(bf16x8, raw);
            f32x4 acc[2];
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0], a, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[1], a, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            const int xo = x0 + 16 * t + m;
            if (xo >= W) continue;
            const long long at = (obase + xo) * kC + 8 * q;
            unsigned short mask[8], out[8];
            if (kEpi == TIGRE_CNN_EPI_RELU_MASK) {
                const unsigned short* am = static_cast<const unsigned short*>(aux) + at;
                if (wide) {
                    const uint4 m4 = *reinterpret_cast<const uint4*>(am);
                    const unsigned word[4] = {m4.x, m4.y, m4.z, m4.w};
#pragma unroll
                    for (int o = 0; o < 8; ++o) mask[o] = (unsigned short)(word[o >> 1] >> (16 * (o & 1)));
                } else {
#pragma unroll
                    for (int o = 0; o < 8; ++o) mask[o] = am[o];
                }
            }
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                float v = acc[o >> 2][o & 3];
                if (kEpi == TIGRE_CNN_EPI_BIAS_RELU) {
                    v += bias_lane[o];
                    v = v > 0.0f ? v : 0.0f;
                } else {
                    v = (mask[o] != 0 && (mask[o] & 0x8000u) == 0) ? v : 0.0f;  // activation > 0
                }
                out[o] = bf16_bits(v);
            }
            unsigned short* ym = static_cast<unsigned short*>(y) + at;
            if (wide) {
                *reinterpret_cast<uint4*>(ym) = make_uint4(out[0] | ((unsigned)out[1] << 16), out[2] | ((unsigned)out[3] << 16),
                                                           out[4] | ((unsigned)out[5] << 16), out[6] | ((unsigned)out[7] << 16));
            } else {
#pragma unroll
                for (int o = 0; o < 8; ++o) ym[o] = out[o];
            }
        }
        __syncthreads();  // plane z - 1 is no longer read
        if (z + 1 < z1) keep((z - z0) % 3, next);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (8 * q + j < 27) toff[j] += toff[j] < 2 * kPlane ? kPlane : -2 * kPlane;
    }
}

// Weight gradient: dw[tap][o][i] = sum_v x[v + tap][i] dy[v][o], one GEMM per tap with k = voxels.
//
// A workgroup of 8 wavefronts owns tiles of kWgRows x-rows by 32 voxels (one k block of the MFMA) and
// marches along z through a chunk of planes; every wavefront keeps the 16 x 16 blocks (input channels
// 16 (w & 1) .., output channels 16 ((w >> 1) & 1) ..) of all 27 taps and of the bias in registers, the
// two groups of four wavefronts take the upper and lower half of the tile's rows and are added in LDS at the end.  So x and dy are read once
// per tile (dy with a halo of one row and one plane) instead of once per tap, and every staged fragment
// feeds up to 27 MFMAs: a row of x meets the nine dy rows (z - dz, y - dy), which slide through registers.
// Planes are staged as they lie in memory, channel fastest; the fragments need eight voxels of one
// channel per lane, which ds_read_b64_tr_b16 gives (in each group of 16 lanes, lane l names row l / 4,
// columns 4 (l % 4) .. + 3 of a 4 x 16 block and receives column l), at any voxel offset, so the dx
// shifts cost nothing.  The two 32-byte channel halves of voxels with bit 3 set are swapped, which
// keeps the eight-byte reads of two lane groups on different banks.  The next plane's loads go to
// registers before the MFMAs of the current one and to LDS after them.
//
// Measured, 8 x 32^3 voxels, 32 -> 32 channels: 24 us a layer (0.6 PFLOP/s; the fragment reads
// and the halo of dy, 1.25 x 1.5, are what keeps it from the matrix rate), 193 us with one workgroup per tap
// and chunk of rows, which read x and dy 28 times and staged them with two-byte LDS writes.
constexpr int kWgRows = 8;                         // x-rows of a tile
constexpr int kWgXW = 34;                          // staged x voxels of a row (halo of one on either side)
constexpr int kWgThreads = 512;
constexpr int kWgXChunks = kWgRows * kWgXW * 4;    // 16-byte chunks of a staged x plane
constexpr int kWgDChunks = (kWgRows + 2) * 32 * 4; // of a staged dy plane
constexpr int kWgXIters = (kWgXChunks + kWgThreads - 1) / kWgThreads;
constexpr int kWgDIters = (kWgDChunks + kWgThreads - 1) / kWgThreads;
constexpr int kWgMaxBlocks = 256;                  // partial sums, at most

typedef f32x4 f32x4u __attribute__((aligned(4)));  // in a caller's buffer
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// Eight voxels of one channel: two transposing reads (voxels 0 .. 3 and 4 .. 7 of the lane group's eight).
__device__ __forceinline__ bf16x8 tr_frag(const char* lo, const char* hi) {
    using P = __attribute__((address_space(3))) s16x4*;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)lo);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)hi);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// A fragment with each pair of voxels masked.
__device__ __forceinline__ bf16x8 masked(bf16x8 f, unsigned m0, unsigned m1, unsigned m2, unsigned m3) {
    const uint4 u = __builtin_bit_cast(uint4, f);
    return __builtin_bit_cast(bf16x8, make_uint4(u.x & m0, u.y & m1, u.z & m2, u.w & m3));
}

// A 16-byte chunk (channels 8 c .. 8 c + 7) of a voxel, or zeros for off < 0.
template <int kIn>
__device__ __forceinline__ uint4 load_chunk(const void* __restrict__ plane, int off, int c) {
    uint4 raw = make_uint4(0u, 0u, 0u, 0u);
    if (kIn == TIGRE_CNN_IN_BF16X32) {
        if (off >= 0) raw = *reinterpret_cast<const uint4*>(static_cast<const unsigned short*>(plane) + (long long)off * kC + 8 * c);
    } else if (off >= 0 && c == 0) {
        raw.x = (unsigned)bf16_bits(static_cast<const float*>(plane)[off]);
    }
    return raw;
}

template <int kXin, int kDyin>
__global__ __launch_bounds__(kWgThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void wgrad_kernel(
    const void* __restrict__ x, const void* __restrict__ dy, float* __restrict__ part, int N, int D, int H, int W,
    int zchunk, int units) {
    struct Stage {
        uint4 x[2][kWgXChunks];
        uint4 d[4][kWgDChunks];
    };
    __shared__ union {
        Stage s;
        f32x4 sum[28 * 256];
    } sh;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, q = lane >> 4;
    const int ih = wave & 1, oh = (wave >> 1) & 1, half = wave >> 2;
    // a block whose input or output channels are all padding holds only zeros
    const bool live = (kXin == TIGRE_CNN_IN_BF16X32 || ih == 0) && (kDyin == TIGRE_CNN_IN_BF16X32 || oh == 0);
    const int segW = (W + 31) / 32, tilesY = (H + kWgRows - 1) / kWgRows, chunksZ = (D + zchunk - 1) / zchunk;

    // lane offsets of the fragment reads inside a staged row: voxel 8 q + 4 h + m / 4 (+ dx + 1 for x)
    int xo[3][2], po[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int v = 8 * q + 4 * h + (m >> 2);
        const int in = ((m & 3) >> 1) * 16 + (m & 1) * 8;
        po[h] = v * 64 + (oh ^ ((v >> 3) & 1)) * 32 + in;
#pragma unroll
        for (int d = 0; d < 3; ++d) xo[d][h] = (v + d) * 64 + (ih ^ (((v + d) >> 3) & 1)) * 32 + in;
    }
    const unsigned one = (m == 0 && ih == 0) ? 0x3f803f80u : 0u;  // bias: input channel 0 is 1 everywhere
    const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(one, one, one, one));

    f32x4 acc[28];
#pragma unroll
    for (int t = 0; t < 28; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int u = blockIdx.x; u < units; u += gridDim.x) {  // uniform: the tiles of this workgroup
        const int xs = (u % segW) * 32;
        const int y0 = ((u / segW) % tilesY) * kWgRows;
        const int zc = (u / (segW * tilesY)) % chunksZ;
        const long long n = u / (segW * tilesY * chunksZ);
        const int za = zc * zchunk, zb = min(za + zchunk, D);
        // x voxels that no dy voxel of a tap meets are left out, not multiplied with the zeros around dy (an infinite one
        // would make the tap NaN): here the one that dx = -1 pairs with voxel W, in a segment that W ends
        unsigned edge_x[4];
        const int past = W - xs - 8 * q;
#pragma unroll
        for (int j = 0; j < 4; ++j) edge_x[j] = past == 2 * j ? 0xffff0000u : past == 2 * j + 1 ? 0x0000ffffu : ~0u;
        // this thread's chunks of a staged plane: voxel offsets from the tile's first row (-1: zero)
        int sx[kWgXIters], sd[kWgDIters];
#pragma unroll
        for (int it = 0; it < kWgXIters; ++it) {
            const int v = (it * kWgThreads + tid) >> 2, r = v / kWgXW;
            const int gy = y0 + r, gx = xs - 1 + v - r * kWgXW;
            sx[it] = (r < kWgRows && gy < H && gx >= 0 && gx < W) ? r * W + gx : -1;
        }
#pragma unroll
        for (int it = 0; it < kWgDIters; ++it) {
            const int v = (it * kWgThreads + tid) >> 2, r = v >> 5;
            const int gy = y0 - 1 + r, gx = xs + (v & 31);
            sd[it] = (r < kWgRows + 2 && gy >= 0 && gy < H && gx < W) ? r * W + gx : -1;
        }
        const long long plane = (long long)H * W;
        constexpr long long xb = kXin == TIGRE_CNN_IN_BF16X32 ? 2 * kC : 4, db = kDyin == TIGRE_CNN_IN_BF16X32 ? 2 * kC : 4;
        auto fetch_x = [&](int z, uint4(&v)[kWgXIters]) {
            const void* p = static_cast<const char*>(x) + ((n * D + z) * plane + (long long)y0 * W) * xb;
#pragma unroll
            for (int it = 0; it < kWgXIters; ++it) {
                const int i = it * kWgThreads + tid, w = (i >> 2) % kWgXW;
                v[it] = load_chunk<kXin>(p, sx[it], (i & 3) ^ ((w >> 3 & 1) << 1));
            }
        };
        auto fetch_d = [&](int z, uint4(&v)[kWgDIters]) {
            const void* p = static_cast<const char*>(dy) + ((n * D + z) * plane + (long long)(y0 - 1) * W) * db;
#pragma unroll
            for (int it = 0; it < kWgDIters; ++it) {
                const int i = it * kWgThreads + tid, w = (i >> 2) & 31;
                v[it] = load_chunk<kDyin>(p, sd[it], (i & 3) ^ ((w >> 3 & 1) << 1));
            }
        };
        auto store_x = [&](int z, const uint4(&v)[kWgXIters]) {
#pragma unroll
            for (int it = 0; it < kWgXIters; ++it)
                if (it * kWgThreads + tid < kWgXChunks) sh.s.x[z & 1][it * kWgThreads + tid] = v[it];
        };
        auto store_d = [&](int z, const uint4(&v)[kWgDIters]) {
#pragma unroll
            for (int it = 0; it < kWgDIters; ++it)
                if (it * kWgThreads + tid < kWgDChunks) sh.s.d[z & 3][it * kWgThreads + tid] = v[it];
        };
        uint4 vx[kWgXIters], vd[kWgDIters];
        __syncthreads();  // the previous tile's planes have been read
        for (int z = max(za - 1, 0); z <= min(za + 1, D - 1); ++z) {
            fetch_d(z, vd);
            store_d(z, vd);
        }
        fetch_x(za, vx);
        store_x(za, vx);
        __syncthreads();
        for (int z = za; z < zb; ++z) {
            const bool more_x = z + 1 < zb, more_d = z + 1 < zb && z + 2 < D;  // uniform
            if (more_x) fetch_x(z + 1, vx);
            if (more_d) fetch_d(z + 2, vd);
            if (live) {
                const char* lx = reinterpret_cast<const char*>(sh.s.x[z & 1]) + half * (kWgRows / 2) * (kWgXW * 64);
                const char* ld[3];  // dy planes z + 1, z, z - 1 (taps dz = -1, 0, +1)
                const bool on[3] = {z + 1 < D, true, z >= 1};
#pragma unroll
                for (int dz = 0; dz < 3; ++dz)
                    ld[dz] = reinterpret_cast<const char*>(sh.s.d[(z + 1 - dz) & 3]) + half * (kWgRows / 2) * 2048;
                bf16x8 b[3][3];  // [dz][dy row mod 3]
#pragma unroll
                for (int dz = 0; dz < 3; ++dz)
#pragma unroll
                    for (int r = 0; r < 2; ++r) b[dz][r] = tr_frag(ld[dz] + r * 2048 + po[0], ld[dz] + r * 2048 + po[1]);
#pragma unroll
                for (int r = 0; r < kWgRows / 2; ++r) {
                    bf16x8 a[3];
#pragma unroll
                    for (int d = 0; d < 3; ++d)
                        a[d] = tr_frag(lx + r * (kWgXW * 64) + xo[d][0], lx + r * (kWgXW * 64) + xo[d][1]);
                    a[0] = masked(a[0], edge_x[0], edge_x[1], edge_x[2], edge_x[3]);
                    // (the volume's first row meets no dy row of the taps dy = 1, its last none of dy = -1)
                    const int row = y0 + half * (kWgRows / 2) + r;
#pragma unroll
                    for (int dz = 0; dz < 3; ++dz) {
                        b[dz][(r + 2) % 3] =
                            tr_frag(ld[dz] + (r + 2) * 2048 + po[0], ld[dz] + (r + 2) * 2048 + po[1]);
                        if (!on[dz]) continue;  // uniform
#pragma unroll
                        for (int dyy = 0; dyy < 3; ++dyy) {  // tap dy = dyy - 1 reads dy row r - dy, halo'd index r + 2 - dyy
                            if ((dyy == 0 && row == H - 1) || (dyy == 2 && r == 0 && row == 0)) continue;  // uniform
#pragma unroll
                            for (int d = 0; d < 3; ++d)
                                acc[dz * 9 + dyy * 3 + d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                    a[d], b[dz][(r + 2 - dyy) % 3], acc[dz * 9 + dyy * 3 + d], 0, 0, 0);
                        }
                    }
                    if (ih == 0)
                        acc[27] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, b[1][(r + 1) % 3], acc[27], 0, 0, 0);
                }
            }
            if (more_x) store_x(z + 1, vx);  // the buffers of planes z - 1 (x) and z - 2 (dy), read before the last barrier
            if (more_d) store_d(z + 2, vd);
            __syncthreads();
        }
    }
    // the two halves of the rows, then part[block][tap][o][i]: row i = 16 ih + 4 q + r, column o = 16 oh + m
    __syncthreads();
    if (half == 1) {
#pragma unroll
        for (int t = 0; t < 28; ++t) sh.sum[t * 256 + (tid & 255)] = acc[t];
    }
    __syncthreads();
    if (half == 0) {
        float* p = part + (long long)blockIdx.x * 28 * kC * kC;
#pragma unroll
        for (int t = 0; t < 28; ++t)
            *reinterpret_cast<f32x4u*>(p + (t * kC + 16 * oh + m) * kC + 16 * ih + 4 * q) = acc[t] + sh.sum[t * 256 + tid];
    }
}

// out[i] = sum over the partials part[c][i].  Sixteen lanes of a workgroup's 256 hold four neighbouring
// sums each, and the sixteen groups take every sixteenth partial; the groups are added in a fixed order.
// Measured with 256 partials: 5.9 us, 60 us with one lane per sum.
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const f32x4u* __restrict__ part, int nparts,
                                                           f32x4u* __restrict__ out) {
    constexpr int kQuads = 28 * kC * kC / 4;
    __shared__ f32x4 sum[256];
    const int col = threadIdx.x & 15, grp = threadIdx.x >> 4;
    const int i = blockIdx.x * 16 + col;  // kQuads is a multiple of 16
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int c = grp; c < nparts; c += 16) s += part[(long long)c * kQuads + i];
    sum[threadIdx.x] = s;
    __syncthreads();
    if (grp == 0) {
        for (int g = 1; g < 16; ++g) s += sum[g * 16 + col];
        out[i] = s;
    }
}

long long wgrad_chunks(long long nseg) {
    long long c = (nseg + 15) / 16;  // at least 16 segments per block
    if (c > 256) c = 256;
    return c < 1 ? 1 : c;
}

}  // namespace

namespace {
// Output planes per workgroup of a kernel that marches along z over `tiles` tiles of the plane: 4, 8, 16
// or 32, up to `most`.  A workgroup of c planes runs about c + 5 steps (two planes of halo, and its weights
// and first plane before any step), and `slots` workgroups run at once, so the smallest number of rounds
// times steps is taken; the larger c on ties.  The result does not depend on it.  At 8 x 32^3 chunks of 32 planes
// are 64 workgroups on 256 CUs, 65 us (102 us with the ReLU mask); of 4 planes, 512 workgroups, 20 and 24 us.
int march_chunk(int N, int D, long long tiles, int most, int slots) {
    int best = most;
    long long cost = -1;
    for (int c = most; c >= 4; c /= 2) {
        const long long blocks = tiles * N * ((D + c - 1) / c);
        const long long t = ((blocks + slots - 1) / slots) * ((c < D ? c : D) + 5);
        if (cost < 0 || t < cost) {
            cost = t;
            best = c;
        }
    }
    return best;
}
}  // namespace

size_t cnn_wgrad_workspace(int N, int D, int H, int W) {
    const long long nseg = (long long)N * D * H * ((W + 31) / 32);
    return (size_t)wgrad_chunks(nseg) * 28 * kC * kC * sizeof(float);
}

int launch_cnn_conv(const void* x, int x_mode, const unsigned short* w, const float* bias, const void* aux, void* y,
                    int epi, int N, int D, int H, int W, hipStream_t stream) {
    TIGRE_REQUIRE(N > 0 && D > 0 && H > 0 && W > 0, "empty volume");
    TIGRE_REQUIRE(x_mode == TIGRE_CNN_IN_BF16X32 || x_mode == TIGRE_CNN_IN_F32X1, "unknown input mode");
    TIGRE_REQUIRE(epi == TIGRE_CNN_EPI_BIAS_RELU || epi == TIGRE_CNN_EPI_RELU_MASK || epi == TIGRE_CNN_EPI_RESIDUAL,
                  "unknown epilogue");
    TIGRE_REQUIRE(epi == TIGRE_CNN_EPI_RELU_MASK || bias != nullptr, "missing bias");
    TIGRE_REQUIRE(epi == TIGRE_CNN_EPI_BIAS_RELU || aux != nullptr, "missing mask / residual input");
    TIGRE_REQUIRE((reinterpret_cast<uintptr_t>(x) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0,
                  "activations and weights must be 16-byte aligned");
    const long long rows = (long long)N * D * H;
    TIGRE_REQUIRE((rows + 3) / 4 <= 2147483647LL, "volume too large");
    dim3 grid((unsigned)((W + 16 * kTilesPerWave - 1) / (16 * kTilesPerWave)), (unsigned)((rows + 3) / 4));
#define TIGRE_CONV(I, E) hipLaunchKernelGGL((conv_kernel<I, E>), grid, dim3(256), 0, stream, x, w, bias, aux, y, N, D, H, W)
    if (x_mode == TIGRE_CNN_IN_BF16X32) {
        TIGRE_REQUIRE((long long)N * D <= 65535, "too many planes for one launch");
        const unsigned short* xa = static_cast<const unsigned short*>(x);
        const dim3 lgrid((unsigned)((W + 16 * kLdsTiles - 1) / (16 * kLdsTiles)), (unsigned)((H + 3) / 4),
                         (unsigned)(N * D));
        const unsigned zmx = (unsigned)((W + 16 * kZmTiles - 1) / (16 * kZmTiles));
        const int chunk = march_chunk(N, D, (long long)zmx * lgrid.y, kZmChunk, 512);
        const dim3 zgrid(zmx, lgrid.y, (unsigned)(N * ((D + chunk - 1) / chunk)));  // at most N D planes
        TIGRE_REQUIRE((long long)H * W * kC <= 2147483647LL, "plane too large");
        if (epi != TIGRE_CNN_EPI_RESIDUAL)
            TIGRE_REQUIRE((reinterpret_cast<uintptr_t>(y) & 7) == 0 && (reinterpret_cast<uintptr_t>(aux) & 7) == 0,
                          "32-channel outputs and masks must be 8-byte aligned");
        if (epi == TIGRE_CNN_EPI_BIAS_RELU) {
            hipLaunchKernelGGL((conv_zm_kernel<TIGRE_CNN_EPI_BIAS_RELU>), zgrid, dim3(kZmThreads), 0, stream, xa, w, bias,
                               aux, y, N, D, H, W, chunk);
        } else if (epi == TIGRE_CNN_EPI_RELU_MASK) {
            hipLaunchKernelGGL((conv_zm_kernel<TIGRE_CNN_EPI_RELU_MASK>), zgrid, dim3(kZmThreads), 0, stream, xa, w, bias,
                               aux, y, N, D, H, W, chunk);
        } else {
            TIGRE_REQUIRE((H + kOutTY - 1) / kOutTY <= 65535, "volume too large for one launch");
            const unsigned ox = (unsigned)((W + kOutTX - 1) / kOutTX), oy = (unsigned)((H + kOutTY - 1) / kOutTY);
            const int ochunk = march_chunk(N, D, (long long)ox * oy, kOutZ, 512);
            const dim3 ogrid(ox, oy, (unsigned)(N * ((D + ochunk - 1) / ochunk)));
            hipLaunchKernelGGL(conv_out_kernel, ogrid, dim3(64 * kOutTY), 0, stream, xa, w, bias,
                               static_cast<const float*>(aux), static_cast<float*>(y), N, D, H, W, ochunk);
        }
    } else {
        TIGRE_REQUIRE((long long)N * D <= 65535, "too many planes for one launch");
        const float* xf = static_cast<const float*>(x);
        const unsigned lx = (unsigned)((W + 16 * kLdsTiles - 1) / (16 * kLdsTiles)), ly = (unsigned)((H + 3) / 4);
        const int chunk = march_chunk(N, D, (long long)lx * ly, 16, 1024);
        const dim3 lgrid(lx, ly, (unsigned)(N * ((D + chunk - 1) / chunk)));
        TIGRE_REQUIRE((long long)H * W < 4294967295LL, "plane too large");  // 32-bit offsets in a plane
        // 16-byte stores and mask loads where the pointers allow them
        const uintptr_t mask_at = epi == TIGRE_CNN_EPI_RELU_MASK ? reinterpret_cast<uintptr_t>(aux) : 0;
        const bool wide = ((reinterpret_cast<uintptr_t>(y) | mask_at) & 15) == 0;
        if (epi == TIGRE_CNN_EPI_BIAS_RELU)
            hipLaunchKernelGGL((conv_taps_kernel<TIGRE_CNN_EPI_BIAS_RELU>), lgrid, dim3(256), 0, stream, xf, w, bias,
                               aux, y, N, D, H, W, chunk, wide);
        else if (epi == TIGRE_CNN_EPI_RELU_MASK)
            hipLaunchKernelGGL((conv_taps_kernel<TIGRE_CNN_EPI_RELU_MASK>), lgrid, dim3(256), 0, stream, xf, w, bias,
                               aux, y, N, D, H, W, chunk, wide);
        else TIGRE_CONV(TIGRE_CNN_IN_F32X1, TIGRE_CNN_EPI_RESIDUAL);
    }
#undef TIGRE_CONV
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

int launch_cnn_wgrad(const void* x, int x_mode, const void* dy, int dy_mode, float* dw, int N, int D, int H, int W,
                     void* ws, size_t ws_bytes, hipStream_t stream) {
    TIGRE_REQUIRE(N > 0 && D > 0 && H > 0 && W > 0, "empty volume");
    TIGRE_REQUIRE(x_mode == TIGRE_CNN_IN_BF16X32 || x_mode == TIGRE_CNN_IN_F32X1, "unknown input mode");
    TIGRE_REQUIRE(dy_mode == TIGRE_CNN_IN_BF16X32 || dy_mode == TIGRE_CNN_IN_F32X1, "unknown gradient mode");
    TIGRE_REQUIRE(ws != nullptr && ws_bytes >= cnn_wgrad_workspace(N, D, H, W), "workspace too small");
    TIGRE_REQUIRE(W < (1 << 27), "volume too wide");  // 32-bit offsets inside the ten rows of a tile
    // Planes per tile: as few as fill kWgMaxBlocks workgroups (one per CU), at least 4 (each tile
    // reads two planes of dy more than it has planes of x), at most 16.
    const long long tiles = (long long)N * ((H + kWgRows - 1) / kWgRows) * ((W + 31) / 32);
    const long long want = (tiles * D + kWgMaxBlocks - 1) / kWgMaxBlocks;
    const int zchunk = (int)(want < 4 ? 4 : (want > 16 ? 16 : want));
    const long long units = tiles * ((D + zchunk - 1) / zchunk);
    TIGRE_REQUIRE(units < (1LL << 31) - kWgMaxBlocks, "volume too large");
    const long long nseg = (long long)N * D * H * ((W + 31) / 32);
    const int blocks = (int)(units < wgrad_chunks(nseg) ? units : wgrad_chunks(nseg));
    float* part = static_cast<float*>(ws);
#define TIGRE_WG(XI, DI)                                                                                       \
    hipLaunchKernelGGL((wgrad_kernel<XI, DI>), dim3((unsigned)blocks), dim3(kWgThreads), 0, stream, x, dy, part, N, \
                       D, H, W, zchunk, (int)units)
    if (x_mode == TIGRE_CNN_IN_BF16X32) {
        if (dy_mode == TIGRE_CNN_IN_BF16X32) TIGRE_WG(TIGRE_CNN_IN_BF16X32, TIGRE_CNN_IN_BF16X32);
        else TIGRE_WG(TIGRE_CNN_IN_BF16X32, TIGRE_CNN_IN_F32X1);
    } else {
        if (dy_mode == TIGRE_CNN_IN_BF16X32) TIGRE_WG(TIGRE_CNN_IN_F32X1, TIGRE_CNN_IN_BF16X32);
        else TIGRE_WG(TIGRE_CNN_IN_F32X1, TIGRE_CNN_IN_F32X1);
    }
#undef TIGRE_WG
    TIGRE_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(28 * kC * kC / 64), dim3(256), 0, stream,
                       reinterpret_cast<const f32x4u*>(part), blocks, reinterpret_cast<f32x4u*>(dw));
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

// ---------------------------------------------------------------------------
// Weight gradient without allocation.  The per-block partial sums go to a
// library-held device array sized for the most any volume needs (wgrad_chunks
// caps the chunks at 256: 256 x 28 x 32 x 32 floats, 28 MiB), one copy per GPU
// for the life of the process.  Every partial the reduction reads is written
// by the same call, so nothing needs clearing; calls that overlap on one GPU
// (two streams) share the array and race.  The array's device address is
// looked up once per device, with that device current; host code passes that
// address, never the symbol itself.
// ---------------------------------------------------------------------------
static __device__ __align__(256) float scratch[256 * 28 * kC * kC];

namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchDevices] = {};

int scratch_address(void** out) {
    int dev = 0;
    TIGRE_HIP_TRY(hipGetDevice(&dev));
    TIGRE_REQUIRE(dev >= 0 && dev < kScratchDevices, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        TIGRE_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        TIGRE_REQUIRE(p != nullptr, "no device address for the weight-gradient scratch");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return TIGRE_OK;
}
}  // namespace

size_t cnn_wgrad_static_bytes() { return sizeof(scratch); }

int launch_cnn_wgrad_noalloc(const void* x, int x_mode, const void* dy, int dy_mode, float* dw, int N, int D, int H,
                             int W, hipStream_t stream) {
    TIGRE_REQUIRE(N > 0 && D > 0 && H > 0 && W > 0, "empty volume");
    const size_t need = cnn_wgrad_workspace(N, D, H, W);
    TIGRE_REQUIRE(need <= sizeof(scratch), "weight-gradient partials exceed the library's static scratch");
    void* ws = nullptr;
    TIGRE_CHECK(scratch_address(&ws));
    return launch_cnn_wgrad(x, x_mode, dy, dy_mode, dw, N, D, H, W, ws, sizeof(scratch), stream);
}

}  // namespace tigre
