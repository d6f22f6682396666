// Row filter of the analytic reconstructions for gfx950: every detector row is
// weighted, convolved with a symmetric kernel (the ramp, windowed or not) and
// written, in one pass over memory.
//
// The convolution is a product of spectra.  A row of nU <= M / 2 real pixels is
// one complex signal of length M: pixel n < M / 4 is the real part of element
// n, pixel n + M / 4 its imaginary part, the rest zero.  The kernel is real and
// symmetric, so its spectrum is real, and the inverse transform holds the two
// halves' convolutions c in its real and imaginary part; pixel m of the result
// is Re c[m] + Im c[m - M / 4].  All lags stay below M / 2, so nothing wraps.
// One transform of length M a row then does what a padded real transform of
// length 2 M (or M, for nU between two powers of two) does, without the
// even-odd step, and rows do not mix.
//
// M / 8 lanes share a row, 8 elements each in registers: radix-8 passes by
// decimation in frequency, with a last radix 2 or 4 where M is no power of 8,
// product, and the same passes backwards, so the spectrum is never put in
// order; the response is read in the passes' order instead.  Passes exchange
// through LDS, one wavefront's lanes without a barrier (M <= 512).  A workgroup
// walks over rows and keeps its twiddle factors and its part of the response
// in registers.
//
// What bounds it: vector issue (two radix-8 transforms of 512 elements are
// about 700 instructions a wavefront) next to the LDS exchanges: 46080 rows of
// 256 pixels take 58 us, 20 of them memory.  The padded rows' real FFT (copy
// into zeroed rows, two transforms with their even-odd passes, copies,
// product, scale) took 810 us of the same call.
#include "common.hpp"

namespace tigre {
namespace {

// Workgroups of a launch: enough for every slot of the chip, each with several rows where there are many, so that
// twiddle factors and response are set up a few times only.
constexpr long long kFilterBlocks = 2048;

struct Cplx {
    float x, y;
};
__device__ __forceinline__ Cplx operator+(Cplx a, Cplx b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ Cplx operator-(Cplx a, Cplx b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ Cplx mul(Cplx a, Cplx b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
// a times the conjugate of b
__device__ __forceinline__ Cplx mulc(Cplx a, Cplx b) { return {a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y}; }
// a times -i (kInv: times i)
template <bool kInv>
__device__ __forceinline__ Cplx quarter(Cplx a) {
    return kInv ? Cplx{-a.y, a.x} : Cplx{a.y, -a.x};
}
// a times exp(-i pi / 4) (kInv: its conjugate)
template <bool kInv>
__device__ __forceinline__ Cplx eighth(Cplx a) {
    constexpr float r = 0.70710678118654752f;
    return kInv ? Cplx{(a.x - a.y) * r, (a.x + a.y) * r} : Cplx{(a.x + a.y) * r, (a.y - a.x) * r};
}

template <bool kInv>
__device__ __forceinline__ void dft4(Cplx& a, Cplx& b, Cplx& c, Cplx& d) {
    const Cplx s = a + c, t = a - c, u = b + d, v = quarter<kInv>(b - d);
    a = s + u;
    b = t + v;
    c = s - u;
    d = t - v;
}

// v[q] = sum over n of v[n] exp(-+ 2 pi i n q / 8)
template <bool kInv>
__device__ __forceinline__ void dft8(Cplx (&v)[8]) {
    Cplx s0 = v[0] + v[4], s1 = v[1] + v[5], s2 = v[2] + v[6], s3 = v[3] + v[7];
    Cplx d0 = v[0] - v[4], d1 = eighth<kInv>(v[1] - v[5]), d2 = quarter<kInv>(v[2] - v[6]),
         d3 = quarter<kInv>(eighth<kInv>(v[3] - v[7]));
    dft4<kInv>(s0, s1, s2, s3);
    dft4<kInv>(d0, d1, d2, d3);
    v[0] = s0, v[1] = d0, v[2] = s1, v[3] = d1, v[4] = s2, v[5] = d2, v[6] = s3, v[7] = d3;
}

template <int kLog>
struct Shape {
    static constexpr int kM = 1 << kLog, kT = kM / 8;           // length, lanes of a row
    static constexpr int kThreads = kT < 256 ? 256 : kT;
    static constexpr int kRows = kThreads / kT;                 // rows of a workgroup
    static constexpr int kPasses = kLog / 3, kRest = kLog % 3;  // radix-8 passes, log2 of the last radix
    static constexpr int kTw = kRest ? kPasses : kPasses - 1;   // passes with twiddle factors
    static constexpr int kLds = kM + kM / 8;                    // a gap every 8 elements spreads the banks
};

// Element q of lane t in pass s is at first(t) + q * step.
template <int kLog>
__device__ __forceinline__ int first(int t, int s) {
    using S = Shape<kLog>;
    if (s >= S::kPasses) return 8 * t;
    const int sub = S::kT >> (3 * s);  // an eighth of the pass's transforms
    return (t / sub) * (8 * sub) + t % sub;
}
template <int kLog>
__host__ __device__ constexpr int step(int s) {
    return s >= Shape<kLog>::kPasses ? 1 : Shape<kLog>::kT >> (3 * s);
}

template <int kLog>
__device__ __forceinline__ void meet() {
    if constexpr (Shape<kLog>::kT > 64) {
        __syncthreads();
    } else {  // the LDS operations of one wavefront complete in order
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// The lanes of a row pass their elements from the order of pass `from` to that of pass `to`.
template <int kLog>
__device__ __forceinline__ void exchange(float2* lds, Cplx (&v)[8], int t, int from, int to) {
    const int a = first<kLog>(t, from), b = first<kLog>(t, to);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int p = a + q * step<kLog>(from);
        lds[p + (p >> 3)] = make_float2(v[q].x, v[q].y);
    }
    meet<kLog>();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int p = b + q * step<kLog>(to);
        const float2 e = lds[p + (p >> 3)];
        v[q] = {e.x, e.y};
    }
    meet<kLog>();
}

// The pass after the radix-8 passes, its own inverse but for the sign.
template <int kLog, bool kInv>
__device__ __forceinline__ void last_pass(Cplx (&v)[8]) {
    if constexpr (Shape<kLog>::kRest == 2) {
        dft4<kInv>(v[0], v[1], v[2], v[3]);
        dft4<kInv>(v[4], v[5], v[6], v[7]);
    } else if constexpr (Shape<kLog>::kRest == 1) {
#pragma unroll
        for (int q = 0; q < 8; q += 2) {
            const Cplx a = v[q];
            v[q] = a + v[q + 1];
            v[q + 1] = a - v[q + 1];
        }
    }
}
}  // namespace

// rows rows of nU pixels, weighted by the image weight (nV x nU, row r by its row r % nV) when it is there.
// response: M / 2 + 1 values of the kernel's spectrum over M.
template <int kLog>
__global__ __launch_bounds__(Shape<kLog>::kThreads) void filter_rows_kernel(const float* __restrict__ in,
                                                                            const float* __restrict__ weight,
                                                                            const float* __restrict__ response,
                                                                            float* __restrict__ out, long long rows,
                                                                            int nV, int nU) {
    using S = Shape<kLog>;
    __shared__ float2 lds_all[S::kRows * S::kLds];
    const int sub = threadIdx.x / S::kT, t = threadIdx.x % S::kT;
    float2* lds = lds_all + sub * S::kLds;

    Cplx tw[S::kTw > 0 ? S::kTw : 1][7];
#pragma unroll
    for (int s = 0; s < S::kTw; ++s) {
        const int len = S::kM >> (3 * s), j = t % (len / 8);
#pragma unroll
        for (int q = 1; q < 8; ++q) {
            float sn, cs;
            sincospif(-2.0f * (float)(j * q) / (float)len, &sn, &cs);
            tw[s][q - 1] = {cs, sn};
        }
    }
    float g[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        // the frequency that the passes leave at element 8 t + q: its digits in reverse
        int p = 8 * t + q, f = 0, weightf = 1, len = S::kM;
#pragma unroll
        for (int s = 0; s < S::kPasses; ++s) {
            len /= 8;
            f += p / len * weightf;
            p %= len;
            weightf *= 8;
        }
        f += p * weightf;
        g[q] = response[min(f, S::kM - f)];
    }

    for (long long r0 = (long long)blockIdx.x * S::kRows; r0 < rows; r0 += (long long)gridDim.x * S::kRows) {
        const long long r = r0 + sub;
        const bool live = r < rows;
        const float* x = in + r * nU;
        const float* w = weight ? weight + (long long)(r % nV) * nU : nullptr;
        auto pixel = [&](int m) {
            if (!live || m >= nU) return 0.0f;
            return w ? x[m] * w[m] : x[m];
        };
        // first pass: only elements below M / 4 are not zero
        const Cplx a = {pixel(t), pixel(t + 2 * S::kT)}, b = {pixel(t + S::kT), pixel(t + 3 * S::kT)};
        const Cplx b1 = eighth<false>(b), b2 = quarter<false>(b), b3 = quarter<false>(b1);
        Cplx v[8] = {a + b, a + b1, a + b2, a + b3, a - b, a - b1, a - b2, a - b3};
#pragma unroll
        for (int s = 0; s < S::kPasses; ++s) {
            if (s > 0) {
                exchange<kLog>(lds, v, t, s - 1, s);
                dft8<false>(v);
            }
            if (s < S::kTw) {
#pragma unroll
                for (int q = 1; q < 8; ++q) v[q] = mul(v[q], tw[s][q - 1]);
            }
        }
        if (S::kRest) {
            exchange<kLog>(lds, v, t, S::kPasses - 1, S::kPasses);
            last_pass<kLog, false>(v);
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = {v[q].x * g[q], v[q].y * g[q]};
        if (S::kRest) {
            last_pass<kLog, true>(v);
            exchange<kLog>(lds, v, t, S::kPasses, S::kPasses - 1);
        }
#pragma unroll
        for (int s = S::kPasses - 1; s >= 0; --s) {
            if (s < S::kTw) {
#pragma unroll
                for (int q = 1; q < 8; ++q) v[q] = mulc(v[q], tw[s][q - 1]);
            }
            dft8<true>(v);
            if (s > 0) exchange<kLog>(lds, v, t, s, s - 1);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int m = t + q * S::kT;
            if (live && m < nU) out[r * nU + m] = v[q].x + v[(q + 6) & 7].y;
        }
    }
}

// Cosine weight of every pixel, dsd / sqrt(dsd^2 + x^2 + y^2), in FP64 and rounded once, with the roundings of that
// expression evaluated left to right.  In place of an upload: 64 K pixels take 2 us, and the host has nothing to wait
// for.
__global__ __launch_bounds__(256) void cosine_weight_kernel(float* __restrict__ w, int nV, int nU, double dV, double dU,
                                                            double dsd) {
#pragma clang fp contract(off)
    const long long total = (long long)nV * nU;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256) {
        const int v = (int)(i / nU), u = (int)(i - (long long)v * nU);
        const double x = (u - nU / 2.0 + 0.5) * dU, y = (v - nV / 2.0 + 0.5) * dV;
        w[i] = (float)(dsd / sqrt(dsd * dsd + x * x + y * y));
    }
}

int launch_cosine_weight(float* w, int nV, int nU, double dV, double dU, double dsd, hipStream_t stream) {
    TIGRE_REQUIRE(nV > 0 && nU > 0, "cosine weight: detector sizes must be positive");
    const long long blocks = ((long long)nV * nU + 255) / 256;
    hipLaunchKernelGGL(cosine_weight_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream, w, nV,
                       nU, dV, dU, dsd);
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

int launch_filter_rows(const float* in, const float* weight, const float* response, float* out, long long rows, int nV,
                       int nU, int log2_len, hipStream_t stream) {
    TIGRE_REQUIRE(rows > 0 && nV > 0 && nU > 0, "filter: rows and detector sizes must be positive");
    TIGRE_REQUIRE(log2_len >= kFilterMinLog && log2_len <= kFilterMaxLog && 2LL * nU <= 1LL << log2_len,
                  "filter: the transform must hold two rows, 64 to 4096 elements");
#define TIGRE_FILTER(L)                                                                                       \
    case L: {                                                                                                 \
        const long long blocks = (rows + Shape<L>::kRows - 1) / Shape<L>::kRows;                              \
        hipLaunchKernelGGL(filter_rows_kernel<L>, dim3((unsigned)(blocks < kFilterBlocks ? blocks : kFilterBlocks)), \
                           dim3(Shape<L>::kThreads), 0, stream, in, weight, response, out, rows, nV, nU);     \
        break;                                                                                                \
    }
    switch (log2_len) {
        TIGRE_FILTER(6)
        TIGRE_FILTER(7)
        TIGRE_FILTER(8)
        TIGRE_FILTER(9)
        TIGRE_FILTER(10)
        TIGRE_FILTER(11)
        TIGRE_FILTER(12)
    }
#undef TIGRE_FILTER
    TIGRE_HIP_TRY(hipGetLastError());
    return TIGRE_OK;
}

}  // namespace tigre
