// Kernels of the VAE decoder (the vae-decode stage, reference src/models/vae_decoder.cpp) on
// gfx950. The decoder engine (vae_engine.cpp) keeps activations channels-last, [pixels, channels]
// bf16, so that a 3x3 convolution is an implicit GEMM (conv.hip, launch_conv3x3_bf16) and the
// mid-block attention reads its tokens in place. This file holds what is not a GEMM:
//   - k_transpose       [R, C] -> [C, R] per batch: NCHW <-> NHWC at the stage's two ends, and
//                       the reference's TransposeArgs op (ops.h:184-191);
//   - GroupNorm         fp64 sums and sums of squares in a fixed order (from the convolution that
//                       wrote the tensor, or one pass over it), applied by a pass, or by the
//                       convolution that reads the tensor; rounded to bf16 as the reference stores
//                       it (ops_cpu.cpp:186-224), and with its SiLU both rounded, in the folded form
//                       of norm_silu8 (common.h);
//   - k_conv_direct     a convolution in the reference's summation order, for the single op where
//                       the MFMA tile does not apply (the engine pads its two thin convolutions);
//   - k_upsample_nchw   the reference's UpsampleArgs op (the engine fuses the upsample into the
//                       next convolution's gather instead).
// The convolutions are in conv.hip, the mid-block's attention in flash512.hip.
#include "common.h"

#include <algorithm>
#include <cmath>
#include <mutex>

namespace bh {
namespace {

// ---- [R, C] -> [C, R] per batch --------------------------------------------------------------

__global__ void __launch_bounds__(256) k_transpose(const bf16_t* __restrict__ in, bf16_t* __restrict__ out,
                                                   int64_t R, int64_t C, int64_t keep) {
    __shared__ bf16_t tile[32][33];
    const int64_t b = blockIdx.z;
    in += b * R * C;
    out += b * R * keep;
    const int64_t r0 = static_cast<int64_t>(blockIdx.y) * 32, c0 = static_cast<int64_t>(blockIdx.x) * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
    for (int i = ty; i < 32; i += 8) {
        const int64_t r = r0 + i, c = c0 + tx;
        if (r < R && c < C) tile[i][tx] = in[r * C + c];
    }
    __syncthreads();
#pragma unroll
    for (int i = ty; i < 32; i += 8) {
        const int64_t c = c0 + i, r = r0 + tx;
        if (c < keep && r < R) out[c * R + r] = tile[tx][i];
    }
}

// The same where rows and columns split into 16-byte runs (R, C and keep multiples of 8, 16-byte
// aligned): a 64 x 64 tile, eight lanes to a 128-byte row segment on both sides. The 66-element
// pitch spreads the eight rows a lane gathers (1056 bytes apart) and its neighbours' columns over
// all banks. Bound by HBM: 512 x 36864 values 25 -> 12 us.
__global__ void __launch_bounds__(256) k_transpose_v8(const bf16_t* __restrict__ in, bf16_t* __restrict__ out,
                                                      int64_t R, int64_t C, int64_t keep) {
    __shared__ __attribute__((aligned(16))) bf16_t tile[64][66];
    const int64_t b = blockIdx.z;
    in += b * R * C;
    out += b * R * keep;
    const int64_t r0 = static_cast<int64_t>(blockIdx.y) * 64, c0 = static_cast<int64_t>(blockIdx.x) * 64;
    const int t8 = threadIdx.x & 7, ty = threadIdx.x >> 3;
#pragma unroll
    for (int i = ty; i < 64; i += 32) {
        const int64_t r = r0 + i, c = c0 + 8 * t8;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (r < R && c < C) v = *reinterpret_cast<const uint4*>(in + r * C + c);
        uint32_t* dst = reinterpret_cast<uint32_t*>(&tile[i][8 * t8]);
        dst[0] = v.x;
        dst[1] = v.y;
        dst[2] = v.z;
        dst[3] = v.w;
    }
    __syncthreads();
#pragma unroll
    for (int i = ty; i < 64; i += 32) {
        const int64_t c = c0 + i, r = r0 + 8 * t8;
        if (c >= keep || r >= R) continue;
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            w[e] = tile[8 * t8 + 2 * e][i] | static_cast<uint32_t>(tile[8 * t8 + 2 * e + 1][i]) << 16;
        *reinterpret_cast<uint4*>(out + c * R + r) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// [R, 8] -> [keep, R], a row (16 bytes) per thread: the decoder's image, three of eight channels (1024 x
// 1024: 39 us on 32 x 32 tiles, seven eighths of them empty).
__global__ void __launch_bounds__(256) k_planes8(const bf16_t* __restrict__ in, bf16_t* __restrict__ out, int64_t R,
                                                 int keep) {
    const int64_t r = blockIdx.x * static_cast<int64_t>(256) + threadIdx.x;
    if (r >= R) return;
    const uint4 v = *reinterpret_cast<const uint4*>(in + r * 8);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int c = 0; c < 8; ++c)
        if (c < keep) out[c * R + r] = static_cast<bf16_t>(w[c >> 1] >> (16 * (c & 1)));
}

// ---- GroupNorm over [pixels, C] --------------------------------------------------------------
//
// One pass sums x and x^2 in fp64; the group's mean and variance follow from the two sums. A bf16
// value's square is exact in fp64 and both sums lose nothing that matters (they are exact up to 2^37
// times the smallest square), so the only cancellation is in the variance, n * sum(x^2) - sum(x)^2,
// which is formed in twice the precision: it equals the two-pass form's for any mean. Bound by
// reading x once (the two-pass form read it twice: 1.6 ms of a 1024px decode).
//
// A workgroup owns a chunk of pixels; thread t holds channel octet t % (C/8) of pixels
// t / (C/8), t / (C/8) + 256/(C/8), ...; the workgroup then sums each group's channels and rows in a
// fixed order into part[group][chunk].
constexpr int kGnThreads = 256;

__global__ void __launch_bounds__(kGnThreads) k_gn_stats(const bf16_t* __restrict__ x, int64_t S, int C, int G,
                                                       int64_t px_per_chunk, double* __restrict__ part) {
    __shared__ double red[kGnThreads][17];
    const int oct = C / 8, per_row = kGnThreads / oct;   // C/8 divides 256 (checked by the host)
    const int t = threadIdx.x, o = t % oct, prow = t / oct;
    const int cpg = C / G;
    const int64_t p0 = static_cast<int64_t>(blockIdx.x) * px_per_chunk;
    const int64_t p1 = min(S, p0 + px_per_chunk);
    double sum[8] = {0, 0, 0, 0, 0, 0, 0, 0}, sq[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t p = p0 + prow; p < p1; p += per_row) {
        const uint4 raw = *reinterpret_cast<const uint4*>(x + p * C + o * 8);
        const uint32_t w4[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const double v = __uint_as_float(q & 1 ? (w4[q >> 1] & 0xffff0000u) : (w4[q >> 1] << 16));
            sum[q] += v;
            sq[q] = __builtin_fma(v, v, sq[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        red[t][q] = sum[q];
        red[t][8 + q] = sq[q];
    }
    __syncthreads();
    if (t < 2 * G) {
        const int g = t >> 1, h = (t & 1) * 8;
        double s = 0.0;
        for (int r = 0; r < per_row; ++r)
            for (int c = g * cpg; c < (g + 1) * cpg; ++c) s += red[r * oct + c / 8][h + c % 8];
        part[(static_cast<int64_t>(g) * gridDim.x + blockIdx.x) * 2 + (t & 1)] = s;
    }
}

// Group g's statistics from its `count` pairs at part[g * count]: mean = s1 / n, var = (n s2 - s1^2) /
// n^2, inv = 1 / sqrt(float(var) + eps), the reference's rounding (ops_cpu.cpp:208-210), with the affine
// to the group's channels. One workgroup per group, summed in a fixed order.
constexpr int kGnFinThreads = 512;

__global__ void __launch_bounds__(kGnFinThreads) k_gn_finalize(const double* __restrict__ part, int64_t count,
                                                              double n, float eps, int cpg,
                                                              const bf16_t* __restrict__ w,
                                                              const bf16_t* __restrict__ b,
                                                              NormChannel* __restrict__ channels) {
#pragma clang fp contract(off)
    __shared__ double red[2][kGnFinThreads];
    const int g = blockIdx.x, t = threadIdx.x;
    const double2* src = reinterpret_cast<const double2*>(part) + g * count;
    double x1 = 0.0, x2 = 0.0;
#pragma unroll 4
    for (int64_t c = t; c < count; c += kGnFinThreads) {
        const double2 v = src[c];
        x1 += v.x;
        x2 += v.y;
    }
    red[0][t] = x1;
    red[1][t] = x2;
    __syncthreads();
    for (int w = kGnFinThreads / 2; w > 0; w >>= 1) {
        if (t < w) {
            red[0][t] += red[0][t + w];
            red[1][t] += red[1][t + w];
        }
        __syncthreads();
    }
    const double s1 = red[0][0], s2 = red[1][0];
    // n s2 - s1^2 with each product as a rounded value and its exact remainder
    const double p = n * s2, q = s1 * s1;
    const double num = (p - q) + (__builtin_fma(n, s2, -p) - __builtin_fma(s1, s1, -q));
    const double var = num <= 0.0 ? 0.0 : num / (n * n);   // a NaN stays one
    NormChannel nc;
    nc.mean = static_cast<float>(s1 / n);
    nc.inv = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(static_cast<float>(var), eps)));
    for (int c = g * cpg + t; c < (g + 1) * cpg; c += kGnFinThreads) {
        nc.w = w ? bf2f(w[c]) : 1.0f;
        nc.b = b ? bf2f(b[c]) : -0.0f;   // x + (-0.0) is x exactly
        channels[c] = nc;
    }
}

// norm8 or norm_silu8 over [S, C]. In place is allowed (each element is read before it is written by the same thread). The grid stride is a
// multiple of 256 and C/8 divides 256, so a thread always sees the same eight channels.
template <bool SILU>
__global__ void __launch_bounds__(256) k_gn_apply(const bf16_t* x, bf16_t* out, int64_t S, int C,
                                                  const NormChannel* __restrict__ channels) {
    const int oct = C / 8;
    const int64_t n = S * oct;
    const int64_t first = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    NormChannel nc[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        nc[q] = channels[static_cast<int>(first % oct) * 8 + q];
        if (SILU) nc[q] = norm_silu_channel(nc[q]);
    }
    const uint4* src = reinterpret_cast<const uint4*>(x);
    uint4* dst = reinterpret_cast<uint4*>(out);
    for (int64_t i = first; i < n; i += stride) {
        dst[i] = SILU ? norm_silu8(src[i], nc) : norm8(src[i], nc);
    }
}

// ---- GroupNorm over [C, pixels], the op's layout ------------------------------------------------
//
// A group is n consecutive values, a channel S of them, so both passes walk memory in order: no
// transposes to channels-last and back (97 of the op's 140 us at 512 x 36864). V: values per access,
// 8 (16 bytes) where group, channel and base allow, else 1.

template <int V>
__global__ void __launch_bounds__(kGnThreads) k_gn_stats_nchw(const bf16_t* __restrict__ x, int64_t n,
                                                            int64_t per_chunk, double* __restrict__ part) {
    __shared__ double red[2][kGnThreads];
    const int t = threadIdx.x;
    x += static_cast<int64_t>(blockIdx.y) * n;
    const int64_t i1 = min(n, (static_cast<int64_t>(blockIdx.x) + 1) * per_chunk);
    double a = 0.0, b = 0.0;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * per_chunk + t * V; i < i1; i += kGnThreads * V) {
        if constexpr (V == 8) {
            const uint4 raw = *reinterpret_cast<const uint4*>(x + i);
            const uint32_t w4[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const double v = __uint_as_float(q & 1 ? (w4[q >> 1] & 0xffff0000u) : (w4[q >> 1] << 16));
                a += v;
                b = __builtin_fma(v, v, b);
            }
        } else {
            const double v = bf2f(x[i]);
            a += v;
            b = __builtin_fma(v, v, b);
        }
    }
    red[0][t] = a;
    red[1][t] = b;
    __syncthreads();
    for (int w = kGnThreads / 2; w > 0; w >>= 1) {
        if (t < w) {
            red[0][t] += red[0][t + w];
            red[1][t] += red[1][t + w];
        }
        __syncthreads();
    }
    if (t < 2) part[(static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x) * 2 + t] = red[t][0];
}

// A channel per blockIdx.y. In place is allowed.
template <int V>
__global__ void __launch_bounds__(256) k_gn_apply_nchw(const bf16_t* x, bf16_t* out, int64_t S,
                                                       const NormChannel* __restrict__ channels) {
    NormChannel nc[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) nc[q] = channels[blockIdx.y];
    x += static_cast<int64_t>(blockIdx.y) * S;
    out += static_cast<int64_t>(blockIdx.y) * S;
    for (int64_t i = (blockIdx.x * static_cast<int64_t>(256) + threadIdx.x) * V; i < S;
         i += static_cast<int64_t>(gridDim.x) * 256 * V) {
        if constexpr (V == 8) {
            *reinterpret_cast<uint4*>(out + i) = norm8(*reinterpret_cast<const uint4*>(x + i), nc);
        } else {
            out[i] = static_cast<bf16_t>(norm8(make_uint4(x[i], 0, 0, 0), nc).x & 0xffffu);
        }
    }
}

// ---- direct convolution, channels-last, the reference's summation order ------------------------
//
// out[p, co] = bias[co] + sum over ci, ky, kx (in that order, taps outside the image skipped) of
// x[p + (ky - pad, kx - pad), ci] * w[co, ci, ky, kx], fp32 with separate multiply and add: the
// same operation sequence as conv2d_cpu (ops_cpu.cpp:276-300), so the result is bit-identical.
// A thread owns one pixel and CPT consecutive output channels; with VEC it reads 8 input channels
// of all 9 taps at once (16-byte loads), keeping the per-channel order.
template <int CPT, bool VEC>
__global__ void __launch_bounds__(256) k_conv_direct(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                     const bf16_t* __restrict__ bias, bf16_t* __restrict__ out,
                                                     int H, int W, int ci, int co, int k, int pad) {
    const int groups = (co + CPT - 1) / CPT;
    const int64_t idx = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (idx >= static_cast<int64_t>(H) * W * groups) return;
    const int cg = static_cast<int>(idx % groups);
    const int64_t p = idx / groups;
    const int y = static_cast<int>(p / W), xx = static_cast<int>(p - static_cast<int64_t>(y) * W);
    const int co0 = cg * CPT;
    float acc[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) acc[j] = (bias && co0 + j < co) ? bf2f(bias[co0 + j]) : 0.0f;
    const int kk = k * k;
    if constexpr (VEC) {
        for (int icb = 0; icb < ci; icb += 8) {
            float xv[9][8];
            bool ok[9];
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                const int ky = t / 3, kx = t % 3;
                const int iy = y + ky - pad, ix = xx + kx - pad;
                ok[t] = t < kk && iy >= 0 && iy < H && ix >= 0 && ix < W;
                uint4 raw = make_uint4(0, 0, 0, 0);
                if (ok[t]) raw = *reinterpret_cast<const uint4*>(x + (static_cast<int64_t>(iy) * W + ix) * ci + icb);
                const uint32_t w4[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    xv[t][q] = __uint_as_float(q & 1 ? (w4[q >> 1] & 0xffff0000u) : (w4[q >> 1] << 16));
            }
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int t = 0; t < 9; ++t) {
                    if (!ok[t]) continue;
#pragma unroll
                    for (int j = 0; j < CPT; ++j) {
                        if (co0 + j >= co) continue;
                        const float wv = bf2f(w[((static_cast<int64_t>(co0 + j) * ci + icb + q) * kk) + t]);
                        acc[j] = __fadd_rn(acc[j], __fmul_rn(xv[t][q], wv));
                    }
                }
        }
    } else {
        for (int ic = 0; ic < ci; ++ic)
            for (int ky = 0; ky < k; ++ky) {
                const int iy = y + ky - pad;
                if (iy < 0 || iy >= H) continue;
                for (int kx = 0; kx < k; ++kx) {
                    const int ix = xx + kx - pad;
                    if (ix < 0 || ix >= W) continue;
                    const float xv = bf2f(x[(static_cast<int64_t>(iy) * W + ix) * ci + ic]);
#pragma unroll
                    for (int j = 0; j < CPT; ++j) {
                        if (co0 + j >= co) continue;
                        const float wv = bf2f(w[((static_cast<int64_t>(co0 + j) * ci + ic) * k + ky) * k + kx]);
                        acc[j] = __fadd_rn(acc[j], __fmul_rn(xv, wv));
                    }
                }
            }
    }
#pragma unroll
    for (int j = 0; j < CPT; ++j)
        if (co0 + j < co) out[p * co + co0 + j] = f2bf(acc[j]);
}

// ---- nearest upsample, NCHW (UpsampleArgs, ops_cpu.cpp:384-397) ------------------------------

__global__ void __launch_bounds__(256) k_upsample_nchw(const bf16_t* __restrict__ in, bf16_t* __restrict__ out,
                                                       int64_t planes, int64_t H, int64_t W, int64_t f) {
    const int64_t H2 = H * f, W2 = W * f, n = planes * H2 * W2;
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t x = i % W2, y = (i / W2) % H2, pl = i / (H2 * W2);
        out[i] = in[(pl * H + y / f) * W + x / f];
    }
}

int grid_for(int64_t n, int per_block) {
    return static_cast<int>(std::min<int64_t>((n + per_block - 1) / per_block, 65535LL * 16));
}

// [co][ci][3][3] -> [co][3][3][ci]: the implicit GEMM's k index is (ky, kx, ci).
__global__ void k_repack3x3(const bf16_t* __restrict__ w, bf16_t* __restrict__ out, int64_t co,
                            int64_t ci) {
    const int64_t n = co * ci * 9;
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t c = i % ci, t = (i / ci) % 9, o = i / (ci * 9);
        out[i] = w[(o * ci + c) * 9 + t];
    }
}

// Scratch of the op-level entry points (NCHW at the boundary, channels-last inside): per device
// and slot, grown on demand, zero-filled when grown, kept until the process ends. Calls that
// overlap on one device share it.
enum OpSlot { SLOT_IN = 0, SLOT_OUT = 1, SLOT_W = 2, SLOT_ZERO = 3, SLOT_GN = 4, SLOT_COUNT = 5 };

void* op_workspace(int slot, size_t bytes) {
    static std::mutex mu;
    static void* ptr[64][SLOT_COUNT] = {};
    static size_t cap[64][SLOT_COUNT] = {};
    int dev = 0;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    require(dev >= 0 && dev < 64, "op workspace: device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (cap[dev][slot] < bytes) {
        if (ptr[dev][slot]) hip_check(hipFree(ptr[dev][slot]), "hipFree");
        ptr[dev][slot] = nullptr;
        cap[dev][slot] = 0;
        hip_check(hipMalloc(&ptr[dev][slot], bytes), "hipMalloc (op workspace)");
        hip_check(hipMemset(ptr[dev][slot], 0, bytes), "hipMemset (op workspace)");
        cap[dev][slot] = bytes;
    }
    return ptr[dev][slot];
}

GroupNormScratch op_gn_scratch() {
    GroupNormScratch sc;
    sc.max_chunks = 2048;
    char* base = static_cast<char*>(op_workspace(SLOT_GN, 2048 * 64 * 16 + 2048 * sizeof(NormChannel)));
    sc.part = reinterpret_cast<double*>(base);
    sc.channels = reinterpret_cast<NormChannel*>(base + 2048 * 64 * 16);
    return sc;
}

}  // namespace

void launch_repack3x3(const bf16_t* w, bf16_t* out, int64_t co, int64_t ci, hipStream_t s) {
    k_repack3x3<<<grid_for(co * ci * 9, 256), 256, 0, s>>>(w, out, co, ci);
    launch_check("repack 3x3 weights");
}

// Conv2dArgs (ops.h:120-126) at the op boundary, NCHW bf16, stride 1: per batch image the input
// goes channels-last, the convolution runs on the kernel its shape allows (3x3 "same" with
// c_in % 64 == 0: the MFMA implicit GEMM; 1x1: the MFMA GEMM; other "same" kernels: the direct
// kernel in the reference's order), and the output comes back to NCHW.
void launch_conv2d_nchw(const bf16_t* x, const bf16_t* w, const bf16_t* bias, bf16_t* out,
                        int64_t batch, int64_t ci, int64_t h, int64_t wd, int64_t co, int64_t k,
                        int64_t pad, hipStream_t s) {
    const int64_t ho = h + 2 * pad - k + 1, wo = wd + 2 * pad - k + 1;
    require(ho == h && wo == wd && 2 * pad == k - 1,
            "conv2d (hip-gfx950): only stride-1 'same' convolutions (2 * pad == k - 1) have a kernel");
    if (batch == 0 || co == 0 || h == 0 || wd == 0) return;
    const int64_t S = h * wd;
    bf16_t* xin = static_cast<bf16_t*>(op_workspace(SLOT_IN, static_cast<size_t>(S * ci * 2)));
    bf16_t* yout = static_cast<bf16_t*>(op_workspace(SLOT_OUT, static_cast<size_t>(S * co * 2)));
    const bool mfma3 = k == 3 && ci % 64 == 0 && co % 8 == 0 && h < (1 << 15) && wd < (1 << 15);
    bf16_t* wr = nullptr;
    if (mfma3) {
        wr = static_cast<bf16_t*>(op_workspace(SLOT_W, static_cast<size_t>(co * ci * 9 * 2)));
        launch_repack3x3(w, wr, co, ci, s);
    }
    for (int64_t b = 0; b < batch; ++b) {
        launch_transpose_bf16(x + b * ci * S, xin, 1, ci, S, s);
        if (mfma3) {
            ConvGeom g;
            g.in = xin;
            g.zero = static_cast<const bf16_t*>(op_workspace(SLOT_ZERO, 256));
            g.H = g.in_h = static_cast<int>(h);
            g.W = g.in_w = static_cast<int>(wd);
            g.c_in = static_cast<int>(ci);
            launch_conv3x3_bf16(g, wr, bias, yout, co, GemmEpilogue{}, s);
        } else if (k == 1) {
            launch_gemm_bf16(xin, w, bias, yout, S, co, ci, GemmEpilogue{}, s);
        } else {
            launch_conv_direct_nhwc(xin, w, bias, yout, h, wd, ci, co, k, pad, s);
        }
        launch_transpose_bf16(yout, out + b * co * S, 1, S, co, s);
    }
}

// NormArgs with groups > 0 (ops_cpu.cpp:186-224): rows = batch, cols = channels * spatial, NCHW.
void launch_group_norm_nchw(const bf16_t* x, const bf16_t* w, const bf16_t* b, bf16_t* out,
                            int64_t rows, int64_t cols, float eps, int64_t groups, int64_t channels,
                            hipStream_t s) {
    const int64_t C = channels ? channels : cols;
    require(cols % groups == 0, "groupnorm: channels*spatial not divisible by groups");
    require(C % groups == 0, "groupnorm: channels not divisible by groups");
    require(cols % C == 0, "groupnorm: cols is not a whole number of channel planes");
    require(gn_nhwc_supported(C, groups),
            "groupnorm (hip-gfx950): needs channels % 8 == 0 with channels / 8 dividing 256");
    const int64_t S = cols / C;
    if (rows == 0 || S == 0) return;
    GroupNormScratch sc = op_gn_scratch();
    const bool vec = S % 8 == 0 && (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
    const int64_t n = cols / groups;
    const int gi = static_cast<int>(groups);
    // chunks of a group: enough workgroups for the chip, at least a few passes of each over its chunk
    const int64_t unit = kGnThreads * (vec ? 8 : 1);
    const int64_t chunks = std::max<int64_t>(1, std::min<int64_t>({sc.max_chunks, 4096 / groups, (n + 4 * unit - 1) / (4 * unit)}));
    const int64_t per_chunk = ((n + chunks - 1) / chunks + 7) / 8 * 8;
    const int64_t blocks = std::min<int64_t>((S + 4 * unit - 1) / (4 * unit), 1024);
    ProfileScope ps(K_NORM, s, 6.0 * static_cast<double>(rows * cols));
    for (int64_t r = 0; r < rows; ++r) {
        const bf16_t* xr = x + r * cols;
        bf16_t* outr = out + r * cols;
        const dim3 gs(static_cast<unsigned>(chunks), static_cast<unsigned>(gi));
        const dim3 ga(static_cast<unsigned>(blocks), static_cast<unsigned>(C));
        if (vec) k_gn_stats_nchw<8><<<gs, kGnThreads, 0, s>>>(xr, n, per_chunk, sc.part);
        else k_gn_stats_nchw<1><<<gs, kGnThreads, 0, s>>>(xr, n, per_chunk, sc.part);
        k_gn_finalize<<<gi, kGnFinThreads, 0, s>>>(sc.part, chunks, static_cast<double>(n), eps,
                                                   static_cast<int>(C / groups), w, b, sc.channels);
        if (vec) k_gn_apply_nchw<8><<<ga, 256, 0, s>>>(xr, outr, S, sc.channels);
        else k_gn_apply_nchw<1><<<ga, 256, 0, s>>>(xr, outr, S, sc.channels);
        launch_check("groupnorm (nchw)");
    }
}


// ---- launchers (declared in common.h) ---------------------------------------------------------

namespace {
// 16-byte runs where both sides have them and fill most of a tile's width (8 channels of a 3-channel
// image would leave seven eighths of it idle).
void launch_transpose(const bf16_t* in, bf16_t* out, int64_t batch, int64_t R, int64_t C, int64_t keep, hipStream_t s) {
    const bool vec = R % 8 == 0 && C % 8 == 0 && C >= 32 && R >= 32 &&
                     (reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
    const int side = vec ? 64 : 32;
    const dim3 grid(static_cast<unsigned>((keep + side - 1) / side), static_cast<unsigned>((R + side - 1) / side),
                    static_cast<unsigned>(batch));
    if (C == 8 && batch == 1 && (R + 255) / 256 < (int64_t{1} << 31) && reinterpret_cast<uintptr_t>(in) % 16 == 0)
        k_planes8<<<static_cast<unsigned>((R + 255) / 256), 256, 0, s>>>(in, out, R, static_cast<int>(keep));
    else if (vec) k_transpose_v8<<<grid, 256, 0, s>>>(in, out, R, C, keep);
    else k_transpose<<<grid, 256, 0, s>>>(in, out, R, C, keep);
    launch_check("transpose");
}
}  // namespace

void launch_transpose_bf16(const bf16_t* in, bf16_t* out, int64_t batch, int64_t R, int64_t C,
                           hipStream_t s) {
    if (batch == 0 || R == 0 || C == 0) return;
    require((R + 31) / 32 <= 65535 && batch <= 65535, "transpose: too many rows for one launch");
    ProfileScope ps(K_ELEMENTWISE, s, 4.0 * static_cast<double>(batch * R * C));
    launch_transpose(in, out, batch, R, C, C, s);
}

void launch_transpose_keep_bf16(const bf16_t* in, bf16_t* out, int64_t R, int64_t C, int64_t keep,
                                hipStream_t s) {
    if (R == 0 || keep == 0) return;
    require(keep <= C && (R + 31) / 32 <= 65535, "transpose: kept columns or rows out of range");
    ProfileScope ps(K_ELEMENTWISE, s, 2.0 * static_cast<double>(R * (C + keep)));
    launch_transpose(in, out, 1, R, C, keep, s);
}

// Rows [S][C] -> [S][Cp] with columns C..Cp-1 zero (Cp >= C): the latent, padded to the implicit
// GEMM's 64-channel k-tile.
__global__ void __launch_bounds__(256) k_pad_rows(const bf16_t* __restrict__ in, bf16_t* __restrict__ out,
                                                  int64_t S, int64_t C, int64_t Cp) {
    const int64_t n = S * Cp;
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t c = i % Cp, p = i / Cp;
        out[i] = c < C ? in[p * C + c] : bf16_t{0};
    }
}

void launch_pad_rows(const bf16_t* in, bf16_t* out, int64_t S, int64_t C, int64_t Cp, hipStream_t s) {
    ProfileScope ps(K_ELEMENTWISE, s, 2.0 * static_cast<double>(S * (C + Cp)));
    k_pad_rows<<<grid_for(S * Cp, 256), 256, 0, s>>>(in, out, S, C, Cp);
    launch_check("pad rows");
}

// w [co][ci][3][3] -> out [cop][3][3][cip] zero-padded (cop >= co, cip >= ci).
__global__ void k_repack3x3_pad(const bf16_t* __restrict__ w, bf16_t* __restrict__ out, int64_t co,
                                int64_t ci, int64_t cop, int64_t cip) {
    const int64_t n = cop * cip * 9;
    for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t c = i % cip, t = (i / cip) % 9, o = i / (cip * 9);
        out[i] = (o < co && c < ci) ? w[(o * ci + c) * 9 + t] : bf16_t{0};
    }
}

void launch_repack3x3_pad(const bf16_t* w, bf16_t* out, int64_t co, int64_t ci, int64_t cop,
                          int64_t cip, hipStream_t s) {
    k_repack3x3_pad<<<grid_for(cop * cip * 9, 256), 256, 0, s>>>(w, out, co, ci, cop, cip);
    launch_check("repack 3x3 weights (padded)");
}

bool gn_nhwc_supported(int64_t C, int64_t G) {
    return C % 8 == 0 && C / 8 <= kGnThreads && kGnThreads % (C / 8) == 0 && G > 0 && G <= 64 &&
           C % G == 0;
}

void launch_group_norm_channels(const bf16_t* x, int64_t S, int64_t C, int64_t G, float eps,
                                const bf16_t* w, const bf16_t* b, GroupNormScratch& sc, hipStream_t s,
                                int64_t stats_rows) {
    require(gn_nhwc_supported(C, G), "groupnorm (nhwc): unsupported channel / group count");
    require(stats_rows == 0 || (C / G) % 4 == 0, "groupnorm (nhwc): sums come by runs of four channels");
    const int ci = static_cast<int>(C), gi = static_cast<int>(G);
    ProfileScope ps(K_NORM, s, stats_rows ? 0.0 : 2.0 * static_cast<double>(S * C));
    int64_t count = stats_rows * (C / G / 4);
    if (count == 0) {
        const int chunks = static_cast<int>(std::min<int64_t>(sc.max_chunks, std::max<int64_t>(1, (S + 15) / 16)));
        k_gn_stats<<<chunks, kGnThreads, 0, s>>>(x, S, ci, gi, (S + chunks - 1) / chunks, sc.part);
        count = chunks;
    }
    k_gn_finalize<<<gi, kGnFinThreads, 0, s>>>(sc.part, count, static_cast<double>(S) * (C / G), eps, ci / gi, w, b,
                                               sc.channels);
    launch_check("groupnorm statistics (nhwc)");
}

void launch_group_norm_apply(const bf16_t* x, bf16_t* out, int64_t S, int64_t C, bool silu,
                             const GroupNormScratch& sc, hipStream_t s) {
    ProfileScope ps(K_NORM, s, 4.0 * static_cast<double>(S * C));
    // four octets or more a thread: it reads its eight channels' statistics (128 bytes) once
    const int blocks = grid_for((S * (C / 8) + 3) / 4, 256);
    if (silu) k_gn_apply<true><<<blocks, 256, 0, s>>>(x, out, S, static_cast<int>(C), sc.channels);
    else k_gn_apply<false><<<blocks, 256, 0, s>>>(x, out, S, static_cast<int>(C), sc.channels);
    launch_check("groupnorm (nhwc)");
}

void launch_conv_direct_nhwc(const bf16_t* x, const bf16_t* w, const bf16_t* bias, bf16_t* out,
                             int64_t H, int64_t W, int64_t ci, int64_t co, int64_t k, int64_t pad,
                             hipStream_t s) {
    require(k >= 1 && k <= 3 && 2 * pad == k - 1, "conv (direct): odd kernel up to 3, same padding");
    require(H * W < (int64_t{1} << 31) && co < 65536 && ci < 65536, "conv (direct): too large");
    ProfileScope ps(K_ELEMENTWISE, s, 2.0 * static_cast<double>(H * W) * ci * co * k * k);
    const int hh = static_cast<int>(H), ww = static_cast<int>(W), cii = static_cast<int>(ci),
              coo = static_cast<int>(co), kk = static_cast<int>(k), pp = static_cast<int>(pad);
    const bool vec = ci % 8 == 0 && k == 3 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
    if (co <= 4) {
        const int64_t n = H * W;
        if (vec) k_conv_direct<4, true><<<grid_for(n, 256), 256, 0, s>>>(x, w, bias, out, hh, ww, cii, coo, kk, pp);
        else k_conv_direct<4, false><<<grid_for(n, 256), 256, 0, s>>>(x, w, bias, out, hh, ww, cii, coo, kk, pp);
    } else {
        const int64_t n = H * W * ((co + 7) / 8);
        if (vec) k_conv_direct<8, true><<<grid_for(n, 256), 256, 0, s>>>(x, w, bias, out, hh, ww, cii, coo, kk, pp);
        else k_conv_direct<8, false><<<grid_for(n, 256), 256, 0, s>>>(x, w, bias, out, hh, ww, cii, coo, kk, pp);
    }
    launch_check("conv (direct)");
}

void launch_upsample_nchw(const bf16_t* in, bf16_t* out, int64_t planes, int64_t H, int64_t W,
                          int64_t f, hipStream_t s) {
    const int64_t n = planes * H * W * f * f;
    if (n == 0) return;
    ProfileScope ps(K_ELEMENTWISE, s, 2.0 * static_cast<double>(n + planes * H * W));
    k_upsample_nchw<<<grid_for(n, 256), 256, 0, s>>>(in, out, planes, H, W, f);
    launch_check("upsample");
}

}  // namespace bh
