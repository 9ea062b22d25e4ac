// The VAE mid-block's attention on gfx950: one head, head_dim 512, no mask:
// softmax(Q K^T / sqrt(512)) V over S tokens, bf16 in and out.
//
// A workgroup of four waves owns 128 queries, a wave two 16-query tiles; one wave per SIMD, so each
// has 512 registers: 256 of output sums (O^T as 32 16-dim tiles x 2), 128 of Q. Keys stream in
// blocks of 32 through two K and two V^T stages of 32 KiB each, filled by direct global->LDS loads.
// Both products run on v_mfma_f32_16x16x32_bf16 with transposed tiles (S^T = K Q^T, O^T += V^T P^T), so
// P goes from the score accumulators to the output product without leaving registers.
//
// What bounds it: the fragment reads and the MFMAs. A fragment read (1 KiB) feeds as many MFMAs as
// the wave has query tiles; with one tile per wave (64 queries a workgroup) the LDS had to deliver
// 64 KiB per 64 MFMAs of every wave, and scores, softmax and output product ran one after another:
// 395 TFLOP/s at 16384 tokens. Two tiles halve the reads per MFMA, and the softmax of block j runs
// between the score MFMAs of block j + 1, and the maximum of block j + 1 between the output MFMAs
// of block j. At 16384 tokens 1392 -> 517 us (1063 TFLOP/s; 604 us with a block's sixteen loads
// issued in one burst after the barrier), at 4096 350 -> 53 us and 14 for the combine.
//
// 128 queries a workgroup leave CUs idle below 32768 tokens, so the keys split over up to 16
// workgroups per query block (flash512_splits), which write unnormalised fp32 sums, combined in split
// order.
//
// Softmax in fp32 with the running maximum in log2 units; it moves only when a block beats it by
// more than 8 (any fixed reference gives the same normalised result; the bound keeps P below
// 2^8). P is rounded to bf16 for the MFMA and the denominator sums those rounded values. Keys past S
// score -inf.
#include "common.h"

#include <algorithm>
#include <atomic>
#include <cmath>

namespace bh {
namespace {

constexpr int kD = 512;
constexpr int kQ = 128;                 // queries per workgroup
constexpr int kKv = 32;                 // keys per block
constexpr int kStage = kKv * kD * 2;    // 32 KiB: a block's K rows, or its V^T
constexpr int kMaxSplits = 16;

struct Args {
    const bf16_t* q;
    const bf16_t* k;
    const bf16_t* vt;
    bf16_t* out;
    float* part;    // [splits][S][512] sums, then [splits][S][2] maximum and denominator; or null
    int S;
    int qblocks;
    float c;        // scale * log2(e)
};

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// One global_load_lds_dwordx4: lane L's 16 bytes at `src` land at LDS address lds + 16 L.
__device__ __forceinline__ void dma16(const void* src, const char* lds) {
    const uint32_t l = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)(lds)));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                 :
                 : "s"(l), "v"(src)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

__device__ __forceinline__ bf16x8_t frag(const char* p) { return *reinterpret_cast<const bf16x8_t*>(p); }

// Sum or maximum over the four lanes lr, lr + 16, lr + 32, lr + 48.
__device__ __forceinline__ float over_rows(float v, bool is_max) {
    uint32_t x = __float_as_uint(v);
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    float a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
    v = is_max ? fmaxf(a, b) : a + b;
    x = __float_as_uint(v);
    const auto w = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    a = __uint_as_float(w[0]);
    b = __uint_as_float(w[1]);
    return is_max ? fmaxf(a, b) : a + b;
}

// K rows in LDS are 1 KiB (512 dims); 16-byte chunk c of row r sits at c ^ (r & 15), so the 16
// rows a fragment read touches hit 16 different chunks of one 256-byte span (all 64 banks). V^T is
// stored in global memory the way a wave reads it (k_vt512): both are copied 1 KiB at a time.
// A wave's i-th of eight loads of a block.
__device__ __forceinline__ void dma_k(char* st, const Args& a, int j, int i, int wave, int lane) {
    const int row = i * 4 + wave;
    const int key = min(j * kKv + row, a.S - 1);
    dma16(a.k + static_cast<int64_t>(key) * kD + (lane ^ (row & 15)) * 8, st + row * 1024);
}
__device__ __forceinline__ void dma_v(char* st, const Args& a, int j, int i, int wave, int lane) {
    const int piece = i * 4 + wave;
    dma16(a.vt + static_cast<int64_t>(j) * (kKv * kD) + piece * 512 + lane * 8, st + piece * 1024);
}

// The output product. Its 256 sums live in accumulation registers, which the compiler does not
// choose by itself next to scores that the vector unit reads every block (it copies every sum in
// and out, four moves each way per MFMA, or spills), so this MFMA is written as an instruction. The
// waits the compiler would otherwise insert around it are explicit:
//  - its P operands were written by vector instructions: probs_ready() leaves the two wait states
//    between them and the first of these MFMAs (V^T fragments come from LDS reads, whose
//    completion the compiler waits for);
//  - its sums are read by vector instructions only after settle(): an MFMA of eight passes needs
//    at most 18 wait states before its result may be read;
//  - between MFMAs the same sum returns 62 MFMAs later.
__device__ __forceinline__ void output(f32x4_t& o, const bf16x8_t& v, const bf16x8_t& p) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(o) : "v"(v), "v"(p));
}
__device__ __forceinline__ void probs_ready(bf16x8_t (&p)[2]) {
    asm volatile("s_nop 3" : "+v"(p[0]), "+v"(p[1]));
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void keep_sums(f32x4_t (&o)[32][2]) {   // here the sums are in accumulation registers
#pragma unroll
    for (int i = 0; i < 32; i += 8)
        asm volatile("" : "+a"(o[i][0]), "+a"(o[i][1]), "+a"(o[i + 1][0]), "+a"(o[i + 1][1]), "+a"(o[i + 2][0]),
                     "+a"(o[i + 2][1]), "+a"(o[i + 3][0]), "+a"(o[i + 3][1]), "+a"(o[i + 4][0]), "+a"(o[i + 4][1]),
                     "+a"(o[i + 5][0]), "+a"(o[i + 5][1]), "+a"(o[i + 6][0]), "+a"(o[i + 6][1]), "+a"(o[i + 7][0]),
                     "+a"(o[i + 7][1]));
}
__device__ __forceinline__ void settle(f32x4_t (&o)[32][2]) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 15");
    keep_sums(o);   // and every read of a sum follows the wait
    __builtin_amdgcn_sched_barrier(0);
}

// Every wave's loads have landed and every wave has finished reading the other stages.
__device__ __forceinline__ void join() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    s_waitcnt<0, 0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

__global__ void __launch_bounds__(256, 1) k_flash512(Args a) {
    __shared__ __attribute__((aligned(1024))) char smem[4 * kStage];   // K, K, V^T, V^T
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15, hi = lane >> 4;
    const int nblk_all = (a.S + kKv - 1) / kKv;
    const int splits = gridDim.x / a.qblocks;
    const int qb = blockIdx.x % a.qblocks, sp = blockIdx.x / a.qblocks;
    const int b0 = static_cast<int>(static_cast<int64_t>(nblk_all) * sp / splits);
    const int b1 = static_cast<int>(static_cast<int64_t>(nblk_all) * (sp + 1) / splits);
    const int q0 = qb * kQ + wave * 32;

#pragma unroll
    for (int i = 0; i < 8; ++i) dma_k(smem, a, b0, i, wave, lane);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        dma_v(smem + 2 * kStage, a, b0, i, wave, lane);
        if (b0 + 1 < b1) dma_k(smem + kStage, a, b0 + 1, i, wave, lane);
    }
    bf16x8_t qf[2][16];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int qc = min(q0 + 16 * u + lr, a.S - 1);
#pragma unroll
        for (int ks = 0; ks < 16; ++ks)
            qf[u][ks] = *reinterpret_cast<const bf16x8_t*>(a.q + static_cast<int64_t>(qc) * kD + 32 * ks + 8 * hi);
    }
    f32x4_t o[32][2];
#pragma unroll
    for (int dt = 0; dt < 32; ++dt)
#pragma unroll
        for (int u = 0; u < 2; ++u) o[dt][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    keep_sums(o);
    float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
    f32x4_t s[2][2], sn[2][2];   // [key tile][query tile]

    auto clear = [&](f32x4_t (&x)[2][2]) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int u = 0; u < 2; ++u) x[kt][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    // The K fragments of step ks (32 dims): both key tiles.
    auto k_read = [&](bf16x8_t (&f)[2], const char* st, int ks) {
        const int pc = ((4 * ks + hi) ^ lr) * 16;
        f[0] = frag(st + lr * 1024 + pc);
        f[1] = frag(st + (16 + lr) * 1024 + pc);
    };
    auto score = [&](f32x4_t (&x)[2][2], const bf16x8_t (&f)[2], int ks) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            x[0][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[0], qf[u][ks], x[0][u], 0, 0, 0);
            x[1][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[1], qf[u][ks], x[1][u], 0, 0, 0);
        }
    };
    // Score element e (key tile e / 8, query tile (e / 4) % 2) in log2 units; keys past S never count.
    auto scale = [&](f32x4_t (&x)[2][2], int e, int j) {
        const int kt = e >> 3, u = (e >> 2) & 1, t = e & 3;
        const float v = x[kt][u][t] * a.c;
        x[kt][u][t] = j * kKv + 16 * kt + 4 * hi + t < a.S ? v : -INFINITY;
    };
    auto block_max = [&](const f32x4_t (&x)[2][2], int u) {
        float mx = fmaxf(fmaxf(x[0][u][0], x[0][u][1]), fmaxf(x[0][u][2], x[0][u][3]));
        mx = fmaxf(mx, fmaxf(fmaxf(x[1][u][0], x[1][u][1]), fmaxf(x[1][u][2], x[1][u][3])));
        return over_rows(mx, true);
    };
    auto rescale = [&](const float (&mx)[2]) {
        if (!__any(mx[0] > m[0] + 8.0f || mx[1] > m[1] + 8.0f)) return;
        settle(o);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const float mn = fmaxf(m[u], mx[u]);
            const float alpha = exp2f(m[u] - mn);   // 0 on the first block (m = -inf)
            m[u] = mn;
            l[u] *= alpha;
#pragma unroll
            for (int dt = 0; dt < 32; ++dt) {   // four registers at a time: 256 do not fit beside Q
#pragma unroll
                for (int t = 0; t < 4; ++t) o[dt][u][t] *= alpha;
                asm volatile("" : "+a"(o[dt][u]));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    bf16x8_t pf[2];
    auto prob = [&](int e, int u) {   // element e of the lane's eight keys of query tile u
        const __bf16 pb = static_cast<__bf16>(__builtin_amdgcn_exp2f(s[e >> 2][u][e & 3] - m[u]));
        pf[u][e] = pb;
        l[u] += static_cast<float>(pb);
    };
    auto v_read = [&](const char* st, int dt) { return frag(st + dt * 1024 + lane * 16); };

    if (b0 < b1) {
        join();
        clear(s);
#pragma unroll
        for (int ks = 0; ks < 16; ++ks) {
            bf16x8_t f[2];
            k_read(f, smem, ks);
            score(s, f, ks);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) scale(s, e, b0);
#pragma unroll
        for (int u = 0; u < 2; ++u) m[u] = fmaxf(m[u], block_max(s, u));   // no sums to rescale yet
        for (int j = b0; j + 1 < b1; ++j) {
            const int x = (j - b0) & 1;
            join();   // K of block j + 1 and V^T of block j are complete; K of j and V^T of j - 1 are free
            const char* kst = smem + (x ^ 1) * kStage;
            const char* vst = smem + (2 + x) * kStage;
            bf16x8_t kf[3][2], vf[4];
#pragma unroll
            for (int ks = 0; ks < 3; ++ks) k_read(kf[ks], kst, ks);
            char* k_free = smem + x * kStage;
            char* v_free = smem + (2 + (x ^ 1)) * kStage;
            clear(sn);
            // Scores of block j + 1, a K step's four MFMAs beside one probability of block j;
            // fragments are read three steps ahead. The next loads (the last block's again past it)
            // go out one at a time under the MFMAs: a load holds its wave while the address unit is
            // busy with the other waves' loads.
            const int jk = min(j + 2, b1 - 1);
#pragma unroll
            for (int ks = 0; ks < 16; ++ks) {
                score(sn, kf[ks % 3], ks);
                if (ks + 3 < 16) k_read(kf[ks % 3], kst, ks + 3);
                if (ks >= 12) vf[ks - 12] = v_read(vst, ks - 12);
                if (ks & 1) dma_k(k_free, a, jk, ks >> 1, wave, lane);
                prob(ks >> 1, ks & 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            // Output of block j, beside the maximum of block j + 1.
            probs_ready(pf);
            float mx[2];
#pragma unroll
            for (int dt = 0; dt < 32; ++dt) {
#pragma unroll
                for (int u = 0; u < 2; ++u) output(o[dt][u], vf[dt & 3], pf[u]);
                if (dt + 4 < 32) vf[dt & 3] = v_read(vst, dt + 4);
                if (dt < 16 && (dt & 1)) dma_v(v_free, a, j + 1, dt >> 1, wave, lane);
                if (dt < 16) scale(sn, dt, j + 1);
                if (dt == 17) mx[0] = block_max(sn, 0);
                if (dt == 21) mx[1] = block_max(sn, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            rescale(mx);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int u = 0; u < 2; ++u) s[kt][u] = sn[kt][u];
        }
        join();
#pragma unroll
        for (int e = 0; e < 16; ++e) prob(e >> 1, e & 1);
        const char* vst = smem + (2 + ((b1 - 1 - b0) & 1)) * kStage;
        bf16x8_t vf[4];
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) vf[dt] = v_read(vst, dt);
        probs_ready(pf);
#pragma unroll
        for (int dt = 0; dt < 32; ++dt) {
#pragma unroll
            for (int u = 0; u < 2; ++u) output(o[dt][u], vf[dt & 3], pf[u]);
            if (dt + 4 < 32) vf[dt & 3] = v_read(vst, dt + 4);
            __builtin_amdgcn_sched_barrier(0);
        }
        settle(o);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const float den = over_rows(l[u], false);
        const int q = q0 + 16 * u + lr;
        if (q >= a.S) continue;
        if (a.part) {
            float* row = a.part + (static_cast<int64_t>(sp) * a.S + q) * kD + 4 * hi;
#pragma unroll
            for (int dt = 0; dt < 32; ++dt) *reinterpret_cast<f32x4_t*>(row + 16 * dt) = o[dt][u];
            if (hi == 0) {
                float* ml = a.part + static_cast<int64_t>(splits) * a.S * kD + (static_cast<int64_t>(sp) * a.S + q) * 2;
                ml[0] = m[u];
                ml[1] = den;
            }
            continue;
        }
        bf16_t* row = a.out + static_cast<int64_t>(q) * kD + 4 * hi;
        const float r = __frcp_rn(den);   // one reciprocal per query, a multiply per output
#pragma unroll
        for (int dt = 0; dt < 32; ++dt)
            *reinterpret_cast<uint2*>(row + 16 * dt) =
                make_uint2(f2bf2(o[dt][u][0] * r, o[dt][u][1] * r), f2bf2(o[dt][u][2] * r, o[dt][u][3] * r));
    }
}

// out[q] = sum_s 2^(m_s - M) o_s[q] / sum_s 2^(m_s - M) l_s over the splits in order. A wave per
// query, eight dims a lane; bound by the partials it reads, or by the latency of its loads where there are few: lane s
// holds split s's maximum and denominator (one load for all of them), and kAtOnce splits' sums are requested at once.
template <int kAtOnce>
__global__ void __launch_bounds__(256) k_flash512_combine(const float* __restrict__ part, bf16_t* __restrict__ out,
                                                          int S, int splits) {
    const int q = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (q >= S) return;
    const float* ml = part + static_cast<int64_t>(splits) * S * kD;
    const float2 mine = *reinterpret_cast<const float2*>(ml + (static_cast<int64_t>(min(lane, splits - 1)) * S + q) * 2);
    f32x4_t x[kAtOnce], y[kAtOnce];
    auto request = [&](int s0) {   // splits past the last are read again, unused
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) {
            const float* row = part + (static_cast<int64_t>(min(s0 + i, splits - 1)) * S + q) * kD + lane * 8;
            x[i] = *reinterpret_cast<const f32x4_t*>(row);
            y[i] = *reinterpret_cast<const f32x4_t*>(row + 4);
        }
    };
    request(0);
    float top = mine.x;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = fmaxf(top, __shfl_xor(top, o, 64));
    const float weight = exp2f(mine.x - top);
    f32x4_t lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
    for (int s0 = 0; s0 < splits; s0 += kAtOnce) {
        if (s0 > 0) request(s0);
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i) {
            if (s0 + i >= splits) break;
            const float w = __shfl(weight, s0 + i, 64);
            den += w * __shfl(mine.y, s0 + i, 64);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                lo[t] += w * x[i][t];
                hi[t] += w * y[i][t];
            }
        }
    }
    const float r = __frcp_rn(den);
    *reinterpret_cast<uint4*>(out + static_cast<int64_t>(q) * kD + lane * 8) =
        make_uint4(f2bf2(lo[0] * r, lo[1] * r), f2bf2(lo[2] * r, lo[3] * r), f2bf2(hi[0] * r, hi[1] * r),
                   f2bf2(hi[2] * r, hi[3] * r));
}

// V [S, 512] -> V^T by blocks of 32 keys in the order a wave reads it: block j, 16-dim tile dt, lane
// (lr, hi): the eight keys 4 hi + 0..3 and 16 + 4 hi + 0..3 of dim 16 dt + lr, the keys that lane
// holds after a pair of 16x16 score tiles. Zero past S. A block's 64 dims per workgroup.
__global__ void __launch_bounds__(256) k_vt512(const bf16_t* __restrict__ v, bf16_t* __restrict__ vt, int S) {
    __shared__ __attribute__((aligned(16))) bf16_t tile[kKv][72];
    const int key0 = blockIdx.x * kKv, d0 = blockIdx.y * 64, t = threadIdx.x;
    {
        const int row = t >> 3, c = t & 7, key = key0 + row;
        uint4 x = make_uint4(0, 0, 0, 0);
        if (key < S) x = *reinterpret_cast<const uint4*>(v + static_cast<int64_t>(key) * kD + d0 + c * 8);
        *reinterpret_cast<uint4*>(&tile[row][c * 8]) = x;
    }
    __syncthreads();
    const int dt = t >> 6, lane = t & 63, lr = lane & 15, hi = lane >> 4;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int key = 4 * hi + 2 * (e & 1) + 16 * (e >> 1);
        w[e] = tile[key][16 * dt + lr] | static_cast<uint32_t>(tile[key + 1][16 * dt + lr]) << 16;
    }
    *reinterpret_cast<uint4*>(vt + static_cast<int64_t>(blockIdx.x) * (kKv * kD) + (d0 / 16 + dt) * 512 + lane * 8) =
        make_uint4(w[0], w[1], w[2], w[3]);
}

int device_cus() {
    static std::atomic<int> cus[64] = {};
    int dev = 0;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    require(dev >= 0 && dev < 64, "attention: device index out of range");
    int n = cus[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        hip_check(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev),
                  "hipDeviceGetAttribute");
        require(n > 0, "attention: device reports no compute units");
        cus[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

int64_t vt_elems(int64_t S) { return (S + kKv - 1) / kKv * kKv * kD; }

}  // namespace

int64_t flash512_scratch_elems(int64_t S, int splits) {
    return vt_elems(S) + (splits > 1 ? splits * S * (kD + 2) * 2 : 0);   // bf16 elements
}

// The key splits of S tokens, at most what `scratch_bytes` holds beside V^T: the least estimated
// time. A workgroup takes about 1.7 us per block (4096 tokens in 1, 2 and 4 splits: 224, 128 and 79 us) and
// ~4 us at its ends; the combine ~3 us, and the partials of one split are S x 2 KiB written and read at
// ~4.5 TB/s. Few tokens: 64 in 1 and 2 splits 14.5 and 15.1 us, 100 in 1 and 4 20.7 and 18.4.
int flash512_splits(int64_t S, int64_t scratch_bytes) {
    const int64_t cus = device_cus(), qb = (S + kQ - 1) / kQ, nblk = (S + kKv - 1) / kKv;
    int best = 1;
    double best_cost = -1.0;
    for (int sp = 1; sp <= kMaxSplits && sp <= nblk; ++sp) {
        if (sp > 1 && flash512_scratch_elems(S, sp) * 2 > scratch_bytes) break;
        const int64_t rounds = (qb * sp + cus - 1) / cus;
        const double cost = rounds * (((nblk + sp - 1) / sp) * 1.7 + 4.0) +
                            (sp > 1 ? 3.0 + sp * static_cast<double>(S) * 4096.0 / 4.5e6 : 0.0);
        if (best_cost < 0 || cost < best_cost) {
            best = sp;
            best_cost = cost;
        }
    }
    return best;
}

void launch_attention512(const bf16_t* q, const bf16_t* k, const bf16_t* v, bf16_t* scratch, int splits,
                         bf16_t* out, int64_t S, float scale, hipStream_t s) {
    require(S > 0 && S < (int64_t{1} << 30), "attention (head_dim 512): sequence length");
    require(splits >= 1 && splits <= kMaxSplits, "attention (head_dim 512): key splits");
    const int n = static_cast<int>(S);
    {
        ProfileScope ps(K_ELEMENTWISE, s, 4.0 * static_cast<double>(S) * kD);
        k_vt512<<<dim3(static_cast<unsigned>((S + kKv - 1) / kKv), kD / 64), 256, 0, s>>>(v, scratch, n);
        launch_check("attention (head_dim 512): V transpose");
    }
    Args a{q, k, scratch, out, splits > 1 ? reinterpret_cast<float*>(scratch + vt_elems(S)) : nullptr, n,
           static_cast<int>((S + kQ - 1) / kQ),
           (scale > 0.0f ? scale : 1.0f / std::sqrt(static_cast<float>(kD))) * 1.4426950408889634f};
    ProfileScope ps(K_ATTN_SELF, s, 4.0 * static_cast<double>(S) * S * kD);
    k_flash512<<<static_cast<unsigned>(a.qblocks) * splits, 256, 0, s>>>(a);
    if (splits > 1) {
        auto* combine = splits == 2 ? &k_flash512_combine<2> : splits <= 4 ? &k_flash512_combine<4> : &k_flash512_combine<8>;
        combine<<<static_cast<unsigned>((S + 3) / 4), 256, 0, s>>>(a.part, out, n, splits);
    }
    launch_check("attention (head_dim 512)");
}

}  // namespace bh
