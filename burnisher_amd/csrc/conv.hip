// 3x3 "same" convolution over channels-last bf16 for the VAE decoder on gfx950: an implicit GEMM
// out[pixel, c_out] = sum over (64 input channels, tap) of patch . W^T on the MFMA cores, with the
// input read once per 64-channel chunk instead of once per tap.
//
// A tile is a patch of 4 MT x 16 output pixels by 16 NT output channels. For each chunk of 64
// input channels the patch's input pixels with a one-pixel border ((4 MT + 2) x 18 rows of 128
// bytes) are loaded into LDS once, and the nine taps are nine k-steps that read their activation
// fragments from the same rows at a shift of (ky, kx) pixels; only the weights (16 NT rows of 128
// bytes per step) stream per tap. What bounds an MFMA kernel here is its operand stream into LDS
// (a 256 x 128 tile that gathers every tap moves 48 KiB per 64-deep k-step; this one moves
// 16 KiB of weights and 41 KiB / 9 of patch), so the steps run near the MFMA rate, and a short
// tile (MT = 1: 64 pixels) costs little more operand traffic per step than a tall one: a small
// image is cut finely enough to fill the chip.
//
// Four waves multiply and four move operands, as in the GEMM (gemm_tile.inc): a consumer wave owns
// some patch rows of 16 pixels and all or half of the channels. The weight ring holds S stages; at a step's
// barrier the weights of the NEXT step have landed too, so the consumers read the next step's
// first fragments under the current step's last MFMAs and no LDS latency is exposed between
// steps.
//
// LDS rows are 128 bytes (64 channels) with 16-byte chunk c at slot c ^ swizzle. The patch rows
// swizzle by the pixel's x: the sixteen rows of a fragment are sixteen consecutive pixels of one
// patch row, whatever the tap, so they cover all 64 banks once and the swizzle of a lane depends on
// (lane, kx) only.
//
// With NORM the convolution reads the raw tensor and applies its GroupNorm and SiLU itself: each
// producer wave normalises the patch rows it loaded, in LDS, as soon as they have landed, so the
// normalised tensor is never written to or read from memory. A pixel is normalised once per patch
// and chunk and 128 output channels, border included (1.27 times each on average with patches of 16 rows, 1.41
// with 8, 1.69 with 4), on waves that otherwise only issue
// loads, under the consumers' MFMAs; the ~10 vector instructions per value take issue slots from
// them (512 -> 512 at 128 x 128: 57 -> 75 us with the raw tensor read in place of the normalised
// one), less than the pass they replace as a whole: decode at 512px 3.32 -> 2.84 ms, at 1024px
// 11.95 -> 10.44 ms (interleaved A/B).
//
// Measured against the per-tap gather it replaces (256 x 128 tiles, three 48 KiB stages): 512 ->
// 512 channels at 128 x 128 pixels 74.5 -> 56.7 us (1036 -> 1364 TFLOP/s); 128 -> 128 at
// 512 x 512 (18 steps a tile) 83.5 -> 64 us; 512 -> 512 at 64 x 64 (64 tiles there, 256 here)
// 63 -> 26 us; the decoder's 3-channel output convolution at 512 x 512, on a 32-wide tile instead
// of a 144-wide one, 79 -> 25 us.
#include "common.h"

#include <algorithm>
#include <atomic>

namespace bh {
namespace {

#include "gemm_tile.inc"
using namespace gk;

constexpr int kPW = 18;                 // patch row: 16 output pixels and the border
constexpr int kPRow = kPW * kRowBytes;  // its bytes in LDS

__host__ __device__ constexpr int cmin(int a, int b) { return a < b ? a : b; }

template <int MT, int NT, bool NORM = false>
struct Halo {
    static constexpr int PY = 4 * MT;                          // output rows of a patch
    // The consumers as WM x WN: each reads WM-th of the patch rows' and WN-th of the weights'
    // fragments. A short tile splits both ways (at 4 x 1 every wave would read all the weights
    // for 16 pixels: 18 fragment reads per 16 MFMAs; 2 x 2 reads 12).
    static constexpr int WN = MT == 4 || NT < 8 ? 1 : 2;
    static constexpr int MW = MT * WN, NW = NT / WN;           // a wave's patch rows, 16-channel blocks
    static constexpr int kRows = (PY + 2) * kPW;               // input pixels of a patch
    static constexpr int kABlocks = (kRows + 7) / 8;           // 1 KiB DMA blocks of eight rows
    static constexpr int kABytes = kABlocks * 1024;
    static constexpr int kBBlocks = 2 * NT;
    static constexpr int kBBytes = kBBlocks * 1024;
    static constexpr int kBiasSlots = 4;
    static constexpr int kNormBytes = NORM ? 1024 : 0;         // a chunk's 64 channels of NormChannel
    // weight stages, after two patch buffers, the bias slots and the channels' norm
    static constexpr int S = cmin(8, (160 * 1024 - 2 * kABytes - kBiasSlots * kBiasSlotBytes - 2 * kNormBytes) / kBBytes);
    static constexpr int D = S - 1;                            // steps the weights are issued ahead
    static constexpr int kBOff = 2 * kABytes;
    static constexpr int kBiasOff = kBOff + S * kBBytes;
    static constexpr int kNormOff = kBiasOff + kBiasSlots * kBiasSlotBytes;
    static constexpr int kDumpOff = kNormOff + kNormBytes;     // where items past the patch's end go
    static constexpr int kSmemBytes = kDumpOff + kNormBytes;
    static constexpr int kBItems = (kBBlocks + 3) / 4;         // DMA instructions per wave and step
    static constexpr int kAItems = (kABlocks + 3) / 4;         // per wave and chunk
    // The next chunk's patch goes out in the first kASteps taps of a chunk, kAPer items a tap:
    // before (in issue order) the weights of that chunk's first step, which go out at tap 9 - D.
    // Items of tap t have landed at the barrier of tap t + D - 1; normalised there, they must be
    // complete at the barrier of tap 8, when the consumers read ahead into the next chunk.
    static constexpr int kTaps = 9 - D;
    static constexpr int kAPer = (kAItems + kTaps - 1) / kTaps;
    static constexpr int kASteps = (kAItems + kAPer - 1) / kAPer;
    static_assert(S >= 3 && kASteps + D - 2 <= 7 && kSmemBytes <= 160 * 1024, "LDS plan");
    // DMA instructions a wave issues in a step of this tap (taps count modulo 9).
    static constexpr int issued(int tap) { return kBItems + (tap < kASteps ? kAPer : 0); }
    // At a step's barrier the weights of the next step (issued D - 1 steps ago) have landed: the
    // D - 2 later steps' instructions may still be in flight.
    static constexpr int in_flight(int tap) {
        int n = 0;
        for (int q = 1; q <= D - 2; ++q) n += issued((tap + 9 - q) % 9);
        return n;
    }
};

struct ConvArgs {
    const bf16_t* in;
    const bf16_t* zero;    // 64 zero bf16: the source of pixels outside the image
    const bf16_t* w;       // [c_out][ky][kx][c_in]
    bf16_t* out;
    int H, W, in_w, c_in, up;
    int c_out;
    int tiles_x, tiles_n, tiles;   // patches per row, channel tiles, all tiles
    double* stats;         // or null: see row16_sum
    int64_t stats_rows;
    const NormChannel* norm;   // [c_in], NORM only
};

// Tile v -> patch origin and first channel. Workgroup b runs on XCD b % 8, so tiles are renumbered
// to give each XCD a contiguous band of patches; the channel tiles of one patch are neighbours,
// so a patch is fetched into that XCD's L2 once.
template <int MT, int NT>
__device__ __forceinline__ void conv_tile(const ConvArgs& a, int v, int& y0, int& x0, int& n0) {
    if ((a.tiles & 7) == 0) v = (v & 7) * (a.tiles >> 3) + (v >> 3);
    const int patch = v / a.tiles_n;
    n0 = (v - patch * a.tiles_n) * 16 * NT;
    const int ty = patch / a.tiles_x;
    y0 = ty * Halo<MT, NT>::PY;
    x0 = (patch - ty * a.tiles_x) * 16;
}

__device__ __forceinline__ uint32_t lds_addr(const char* p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)(p)));
}

// The producer waves. `cur` and `next` are the weight sources of the chunk being multiplied and of
// the one after it (across tiles); past the last chunk the sources repeat it, so that every step
// issues the same number of instructions, into buffers nobody reads again.
template <int MT, int NT, bool NORM>
__device__ __forceinline__ void conv_produce(char* smem, const ConvArgs& a, const bf16_t* bias,
                                             int my_tiles, int wave, int lane) {
    using G = Halo<MT, NT, NORM>;
    const int sub = lane >> 3, slot = lane & 7;
    const int chunks = a.c_in >> 6;
    const int64_t k = 9 * static_cast<int64_t>(a.c_in);
    int aoff[G::kAItems];                 // element offset of each patch item's source, -1 outside
    const bf16_t *cur[G::kBItems], *next[G::kBItems];

    // Items past the patch's end, there to keep the count, repeat its last block; where that block
    // may be normalised already, they go to a spare KiB instead.
    auto exists = [&](int i) { return i < G::kAItems && i * 4 + wave < G::kABlocks; };
    auto block_of = [&](int i) { return min(i * 4 + wave, G::kABlocks - 1); };
    const int octet = lane & 7;   // of the channels this lane normalises
    auto tile_sources = [&](int it) {
        int y0, x0, n0;
        conv_tile<MT, NT>(a, blockIdx.x + it * gridDim.x, y0, x0, n0);
#pragma unroll
        for (int i = 0; i < G::kAItems; ++i) {
            const int row = block_of(i) * 8 + sub;
            const int py = row / kPW, px = row - py * kPW;
            int sy = y0 + py - 1, sx = x0 + px - 1;
            const bool inside = row < G::kRows && static_cast<unsigned>(sy) < static_cast<unsigned>(a.H) &&
                                static_cast<unsigned>(sx) < static_cast<unsigned>(a.W);
            if (a.up) {
                sy >>= 1;
                sx >>= 1;
            }
            aoff[i] = inside ? (sy * a.in_w + sx) * a.c_in + (slot ^ ((px >> 1) & 7)) * 8 : -1;
        }
#pragma unroll
        for (int i = 0; i < G::kBItems; ++i) {
            const int row = min(i * 4 + wave, G::kBBlocks - 1) * 8 + sub;
            const int n = min(n0 + b_col(row), a.c_out - 1);
            next[i] = a.w + n * k + (slot ^ ((row >> 1) & 7)) * 8;
        }
        if (bias && wave == 0 && lane < 2 * NT) {
            const int n = min(n0 + lane * 8, a.c_out - 8);
            dma16(bias + n, smem + G::kBiasOff + (it % G::kBiasSlots) * kBiasSlotBytes);
        }
    };
    // kAPer items of a chunk's patch into `buf`
    auto issue_patch = [&](int first, int cb, char* buf) {
#pragma unroll
        for (int q = 0; q < G::kAPer; ++q) {
            const int i = cmin(first + q, G::kAItems - 1);
            const bf16_t* src = aoff[i] < 0 ? a.zero + slot * 8 : a.in + aoff[i] + cb * 64;
            dma16(src, NORM && !exists(first + q) ? smem + G::kDumpOff : buf + block_of(i) * 1024);
        }
    };
    // The channels' norm of chunk cb, 16 bytes a channel, into its LDS slot (wave 0).
    auto issue_norm = [&](int cb) {
        if (NORM && wave == 0) dma16(a.norm + cb * 64 + lane, smem + G::kNormOff);
    };
    // This lane's octet of them, from LDS.
    NormChannel nc[NORM ? 8 : 1];
    auto read_norm = [&]() {
        if constexpr (NORM) {
#pragma unroll
            for (int q = 0; q < 8; ++q)
                nc[q] = norm_silu_channel(reinterpret_cast<const NormChannel*>(smem + G::kNormOff)[octet * 8 + q]);
        }
    };
    // The items of issue_patch(first, ...) normalised in place: lane L takes channel octet L % 8 of
    // the pixel L / 8 of each block, wherever the swizzle put it; pixels outside the image stay
    // zero, as the convolution pads the normalised tensor.
    auto normalise_patch = [&](int first, char* buf) {
        if constexpr (NORM) {
            uint4 raw[G::kAPer];
            char* at[G::kAPer];
#pragma unroll
            for (int q = 0; q < G::kAPer; ++q) {
                const int row = block_of(first + q) * 8 + sub;
                at[q] = buf + row * kRowBytes + (octet ^ (((row % kPW) >> 1) & 7)) * 16;
                if (exists(first + q)) raw[q] = *reinterpret_cast<const uint4*>(at[q]);
            }
#pragma unroll
            for (int q = 0; q < G::kAPer; ++q)
                if (exists(first + q) && aoff[cmin(first + q, G::kAItems - 1)] >= 0)
                    *reinterpret_cast<uint4*>(at[q]) = norm_silu8(raw[q], nc);
        }
    };
    int bst = 0;   // the stage the next weights go to
    auto issue_weights = [&](const bf16_t* const (&src)[G::kBItems], int tap) {
        char* stage = smem + G::kBOff + bst * G::kBBytes;
#pragma unroll
        for (int i = 0; i < G::kBItems; ++i)
            dma16(src[i] + tap * a.c_in, stage + min(i * 4 + wave, G::kBBlocks - 1) * 1024);
        bst = bst == G::S - 1 ? 0 : bst + 1;
    };
    tile_sources(0);
#pragma unroll
    for (int i = 0; i < G::kBItems; ++i) cur[i] = next[i];
    issue_norm(0);
#pragma unroll
    for (int q = 0; q < G::kASteps; ++q) issue_patch(q * G::kAPer, 0, smem);
#pragma unroll
    for (int t = 0; t < G::D; ++t) issue_weights(cur, t);
    if (NORM) {
        wait_and_join<0>();   // every wave sees the channels' norm
        read_norm();
#pragma unroll
        for (int q = 0; q < G::kASteps; ++q) normalise_patch(q * G::kAPer, smem);
    }
    const int total = my_tiles * chunks;
    int it = 0, cb = 0;   // of the chunk after the one being multiplied
    for (int c = 0; c < total; ++c) {
        char* nbuf = smem + ((c + 1) & 1) * G::kABytes;
        if (c + 1 < total) {
            if (++cb == chunks) {
                cb = 0;
                ++it;
            }
        }
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            // unrolled, so the wait count is a constant of each copy
            switch (tap) {
                case 0: wait_and_join<G::in_flight(0)>(); break;
                case 1: wait_and_join<G::in_flight(1)>(); break;
                case 2: wait_and_join<G::in_flight(2)>(); break;
                case 3: wait_and_join<G::in_flight(3)>(); break;
                case 4: wait_and_join<G::in_flight(4)>(); break;
                case 5: wait_and_join<G::in_flight(5)>(); break;
                case 6: wait_and_join<G::in_flight(6)>(); break;
                case 7: wait_and_join<G::in_flight(7)>(); break;
                default: wait_and_join<G::in_flight(8)>(); break;
            }
            if (tap == 0 && c + 1 < total) {
                if (cb == 0) {
                    tile_sources(it);
                } else {
#pragma unroll
                    for (int i = 0; i < G::kBItems; ++i) next[i] = cur[i] + 64;
                }
            }
            if (tap == 0) issue_norm(cb);
            if (tap < G::kASteps) issue_patch(tap * G::kAPer, cb, nbuf);
            if (tap + G::D < 9) issue_weights(cur, tap + G::D);
            else issue_weights(next, tap + G::D - 9);
            if (tap == G::D - 1) read_norm();
            if (tap >= G::D - 1 && tap - (G::D - 1) < G::kASteps)
                normalise_patch((tap - (G::D - 1)) * G::kAPer, nbuf);
        }
#pragma unroll
        for (int i = 0; i < G::kBItems; ++i) cur[i] = next[i];
    }
    s_waitcnt<0, 0>();   // no DMA may outlive the workgroup's LDS
}

__device__ __forceinline__ void conv_join() {
    // No MFMA or LDS read of a finished step may sink below the barrier that frees its stage.
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// LDS by 32-bit address.
__device__ __forceinline__ bf16x8_t lds_frag(uint32_t addr) {
    return *reinterpret_cast<__attribute__((address_space(3))) const bf16x8_t*>(addr);
}
// One k-step: a0 and b hold the first K=32 half's fragments (read during the step before); the
// second half's (64 bytes further, in swizzled slots: address ^ 64) are read under the first
// half's MFMAs and the next step's first half under the second half's.
template <int MT, int NT>
__device__ __forceinline__ void conv_step(f32x4_t (&acc)[MT][NT], bf16x8_t (&a0)[MT], bf16x8_t (&b)[NT],
                                          uint32_t a_row, uint32_t b_row, uint32_t a_next, uint32_t b_next) {
    bf16x8_t a1[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) a1[i] = lds_frag((a_row ^ 64) + i * kPRow);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a0[i], acc[i][j], 0, 0, 0);
        b[j] = lds_frag((b_row ^ 64) + j * 16 * kRowBytes);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a1[i], acc[i][j], 0, 0, 0);
        b[j] = lds_frag(b_next + j * 16 * kRowBytes);
        if (j < MT) a0[j] = lds_frag(a_next + j * kPRow);
    }
#pragma unroll
    for (int i = NT; i < MT; ++i) a0[i] = lds_frag(a_next + i * kPRow);
    __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x008, MT, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    constexpr int kBoth = cmin(MT, NT);
#pragma unroll
    for (int j = 0; j < kBoth; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x008, MT, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
#pragma unroll
    for (int j = kBoth; j < NT; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x008, MT, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
}

// Sums of the stored outputs for the GroupNorm that follows: for each run of four channels, the sum
// and the sum of squares in fp64 over a wave's pixels of it, at
// stats[(channel / 4) * stats_rows + row] with row = patch * waves + wave. Both are sums of exactly
// converted bf16 values (a square has 16 significant bits), so neither loses a bit that matters at
// any image size. The sixteen pixels of a patch row are sixteen neighbouring lanes, summed with
// rotations within them. Costs ~1.2 us per 256 x 128 tile; a pass over the output costs 14 us at
// 128 channels of 512 x 512 (54 at 1024 x 1024) and two launches.
__device__ __forceinline__ double row16_sum(double v) {
#define BH_ROR(N)                                                                                  \
    {                                                                                              \
        const uint64_t b = __builtin_bit_cast(uint64_t, v);                                        \
        const uint32_t lo = __builtin_amdgcn_mov_dpp(static_cast<int>(b), 0x120 + N, 0xf, 0xf, false);       \
        const uint32_t hi = __builtin_amdgcn_mov_dpp(static_cast<int>(b >> 32), 0x120 + N, 0xf, 0xf, false); \
        v += __builtin_bit_cast(double, static_cast<uint64_t>(hi) << 32 | lo);                     \
    }
    BH_ROR(8) BH_ROR(4) BH_ROR(2) BH_ROR(1)
#undef BH_ROR
    return v;
}

// A wave's MW x 16 pixels by 16 NW channels, from image row y0 and channel n0: bias, then the
// residual add (the sum rounded first where the reference stores it), one rounding. A lane holds 8
// consecutive channels of one pixel of each row per 32 channels. The residual's loads are issued
// before the stores: a load behind a store waits for that store's acknowledgement. Rows are addressed by
// a scalar base and one 32-bit lane offset.
template <int MW, int MODE, int NW, bool STATS>
__device__ __forceinline__ void conv_epilogue(const f32x4_t (&acc)[MW][NW], const ConvArgs& a, const Epi& e,
                                              int y0, int x0, int n0, int lane, const bf16_t* bl,
                                              int64_t stats_row) {
    constexpr int kP = NW / 2;
    const int lr = lane & 15, hi = lane >> 4;
    const bool xok = x0 + lr < a.W;
    const uint32_t lo = lr * static_cast<uint32_t>(e.ld_out) + 8 * hi;
    const int64_t base = (static_cast<int64_t>(y0) * a.W + x0) * e.ld_out + n0;
    const int64_t row = static_cast<int64_t>(a.W) * e.ld_out;
    uint4 res[kP][MW];
    auto load = [&](int p) {
        if (MODE != EPI_RESIDUAL) return;
#pragma unroll
        for (int i = 0; i < MW; ++i)
            if (y0 + i < a.H && xok && n0 + 32 * p + 8 * hi < a.c_out)
                res[p][i] = *reinterpret_cast<const uint4*>(e.residual + base + i * row + 32 * p + lo);
    };
#pragma unroll
    for (int p = 0; p < cmin(kP, 2); ++p) load(p);
#pragma unroll
    for (int p = 0; p < kP; ++p) {
        if (p > 0 && p + 1 < kP) load(p + 1);
        if (n0 + 32 * p + 8 * hi >= a.c_out) break;
        float bias[8];
        bias_or_neg_zero(e, e.bias ? ld_raw<8>(bl + 32 * p + 8 * hi) : uint4{}, bias);
        double sum[2] = {0.0, 0.0}, sq[2] = {0.0, 0.0};
#pragma unroll
        for (int i = 0; i < MW; ++i) {
            if (y0 + i >= a.H || !xok) continue;
            float v[8], t[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = __fadd_rn(acc[i][2 * p + (q >> 2)][q & 3], bias[q]);
            if (MODE == EPI_RESIDUAL) {
                unpack8(res[p][i], t);
#pragma unroll
                for (int q = 0; q < 8; ++q) v[q] = __fadd_rn(t[q], e.round_mid ? round_bf16(v[q]) : v[q]);
            }
            const uint4 packed = pack8(v);
            *reinterpret_cast<uint4*>(a.out + base + i * row + 32 * p + lo) = packed;
            if (STATS && a.stats) {
                unpack8(packed, v);
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const double x = static_cast<double>(v[q]);
                    sum[q >> 2] += x;
                    sq[q >> 2] = __builtin_fma(x, x, sq[q >> 2]);
                }
            }
        }
        if (STATS && a.stats) {   // a lane's sixteen neighbours share its channels, so none has left the loop
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const double s1 = row16_sum(sum[h]), s2 = row16_sum(sq[h]);
                double* to = a.stats + ((static_cast<int64_t>(n0 + 32 * p + 8 * hi) / 4 + h) * a.stats_rows + stats_row) * 2;
                if (lr == 0) {
                    to[0] = s1;
                    to[1] = s2;
                }
            }
        }
    }
}

template <int MT, int MODE, int NT, bool STATS, bool NORM>
__device__ __forceinline__ void conv_consume(char* smem, const ConvArgs& a, const Epi& e, int my_tiles,
                                             int wave, int lane) {
    using G = Halo<MT, NT, NORM>;
    if (NORM) wait_and_join<63>();   // the producers' barrier over the first chunk's norm
    const int lr = lane & 15, hi = lane >> 4, sw = (lr >> 1) & 7;
    // this lane's offset in a 16-row weight block and in a patch row for tap column kx
    const uint32_t lb = lr * kRowBytes + ((hi ^ sw) * 16);
    uint32_t la[3];
#pragma unroll
    for (int kx = 0; kx < 3; ++kx) la[kx] = (lr + kx) * kRowBytes + ((hi ^ (((lr + kx) >> 1) & 7)) * 16);
    const int chunks = a.c_in >> 6;
    constexpr int MW = G::MW, NW = G::NW;
    const int wm = wave / G::WN, wn = wave % G::WN;
    const uint32_t patch = lds_addr(smem) + wm * MW * kPRow;
    const uint32_t ring = lds_addr(smem) + G::kBOff + wn * NW * 16 * kRowBytes;
    int st = 0, buf = 0;
    for (int it = 0; it < my_tiles; ++it) {
        f32x4_t acc[MW][NW];
#pragma unroll
        for (int i = 0; i < MW; ++i)
#pragma unroll
            for (int j = 0; j < NW; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        bf16x8_t a0[MW], b[NW];
        for (int cb = 0; cb < chunks; ++cb) {
            const uint32_t pa = patch + buf * G::kABytes, pn = patch + (buf ^ 1) * G::kABytes;
#pragma unroll
            for (int tap = 0; tap < 9; ++tap) {
                conv_join();
                // formed anew each step: kept across steps, the 36 addresses of a chunk would spill
                asm volatile("" : "+v"(la[0]), "+v"(la[1]), "+v"(la[2]));
                const uint32_t ar = pa + la[tap % 3] + (tap / 3) * kPRow, br = ring + st * G::kBBytes + lb;
                if (tap == 0 && cb == 0) {   // a tile's first fragments: nothing read them ahead
#pragma unroll
                    for (int i = 0; i < MW; ++i) a0[i] = lds_frag(ar + i * kPRow);
#pragma unroll
                    for (int j = 0; j < NW; ++j) b[j] = lds_frag(br + j * 16 * kRowBytes);
                }
                st = st == G::S - 1 ? 0 : st + 1;
                const int nt = (tap + 1) % 9;
                conv_step<MW, NW>(acc, a0, b, ar, br, (tap == 8 ? pn : pa) + la[nt % 3] + (nt / 3) * kPRow,
                                  ring + st * G::kBBytes + lb);
            }
            buf ^= 1;
        }
        int y0, x0, n0;
        conv_tile<MT, NT>(a, blockIdx.x + it * gridDim.x, y0, x0, n0);
        const char* slot = smem + G::kBiasOff + (it % G::kBiasSlots) * kBiasSlotBytes;
        constexpr int kWM = 4 / G::WN;
        const int64_t patch_index = static_cast<int64_t>(y0 / G::PY) * a.tiles_x + x0 / 16;
        conv_epilogue<MW, MODE, NW, STATS>(acc, a, e, y0 + MW * wm, x0, n0 + 16 * NW * wn, lane,
                                           reinterpret_cast<const bf16_t*>(slot) + 16 * NW * wn,
                                           patch_index * kWM + wm);
    }
}

template <int MT, int MODE, int NT, bool STATS, bool NORM>
__global__ void __launch_bounds__(kWgThreads, 1) k_conv3x3(ConvArgs a, Epi e) {
    __shared__ __attribute__((aligned(1024))) char smem[Halo<MT, NT, NORM>::kSmemBytes];
    const int my_tiles = (a.tiles - static_cast<int>(blockIdx.x) + static_cast<int>(gridDim.x) - 1) /
                         static_cast<int>(gridDim.x);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (wave >= kConsumers) conv_produce<MT, NT, NORM>(smem, a, e.bias, my_tiles, wave - kConsumers, lane);
    else conv_consume<MT, MODE, NT, STATS, NORM>(smem, a, e, my_tiles, wave, lane);
}

int device_cus() {
    static std::atomic<int> cus[64] = {};
    int dev = 0;
    hip_check(hipGetDevice(&dev), "hipGetDevice");
    require(dev >= 0 && dev < 64, "conv3x3: device index out of range");
    int n = cus[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        hip_check(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev),
                  "hipDeviceGetAttribute");
        require(n > 0, "conv3x3: device reports no compute units");
        cus[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

int patches(const ConvGeom& cv, int mt) { return ((cv.H + 4 * mt - 1) / (4 * mt)) * ((cv.W + 15) / 16); }

struct ConvExtra {
    double* stats;
    const NormChannel* norm;
};

template <int MT, int NT>
void launch_conv(const ConvGeom& cv, const bf16_t* w, bf16_t* out, int64_t c_out, const Epi& e,
                 const ConvExtra& x, hipStream_t s) {
    ConvArgs a{cv.in, cv.zero, w, out, cv.H, cv.W, cv.in_w, cv.c_in, cv.up, static_cast<int>(c_out), 0, 0, 0,
               x.stats, static_cast<int64_t>(patches(cv, MT)) * (4 / Halo<MT, NT>::WN), x.norm};
    a.tiles_x = (cv.W + 15) / 16;
    a.tiles_n = static_cast<int>((c_out + 16 * NT - 1) / (16 * NT));
    a.tiles = patches(cv, MT) * a.tiles_n;
    int grid = min(a.tiles, device_cus() & ~7);
    if (grid < 8) grid = min(a.tiles, device_cus());
    // The combinations the decoder and the single op use; null sums are skipped. Above 32 channels a tile is 128
    // wide whatever the width: 136 or 144 channels multiply 256 columns, where tiles of 144 multiplied 144, and the op
    // is still the shorter one (256 channels to 144 at 256 x 256: 92 -> 75 us; 512 to 144 at 192 x 192: 108 -> 97,
    // the least gain of 77 such sizes; 512 to 288 at 256 x 256: 237 -> 185).
    if constexpr (NT == 8) {
        if (x.norm) {
            if (e.residual) k_conv3x3<MT, EPI_RESIDUAL, NT, true, true><<<grid, kWgThreads, 0, s>>>(a, e);
            else k_conv3x3<MT, EPI_STORE, NT, true, true><<<grid, kWgThreads, 0, s>>>(a, e);
            return;
        }
        if (e.residual) k_conv3x3<MT, EPI_RESIDUAL, NT, true, false><<<grid, kWgThreads, 0, s>>>(a, e);
        else if (x.stats) k_conv3x3<MT, EPI_STORE, NT, true, false><<<grid, kWgThreads, 0, s>>>(a, e);
        else k_conv3x3<MT, EPI_STORE, NT, false, false><<<grid, kWgThreads, 0, s>>>(a, e);
    } else {
        k_conv3x3<MT, EPI_STORE, NT, false, false><<<grid, kWgThreads, 0, s>>>(a, e);
    }
}

// The patch height: the least estimated time, rounds of tiles over the CUs times a step's cycles.
// A step is bound by its MFMAs (256 cycles per patch-row block) or, on the short tiles, by the
// weights that stream per step whatever the height; the figures are a step's cycles by height.
int conv_rows(const ConvGeom& cv, int64_t c_out) {
    const int64_t cus = device_cus(), tiles_n = (c_out + 127) / 128;
    const int step[5] = {0, 400, 620, 0, 1180};
    int best = 4;
    int64_t best_cost = -1;
    for (int mt : {4, 2, 1}) {
        const int64_t tiles = patches(cv, mt) * tiles_n;
        const int64_t cost = (tiles + cus - 1) / cus * step[mt];
        if (best_cost < 0 || cost < best_cost) {
            best = mt;
            best_cost = cost;
        }
    }
    return best;
}

bool aligned(const void* p, int bytes) { return (reinterpret_cast<uintptr_t>(p) % bytes) == 0; }

}  // namespace

int64_t conv3x3_stats_rows(const ConvGeom& cv, int64_t c_out) {
    if (c_out <= 32) return 0;
    switch (conv_rows(cv, c_out)) {
        case 1: return static_cast<int64_t>(patches(cv, 1)) * (4 / Halo<1, 8>::WN);
        case 2: return static_cast<int64_t>(patches(cv, 2)) * (4 / Halo<2, 8>::WN);
        default: return static_cast<int64_t>(patches(cv, 4)) * (4 / Halo<4, 8>::WN);
    }
}

void launch_conv3x3_bf16(const ConvGeom& cv, const bf16_t* wr, const bf16_t* bias, bf16_t* out,
                         int64_t c_out, const GemmEpilogue& ep, hipStream_t s, double* stats,
                         const NormChannel* norm) {
    const int64_t m = static_cast<int64_t>(cv.H) * cv.W, k = 9 * static_cast<int64_t>(cv.c_in);
    if (m == 0 || c_out == 0) return;
    require(cv.in && cv.zero && wr && out, "conv3x3: null operand");
    require(cv.c_in % 64 == 0 && cv.c_in > 0, "conv3x3 (mfma): c_in must be a positive multiple of 64");
    require(c_out % 8 == 0, "conv3x3 (mfma): c_out must be a multiple of 8");
    require(cv.up ? (cv.in_h * 2 == cv.H && cv.in_w * 2 == cv.W) : (cv.in_h == cv.H && cv.in_w == cv.W),
            "conv3x3: input and output sizes disagree");
    require(!ep.vt && !ep.row_add && !ep.gate, "conv3x3: epilogue must be a plain store or a residual add");
    require(aligned(cv.in, 16) && aligned(cv.zero, 16) && aligned(wr, 16) && aligned(out, 16) &&
                (!bias || aligned(bias, 16)) && (!ep.residual || aligned(ep.residual, 16)),
            "conv3x3: operands must be 16-byte aligned");
    require(static_cast<int64_t>(cv.in_h) * cv.in_w * cv.c_in < (int64_t{1} << 31),
            "conv3x3: input too large for 32-bit pixel offsets");
    Epi e{bias, ep.act, ep.round_mid, nullptr, 1, ep.residual, nullptr, 1,
          ep.ld_out > 0 ? ep.ld_out : c_out, 0, nullptr, 0, 0, 0, 0, 0, 72};
    require(ep.act == 0, "conv3x3: no activation epilogue (the decoder's SiLU follows a GroupNorm)");
    ProfileScope ps(K_GEMM, s, 2.0 * static_cast<double>(m) * c_out * k);
    require(!stats || conv3x3_stats_rows(cv, c_out) > 0, "conv3x3: this shape sums no statistics");
    require((!ep.residual && !norm) || c_out > 32, "conv3x3: the narrow tile is a plain store");
    require(!norm || (!cv.up && aligned(norm, 16)), "conv3x3: a normalised input is not upsampled");
    const ConvExtra x{stats, norm};
    if (c_out <= 32) {   // the decoder's conv_out: one 32-wide tile column
        launch_conv<4, 2>(cv, wr, out, c_out, e, x, s);
    } else {
        switch (conv_rows(cv, c_out)) {
            case 1: launch_conv<1, 8>(cv, wr, out, c_out, e, x, s); break;
            case 2: launch_conv<2, 8>(cv, wr, out, c_out, e, x, s); break;
            default: launch_conv<4, 8>(cv, wr, out, c_out, e, x, s); break;
        }
    }
    launch_check("conv3x3 (mfma)");
}

}  // namespace bh
