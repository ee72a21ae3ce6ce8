// Which 64-key tiles of a mask tensor the pipelined attention kernel has to visit (gfx950): one pass over a mask that the heads
// share, and over V, ahead of the attention launch.
//
// FlagAttention src/flag_attn/sage_attention/attn_qk_int8_per_block.py:33-36 skips the 128 x 64 tiles of a bool mask without a
// visible key; under an additive mask it computes every tile.  There a tile can be left out where it changes nothing: its largest
// entry lies so far below the largest entry of every row that every P of the tile is exactly 0, whatever the scores (bounded by
// the block scales, which the attention kernel looks at: `visits` in attn_fast_kernel.h).  Padding and causal masks in additive
// form, the ones model code builds, leave out their hidden half that way; a row that sees no key at all makes its q-block visit
// every tile.  A tile of V with an Inf or NaN is visited by all (0 times those is NaN).
// The scan also tells the tiles whose entries are all 0 (bool: all visible), whose steps need no mask arithmetic: +0 stands for them,
// -0 for any other tile with 0 as its largest entry.
//
// Bound by the bytes of the mask and of V.  A workgroup takes a strip of 16 mask rows, a thread 16 bytes of each of them at a time
// (16 loads on their way), so that the scan of one [M, N] mask fills the chip; or one 64-key tile of V.
// 10 to 25 us at 4 TB/s (4.7 is a copy's); taking note of the zeros costs it nothing that shows (bool B4 N1536 10.1 -> 10.3 us, B1
// N4096 12.4 -> 11.6, at 125 registers and four waves per SIMD; bf16 12.4 -> 12.5 and 15.0 -> 15.4).
// Attention call without the scan -> with it, launch and all: B4 H16 M1536 N1536 D128, [B, 1, M, N] bf16 mask (19 MB, V 25 MB) with
// causal and padding in one 96 -> 66 us; B1 H32/8 M2560 N2560 D128, causal, bool 135 -> 76; B2 H24 M3840 N3840 D64, causal and
// padding, fp32 entries (118 MB) 270 -> 134 us.
#include <type_traits>

#include "attn_common.h"

namespace sage {
namespace {

using attn::AttnArgs;
using attn::BN;
using attn::kScanRows;

constexpr int kScanThreads = 256;

struct ScanArgs {
    const unsigned char* mask;
    const unsigned char* v;
    float* top;
    float* low;
    unsigned* odd;
    int64_t ms_b, ms_m;        // bytes
    int64_t vs_b, vs_h, vs_n;  // bytes
    int32_t M, N, nk, Hkv;
    int32_t strips, mask_wgs;  // strips of a mask batch; workgroups that scan the mask (the others: V)
    int32_t v_tiles;           // batch * Hkv * nk
};

// the largest of the first `live` entries of a 16-byte chunk; NaN counts as +inf (bool: 0 where a key is visible, else -inf)
template <typename MT>
__device__ __forceinline__ float chunk_max(uint4 w, int live) {
    constexpr int E = 16 / sizeof(MT);
    const unsigned word[4] = {w.x, w.y, w.z, w.w};
    float m = -INFINITY;
    if constexpr (sizeof(MT) == 1) {
        unsigned any = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int bytes = live - 4 * i;
            any |= bytes >= 4 ? word[i] : bytes <= 0 ? 0u : word[i] & ((1u << (8 * bytes)) - 1);
        }
        m = any ? 0.0f : -INFINITY;
    } else {
#pragma unroll
        for (int i = 0; i < E; i++) {
            float x;
            if constexpr (sizeof(MT) == 4) x = __builtin_bit_cast(float, word[i]);
            else {
                const unsigned short bits = (unsigned short)(i & 1 ? word[i >> 1] >> 16 : word[i >> 1]);
                x = (float)__builtin_bit_cast(MT, bits);
            }
            x = x == x ? x : INFINITY;
            m = i < live ? fmaxf(m, x) : m;
        }
    }
    return m;
}

// do all entries of a 16-byte chunk leave their scores as they are?  (additive: zeros of either sign; bool: non-zero bytes)
template <typename MT>
__device__ __forceinline__ bool chunk_plain(uint4 w) {
    const unsigned word[4] = {w.x, w.y, w.z, w.w};
    unsigned changes = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if constexpr (sizeof(MT) == 1) changes |= (word[i] - 0x01010101u) & ~word[i] & 0x80808080u;  // a zero byte sets bits from its own up
        else changes |= word[i] & (sizeof(MT) == 4 ? 0x7fffffffu : 0x7fff7fffu);
    }
    return changes == 0;
}

template <typename MT>
__device__ __forceinline__ void scan_strip(const ScanArgs& a, int wg) {
    constexpr int E = 16 / sizeof(MT), LPT = BN / E;  // entries per chunk; chunks (lanes) per tile
    __shared__ float row_top[kScanThreads / 64][kScanRows];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int mb = wg / a.strips, strip = wg % a.strips;
    const unsigned char* base = a.mask + mb * a.ms_b;
    float row[kScanRows];
#pragma unroll
    for (int r = 0; r < kScanRows; r++) row[r] = -INFINITY;
    const int chunks = a.nk * LPT;
    for (int c0 = 0; c0 < chunks; c0 += kScanThreads) {
        const int c = c0 + tid, live = a.N - c * E;  // entries of the chunk that are keys
        float t = -INFINITY;
        bool plain = live >= E;
        if (live > 0) {
            uint4 w[kScanRows];
#pragma unroll
            for (int r = 0; r < kScanRows; r++)  // (rows past the last one: that one again)
                w[r] = *reinterpret_cast<const uint4*>(base + (int64_t)min(strip * kScanRows + r, a.M - 1) * a.ms_m + (int64_t)16 * c);
#pragma unroll
            for (int r = 0; r < kScanRows; r++) {
                const float m = chunk_max<MT>(w[r], live);
                row[r] = fmaxf(row[r], m);
                t = fmaxf(t, m);
                plain &= chunk_plain<MT>(w[r]);
            }
        }
#pragma unroll
        for (int x = 1; x < LPT; x <<= 1) {
            t = fmaxf(t, __shfl_xor(t, x));
            plain &= __shfl_xor((int)plain, x) != 0;
        }
        if (t == 0.0f) t = plain ? 0.0f : -0.0f;
        const int tile = c / LPT;
        if (c < chunks && c % LPT == 0) {
            // (additive: the last tile of a kv_len that is not a multiple of 64 also holds keys that score -1e6)
            if (sizeof(MT) > 1 && tile == a.nk - 1 && a.N % BN) t = fmaxf(t, attn::kMasked);
            a.top[(int64_t)wg * a.nk + tile] = t;
        }
    }
#pragma unroll
    for (int r = 0; r < kScanRows; r++) {
#pragma unroll
        for (int x = 1; x < 64; x <<= 1) row[r] = fmaxf(row[r], __shfl_xor(row[r], x));
        if (lane == 0) row_top[wave][r] = row[r];
    }
    __syncthreads();
    if (tid == 0) {
        float low = INFINITY;
        for (int r = 0; r < kScanRows; r++) {
            float m = row_top[0][r];
            for (int w = 1; w < kScanThreads / 64; w++) m = fmaxf(m, row_top[w][r]);
            low = fminf(low, m);
        }
        a.low[wg] = low;
    }
}

// A wave takes a 64-key tile of V, every load of it on its way before the first is looked at.
template <int D, typename VT>
__device__ __forceinline__ void scan_v(const ScanArgs& a, int wg) {
    constexpr int CPR = 2 * D / 16, LOADS = BN * CPR / 64;  // 16-byte chunks per row; of a tile per lane
    constexpr unsigned exponent = std::is_same_v<VT, __bf16> ? 0x7f807f80u : 0x7c007c00u;  // all ones: Inf or NaN
    const int i = wg * (kScanThreads / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= a.v_tiles) return;
    const int t = i % a.nk, bh = i / a.nk, hk = bh % a.Hkv, b = bh / a.Hkv;
    const unsigned char* base = a.v + b * a.vs_b + hk * a.vs_h + 16 * (lane % CPR);
    uint4 w[LOADS];
#pragma unroll
    for (int x = 0; x < LOADS; x++)
        w[x] = *reinterpret_cast<const uint4*>(base + (int64_t)min(BN * t + x * (64 / CPR) + lane / CPR, a.N - 1) * a.vs_n);
    bool odd = false;
#pragma unroll
    for (int x = 0; x < LOADS; x++) {
        const unsigned word[4] = {w[x].x, w[x].y, w[x].z, w[x].w};
#pragma unroll
        for (int y = 0; y < 4; y++) {
            const unsigned e = word[y] & exponent;
            odd |= (e & 0xffffu) == (exponent & 0xffffu) || (e >> 16) == (exponent >> 16);
        }
    }
    const bool any = __builtin_amdgcn_ballot_w64(odd) != 0;
    if (lane == 0) a.odd[i] = any ? 1u : 0u;
}

template <int D, typename VT, typename MT>
__global__ __launch_bounds__(kScanThreads) void mask_scan_kernel(ScanArgs a) {
    const int wg = blockIdx.x;
    if (wg < a.mask_wgs) scan_strip<MT>(a, wg);
    else scan_v<D, VT>(a, wg - a.mask_wgs);
}

int64_t mask_batches(const AttnArgs& a, int64_t batch) { return a.ms_b ? batch : 1; }
int64_t scan_strips(const AttnArgs& a) { return a.ms_m ? (a.M + kScanRows - 1) / kScanRows : 1; }

template <int D, typename VT>
int launch_scan(const AttnArgs& a, const ScanArgs& s, int64_t wgs, hipStream_t stream) {
    dim3 grid((unsigned)wgs), block(kScanThreads);
    if (!a.mask_additive) hipLaunchKernelGGL((mask_scan_kernel<D, VT, uint8_t>), grid, block, 0, stream, s);
    else if (a.mask_dt == SAGE_F32) hipLaunchKernelGGL((mask_scan_kernel<D, VT, float>), grid, block, 0, stream, s);
    else if (a.mask_dt == SAGE_BF16) hipLaunchKernelGGL((mask_scan_kernel<D, VT, __bf16>), grid, block, 0, stream, s);
    else hipLaunchKernelGGL((mask_scan_kernel<D, VT, _Float16>), grid, block, 0, stream, s);
    return check_launch("mask_scan_kernel");
}

}  // namespace

namespace attn {

// us: of a step of the attention kernel under a mask, and of the scan
static float step_us(int head_dim) { return head_dim == 128 ? 1.5f : 0.85f; }
static float scan_us(const AttnArgs& a, int64_t batch, int head_dim) {
    const float esz = a.mask_additive ? (float)dtype_bytes(a.mask_dt) : 1.0f;
    return 5.0f + ((float)mask_batches(a, batch) * (a.ms_m ? (float)a.M : 1.0f) * (float)a.N * esz +
                   (float)(batch * a.Hkv) * (float)a.N * (float)(2 * head_dim)) * (1e-6f / 4.5f);
}

// Few q-blocks: the tiles left to visit are split over several workgroups each, like the keys of a call without a mask, where the
// steps that saves are worth the scan, the second launch and the partial results (B2 H2 M3072 N3072 D128 causal and padded, bool:
// 96 us whole, 62 in five runs; but B1 H32 M732 45, 55 in two, B2 H8 M832 48, 54 in three).
int mask_splits(const AttnArgs& a, int64_t batch, int head_dim) {
    const int64_t q_blocks = batch * a.Hq * ((a.M + kFastRows - 1) / kFastRows);
    const float whole = 7.0f + step_us(head_dim) * (float)a.nk, rows = (float)(batch * a.Hq) * (float)a.M;
    float best = 0.9f * whole;
    int runs = 1;
    if (a.ms_h != 0 || a.Hq < 2 || a.causal) return 1;  // (not scanned)
    for (int s = 2; s <= 16 && s <= a.nk / 4 && s * q_blocks <= 256; s++) {
        const float cost = scan_us(a, batch, head_dim) + 7.0f + step_us(head_dim) * (float)((a.nk + s - 1) / s) + 4.0f +
                           (float)s * rows * (float)head_dim * (8e-6f / 4.0f);
        if (cost < best) { best = cost; runs = s; }
    }
    return runs;
}

// Worth its launch where the heads share the mask (one read of it serves all of them; a mask per head is a position bias as a
// rule, and read once either way) and enough steps can go.  What it costs (a launch, the bytes of the mask and of V, 1 to 2 us in
// every workgroup) a mask that hides no tile loses; what it gains lies in the entries, which the rule does not see.  The lines lie
// where the masks that model code builds gain, a causal one or the padding of sequences between half as long and as long as the
// keys.  Attention call with the scan over the one without, every shape run both ways (means of 2500 shapes, in brackets the
// tenths of them at either end: 2 to 32 heads, 1 to 8 sequences, 512 to 8192 keys; "entries" change a score in every tile,
// "zeros" in none):
//   more q-blocks than compute units   entries             zeros               causal              causal and padding
//     rows of entries, 8 to 11 tiles   1.29 (1.24 - 1.34)  1.22 (1.17 - 1.27)  0.92 (0.81 - 1.05)  0.91 (0.80 - 1.03)  (not scanned)
//     12 to 20                         1.22 (1.17 - 1.28)  1.12 (1.06 - 1.18)  0.81 (0.69 - 0.93)  0.79 (0.68 - 0.92)
//     21 to 35                         1.16 (1.11 - 1.21)  1.04 (0.98 - 1.09)  0.68 (0.59 - 0.76)  0.66 (0.54 - 0.74)
//     36 to 64                         1.13 (1.08 - 1.21)  0.99 (0.92 - 1.06)  0.59 (0.52 - 0.67)  0.55 (0.45 - 0.65)
//     65 to 128                        1.17 (1.08 - 1.31)  1.17 (1.08 - 1.32)  0.67 (0.59 - 0.81)  0.61 (0.48 - 0.78)
//   more q-blocks than compute units   entries             zeros               padding
//     one row of entries, 8 to 27      1.19 (1.13 - 1.27)  1.09 (1.00 - 1.20)  0.99 (0.84 - 1.16)  (not scanned)
//     28 to 64                         1.11 (1.08 - 1.14)  0.96 (0.89 - 1.02)  0.82 (0.67 - 0.94)
//     65 to 128                        1.08 (1.06 - 1.10)  1.08 (1.06 - 1.10)  0.91 (0.69 - 1.05)
//     causal mask folded into a bool one, whose walk ends at the limit anyway, 8 to 35 tiles 1.13 (0.98 - 1.33) with padding (not
//     scanned), 0.80 (0.59 - 1.13) from 36
//   fewer, unsplit, 48 us of steps and more: the longest q-block alone counts, which a causal mask does not shorten and padding
//   seldom where there are several sequences, the longest of which is nearly full
//                                      entries             causal              causal and padding
//     one sequence                     1.18 (1.13 - 1.25)  1.09 (0.95 - 1.19)  0.87 (0.71 - 1.06)
//     two to eight                     1.30 (1.18 - 1.43)  1.19 (1.04 - 1.36)  1.07 (0.86 - 1.27)  (not scanned)
// V is read once more, so the queries per K/V head have to be many as well.
int64_t mask_scan_bytes(const AttnArgs& a, int64_t batch, int head_dim) {
    const int64_t q_blocks = batch * a.Hq * ((a.M + kFastRows - 1) / kFastRows);
    if (a.causal) return 0;  // (the largest entry of a row may lie where the causal mask adds -1e6 to it)
    if (a.ms_h != 0 || a.Hq < 2) return 0;
    if (mask_splits(a, batch, head_dim) == 1) {
        if (q_blocks > 256) {
            if (a.nk < (a.mask_causal ? 36 : a.ms_m == 0 ? 28 : 12)) return 0;
        } else if (a.ms_m == 0 || batch > 1 || step_us(head_dim) * (float)a.nk < 48.0f) {
            return 0;
        }
        if ((int64_t)a.groups * a.M < 512) return 0;
    }
    const int64_t mask_wgs = mask_batches(a, batch) * scan_strips(a), v_tiles = batch * a.Hkv * a.nk;
    if (mask_wgs + v_tiles > 0x7fffffffLL) return 0;
    const int64_t bytes = 4 * (mask_wgs * (a.nk + 1) + v_tiles);
    return (bytes + 15) / 16 * 16;
}

int launch_mask_scan(AttnArgs& a, int64_t batch, int head_dim, int v_dtype, void* workspace, hipStream_t stream) {
    const int64_t strips = scan_strips(a), mask_wgs = mask_batches(a, batch) * strips, v_tiles = batch * a.Hkv * a.nk;
    ScanArgs s{};
    s.mask = static_cast<const unsigned char*>(a.mask); s.v = static_cast<const unsigned char*>(a.v);
    s.top = static_cast<float*>(workspace); s.low = s.top + mask_wgs * a.nk; s.odd = reinterpret_cast<unsigned*>(s.low + mask_wgs);
    const int64_t esz = a.mask_additive ? dtype_bytes(a.mask_dt) : 1;
    s.ms_b = a.ms_b * esz; s.ms_m = a.ms_m * esz;
    s.vs_b = 2 * a.vs_b; s.vs_h = 2 * a.vs_h; s.vs_n = 2 * a.vs_n;
    s.M = a.M; s.N = a.N; s.nk = a.nk; s.Hkv = a.Hkv; s.strips = (int)strips; s.mask_wgs = (int)mask_wgs; s.v_tiles = (int)v_tiles;
    const int64_t v_wgs = (v_tiles + kScanThreads / 64 - 1) / (kScanThreads / 64);
    a.scan_top = s.top; a.scan_low = s.low; a.scan_v = s.odd; a.scan_strips = s.strips;
    a.longest_first = a.ms_m != 0;
    if (head_dim == 128)
        return v_dtype == SAGE_BF16 ? launch_scan<128, __bf16>(a, s, mask_wgs + v_wgs, stream) : launch_scan<128, _Float16>(a, s, mask_wgs + v_wgs, stream);
    return v_dtype == SAGE_BF16 ? launch_scan<64, __bf16>(a, s, mask_wgs + v_wgs, stream) : launch_scan<64, _Float16>(a, s, mask_wgs + v_wgs, stream);
}

}  // namespace attn
}  // namespace sage
