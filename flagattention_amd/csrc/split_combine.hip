// How launches of the pipelined attention kernel for gfx950 are laid out over the 256 compute units, and the kernels that
// combine partial results.  Key split: a launch with few (batch, head, q-block) items leaves most CUs idle; the keys of
// every item are then cut into `nsplit` runs of whole 64-key steps, one workgroup each, which write a normalized
// fp32 partial output o_s and its base-2 log-sum-exp lse_s.  Cut launch: all steps of the launch form one line
// (CutLine), of which every workgroup takes an equal share.  Either way the combine kernel forms
//     lse = log2 sum_s 2^lse_s,      out = sum_s 2^(lse_s - lse) o_s
// (FlagAttention src/flag_attn/flash.py:73-75, :106-141 is the dense forward's use of the same idea,
// split_kv.py:250-278 its choice of the number of runs, :155-214 its combine kernel).
#include "attn_common.h"

namespace sage {
namespace attn {
namespace {

constexpr int kComputeUnits = 256;
constexpr int kMaxSplits = 64;
constexpr int kMinStepsPerSplit = 4;   // 256 keys: below that the prologue and epilogue of a workgroup dominate
constexpr int kFewItems = 16;          // up to here every piece of the work has a CU to itself: the longest run alone counts
constexpr int kMinStepsPerShare = 8;   // of a cut launch: a share may hold two pieces

struct CombineArgs {
    const float* part_o;    // [nsplit, rows, D]
    const float* part_lse;  // [nsplit, rows], base 2
    void* out;
    float* lse;             // [rows] or null
    int64_t os_b, os_h, os_n;
    int64_t rows;           // batch * heads_q * qo_len
    int32_t Hq, M, nsplit, out_dt;
    float lse_mul, lse_shift_mul;
    const float* lse_shift;
};

constexpr int kCombineThreads = 256;

// Maximum of log-sum-exps.  NaN stays: it stands for NaN scores (a NaN or an infinity in Q or K), which make the whole row
// NaN, where fmaxf would leave the -inf of a row that saw no key, or the other runs alone.
__device__ __forceinline__ float max_or_nan(float m, float x) { return x > m || x != x ? x : m; }

__device__ __forceinline__ void store4(void* out, int out_dt, int64_t o, v4f r) {
    if (out_dt == SAGE_BF16) {
        typedef __bf16 b4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<b4*>(static_cast<__bf16*>(out) + o) = b4{(__bf16)r[0], (__bf16)r[1], (__bf16)r[2], (__bf16)r[3]};
    } else if (out_dt == SAGE_F16) {
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<h4*>(static_cast<_Float16*>(out) + o) = h4{(_Float16)r[0], (_Float16)r[1], (_Float16)r[2], (_Float16)r[3]};
    } else {
        *reinterpret_cast<v4f*>(static_cast<float*>(out) + o) = r;
    }
}

// TPR threads per row, four channels each; SG groups of them share the runs of a row (group g takes runs g, g + SG, ...)
// and meet through LDS.  SG = 1 where the rows alone fill the chip; with few rows (decoding) the runs of a row are read
// side by side instead of one after the other.
template <int D, int SG>
__global__ __launch_bounds__(kCombineThreads) void split_combine_kernel(CombineArgs a) {
    constexpr int TPR = D / 4;
    constexpr int ROWS = kCombineThreads / (TPR * SG);  // rows per workgroup
    __shared__ float sm_m[SG > 1 ? kCombineThreads : 1], sm_den[SG > 1 ? kCombineThreads : 1];
    __shared__ v4f sm_acc[SG > 1 ? kCombineThreads : 1];
    const int c = threadIdx.x % TPR, sg = (threadIdx.x / TPR) % SG;
    const int64_t row = (int64_t)blockIdx.x * ROWS + threadIdx.x / (TPR * SG);
    const bool ok = row < a.rows;
    const float* pl = a.part_lse + (ok ? row : 0);
    // The loads of kBatch runs are on their way together, the last run again past the end (one after the other a row of seven
    // runs took ten trips to memory).
    constexpr int kBatch = 8;
    const int last = a.nsplit - 1;
    float m = -INFINITY;
    for (int s0 = sg; s0 <= last; s0 += SG * kBatch) {
        float x[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) x[u] = pl[(int64_t)min(s0 + SG * u, last) * a.rows];
#pragma unroll
        for (int u = 0; u < kBatch; u++) m = max_or_nan(m, x[u]);
    }
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    float den = 0.0f;
    if (m != -INFINITY) {  // (a row that saw no key in any run: every partial is 0 and every lse_s -inf)
        const float* po = a.part_o + (ok ? row : 0) * D + 4 * c;
        for (int s0 = sg; s0 <= last; s0 += SG * kBatch) {
            v4f o[kBatch];
            float x[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                const int64_t s = min(s0 + SG * u, last);
                x[u] = pl[s * a.rows];
                o[u] = *reinterpret_cast<const v4f*>(po + s * a.rows * D);
            }
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                if (s0 + SG * u > last) break;
                const float w = __builtin_amdgcn_exp2f(x[u] - m);
                den += w;
#pragma unroll
                for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(w, o[u][i], acc[i]);
            }
        }
    }
    if constexpr (SG > 1) {
        sm_m[threadIdx.x] = m;
        sm_den[threadIdx.x] = den;
        sm_acc[threadIdx.x] = acc;
        __syncthreads();
        if (sg != 0) return;
        const int t0 = threadIdx.x;
#pragma unroll
        for (int g = 1; g < SG; g++) m = max_or_nan(m, sm_m[t0 + g * TPR]);
        acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        den = 0.0f;
        if (m != -INFINITY) {
#pragma unroll
            for (int g = 0; g < SG; g++) {
                const float w = __builtin_amdgcn_exp2f(sm_m[t0 + g * TPR] - m);
                const v4f o = sm_acc[t0 + g * TPR];
                den = __builtin_fmaf(w, sm_den[t0 + g * TPR], den);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(w, o[i], acc[i]);
            }
        }
    }
    if (!ok) return;
    const float inv = den > 0.0f ? 1.0f / den : 0.0f;
    v4f r;
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = acc[i] * inv;
    const int mi = (int)(row % a.M), h = (int)((row / a.M) % a.Hq);
    const int64_t b = row / ((int64_t)a.M * a.Hq);
    const int64_t o = b * a.os_b + (int64_t)h * a.os_h + (int64_t)mi * a.os_n + 4 * c;
    store4(a.out, a.out_dt, o, r);
    if (a.lse && c == 0) a.lse[row] = lse_out(__builtin_log2f(den) + m, a.lse_mul, a.lse_shift, a.lse_shift_mul, row);  // den = 0: log2(0) + (-inf) = -inf
}

// One wave tile (32 rows) of one item of a cut launch: the parts lie in the order of the accumulator registers, so a
// thread adds up four-channel pieces of one row; the sum is turned through LDS and written as whole rows.  Bound by the
// bytes of the parts: 67 MB at head_dim 128 when every share leaves two, 11.5 us (5.8 TB/s).  With fewer items to combine
// (64 of them from 288 parts, 38 MB) a quarter of the workgroups have work, and it takes 11 to 13 us (about 3 TB/s).
template <int D>
__global__ __launch_bounds__(kCombineThreads) void cut_combine_kernel(AttnArgs a) {
    constexpr int kPieces = 32 * D / 4 / kCombineThreads;  // per thread: 4 | 2
    constexpr int RS = D + 4;                              // floats per row in LDS
    __shared__ float rows[32 * RS];
    // blockIdx: one of the cuts between two shares x tile.  The first cut inside an item takes care of the item.
    const int tile = blockIdx.x % 8, cut = blockIdx.x / 8 + 1, pos = cut_begin(cut, a.cut_wgs, a.cut_total);
    const CutLine line(a.M, a.N, a.causal);
    const int bh = pos / line.head, iq = line.item(pos - bh * line.head);
    const int begin = bh * line.head + line.start(iq), m0 = kFastRows * iq + 32 * tile;
    const int first = cut_owner(begin, a.cut_wgs, a.cut_total);
    if (begin == pos || first + 1 != cut || m0 >= a.M) return;
    const int last = cut_owner(begin + line.len(iq) - 1, a.cut_wgs, a.cut_total);
    const int t = threadIdx.x, lane = t & 63, row = t & 31;
    auto slot = [&](int w) { return 2 * w + (w == first && begin != cut_begin(w, a.cut_wgs, a.cut_total)); };
    float m = -INFINITY;
    for (int w = first; w <= last; w++) m = max_or_nan(m, a.part_lse[(int64_t)slot(w) * kFastRows + 32 * tile + row]);
    v4f acc[kPieces];
#pragma unroll
    for (int e = 0; e < kPieces; e++) acc[e] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    float den = 0.0f;
    if (m != -INFINITY) {  // (a row that saw no key)
#pragma unroll 2
        for (int w = first; w <= last; w++) {
            const int64_t s = slot(w);
            const float f = __builtin_amdgcn_exp2f(a.part_lse[s * kFastRows + 32 * tile + row] - m);
            const v4f* po = reinterpret_cast<const v4f*>(a.part_o) + (s * 8 + tile) * (8 * D) + t;
            den += f;
#pragma unroll
            for (int e = 0; e < kPieces; e++) {
                const v4f o = po[kCombineThreads * e];
#pragma unroll
                for (int i = 0; i < 4; i++) acc[e][i] = __builtin_fmaf(f, o[i], acc[e][i]);
            }
        }
    }
    const float inv = den > 0.0f ? 1.0f / den : 0.0f;
    const int b = bh / a.Hq, h = bh % a.Hq;
    if (a.lse && t < 32 && m0 + row < a.M) {
        const int64_t r = (int64_t)bh * a.M + m0 + row;
        a.lse[r] = lse_out(__builtin_log2f(den) + m, a.lse_mul, a.lse_shift, a.lse_shift_mul, r);
    }
#pragma unroll
    for (int e = 0; e < kPieces; e++) {
        const int piece = t / 64 + 4 * e;  // 4 * (32-channel tile) + register group
        v4f r;
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = acc[e][i] * inv;
        *reinterpret_cast<v4f*>(rows + row * RS + 32 * (piece / 4) + 8 * (piece % 4) + 4 * (lane >> 5)) = r;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kPieces; e++) {
        const int p = t + kCombineThreads * e, r = p / (D / 4), c = 4 * (p % (D / 4));
        if (m0 + r >= a.M) continue;
        const v4f x = *reinterpret_cast<const v4f*>(rows + r * RS + c);
        const int64_t o = (int64_t)b * a.os_b + (int64_t)h * a.os_h + (int64_t)(m0 + r) * a.os_n + c;
        store4(a.out, a.out_dt, o, x);
    }
}

// lse = ln 2 * lse + shift_mul * shift, in place: 12 bytes per row, a launch of 2-3 us.
__global__ __launch_bounds__(kCombineThreads) void lse_natural_kernel(float* lse, const float* shift, float shift_mul, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * kCombineThreads + threadIdx.x;
    if (i >= n) return;
    const float x = lse[i] * 0.693147180559945309f;
    lse[i] = shift ? __builtin_fmaf(shift[i], shift_mul, x) : x;
}

}  // namespace

int launch_lse_natural(float* lse, const float* shift, float shift_mul, int64_t n, hipStream_t stream) {
    const int64_t wgs = (n + kCombineThreads - 1) / kCombineThreads;
    if (wgs > 0x7fffffffLL) return fail(SAGE_E_UNSUPPORTED, "sage_lse_natural: too many rows for one launch");
    hipLaunchKernelGGL(lse_natural_kernel, dim3((unsigned)wgs), dim3(kCombineThreads), 0, stream, lse, shift, shift_mul, n);
    return check_launch("lse_natural_kernel");
}

// One row tile always: B1 H8/8 M1 N8192 19 us against 24 us on the 256-row tiles of the pipelined kernel, B4 H32/32 M1 N4096
// 46 against 57 us (bf16, head_dim 128, dense).  Two row tiles (one wave per SIMD) where they hold several heads that
// would otherwise walk over K and V one by one: B8 H32/4 M8 N8192 36 against 185 us.  A head that fills them alone
// gains nothing (SageAttention B16 H32/32 M64 N1024: 54 against 52 us).
bool decode_serves(int64_t heads_q, int64_t heads_kv, int64_t qo_len) {
    const int64_t groups = heads_q / heads_kv, rows = groups * qo_len;
    return rows <= 32 || (groups > 1 && rows <= kDecodeRows);
}

// Runs of the keys of one (batch, K/V head) for attn_decode_kernel: a workgroup for every CU, whose eight waves keep
// the HBM busy; at least one 32-key tile per wave.
static int plan_decode_split(int64_t items, int64_t rows, int64_t nk) {
    const int64_t smax = nk / kMinStepsPerSplit < kMaxSplits ? nk / kMinStepsPerSplit : kMaxSplits;
    float best = 0.0f;
    int best_s = 1;
    for (int64_t s = 1; s <= smax; s++) {
        const int64_t steps = (nk + s - 1) / s;
        if ((nk + steps - 1) / steps != s) continue;  // (a run without a key)
        // (unsplit with more items than CUs: four-wave workgroups, two per CU; two row tiles: four waves, one per CU)
        const bool pairs = s == 1 && rows <= 32 && items > kComputeUnits;
        const int64_t slots = pairs ? 2 * kComputeUnits : kComputeUnits, waves = pairs || rows > 32 ? 4 : 8;
        const int64_t rounds = (items * s + slots - 1) / slots, tiles = (2 * steps + waves - 1) / waves;  // tiles per wave
        const float cost = (float)rounds * ((float)tiles + 2.0f) + (s > 1 ? 0.5f + 0.01f * (float)s : 0.0f);
        if (s == 1 || cost < 0.97f * best) { best = cost; best_s = (int)s; }
    }
    return best_s;
}

// Short calls on attn_decode_kernel, a workgroup per 32-row tile of a K/V head's packed query rows (and run of its keys), instead
// of one per 256 rows: they end in the time one workgroup takes, in which eight waves walk over the keys side by side instead of
// one after the other, and a kernel that runs only a few steps spends less on its start.  Returns the runs of the keys, 0: not here.
// Every workgroup has a compute unit of its own; or there are two or three for each where half of them are short (causal), where two
// fit a CU (head_dim 64) or where the pipelined kernel runs its instance that hides keys (a ragged last tile).  The K/V rows that
// all of them read, once per row tile, stay below 100 MB (causal, half of them: 130).  Times in us fitted to 350 launches within
// 12 %; over 1750 others of its range 0.72 (int8) and 0.79 (dense) of the time on the pipelined kernel on average, five and 25 of them more
// than 2.5 % slower (worst: int8 B6 H2 M67 N13312 D64 21.0 -> 23.3, dense B1 H8 M82 N3584 D128 17.3 -> 20.1).
// Measured, pipelined kernel -> here (us, in a graph):
//   int8  D64  B1 H2 M256 N256 8.0 -> 5.4, H8 N512 causal 22 -> 6.6, H8 N1024 18 -> 9.2, H2 N2048 causal 25 -> 12; D128 H8 N512 17 -> 10.4
//   dense D128 H2 N200 13.2 -> 9.4, H8 N512 causal 35 -> 12.6, H8 N128 causal 10.3 -> 7.5, H2 N2048 28 -> 23
//   more than one per CU: int8 D64 H32 M512 N512 11.6 -> 9.1, H96 N200 causal 10.7 -> 7.3, H64 N384 causal 12.1 -> 9.1, dense D64 H64 N200
//   10.0 -> 8.0; beyond: int8 D64 H96 N256 8.6 (10.3 here), dense D64 H64 N256 8.3 (9.2), int8 D128 H64 N256 10.2 (14.7)
//   not here: int8 D128 H32 M64 N16384 52 (65 here), dense D128 H32/32 M128 N128 9.1 (11.5), H32 M64 N1024 15.0 (16.1)
static int plan_row_tiles(int64_t batch, int64_t heads_q, int64_t heads_kv, int64_t qo_len, int64_t kv_len, bool causal,
                          int64_t head_dim, bool int8, bool with_workspace) {
    const int64_t rows = heads_q / heads_kv * qo_len, wgs = batch * heads_kv * ((rows + 31) / 32), nk = (kv_len + BN - 1) / BN;
    const bool ragged = kv_len % BN != 0;
    const int64_t halves = causal ? (head_dim == 64 ? (int8 ? 6 : 5) : 4)  // workgroups per two CUs
                         : (head_dim == 64 && int8) || (ragged && (head_dim == 64 || int8)) ? 4 : 2;
    if (2 * wgs > halves * kComputeUnits || kv_len >= (1 << 22)) return 0;
    const float mb = (float)wgs * (float)(kv_len * head_dim * (int8 ? 3 : 4)) * 1e-6f;
    if (mb > (causal ? 130.0f : 100.0f) || (rows <= 64 && !int8 && kv_len >= 1024)) return 0;  // (two row tiles of a head: no gain in 16 bits)
    if (qo_len > kv_len && kv_len >= 512) return 0;  // (cross attention over keys that can be split keeps the key split of 256-row blocks)
    // a workgroup: its start and end, and each turn of its waves over 32 keys each; the K/V bytes; the second launch
    const float start = int8 ? (head_dim == 64 ? 4.5f : 7.1f) : (head_dim == 64 ? 5.7f : 8.4f);
    const float turn = int8 ? (head_dim == 64 ? 0.9f : 1.4f) : (head_dim == 64 ? 1.0f : 2.2f);
    const float combine = head_dim == 64 ? 2.2f : 3.6f;
    const int64_t smax = with_workspace ? (nk / kMinStepsPerSplit < kMaxSplits ? nk / kMinStepsPerSplit : kMaxSplits) : 1;
    float best = 0.0f;
    int best_s = 1;
    for (int64_t s = 1; s <= smax; s++) {
        const int64_t steps = (nk + s - 1) / s;
        if ((nk + steps - 1) / steps != s || (s > 1 && wgs * s > kComputeUnits)) continue;  // (a run without a key; a second round)
        const float cost = start + turn * (float)((2 * steps + 7) / 8) +
                           (s > 1 ? combine + (head_dim == 64 ? 4.8f : 0.7f) * (float)(s * batch * heads_q * qo_len * head_dim) * 1e-6f : 0.0f);
        if (s == 1 || cost < best) { best = cost; best_s = (int)s; }
    }
    return best_s;
}

// Plans of the pipelined kernel, in steps.  Fitted to 38 shapes (1 to 96 heads, 512 to 16384 keys, both flags, both
// head_dims, int8 and 16-bit Q and K) within 5 % for the cut launch and 10 % for the others: a workgroup spends kFixed on
// the prologue and epilogue of each item or piece of one, a launch kLaunch, a second one kCombine, a piece that leaves a
// partial result kPartial (132 KB stored, read again by the combine kernel).  A chip that is partly idle clocks higher
// (head_dim 128: 79 us a workgroup at half the CUs, 100 us at all of them).
constexpr float kFixed = 5.0f, kLaunch = 4.0f, kCombine = 3.0f, kPartial = 2.5f;
constexpr float kCombineRows = 4.0f, kPartialRows = 4.0f;  // the key split stores its partial results row by row, in 16-byte pieces; per 256 rows of each CU

// Measured (us, pairs or key split -> plan taken; SageAttention / dense, bf16):
//   longest first  B1 H32/8 N3001 causal 86 -> 78 / 99 -> 93, B1 H40 N4096 causal 189 -> 157 / 246 -> 192,
//                  B2 H24 N3001 D64 causal 113 -> 84 / 120 -> 84; many heads per XCD lose the L2 (B16 H32 N2048 536 -> 599)
//   cut            B1 H16 N4096 causal 108 -> 79 / 129 -> 91, B1 H12 N8192 D64 causal 206 -> 127 / 222 -> 131,
//                  B1 H33 N4096 250 -> 215 / 303 -> 259, B1 H5 N14000 524 -> 372 / 709 -> 488;
//                  short items lose (B6 H16 N1000 causal 46 -> 62)
//   key split      B1 H30 M512 N4096 70 -> 44 / 76 -> 48; not B2 H16 N512 (25 against 14), B1 H20 N1024 (31 against 23)
LaunchPlan plan_launch(int64_t batch, int64_t heads_q, int64_t heads_kv, int64_t qo_len, int64_t kv_len, bool causal,
                       int64_t head_dim, bool int8, bool with_workspace) {
    LaunchPlan plan{1, 0, false, false};
    const int64_t nk = (kv_len + BN - 1) / BN;
    if (decode_serves(heads_q, heads_kv, qo_len)) {
        if (with_workspace) plan.nsplit = plan_decode_split(batch * heads_kv, heads_q / heads_kv * qo_len, nk);
        return plan;
    }
    if (const int runs = plan_row_tiles(batch, heads_q, heads_kv, qo_len, kv_len, causal, head_dim, int8, with_workspace)) {
        plan.nsplit = runs;
        plan.row_tiles = true;
        return plan;
    }
    const int64_t nq = (qo_len + kFastRows - 1) / kFastRows, heads = batch * heads_q;
    const int64_t per_head = causal ? (nq + 1) / 2 : nq;  // pairs under the causal flag
    const int64_t base = heads * per_head;
    // beyond eight rounds the hand-over between rounds hides what a plan could gain
    if (heads <= 0 || base >= 8 * kComputeUnits || qo_len >= (1 << 22) || kv_len >= (1 << 22)) return plan;
    const CutLine line((int)qo_len, (int)kv_len, causal);
    const int64_t items = heads * line.nq, total = heads * line.head;
    const float cus = (float)kComputeUnits;
    auto busy = [&](float longest) {  // the chip's higher clock while CUs idle
        const float util = (float)total / (cus * longest);
        return util < 1.0f ? 0.7f + 0.3f * util : 1.0f;
    };
    // ---- whole items: as they come, or in pairs
    const int shorter = causal && nq > 1 ? line.len((int)(nq / 2 - 1)) : 0;  // the most even pair is the longest
    const int mirror = line.len((int)(nq - 1 - (nq > 1 ? nq / 2 - 1 : 0)));
    const float pair = causal ? fmaxf((float)(shorter + mirror), (float)(line.len((int)nq - 1) + (nq > 1 ? line.len(0) : 0))) : (float)nk;
    const float each = pair + kFixed * (causal && nq > 1 ? 2.0f : 1.0f);
    const int64_t full = base / kComputeUnits, rest = base % kComputeUnits;
    float best = kLaunch;
    if (full == 0) best += each * busy(pair);
    else best += each * ((float)full + (rest == 0 ? 0.0f : 0.66f + 0.34f * fmaxf(0.0f, (float)(2 * rest) / cus - 1.0f)));
    // ---- one workgroup per item, longest first (causal): the bounds of any such order
    if (causal && nq > 1) {
        float lpt = fmaxf(((float)nk + kFixed) * busy((float)nk), ((float)total + kFixed * (float)items) / cus + 3.0f);
        for (int64_t i = kComputeUnits, k = 2; i < items; i += kComputeUnits, k++)
            lpt = fmaxf(lpt, (float)k * ((float)line.len((int)(line.nq - 1 - i / heads)) + kFixed));
        lpt += kLaunch;
        if (lpt < 0.95f * best) { best = lpt; plan.longest_first = true; }
    }
    // ---- the keys of every item (pair) split, where the chip would be less than 80 % busy
    const int smax = !with_workspace || base * 5 >= kComputeUnits * 4 ? 1
                     : (int)(nk / kMinStepsPerSplit < kMaxSplits ? nk / kMinStepsPerSplit : kMaxSplits);
    const bool few = items <= kFewItems;
    if (few) best = pair + 6.0f;
    for (int s = 2; s <= smax; s++) {
        const int64_t steps = (nk + s - 1) / s;
        if ((nk + steps - 1) / steps != s) continue;  // (a run without a key)
        const float rounds = (float)((base * s + kComputeUnits - 1) / kComputeUnits);
        const float run = causal && nq > 1 ? (float)steps + fminf((float)steps, (float)shorter) + 2.0f * kFixed : (float)steps + kFixed;
        const float cost = few ? (float)steps + 6.0f + 0.25f * (float)s
                               : kLaunch + kCombineRows + rounds * run + kPartialRows * (float)(s * heads * qo_len) / (cus * (float)kFastRows) + 0.25f * (float)s;
        if (cost < 0.95f * best) { best = cost; plan.nsplit = s; plan.longest_first = false; }
    }
    if (few) return plan;
    // ---- the launch cut into equal shares.  (Without the causal flag not where one round fills 80 % of the chip.)
    const bool one_round = !causal && base * 5 >= kComputeUnits * 4 && base <= kComputeUnits;
    if (with_workspace && !one_round && total < (1 << 23) && total >= 2 * kMinStepsPerShare) {
        const int64_t wgs = total / kMinStepsPerShare < kComputeUnits ? total / kMinStepsPerShare : kComputeUnits;
        const float cost = kLaunch + kCombine + (float)total / (float)wgs + kFixed * (1.0f + (float)items / (float)wgs) + 2.0f * kPartial +
                           0.25f * (float)nk * (float)wgs / (float)total;  // (the parts of an item)
        if (cost < 0.93f * best) plan = LaunchPlan{1, (int)wgs, false, false};
    }
    return plan;
}

int64_t plan_workspace_bytes(const LaunchPlan& plan, int64_t batch, int64_t heads_q, int64_t qo_len, int64_t head_dim) {
    if (plan.cut_wgs > 0) return (int64_t)2 * plan.cut_wgs * kFastRows * (head_dim + 1) * (int64_t)sizeof(float);
    if (plan.nsplit > 1) return (int64_t)plan.nsplit * batch * heads_q * qo_len * (head_dim + 1) * (int64_t)sizeof(float);
    return 0;
}

void apply_cut(AttnArgs& a, int cut_wgs, int64_t batch, int head_dim, void* workspace) {
    a.cut_wgs = cut_wgs;
    a.cut_total = (int)(batch * a.Hq * CutLine(a.M, a.N, a.causal).head);
    a.part_o = static_cast<float*>(workspace);
    a.part_lse = a.part_o + (int64_t)2 * cut_wgs * kFastRows * head_dim;
}

int launch_cut_combine(const AttnArgs& a, int head_dim, hipStream_t stream) {
    dim3 grid((unsigned)((a.cut_wgs - 1) * 8)), block(kCombineThreads);
    if (head_dim == 128) hipLaunchKernelGGL((cut_combine_kernel<128>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((cut_combine_kernel<64>), grid, block, 0, stream, a);
    return check_launch("cut_combine_kernel");
}

// Points `a` (a complete description of the unsplit launch) at the workspace and sets the split fields.
void apply_key_split(AttnArgs& a, int nsplit, int64_t batch, int head_dim, void* workspace) {
    const int64_t rows = batch * a.Hq * a.M;
    a.nsplit = nsplit;
    a.split_steps = (a.nk + nsplit - 1) / nsplit;
    a.out = workspace;
    a.out_dt = SAGE_F32;
    a.os_n = head_dim; a.os_h = (int64_t)a.M * head_dim; a.os_b = (int64_t)a.Hq * a.M * head_dim;
    a.out_split_stride = rows * head_dim;
    a.lse = static_cast<float*>(workspace) + (int64_t)nsplit * rows * head_dim;
    a.lse_split_stride = rows;
    a.lse_mul = 1.0f;
    a.lse_shift = nullptr;
}

int launch_split_combine(const AttnArgs& split, const AttnArgs& whole, int head_dim, int64_t batch, hipStream_t stream) {
    CombineArgs c{};
    c.part_o = static_cast<const float*>(split.out);
    c.part_lse = split.lse;
    c.out = whole.out; c.lse = whole.lse;
    c.os_b = whole.os_b; c.os_h = whole.os_h; c.os_n = whole.os_n;
    c.rows = batch * whole.Hq * whole.M;
    c.Hq = whole.Hq; c.M = whole.M; c.nsplit = split.nsplit; c.out_dt = whole.out_dt;
    c.lse_mul = whole.lse_mul; c.lse_shift = whole.lse_shift; c.lse_shift_mul = whole.lse_shift_mul;
    // eight groups per row while rows alone would leave compute units idle
    const int sg = c.rows * (head_dim / 4) < kComputeUnits * kCombineThreads && c.nsplit >= 8 ? 8 : 1;
    const int rows_per_wg = kCombineThreads / (head_dim / 4 * sg);
    const int64_t wgs = (c.rows + rows_per_wg - 1) / rows_per_wg;
    if (wgs > 0x7fffffffLL) return fail(SAGE_E_UNSUPPORTED, "split combine: too many rows for one launch");
    dim3 grid((unsigned)wgs), block(kCombineThreads);
    if (head_dim == 128) {
        if (sg == 8) hipLaunchKernelGGL((split_combine_kernel<128, 8>), grid, block, 0, stream, c);
        else hipLaunchKernelGGL((split_combine_kernel<128, 1>), grid, block, 0, stream, c);
    } else {
        if (sg == 8) hipLaunchKernelGGL((split_combine_kernel<64, 8>), grid, block, 0, stream, c);
        else hipLaunchKernelGGL((split_combine_kernel<64, 1>), grid, block, 0, stream, c);
    }
    return check_launch("split_combine_kernel");
}

}  // namespace attn
}  // namespace sage
