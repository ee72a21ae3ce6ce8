// Types shared by the attention kernels of libsage_attention_hip.so (gfx950).
#pragma once
#include <utility>

#include "common.h"

namespace sage {
namespace attn {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// compile-time loops: f(IC<0>{}), f(IC<1>{}), ...
template <int I> struct IC { static constexpr int value = I; };
template <typename Fn, int... Is>
__device__ __forceinline__ void sfor_impl(Fn&& f, std::integer_sequence<int, Is...>) { (f(IC<Is>{}), ...); }
template <int N, typename Fn>
__device__ __forceinline__ void sfor(Fn&& f) { sfor_impl(f, std::make_integer_sequence<int, N>{}); }

constexpr int kThreads = 256;
constexpr int BM = 128;  // query rows per workgroup (= Q quantization block)
constexpr int BN = 64;   // keys per step (= K quantization block)
constexpr int kFastRows = 256;  // query rows per workgroup of the pipelined kernel (attn_fast_kernel.h)
constexpr int kScanRows = 16;  // mask rows per strip of mask_scan_kernel
constexpr float kMasked = -1.0e6f;
constexpr float kTau = 8.0f;  // log2 of the largest P tolerated before the running maximum is advanced

enum { MODE_PLAIN = 0, MODE_CAUSAL = 1, MODE_MASK_BOOL = 2, MODE_MASK_F32 = 3 };

struct AttnArgs {
    const int8_t* q;
    const int8_t* k;
    const void* v;
    void* out;
    const float* q_scale;
    const float* k_scale;
    float* lse;
    const void* mask;
    int64_t qs_b, qs_h, qs_n;
    int64_t ks_b, ks_h, ks_n;
    int64_t vs_b, vs_h, vs_n;
    int64_t os_b, os_h, os_n;
    int64_t ms_b, ms_h, ms_m, ms_n;
    int32_t Hq, Hkv, M, N, nq, nk, groups;
    int32_t out_dt, causal;
    int32_t total_wg;
    int32_t mask_vec;  // mask rows are contiguous along the keys and every group of four entries is naturally aligned
    int32_t mask_dt;   // storage type of an additive mask (SAGE_F32 / SAGE_F16 / SAGE_BF16)
    int32_t mask_additive;  // the mask tensor is additive (entries of type mask_dt), not bool
    int32_t mask_padded;  // mask rows are readable (bool: and zero) up to the next multiple of 16 bytes past kv_len
    int32_t mask_causal;  // the bool mask is False wherever n > m + (kv_len - qo_len): tiles beyond need no visit
    // Heads that take turns within one q-block in the order of the workgroups (1: a head's q-blocks follow each
    // other).  Under a mask shared by the heads, head_tile heads x several q-blocks run side by side on an XCD, so
    // that both the mask tiles (shared by the heads) and the K/V tiles (shared by the q-blocks) are re-read from L2.
    int32_t head_tile;
    // Split of the keys (under a mask tensor: of the tiles it leaves to visit) over several workgroups per (batch, head, q-block): workgroup s
    // of `nsplit` takes steps s * split_steps .. and writes an fp32 partial output and its base-2 log-sum-exp to
    // out + s * out_split_stride / lse + s * lse_split_stride, which a second kernel combines.  Unsplit: 1, nk, 0, 0.
    int32_t nsplit, split_steps;
    int64_t out_split_stride, lse_split_stride;
    int32_t longest_first;  // (causal, pipelined kernel) a workgroup per q-block, those with the most steps first over all heads; 0: pairs
    // Cut of the whole launch into cut_wgs equal shares of its steps (0: a workgroup per q-block, or pair of them): see
    // CutLine.  Items cut in two or more leave normalized fp32 outputs in part_o and base-2 log-sum-exps in part_lse.
    int32_t cut_wgs, cut_total;  // workgroups; steps of the whole launch
    float* part_o;     // [2 * cut_wgs slots][256 rows x D, in the order of the accumulator registers]
    float* part_lse;   // [2 * cut_wgs][256]
    float lse_mul;     // factor on the base-2 log-sum-exp on its way out (1: as is; ln 2: natural log)
    const float* lse_shift;  // (null: none) [B, Hq, M], added to it with the factor lse_shift_mul: what K smoothing took off the logits
    float lse_shift_mul;
    // (mask tensors, pipelined kernel) what mask_scan_kernel found (null: every tile is visited): per strip of kScanRows mask
    // rows and 64-key tile the largest entry, per strip the smallest of its rows' largest entries, per 64-key tile of V
    // whether it holds an Inf or NaN.  scan_strips: strips of a mask batch.  visit_group: tiles per bit of the visit word.
    const float* scan_top;  // [mask batches][scan_strips][nk]  (+0: every entry is 0, -0: the largest one is)
    const float* scan_low;  // [mask batches][scan_strips]
    const unsigned* scan_v; // [B][Hkv][nk]
    int32_t scan_strips, visit_group;
    float qk_scale;    // 16-bit Q and K only: sm_scale * log2(e), the one scale of every score (q/k point at 16-bit data)
};

// The steps of a launch as one line, which is cut into equal shares: head after head, within a head its items
// (q-blocks of 256 rows), within an item its 64-key steps.  Under the causal flag the items of a head lie in pairs of a
// long and a short one (nq - 1 - j, then j), whose lengths add up to the same: where a share is a pair's length over a
// whole number, every pair ends at a cut.  `dead` leading items see no key (qo_len > kv_len): one step each (all of it
// hidden), at the end of the head.
struct CutLine {
    int nq, nk, dead, c, first_pair, pair, head;  // live item i (counted from `dead`): 4 (i + 1) + c steps, the last one nk
    bool causal;
    __host__ __device__ CutLine(int M, int N, bool causal_) : nq((M + kFastRows - 1) / kFastRows), nk((N + BN - 1) / BN), causal(causal_) {
        dead = 0; c = 0; first_pair = nk; pair = nk; head = nq * nk;
        if (!causal) return;
        const int shift = N - M;
        c = shift >= 0 ? (shift + BN - 1) / BN : -((-shift) / BN);  // floor((shift + 63) / 64)
        dead = c < 0 ? (-c) / 4 : 0;
        if (dead >= nq) dead = nq - 1;
        c += 4 * dead;
        const int live = nq - dead;
        first_pair = nk + (live > 1 ? 4 + c : 0);
        pair = 4 * (live + 1) + 2 * c;
        const int pairs = live / 2;  // whole ones; an odd count leaves the middle item alone
        head = (pairs > 0 ? first_pair + (pairs - 1) * pair : 0) + (live & 1 ? len(dead + live / 2) : 0) + dead;
    }
    __host__ __device__ int len(int iq) const {  // steps of item iq
        if (!causal) return nk;
        return iq < dead ? 1 : iq == nq - 1 ? nk : 4 * (iq - dead + 1) + c;
    }
    __host__ __device__ int start(int iq) const {  // of item iq, within its head
        if (!causal) return iq * nk;
        if (iq < dead) return head - dead + iq;
        const int live = nq - dead, i = iq - dead, mirror = live - 1 - i, p = i < mirror ? i : mirror;
        return (p == 0 ? 0 : first_pair + (p - 1) * pair) + (i < mirror ? len(dead + mirror) : 0);
    }
    __host__ __device__ int item(int r) const {  // the item that holds position r of a head
        if (!causal) return r / nk;
        if (r >= head - dead) return r - (head - dead);
        const int live = nq - dead, p = r < first_pair ? 0 : 1 + (r - first_pair) / pair;
        const int longer = nq - 1 - p;
        return r - (p == 0 ? 0 : first_pair + (p - 1) * pair) < len(longer) || 2 * p == live - 1 ? longer : dead + p;
    }
};
// the log-sum-exp of a row as the caller gets it, from its base-2 one
__device__ __forceinline__ float lse_out(float lse2, float mul, const float* shift, float shift_mul, int64_t row) {
    const float x = lse2 * mul;
    return shift ? __builtin_fmaf(shift[row], shift_mul, x) : x;
}

// first step of share w of W (total steps < 2^23, W <= 256), and the share that holds step pos
__host__ __device__ inline int cut_begin(int w, int W, int total) { return (int)((unsigned)w * (unsigned)total / (unsigned)W); }
__host__ __device__ inline int cut_owner(int pos, int W, int total) {
    return (int)((((unsigned)pos + 1u) * (unsigned)W - 1u) / (unsigned)total);
}

template <typename VT> struct PV;
template <> struct PV<__bf16> {
    typedef bf16x8 vec;
    static __device__ __forceinline__ v16f mfma(vec a, vec b, v16f c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ v4f mfma16(vec a, vec b, v4f c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    // acc + p[2c] + p[2c+1]
    static __device__ __forceinline__ float dot2_ones(vec p, int c, float acc) {
        typedef __bf16 v2 __attribute__((ext_vector_type(2)));
        const v2 ones = {(__bf16)1.0f, (__bf16)1.0f};
        const v2 pr = {p[2 * c], p[2 * c + 1]};
        return __builtin_amdgcn_fdot2_f32_bf16(pr, ones, acc, false);
    }
};
template <> struct PV<_Float16> {
    typedef f16x8 vec;
    static __device__ __forceinline__ v16f mfma(vec a, vec b, v16f c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ v4f mfma16(vec a, vec b, v4f c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ float dot2_ones(vec p, int c, float acc) {
        typedef _Float16 v2 __attribute__((ext_vector_type(2)));
        const v2 ones = {(_Float16)1.0f, (_Float16)1.0f};
        const v2 pr = {p[2 * c], p[2 * c + 1]};
        return __builtin_amdgcn_fdot2(pr, ones, acc, false);
    }
};


// Launches the software-pipelined kernel: no mask tensor, and qo_len <= kv_len when causal.
// head_dim 64 / 128, V dtype fp16 / bf16.
int launch_fast(const AttnArgs& a, int head_dim, int v_dtype, bool causal, hipStream_t stream);

// How a launch is laid out (split_combine.hip).  Whole: a workgroup per item (256 queries of a head), or under the causal
// flag per pair of a short and a long one; longest_first: per item under the causal flag too, the longest first.  With a
// workspace, where that leaves compute units idle: nsplit > 1 workgroups share the keys of each item (pair), or cut_wgs > 0
// workgroups take equal shares of all steps of the launch.  row_tiles: short calls, on attn_decode_kernel (launch_decode).  apply_* turn the arguments of the whole launch into those of
// the other (partial results in `workspace`, plan_workspace_bytes large); launch_*_combine then write what the whole launch would have.
struct LaunchPlan { int nsplit, cut_wgs; bool longest_first, row_tiles; };
LaunchPlan plan_launch(int64_t batch, int64_t heads_q, int64_t heads_kv, int64_t qo_len, int64_t kv_len, bool causal,
                       int64_t head_dim, bool int8, bool with_workspace);
int64_t plan_workspace_bytes(const LaunchPlan& plan, int64_t batch, int64_t heads_q, int64_t qo_len, int64_t head_dim);
void apply_cut(AttnArgs& a, int cut_wgs, int64_t batch, int head_dim, void* workspace);
int launch_cut_combine(const AttnArgs& a, int head_dim, hipStream_t stream);
void apply_key_split(AttnArgs& a, int nsplit, int64_t batch, int head_dim, void* workspace);
int launch_split_combine(const AttnArgs& split, const AttnArgs& whole, int head_dim, int64_t batch, hipStream_t stream);

// The kernel for few query rows (attn_decode.hip): no mask tensor, qo_len rows of each query head that shares a K/V
// head, up to kDecodeRows in a workgroup (decode_serves), more in tiles of 32 (row_tiles); any kv_len, causal with any qo_len.  Splits its keys like the pipelined kernel.
constexpr int kDecodeRows = 64;
bool decode_serves(int64_t heads_q, int64_t heads_kv, int64_t qo_len);
int launch_decode(const AttnArgs& a, int64_t batch, int head_dim, int v_dtype, bool int8, hipStream_t stream);

// The pipelined kernel under a bool mask tensor or an additive fp16 / bf16 one, where fast_serves_mask() says so (a.mask
// set; esz: bytes per mask entry).
bool fast_serves_mask(const AttnArgs& a, int head_dim, int esz);
int launch_fast_masked(const AttnArgs& a, int head_dim, int v_dtype, hipStream_t stream);
int launch_fast_additive(const AttnArgs& a, int head_dim, int v_dtype, hipStream_t stream);
int launch_fast_additive_causal(const AttnArgs& a, int head_dim, int v_dtype, hipStream_t stream);

// The scan of a mask that the heads share, ahead of the pipelined kernel (mask_scan.hip): bytes of workspace it takes (0: the
// rule on sizes says no), and its launch, which fills the scan fields of `a`.
int64_t mask_scan_bytes(const AttnArgs& a, int64_t batch, int head_dim);
int mask_splits(const AttnArgs& a, int64_t batch, int head_dim);  // runs of the tiles to visit, where the mask is scanned
int launch_mask_scan(AttnArgs& a, int64_t batch, int head_dim, int v_dtype, void* workspace, hipStream_t stream);

// The pipelined kernel on 16-bit Q and K (dense attention); causal with any qo_len / kv_len.
int launch_flash(const AttnArgs& a, int head_dim, int dtype, bool causal, hipStream_t stream);

}  // namespace attn
}  // namespace sage
