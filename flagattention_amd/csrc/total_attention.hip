// Total attention of the dense flash_attention for gfx950: tot[b, h, n] = sum over queries m of
// softmax(sm_scale * q.k^T)[m, n], recomputed from Q, K and the log normalizer the forward pass returned
// (FlagAttention src/flag_attn/total.py:64-160 is the kernel it stands in for, flash.py:142-157 its call site).
//
// A wave keeps 64 keys in registers for the whole launch and the workgroup's four waves (256 keys) walk over the queries
// together, 32 at a time:
//   S^T[key, query] = K . Q^T   (v_mfma_f32_32x32x16_{bf16,f16}: A = the wave's K rows, B = the query rows from LDS)
//   p = exp2(S^T * sm_scale * log2(e) - L[query] * log2(e)),   zero where the causal mask hides the key.
// A lane owns one query column of every tile and 32 of the 64 keys, so the sum over queries is first kept per lane (32
// running sums) and folded across the 32 lanes of each half of the wave once, at the end.
//
// Bound by vector and matrix instructions (about 700 and 512 issue cycles per wave and tile at head_dim 128; full tiles
// run at about 930 cycles each).  Query tiles go through LDS because four waves read each: every wave loading its own
// (with only 32 keys per wave) asked the L1 for twice the bytes it delivers.  The tiles are loaded three ahead, straight
// into LDS.  Workgroups are handed out longest first over all heads: with the key blocks of one head side by side, the
// last heads' long blocks started late (B4 H32 M4096 N4096 D128 fp16 causal 425 us, longest first 280 us; without the
// causal flag 523 us).  Where key blocks alone do not fill the chip the queries are cut into runs (total_chunk), whose
// sums go to a workspace and are added in order.  Before, with a wave per 32 keys loading queries into registers:
// B1 H16 M4096 N4096 D128 causal 212 -> 41 us, B4 H32 M4096 N4096 1739 -> 275 us, B8 H16 M2048 N2048 D64 210 -> 50 us.
// Issuing the matrix instructions of the next tile between the exponentials of the current one (two score sets, two
// waves per SIMD) ran no faster than three waves in different phases.
#include "attn_common.h"

namespace sage {
namespace {

using namespace attn;

struct TotalArgs {
    const void* q;
    const void* k;
    const float* log_normalizer;  // [B, Hq, M], natural log
    float* total;                 // [B, Hq, N]; of run r at total + r * run_stride
    int64_t run_stride;
    int32_t chunk;                // query tiles of a run at most (TotalRuns)
    int32_t BH;                   // batch * heads
    int64_t qs_b, qs_h, qs_n;
    int64_t ks_b, ks_h, ks_n;
    int32_t Hq, M, N, groups, causal;
    float qk_scale;  // sm_scale * log2(e)
};

constexpr int kTotalWaves = 4;
constexpr int kTotalThreads = 64 * kTotalWaves;
constexpr int kWaveKeys = 64;
constexpr int kWgKeys = kWaveKeys * kTotalWaves;
constexpr int kTileQ = 32;
// The queries that see a key block, cut into runs of about equal length, one workgroup each.
struct TotalRuns {
    int tiles, chunk, shift;  // query tiles in all; of a run at most; kv_len - qo_len
    bool causal;
    __host__ __device__ int first(int kb) const {  // first query tile that sees a key of block kb: m + shift >= its first key
        const int m = causal ? kb * kWgKeys - shift : 0;
        return m > 0 ? m / kTileQ : 0;
    }
    __host__ __device__ int count(int kb) const { return (tiles - first(kb) + chunk - 1) / chunk; }
    __host__ __device__ int len(int kb) const { const int c = count(kb); return (tiles - first(kb) + c - 1) / c; }
};
constexpr int kRing = 4;  // query tiles resident in LDS: the one in work and three on their way

// WIDE: the rows of a query tile lie further apart than 32-bit byte offsets reach, or in descending order (64-bit addresses
// per lane).
template <int D, typename VT, bool WIDE>
__global__ __launch_bounds__(kTotalThreads, 3) void total_attention_kernel(TotalArgs a) {
    using PVT = PV<VT>;
    using vec16 = typename PVT::vec;
    constexpr int KS = D / 16;      // matrix instructions per 32 x 32 tile
    constexpr int RS = 2 * D;       // bytes per query row
    constexpr int CPR = RS / 16;    // 16-byte chunks per query row
    constexpr int LOADS = kTileQ * CPR / kTotalThreads;  // 1 KB loads per wave and tile
    __shared__ __attribute__((aligned(16))) unsigned char qtile[kRing][kTileQ * RS];
    __shared__ float ltile[kRing][kTotalWaves][64];      // log normalizers of a tile's queries, a copy per wave
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    // Heads fastest, so that a head stays on one XCD and the workgroups with the most tiles come first: under the causal
    // flag the last queries see every key and the first keys are seen by every query.
    const int nkb = (a.N + kWgKeys - 1) / kWgKeys;
    const int bh = blockIdx.x % a.BH, rest = blockIdx.x / a.BH;
    const TotalRuns runs{(a.M + kTileQ - 1) / kTileQ, a.chunk, a.N - a.M, a.causal != 0};
    int kb = 0, run = rest;
    if (a.chunk >= runs.tiles) kb = rest, run = 0;  // (one run per block)
    else
        for (int c; kb < nkb - 1 && run >= (c = runs.count(kb)); kb++) run -= c;
    const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.groups;
    const int n0 = kb * kWgKeys + wave * kWaveKeys;  // (may lie past the last key: such a wave multiplies copies of it)
    const int shift = a.N - a.M;
    const int m_sees = a.causal ? max(-shift, 0) : 0;  // first query that sees a key

    // K rows of this wave: lane (key l32, half) holds elements 16 t + 8 half .. + 7 of its row for step t
    vec16 kf[2][KS];
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
        const int key = min(n0 + 32 * kt + l32, a.N - 1);  // keys past the end re-read the last one; their sums are not stored
        const VT* kp = static_cast<const VT*>(a.k) + (int64_t)b * a.ks_b + (int64_t)hk * a.ks_h + (int64_t)key * a.ks_n + 8 * half;
#pragma unroll
        for (int t = 0; t < KS; t++) kf[kt][t] = *reinterpret_cast<const vec16*>(kp + 16 * t);
    }
    const VT* qbase = static_cast<const VT*>(a.q) + (int64_t)b * a.qs_b + (int64_t)h * a.qs_h;
    const float* lbase = a.log_normalizer + ((int64_t)b * a.Hq + h) * a.M;

    // the run's queries
    const int m_lo = (runs.first(kb) + run * runs.len(kb)) * kTileQ;
    const int m_hi = min(m_lo + runs.len(kb) * kTileQ, a.M);

    const int ntiles = max(m_hi - m_lo + kTileQ - 1, 0) / kTileQ;

    // Query tile t of the run -> ring buffer t % 4, straight into LDS (16 bytes per lane; written in assembly because the
    // compiler would wait for every outstanding load before each LDS read, tracked with s_waitcnt vmcnt below).  Chunk c
    // of row r lies at chunk c ^ r of its LDS row (modulo the chunks of a row), so that the fragment reads, one chunk of
    // 32 rows at a time, spread over all banks: the load fetches the chunk that belongs where a lane writes.
    // m0 holds the LDS address of the load; nothing else in this kernel uses it.  Tiles past the last one load it again.
    const unsigned lds_q = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)&qtile[0][0];
    const unsigned lds_l = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)&ltile[0][0][0];
    unsigned qoff[LOADS];  // byte offsets of this lane's pieces of a tile
    auto set_offsets = [&](int last) {  // last: the tile's last row
#pragma unroll
        for (int e = 0; e < LOADS; e++) {
            const int row = (64 / CPR) * (LOADS * wave + e) + lane / CPR;
            qoff[e] = (unsigned)min(row, last) * (unsigned)(a.qs_n * 2) + 16 * ((lane % CPR) ^ (row & (CPR - 1)));
        }
    };
    set_offsets(kTileQ - 1);
    auto fetch = [&](int t) {
        const int m0 = m_lo + kTileQ * min(t, ntiles - 1), buf = t & (kRing - 1);
        if (!WIDE && m0 + kTileQ > a.M) set_offsets(a.M - 1 - m0);  // (every later tile is this one again)
        const unsigned char* base = reinterpret_cast<const unsigned char*>(qbase + (int64_t)m0 * a.qs_n);
#pragma unroll
        for (int e = 0; e < LOADS; e++) {
            const unsigned dst = lds_q + (unsigned)(buf * kTileQ * RS + 1024 * (LOADS * wave + e));
            if constexpr (WIDE) {
                const int row = (64 / CPR) * (LOADS * wave + e) + lane / CPR;
                const unsigned char* src = base + (int64_t)min(row, a.M - 1 - m0) * (a.qs_n * 2) + 16 * ((lane % CPR) ^ (row & (CPR - 1)));
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(src), "s"(dst) : "memory");
            } else {
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(qoff[e]), "s"(base), "s"(dst) : "memory");
            }
        }
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                     :: "v"((unsigned)(4 * min(l32, a.M - 1 - m0))), "s"(lbase + m0), "s"(lds_l + (unsigned)(256 * (kTotalWaves * buf + wave))) : "memory");
    };
    if (ntiles > 0) {
        fetch(0);
        fetch(1);
        fetch(2);
    }
    // (waited for here: inside the loop the compiler's waits for them would also wait for the query tiles on their way)
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int t = 0; t < KS; t++) {
            v4i bits = __builtin_bit_cast(v4i, kf[kt][t]);
            asm volatile("" : "+v"(bits));
            kf[kt][t] = __builtin_bit_cast(vec16, bits);
        }
    float tot[2][16];
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++) tot[kt][i] = 0.0f;

    for (int t = 0; t < ntiles; t++) {
        // all but the two youngest tiles' loads of this wave have landed; past the barrier, those of all waves, and
        // nobody reads the buffer of tile t - 1 any more
        __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * (LOADS + 1)));
        __builtin_amdgcn_s_barrier();
        fetch(t + 3);
        const int mq = m_lo + kTileQ * t, buf = t & (kRing - 1);
        if (a.causal && mq + kTileQ - 1 + shift < n0) continue;  // (the tile's last query sees no key of this wave)
        // queries past the end, and queries that see no key, take L = +inf: every p of theirs is exp2(-inf) = 0
        const float L = ltile[buf][wave][lane];
        float l2 = (unsigned)(mq + l32 - m_sees) < (unsigned)(a.M - m_sees) ? L * 1.44269504088896340736f : INFINITY;
        v16f s[2];
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int i = 0; i < 16; i++) s[kt][i] = 0.0f;
        const unsigned char* row = &qtile[buf][l32 * RS];
#pragma unroll
        for (int c = 0; c < KS; c++) {
            const vec16 qf = *reinterpret_cast<const vec16*>(row + 16 * ((2 * c + half) ^ (l32 & (CPR - 1))));
            s[0] = PVT::mfma(kf[0][c], qf, s[0]);
            s[1] = PVT::mfma(kf[1][c], qf, s[1]);
        }
        if (a.causal && mq + shift < n0 + kWaveKeys - 1) {  // the tile's first query does not see the wave's last key
            const int last = mq + l32 + shift - n0 - 4 * half;  // last key the query sees, from the lane's first one on
            // A log normalizer of NaN (NaN scores) or -inf joins the scores of the keys the query sees: in the exponent it
            // would make the hidden ones NaN as well.
            const float odd = l2 > -INFINITY ? 0.0f : -l2;
            l2 = l2 > -INFINITY ? l2 : 0.0f;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int i = 0; i < 16; i++)  // accumulator register i: key 32 kt + 8 (i / 4) + i % 4 from there
                    s[kt][i] = 32 * kt + 8 * (i >> 2) + (i & 3) <= last ? s[kt][i] + odd : -INFINITY;
        }
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int i = 0; i < 16; i++) tot[kt][i] += __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][i], a.qk_scale, -l2));
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // nothing of this workgroup is on its way into LDS when it ends
    // Fold the 32 query columns of a key through LDS (the ring is free once every wave is here; 4 KB per wave): 32 keys at
    // a time, entry (key, query) at column query ^ key of its row, so that neither the writes (a row at a time) nor the
    // reads (a lane per key, both halves of the wave taking 16 columns each) meet in a bank.  Five rounds of lane
    // exchanges per sum instead took as long as eight tiles.
    __syncthreads();
    float* out = a.total + ((int64_t)b * a.Hq + h) * a.N + run * a.run_stride;
    float* fold = reinterpret_cast<float*>(&qtile[0][0]) + wave * 1024;
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int key = 8 * (i >> 2) + 4 * half + (i & 3);
            fold[32 * key + (l32 ^ key)] = tot[kt][i];
        }
        float x = 0.0f;
#pragma unroll
        for (int c = 0; c < 16; c++) x += fold[32 * l32 + ((16 * half + c) ^ l32)];
        x += __shfl_xor(x, 32);
        const int n = n0 + 32 * kt + l32;
        if (half == 0 && n < a.N) out[n] = x;
    }
}

// total[i] = sum of the runs' sums, in order
__global__ __launch_bounds__(256) void total_runs_kernel(const float* part, float* total, int64_t count, int N, TotalRuns runs) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    const int n = runs.count((int)(i % N) / kWgKeys);
    float x = 0.0f;
    for (int r = 0; r < n; r += 8) {  // eight loads on their way together, the last run again past the end
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = part[(int64_t)min(r + u, n - 1) * count + i];
#pragma unroll
        for (int u = 0; u < 8; u++) x = r + u < n ? x + v[u] : x;
    }
    total[i] = x;
}

// Longest run of queries (in tiles): where the key blocks alone do not fill the chip the queries of each are cut into equal
// runs of at least eight tiles, as many as make three workgroups per CU, all of them resident at once.  (With the same four
// ranges of queries for every block some CUs held 84 tiles and others 40: B1 H16 M4096 N4096 D128 causal, whole call, 142 -> 135
// us; B1 H16/2 M4032 136 -> 128, B3 H8/1 M2048 86.5 -> 83.)  Runs that would be long: three times as many, handed out as others
// end (B6 H2 M9728 D64 causal 285 -> 280 us, 300 with what is resident at once; B1 H32/4 M6995, 896 key blocks, 1204, 1249 uncut).
int total_chunk(int64_t BH, int64_t M, int64_t N, bool causal) {
    constexpr int64_t kResident = 3 * 256, kLongRun = 32;
    const int64_t nkb = (N + kWgKeys - 1) / kWgKeys, tiles = (M + kTileQ - 1) / kTileQ;
    if (BH * nkb >= 4 * 256 || tiles < 16 || tiles > (1 << 24) || N > (1 << 29)) return (int)tiles;
    TotalRuns runs{(int)tiles, 1, (int)(N - M), causal};
    int64_t all = 0;
    for (int kb = 0; kb < nkb; kb++) all += runs.count(kb);
    int64_t slots = kResident, chunk = (BH * all + slots - 1) / slots;
    if (chunk > kLongRun) {
        slots = 3 * kResident;
        chunk = (BH * all + slots - 1) / slots;
        if (chunk < kLongRun) chunk = kLongRun;
    }
    if (chunk < (tiles + 63) / 64) chunk = (tiles + 63) / 64;  // (64 runs at most)
    const int64_t most = tiles / 8;  // (at least eight tiles each)
    if (chunk < (tiles + most - 1) / most) chunk = (tiles + most - 1) / most;
    for (; chunk < tiles; chunk++) {
        runs.chunk = (int)chunk;
        int64_t wgs = 0;
        for (int kb = 0; kb < nkb; kb++) wgs += BH * runs.count(kb);
        if (wgs <= slots) break;
    }
    return (int)(chunk < tiles ? chunk : tiles);
}

int64_t total_run_count(int64_t M, int chunk) { return ((M + kTileQ - 1) / kTileQ + chunk - 1) / chunk; }  // (of the first key block, which has the most)

template <int D, typename VT>
int launch_total(const TotalArgs& a, hipStream_t stream) {
    const int64_t nkb = (a.N + kWgKeys - 1) / kWgKeys;
    const TotalRuns runs{(a.M + kTileQ - 1) / kTileQ, a.chunk, a.N - a.M, a.causal != 0};
    int64_t wgs = nkb;
    if (a.chunk < runs.tiles) {
        wgs = 0;
        for (int kb = 0; kb < nkb; kb++) wgs += runs.count(kb);
    }
    wgs *= a.BH;
    if (wgs > 0x7fffffffLL) return fail(SAGE_E_UNSUPPORTED, "sage_flash_total_attention: too many key blocks for one launch");
    dim3 grid((unsigned)wgs), block(kTotalThreads);
    const bool wide = a.qs_n < 0 || a.qs_n >= (1LL << 25);  // 31 rows of 2-byte elements pass 2^31 bytes
    if (wide) hipLaunchKernelGGL((total_attention_kernel<D, VT, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((total_attention_kernel<D, VT, false>), grid, block, 0, stream, a);
    return check_launch("total_attention_kernel");
}

}  // namespace

int64_t total_workspace_bytes(const sage_flash_params& p) {
    const int64_t runs = total_run_count(p.qo_len, total_chunk(p.batch * p.heads_q, p.qo_len, p.kv_len, p.causal != 0));
    return runs > 1 ? runs * p.batch * p.heads_q * p.kv_len * (int64_t)sizeof(float) : 0;
}

int launch_flash_total_attention(const sage_flash_params& p, const float* log_normalizer, float* total, void* workspace,
                                 int64_t workspace_bytes, hipStream_t stream) {
    TotalArgs a{};
    a.q = p.q.ptr; a.k = p.k.ptr; a.log_normalizer = log_normalizer; a.total = total;
    a.qs_b = p.q.stride_b; a.qs_h = p.q.stride_h; a.qs_n = p.q.stride_n;
    a.ks_b = p.k.stride_b; a.ks_h = p.k.stride_h; a.ks_n = p.k.stride_n;
    a.Hq = (int)p.heads_q; a.M = (int)p.qo_len; a.N = (int)p.kv_len; a.groups = (int)(p.heads_q / p.heads_kv);
    a.causal = p.causal ? 1 : 0;
    a.qk_scale = p.sm_scale * 1.44269504089f;
    a.BH = (int)(p.batch * p.heads_q);
    const int tiles = (int)((p.qo_len + kTileQ - 1) / kTileQ);
    a.chunk = workspace && workspace_bytes >= total_workspace_bytes(p) ? total_chunk(a.BH, p.qo_len, p.kv_len, p.causal != 0) : tiles;
    const int64_t runs = total_run_count(p.qo_len, a.chunk);
    const int64_t count = p.batch * p.heads_q * p.kv_len;
    if (runs > 1) {
        a.total = static_cast<float*>(workspace);
        a.run_stride = count;
    }
    int rc;
    if (p.head_dim == 128)
        rc = p.dtype == SAGE_BF16 ? launch_total<128, __bf16>(a, stream) : launch_total<128, _Float16>(a, stream);
    else
        rc = p.dtype == SAGE_BF16 ? launch_total<64, __bf16>(a, stream) : launch_total<64, _Float16>(a, stream);
    if (rc || runs == 1) return rc;
    const int64_t wgs = (count + 255) / 256;
    if (wgs > 0x7fffffffLL) return fail(SAGE_E_UNSUPPORTED, "sage_flash_total_attention: too many keys for one launch");
    hipLaunchKernelGGL(total_runs_kernel, dim3((unsigned)wgs), dim3(256), 0, stream, (const float*)workspace, total, count, a.N,
                       TotalRuns{tiles, a.chunk, a.N - a.M, a.causal != 0});
    return check_launch("total_runs_kernel");
}

}  // namespace sage
