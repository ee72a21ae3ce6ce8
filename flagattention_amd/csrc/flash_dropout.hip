// Dense attention forward with dropout on P for gfx950, and the dropout mask on its own
// (FlagAttention src/flag_attn/flash.py:387-391, :467-502 is the kernel branch it stands in for;
// src/flag_attn/testing/dropout.py:19-39 the helper that recomputes the mask).
//
// Element (b, h, m, n) of P survives iff rand(seed, offset + ((b H + h) M + m) N + n) > dropout_p, where rand is
// Triton's tl.rand with six rounds: Philox-4x32 on the counter (low word, high word, 0, 0) of the 64-bit sum,
// key (low, high) word of the seed, first output word x -> fp32 (x >= 0 ? x : -x - 1) * 4.6566127342e-10
// (x read as int32).  The row sums of the softmax are taken BEFORE the mask, the output is scaled by
// 1 / (1 - dropout_p) at the end (flash.py:470-477, :499-502).
//
// Six rounds of 32 x 32 -> 64 bit products per score cost more vector instructions than the softmax, so this kernel is
// bound by the vector issue port and is built for it (rates measured with four waves per SIMD, in cycles at 2.4 GHz: integer
// products 5.5, three-input XOR 4.8, exponential 9, FMA and XOR 3; with two waves per SIMD everything takes 5.7 or more):
// * the generator is unrolled by hand (philox6_from_product): 4 full products, 3 high and 1 low half and one 64-bit addition per
//   score instead of 12 full products; what depends on the row only is computed once per row;
// * exclusive ors of three operands are one instruction each (xor3), and so are the last exclusive or and the subtraction of the
//   keep decision;
// * the keep decision is an integer threshold and a sign, applied to two 16-bit P at a time (no compare, no select);
// * the rest is kept small: K and V tiles of 32 keys go straight into LDS for the four waves of a workgroup (32 queries
//   each, S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_32x32x16, V^T by ds_read_b64_tr_b16), one barrier per tile, loads
//   one tile ahead (a tile takes microseconds), registers for four (head_dim 128: three) waves per SIMD;
// * workgroups are handed out longest first over all heads.
// B4 H16 M2048 N2048 D64 fp16 causal 397 -> 143 us, without the causal flag 404 -> 272 us; B2 H32 M4096 N4096 D128 3475 -> 1207
// us, causal 3445 -> 619 us (before: the generator rolled out by the compiler, V^T gathered from LDS entry by entry,
// short rows first).  With xor3, the addends of the counters' products in scalar registers (30 vector registers less at head_dim
// 128) and an exchange of row maxima only where a tile raises one 119, 224, 1031 and 536 us.  Reference points that lag behind
// the maximum of their row by up to 2^8 would make it 112, 212, 977 and 505 us, but P is then rounded at another place than where its
// row's largest is exactly 1, and the error of the output grows by 2 to 23 %.
#include "attn_common.h"

namespace sage {
namespace {

using namespace attn;

// ---- Philox-4x32, six rounds, counter (c0, c1, 0, 0): the first output word
__device__ __forceinline__ uint32_t philox6_first_word(uint32_t c0, uint32_t c1, uint32_t k0, uint32_t k1) {
    constexpr uint32_t KEY_A = 0x9E3779B9u, KEY_B = 0xBB67AE85u, ROUND_A = 0xD2511F53u, ROUND_B = 0xCD9E8D57u;
    uint32_t c2 = 0, c3 = 0;
#pragma unroll
    for (int r = 0; r < 6; r++) {
        const uint64_t pb = (uint64_t)ROUND_B * c2, pa = (uint64_t)ROUND_A * c0;
        const uint32_t hi_b = (uint32_t)(pb >> 32), lo_b = (uint32_t)pb;
        const uint32_t hi_a = (uint32_t)(pa >> 32), lo_a = (uint32_t)pa;
        c0 = hi_b ^ c1 ^ k0;
        c2 = hi_a ^ c3 ^ k1;
        c1 = lo_b;
        c3 = lo_a;
        k0 += KEY_A;
        k1 += KEY_B;
    }
    return c0;
}

// does the element with this 64-bit offset survive?
__device__ __forceinline__ bool dropout_keeps(uint64_t offset, uint32_t k0, uint32_t k1, float dropout_p) {
    const int32_t x = (int32_t)philox6_first_word((uint32_t)offset, (uint32_t)(offset >> 32), k0, k1);
    const int32_t folded = x ^ (x >> 31);  // x >= 0 ? x : -x - 1
    return (float)folded * 4.6566127342e-10f > dropout_p;
}

struct DropArgs {
    const void* q;
    const void* k;
    const void* v;
    void* out;
    float* log_normalizer;  // [B, Hq, M] natural log, or null
    int64_t qs_b, qs_h, qs_n, ks_b, ks_h, ks_n, vs_b, vs_h, vs_n, os_b, os_h, os_n;
    int32_t Hq, M, N, groups, causal, out_dt;
    int32_t BH, nmb;   // batch * heads, 128-query blocks
    int32_t snake;     // blocks of one round over the CUs, 0: plain order
    uint32_t minus_keep_from; // minus the smallest folded output word that is kept
    float qk_scale;    // sm_scale * log2(e)
    float dropout_p, keep_scale;  // keep_scale = 1 / (1 - dropout_p)
    uint32_t seed_lo, seed_hi;
    uint64_t offset;
};

constexpr int kDropWaves = 4;  // 128 queries per workgroup
constexpr int kDropThreads = 64 * kDropWaves;
constexpr int kDropKeys = 32;  // keys per tile

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;

// Philox-4x32 of six rounds for consecutive counters whose high word does not change: what six rounds of
//   (c0, c1, c2, c3) <- (hi(B c2) ^ c1 ^ k0, lo(B c2), hi(A c0) ^ c3 ^ k1, lo(A c0))
// from (low, high, 0, 0) leave to be computed per low word for the first output word.
struct PhiloxRow {
    uint32_t hi_word;  // the counters' high word
    uint32_t x2, x3;   // key words mixed with the product of round two, which depends on the high word only
};

constexpr uint32_t kPhiloxA = 0xD2511F53u, kPhiloxB = 0xCD9E8D57u, kPhiloxKeyA = 0x9E3779B9u, kPhiloxKeyB = 0xBB67AE85u;

__device__ __forceinline__ PhiloxRow philox_row(uint32_t hi_word, uint32_t k0, uint32_t k1) {
    const uint64_t u = (uint64_t)kPhiloxA * (hi_word ^ k0);
    return {hi_word, (uint32_t)(u >> 32) ^ (k1 + kPhiloxKeyB), (uint32_t)u ^ (k1 + 2 * kPhiloxKeyB)};
}

// Three operands in one instruction.  As two XORs (what the compiler makes of a ^ b ^ c) the six rounds and the decision took
// 110 instead of 89 cycles per score and SIMD at four waves, 113 instead of 93 at two.
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) { return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96); }

// a + b, b the same for all lanes: one instruction, b in scalar registers (as the addend of a product, where the compiler puts it, every
// b of the tile would keep two vector registers)
__device__ __forceinline__ uint64_t add_u64(uint64_t a, uint64_t b) {
    uint64_t r;
    asm("v_lshl_add_u64 %0, %1, 0, %2" : "=v"(r) : "v"(a), "s"(b));
    return r;
}

// first: A * low word, all 64 bits
__device__ __forceinline__ uint32_t philox6_from_product(uint64_t first, const PhiloxRow& r, uint32_t k0, uint32_t k1) {
    auto hi = [](uint64_t x) { return (uint32_t)(x >> 32); };
    const uint64_t b1 = (uint64_t)kPhiloxB * (hi(first) ^ k1);
    const uint64_t a2 = (uint64_t)kPhiloxA * (hi(b1) ^ (k0 + kPhiloxKeyA));
    const uint64_t b2 = (uint64_t)kPhiloxB * ((uint32_t)first ^ r.x2);
    const uint64_t a3 = (uint64_t)kPhiloxA * xor3(hi(b2), (uint32_t)b1, k0 + 2 * kPhiloxKeyA);
    const uint32_t c2 = hi(a2) ^ r.x3;
    const uint32_t c0 = xor3(__umulhi(kPhiloxB, c2), (uint32_t)b2, k0 + 3 * kPhiloxKeyA);
    const uint32_t d2 = xor3(hi(a3), (uint32_t)a2, k1 + 3 * kPhiloxKeyB);
    const uint32_t e2 = xor3(__umulhi(kPhiloxA, c0), (uint32_t)a3, k1 + 4 * kPhiloxKeyB);
    return xor3(__umulhi(kPhiloxB, e2), kPhiloxB * d2, k0 + 5 * kPhiloxKeyA);
}

// negative iff the element with this output word is dropped: the word folds to [0, 2^31) and is kept from keep_from on
// (exclusive or and addition are one instruction)
__device__ __forceinline__ int32_t drop_sign(uint32_t word, uint32_t minus_keep_from) {
    const int32_t x = (int32_t)word;
    return (int32_t)((uint32_t)(x ^ (x >> 31)) + minus_keep_from);
}

template <int D> __device__ __forceinline__ int drop_v_swizzle(int row) { return D == 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1); }

// KG: groups of four waves that share the queries of a workgroup and take its key tiles in turn (drop_groups).  The second
// launch bound is waves per SIMD, whatever KG is: with fewer asked for, two groups at head_dim 64 took 132 registers and one
// workgroup filled a CU (B1 H32 M2048 N2048 D64 153 -> 140 us, causal 107 -> 80 us, B4 H16 M1024 N1024 83 -> 77 and 58 -> 45
// us; three instead of two at head_dim 128: 131 -> 120 us for B3 H16 M2048 N2048 causal, whose blocks are then resident at once, 85 ->
// 80 us for M1500; nothing in longer launches, B2 H32 M4096 N4096 1028 and 1031 us).
constexpr int drop_waves_per_simd(int head_dim) { return head_dim == 128 ? 3 : 4; }

// WIDE: the rows of a K or V tile lie further apart than 32-bit byte offsets reach, or in descending order (64-bit
// addresses per lane; one group of waves only).
template <int D, typename VT, int KG, bool WIDE = false>
__global__ __launch_bounds__(kDropThreads * KG, drop_waves_per_simd(D)) void flash_dropout_fwd_kernel(DropArgs a) {
    using PVT = PV<VT>;
    using vec16 = typename PVT::vec;
    constexpr int KS = D / 16;      // matrix instructions of one 32 x 32 score tile
    constexpr int DT = D / 32;      // 32-channel tiles of the output
    constexpr int RS = 2 * D;       // bytes per K / V row
    constexpr int CPR = RS / 16;    // 16-byte chunks per row
    constexpr int TILE = kDropKeys * RS;
    constexpr int LOADS = TILE / 1024 / kDropWaves;  // 1 KB loads per wave of a K (of a V) tile
    __shared__ __attribute__((aligned(16))) unsigned char smem[KG][2][2][TILE];  // [group][buffer][K, V]
    __shared__ float row_m[KG > 1 ? KG * 32 * kDropWaves : 1], row_l[KG > 1 ? KG * 32 * kDropWaves : 1];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave_all % kDropWaves, group = wave_all / kDropWaves;
    const int l32 = lane & 31, half = lane >> 5;
    // heads fastest (a head stays on one XCD); under the causal flag the last queries, which see the most keys, first
    // (snake: all workgroups are resident at once, so every second round of 256, one per CU, goes in the reverse order of
    // blocks and a CU holds long and short ones: B4 H16 M2048 N2048 D64 causal 177 -> 166 us, B3 H16 M2048 N2048 D128
    // 132 -> 120)
    const int bh = blockIdx.x % a.BH;
    int rank = blockIdx.x / a.BH;
    if (a.snake > 0 && a.snake < a.nmb && a.nmb < 2 * a.snake) {
        // a second round on some of the CUs only: these, the first ones, hold the shorter blocks of the first round (in plain
        // order B2 H16 M1500 N1500 D64 causal, 384 blocks, takes 68 us instead of 60)
        const int extra = a.nmb - a.snake;
        rank = rank < extra ? a.snake - extra + rank : rank < a.snake ? rank - extra : a.nmb - 1 - (rank - a.snake);
    } else if (a.snake > 0 && (rank / a.snake) % 2 == 1 && (rank / a.snake + 1) * a.snake <= a.nmb) {
        rank = (rank / a.snake) * a.snake + a.snake - 1 - rank % a.snake;
    }
    const int mb = a.nmb - 1 - rank;
    const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.groups;
    const int m0 = mb * (32 * kDropWaves);
    const int my_m = m0 + 32 * wave + l32;
    const bool row_ok = my_m < a.M;
    const int shift = a.N - a.M;

    // Q rows as the B operand: lane (query l32, half) holds elements 16 t + 8 half .. + 7 of its row for step t
    vec16 qf[KS];
    {
        const VT* qp = static_cast<const VT*>(a.q) + (int64_t)b * a.qs_b + (int64_t)h * a.qs_h +
                       (int64_t)min(my_m, a.M - 1) * a.qs_n + 8 * half;
#pragma unroll
        for (int t = 0; t < KS; t++) qf[t] = *reinterpret_cast<const vec16*>(qp + 16 * t);
    }
    // (waited for here: inside the loop the compiler's waits for them would also wait for the tile on its way)
#pragma unroll
    for (int t = 0; t < KS; t++) {
        v4i bits = __builtin_bit_cast(v4i, qf[t]);
        asm volatile("" : "+v"(bits));
        qf[t] = __builtin_bit_cast(vec16, bits);
    }
    const VT* kbase = static_cast<const VT*>(a.k) + (int64_t)b * a.ks_b + (int64_t)hk * a.ks_h;
    const VT* vbase = static_cast<const VT*>(a.v) + (int64_t)b * a.vs_b + (int64_t)hk * a.vs_h;

    // keys that any row of the workgroup / of this wave can see
    int n_end = a.N, wave_end = a.N;
    if (a.causal) {
        n_end = max(min(a.N, min(m0 + 32 * kDropWaves, a.M) + shift), 0);
        wave_end = min(m0 + 32 * wave + 32, a.M) + shift;
    }
    const int my_lim = a.causal ? min(my_m + shift, a.N - 1) : a.N - 1;              // last key this lane's query sees
    const int first_lim = a.causal ? min(m0 + 32 * wave + shift, a.N - 1) : a.N - 1;  // ... the wave's first query
    const int ntiles = (n_end + kDropKeys - 1) / kDropKeys;

    // Tile t of K and V -> one of the group's two buffers, straight into LDS (written in assembly, as in attn_fast_kernel.h: the compiler would
    // wait for every outstanding load before each LDS read; m0 holds the LDS address and nothing else here uses it).  Chunk
    // c of row r lies at chunk c ^ (r mod chunks) for K and at c ^ drop_v_swizzle(r) for V: the load fetches the chunk
    // that belongs where a lane writes, the fragment reads spread over all banks.  Rows past the end re-read the last one.
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)&smem[group][0][0][0];
    unsigned koff[LOADS], voff[LOADS];
    auto set_offsets = [&](int last) {  // last: the tile's last row
#pragma unroll
        for (int e = 0; e < LOADS; e++) {
            const int row = (64 / CPR) * (LOADS * wave + e) + lane / CPR;
            koff[e] = (unsigned)min(row, last) * (unsigned)(a.ks_n * 2) + 16 * ((lane % CPR) ^ (row & (CPR - 1)));
            voff[e] = (unsigned)min(row, last) * (unsigned)(a.vs_n * 2) + 16 * ((lane % CPR) ^ drop_v_swizzle<D>(row));
        }
    };
    set_offsets(kDropKeys - 1);
    auto fetch = [&](int t, int buf) {
        const int n0 = kDropKeys * t;
        if (!WIDE && n0 + kDropKeys > a.N) set_offsets(a.N - 1 - n0);  // (the last tile)
        const VT* kt = kbase + (int64_t)n0 * a.ks_n;
        const VT* vt = vbase + (int64_t)n0 * a.vs_n;
        const unsigned dst = lds0 + (unsigned)(buf * 2 * TILE + 1024 * LOADS * wave);
#pragma unroll
        for (int e = 0; e < LOADS; e++) {
            if constexpr (WIDE) {
                const int row = (64 / CPR) * (LOADS * wave + e) + lane / CPR, r = min(row, a.N - 1 - n0);
                const VT* ksrc = kt + (int64_t)r * a.ks_n + 8 * ((lane % CPR) ^ (row & (CPR - 1)));
                const VT* vsrc = vt + (int64_t)r * a.vs_n + 8 * ((lane % CPR) ^ drop_v_swizzle<D>(row));
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(ksrc), "s"(dst + 1024 * e) : "memory");
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(vsrc), "s"(dst + TILE + 1024 * e) : "memory");
            } else {
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(koff[e]), "s"(kt), "s"(dst + 1024 * e) : "memory");
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff[e]), "s"(vt), "s"(dst + TILE + 1024 * e) : "memory");
            }
        }
    };
    int vtr[DT];  // LDS offsets of the transposed fragment reads (see attn_fast_kernel.h)
    {
        const int s4 = (lane >> 2) & 3, a4 = lane & 3, g1 = (lane >> 4) & 1;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
            vtr[dt] = (4 * half + s4) * RS + 16 * ((4 * dt + 2 * g1 + (a4 >> 1)) ^ drop_v_swizzle<D>(s4)) + 8 * (a4 & 1);
    }

    // offset of element (b, h, my_m, 4 half) in the random stream: this lane's first key of a tile, from the tile's start on
    const uint64_t rng_row = a.offset + (((uint64_t)b * a.Hq + h) * (uint64_t)a.M + (uint64_t)my_m) * (uint64_t)a.N + 4 * half;
    PhiloxRow prow = philox_row((uint32_t)(rng_row >> 32), a.seed_lo, a.seed_hi);

    v16f acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[dt][i] = 0.0f;
    float m_i = -INFINITY, l_i = 0.0f;  // running maximum (unscaled scores) and this half's part of the row sum

    if (group < ntiles) fetch(group, 0);
    const int rounds = (ntiles + KG - 1) / KG;
    for (int r = 0; r < rounds; r++) {
        // vmcnt(0): this round's tiles have landed, for all waves past the barrier; the last round's have been read
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __builtin_amdgcn_s_barrier();
        const int t = r * KG + group;
        if (t + KG < ntiles) fetch(t + KG, (r + 1) & 1);
        const int n0 = kDropKeys * t;
        if (t >= ntiles || (a.causal && n0 >= wave_end)) continue;  // (no query of this wave sees a key of the tile)
        const unsigned char* ktile = smem[group][r & 1][0];
        const unsigned char* vtile = smem[group][r & 1][1];

        v16f s;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.0f;
        int krow = l32 * RS + 16 * (half ^ (l32 & (CPR - 1)));
        asm volatile("" : "+v"(krow));  // (the addresses of the fragments, krow ^ 32 c, are not kept from tile to tile)
#pragma unroll
        for (int c = 0; c < KS; c++) s = PVT::mfma(*reinterpret_cast<const vec16*>(ktile + (krow ^ (32 * c))), qf[c], s);

        // accumulator i of this lane: key n0 + 8 (i / 4) + 4 half + i % 4 of query my_m
        if (n0 + kDropKeys - 1 > first_lim) {
            const int last = my_lim - n0 - 4 * half;
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] = 8 * (i >> 2) + (i & 3) <= last ? s[i] : -INFINITY;
        }
        float tile_max = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; i++) tile_max = fmaxf(tile_max, s[i]);
        // A row's exponentials are taken against its maximum so far, so that its largest P is exactly 1 in 16 bits: the row sum adds P
        // before they are rounded.  A tile that raises no row of the wave needs no exchange between the two lanes of a row (1 %).
        if (__builtin_amdgcn_ballot_w64(tile_max > m_i) != 0) {
            const float m_new = fmaxf(m_i, fmaxf(tile_max, __shfl_xor(tile_max, 32)));
            // (a query that has seen no key yet keeps m = -inf: every p below is then 0)
            const float alpha = m_i == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(__builtin_fmaf(m_i, a.qk_scale, -(m_new * a.qk_scale)));
            l_i *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[dt][i] *= alpha;
            m_i = m_new;
        }
        const float m_use = m_i == -INFINITY ? 0.0f : m_i * a.qk_scale;
        // ---- P, its row sum (which does not see the dropout mask), and the mask
        const uint64_t first = rng_row + (uint64_t)n0;
        const uint32_t lo = (uint32_t)first;
        // (the low words of the tile run over 28 consecutive values; once per 2^32 draws they wrap inside one)
        const bool wraps = __builtin_amdgcn_ballot_w64(lo + 27u < lo) != 0;
        if ((uint32_t)(first >> 32) != prow.hi_word) prow = philox_row((uint32_t)(first >> 32), a.seed_lo, a.seed_hi);
        vec16 pf[2];
        float psum = 0.0f;
        uint32_t pbits[8];
        // two scores and the signs of their words (bit 31 set: dropped) -> two 16-bit P
        auto put = [&](int i, int32_t sign0, int32_t sign1) {
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.qk_scale, -m_use));  // hidden keys: exp2(-inf) = 0
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i + 1], a.qk_scale, -m_use));
            psum += p0;
            psum += p1;
            typedef VT vt2 __attribute__((ext_vector_type(2)));
            // bytes of the mask: the sign of the first word twice, that of the second twice (v_perm_b32 replicates bit 31)
            const uint32_t dropped = __builtin_amdgcn_perm((uint32_t)sign1, (uint32_t)sign0, 0x0b0b0909u);
            pbits[i / 2] = __builtin_bit_cast(uint32_t, vt2{(VT)p0, (VT)p1}) & ~dropped;
        };
        if (!wraps) {
            const uint64_t product = (uint64_t)kPhiloxA * lo;
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                int32_t sign[2];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int k = 8 * ((i + e) >> 2) + ((i + e) & 3);
                    sign[e] = drop_sign(philox6_from_product(add_u64(product, (uint64_t)kPhiloxA * k), prow, a.seed_lo, a.seed_hi), a.minus_keep_from);
                }
                put(i, sign[0], sign[1]);
                __builtin_amdgcn_sched_barrier(0);  // (two scores at a time: all sixteen side by side would not fit the registers)
            }
        } else {  // every counter with a high word of its own
            uint32_t dropped = 0;
#pragma unroll 1
            for (int i = 0; i < 16; i++)
                dropped |= (dropout_keeps(first + (uint64_t)(8 * (i >> 2) + (i & 3)), a.seed_lo, a.seed_hi, a.dropout_p) ? 0u : 1u) << i;
#pragma unroll
            for (int i = 0; i < 16; i += 2) put(i, (int32_t)(dropped << (31 - i)), (int32_t)(dropped << (30 - i)));
        }
        l_i += psum;
#pragma unroll
        for (int c = 0; c < 2; c++) pf[c] = __builtin_bit_cast(vec16, v4i{(int)pbits[4 * c], (int)pbits[4 * c + 1], (int)pbits[4 * c + 2], (int)pbits[4 * c + 3]});
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                const unsigned char* p0 = vtile + vtr[dt] + 16 * c * RS;
                const s16x4 v_lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)p0);
                const s16x4 v_hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p0 + 8 * RS));
                acc[dt] = PVT::mfma(__builtin_bit_cast(vec16, __builtin_shufflevector(v_lo, v_hi, 0, 1, 2, 3, 4, 5, 6, 7)), pf[c], acc[dt]);
            }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // nothing of this workgroup is on its way into LDS when it ends

    float l_tot = l_i + __shfl_xor(l_i, 32);
    if constexpr (KG > 1) {  // the groups' shares of a row -> group 0
        static_assert(sizeof(float) * 32 * kDropWaves * D <= sizeof(smem), "one group's accumulators fit the tile buffers");
        const int slot = 32 * wave + l32;
        if (half == 0) {
            row_m[group * 32 * kDropWaves + slot] = m_i;
            row_l[group * 32 * kDropWaves + slot] = l_tot;
        }
        __syncthreads();
        float m = -INFINITY, l = 0.0f;
#pragma unroll
        for (int g = 0; g < KG; g++) m = fmaxf(m, row_m[g * 32 * kDropWaves + slot]);
        const float base = m == -INFINITY ? 0.0f : m * a.qk_scale;
#pragma unroll
        for (int g = 0; g < KG; g++)
            l += row_l[g * 32 * kDropWaves + slot] * __builtin_amdgcn_exp2f(__builtin_fmaf(row_m[g * 32 * kDropWaves + slot], a.qk_scale, -base));
        const float mine = __builtin_amdgcn_exp2f(__builtin_fmaf(m_i, a.qk_scale, -base));
        float* park = reinterpret_cast<float*>(&smem[0][0][0][0]) + wave * 32 * D + lane;  // entry e of a lane: 64 e further on
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[dt][i] *= mine;
        for (int g = 1; g < KG; g++) {
            if (group == g) {
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int i = 0; i < 16; i++) park[64 * (16 * dt + i)] = acc[dt][i];
            }
            __syncthreads();
            if (group == 0) {
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[dt][i] += park[64 * (16 * dt + i)];
            }
            __syncthreads();
        }
        if (group != 0) return;
        m_i = m;
        l_tot = l;
    }
    // l = 0: a query that saw no key: zero row.  (NaN stays, also where every NaN element of the row was dropped.)
    const float inv = l_tot != 0.0f ? a.keep_scale / l_tot : 0.0f;
    if (!row_ok) return;
    // accumulator i of tile dt: channel 32 dt + 8 (i / 4) + 4 half + i % 4 of query my_m
    const int64_t obase = (int64_t)b * a.os_b + (int64_t)h * a.os_h + (int64_t)my_m * a.os_n;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int d = 32 * dt + 8 * g + 4 * half;
            float r[4];
#pragma unroll
            for (int i = 0; i < 4; i++) r[i] = acc[dt][4 * g + i] * inv;
            if (a.out_dt == SAGE_BF16) {
                typedef __bf16 b4 __attribute__((ext_vector_type(4)));
                *reinterpret_cast<b4*>(static_cast<__bf16*>(a.out) + obase + d) = b4{(__bf16)r[0], (__bf16)r[1], (__bf16)r[2], (__bf16)r[3]};
            } else if (a.out_dt == SAGE_F16) {
                typedef _Float16 h4 __attribute__((ext_vector_type(4)));
                *reinterpret_cast<h4*>(static_cast<_Float16*>(a.out) + obase + d) = h4{(_Float16)r[0], (_Float16)r[1], (_Float16)r[2], (_Float16)r[3]};
            } else {
                *reinterpret_cast<v4f*>(static_cast<float*>(a.out) + obase + d) = v4f{r[0], r[1], r[2], r[3]};
            }
        }
    if (a.log_normalizer && half == 0)
        a.log_normalizer[((int64_t)b * a.Hq + h) * a.M + my_m] =
            l_tot != 0.0f ? (__builtin_log2f(l_tot) + m_i * a.qk_scale) * 0.693147180559945309f : -INFINITY;
}

__global__ void dropout_mask_kernel(uint8_t* mask, int64_t count, uint64_t offset, uint32_t seed_lo, uint32_t seed_hi,
                                    float dropout_p) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) mask[i] = dropout_keeps(offset + (uint64_t)i, seed_lo, seed_hi, dropout_p) ? 1 : 0;
}

// Groups of waves per workgroup: as many as the SIMDs hold waves for, where there are fewer workgroups than that takes (a
// SIMD with one wave issues a vector instruction every 5.7 cycles, with four waves every 3).  Two at most at head_dim 128, up to 256
// workgroups (three groups: B1 H4 M4096 N4096 148 -> 140 us, but B1 H8 M512 N512 25.0 -> 25.8).
int drop_groups(int64_t wgs, int head_dim) {
    int groups = 1;
    while (2 * groups <= drop_waves_per_simd(head_dim) && wgs * 2 * groups <= 256 * (drop_waves_per_simd(head_dim) & ~1)) groups *= 2;
    return groups;
}

template <int D, typename VT>
int launch_drop(DropArgs a, int64_t B, hipStream_t stream) {
    const int64_t wgs = B * a.Hq * a.nmb;
    if (wgs > 0x7fffffffLL) return fail(SAGE_E_UNSUPPORTED, "sage_flash_attn_fwd_dropout: too many query blocks for one launch");
    auto far = [](int64_t stride) { return stride < 0 || stride >= (1LL << 25); };  // 31 rows of 2-byte elements pass 2^31 bytes
    const bool wide = far(a.ks_n) || far(a.vs_n);
    const int groups = wide ? 1 : drop_groups(wgs, D);
    if (a.causal && wgs * groups <= 256 * drop_waves_per_simd(D) && a.BH < 256) a.snake = 256 / a.BH;
    dim3 grid((unsigned)wgs);
    if (wide) {
        hipLaunchKernelGGL((flash_dropout_fwd_kernel<D, VT, 1, true>), grid, dim3(kDropThreads), 0, stream, a);
        return check_launch("flash_dropout_fwd_kernel (wide rows)");
    }
    if constexpr (D == 64) {
        if (groups == 4) hipLaunchKernelGGL((flash_dropout_fwd_kernel<D, VT, 4>), grid, dim3(4 * kDropThreads), 0, stream, a);
    }
    if (groups == 2) hipLaunchKernelGGL((flash_dropout_fwd_kernel<D, VT, 2>), grid, dim3(2 * kDropThreads), 0, stream, a);
    else if (groups == 1) hipLaunchKernelGGL((flash_dropout_fwd_kernel<D, VT, 1>), grid, dim3(kDropThreads), 0, stream, a);
    return check_launch("flash_dropout_fwd_kernel");
}

}  // namespace

int launch_flash_dropout(const sage_flash_params& p, float dropout_p, uint64_t seed, uint64_t offset, hipStream_t stream) {
    DropArgs a{};
    a.q = p.q.ptr; a.k = p.k.ptr; a.v = p.v.ptr; a.out = p.out.ptr; a.log_normalizer = p.log_normalizer;
    a.qs_b = p.q.stride_b; a.qs_h = p.q.stride_h; a.qs_n = p.q.stride_n;
    a.ks_b = p.k.stride_b; a.ks_h = p.k.stride_h; a.ks_n = p.k.stride_n;
    a.vs_b = p.v.stride_b; a.vs_h = p.v.stride_h; a.vs_n = p.v.stride_n;
    a.os_b = p.out.stride_b; a.os_h = p.out.stride_h; a.os_n = p.out.stride_n;
    a.Hq = (int)p.heads_q; a.M = (int)p.qo_len; a.N = (int)p.kv_len; a.groups = (int)(p.heads_q / p.heads_kv);
    a.causal = p.causal ? 1 : 0; a.out_dt = p.out_dtype;
    a.qk_scale = p.sm_scale * 1.44269504089f;
    a.dropout_p = dropout_p;
    a.keep_scale = 1.0f / (1.0f - dropout_p);
    a.seed_lo = (uint32_t)seed; a.seed_hi = (uint32_t)(seed >> 32);
    a.offset = offset;
    // the threshold on the folded word, from the comparison it stands for: (float)word * 4.6566127342e-10f > dropout_p
    {
        int64_t lo = 0, hi = 1LL << 31;  // hi: none is kept (drop_sign is then negative for every word)
        while (lo < hi) {
            const int64_t mid = (lo + hi) / 2;
            if ((float)(int32_t)mid * 4.6566127342e-10f > dropout_p) hi = mid;
            else lo = mid + 1;
        }
        a.minus_keep_from = 0u - (uint32_t)lo;
    }
    a.BH = (int)(p.batch * p.heads_q);
    a.nmb = (a.M + 32 * kDropWaves - 1) / (32 * kDropWaves);
    if (p.head_dim == 128)
        return p.dtype == SAGE_BF16 ? launch_drop<128, __bf16>(a, p.batch, stream) : launch_drop<128, _Float16>(a, p.batch, stream);
    return p.dtype == SAGE_BF16 ? launch_drop<64, __bf16>(a, p.batch, stream) : launch_drop<64, _Float16>(a, p.batch, stream);
}

int launch_dropout_mask(uint8_t* mask, int64_t count, float dropout_p, uint64_t seed, uint64_t offset, hipStream_t stream) {
    if (count == 0) return SAGE_OK;
    const int64_t blocks = (count + 255) / 256;
    if (blocks > 0x7fffffffLL) return fail(SAGE_E_UNSUPPORTED, "sage_flash_dropout_mask: too many elements for one launch");
    hipLaunchKernelGGL(dropout_mask_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, mask, count, offset,
                       (uint32_t)seed, (uint32_t)(seed >> 32), dropout_p);
    return check_launch("dropout_mask_kernel");
}

}  // namespace sage
