// Attention forward for few query rows against many keys (decoding, speculative tokens), gfx950: int8 Q and K with
// block scales (SageAttention) and 16-bit Q and K (dense attention).
//
// Bound by the bytes of K and V: a K/V head is read once for ALL query rows that share it.  The rows of a call that
// belong to one K/V head, qo_len rows of each of its `groups` query heads, are packed into one or two 32-row tiles
// (row r = head r / qo_len of the group, query r % qo_len), where the kernel of attn_fast_kernel.h spends a 256-row
// tile, and a walk over K and V of its own, on every query head.
//
// * A workgroup is eight waves (four with two row tiles), and a wave walks over 32-key tiles of its own (tile w, w + 8,
//   ... of the workgroup's keys) with no barrier: S^T = K.Q^T and O^T += V^T.P^T on the 32x32 matrix instructions, so a lane owns one query
//   row.  Matrix and vector work of a tile is a small part of the time its 12-16 KB take to arrive.
// * K rows are loaded straight into the A operand; V goes through registers into the wave's own slice of LDS, from
//   where ds_read_b64_tr_b16 returns the transposed operand (chunks XOR-swizzled as in attn_fast_kernel.h).  The
//   registers of a tile are requested anew as soon as their contents have been consumed: eight waves on a CU keep up
//   to 128 KB in flight, about six times bandwidth x latency of its share of the HBM.
//   Measured (bf16, head_dim 128, with the combine launch; before: the 256-row tiles of the pipelined kernel): dense
//   B8 H32/8 M1 N8192 197 -> 46 us = 5.8 TB/s of K and V (a 1 GiB copy moves 5.2 TB/s here), SageAttention on the same
//   shape 144 -> 37 us = 5.4 TB/s, dense B64 H32/8 M1 N1024 229 -> 42 us = 6.4 TB/s.
// * Short calls with more rows (plan_row_tiles) come here too, a workgroup per 32 packed rows: what counts there is the time of
//   one workgroup.  The waves' results meet in LDS in one go where eight waves share it (32 channels at a time before: B1 H8
//   N256 D128 int8 9.0 -> 8.2 us, N64 6.7 -> 5.9).
// * The keys of a (batch, K/V head) are cut into runs (plan_decode_split) so that every CU holds eight waves; the
//   waves of a workgroup are combined through LDS, the runs by split_combine_kernel.
#include "attn_common.h"

namespace sage {
namespace attn {
namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;

constexpr int kTileKeys = 32;

template <int D>
__device__ __forceinline__ int v_swizzle(int row) { return D == 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1); }

// RT: 32-row tiles of packed query rows (groups * qo_len) per workgroup
// kDecodeWaves: eight (one workgroup per CU), or four: with one row tile where the items alone fill the chip (two
// workgroups per CU, finer rounds: B11 H32/32 M1 N700 D128 26 us against 32 us), and with two row tiles, which leave
// registers for one wave per SIMD only.
template <int D, typename VT, int QB, int RT, int kDecodeWaves>
__global__ __launch_bounds__(64 * kDecodeWaves, RT == 1 ? 8 / kDecodeWaves : 1) void attn_decode_kernel(AttnArgs a) {
    using PVT = PV<VT>;
    using vec16 = typename PVT::vec;
    constexpr bool INT8 = QB == 1;
    constexpr int KSTEPS = D * QB / 32;   // matrix instructions of a 32 x 32 score tile: 32 bytes of a row each
    constexpr int DT = D / 32;
    constexpr int V_RS = 2 * D;           // bytes per V row in LDS
    constexpr int VCPR = V_RS / 16;       // 16-byte chunks per V row
    constexpr int VLOADS = kTileKeys * VCPR / 64;
    constexpr int V_TILE = kTileKeys * V_RS;
    constexpr int CH = kDecodeWaves == 8 ? D : 32;  // channels of the waves' results that meet in LDS at a time
    constexpr int SL_RS = CH + 4;         // floats per row of the combine buffer
    constexpr int SLICE = kDecodeWaves * 32 * SL_RS * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[kDecodeWaves * V_TILE > SLICE ? kDecodeWaves * V_TILE : SLICE];
    __shared__ float row_m[kDecodeWaves][32 * RT], row_l[kDecodeWaves][32 * RT];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the runs, then the row tiles, of one (batch, K/V head) are neighbours in the grid
    const int rows = a.groups * a.M, row_tiles = (rows + 32 * RT - 1) / (32 * RT);
    const int split = blockIdx.x % a.nsplit;
    const int row0 = blockIdx.x / a.nsplit % row_tiles * (32 * RT);  // first row of the workgroup
    const int item = blockIdx.x / a.nsplit / row_tiles;
    const int hk = item % a.Hkv, b = item / a.Hkv;
    // queries of the workgroup's rows: from q_lo to q_hi, all of a head's where the rows belong to several heads
    const int q_first = row0 % a.M, in_head = min(a.M - q_first, rows - row0);
    const bool one_head = in_head >= min(32 * RT, rows - row0);
    const int q_lo = one_head ? q_first : 0, q_hi = one_head ? min(q_first + 32 * RT, a.M) - 1 : a.M - 1;
    const int kbeg = split * a.split_steps * BN;
    const int kend = min(kbeg + a.split_steps * BN, a.causal ? min(q_hi + a.N - a.M + 1, a.N) : a.N);  // (0 or less: no row sees a key)

    // this lane's query rows
    v4i qf[RT][KSTEPS];
    int lim[RT];       // last key the row sees
    float qs[RT];      // scale of the row's scores (int8: still to be multiplied by the K block's)
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        const int r = row0 + 32 * rt + l32;
        const bool ok = r < rows;  // (rows past the last one multiply a copy of the group's first: nothing of theirs is stored)
        const int g = ok ? r / a.M : 0, mi = ok ? r - g * a.M : 0, h = hk * a.groups + g;
        const int8_t* qp = a.q + ((int64_t)b * a.qs_b + (int64_t)h * a.qs_h + (int64_t)mi * a.qs_n) * QB + 16 * half;
#pragma unroll
        for (int t = 0; t < KSTEPS; t++) qf[rt][t] = *reinterpret_cast<const v4i*>(qp + 32 * t);
        lim[rt] = ok && a.causal ? min(mi + a.N - a.M, a.N - 1) : a.N - 1;
        qs[rt] = INT8 ? a.q_scale[((int64_t)b * a.Hq + h) * a.nq + mi / BM] : a.qk_scale;
    }
    // keys below this one are visible to every row of the workgroup
    const int all_see = a.causal ? min(q_lo + a.N - a.M + 1, a.N) : a.N;
    // (constant address space: scalar loads, which the waits for K and V do not count)
    typedef __attribute__((address_space(4))) const float* const_f32_ptr;
    const const_f32_ptr ksp = (const_f32_ptr)(uintptr_t)(INT8 ? a.k_scale + ((int64_t)b * a.Hkv + hk) * a.nk : nullptr);

    const unsigned char* kg = reinterpret_cast<const unsigned char*>(a.k) + ((int64_t)b * a.ks_b + (int64_t)hk * a.ks_h) * QB;
    const unsigned char* vg = static_cast<const unsigned char*>(a.v) + ((int64_t)b * a.vs_b + (int64_t)hk * a.vs_h) * 2;
    const int64_t krow = a.ks_n * QB, vrow = a.vs_n * 2;  // bytes from one key to the next
    const int vr0 = lane / VCPR, vchunk = lane % VCPR;    // V load e of a lane: row vr0 + e * 64 / VCPR, this chunk
    unsigned char* vlds = smem + wave * V_TILE;

    v4i kf[KSTEPS], vr[VLOADS];
    // Rows past the last key re-read it (finite values under hidden scores).  The loads of a tile are unconditional and
    // without branches, so that the waits for older loads leave them in flight.
    auto load_k = [&](int key0) {
        const unsigned char* p = kg + (int64_t)key0 * krow;
        const unsigned off = (unsigned)(min(l32, a.N - 1 - key0) * (int)krow + 16 * half);
#pragma unroll
        for (int t = 0; t < KSTEPS; t++) kf[t] = *reinterpret_cast<const v4i*>(p + off + 32 * t);
    };
    auto load_v = [&](int key0) {
        const unsigned char* p = vg + (int64_t)key0 * vrow;
        const int last = a.N - 1 - key0;
#pragma unroll
        for (int e = 0; e < VLOADS; e++)
            vr[e] = *reinterpret_cast<const v4i*>(p + (unsigned)(min(vr0 + e * (64 / VCPR), last) * (int)vrow + 16 * vchunk));
    };
    int vtr[DT];  // LDS offsets of the transposed fragment reads (see attn_fast_kernel.h)
    {
        const int s4 = (lane >> 2) & 3, a4 = lane & 3, g1 = (lane >> 4) & 1;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
            vtr[dt] = (4 * half + s4) * V_RS + 16 * ((4 * dt + 2 * g1 + (a4 >> 1)) ^ v_swizzle<D>(s4)) + 8 * (a4 & 1);
    }

    float m_i[RT], l_i[RT];
    v16f o[RT][DT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        m_i[rt] = -INFINITY;
        l_i[rt] = 0.0f;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int i = 0; i < 16; i++) o[rt][dt][i] = 0.0f;
    }

    int key0 = kbeg + kTileKeys * wave;
    if (key0 < kend) {
        load_k(key0);
        load_v(key0);
    }
    for (; key0 < kend; key0 += kTileKeys * kDecodeWaves) {
        const int next = key0 + kTileKeys * kDecodeWaves;
        const int fetch = next < kend ? next : key0;  // (behind the last tile: the same lines once more)
        // ---- S^T = K.Q^T; the K registers are requested anew right behind it
        v16i s[RT];
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
#pragma unroll
            for (int i = 0; i < 16; i++) s[rt][i] = 0;
#pragma unroll
            for (int t = 0; t < KSTEPS; t++) {
                if constexpr (INT8) s[rt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[t], qf[rt][t], s[rt], 0, 0, 0);
                else s[rt] = __builtin_bit_cast(v16i, PVT::mfma(__builtin_bit_cast(vec16, kf[t]), __builtin_bit_cast(vec16, qf[rt][t]),
                                                                __builtin_bit_cast(v16f, s[rt])));
            }
        }
        load_k(fetch);
        __builtin_amdgcn_sched_barrier(0);
        // ---- V tile -> LDS (the wave's own slice: a wave's LDS instructions run in order, no barrier)
#pragma unroll
        for (int e = 0; e < VLOADS; e++) {
            const int row = vr0 + e * (64 / VCPR);
            *reinterpret_cast<v4i*>(vlds + row * V_RS + 16 * (vchunk ^ v_swizzle<D>(row))) = vr[e];
        }
        load_v(fetch);
        __builtin_amdgcn_sched_barrier(0);
        // ---- online softmax: register i of this lane is key key0 + 8 (i / 4) + 4 half + i % 4 of its row
        const float ks = INT8 ? ksp[key0 / BN] : 1.0f;
        const bool hides = key0 + kTileKeys > all_see || key0 + kTileKeys > kend;
        vec16 pf[RT][2];
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const float sc = qs[rt] * ks;
            const int last = min(lim[rt], kend - 1);
            float x[16];
            float mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int bits = s[rt][i];
                x[i] = (INT8 ? (float)bits : __builtin_bit_cast(float, bits)) * sc;
                if (hides) x[i] = key0 + 8 * (i >> 2) + 4 * half + (i & 3) <= last ? x[i] : -INFINITY;
                mx = fmaxf(mx, x[i]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float m_new = fmaxf(m_i[rt], mx);
            const float m_use = m_new == -INFINITY ? 0.0f : m_new;  // (no key seen yet: every P below is exp2(-inf) = 0)
            if (__builtin_amdgcn_ballot_w64(m_new > m_i[rt]) != 0) {
                const float alpha = __builtin_amdgcn_exp2f(m_i[rt] - m_use);  // 0 for a row without a reference point
                l_i[rt] *= alpha;
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int i = 0; i < 16; i++) o[rt][dt][i] *= alpha;
                m_i[rt] = m_new;
            }
            float lsum = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; i++) pf[rt][i >> 3][i & 7] = (VT)__builtin_amdgcn_exp2f(x[i] - m_use);
#pragma unroll
            for (int c = 0; c < 8; c++) lsum = PVT::dot2_ones(pf[rt][c >> 2], c & 3, lsum);
            l_i[rt] += lsum;
        }
        // ---- O^T += V^T.P^T
#pragma unroll
        for (int tp = 0; tp < 2; tp++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                const unsigned char* p0 = vlds + vtr[dt] + 16 * tp * V_RS;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)p0);
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p0 + 8 * V_RS));
                const vec16 vf = __builtin_bit_cast(vec16, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
                for (int rt = 0; rt < RT; rt++) o[rt][dt] = PVT::mfma(vf, pf[rt][tp], o[rt][dt]);
            }
    }

    // ---- the waves of the workgroup -> one normalized result and its log-sum-exp
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        const float l_tot = l_i[rt] + __shfl_xor(l_i[rt], 32);
        if (half == 0) {
            row_m[wave][32 * rt + l32] = m_i[rt];
            row_l[wave][32 * rt + l32] = l_tot;
        }
    }
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        if (row0 + 32 * rt >= rows) break;
        const int r = 32 * rt + l32;  // (within the workgroup)
        float m = -INFINITY, l = 0.0f;
#pragma unroll
        for (int w = 0; w < kDecodeWaves; w++) m = fmaxf(m, row_m[w][r]);
        const float m_use = m == -INFINITY ? 0.0f : m;
#pragma unroll
        for (int w = 0; w < kDecodeWaves; w++) l += row_l[w][r] * __builtin_amdgcn_exp2f(row_m[w][r] - m_use);
        // l = 0: a row that saw no key; its output is 0, its log-sum-exp -inf
        const float f = l > 0.0f ? __builtin_amdgcn_exp2f(m_i[rt] - m_use) / l : 0.0f;
        if (a.lse && wave == 0 && half == 0 && row0 + r < rows) {
            const int g = (row0 + r) / a.M, mi = row0 + r - g * a.M;
            const int64_t row = ((int64_t)b * a.Hq + hk * a.groups + g) * a.M + mi;
            a.lse[row + split * a.lse_split_stride] = lse_out(__builtin_log2f(l) + m, a.lse_mul, a.lse_shift, a.lse_shift_mul, row);
        }
        // CH channels of every wave's rows at a time through LDS: all of them where a wave slice fits, else 32
        float* slice = reinterpret_cast<float*>(smem);
#pragma unroll
        for (int d0 = 0; d0 < D; d0 += CH) {
            __syncthreads();  // the V tiles / the previous channels have been read
#pragma unroll
            for (int dt = 0; dt < CH / 32; dt++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const v16f& x = o[rt][d0 / 32 + dt];
                    *reinterpret_cast<v4f*>(slice + (wave * 32 + l32) * SL_RS + 32 * dt + 8 * g + 4 * half) =
                        v4f{x[4 * g] * f, x[4 * g + 1] * f, x[4 * g + 2] * f, x[4 * g + 3] * f};
                }
            __syncthreads();
            constexpr int GROUPS = CH / 4;  // groups of four channels per row
#pragma unroll
            for (int e = 0; e < (32 * GROUPS + 64 * kDecodeWaves - 1) / (64 * kDecodeWaves); e++) {
                const int piece = tid + 64 * kDecodeWaves * e;
                const int orow = row0 + 32 * rt + piece / GROUPS, c = 4 * (piece % GROUPS);
                if (piece >= 32 * GROUPS || orow >= rows) continue;
                v4f sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int w = 0; w < kDecodeWaves; w++) {
                    const v4f x = *reinterpret_cast<const v4f*>(slice + (w * 32 + piece / GROUPS) * SL_RS + c);
#pragma unroll
                    for (int i = 0; i < 4; i++) sum[i] += x[i];
                }
                const int g = orow / a.M, mi = orow - g * a.M;
                const int64_t off = (int64_t)b * a.os_b + (int64_t)(hk * a.groups + g) * a.os_h + (int64_t)mi * a.os_n +
                                    split * a.out_split_stride + d0 + c;
                if (a.out_dt == SAGE_BF16) {
                    typedef __bf16 b4 __attribute__((ext_vector_type(4)));
                    *reinterpret_cast<b4*>(static_cast<__bf16*>(a.out) + off) = b4{(__bf16)sum[0], (__bf16)sum[1], (__bf16)sum[2], (__bf16)sum[3]};
                } else if (a.out_dt == SAGE_F16) {
                    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
                    *reinterpret_cast<h4*>(static_cast<_Float16*>(a.out) + off) = h4{(_Float16)sum[0], (_Float16)sum[1], (_Float16)sum[2], (_Float16)sum[3]};
                } else {
                    *reinterpret_cast<v4f*>(static_cast<float*>(a.out) + off) = sum;
                }
            }
        }
    }
}

template <int D, typename VT, int QB>
int launch_rt(const AttnArgs& a, int64_t batch, hipStream_t stream) {
    const int64_t rows = (int64_t)a.groups * a.M;
    const bool two = rows > 32 && rows <= kDecodeRows && a.groups > 1;  // two row tiles per workgroup
    const int64_t wgs = batch * a.Hkv * a.nsplit * (two ? 1 : (rows + 31) / 32);
    if (wgs > 0x7fffffffLL) return fail(SAGE_E_UNSUPPORTED, "attention over few query rows: too many workgroups for one launch");
    dim3 grid((unsigned)wgs);
    if (two) hipLaunchKernelGGL((attn_decode_kernel<D, VT, QB, 2, 4>), grid, dim3(256), 0, stream, a);
    else if (a.nsplit == 1 && wgs > 256) hipLaunchKernelGGL((attn_decode_kernel<D, VT, QB, 1, 4>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((attn_decode_kernel<D, VT, QB, 1, 8>), grid, dim3(512), 0, stream, a);
    return check_launch("attn_decode_kernel");
}

template <int D, typename VT>
int launch_qb(const AttnArgs& a, int64_t batch, bool int8, hipStream_t stream) {
    return int8 ? launch_rt<D, VT, 1>(a, batch, stream) : launch_rt<D, VT, 2>(a, batch, stream);
}

}  // namespace

int launch_decode(const AttnArgs& a, int64_t batch, int head_dim, int v_dtype, bool int8, hipStream_t stream) {
    if (head_dim == 128)
        return v_dtype == SAGE_BF16 ? launch_qb<128, __bf16>(a, batch, int8, stream) : launch_qb<128, _Float16>(a, batch, int8, stream);
    return v_dtype == SAGE_BF16 ? launch_qb<64, __bf16>(a, batch, int8, stream) : launch_qb<64, _Float16>(a, batch, int8, stream);
}

}  // namespace attn
}  // namespace sage
