// Attention of a block of prompt rows over the history and themselves (causal), on the matrix cores.
//
// The decode step's chunk pass (attn_mfma_kernel) serves up to 32 rows: 16 (row, query head) pairs per
// workgroup, partial results through memory.  A prompt has rows enough to keep the chip busy without
// splitting the history, so here a workgroup of four waves owns 128 pairs of one kv head for good --
// 128 / heads-per-group consecutive rows with all their query heads, 32 pairs a wave -- and walks the
// 64-slot chunks they see; nothing is merged.
//
//   S^T = K Q^T   2 x 8 v_mfma_f32_32x32x16_bf16: a lane owns ONE query (column) and half of the
//                 chunk's slots, so the softmax is in-lane but for one exchange of the maximum with
//                 lane + 32; the running sum stays a half per lane until the end
//   O^T += V^T P^T   4 x 4 more: the slots a lane half holds after S^T (4 h + 0..3 of every eight) are
//                 the slots its B operand takes, so P goes from the softmax registers straight into the
//                 matrix core (rounded to bf16 as everywhere); V^T is read with the same slot order
//
// K rows are staged as they are (pitch 272 bytes: 32 rows at one column meet every bank once), V
// transposed 4 slots x 8 dims at a time in registers (16 v_perm per thread and chunk; pitch 136).  Two
// buffers of each, shared by the four waves, which is what bounds the LDS traffic.  Keys run a chunk ahead of values:
// chunk c + 1's scores are multiplied in front of chunk c's softmax, so that a wave's matrix instructions run beside its
// exponentials; keys c + 2 and values c + 1 are parked meanwhile and the loads of the ones after them are in flight.
// 3001 rows of 32 query heads: 105 us with each chunk in turn (matrix cores and vector ALU busy for a third of the cycles:
// two waves a SIMD that meet at a barrier every chunk do not cover a wave's chain scores -> maximum -> exponentials ->
// product), 96 so, 0.78 PFLOP/s over the slots seen.  (Half the scores beside the maximum and half beside the exponentials:
// 97; the order of the two kinds of instructions prescribed: 103.)
//
// Longest rows first, but the second workgroup of each CU the other way round: the longest rows' CUs get the shorter ones of that
// batch beside them (us, all longest first -> so: 32 heads, 2048 rows 58.0 -> 54.4, 3001 level, 4096 171 -> 161; 16 heads, 3001
// 76.7 -> 74.0, 4096 106 -> 99.6; every other batch the other way round 4096 165).  The kv head is the low part of the block number, so that with eight of them an
// XCD's L2 holds one head's history.
// Reference: the prompt forward's causal attention, src/bonsai_sft/gpu/model.py:996-1005 with the mask
// of fast_generate.py:949-953.
#ifndef BONSAI_PREFILL_ATTN_HIP_H
#define BONSAI_PREFILL_ATTN_HIP_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wave_reduce.h"

namespace bonsai_prefill {

constexpr int kHead = 128;
constexpr int kSlots = 64;             // slots of a chunk
constexpr int kWaves = 4;
constexpr int kPairs = 32 * kWaves;    // (row, query head) pairs of a workgroup
constexpr int kKPitch = 2 * kHead + 16;
constexpr int kVPitch = 2 * kSlots + 8;
constexpr int kKBytes = kSlots * kKPitch, kVBytes = kHead * kVPitch;
constexpr int kLds = 2 * (kKBytes + kVBytes);
constexpr int kRawBuffer = 0x00020000;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32v4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8 frag(u32v4 v) {
    bf16x8 r;
    __builtin_memcpy(&r, &v, 16);
    return r;
}

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    const bf16x2 p = {(__bf16)a, (__bf16)b};
    uint32_t u;
    __builtin_memcpy(&u, &p, 4);
    return u;
}

// What a workgroup of `tokens` consecutive rows, the last of them m0 + tokens - 1 at most, sees and where its lanes' pairs sit.
struct Rows {
    int m0, seen, chunks, masked_from;
    __device__ __forceinline__ Rows(int tile, int tokens, int M, int base) {
        m0 = tile * tokens;
        seen = base + (M - m0 < tokens ? M : m0 + tokens);  // slots the last row sees
        chunks = (seen + kSlots - 1) / kSlots;
        masked_from = (base + m0 + 1) / kSlots;             // from here on some row does not see all slots
    }
};

// Which of `tiles` tiles, longest first, comes at place `i`: places batch .. 2 batch - 1 the other way round.
__device__ __forceinline__ int turn_of(int i, int tiles, int batch) {
    if (i < batch || i >= 2 * batch) return i;
    return batch + (tiles < 2 * batch ? tiles : 2 * batch) - 1 - i;
}

// A lane's pair: (row, query head) number `pair` of the workgroup; pairs without a row repeat the block's last one.
struct Pair {
    u32v4 q[8];   // its query, dims 16 j + 8 h + 0..7
    int pos;      // the last slot it sees
    size_t row;   // element its output row starts at
    bool valid;
    __device__ __forceinline__ Pair(const uint16_t *qs, int pair, int h, int m0, int tokens, int M, int base, int n_heads,
                                    int hpg, int kvh) {
        const int tok = pair / hpg, g = pair - tok * hpg;
        valid = tok < tokens && m0 + tok < M;
        const int m = valid ? m0 + tok : M - 1;
        pos = base + m;
        row = (size_t)m * n_heads * kHead + (size_t)(kvh * hpg + g) * kHead;
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = *reinterpret_cast<const u32v4 *>(qs + row + 16 * j + 8 * h);
    }
};

// The running softmax of a lane's query: o[d][r] is dim 32 d + 8 (r / 4) + 4 h + r % 4, l the sum of the lane's half of
// the slots, both against the maximum m.
struct Softmax {
    f32x16 o[4];
    float m, l;
    __device__ __forceinline__ Softmax() : m(-INFINITY), l(0.0f) {
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
    }
};

// A block of 4 slots x 8 dims of V, transposed: 8 stores of 4 slots each.
__device__ __forceinline__ void park_v(unsigned char *vb, const u32v4 (&v)[4], int dim, int slot) {
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        const uint32_t sel = d & 1 ? 0x07060302u : 0x05040100u;
        uint2 t;
        t.x = __builtin_amdgcn_perm(v[1][d / 2], v[0][d / 2], sel);
        t.y = __builtin_amdgcn_perm(v[3][d / 2], v[2][d / 2], sel);
        *reinterpret_cast<uint2 *>(vb + (dim + d) * kVPitch + slot * 2) = t;
    }
}

// Scores of a chunk's keys, parked at kb: s[t][r] is slot 32 t + 8 (r / 4) + 4 h + r % 4 of it.
__device__ __forceinline__ void scores(const unsigned char *kb, const Pair &p, int col, int h, f32x16 (&s)[2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[t][r] = 0.0f;
        const unsigned char *kp = kb + (32 * t + col) * kKPitch + 16 * h;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(*reinterpret_cast<const u32v4 *>(kp + 32 * j)),
                                                           frag(p.q[j]), s[t], 0, 0, 0);
    }
}
// Chunk c with its scores and its values, parked at vb, into the running softmax of a wave's 32 queries.
__device__ __forceinline__ void take(f32x16 (&s)[2], const unsigned char *vb, const Pair &p, int c, int masked_from, int col,
                                     int h, float scale_log2e, Softmax &x) {
    if (c >= masked_from) {
        const int rel = p.pos - c * kSlots - 4 * h;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (32 * t + 8 * (r / 4) + r % 4 > rel) s[t][r] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[t][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(x.m, mx * scale_log2e);
    // A row may have met nothing but -inf so far: a wave that does not start at slot 0 can see nothing of its first
    // chunk, and scores themselves can be -inf.  Its exponentials are then 0 against any finite maximum.
    const float shift = m_new == -INFINITY ? 0.0f : m_new;
    if (__any(m_new > x.m)) {
        const float alpha = __builtin_amdgcn_exp2f(x.m - shift);
        x.l *= alpha;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) x.o[d][r] *= alpha;
        x.m = m_new;
    }
    uint32_t e[2][8];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const float a = __builtin_amdgcn_exp2f(fmaf(s[t][2 * r], scale_log2e, -shift));
            const float b = __builtin_amdgcn_exp2f(fmaf(s[t][2 * r + 1], scale_log2e, -shift));
            e[t][r] = pack_bf16(a, b);
            bf16x2 pv;
            __builtin_memcpy(&pv, &e[t][r], 4);
            const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};
            x.l = __builtin_amdgcn_fdot2_f32_bf16(pv, ones, x.l, false);
        }
    // K-step ks takes slots 16 ks + 4 h + 0..3 and 16 ks + 8 + 4 h + 0..3 of each lane half
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const uint32_t *pp = e[ks / 2] + 4 * (ks & 1);
        const bf16x8 pf = frag(u32v4{pp[0], pp[1], pp[2], pp[3]});
        const unsigned char *vp = vb + col * kVPitch + (16 * ks + 4 * h) * 2;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const uint2 lo = *reinterpret_cast<const uint2 *>(vp + 32 * d * kVPitch);
            const uint2 hi = *reinterpret_cast<const uint2 *>(vp + 32 * d * kVPitch + 16);
            x.o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(u32v4{lo.x, lo.y, hi.x, hi.y}), pf, x.o[d], 0, 0, 0);
        }
    }
}

// A kv head's K or V, slots from `seen` on read as zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t history(const uint16_t *layer, int kvh, int slots, int seen) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(layer + (size_t)kvh * slots * kHead), 0, seen * 2 * kHead,
                                             kRawBuffer);
}

__global__ void __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
prefill_attn_kernel(const uint16_t *q, const uint16_t *k_layer, const uint16_t *v_layer, uint16_t *out,
                    float scale_log2e, int M, int n_heads, int n_kv, int hpg, int slots, int base, int tokens,
                    int tiles, int batch) {
    __shared__ __align__(16) unsigned char smem[kLds];
    const int kvh = (int)blockIdx.x % n_kv;
    const Rows w(tiles - 1 - turn_of((int)blockIdx.x / n_kv, tiles, batch), tokens, M, base);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, h = lane >> 5;
    const Pair p(q, wave * 32 + col, h, w.m0, tokens, M, base, n_heads, hpg, kvh);
    const __amdgpu_buffer_rsrc_t rK = history(k_layer, kvh, slots, w.seen), rV = history(v_layer, kvh, slots, w.seen);

    const int k_slot = tid >> 4, k_col = tid & 15;           // K: 16-byte column of slots k_slot + 16 i
    const int v_slot = (tid & 15) * 4, v_dim = (tid >> 4) * 8;  // V: a block of 4 slots x 8 dims
    const int k_off = k_slot * 2 * kHead + k_col * 16;
    const int v_off = v_slot * 2 * kHead + v_dim * 2;
    u32v4 kr[4], vr[4];
    const auto load_k = [&](int c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) kr[i] = __builtin_amdgcn_raw_buffer_load_b128(rK, k_off + i * 16 * 2 * kHead, c * kSlots * 2 * kHead, 0);
    };
    const auto load_v = [&](int c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) vr[i] = __builtin_amdgcn_raw_buffer_load_b128(rV, v_off + i * 2 * kHead, c * kSlots * 2 * kHead, 0);
    };
    unsigned char *const kbs = smem, *const vbs = smem + 2 * kKBytes;
    const auto park_k = [&](int c) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<u32v4 *>(kbs + (c & 1) * kKBytes + (k_slot + 16 * i) * kKPitch + k_col * 16) = kr[i];
    };
    const auto park = [&](int c) { park_v(vbs + (c & 1) * kVBytes, vr, v_dim, v_slot); };
    // (loads for later chunks stay in flight)
    const auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // Keys are a chunk ahead of values: chunk c + 1's scores are multiplied while chunk c's softmax is computed.
    Softmax x;
    f32x16 s[2];
    load_k(0);
    load_v(0);
    park_k(0);
    park(0);
    if (w.chunks > 1) load_k(1);
    meet();
    scores(kbs, p, col, h, s);
    if (w.chunks > 1) {
        park_k(1);
        load_v(1);
    }
    if (w.chunks > 2) load_k(2);
    for (int c = 0; c < w.chunks; ++c) {
        // keys c + 1 and values c are parked; keys c and values c - 1 are no longer read
        meet();
        if (c + 1 < w.chunks) park(c + 1);
        if (c + 2 < w.chunks) {
            park_k(c + 2);
            load_v(c + 2);
        }
        if (c + 3 < w.chunks) load_k(c + 3);
        f32x16 ahead[2];
        scores(kbs + ((c + 1) & 1) * kKBytes, p, col, h, ahead);   // (behind the last chunk: of what lies there, not used)
        take(s, vbs + (c & 1) * kVBytes, p, c, w.masked_from, col, h, scale_log2e, x);
#pragma unroll
        for (int t = 0; t < 2; ++t) s[t] = ahead[t];
    }

    const float l = x.l + __shfl_xor(x.l, 32);
    if (!p.valid) return;
    const float inv = 1.0f / l;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint2 v;
            v.x = pack_bf16(x.o[d][4 * k] * inv, x.o[d][4 * k + 1] * inv);
            v.y = pack_bf16(x.o[d][4 * k + 2] * inv, x.o[d][4 * k + 3] * inv);
            *reinterpret_cast<uint2 *>(out + p.row + 32 * d + 8 * k + 4 * h) = v;
        }
}

// Few rows: the kernel above has 128 pairs a workgroup, which leaves most CUs idle (256 rows of two query heads a
// kv head: 32 workgroups) and one workgroup walks all chunks.  Here the four waves of a workgroup share 32 pairs
// and take every fourth chunk each, staged by the wave for itself (program order instead of barriers); the four
// results meet in LDS.  Same operations; the softmax's running maxima are those of a wave's own chunks.
constexpr int kSplitStage = kKBytes + kVBytes;
constexpr int kSplitLds = kWaves * kSplitStage;
static_assert(kWaves * 64 * 64 * 4 + kWaves * 64 * 8 <= kSplitLds, "the merge reuses the staging areas");

__global__ void __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(1)))
prefill_attn_split_kernel(const uint16_t *q, const uint16_t *k_layer, const uint16_t *v_layer, uint16_t *out,
                          float scale_log2e, int M, int n_heads, int n_kv, int hpg, int slots, int base, int tokens,
                          int tiles, int) {
    __shared__ __align__(16) unsigned char smem[kSplitLds];
    const int kvh = (int)blockIdx.x % n_kv;
    const Rows rows(tiles - 1 - (int)blockIdx.x / n_kv, tokens, M, base);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int col = lane & 31, h = lane >> 5;
    const Pair p(q, col, h, rows.m0, tokens, M, base, n_heads, hpg, kvh);
    const __amdgpu_buffer_rsrc_t rK = history(k_layer, kvh, slots, rows.seen), rV = history(v_layer, kvh, slots, rows.seen);
    unsigned char *kb = smem + wave * kSplitStage, *vb = kb + kKBytes;
    const int k_slot = lane >> 4, k_col = lane & 15;            // slots k_slot + 4 i
    const int v_slot = (lane & 15) * 4, v_dim = (lane >> 4) * 8;  // dims v_dim + 32 i
    u32v4 kr[16], vr[4][4];
    const auto load = [&](int c) {
        const int s = c * kSlots * 2 * kHead;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            kr[i] = __builtin_amdgcn_raw_buffer_load_b128(rK, (k_slot + 4 * i) * 2 * kHead + k_col * 16, s, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                vr[i][t] = __builtin_amdgcn_raw_buffer_load_b128(rV, (v_slot + t) * 2 * kHead + (v_dim + 32 * i) * 2, s, 0);
    };

    Softmax x;
    if (wave < rows.chunks) load(wave);
    for (int c = wave; c < rows.chunks; c += kWaves) {
        bonsai_wave::order_lds();  // the chunk before is no longer read
#pragma unroll
        for (int i = 0; i < 16; ++i) *reinterpret_cast<u32v4 *>(kb + (k_slot + 4 * i) * kKPitch + k_col * 16) = kr[i];
#pragma unroll
        for (int i = 0; i < 4; ++i) park_v(vb, vr[i], v_dim + 32 * i, v_slot);
        bonsai_wave::order_lds();
        if (c + kWaves < rows.chunks) load(c + kWaves);
        f32x16 s[2];
        scores(kb, p, col, h, s);
        take(s, vb, p, c, rows.masked_from, col, h, scale_log2e, x);
    }

    // ---- the waves' results: [wave][register][lane], maxima and sums behind them
    __syncthreads();
    float *meet = reinterpret_cast<float *>(smem);
    float *stat = meet + kWaves * 64 * 64;  // [wave][maximum, sum][lane]
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) meet[(wave * 64 + d * 16 + r) * 64 + lane] = x.o[d][r];
    stat[wave * 128 + lane] = x.m;
    stat[wave * 128 + 64 + lane] = x.l;
    __syncthreads();
    float top = -INFINITY, l = 0.0f, e[kWaves];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) top = fmaxf(top, stat[w * 128 + lane]);
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        e[w] = __builtin_amdgcn_exp2f(stat[w * 128 + lane] - top);
        l = fmaf(e[w], stat[w * 128 + 64 + lane], l);
    }
    l += __shfl_xor(l, 32);
    if (!p.valid) return;
    const float inv = 1.0f / l;
    // wave d finishes dims 32 d + 8 (r / 4) + 4 h + r % 4
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float sum = 0.0f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) sum = fmaf(e[w], meet[(w * 64 + wave * 16 + 4 * k + i) * 64 + lane], sum);
            v[i] = sum * inv;
        }
        *reinterpret_cast<uint2 *>(out + p.row + 32 * wave + 8 * k + 4 * h) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
    }
}

}  // namespace bonsai_prefill
#endif  // BONSAI_PREFILL_ATTN_HIP_H
