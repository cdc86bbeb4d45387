// Matrix-core kernel for wide blocks (prompts, batches of requests): more than 16 tokens.
//
// Below 16 tokens a packed projection streams its weights and is bound by latency and bytes; here
// every weight is multiplied with tens to thousands of tokens, and what bounds the kernel is the issue
// of vector instructions: per scale group (128 of K) the exact int32 sums must become fp32 and meet the
// group's scale, two operations a result (eight per 16 x 16 results, against two matrix instructions),
// beside unpacking the weights and arranging the activations.  (A wave alone issues a vector instruction
// every 2.25 ns, whichever it is, two or more together one every 1.15 ns -- left shifts, byte permutations and
// three-operand integer ones every 1.9; a matrix instruction takes 13.6.)  So
//   * v_mfma_i32_32x32x32_i8: half the matrix instructions of the 16 x 16 form;
//   * weights are unpacked to 64 times their value (wide_unpack), which needs no offset term -- the
//     other forms feed -2 sum(a) through the accumulator, 8 more matrix instructions per 16 x 64 x 64 --
//     and the factor, a power of two, goes out with the division;
//   * the accumulators start from the bits of 1.5 * 2^23, so that a sum is a float and one exact
//     subtraction stands for the conversion;
//   * 64 tokens x 32 rows a wave in 128 registers, four waves a SIMD, are ahead where the rows fill the
//     chip; where they do not, 128 tokens x 32 rows, two waves a SIMD, unpack a weight once for twice the tokens.
//     They run as a pipeline (gemv_wide_kernel): waves that keep step at the barriers otherwise all read LDS, all
//     multiply and all add at the same time.  64 x 64 a wave without it before -> now: 2560 x 9728 at 3001 tokens 94 -> 87 us,
//     2560 x 4096 45 -> 41, 2560 x 9728 at 2048 91 -> 78; 12288 x 2048 at 514 (64 x 256 tiles then) 24.7 -> 23.5.
// Back to back on random bytes, activations in their own order, with 16 x 16 instructions before -> now: 19456 x 2560 at 3001 tokens
// 254 -> 194 us (1.54 POP/s; PyTorch's int8 product reaches 1.99 at 16384^3), 2560 x 9728 123 -> 87,
// 12288 x 2048 at 514 35 -> 23.5, at 256 19.6 -> 16.7, 2048 x 2048 at 256 7.1 -> 6.6.
//
//   WM x WN waves share a staged block of WM*MT*32 tokens x WN*NT*32 rows; KS such sets of waves
//   split K and add their fp32 results up in slice order (narrower blocks and few rows, where a
//   tile per workgroup would leave most CUs idle).
//
// Activations that a quantiser has left in operand order (ORDERED: a prompt's) go from memory to LDS without passing
// registers, and nothing is transposed here: once per weight row tile it was, and is once now, by the quantiser.
// Own order -> operand order, each on its own tiles, within a prompt, us: at 3001 tokens 6144 x 2560 71.6 -> 59.5, 19456 x 2560 with SiLU
// 198 -> 176.5 (1.69 POP/s), 2560 x 4096 46.2 -> 38.7, 2560 x 9728 98 -> 80 (1.87); at 256 12288 x 2048 with SiLU 18.1 -> 15.3,
// 4096 x 2048 10.1 -> 8.6, 2048 x 6144 13.8 -> 12.6, 2048 x 2048 7.1 -> 6.8.
//
// Per group a set stages 128 bytes of K for its tokens (16-byte units XORed with half the row number, so that a ds_read_b128 of
// 16 rows meets every bank once) and the packed rows (a wave's operand read is 512 or 1024 contiguous bytes).  In their own order
// activations pass registers (4 x 4 byte transposes: operand order, see gemv_core.h), and rows are inverted there where the
// unpacking wants it: the loads of group g + 2 are in flight and group g + 1 is being parked while group g is multiplied.  In
// operand order group g + 1 is on its way, with three buffers g + 2 as well, and rows are inverted behind their read.  One barrier
// per group, none where a set is a single wave.  All scales of
// the row block (G x rows, transposed), the multipliers and their reciprocals are staged once.  Rows past
// N and tokens past M read as zero through the buffer range check.
//
// Arithmetic and rounding points are those of the other kernels: exact G, fp32 scale-accumulate with
// groups in ascending order inside a slice, slices in order, division by s[m], bf16 RNE.
//
// gate|up of a prompt (`PAIRS`): a tile has gate rows and their up rows, and silu(gate) * up leaves the tile instead, 16 bytes
// a lane as before: half the bytes out, and what follows reads half (3001 tokens of the 4B shape: 191.2 us as without it,
// the activation launch behind it 32.7 -> 18.9; 256 tokens of the 1.7B one: 18.4 and 4.5 us, level).  Builds of their own: with
// a flag for it, all the others were slower, 4096 x 2048 at 128 tokens 6.59 us instead of 6.45, 2048 x 2048 at 514 10.5
// instead of 10.2, long ones level.
//
// Block numbers go round the eight XCDs, so an XCD takes a contiguous range of tiles, eight token
// tiles by consecutive row tiles: its L2 sees the same activations and the same rows again.
//
// Replaces, for these widths, the launch-per-projection path of
// src/bonsai_sft/gpu/t2g128_kernels/t2g128_kernels.cu:94-148 (any M).
#ifndef BONSAI_GEMV_WIDE_HIP_H
#define BONSAI_GEMV_WIDE_HIP_H

#include <type_traits>

#include "../../include/bonsai_gemv.h"
#include "gemv_mxl.hip.h"

namespace bonsai {

constexpr int kWideXcds = 8;
constexpr int kWideTokenGroup = 8;  // token tiles walked before the next row tile

// Weights as 64 times their value (mfma_flip), two dwords at a time: one shift of 64 bits for both (left shifts run at half the rate
// of other instructions, and this one at that of a 32-bit one; what crosses from one dword to the other is masked): 6144 x 2560 at
// 3001 ordered tokens 63.9 -> 62.9 us, 2560 x 9728 82.0 -> 81.3; at 256 12288 x 2048 14.6 -> 14.5, 4096 x 2048 7.4 -> 7.2,
// 2048 x 6144 10.4 -> 10.0.  H: which two operands, and from which dwords -- T2 2H and 2H + 1 from the dwords of those numbers,
// Q1 H and H + 2 from dwords 0 and 2.
template <int BITS, int H, typename V>
__device__ __forceinline__ void wide_unpack(const uint32_t (&p)[4], V (&vb)[4]) {
    const uint64_t q = BITS == 2 ? (uint64_t)p[2 * H + 1] << 32 | p[2 * H] : (uint64_t)p[2] << 32 | p[0];
    V &lo = vb[BITS == 2 ? 2 * H : H], &hi = vb[BITS == 2 ? 2 * H + 1 : H + 2];
    const auto place = [&](int k, uint64_t x) {
        lo[k] = (int)(BITS == 2 ? (uint32_t)x & 0xC0C0C0C0u : ((uint32_t)x & 0x80808080u) | 0x40404040u);
        hi[k] = (int)(BITS == 2 ? (uint32_t)(x >> 32) & 0xC0C0C0C0u : ((uint32_t)(x >> 32) & 0x80808080u) | 0x40404040u);
    };
    const auto shifted = [&](auto by) {
        uint64_t x = q << decltype(by)::value;
        if (decltype(by)::value != 0) asm("" : "+v"(x));  // (or the masks would let the compiler split it into two)
        return x;
    };
    constexpr int from = BITS == 2 ? 6 : (H == 0 ? 7 : 3), step = BITS == 2 ? 2 : 1;
    place(0, shifted(std::integral_constant<int, from>{}));
    place(1, shifted(std::integral_constant<int, from - step>{}));
    place(2, shifted(std::integral_constant<int, from - 2 * step>{}));
    place(3, shifted(std::integral_constant<int, from - 3 * step>{}));
}

template <int BITS, int WM, int WN, int KS, int MT, int NT>
struct WideShape {
    static constexpr int kTokens = WM * MT * 32, kRows = WN * NT * 32;
    static constexpr int kSet = 64 * WM * WN;  // threads that share a staged block
    static constexpr int kThreads = kSet * KS;
    static constexpr bool kPrivate = WM * WN == 1;  // a set is one wave: program order is enough
    static constexpr bool kPiped = KS == 1 && WM == 1 && NT == 1 && MT % 2 == 0 && MT > 2;  // (all but group sums)
    static constexpr int kBufs = kPrivate ? 1 : 2;
    static constexpr int kABytes = kTokens * 128, kBBytes = kRows * 16 * BITS;
    static constexpr int kSetBytes = kBufs * (kABytes + kBBytes);
    static constexpr bool kDeep = !kPrivate && KS > 1;  // has three buffers of ordered activations where they fit
    static constexpr int kElems = MT * NT * 16;  // results per lane
    static constexpr int kOutPitch = kRows * 2 + 16;
    static constexpr int kShare = kElems / KS;  // results per lane that a K slice finishes
    static constexpr int kRedBytes = (KS - 1) * kSet * kElems * 4;
    // scales [G][rows] u16, then multipliers and their reciprocals [tokens] (they stay), then the staged blocks, whose
    // space the K slices' partial sums and the outgoing tile take over
    static size_t lds_bytes(int K, bool deep) {
        const size_t keep = (size_t)(K / kGroup) * kRows * 2 + kTokens * 8;
        const size_t stage = (size_t)KS * (kSetBytes + (deep && kDeep ? kABytes + kBBytes : 0));
        const size_t after = kRedBytes + (size_t)kTokens * kOutPitch;
        return keep + (stage > after ? stage : after);
    }
};

// The barrier of the staging pipeline: LDS traffic of the group is done, loads for later ones stay
// in flight (a __syncthreads() would wait for them as well).
__device__ __forceinline__ void wide_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// .. and what was sent to LDS has arrived
__device__ __forceinline__ void wide_barrier_landed() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// .. but for the last N loads (or fewer: what is waited for is older than the last block, of N loads at least)
template <int N>
__device__ __forceinline__ void wide_barrier_landed_but() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// 16 bytes a lane from memory to LDS, a wave's 1 KB from `lds` on (wave-uniform)
__device__ __forceinline__ void wide_load_to_lds(__amdgpu_buffer_rsrc_t r, unsigned char *lds, uint32_t voffset, uint32_t soffset) {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16, voffset, soffset, 0, 0);
#endif
}

// ORDERED: activations in operand order, as bonsai_*_quant_ordered write them
template <int BITS, int WM, int WN, int KS, int MT, int NT, bool SF16, bool G32, bool PAIRS, bool ORDERED>
__device__ __forceinline__ void gemv_wide_tile(const int8_t *A, const uint8_t *B, void *out, const float *s, const uint16_t *ws,
                                               int M, int N, int K, int out_f32, int tiles_m, int tiles_n, int flags) {
    using S = WideShape<BITS, WM, WN, KS, MT, NT>;
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr bool kPiped = S::kPiped && !G32;
    constexpr int kAhead = S::kPrivate ? 2 : 1;  // register sets of staging loads in flight
    const int G = K >> 7;
    const int row_bytes = K * BITS / 8;

    // ---- tile of this workgroup
    const int total = tiles_m * tiles_n;
    const int per = (total + kWideXcds - 1) / kWideXcds;
    const int t = ((int)blockIdx.x & (kWideXcds - 1)) * per + ((int)blockIdx.x >> 3);
    if (t >= total) return;
    const int band = kWideTokenGroup * tiles_n;
    const int mg = t / band, rem = t - mg * band;
    const int gm = tiles_m - mg * kWideTokenGroup < kWideTokenGroup ? tiles_m - mg * kWideTokenGroup : kWideTokenGroup;
    const int tn = rem / gm;
    const int m0 = (mg * kWideTokenGroup + rem - tn * gm) * S::kTokens;
    // PAIRS: the tile's rows are kRows / 2 gate rows and, behind them, their up rows, of N / 2 each
    constexpr int kHalf = S::kRows / 2;
    const int n0 = tn * (PAIRS ? kHalf : S::kRows);
    const int mv = M - m0 < S::kTokens ? M - m0 : S::kTokens;
    const int nv = PAIRS ? (N / 2 - n0 < kHalf ? N / 2 - n0 : kHalf) : (N - n0 < S::kRows ? N - n0 : S::kRows);
    // row r of the tile as a row of what rB and rS cover (a pair's matrix whole: rows past its end repeat the last)
    const auto at_row = [&](int r) {
        if (!PAIRS) return r;
        const int p = r < kHalf ? r : r - kHalf;
        return n0 + (p < nv ? p : nv - 1) + (r < kHalf ? 0 : N / 2);
    };
    const int base_row = PAIRS ? 0 : n0, rows_there = PAIRS ? N : nv;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int set = wave / (WM * WN), wsub = wave % (WM * WN);
    const int stid = tid - set * S::kSet;
    const int wm = wsub / WN, wn = wsub % WN;
    const int op_row = lane & 31, kb = lane >> 5;

    uint16_t *scales = reinterpret_cast<uint16_t *>(smem);
    float2 *mult = reinterpret_cast<float2 *>(smem + (size_t)G * S::kRows * 2);
    unsigned char *work = reinterpret_cast<unsigned char *>(mult + S::kTokens);
    // three buffers (ORDERED): two groups are on their way while one is multiplied
    const int bufs = ORDERED && S::kDeep && (flags & 4) != 0 ? 3 : S::kBufs;
    unsigned char *abuf = work + set * (bufs * (S::kABytes + S::kBBytes));
    unsigned char *bbuf = abuf + bufs * S::kABytes;

    const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t *>(A + (size_t)m0 * K), 0, mv * K, kMxlBufferWord3);
    const __amdgpu_buffer_rsrc_t rB = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(B + (size_t)base_row * row_bytes), 0, rows_there * row_bytes, kMxlBufferWord3);

    // ---- K slice of this set (whole 512-wide tiles where K has them: the slices of gemv_mxl.hip.h)
    const int unit = (G & 3) == 0 ? 4 : 1;
    const int units = G / unit;
    const int gb = KS == 1 ? 0 : (units * set / KS) * unit;
    const int ge = KS == 1 ? G : (units * (set + 1) / KS) * unit;
    const int iters = KS == 1 ? G : ((units + KS - 1) / KS) * unit;  // of the longest slice

    // ---- staging roles
    constexpr int QB = mfma_quarter_bytes<BITS>();
    constexpr int QW = QB / 16;
    constexpr int QPR = 128 / QB;                       // quarters of a token row
    constexpr int AN_TASKS = S::kTokens * QPR;
    constexpr int AL = (AN_TASKS + S::kSet - 1) / S::kSet;  // quarters a thread stages
    constexpr int BCH = BITS;                           // 16-byte chunks of a packed row
    constexpr int BN_TASKS = S::kRows * BCH;
    constexpr int BL = (BN_TASKS + S::kSet - 1) / S::kSet;
    // Activations in operand order need no registers on their way: whole blocks go from memory to LDS, 64 units of 16 bytes a
    // wave and load, each lane reading the unit that belongs where it writes.
    static_assert(!ORDERED || !S::kPrivate, "sets of one wave have one buffer");
    constexpr int UL = S::kTokens * 8 / S::kSet;
    static_assert(UL * S::kSet == S::kTokens * 8 && UL >= AL && BN_TASKS % 64 == 0, "whole waves");
    uint32_t a_off[UL], b_off[BL];
#pragma unroll
    for (int i = 0; i < UL; ++i) {
        const int task = stid + i * S::kSet;
        a_off[i] = ORDERED
                       ? (uint32_t)(task >> 3) * (uint32_t)K + (uint32_t)((task & 7) ^ ((task >> 4) & 7)) * 16
                       : (uint32_t)(task / QPR) * (uint32_t)K + (uint32_t)((task % QPR) * QB);
    }
#pragma unroll
    for (int i = 0; i < BL; ++i) {
        const int task = stid + i * S::kSet;
        b_off[i] = (uint32_t)at_row(task / BCH) * (uint32_t)row_bytes + (uint32_t)((task % BCH) * 16);
    }
    u32x4 ars[kAhead][AL][QW], brs[kAhead][BL];
    auto load = [&](auto &ar, auto &br, int g) {
#pragma unroll
        for (int i = 0; i < AL; ++i)
            if (AN_TASKS % S::kSet == 0 || stid + i * S::kSet < AN_TASKS) {
#pragma unroll
                for (int q = 0; q < QW; ++q) ar[i][q] = mxl_load_b128(rA, a_off[i] + q * 16, (uint32_t)(g * 128));
            }
#pragma unroll
        for (int i = 0; i < BL; ++i)
            if (BN_TASKS % S::kSet == 0 || stid + i * S::kSet < BN_TASKS)
                br[i] = mxl_load_b128(rB, b_off[i], (uint32_t)(g * 16 * BITS));
    };
    auto park = [&](const auto &ar, const auto &br, int buf) {
        u32x4 *a = reinterpret_cast<u32x4 *>(abuf + buf * S::kABytes);
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            const int task = stid + i * S::kSet;
            if (AN_TASKS % S::kSet != 0 && task >= AN_TASKS) continue;
            const int row = task / QPR, q = task % QPR;
            u32x4 *dst = a + row * 8;
            const int x = (row >> 1) & 7;
            if (BITS == 2) {
                const u32x4 v = ar[i][0];
                dst[q ^ x] = transpose4x4_bytes(v.x, v.y, v.z, v.w);
            } else {
                const u32x4 lo = ar[i][0], hi = ar[i][QW - 1];
                dst[(2 * q) ^ x] = transpose4x4_bytes(lo.x, lo.z, hi.x, hi.z);
                dst[(2 * q + 1) ^ x] = transpose4x4_bytes(lo.y, lo.w, hi.y, hi.w);
            }
        }
        u32x4 *b = reinterpret_cast<u32x4 *>(bbuf + buf * S::kBBytes);
#pragma unroll
        for (int i = 0; i < BL; ++i)
            if (BN_TASKS % S::kSet == 0 || stid + i * S::kSet < BN_TASKS)
                b[stid + i * S::kSet] = u32x4{mfma_flip<BITS>(br[i].x), mfma_flip<BITS>(br[i].y), mfma_flip<BITS>(br[i].z), mfma_flip<BITS>(br[i].w)};
    };

    const auto send = [&](int g, int buf) {
#pragma unroll
        for (int i = 0; i < UL; ++i)
            wide_load_to_lds(rA, abuf + buf * S::kABytes + (i * S::kSet + wsub * 64) * 16, a_off[i], (uint32_t)(g * 128));
#pragma unroll
        for (int i = 0; i < BL; ++i)
            if (BN_TASKS % S::kSet == 0 || wsub * 64 + i * S::kSet < BN_TASKS)
                wide_load_to_lds(rB, bbuf + buf * S::kBBytes + (i * S::kSet + wsub * 64) * 16, b_off[i], (uint32_t)(g * 16 * BITS));
    };
    if (ORDERED) {
        if (gb < ge) send(gb, 0);
    } else {
        load(ars[0], brs[0], gb < ge ? gb : 0);
    }

    // ---- scales of the row block, transposed, and the multipliers
    if (!G32) {
        const __amdgpu_buffer_rsrc_t rS = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t *>(ws + (size_t)base_row * G), 0, rows_there * G * 2, kMxlBufferWord3);
        if (flags & 1) {  // whole quads of groups, aligned: a thread's quads are those of one row
            typedef unsigned int v2u __attribute__((ext_vector_type(2)));
            constexpr int kPerRow = S::kThreads / S::kRows;
            static_assert(kPerRow * S::kRows == S::kThreads, "threads divide among the rows");
            const int row = tid % S::kRows;
            for (int q = tid / S::kRows; q < G >> 2; q += kPerRow) {
                const v2u v = __builtin_amdgcn_raw_buffer_load_b64(rS, at_row(row) * (G * 2) + q * 8, 0, 0);
                uint16_t *d = scales + (q * 4) * S::kRows + row;
                d[0] = (uint16_t)v.x;
                d[S::kRows] = (uint16_t)(v.x >> 16);
                d[2 * S::kRows] = (uint16_t)v.y;
                d[3 * S::kRows] = (uint16_t)(v.y >> 16);
            }
        } else {
            for (int i = tid; i < S::kRows * G; i += S::kThreads) {
                const int row = i / G, g = i - row * G;
                scales[g * S::kRows + row] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rS, (at_row(row) * G + g) * 2, 0, 0);
            }
        }
        // (the sums come out 64 times too large, wide_unpack: so does what divides them)
        for (int i = tid; i < S::kTokens; i += S::kThreads) {
            const float d = s[m0 + (i < mv ? i : mv - 1)] * 64.0f;
            mult[i] = make_float2(d, 1.0f / d);
        }
    }

    const auto flip = [](uint32_t (&p)[4]) {  // (as parking does for the others)
#pragma unroll
        for (int t = 0; t < 4; t += BITS == 2 ? 1 : 2) p[t] = mfma_flip<BITS>(p[t]);
    };
    typedef int v16i __attribute__((ext_vector_type(16)));
    float acc[MT][NT][16];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    // The accumulators start from the bits of 1.5 * 2^23 (|G| < 2^22): the sums then ARE floats,
    // 12582912 + G, and one exact subtraction at full rate takes the place of an int-to-float conversion.
    constexpr int kBias = 0x4B400000;
    constexpr float kBiasF = 12582912.0f;
    v16i bias16;
#pragma unroll
    for (int r = 0; r < 16; ++r) bias16[r] = kBias;
    if (kPiped || ORDERED) asm volatile("" : "+v"(bias16));  // in registers for good: no copies in front of the products
    if (S::kPrivate) {
        if (kAhead > 1 && gb + 1 < ge) load(ars[kAhead - 1], brs[kAhead - 1], gb + 1);
    } else if (!ORDERED) {
        park(ars[0], brs[0], 0);
        if (gb + 1 < ge) load(ars[0], brs[0], gb + 1);
    }
    if (ORDERED) {
        wide_barrier_landed();
        if ((kPiped || (S::kDeep && bufs == 3)) && gb + 1 < ge) send(gb + 1, 1);
    } else {
        __syncthreads();
    }

    int now = 0;  // buffer of the group, of three
    const auto step = [&](int it, auto set_of) {
        constexpr int R = decltype(set_of)::value;  // register set of this group
        const int g = gb + it;
        const int buf = S::kPrivate ? 0 : (S::kDeep && ORDERED ? now : it & 1);
        if (S::kPrivate) {
            bonsai_wave::order_lds();  // group g - 1 is no longer read
            if (g < ge) park(ars[R], brs[R], 0);
            bonsai_wave::order_lds();
            if (g + kAhead < ge) load(ars[R], brs[R], g + kAhead);
        } else if (ORDERED) {
            // group g is there; group g - 1 is no longer read
            if (S::kDeep && bufs == 3 && g + 1 < ge) {
                if (it > 0) wide_barrier_landed_but<UL + (BN_TASKS % S::kSet == 0 ? BL : 0)>();
                if (g + 2 < ge) send(g + 2, now == 0 ? 2 : now - 1);
            } else {
                if (it > 0) wide_barrier_landed();
                if (bufs != 3 && g + 1 < ge) send(g + 1, buf ^ 1);
            }
            if (S::kDeep) now = now + 1 == bufs ? 0 : now + 1;
        } else {
            if (it > 0) wide_barrier();  // group g is parked; group g - 1 is no longer read
            if (g + 1 < ge) park(ars[0], brs[0], buf ^ 1);
            if (g + 2 < ge) load(ars[0], brs[0], g + 2);
        }
        if (g >= ge) return;  // (uniform in a set)
        // lane half kb takes 16-byte units 4 kb + t of the group, t the number of the matrix instruction
        const u32x4 *a = reinterpret_cast<const u32x4 *>(abuf + buf * S::kABytes) + (wm * MT * 32 + op_row) * 8;
        const unsigned char *b = bbuf + buf * S::kBBytes + (wn * NT * 32 + op_row) * (16 * BITS) + kb * (8 * BITS);
        const int x = (op_row >> 1) & 7;
        v4i vb[NT][4];
        float w[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            uint32_t p[4] = {0u, 0u, 0u, 0u};
            if (BITS == 2) {
                const u32x4 pp = *reinterpret_cast<const u32x4 *>(b + j * 32 * 16 * BITS);
                p[0] = pp.x;
                p[1] = pp.y;
                p[2] = pp.z;
                p[3] = pp.w;
            } else {
                const uint2 pp = *reinterpret_cast<const uint2 *>(b + j * 32 * 16 * BITS);
                p[0] = pp.x;
                p[2] = pp.y;
            }
            if (ORDERED) flip(p);
            w[j] = G32 ? 0.0f : scale_to_f32<SF16>(scales[g * S::kRows + (wn * NT + j) * 32 + op_row]);
            wide_unpack<BITS, 0>(p, vb[j]);
            wide_unpack<BITS, 1>(p, vb[j]);
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            v4i va[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const u32x4 u = a[i * 256 + ((4 * kb + t) ^ x)];
                va[t] = v4i{(int)u.x, (int)u.y, (int)u.z, (int)u.w};
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                v16i dd = bias16;
#pragma unroll
                for (int t = 0; t < 4; ++t) dd = __builtin_amdgcn_mfma_i32_32x32x32_i8(va[t], vb[j][t], dd, 0, 0, 0);
                if (G32) {
                    const int n = (wn * NT + j) * 32 + op_row;
                    int stride = N;
                    asm volatile("" : "+s"(stride));  // addresses made here: 16 of them held over the loop would spill
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int m = (wm * MT + i) * 32 + 8 * (r / 4) + 4 * kb + r % 4;
                        if (m < mv && n < nv)
                            reinterpret_cast<int32_t *>(out)[((size_t)(m0 + m) * stride + n0 + n) * G + g] = (dd[r] - kBias) >> 6;
                    }
                    continue;
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] += (__int_as_float(dd[r]) - kBiasF) * w[j];
            }
        }
    };
    if constexpr (kPiped) {
        // A wave's token tiles one after another, as a pipeline.  While the four products of a tile run, the sums of the tile
        // before join their results, the activations of the tile behind are on their way from LDS, and group g + 1 is parked; the
        // barrier stands in front of the last tile, which has its operands, so that the first ones of group g + 1 arrive
        // under it.  (sched_barrier and the empty asm hold the order: left alone, the compiler keeps all sums to the end.)
        v4i va[2][4], vb[4];
        v16i dd[2];
        uint32_t packed[4] = {0u, 0u, 0u, 0u};
        float w[2] = {0.0f, 0.0f};
        const int x = (op_row >> 1) & 7;
        const unsigned char *a0 = abuf + op_row * 128, *b0 = bbuf + (wn * 32 + op_row) * (16 * BITS) + kb * (8 * BITS);
        const uint16_t *sc = scales + wn * 32 + op_row;
        const auto read_a = [&](int i, int buf) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const u32x4 u = *reinterpret_cast<const u32x4 *>(a0 + buf * S::kABytes + i * 4096 + ((4 * kb + t) ^ x) * 16);
                va[i & 1][t] = v4i{(int)u.x, (int)u.y, (int)u.z, (int)u.w};
            }
        };
        const auto read_b = [&](int g, int buf, float &scale) {  // (behind the last group: what stands there, unused)
            if (BITS == 2) {
                const u32x4 p = *reinterpret_cast<const u32x4 *>(b0 + buf * S::kBBytes);
                packed[0] = p.x;
                packed[1] = p.y;
                packed[2] = p.z;
                packed[3] = p.w;
            } else {
                const uint2 p = *reinterpret_cast<const uint2 *>(b0 + buf * S::kBBytes);
                packed[0] = p.x;
                packed[2] = p.y;
            }
            if (ORDERED) flip(packed);
            scale = scale_to_f32<SF16>(sc[g * S::kRows]);
        };
        const auto join = [&](int i, float scale, int from, int to) {
#pragma unroll
            for (int r = from; r < to; ++r) {
                acc[i][0][r] += (__int_as_float(dd[i & 1][r]) - kBiasF) * scale;
                asm volatile("" : "+v"(acc[i][0][r]));
            }
        };
        const auto group = [&](int g, auto parity) {
            constexpr int P = decltype(parity)::value;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                __builtin_amdgcn_sched_barrier(0);
                if (i + 1 < MT) {
                    read_a(i + 1, P);
                } else {
                    if (ORDERED) {
                        wide_barrier_landed();  // group g + 1 is there; group g is no longer read
                        if (g + 2 < ge) send(g + 2, P);
                    } else {
                        wide_barrier();  // group g + 1 is parked; group g is no longer read
                    }
                    read_b(g + 1, P ^ 1, w[P ^ 1]);
                    read_a(0, P ^ 1);
                }
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    dd[i & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(va[i & 1][t], vb[t], t ? dd[i & 1] : bias16, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (t == 0) {
                        if (!ORDERED && i == 0 && g + 1 < ge) park(ars[0], brs[0], P ^ 1);
                        if (!ORDERED && i == 1 && g + 2 < ge) load(ars[0], brs[0], g + 2);
                    } else {
                        join(i ? i - 1 : MT - 1, w[i ? P : P ^ 1], t * 5 - 5, t == 3 ? 16 : t * 5);
                        if (i == MT - 1 && t > 1) {  // (operands that the products so far have taken)
                            if (t == 2)
                                wide_unpack<BITS, 0>(packed, vb);
                            else
                                wide_unpack<BITS, 1>(packed, vb);
#pragma unroll
                            for (int u = 0; u < 4; ++u) asm volatile("" : "+v"(vb[u]));
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        read_b(0, 0, w[0]);
        read_a(0, 0);
        wide_unpack<BITS, 0>(packed, vb);
        wide_unpack<BITS, 1>(packed, vb);
        dd[(MT - 1) & 1] = bias16;  // "group -1": nothing, at scale 0
        for (int g = 0; g < ge; g += 2) {
            group(g, std::integral_constant<int, 0>{});
            if (g + 1 < ge) group(g + 1, std::integral_constant<int, 1>{});
        }
        join(MT - 1, w[(ge - 1) & 1], 0, 16);
    } else {
        for (int it = 0; it < iters; it += kAhead) {
            step(it, std::integral_constant<int, 0>{});
            if (kAhead > 1) step(it + 1, std::integral_constant<int, kAhead - 1>{});
        }
    }
    if (G32) return;

    // ---- y / s: the reciprocal is correctly rounded and one residual step makes the quotient so
    const auto divide = [&](float y, float d, float inv) {
        const float q = y * inv;
        const float c = fmaf(fmaf(-q, d, y), inv, q);
        return c == c ? c : q;  // (infinite or NaN y)
    };
    __syncthreads();  // the staged blocks are free
    unsigned char *tile = work + S::kRedBytes;
    const auto place = [&](int i, int j, int r, int &m, int &n) {
        m = (wm * MT + i) * 32 + 8 * (r / 4) + 4 * kb + r % 4;
        n = (wn * NT + j) * 32 + op_row;
    };
    const auto finish = [&](int i, int j, int r, float y0, float y1) {  // results r, r + 1
        int m, n;
        place(i, j, r, m, n);
        const float2 d0 = mult[m], d1 = mult[m + 1];
        y0 = divide(y0, d0.x, d0.y);
        y1 = divide(y1, d1.x, d1.y);
        if (out_f32) {
            float *o = reinterpret_cast<float *>(out) + (size_t)(m0 + m) * N + n0 + n;
            if (m < mv && n < nv) o[0] = y0;
            if (m + 1 < mv && n < nv) o[N] = y1;
        } else {
            typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
            const bf2 p = {static_cast<__bf16>(y0), static_cast<__bf16>(y1)};  // round to nearest even
            uint16_t u[2];
            __builtin_memcpy(u, &p, 4);
            *reinterpret_cast<uint16_t *>(tile + m * S::kOutPitch + n * 2) = u[0];
            *reinterpret_cast<uint16_t *>(tile + (m + 1) * S::kOutPitch + n * 2) = u[1];
        }
    };
    if (KS > 1) {
        // slice z finishes the results [z * kShare, ..) of every lane and takes the other slices'
        // values of them, slot by slot, from red[z]
        static_assert(S::kShare * KS == S::kElems, "results divide among the slices");
        float *red = reinterpret_cast<float *>(work) + stid;
        const auto slot = [&](int dst, int src, int k) -> float & {
            return red[((dst * (KS - 1) + (src < dst ? src : src - 1)) * S::kShare + k) * S::kSet];
        };
#pragma unroll
        for (int z = 0; z < KS; ++z)
            if (z != set) {
#pragma unroll
                for (int k = 0; k < S::kShare; ++k) {
                    const int e = z * S::kShare + k;
                    slot(z, set, k) = acc[e / (NT * 16)][e / 16 % NT][e % 16];
                }
            }
        __syncthreads();
#pragma unroll
        for (int z = 0; z < KS; ++z)
            if (z == set) {
#pragma unroll
                for (int k = 0; k < S::kShare; k += 2) {
                    float y[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int e = z * S::kShare + k + h;
                        const float own = acc[e / (NT * 16)][e / 16 % NT][e % 16];
                        y[h] = z == 0 ? own : slot(z, 0, k + h);
#pragma unroll
                        for (int src = 1; src < KS; ++src) y[h] += src == z ? own : slot(z, src, k + h);
                    }
                    const int e = z * S::kShare + k;
                    finish(e / (NT * 16), e / 16 % NT, e % 16, y[0], y[1]);
                }
            }
    } else {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 16; r += 2) finish(i, j, r, acc[i][j][r], acc[i][j][r + 1]);
    }
    if (out_f32) return;
    __syncthreads();
    // ---- the tile leaves in 16-byte pieces of whole rows
    uint16_t *o = reinterpret_cast<uint16_t *>(out);
    if constexpr (PAIRS) {   // .. as bf16(bf16(silu(gate)) * up)
        constexpr int kPairs = kHalf / 8;
        for (int i = tid; i < S::kTokens * kPairs; i += S::kThreads) {
            const int m = i / kPairs, c = (i % kPairs) * 8;
            if (m >= mv || c >= nv) continue;
            const uint16_t *gate = reinterpret_cast<const uint16_t *>(tile + m * S::kOutPitch) + c, *up = gate + kHalf;
            const u32x4 g = *reinterpret_cast<const u32x4 *>(gate), u = *reinterpret_cast<const u32x4 *>(up);
            const auto two = [](uint32_t x, uint32_t y) {   // (the products are rounded already)
                const float lo = silu_mul_bf16(__uint_as_float(x << 16), __uint_as_float(y << 16));
                const float hi = silu_mul_bf16(__uint_as_float(x & 0xffff0000u), __uint_as_float(y & 0xffff0000u));
                return (__float_as_uint(lo) >> 16) | (__float_as_uint(hi) & 0xffff0000u);
            };
            const u32x4 r = u32x4{two(g.x, u.x), two(g.y, u.y), two(g.z, u.z), two(g.w, u.w)};
            *reinterpret_cast<u32x4 *>(o + (size_t)(m0 + m) * (N / 2) + n0 + c) = r;
        }
        return;
    }
    constexpr int CPR = S::kRows / 8;
    for (int i = tid; i < S::kTokens * CPR; i += S::kThreads) {
        const int m = i / CPR, c = (i % CPR) * 8;
        if (m >= mv || c >= nv) continue;
        const unsigned char *src = tile + m * S::kOutPitch + c * 2;
        uint16_t *dst = o + (size_t)(m0 + m) * N + n0 + c;
        if (flags & 2) {  // N a multiple of 8, rows 16-byte aligned
            *reinterpret_cast<u32x4 *>(dst) = *reinterpret_cast<const u32x4 *>(src);
        } else {
            for (int k = 0; k < 8 && c + k < nv; ++k) dst[k] = reinterpret_cast<const uint16_t *>(src)[k];
        }
    }
}

template <int BITS, int WM, int WN, int KS, int MT, int NT, bool SF16, bool G32, bool PAIRS>
__global__ void __launch_bounds__(64 * WM * WN * KS) __attribute__((amdgpu_waves_per_eu(MT * NT >= 4 || WM * WN == 1 ? 2 : 4)))
gemv_wide_kernel(const int8_t *A, const uint8_t *B, void *out, const float *s, const uint16_t *ws, int M,
                 int N, int K, int out_f32, int tiles_m, int tiles_n, int flags) {
    gemv_wide_tile<BITS, WM, WN, KS, MT, NT, SF16, G32, PAIRS, false>(A, B, out, s, ws, M, N, K, out_f32, tiles_m, tiles_n, flags);
}

// (six waves a SIMD where a wave has one tile: three workgroups a CU.  4096 x 2048 at 256 tokens level, 6144 x 2560 at 3001
// 117 -> 99 us.  In the kernel above, with its staging registers, that spills: 8.1 -> 9.1.)
template <int BITS, int WM, int WN, int KS, int MT, int NT, bool PAIRS>
__global__ void __launch_bounds__(64 * WM * WN * KS) __attribute__((amdgpu_waves_per_eu(MT * NT >= 4 || WM * WN == 1 ? 2 : (MT * NT == 1 ? 6 : 4))))
gemv_wide_ordered_kernel(const int8_t *A, const uint8_t *B, void *out, const float *s, const uint16_t *ws, int M,
                         int N, int K, int out_f32, int tiles_m, int tiles_n, int flags) {
    gemv_wide_tile<BITS, WM, WN, KS, MT, NT, false, false, PAIRS, true>(A, B, out, s, ws, M, N, K, out_f32, tiles_m, tiles_n, flags);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
using WideKernelFn = void (*)(const int8_t *, const uint8_t *, void *, const float *, const uint16_t *, int, int,
                              int, int, int, int, int);

struct WideVariant {
    WideKernelFn fn[4];  // bf16 scales, fp16 scales, group sums, pairs (bf16 scales); on ordered activations the first and the last
    int tokens, rows, threads;
    size_t (*lds)(int K, bool deep);
    bool deep;
    int t[5];  // template arguments, for the launch record
};

template <int BITS, int WM, int WN, int KS, int MT, int NT>
constexpr WideVariant wide_variant() {
    using S = WideShape<BITS, WM, WN, KS, MT, NT>;
    return WideVariant{{gemv_wide_kernel<BITS, WM, WN, KS, MT, NT, false, false, false>,
                        gemv_wide_kernel<BITS, WM, WN, KS, MT, NT, true, false, false>,
                        gemv_wide_kernel<BITS, WM, WN, KS, MT, NT, false, true, false>,
                        gemv_wide_kernel<BITS, WM, WN, KS, MT, NT, false, false, true>},
                       S::kTokens, S::kRows, S::kThreads, S::lds_bytes, S::kDeep, {WM, WN, KS, MT, NT}};
}

template <int WM, int WN, int KS, int MT, int NT>
constexpr WideVariant wide_ordered_variant() {
    using S = WideShape<2, WM, WN, KS, MT, NT>;
    return WideVariant{{gemv_wide_ordered_kernel<2, WM, WN, KS, MT, NT, false>, nullptr, nullptr,
                        gemv_wide_ordered_kernel<2, WM, WN, KS, MT, NT, true>},
                       S::kTokens, S::kRows, S::kThreads, S::lds_bytes, S::kDeep, {WM, WN, KS, MT, NT}};
}

// (tokens x rows of a workgroup, K slices)
enum : int { WIDE_64x256 = 0, WIDE_64x128_K2, WIDE_32x64_K4, WIDE_32x64_K8, WIDE_64x128_K4, WIDE_128x256, kWideVariants };

template <int BITS>
const WideVariant &wide_kernel(int v) {
    static const WideVariant t[kWideVariants] = {wide_variant<BITS, 1, 8, 1, 2, 1>(), wide_variant<BITS, 1, 4, 2, 2, 1>(),
                                                 wide_variant<BITS, 1, 2, 4, 1, 1>(), wide_variant<BITS, 1, 1, 8, 1, 2>(),
                                                 wide_variant<BITS, 1, 4, 4, 2, 1>(), wide_variant<BITS, 1, 8, 1, 4, 1>()};
    return t[v];
}

// On ordered activations (T2 alone: half the weight bytes leave Q1 little to gain, 0.3 % over 131 sizes; T2 9 %): without staging
// registers and instructions smaller tiles are ahead, and these six stand for all (over 267 sizes 0.6 % behind the best of
// nine in the mean, 10 % at most; the six above, by their estimates, 3.4 % and 22 %; without the last one 1.2 % and 20 %).
enum : int { ORDERED_32x64_K4 = 0, ORDERED_128x256, ORDERED_64x64_K2, ORDERED_64x128, ORDERED_64x64_K4, ORDERED_64x128_K4, kOrderedVariants };

inline const WideVariant &wide_kernel_ordered(int v) {
    static const WideVariant t[kOrderedVariants] = {wide_ordered_variant<1, 2, 4, 1, 1>(), wide_ordered_variant<1, 8, 1, 4, 1>(),
                                                    wide_ordered_variant<1, 2, 2, 2, 1>(), wide_ordered_variant<1, 4, 1, 2, 1>(),
                                                    wide_ordered_variant<1, 2, 4, 2, 1>(), wide_ordered_variant<1, 4, 4, 2, 1>()};
    return t[v];
}

template <int BITS>
const WideVariant &wide_of(int v, bool ordered) {
    if constexpr (BITS == 2)
        if (ordered) return wide_kernel_ordered(v);
    return wide_kernel<BITS>(v);
}

template <int BITS>
int wide_init_device(int max_lds) {
    const auto init = [&](const WideVariant &k) {
        for (WideKernelFn fn : k.fn)
            if (fn != nullptr && hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     max_lds) != hipSuccess)
                return false;
        return true;
    };
    for (int v = 0; v < kWideVariants; ++v)
        if (!init(wide_kernel<BITS>(v))) return 2;
    if constexpr (BITS == 2)
        for (int v = 0; v < kOrderedVariants; ++v)
            if (!init(wide_kernel_ordered(v))) return 2;
    return 0;
}

// What a launch takes, in microseconds: a fixed part, the scale groups of a K slice times the length of one
// -- bound by latency up to some tiles per CU, then by what they issue -- and a part per tile for its scales
// and its results.  Fitted to 17 ... 4096 tokens of 13 matrices (1024 x 1024 ... 20000 x 9728), then moved for
// the choice between them.  Over 220 drawn blocks with weights from HBM each is off by 13-18 % rms, mostly by a
// part that all share (9-16 % low).
// Those on ordered activations are fitted to 267 sizes from 17 to 3500 tokens and moved, by a tenth at most, for the choice (7-8 %
// rms where they are near the best).
inline double wide_estimate(int v, int M, int N, int K, int n_cus, bool ordered = false) {
    struct Cost {
        int tokens, rows, slices;
        double fixed, group_min, group_tile, tile;
    };
    static constexpr Cost o[kOrderedVariants] = {{32, 64, 4, 2.993, 0.581, 0.424, 0.468}, {128, 256, 1, 2.101, 0.737, 0.846, 7.022},
                                                 {64, 64, 2, 3.2, 0.539, 0.314, 0.827},   {64, 128, 1, 5.267, 0.422, 0.263, 0.599},
                                                 {64, 64, 4, 1.752, 0.784, 0.833, 1.975}, {64, 128, 4, 1.026, 1.161, 1.141, 3.872}};
    static constexpr Cost c[kWideVariants] = {{64, 256, 1, 3.7, 0.752, 0.571, 1.47},   {64, 128, 2, 2.94, 0.882, 0.577, 1.565},
                                              {32, 64, 4, 3.27, 0.595, 0.498, 0.554},  {32, 64, 8, 1.87, 0.791, 0.889, 2.54},
                                              {64, 128, 4, 1.5, 1.25, 1.25, 3.0},      {128, 256, 1, 2.0, 0.88, 1.03, 6.0}};
    const Cost &k = ordered ? o[v] : c[v];
    const int G = K / kGroup, unit = G % 4 == 0 ? 4 : 1;
    const int groups = (G / unit + k.slices - 1) / k.slices * unit;
    const long tiles = (long)((M + k.tokens - 1) / k.tokens) * ((N + k.rows - 1) / k.rows);
    const double per_cu = (double)((tiles + n_cus - 1) / n_cus);
    const double busy = k.group_tile * per_cu;
    return k.fixed + groups * (busy > k.group_min ? busy : k.group_min) + k.tile * per_cu;
}

// Whether variant v takes rows of K weights: all scales of its row block are staged at once, 2 bytes per row and group,
// so that 64x128_K4 and 128x256 stop at K = 23,808, 64x256 at 32,384 and 64x128_K2 at 56,576 (160 KB of LDS; the other tiles of
// ordered activations take all rows that there are), and its offsets are 32-bit.
template <int BITS>
bool wide_fits(int v, int K, int lds_limit, bool ordered = false) {
    const WideVariant &k = wide_of<BITS>(v, ordered);
    if (ordered && K > BONSAI_ORDERED_MAX_K) return false;  // (no quantiser writes such rows)
    return k.lds(K, false) <= (size_t)lds_limit && (long)k.rows * K <= (1L << 30) && (long)k.tokens * K <= (1L << 30);
}

// The variant with the smallest estimate among those that take rows of K weights: over 220 drawn blocks 0.8 % behind
// the best of them in the mean, within 0.8 % on nine in ten, 21 % at most (16586 x 2560 of sign weights at 89 tokens:
// 64x128_K2 for 32x64_K4).  -1: none does.
template <int BITS>
int wide_pick(int M, int N, int K, int n_cus, int lds_limit, bool ordered = false) {
    int best = -1;
    for (int v = 0; v < (ordered ? kOrderedVariants : kWideVariants); ++v)
        if (wide_fits<BITS>(v, K, lds_limit, ordered) &&
            (best < 0 || wide_estimate(v, M, N, K, n_cus, ordered) < wide_estimate(best, M, N, K, n_cus, ordered)))
            best = v;
    return best;
}

// Launches one problem as variant v; -1 when it does not fit (the caller falls back).  ask: the answer alone, 0 or -1
template <int BITS>
int launch_wide(int v, const GemvProblem &q, int out_kind, int scale_kind, int lds_limit, hipStream_t stream, bool pairs = false,
                bool ordered = false, bool ask = false, int n_cus = 0) {
    const WideVariant &k = wide_of<BITS>(v, ordered);
    if (!wide_fits<BITS>(v, q.K, lds_limit, ordered)) return -1;
    // pairs: N / 2 gate rows, N / 2 up rows -> silu(gate) * up, 16-byte pieces of whole rows; one resource over all of B
    if (pairs && (out_kind != OUT_BF16 || scale_kind != 0 || q.N % 16 != 0 || (reinterpret_cast<uintptr_t>(q.out) & 15) != 0 ||
                  (long)q.N * q.K * BITS / 8 > (1L << 30)))
        return -1;
    const int tile_rows = pairs ? k.rows / 2 : k.rows, all_rows = pairs ? q.N / 2 : q.N;
    const int tm = (q.M + k.tokens - 1) / k.tokens, tn = (all_rows + tile_rows - 1) / tile_rows;
    if ((long)tm * tn > (1L << 28)) return -1;
    if (ask) return 0;
    const int per = (tm * tn + kWideXcds - 1) / kWideXcds;
    const int flags = ((q.K / kGroup) % 4 == 0 && (reinterpret_cast<uintptr_t>(q.ws) & 7) == 0 ? 1 : 0) |
                      (q.N % 8 == 0 && (reinterpret_cast<uintptr_t>(q.out) & 15) == 0 ? 2 : 0);
    // Weights from HBM and activations that another die has written take longer than a group: three buffers where no second
    // workgroup on the CU fills the wait.  256 tokens within a prompt, us, two -> three: 2048 x 6144 (256 tiles) 13.0 -> 11.2, 2048 x 2048
    // level; 4096 x 2048 (512 tiles) 8.7 -> 9.0, gate|up 12288 x 2048 (384 tiles) 16.1 -> 16.4.
    const size_t three = k.lds(q.K, true);
    const bool deep = ordered && k.deep && tm * tn <= n_cus && three <= (size_t)lds_limit;
    const int variant = pairs ? 3 : (out_kind == OUT_G32 ? 2 : scale_kind);
    hipLaunchKernelGGL(k.fn[variant], dim3(per * kWideXcds, 1, 1), dim3(k.threads, 1, 1), deep ? three : k.lds(q.K, false), stream, q.A, q.B, q.out,
                       q.s, reinterpret_cast<const uint16_t *>(q.ws), q.M, q.N, q.K, out_kind == OUT_F32 ? 1 : 0, tm,
                       tn, flags | (deep ? 4 : 0));
    note_kernel(ordered ? "gemv_wide_ordered_kernel" : "gemv_wide_kernel", BITS, k.t[0], k.t[1], k.t[2], k.t[3], k.t[4], variant);
    return hipGetLastError() == hipSuccess ? 0 : 2;
}

}  // namespace bonsai
#endif  // BONSAI_GEMV_WIDE_HIP_H
