// All layers of a one-token decode step in one launch (`bonsai_decode_step_one`).
//
// A one-token step is a chain of small operations.  With a launch for each (five a layer, the projections with their
// element-wise neighbours folded in) a 1.7B-shaped layer took 23.5 us, of which reading its weights is 2.7 us: the rest is
// launches (1.6 us for an empty one), waves starting, and first loads that nothing could request earlier.  Here one
// workgroup per compute unit stays for the whole step and owns a fixed share of the output rows of every projection:
//   * weights are requested most of a layer ahead, into registers (a unit's share of a layer is 52 KB with the 1.7B
//     shape, 105 KB with the 4B one), and only while no row is on its way: what shares the memory system with a
//     hand-over delays it (1 us each);
//   * a row goes from one phase to the next through memory, without a barrier: the producer stores it past its L2 (sc1),
//     the consumer reads it past its own until every dword has arrived.  Measured between 256 workgroups: 1.0 to 1.2 us
//     for 2048 to 9728 values, 1.9 where everybody polls from the start, 1.5 where a workgroup's values go out in several
//     stores (a line that is being polled has to be taken out of eight L2s for each of them), hence one store a workgroup
//     and a pause before the first poll;
//   * q|k|v's rows are dealt out by kv head, so that the hand-over to the attention, and of its parts, stays within a die's
//     L2 (near_heads): 0.2 us instead of 0.6 between two workgroups.  With the pauses that fit it the 1.7B shape takes 379 /
//     432 / 483 us at a history of 24 / 300 / 1500 (before: 386 / 455 / 517), the 4B one 698 / 771 / 871 (720 / 803 / 902).  At 300
//     slots, us without both / near alone / the pauses alone / both: 451 / 448 / 439 / 426 and 814 / 811 / 773 / 764;
//   * what needs a value of the whole row (the norm's sum of squares, the maximum the quantisation scales by) is computed
//     by every workgroup from the row it has read anyway.
// What bounds it now is the length of the chain: per phase a hand-over, about 0.8 us for norm and quantisation, 0.5 us
// from the row in LDS to the results.
//
// Two kinds of waves.  Four front waves, one a SIMD, receive rows, norm and quantise them into LDS and attend; twelve back
// waves hold the weights and multiply, so that waiting for a row (loads return in order) never waits for weights.
//
// Phases of a layer, each ending in a hand-over:
//     q|k|v (norm, quantise)  ->  attention  [-> merge of its parts]  ->  o (quantise, add)  ->  gate|up (norm, quantise,
//     SiLU * up)  ->  down (quantise, add)
//
// Exchange memory.  Rows are bf16 and a dword that has not arrived holds 0xffffffff, which no producer stores (two
// NaNs of that pattern become 0x7fff7fff): every dword vouches for itself, so neither ordering nor the width of a store
// matters.  There are two sets of rows; a launch uses one and refills its own part of the other with that pattern as it
// goes, which is safe because the readers of the other set belong to the launch before.  The set is picked by a counter
// in the exchange memory that workgroup 0 advances at its end (every workgroup that takes part has read it by then: the
// last phases depend on all of them, given two layers).  Parts of the attention carry a tag instead (step and layer).
//
// Waits are bounded.  A workgroup that waits longer than kStartTicks in the first layer (the launch did not get all of
// its compute units) or kRunTicks later leaves, marks the exchange memory so that workgroups that start late leave at
// once, and sets *status.  A step writes nothing but its workspace slot, its exchange memory and its output row, so it
// can be repeated: the launch behind this one does so where it finds the mark (step_finish.hip.h).
//
// Arithmetic: operations and rounding points of the stand-alone producers; group sums exact (see Codes), scaled and summed
// in fp32 over K: two or four groups a unit, then the units of a row.  The attention keeps its probabilities in fp32.
#ifndef BONSAI_STEP_ONE_HIP_H
#define BONSAI_STEP_ONE_HIP_H

namespace step_one {

constexpr int kFrontWaves = 4, kBackWaves = 12;
constexpr int kFront = kFrontWaves * 64, kBack = kBackWaves * 64, kThreads = kFront + kBack;
constexpr uint32_t kEmpty = 0xffffffffu;
constexpr int kMaxSplits = 32;             // attention parts per head
constexpr int kSingle = 128;               // slots one workgroup takes alone: up to here no parts to merge
constexpr int kRounds = 2;                 // rounds of eight slots a wave requests ahead
constexpr int kPartEntries = kHd + 4;      // 8-byte entries of a part: 128 sums, maximum, sum, pad
constexpr uint32_t kStartTicks = 500000;   // 5 ms of the 100 MHz counter
constexpr uint32_t kRunTicks = 20000000;   // 200 ms
// s_sleep(1) steps (27 ns each) before the first look.  One that comes too early costs a look, about 1 us with those of 255
// others on their way, and delays what it looks for; one that comes too late costs what it is late by.  By sweep, us a step at a
// history of 24 / 300 / 900, from 8 (10 for the attention's row and the down projection's) everywhere: gate|up's row 12 steps and
// the down projection's 18 382 / 439 / 458 -> 377 / 431 / 438 (1.7B shape), 729 / 802 / 854 -> 705 / 779 / 830 (4B); q|k|v's row
// 12 level and 698 / 772 / 825, 16 1 % behind and 692 / 766 / 817; two more or fewer of any: within 1 %.  They are numbers that
// fit these two shapes: how long others take depends on every row, and only the norm's pause follows one.  On two other shapes each
// of them is within 1 % of the best at any of those histories (1024 x 3072 352 / 404 / 407, 2304 x 6400 542 / 594 / 636; from 8 and 10
// everywhere 361 / 422 / 433 and 547 / 606 / 649).
constexpr int kPauseHead = 4, kPauseParts = 2;   // near hand-overs
constexpr int kPauseAtt = 10, kPauseH2 = 12, kPauseInner = 18;
__host__ __device__ constexpr int pause_row(int words) { return 8 + 4 * words; }   // words a lane of a row of dim
constexpr int kBufFlags = 0x00020000;
constexpr int kOob = 0x7ffffff0;           // an offset no buffer reaches: loads give 0, stores are dropped

struct Layer {
    const uint8_t *w[4];    // q|k|v, o, gate|up, down
    const uint16_t *s[4];   // their group scales (bf16)
    const uint16_t *ln1, *ln2, *qn, *kn;
};

struct Args {
    const Layer *layers;
    const uint16_t *embed;
    const int32_t *step_in;   // cache_len, hide, row mask, position, token
    uint16_t *kv;             // [2, n_layers, n_kv, slots, 128]
    const uint16_t *cos_t, *sin_t;
    uint8_t *exchange;
    uint16_t *h_out;          // bf16 [dim]: the residual stream behind the last layer
    int32_t *status;
    int n_layers, dim, ffn, n_heads, n_kv, slots, sigma, max_pos, vocab, groups;
    float eps, scale;
    uint32_t first_wait, later_wait;   // ticks, in the first layer and in the others
};

// ---- sizes --------------------------------------------------------------------------------
// A projection's share of a workgroup is cut into units of 16 rows x 64 bytes of each (256 ternary or 512 sign
// weights): one 16-byte load a lane.  Unit i of the share (row tile i / units, stretch of K i % units) belongs to back
// wave i % 12.
__host__ __device__ constexpr int unit_k(int bits) { return 512 / bits; }
struct Share {
    int units, rows, count;   // stretches of K; rows of a workgroup, whole pairs of values; units of a workgroup
    __host__ __device__ Share(int k, int n, int groups, int bits, bool pairs) {
        units = k / unit_k(bits);
        const int values = pairs ? n / 2 : n;
        rows = 2 * ((values + 2 * groups - 1) / (2 * groups));
        if (pairs) rows *= 2;
        count = (rows + 15) / 16 * units;
    }
    __host__ __device__ int loads() const { return (count + kBackWaves - 1) / kBackWaves; }
    __host__ __device__ int pitch() const { return (units + 3) & ~3; }   // floats a row of the results
    __host__ __device__ int results() const { return (rows + 15) / 16 * 16 * pitch(); }
};

// q|k|v's rows in the order of the kv heads: a head's queries, its key, its value.  A kv head's rows are computed and attended
// to by the same workgroups, those whose number is the head's modulo n_kv.
struct HeadOrder {
    int n_heads, n_kv, gqa;
    __host__ __device__ int rows() const { return (gqa + 2) * kHd; }   // of a kv head
    __device__ int row_of(int kvh, int i) const {                     // its i-th one, as a row of the matrix
        const int which = (uint32_t)i / kHd;
        return (which < gqa ? kvh * gqa + which : n_heads + (which - gqa) * n_kv + kvh) * kHd + (int)((uint32_t)i % kHd);
    }
};

__host__ __device__ inline int align128(int bytes) { return (bytes + 127) & ~127; }
struct Rows {   // byte offsets of a layer's rows in a set
    int qkv, att, h2, inner, size;
    __host__ __device__ Rows(int dim, int ffn, int n_heads, int n_kv) {
        qkv = align128(2 * dim);
        att = qkv + align128(2 * kHd * (n_heads + 2 * n_kv));
        h2 = att + align128(2 * kHd * n_heads);
        inner = h2 + align128(2 * dim);
        size = inner + align128(2 * ffn);
    }
};
constexpr int kControlBytes = 256;
// Control words beside those of step_finish.hip.h, which leaves these: whether the workgroups of a kv head share a die, and the
// dies of the workgroups with the same number modulo eight, a bit each.
enum { kDiesShared = 16, kDieOf = 24, kDies = 8 };

// LDS: planes of the row (two bytes a value), its group sums, results of all units, raw row of the down projection
struct Lds {
    int sums, red, raw, size;
    __host__ __device__ Lds(int k_max, int results_max, int ffn) {
        sums = 2 * k_max + 64;                 // (64 zero bytes behind the planes)
        red = sums + k_max / 128 * 4;
        red = (red + 63) & ~63;
        raw = red + results_max * 4;
        size = raw + 2 * ffn;
    }
};

// ---- device pieces ------------------------------------------------------------------------
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, kBufFlags);
}

typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

// What is computed from the value is computed here again: kept over the layers, the addresses of all loads and stores
// would take more registers than there are.
__device__ __forceinline__ int afresh(int x) {
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ int afresh_scalar(int x) {
    x = __builtin_amdgcn_readfirstlane(x);
    asm volatile("" : "+s"(x));
    return x;
}

// An offset that gives nothing where it is not wanted.  (Left to itself the compiler makes two loads of it, in a branch
// each, and has the second one wait for everything the first could have asked for.)
__device__ __forceinline__ int wanted(bool ok, int offset) { return afresh(ok ? offset : kOob); }

// The value of lane ^ 8, ^ 16, ^ 32 and sums and maxima over such pairs, without a trip through LDS.
constexpr int kRor8 = 0x128;
__device__ __forceinline__ float from_xor8(float v) { return bonsai_wave::partner<kRor8>(v); }
struct Pair {
    float a, b;   // the two lanes of a pair, the lower one first, in both of them
};
__device__ __forceinline__ Pair pair16(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return Pair{__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ Pair pair32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return Pair{__uint_as_float(r[0]), __uint_as_float(r[1])};
}

// Maximum of non-negative values and sum over sixteen lanes; the lane moves are part of the operations.
template <int CTRL>
__device__ __forceinline__ float max_step(float v) {
    const uint32_t x = __float_as_uint(v);
    const uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
    return __uint_as_float(x > y ? x : y);
}
template <int CTRL>
__device__ __forceinline__ float sum_step(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum_of_16(float v) {
    v = sum_step<bonsai_wave::kXor1>(v);
    v = sum_step<bonsai_wave::kXor2>(v);
    v = sum_step<bonsai_wave::kHalfMirror>(v);
    return sum_step<bonsai_wave::kMirror>(v);
}
__device__ __forceinline__ float top_of_64(float v) {
    v = max_step<bonsai_wave::kXor1>(v);
    v = max_step<bonsai_wave::kXor2>(v);
    v = max_step<bonsai_wave::kHalfMirror>(v);
    v = max_step<bonsai_wave::kMirror>(v);
    Pair p = pair16(v);
    p = pair32(fmaxf(p.a, p.b));
    return fmaxf(p.a, p.b);
}

// The value K lanes on within sixteen (0 past the end).
template <int K>
__device__ __forceinline__ float lanes_on(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + K, 0xf, 0xf, true));
}

// ---- hand-over ----------------------------------------------------------------------------
__device__ __forceinline__ int first_spin(uint32_t limit) { return limit ? 1 : 64; }   // (0: does not wait at all)
__device__ __forceinline__ bool timed_out(int spins, uint32_t &since, uint32_t limit) {
    if (spins & 63) return false;
    const uint32_t now = (uint32_t)wall_clock64() | 1u;
    if (since == 0) since = now;
    return now - since >= limit;
}

// A row of `words` 16-byte words at `from`: word tid + 256 i into v[i] (zero past the end), once all of them have arrived.
template <int U>
__device__ __forceinline__ bool receive(const __amdgpu_buffer_rsrc_t r, int from, int words, v4u *v, int pause, uint32_t limit) {
    const int tid = afresh((int)threadIdx.x);
    for (int z = 0; z < pause; ++z) __builtin_amdgcn_s_sleep(1);
    uint32_t since = 0;
    for (int spins = first_spin(limit);; ++spins) {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < U; ++i)
            v[i] = __builtin_amdgcn_raw_buffer_load_b128(r, wanted(tid + i * kFront < words, (tid + i * kFront) * 16), from, kDeviceScope);
#pragma unroll
        for (int i = 0; i < U; ++i)
            ok = ok & (v[i].x != kEmpty) & (v[i].y != kEmpty) & (v[i].z != kEmpty) & (v[i].w != kEmpty);
        if (__all(ok)) return true;
        if (timed_out(spins, since, limit)) return false;
        __builtin_amdgcn_s_sleep(1);
    }
}

// Two neighbouring values of a row.  A workgroup's values go out in one instruction: a line that others poll is taken
// out of eight L2s for every store that reaches it.
__device__ __forceinline__ void hand_over(const __amdgpu_buffer_rsrc_t set, int row, int off, uint32_t d) {
    d = d == kEmpty ? 0x7fff7fffu : d;
    __builtin_amdgcn_raw_buffer_store_b32(d, set, off, row, kDeviceScope);
}
// What only workgroups of the same die wait for stays in its L2: from one workgroup to another 0.21 us instead of 0.57 to
// another die (0.38 on the same one past the L2).  `near`: see near_heads.
__device__ __forceinline__ void hand_over_near(const __amdgpu_buffer_rsrc_t set, int row, int off, uint32_t d, bool near) {
    d = d == kEmpty ? 0x7fff7fffu : d;
    if (near)
        __builtin_amdgcn_raw_buffer_store_b32(d, set, off, row, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b32(d, set, off, row, kDeviceScope);
}
// Workgroups go round the dies in the order of their numbers, so that those of a kv head (n_kv a multiple of eight) share
// one.  The exchange memory's reset has looked whether they do (dies_kernel).  A workgroup that is not where it was then
// stores past its L2, which all see; what the others leave in theirs it does not see, and a step in which it would have to
// ends at its limit and is done again (step_finish.hip.h).
__device__ __forceinline__ bool near_heads(const __attribute__((address_space(4))) uint32_t *control, int wg) {
    uint32_t die;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(die));
    return control[kDiesShared] != 0 && ((control[kDieOf + wg % kDies] >> die) & 1u) != 0;
}
// `values` values of a row from `first` on, for the next launch
__device__ __forceinline__ void empty(const __amdgpu_buffer_rsrc_t set, int row, int first, int values) {
    const int i = afresh((int)threadIdx.x & 63);
    for (int d = 0; d < values; d += 128)
        __builtin_amdgcn_raw_buffer_store_b32(kEmpty, set, wanted(d + 2 * i < values, 2 * (first + d) + 4 * i), row, 0);
}

// ---- a row into LDS -----------------------------------------------------------------------
// Eight neighbouring activations (word w of the row), quantised with s, as two planes of E4M3 bytes, a = 16 hi + lo with
// hi in -8 .. 7 and lo in 0 .. 15.  32 values form a block of 32 bytes hi, 32 bytes lo, in the order in which a code
// dword masked to nibbles gives its weights: ternary 0 2 .. 14, 1 3 .. 15, 16 18 ..; sign 0 4 .. 28, 1 5 .. 29, ..
// Also the negative sum of the word's group, scaled as the matrix cores' results are (see Codes).
template <int BITS>
__device__ __forceinline__ void put_word(unsigned char *planes, float *sums, int w, const float *x, float s, bool ok) {
    float hi[8], lo[8], sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float r = __builtin_rintf(__builtin_amdgcn_fmed3f(x[i] * s, -128.0f, 127.0f));
        hi[i] = __builtin_floorf(r * 0.0625f);
        lo[i] = __builtin_fmaf(hi[i], -16.0f, r);
        sum += r;
    }
    if (!ok) sum = 0.0f;
    sum = sum_of_16(sum);
    if (!ok) return;
    if ((w & 15) == 0) sums[w >> 4] = BITS == 2 ? -sum : -0.25f * sum;
    unsigned char *p = planes + (w >> 2) * 64;
    if constexpr (BITS == 2) {
        p += ((w >> 1) & 1) * 16 + (w & 1) * 4;
#pragma unroll
        for (int odd = 0; odd < 2; ++odd) {
            int h = __builtin_amdgcn_cvt_pk_fp8_f32(hi[odd], hi[2 + odd], 0, false);
            h = __builtin_amdgcn_cvt_pk_fp8_f32(hi[4 + odd], hi[6 + odd], h, true);
            int l = __builtin_amdgcn_cvt_pk_fp8_f32(lo[odd], lo[2 + odd], 0, false);
            l = __builtin_amdgcn_cvt_pk_fp8_f32(lo[4 + odd], lo[6 + odd], l, true);
            *reinterpret_cast<int *>(p + 8 * odd) = h;
            *reinterpret_cast<int *>(p + 32 + 8 * odd) = l;
        }
    } else {
        p += (w & 3) * 2;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            *reinterpret_cast<uint16_t *>(p + 8 * j) = (uint16_t)__builtin_amdgcn_cvt_pk_fp8_f32(hi[j], hi[4 + j], 0, false);
            *reinterpret_cast<uint16_t *>(p + 32 + 8 * j) = (uint16_t)__builtin_amdgcn_cvt_pk_fp8_f32(lo[j], lo[4 + j], 0, false);
        }
    }
}
__device__ __forceinline__ void unpack_word(const v4u v, float *f) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f[2 * j] = __uint_as_float(v[j] << 16);
        f[2 * j + 1] = __uint_as_float(v[j] & 0xffff0000u);
    }
}

struct Meet {   // LDS where the waves meet
    double sumsq[kFrontWaves];
    float top[kFrontWaves];
    int bad;
};
__device__ __forceinline__ bool given_up(const Meet &m) { return __builtin_amdgcn_readfirstlane(m.bad) != 0; }
__device__ __forceinline__ float multiplier(const Meet &m) {
    float amax = m.top[0];
#pragma unroll
    for (int i = 1; i < kFrontWaves; ++i) amax = fmaxf(amax, m.top[i]);
    const float recip = 1.0f / fmaxf(amax, 1e-5f);
    return recip * 127.0f;
}

// Words v of a row, a front wave's share of it, normed with weights w into f; their maximum is one of meet.top's when the
// waves have met.  false: give up.
template <int U>
__device__ __forceinline__ bool norm(Meet &meet, const v4u *v, const v4u *w, int dim, float eps, int wave, int lane, bool ok, float (*f)[8]) {
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < U; ++i) {
        unpack_word(v[i], f[i]);
#pragma unroll
        for (int j = 0; j < 8; j += 2) ss += (double)(f[i][j] * f[i][j]) + (double)(f[i][j + 1] * f[i][j + 1]);
    }
    const double wsum = bonsai_wave::sum64(ss);
    if (lane == 0) {
        meet.sumsq[wave] = wsum;
        if (!ok) meet.bad = 1;
    }
    __syncthreads();
    if (given_up(meet)) return false;
    double total = 0.0;
#pragma unroll
    for (int i = 0; i < kFrontWaves; ++i) total += meet.sumsq[i];
    const float var = (float)total / (float)dim;
    const float rs = 1.0f / sqrtf(var + eps);
    float top = 0.0f;
#pragma unroll
    for (int i = 0; i < U; ++i) {
        float wf[8];
        unpack_word(w[i], wf);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            f[i][j] = bf16_round(wf[j] * bf16_round(f[i][j] * rs));
            top = fmaxf(top, fabsf(f[i][j]));
        }
    }
    top = top_of_64(top);
    if (lane == 0) meet.top[wave] = top;
    __syncthreads();
    return true;
}
// Maximum of |value| over a wave's words.
template <int U>
__device__ __forceinline__ float top_of(const v4u *v) {
    float top = 0.0f;
#pragma unroll
    for (int i = 0; i < U; ++i) {
        float f[8];
        unpack_word(v[i], f);
#pragma unroll
        for (int j = 0; j < 8; ++j) top = fmaxf(top, fabsf(f[j]));
    }
    return top_of_64(top);
}

// ---- the projections ----------------------------------------------------------------------
// A lane's loads for one projection.
template <int N>
struct Weights {
    v4u w[N];
    uint32_t s[N];   // two group scales

    // Loads FROM .. TO - 1 of back wave `bw`: `rows` rows, i-th one row place(i) of n.  `on` = 0 asks for nothing.
    template <int BITS, int FROM, int TO, class Place>
    __device__ __forceinline__ void ask(uintptr_t weights, uintptr_t scales, const Share &sh, int bw, int rows, int n, Place place,
                                        int on) {
        const int total = on ? n * sh.units : 0;
        const __amdgpu_buffer_rsrc_t rw = rsrc_of(reinterpret_cast<const void *>(weights), total * 64);
        const __amdgpu_buffer_rsrc_t rs = rsrc_of(reinterpret_cast<const void *>(scales), total * (BITS == 2 ? 4 : 8));
        const int lane = afresh((int)threadIdx.x & 63);
        const int recip = 65536 / sh.units + 1;
#pragma unroll
        for (int i = FROM; i < TO; ++i) {
            const int idx = bw + i * kBackWaves;
            const int tile = (idx * recip) >> 16, u = idx - tile * sh.units;
            const int row = tile * 16 + (lane & 15);
            const int at = place(row) * sh.units + u;
            const int off = wanted(row < rows, at * 64 + (lane >> 4) * 16);
            w[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, off, 0, 0);
            const int o = BITS == 2 ? (off >> 6) * 4 : (off >> 6) * 8 + ((off >> 2) & 4);
            s[i] = __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0);
        }
    }
};

// One unit on the matrix cores (v_mfma_f32_16x16x128_f8f6f4, E4M3 x E2M1): weight rows are B's columns, and a code
// dword masked to nibbles already is E2M1: codes 0 .. 3 are 0, 0.5, 1, 1.5.  Four lanes share a row's 64 bytes, 16 each,
// so that one instruction sees pieces of two (sign weights: four) scale groups; A's rows keep them apart: row 2 g + p
// holds plane p of the activations of group g and zero where a lane's weights belong to another one.  With the sums of
// the activations going in as C, rows 2 g and 2 g + 1 of the result give 16 hi + lo = G / 2 (sign: G / 4), exactly.
template <int BITS>
struct Codes {
    static constexpr int kSteps = BITS == 2 ? 2 : 4;   // instructions a unit
    v8i b[kSteps];
    __device__ __forceinline__ explicit Codes(const v4u w) {
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            if constexpr (BITS == 2) {
                const uint32_t p = w[2 * i], q = w[2 * i + 1];
                b[i] = v8i{(int)(p & 0x33333333u), (int)((p >> 2) & 0x33333333u), (int)(q & 0x33333333u),
                           (int)((q >> 2) & 0x33333333u), 0, 0, 0, 0};
            } else {
                const uint32_t p = w[i];
                b[i] = v8i{(int)(p & 0x11111111u), (int)((p >> 1) & 0x11111111u), (int)((p >> 2) & 0x11111111u),
                           (int)((p >> 3) & 0x11111111u), 0, 0, 0, 0};
            }
        }
    }
};
// Where a lane finds its part of A: A's lane kb holds, in its first sixteen bytes, what meets half kb & 1 of the weights
// of B's lane kb >> 1 and, in the others, of lane 2 + (kb >> 1).  Byte offsets into the planes of unit 0 and from one
// unit and one instruction to the next; all three are that of the zero bytes, 0 and 0 where the row has another group.
template <int BITS>
struct Operand {
    static constexpr int kBlocks = BITS == 2 ? 2 : 4;   // blocks of 32 values a lane of B
    int x, y, unit_x, unit_y, step_x, step_y, sums;
    __device__ __forceinline__ Operand(int lane, int zero_at) {
        const int kb = lane >> 4, mm = lane & (BITS == 2 ? 3 : 7), g = mm >> 1;
        const int kx = kb >> 1, ky = 2 + kx, from = (mm & 1) * 32 + (kb & 1) * 16;
        const bool has_x = BITS == 2 ? g == 0 : g == kx, has_y = BITS == 2 ? g == 1 : g == ky;
        x = has_x ? kx * kBlocks * 64 + from : zero_at;
        y = has_y ? ky * kBlocks * 64 + from : zero_at;
        unit_x = has_x ? 4 * kBlocks * 64 : 0;
        unit_y = has_y ? 4 * kBlocks * 64 : 0;
        step_x = has_x ? 64 : 0;
        step_y = has_y ? 64 : 0;
        sums = BITS == 2 ? 0 : (kb & 1) * 2;
    }
};
// G x scale, summed over the unit's groups, in lanes 0 .. 15 (of the row), times 1 / 2 (sign: 1 / 4)
template <int BITS>
__device__ __forceinline__ float unit_product(const v4u w, uint32_t scales, const unsigned char *planes, const float *sums,
                                              const Operand<BITS> &op, int u) {
    const Codes<BITS> c(w);
    const unsigned char *px = planes + (op.x + u * op.unit_x), *py = planes + (op.y + u * op.unit_y);
    const float *so = sums + (u * (BITS == 2 ? 2 : 4) + op.sums);
    v4f d = v4f{0.0f, so[0], 0.0f, so[1]};
#pragma unroll
    for (int i = 0; i < Codes<BITS>::kSteps; ++i) {
        const v4u x = *reinterpret_cast<const v4u *>(px + i * op.step_x), y = *reinterpret_cast<const v4u *>(py + i * op.step_y);
        const v8i a = v8i{(int)x.x, (int)x.y, (int)x.z, (int)x.w, (int)y.x, (int)y.y, (int)y.z, (int)y.w};
        d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, c.b[i], d, 0, 4, 0, 0, 0, 0);
    }
    const float g0 = __builtin_fmaf(d[0], 16.0f, d[1]), g1 = __builtin_fmaf(d[2], 16.0f, d[3]);
    float v = g0 * __uint_as_float(scales << 16) + g1 * __uint_as_float(scales & 0xffff0000u);
    if constexpr (BITS == 1) {   // the other two groups are sixteen lanes further
        const Pair p = pair16(v);
        v = p.a + p.b;
    }
    return v;
}

__device__ __forceinline__ float silu_mul(float g, float u) {
    const float ex = __builtin_amdgcn_exp2f(g * -1.44269504088896341f);
    const float sg = bf16_round(g * __builtin_amdgcn_rcpf(1.0f + ex));
    return bf16_round(sg * u);
}

// What both kinds of waves know.
struct Common {
    const Args &a;
    int wg, lane, gqa, q_dim, n_qkv;
    Share sq, so, sg, sd;
    Rows lay;
    int rows_q, rows_o, rows_g, rows_d;
    __amdgpu_buffer_rsrc_t here, other;   // this launch's set and the other one
    uint8_t *parts;
    uint32_t epoch;
    bool attends, merges, near;
    int n, hide, sees_itself, position, token, kvh, unit, split, head, per, splits;
    HeadOrder order;
    int head_row0;   // of the kv head's rows of q|k|v, the workgroup's first
    __device__ int qkv_at() const { return kvh * order.rows() + head_row0; }   // .. in the exchange memory
    unsigned char *planes;
    float *sums, *red, *resid;
    uint16_t *raw;
    int zero_at;
    Meet &meet;
};

// a layer's addresses, one a lane
template <class Args>
__device__ __forceinline__ v2u ask_layer(const Args &a, int l) {
    const int i = afresh((int)threadIdx.x & 63);
    return __builtin_amdgcn_raw_buffer_load_b64(rsrc_of(a.layers, a.n_layers * (int)sizeof(Layer)),
                                                wanted(i < (int)sizeof(Layer) / 8, l * (int)sizeof(Layer) + i * 8), 0, 0);
}
__device__ __forceinline__ uintptr_t address(const v2u &t, int i) {
    return (uintptr_t)(uint32_t)__builtin_amdgcn_readlane((int)t.x, i) | (uintptr_t)(uint32_t)__builtin_amdgcn_readlane((int)t.y, i) << 32;
}

// ---- the back waves: weights, dot products, results ----------------------------------------
// NQ, NO, NG, ND: loads a lane for q|k|v, o, gate|up and down; TQ, TO: lanes a row that add up the results of q|k|v and
// of o and down (gate|up: one).  Returns false when the front waves gave up.
template <int BITS, int NQ, int NO, int NG, int ND, int TQ, int TO>
__device__ __forceinline__ bool back(const Common &c, int bw) {
    const Args &a = c.a;
    Weights<NQ> w_q;
    Weights<NO> w_o;
    Weights<NG> w_g;
    Weights<ND> w_d;
    constexpr int kHalfG = (NG + 1) / 2;
    const auto head_row = [&](int row) { return c.order.row_of(c.kvh, c.head_row0 + row); };
    const auto from = [&](const Share &sh) { return [&](int row) { return c.wg * sh.rows + row; }; };
    const auto in_turn = [&](int row) { return c.wg * c.sg.rows / 2 + (row & 1) * a.ffn + (row >> 1); };   // gate, up
    const auto ask_q = [&](const v2u &t, int on) { w_q.template ask<BITS, 0, NQ>(address(t, 0), address(t, 4), c.sq, bw, c.rows_q, c.n_qkv, head_row, on); };
    const auto ask_o = [&](const v2u &t, int on) { w_o.template ask<BITS, 0, NO>(address(t, 1), address(t, 5), c.so, bw, c.rows_o, a.dim, from(c.so), on); };
    const auto ask_g1 = [&](const v2u &t, int on) { w_g.template ask<BITS, 0, kHalfG>(address(t, 2), address(t, 6), c.sg, bw, c.rows_g, 2 * a.ffn, in_turn, on); };
    const auto ask_g2 = [&](const v2u &t, int on) { w_g.template ask<BITS, kHalfG, NG>(address(t, 2), address(t, 6), c.sg, bw, c.rows_g, 2 * a.ffn, in_turn, on); };
    const auto ask_d = [&](const v2u &t, int on) { w_d.template ask<BITS, 0, ND>(address(t, 3), address(t, 7), c.sd, bw, c.rows_d, a.dim, from(c.sd), on); };
    v2u cur = ask_layer(a, 0);
    ask_q(cur, 1);
    ask_o(cur, 1);
    ask_g1(cur, 1);

    // Units into red; then the first back wave alone adds up every row's, T lanes a row, and calls done(row, sum) in all
    // of its lanes.  The barrier behind it is where the front waves may begin to look for the next row.
    const auto project = [&](const auto &wt, auto n_c, auto t_c, const Share &sh, int rows, float &s, auto done) {
        constexpr int T = decltype(t_c)::value;
        constexpr int N = decltype(n_c)::value;
        const int lane = afresh(c.lane);
        const int recip = 65536 / sh.units + 1, pitch = sh.pitch();
        s = multiplier(c.meet);
        const Operand<BITS> operand(lane, c.zero_at);
        __syncthreads();   // the row is in LDS
        float v[N];
        int tile[N], u[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {   // (units past the last one are unit 0 of rows that do not exist)
            const int idx = bw + i * kBackWaves;
            tile[i] = (idx * recip) >> 16;
            u[i] = idx - tile[i] * sh.units;
            if (i > 0 && (i & 1) == 0) __builtin_amdgcn_sched_barrier(0);   // two units' operands at a time
            v[i] = unit_product<BITS>(wt.w[i], wt.s[i], c.planes, c.sums, operand, u[i]);
        }
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (bw + i * kBackWaves < sh.count && lane < 16) {
                float *to = c.red + (tile[i] * 16 + lane) * pitch + u[i];
                *to = v[i];
                if (u[i] == sh.units - 1)   // (whole words of four are read)
                    for (int e = sh.units; e < pitch; ++e) *++to = 0.0f;
            }
        __syncthreads();
        if (bw == 0) {
            const int quads = pitch >> 2;   // (behind a row's units come zeros)
            for (int base = 0; base < rows; base += 64 / T) {
                const int row = base + lane / T;
                const v4f *p = reinterpret_cast<const v4f *>(c.red + (row < rows ? row : 0) * pitch);
                float sum = 0.0f;
                for (int q = 0; q < quads; q += 2 * T) {
                    const int q0 = q + (lane & (T - 1)), q1 = q0 + T;
                    const v4f x = p[q0 < quads ? q0 : 0], y = p[q1 < quads ? q1 : 0];
                    const float sx = (x[0] + x[1]) + (x[2] + x[3]), sy = (y[0] + y[1]) + (y[2] + y[3]);
                    sum += (q0 < quads ? sx : 0.0f) + (q1 < quads ? sy : 0.0f);
                }
                if (T > 1) sum = sum_step<bonsai_wave::kXor1>(sum);
                if (T > 2) sum = sum_step<bonsai_wave::kXor2>(sum);
                if (T > 4) sum = sum_step<bonsai_wave::kHalfMirror>(sum);
                done(row, sum * (BITS == 2 ? 2.0f : 4.0f));
            }
        }
        __syncthreads();
    };
    const int lane = c.lane;
    for (int layer = 0; layer < a.n_layers; ++layer) {
        const int l = afresh_scalar(layer);
        const int row0 = l * c.lay.size;   // of the layer's rows in a set
        const int more = l + 1 < a.n_layers;
        const v2u nxt = ask_layer(a, more ? l + 1 : l);
        float s;

        // Weights are asked for where a row has just come in and none is on its way: what shares the memory system with
        // a hand-over delays it.
        if (c.rows_q) __syncthreads();   // sum of squares
        ask_d(cur, 1);
        ask_g2(cur, 1);
        if (bw == 1 && l > 0) empty(c.other, row0, c.wg * c.sd.rows, c.rows_d);
        if (c.rows_q) {
            if (given_up(c.meet)) return false;
            __syncthreads();   // maximum
            project(w_q, std::integral_constant<int, NQ>{}, std::integral_constant<int, TQ>{}, c.sq, c.rows_q, s, [&](int row, float v) {
                const float y = v / s, z = lanes_on<TQ>(y);
                if ((lane & (2 * TQ - 1)) == 0 && row < c.rows_q) hand_over_near(c.here, row0 + c.lay.qkv, (c.qkv_at() + row) * 2, pack_bf16(y, z), c.near);
            });
        }

        if (c.attends) {
            __syncthreads();   // query, key and value
            if (given_up(c.meet)) return false;
            __syncthreads();   // the waves' sums
        }
        if (c.merges) {
            __syncthreads();
            if (given_up(c.meet)) return false;
            __syncthreads();
        }

        const auto add = [&](const Share &sh, int rows, bool last, int to) {
            return [&, rows, last, to](int row, float v) {
                const float h = bf16_round(bf16_round(v / s) + c.resid[row < rows ? row : 0]);
                const float z = lanes_on<TO>(h);
                if ((lane & (TO - 1)) == 0 && row < rows) c.resid[row] = h;
                if ((lane & (2 * TO - 1)) == 0 && row < rows) {
                    const int at = (c.wg * sh.rows + row) * 2;
                    if (last)
                        *reinterpret_cast<uint32_t *>(reinterpret_cast<uint8_t *>(a.h_out) + at) = pack_bf16(h, z);
                    else
                        hand_over(c.here, to, at, pack_bf16(h, z));
                }
            };
        };
        if (c.rows_o) __syncthreads();   // maximum
        ask_q(nxt, more);
        if (bw == 1) empty(c.other, row0 + c.lay.qkv, c.qkv_at(), c.rows_q);
        if (c.rows_o) {
            if (given_up(c.meet)) return false;
            project(w_o, std::integral_constant<int, NO>{}, std::integral_constant<int, TO>{}, c.so, c.rows_o, s,
                    add(c.so, c.rows_o, false, row0 + c.lay.h2));
        }

        if (c.rows_g) __syncthreads();   // sum of squares
        ask_o(nxt, more);
        if (bw == 1) empty(c.other, row0 + c.lay.h2, c.wg * c.so.rows, c.rows_o);
        if (bw == 1 && c.unit < c.gqa) empty(c.other, row0 + c.lay.att, c.head * kHd, kHd);
        if (c.rows_g) {
            if (given_up(c.meet)) return false;
            __syncthreads();   // maximum
            project(w_g, std::integral_constant<int, NG>{}, std::integral_constant<int, 1>{}, c.sg, c.rows_g, s, [&](int row, float v) {
                const float y = bf16_round(v / s), up = lanes_on<1>(y);
                const float inner = silu_mul(y, up), z = lanes_on<2>(inner);
                if ((lane & 3) == 0 && row < c.rows_g) hand_over(c.here, row0 + c.lay.inner, c.wg * c.sg.rows + row, pack_bf16(inner, z));
            });
        }

        if (c.rows_d) __syncthreads();   // maximum, and the row itself, which all waves quantise
        ask_g1(nxt, more);
        if (bw == 1) empty(c.other, row0 + c.lay.inner, c.wg * c.sg.rows / 2, c.rows_g / 2);
        if (c.rows_d) {
            if (given_up(c.meet)) return false;
            const float sd = multiplier(c.meet);
            const int tid = afresh((int)threadIdx.x);
            for (int w = tid; (w & ~63) < (a.ffn >> 3); w += kThreads) {
                const bool ok = w < (a.ffn >> 3);
                float f[8];
                unpack_word(*reinterpret_cast<const v4u *>(c.raw + (ok ? w : 0) * 8), f);
                put_word<BITS>(c.planes, c.sums, w, f, sd, ok);
            }
            project(w_d, std::integral_constant<int, ND>{}, std::integral_constant<int, TO>{}, c.sd, c.rows_d, s,
                    add(c.sd, c.rows_d, !more, row0 + c.lay.size));
        }
        cur = nxt;
    }
    return true;
}

// ---- the front waves: rows in, norms, quantisation, attention -------------------------------
// UD, UQ, UF: 16-byte words a lane of a row of dim, of the attention's output, of ffn.  Returns false when a wait was
// too long.
template <int BITS, int UD, int UQ, int UF>
__device__ __forceinline__ bool front(const Common &c, int wave) {
    const Args &a = c.a;
    const int tid = threadIdx.x, lane = c.lane, n = c.n;
    __shared__ __align__(16) uint16_t q_lds[3 * kHd];            // query, key, value
    __shared__ __align__(16) float att_acc[kFrontWaves * kHd];
    __shared__ float att_ml[kFrontWaves * 2];
    __shared__ float weight_of[kMaxSplits];
    v2u cur = ask_layer(a, 0);
    v4u ln1[UD], ln2[UD], row_d[UD];
    const auto ask_row = [&](v4u *v, const void *p) {
        const __amdgpu_buffer_rsrc_t r = rsrc_of(p, 2 * a.dim);
        const int at = afresh(tid);
#pragma unroll
        for (int i = 0; i < UD; ++i)
            v[i] = __builtin_amdgcn_raw_buffer_load_b128(r, wanted(at + i * kFront < (a.dim >> 3), (at + i * kFront) * 16), 0, 0);
    };
    uint32_t head_w[2];   // norm weights of the wave's head row: wave 0 the query's, wave 1 the key's
    const auto ask_head = [&](const v2u &t) {
        const __amdgpu_buffer_rsrc_t r = rsrc_of(reinterpret_cast<const void *>(address(t, wave == 0 ? 10 : 11)), 2 * kHd);
        const int i = afresh(lane);
        head_w[0] = __builtin_amdgcn_raw_buffer_load_b16(r, 2 * i, 0, 0);
        head_w[1] = __builtin_amdgcn_raw_buffer_load_b16(r, 2 * i + 128, 0, 0);
    };
    // keys and values of the wave's first slots: eight lanes a slot, sixteen dims a lane
    const int per_wave = c.per / kFrontWaves;             // a multiple of 16
    const int slot0 = c.split * c.per + wave * per_wave;
    const int slots_end = slot0 + per_wave < n ? slot0 + per_wave : n;   // of the history
    v4u keys[kRounds][2], vals[kRounds][2];
    const auto ask_history = [&](int l, int at, int on) {
        const size_t plane = (size_t)a.n_kv * a.slots * kHd;
        const uint16_t *k = a.kv + (size_t)l * plane + (size_t)c.kvh * a.slots * kHd;
        const int bytes = on && slots_end > 0 ? slots_end * 256 : 0;
        const __amdgpu_buffer_rsrc_t rk = rsrc_of(k, bytes), rv = rsrc_of(k + (size_t)a.n_layers * plane, bytes);
        const int i = afresh(lane);
        const int off = (at + (i >> 3)) * 256 + (i & 7) * 32;
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            keys[r][0] = __builtin_amdgcn_raw_buffer_load_b128(rk, off + r * 2048, 0, 0);
            keys[r][1] = __builtin_amdgcn_raw_buffer_load_b128(rk, off + r * 2048 + 16, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            vals[r][0] = __builtin_amdgcn_raw_buffer_load_b128(rv, off + r * 2048, 0, 0);
            vals[r][1] = __builtin_amdgcn_raw_buffer_load_b128(rv, off + r * 2048 + 16, 0, 0);
        }
    };
    const auto norm_weights = [&](const v2u &t, int which) { return reinterpret_cast<const void *>(address(t, 8 + which)); };
    {
        const uint32_t tok = (uint32_t)c.token;
        const uint16_t *e = a.embed + (size_t)(tok < (uint32_t)a.vocab ? tok : (uint32_t)a.vocab - 1) * a.dim;
        ask_row(row_d, e);
        if (tid < c.rows_d) c.resid[tid] = bf16_bits_to_f32(e[c.wg * c.sd.rows + tid]);
        if (tid < 16) reinterpret_cast<uint32_t *>(c.planes + c.zero_at)[tid] = 0;
    }
    ask_row(ln1, norm_weights(cur, 0));
    // (the position is the same in every layer)
    const int pos = c.position < 0 ? 0 : (c.position >= a.max_pos ? a.max_pos - 1 : c.position);
    const uint32_t c0 = a.cos_t[(size_t)pos * kHd + lane], c1 = a.cos_t[(size_t)pos * kHd + lane + 64];
    const uint32_t s0 = a.sin_t[(size_t)pos * kHd + lane], s1 = a.sin_t[(size_t)pos * kHd + lane + 64];
    ask_head(cur);
    ask_history(0, slot0, c.attends);
    ask_row(ln2, norm_weights(cur, 1));

    // norm + quantisation of a row of dim values; false: give up
    const auto stage_norm = [&](const v4u *v, const v4u *w, bool ok) -> bool {
        float f[UD][8];
        if (!norm<UD>(c.meet, v, w, a.dim, a.eps, wave, lane, ok, f)) return false;
        const float s = multiplier(c.meet);
        const int t = afresh(tid);
#pragma unroll
        for (int i = 0; i < UD; ++i) put_word<BITS>(c.planes, c.sums, t + i * kFront, f[i], s, t + i * kFront < (a.dim >> 3));
        __syncthreads();
        __syncthreads();   // the back waves' units
        __syncthreads();   // and their results
        return true;
    };

    for (int layer = 0; layer < a.n_layers; ++layer) {
        const int l = afresh_scalar(layer);
        const uint32_t limit = l == 0 ? a.first_wait : a.later_wait;
        const int row0 = l * c.lay.size;   // of the layer's rows in a set
        const int more = l + 1 < a.n_layers;
        const int nl = more ? l + 1 : l;
        v2u nxt;

        // ---- q | k | v
        {
            bool ok = true;
            if (l > 0 && c.rows_q) ok = receive<UD>(c.here, row0, a.dim >> 3, row_d, pause_row(UD), limit);
            nxt = ask_layer(a, nl);
            if (c.rows_q && !stage_norm(row_d, ln1, ok)) return false;
        }

        // ---- attention
        if (c.attends) {
            const int tid = afresh((int)threadIdx.x), lane = tid & 63;
            const bool has_token = n >= c.split * c.per && n < (c.split + 1) * c.per;   // the part that holds the token itself
            bool ok = true;
            if (wave < (has_token ? 3 : 1)) {
                const int row = wave == 0 ? c.head - c.kvh * c.gqa : c.gqa + wave - 1;   // of the kv head's
                const int from = row0 + c.lay.qkv + (c.kvh * (c.gqa + 2) + row) * 256;
                uint32_t d = kEmpty;
                uint32_t since = 0;
                for (int z = 0; z < kPauseHead; ++z) __builtin_amdgcn_s_sleep(1);
                for (int spins = first_spin(limit);; ++spins) {
                    d = __builtin_amdgcn_raw_buffer_load_b32(c.here, lane * 4, from, kDeviceScope);
                    if (__all(d != kEmpty)) break;
                    if (timed_out(spins, since, limit)) {
                        ok = false;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
                uint16_t *dst = q_lds + wave * kHd;
                const bool writes = wave > 0 && c.unit == c.split * c.gqa;   // the first c.head's workgroup fills the cache
                uint16_t *cache = a.kv + ((size_t)((wave == 2 ? a.n_layers : 0) + l) * a.n_kv + c.kvh) * a.slots * kHd + (size_t)a.sigma * kHd;
                if (wave == 2) {
                    reinterpret_cast<uint32_t *>(dst)[lane] = d;
                    if (writes) reinterpret_cast<uint32_t *>(cache)[lane] = d;
                } else {
                    const uint32_t lo_d = (uint32_t)__shfl((int)d, lane >> 1), hi_d = (uint32_t)__shfl((int)d, 32 + (lane >> 1));
                    const RopeRowIn x{lane & 1 ? lo_d >> 16 : lo_d & 0xffffu, lane & 1 ? hi_d >> 16 : hi_d & 0xffffu,
                                      head_w[0], head_w[1], c0, c1, s0, s1};
                    uint32_t o0, o1;
                    rope_row_math(x, a.eps, o0, o1);
                    dst[lane] = (uint16_t)o0;
                    dst[lane + 64] = (uint16_t)o1;
                    if (writes) {
                        cache[lane] = (uint16_t)o0;
                        cache[lane + 64] = (uint16_t)o1;
                    }
                }
            }
            if (lane == 0 && !ok) c.meet.bad = 1;
            __syncthreads();
            if (given_up(c.meet)) return false;
            float m_run = -INFINITY, l_run = 0.0f, acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            const float to_log2 = a.scale * 1.44269504088896341f;
            const int group = lane >> 3, sub = lane & 7;
            const v4u *row_q = reinterpret_cast<const v4u *>(q_lds + sub * 16);
            const v4u q0 = row_q[0], q1 = row_q[1];
            for (int at = 0; at < per_wave && slot0 + at <= n; at += 8 * kRounds) {
                if (at) ask_history(l, slot0 + at, 1);
                float x[kRounds];
                const int left = (per_wave - at) >> 3;
#pragma unroll
                for (int r = 0; r < kRounds; ++r) {
                    x[r] = -INFINITY;
                    if (r >= left) continue;
                    const int slot = slot0 + at + 8 * r + group;
                    if (slot == n) {   // the token itself
                        keys[r][0] = row_q[16];
                        keys[r][1] = row_q[17];
                        vals[r][0] = row_q[32];
                        vals[r][1] = row_q[33];
                    }
                    const v4u k0 = keys[r][0], k1 = keys[r][1];
                    float d = dot2_bf16(k0.x, q0.x, 0.0f), e = dot2_bf16(k1.x, q1.x, 0.0f);
                    d = dot2_bf16(k0.y, q0.y, d);
                    e = dot2_bf16(k1.y, q1.y, e);
                    d = dot2_bf16(k0.z, q0.z, d);
                    e = dot2_bf16(k1.z, q1.z, e);
                    d = dot2_bf16(k0.w, q0.w, d);
                    e = dot2_bf16(k1.w, q1.w, e);
                    d += e;
                    d += bonsai_wave::partner<bonsai_wave::kXor1>(d);
                    d += bonsai_wave::partner<bonsai_wave::kXor2>(d);
                    d += bonsai_wave::partner<bonsai_wave::kHalfMirror>(d);
                    x[r] = slot < n + c.sees_itself && slot != c.hide ? d * to_log2 : -INFINITY;
                }
                float m = x[0];
#pragma unroll
                for (int r = 1; r < kRounds; ++r) m = fmaxf(m, x[r]);
                m = fmaxf(m, from_xor8(m));
                Pair p = pair16(m);
                p = pair32(fmaxf(p.a, p.b));
                m = fmaxf(m_run, fmaxf(p.a, p.b));
                const float base = m == -INFINITY ? 0.0f : m;
                const float keep = __builtin_amdgcn_exp2f(m_run - base);
                l_run *= keep;   // of the lane's own slots
                m_run = m;
                // the lane's sixteen dims over its slots, then over the eight groups of lanes: the swaps leave four of
                // the sixteen sums a lane
                float t[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) t[i] = 0.0f;
#pragma unroll
                for (int r = 0; r < kRounds; ++r) {
                    if (r >= left) continue;
                    const float w = __builtin_amdgcn_exp2f(x[r] - base);
                    l_run += w;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint32_t v = vals[r][i >> 2][i & 3];
                        t[2 * i] += w * __uint_as_float(v << 16);
                        t[2 * i + 1] += w * __uint_as_float(v & 0xffff0000u);
                    }
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) {   // lanes below 32: dims 0 .. 7, above: 8 .. 15
                    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(t[i]), __float_as_uint(t[i + 8]), false, false);
                    t[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {   // even rows of sixteen lanes: the lower four of these
                    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(t[i]), __float_as_uint(t[i + 4]), false, false);
                    t[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = acc[i] * keep + (t[i] + from_xor8(t[i]));
            }
            l_run += from_xor8(l_run);
            Pair lp = pair16(l_run);
            lp = pair32(lp.a + lp.b);
            if ((lane & 8) == 0) {
                const int d = sub * 16 + (lane >> 5) * 8 + ((lane >> 4) & 1) * 4;
                *reinterpret_cast<v4u *>(att_acc + wave * kHd + d) =
                    v4u{__float_as_uint(acc[0]), __float_as_uint(acc[1]), __float_as_uint(acc[2]), __float_as_uint(acc[3])};
            }
            if (lane == 0) {
                att_ml[wave * 2] = m_run;
                att_ml[wave * 2 + 1] = lp.a + lp.b;
            }
            __syncthreads();
            if (tid < kHd) {   // the waves' sums together, a thread a dim
                float ml[2 * kFrontWaves], o = 0.0f, sum = 0.0f, m = -INFINITY;
#pragma unroll
                for (int w = 0; w < 2 * kFrontWaves; ++w) ml[w] = att_ml[w];
#pragma unroll
                for (int w = 0; w < kFrontWaves; ++w) m = fmaxf(m, ml[2 * w]);
                const float base = m == -INFINITY ? 0.0f : m;
#pragma unroll
                for (int w = 0; w < kFrontWaves; ++w) {
                    const float f = __builtin_amdgcn_exp2f(ml[2 * w] - base);
                    o += f * att_acc[w * kHd + tid];
                    sum += f * ml[2 * w + 1];
                }
                if (c.splits == 1) {
                    const float y = sum > 0.0f ? o / sum : 0.0f;
                    const float z = bonsai_wave::partner<bonsai_wave::kXor1>(y);
                    if ((tid & 1) == 0)
                        hand_over(c.here, row0 + c.lay.att, (c.head * kHd + tid) * 2, pack_bf16(y, z));
                } else {
                    const uint32_t tag = c.epoch * (uint32_t)a.n_layers + (uint32_t)l + 1u;
                    const __amdgpu_buffer_rsrc_t r = rsrc_of(c.parts + (size_t)(c.head * kMaxSplits + c.split) * (kPartEntries * 8), kPartEntries * 8);
                    const v2u part = v2u{__float_as_uint(o), tag}, of_all = v2u{__float_as_uint(tid ? sum : m), tag};
                    const int last = wanted(tid < 2, (kHd + tid) * 8);
                    if (c.near) {
                        __builtin_amdgcn_raw_buffer_store_b64(part, r, tid * 8, 0, 0);
                        __builtin_amdgcn_raw_buffer_store_b64(of_all, r, last, 0, 0);
                    } else {
                        __builtin_amdgcn_raw_buffer_store_b64(part, r, tid * 8, 0, kDeviceScope);
                        __builtin_amdgcn_raw_buffer_store_b64(of_all, r, last, 0, kDeviceScope);
                    }
                }
            }
        }
        if (c.merges) {   // the c.head's c.parts together, a thread a (quarter of the c.parts, dim)
            const int tid = afresh((int)threadIdx.x), lane = tid & 63;
            const uint32_t tag = c.epoch * (uint32_t)a.n_layers + (uint32_t)l + 1u;
            const __amdgpu_buffer_rsrc_t r = rsrc_of(c.parts + (size_t)c.head * kMaxSplits * (kPartEntries * 8), kMaxSplits * kPartEntries * 8);
            const int d = tid & 127, q = tid >> 7;
            bool ok = true;
            uint32_t since = 0;
            v2u o[kMaxSplits / 2];
            v4u ml;
            for (int z = 0; z < kPauseParts; ++z) __builtin_amdgcn_s_sleep(1);
            for (int spins = first_spin(limit);; ++spins) {
#pragma unroll
                for (int i = 0; i < kMaxSplits / 2; ++i)
                    o[i] = __builtin_amdgcn_raw_buffer_load_b64(r, wanted(q + 2 * i < c.splits, ((q + 2 * i) * kPartEntries + d) * 8), 0, kDeviceScope);
                ml = __builtin_amdgcn_raw_buffer_load_b128(r, wanted(wave == 0 && lane < c.splits, (lane * kPartEntries + kHd) * 8), 0, kDeviceScope);
                bool all = wave != 0 || lane >= c.splits || ((ml.y == tag) & (ml.w == tag));
#pragma unroll
                for (int i = 0; i < kMaxSplits / 2; ++i) all = all & ((q + 2 * i >= c.splits) | (o[i].y == tag));
                if (__all(all)) break;
                if (timed_out(spins, since, limit)) {
                    ok = false;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (wave == 0) {
                const float m = lane < c.splits ? __uint_as_float(ml.x) : -INFINITY;
                const float top = wave_max(m);
                const float f = __builtin_amdgcn_exp2f(m - (top == -INFINITY ? 0.0f : top));
                const float sum = wave_sum(lane < c.splits ? f * __uint_as_float(ml.z) : 0.0f);
                if (lane < c.splits) weight_of[lane] = sum > 0.0f ? f / sum : 0.0f;
            }
            if (lane == 0 && !ok) c.meet.bad = 1;
            __syncthreads();
            if (given_up(c.meet)) return false;
            float y = 0.0f;
#pragma unroll
            for (int i = 0; i < kMaxSplits / 2; ++i)
                if (q + 2 * i < c.splits) y += weight_of[q + 2 * i] * __uint_as_float(o[i].x);
            att_acc[tid] = y;
            __syncthreads();
            if (tid < 64) {
                float z[2];
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    z[i] = att_acc[2 * tid + i] + att_acc[128 + 2 * tid + i];
                hand_over(c.here, row0 + c.lay.att, (c.head * kHd + 2 * tid) * 2,
                          pack_bf16(z[0], z[1]));
            }
        }

        // ---- o
        {
            v4u row_a[UQ];
            if (c.rows_o) {
                const bool ok = receive<UQ>(c.here, row0 + c.lay.att, c.q_dim >> 3, row_a, kPauseAtt, limit);
                const float top = top_of<UQ>(row_a);
                if (lane == 0) {
                    c.meet.top[wave] = top;
                    if (!ok) c.meet.bad = 1;
                }
                __syncthreads();
                if (given_up(c.meet)) return false;
                const float s = multiplier(c.meet);
                const int t = afresh(tid);
#pragma unroll
                for (int i = 0; i < UQ; ++i) {
                    float f[8];
                    unpack_word(row_a[i], f);
                    put_word<BITS>(c.planes, c.sums, t + i * kFront, f, s, t + i * kFront < (c.q_dim >> 3));
                }
                __syncthreads();
                __syncthreads();
                __syncthreads();
            }
        }

        // ---- gate | up
        {
            bool ok = true;
            if (c.rows_g) ok = receive<UD>(c.here, row0 + c.lay.h2, a.dim >> 3, row_d, kPauseH2, limit);
            ask_row(ln1, norm_weights(nxt, 0));
            ask_head(nxt);
            ask_history(nl, slot0, c.attends && more);
            if (c.rows_g && !stage_norm(row_d, ln2, ok)) return false;
        }

        // ---- down
        {
            v4u row_f[UF];
            bool ok = true;
            if (c.rows_d) ok = receive<UF>(c.here, row0 + c.lay.inner, a.ffn >> 3, row_f, kPauseInner, limit);
            ask_row(ln2, norm_weights(nxt, 1));
            if (c.rows_d) {
                const int t = afresh(tid);
#pragma unroll
                for (int i = 0; i < UF; ++i)
                    if (t + i * kFront < (a.ffn >> 3)) *reinterpret_cast<v4u *>(c.raw + (t + i * kFront) * 8) = row_f[i];
                const float top = top_of<UF>(row_f);
                if (lane == 0) {
                    c.meet.top[wave] = top;
                    if (!ok) c.meet.bad = 1;
                }
                __syncthreads();
                if (given_up(c.meet)) return false;
                const float s = multiplier(c.meet);
                for (int w = t; (w & ~63) < (a.ffn >> 3); w += kThreads) {
                    const bool in = w < (a.ffn >> 3);
                    float f[8];
                    unpack_word(*reinterpret_cast<const v4u *>(c.raw + (in ? w : 0) * 8), f);
                    put_word<BITS>(c.planes, c.sums, w, f, s, in);
                }
                __syncthreads();
                __syncthreads();
                __syncthreads();
            }
        }
        cur = nxt;
    }
    return true;
}

template <int BITS, int NQ, int NO, int NG, int ND, int TQ, int TO, int UD, int UQ, int UF>
__global__ void __launch_bounds__(kThreads)
step_one_kernel(const Args a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wg = blockIdx.x;
    __shared__ Meet meet;
    __shared__ float resid[256];
    const int groups = a.groups, gqa = a.n_heads / a.n_kv;
    const int q_dim = a.n_heads * kHd, n_qkv = (a.n_heads + 2 * a.n_kv) * kHd;
    const HeadOrder order{a.n_heads, a.n_kv, gqa};
    const Share sq(a.dim, order.rows(), groups / a.n_kv, BITS, false), so(q_dim, a.dim, groups, BITS, false),
        sg(a.dim, 2 * a.ffn, groups, BITS, true), sd(a.ffn, a.dim, groups, BITS, false);
    const auto mine = [](const Share &s, int n, int i) {
        const int left = n - i * s.rows;
        return left < 0 ? 0 : (left < s.rows ? left : s.rows);
    };
    const int kvh = wg % a.n_kv, unit = wg / a.n_kv;
    const int rows_q = mine(sq, order.rows(), unit), rows_o = mine(so, a.dim, wg), rows_g = mine(sg, 2 * a.ffn, wg), rows_d = mine(sd, a.dim, wg);

    // The attention's share: the slots [0, n] (slot n is the token itself, whose key and value come from the exchange
    // memory) of one head, or a part of them.  A workgroup a query head rather than a kv head: the chain is shorter, and
    // the heads' second reads of keys and values come from their common L2.
    const auto in = (const __attribute__((address_space(4))) int32_t *)(uintptr_t)a.step_in;
    const int n = in[0] < 0 ? 0 : (in[0] < a.sigma ? in[0] : a.sigma);   // as everywhere: a history within its slots
    const int split = unit / gqa;
    const int head = kvh * gqa + unit - split * gqa;
    const int room = groups / (a.n_kv * gqa);
    const int max_splits = room < kMaxSplits ? room : kMaxSplits;
    const int per = n < kSingle ? (n < 64 ? 64 : kSingle) : 64 * ((n + 64 * max_splits) / (64 * max_splits));
    const int splits = n < kSingle ? 1 : (n + per) / per;
    const bool attends = split < splits, merges = splits > 1 && split == 0;
    if (rows_q + rows_o + rows_g + rows_d == 0 && !attends) return;

    uint32_t *control = reinterpret_cast<uint32_t *>(a.exchange);
    const auto state = (const __attribute__((address_space(4))) uint32_t *)(uintptr_t)control;
    const uint32_t epoch = state[0];
    if (state[1]) {
        if (wg == 0 && tid == 0) *a.status = 1;
        return;
    }
    const Rows lay(a.dim, a.ffn, a.n_heads, a.n_kv);
    const int set_bytes = a.n_layers * lay.size;
    uint8_t *const sets = a.exchange + kControlBytes;
    const int k_max = a.ffn > q_dim ? (a.ffn > a.dim ? a.ffn : a.dim) : (q_dim > a.dim ? q_dim : a.dim);
    int results = sq.results() > so.results() ? sq.results() : so.results();
    results = results > sg.results() ? results : sg.results();
    results = results > sd.results() ? results : sd.results();
    const Lds at(k_max, results, a.ffn);
    const Common c{a, wg, tid & 63, gqa, q_dim, n_qkv, sq, so, sg, sd, lay, rows_q, rows_o, rows_g, rows_d,
                   rsrc_of(sets + (size_t)(epoch & 1) * set_bytes, set_bytes), rsrc_of(sets + (size_t)((epoch & 1) ^ 1) * set_bytes, set_bytes), sets + (size_t)2 * set_bytes,
                   epoch, attends, merges, near_heads(state, wg), n, in[1], in[2] & 1, in[3], in[4], kvh, unit, split, head, per, splits, order,
                   unit * sq.rows, smem,
                   reinterpret_cast<float *>(smem + at.sums), reinterpret_cast<float *>(smem + at.red), resid,
                   reinterpret_cast<uint16_t *>(smem + at.raw), 2 * k_max, meet};
    if (tid == 0) meet.bad = 0;
    __syncthreads();
    const bool done = wave < kFrontWaves ? front<BITS, UD, UQ, UF>(c, wave) : back<BITS, NQ, NO, NG, ND, TQ, TO>(c, wave - kFrontWaves);
    if (tid == 0) {
        if (!done) {
            *a.status = 1;
            control[1] = 1;
        } else if (wg == 0) {
            control[0] = epoch + 1;
        }
    }
}

__global__ void __launch_bounds__(256) exchange_reset_kernel(v4u *p, size_t words, size_t rows_from, size_t rows_to) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < words; i += (size_t)gridDim.x * 256)
        p[i] = i >= rows_from && i < rows_to ? v4u{kEmpty, kEmpty, kEmpty, kEmpty} : v4u{0, 0, 0, 0};
}

// The dies of the workgroups of a launch, then whether those with the same number modulo eight share one.
__global__ void __launch_bounds__(64) dies_kernel(uint32_t *control) {
    uint32_t die;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(die));
    if (threadIdx.x == 0) __hip_atomic_fetch_or(control + kDieOf + blockIdx.x % kDies, 1u << die, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__global__ void __launch_bounds__(64) dies_shared_kernel(uint32_t *control, int n_kv) {
    const uint32_t dies = control[kDieOf + threadIdx.x % kDies];
    const bool one = __all(dies != 0 && (dies & (dies - 1)) == 0);
    if (threadIdx.x == 0) control[kDiesShared] = one && n_kv % kDies == 0;
}

// ---- host ---------------------------------------------------------------------------------
inline hipError_t look_at_dies(void *exchange, int n_kv, int groups, hipStream_t stream) {
    uint32_t *control = static_cast<uint32_t *>(exchange);
    hipLaunchKernelGGL(dies_kernel, dim3(groups), dim3(64), 0, stream, control);
    hipLaunchKernelGGL(dies_shared_kernel, dim3(1), dim3(64), 0, stream, control, n_kv);
    return hipGetLastError();
}
// The builds: loads a lane per projection and words a lane per row that each of them holds.
struct Build {
    int bits, nq, no, ng, nd, ud, uq, uf;
};
constexpr Build kBuilds[] = {
    {2, 1, 1, 2, 2, 1, 1, 3},   // the 1.7B shape and below: 30 registers of weights
    {2, 2, 2, 5, 4, 2, 2, 5},   // the 4B shape: 65
    {1, 1, 1, 1, 1, 1, 1, 3},
    {1, 1, 1, 3, 2, 2, 2, 5},
};
struct Fit {
    int build = -1, lds = 0;
    int64_t bytes = 0, marked = 0;   // exchange memory; behind the control words, up to here, marks of empty rows
};
inline Fit fit(int bits, int n_layers, int dim, int ffn, int n_heads, int n_kv, int groups) {
    Fit f;
    const int q_dim = n_heads * kHd;
    if ((bits != 1 && bits != 2) || n_layers < 2 || n_kv < 1 || n_heads < 1 || n_heads % n_kv != 0 || groups / n_heads < 1 ||
        groups > 65535 || dim < 128 || ffn < 128 || dim % unit_k(bits) != 0 || ffn % unit_k(bits) != 0 || q_dim % unit_k(bits) != 0)
        return f;
    const int64_t n_qkv = (int64_t)(n_heads + 2 * n_kv) * kHd;
    // 32-bit offsets into a matrix
    if (2 * (int64_t)ffn * dim >= kOob || n_qkv * dim >= kOob) return f;
    const HeadOrder order{n_heads, n_kv, n_heads / n_kv};
    const Share s[4] = {{dim, order.rows(), groups / n_kv, bits, false}, {q_dim, dim, groups, bits, false},
                        {dim, 2 * ffn, groups, bits, true}, {ffn, dim, groups, bits, false}};
    int results = 0;
    for (const Share &x : s) {
        if (x.rows > 256 || x.count > 2048) return f;
        if (x.results() > results) results = x.results();
    }
    const int k = ffn > q_dim ? (ffn > dim ? ffn : dim) : (q_dim > dim ? q_dim : dim);
    f.lds = Lds(k, results, ffn).size;
    if (f.lds > 58 * 1024) return f;
    const Rows lay(dim, ffn, n_heads, n_kv);
    if ((int64_t)n_layers * lay.size > 0x7fffffff) return f;
    f.marked = kControlBytes + 2 * (int64_t)n_layers * lay.size;
    f.bytes = f.marked + (int64_t)n_heads * kMaxSplits * kPartEntries * 8;
    const auto words = [](int k) { return (k / 8 + kFront - 1) / kFront; };
    for (int i = 0; i < (int)(sizeof kBuilds / sizeof kBuilds[0]); ++i) {
        const Build &b = kBuilds[i];
        if (b.bits == bits && s[0].loads() <= b.nq && s[1].loads() <= b.no && s[2].loads() <= b.ng && s[3].loads() <= b.nd &&
            words(dim) <= b.ud && words(q_dim) <= b.uq && words(ffn) <= b.uf) {
            f.build = i;
            break;
        }
    }
    return f;
}
inline const void *kernel_of(int build) {
    switch (build) {
        case 0: return reinterpret_cast<const void *>(&step_one_kernel<2, 1, 1, 2, 2, 4, 8, 1, 1, 3>);
        case 1: return reinterpret_cast<const void *>(&step_one_kernel<2, 2, 2, 5, 4, 2, 4, 2, 2, 5>);
        case 2: return reinterpret_cast<const void *>(&step_one_kernel<1, 1, 1, 1, 1, 4, 8, 1, 1, 3>);
        default: return reinterpret_cast<const void *>(&step_one_kernel<1, 1, 1, 3, 2, 2, 4, 2, 2, 5>);
    }
}

}  // namespace step_one
#endif  // BONSAI_STEP_ONE_HIP_H
