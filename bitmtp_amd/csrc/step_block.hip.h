// All layers of a decode step of 2 to 16 rows in one launch (`bonsai_decode_step_block`): draft and verify blocks.
//
// With a launch for each operation (ten a layer) a nine-row step of the 1.7B shape took 33 us a layer, of which reading its
// weights is 2.7 us.  As in the one-token form (step_one.hip.h) one workgroup per compute unit stays for the whole step and
// owns a share of every projection's rows.  What differs is that a workgroup cannot norm and quantise sixteen rows for itself
// (2.5 us a phase): the rows' workgroups do, one row each, and leave the int8 row for everybody.  So a layer alternates
// between
//     row phases (workgroup m: row m)      norm + quantise | merge of the attention's parts + quantise | norm + quantise |
//                                          quantise
//     projections (all workgroups)         q|k|v | o, add | gate|up, SiLU * up | down, add
// and the attention between the first projection and the second row phase, a query head or a part of its slots a workgroup,
// from the last workgroup on, so that the rows' ones, which everybody waits for, have none of it, of o or of down.
//
// Hand-overs, eight a layer of 1.0 - 1.4 us each, are what bounds it now: the nine-row step takes 22 us a layer, and bytes and
// instructions little of that.  To a row phase: two bf16 values and a tag (step and layer) in eight bytes, which nothing but
// the value itself makes valid; few readers wait for them.  From a row phase: int8 rows and, stored with them, their
// multipliers, in one of two sets of places, one for each layer, of which a step empties the other; no int8 row holds -128.
// One wave of a workgroup looks for a row's announcement (in eight copies: all 256 looking at one line took 0.3 us longer);
// then the others look for their stretch of the rows and it for the multipliers.  (All looking at the rows from the start
// took 4 us a layer more; only behind the multipliers, 1 % more of a step.)  Waits are bounded and handled as in the
// one-token form.
//
// Projections: 16 rows of weights x 128 of K x 16 tokens are two v_mfma_i32_16x16x64_i8, exact group sums.  A back wave
// owns a stretch of K for all rows of the workgroup and reads that stretch of the tokens once; the waves' results meet in
// LDS in the order of K.
//
// The rows of q|k|v are dealt out by kv head, so that the hand-over to the attention stays within a die (near_heads of
// step_one.hip.h): nine rows 610 -> 594 us (1.7B shape), 1006 -> 992 (4B), sixteen 661 -> 636, of which the near stores are 6 and 11 us
// at nine rows.
//
// Layers of nine rows, 1.7B / 4B shape, us at a history of 24, 300, 1500: 934 / 961 / 1034 -> 590 / 645 / 761 and
// 1521 / 1543 / 1657 -> 988 / 1092 / 1289; two rows (1.7B) 812 / 818 / 900 -> 539 / 581 / 702; sixteen 987 / 1011 / 1089 ->
// 637 / 692 / 817.
#ifndef BONSAI_STEP_BLOCK_HIP_H
#define BONSAI_STEP_BLOCK_HIP_H

namespace step_block {

using step_one::address;
using step_one::afresh;
using step_one::afresh_scalar;
using step_one::ask_layer;
using step_one::given_up;
using step_one::HeadOrder;
using step_one::kBack;
using step_one::kBackWaves;
using step_one::kFront;
using step_one::kFrontWaves;
using step_one::kOob;
using step_one::kThreads;
using step_one::Layer;
using step_one::Meet;
using step_one::multiplier;
using step_one::pair16;
using step_one::pair32;
using step_one::rsrc_of;
using step_one::top_of;
using step_one::unpack_word;
using step_one::v2u;
using step_one::v4f;
using step_one::v4u;
using step_one::wanted;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));

constexpr int kRows = 16;                   // rows of a block at most
constexpr int kMaxSplits = 32;              // attention parts per head
constexpr int kPartBytes = (kHd + 4) * 8;   // of a (head, part, row): 128 sums, maximum, sum, each with its tag
constexpr int kControlBytes = 256;
constexpr int kMostLds = 159 * 1024;        // beside what is declared in place
constexpr uint32_t kEmpty = 0x80808080u;    // int8 rows hold no -128, a multiplier is positive
constexpr int kCopies = 8;                  // of the multipliers' line, one for each XCD's workgroups
constexpr int kNap = 1;                     // of 64 cycles, between two looks
// .. and before a row's workgroup looks for its row (27 ns each): none 593, 10 588, 20 589 us a nine-row step (1.7B shape, 24 slots), 991,
// 984 and 993 with the 4B one; none and 10 level at 300 and 900 slots, and at all three with 1024 x 3072 and 2304 x 6400.
constexpr int kPause = 10;
constexpr int kVPitch = 272, kOPitch = 132; // bytes of a slot's values, floats of a row's sums in LDS

struct Args {
    const Layer *layers;
    const uint16_t *embed;
    const int32_t *step_in;   // cache_len, hide, row masks, positions, tokens
    uint16_t *kv;
    const uint16_t *cos_t, *sin_t;
    uint8_t *exchange;
    uint16_t *h_out;          // bf16 [rows, dim]
    int32_t *status;
    int rows, n_layers, dim, ffn, n_heads, n_kv, slots, sigma, max_pos, vocab, groups;
    float eps, scale;
    uint32_t first_wait, later_wait;
};

// ---- sizes --------------------------------------------------------------------------------
// A workgroup's share of a projection: `rows` output rows in tiles of 16; back wave b takes the scale groups
// [b stretch, (b + 1) stretch) of K.  `apart`: none for the rows' workgroups, whose row phase ends last: whole tiles for the
// others (half of them idle at 2048 rows; with eight rows each for all 256 everything waited for the rows' 0.8 - 1.3 us more).
struct Share {
    int k, groups, stretch, first, rows, tiles;
    bool pairs;
    int chunks, blocks;         // of a row's weights: 16 bytes, eight of those
    int weight_bytes, part_bytes, bytes;   // in LDS: weights, scales (of the gate or the up rows), all
    __host__ __device__ Share(int bits, int k_, int n, int wgs, bool pairs_, bool apart) {
        k = k_;
        pairs = pairs_;
        groups = k / 128;
        stretch = (groups + kBackWaves - 1) / kBackWaves;
        first = apart ? kRows : 0;
        if (apart) {
            rows = 16 * ((n + 16 * (wgs - kRows) - 1) / (16 * (wgs - kRows)));
        } else {
            const int values = pairs ? n / 2 : n;
            rows = 2 * ((values + 2 * wgs - 1) / (2 * wgs));
            if (pairs) rows *= 2;
        }
        tiles = (rows + 15) / 16;
        chunks = groups * bits;
        blocks = (chunks + 7) / 8;
        weight_bytes = tiles * blocks * 2048;
        part_bytes = ((pairs ? rows / 2 : rows) * groups * 2 + 255) & ~255;
        bytes = weight_bytes + (pairs ? 2 : 1) * part_bytes;
    }
};
__host__ __device__ inline int room_of(int wgs, int n_heads) {   // parts of a head's slots at most; the rows' workgroups have none
    const int room = (wgs - kRows) / n_heads;
    return room < kMaxSplits ? room : kMaxSplits;
}
struct Places {   // byte offsets in the exchange memory
    int64_t h, h2, qkv, inner, parts, q8, size;
    int layer8, o8, g8, d8, s8;   // int8 rows of a layer: q|k|v's at 0, then o's, gate|up's, down's, multipliers
    __host__ __device__ Places(int n_layers, int dim, int ffn, int n_heads, int n_kv, int wgs) {
        const int64_t pair = 4;   // bytes a value with its tag
        h = kControlBytes;
        h2 = h + kRows * dim * pair;
        qkv = h2 + kRows * dim * pair;
        inner = qkv + kRows * (int64_t)(n_heads + 2 * n_kv) * kHd * pair;
        parts = inner + kRows * ffn * pair;
        const int room = room_of(wgs, n_heads);
        q8 = parts + (int64_t)n_heads * room * kRows * kPartBytes;
        q8 = (q8 + 255) & ~(int64_t)255;
        o8 = kRows * dim;
        g8 = o8 + kRows * n_heads * kHd;
        d8 = g8 + kRows * dim;
        s8 = d8 + kRows * ffn;
        layer8 = s8 + 8 * kCopies * 128;   // a line a phase and copy, multipliers and announcements
        size = q8 + 2 * (int64_t)n_layers * layer8;   // two sets, in turn
    }
};
struct Lds {
    int wave, once, gate, resid, mult, size;   // `once`: weights of q|k|v, o and down in turn, `gate`: of gate|up
    // (tiles: at most, of the build, which computes as many everywhere)
    __host__ __device__ Lds(const Share &q, const Share &o, const Share &g, const Share &d, int q_dim, int build_tiles) {
        const auto most = [](int a, int b) { return a > b ? a : b; };
        wave = 1024 * most(4, build_tiles);   // a back wave's tokens, then its results
        const int att = 3 * kRows * kHd * 2 + kFrontWaves * 16 * kVPitch + kFrontWaves * kRows * kOPitch * 4 + 1024;
        once = (most(most(kBackWaves * wave, att), 2 * q_dim) + 255) & ~255;
        gate = once + most(q.bytes, most(o.bytes, d.bytes));
        resid = gate + g.bytes;
        mult = resid + 4 * kRows * o.rows;
        size = mult + 4 * kRows;
    }
};

// ---- rows as eight bytes a pair of values ----------------------------------------------------
__device__ __forceinline__ void hand_over(const __amdgpu_buffer_rsrc_t rows, int value, uint32_t d, uint32_t tag) {
    __builtin_amdgcn_raw_buffer_store_b64(v2u{d, tag}, rows, value * 4, 0, kDeviceScope);
}
__device__ __forceinline__ void hand_over_near(const __amdgpu_buffer_rsrc_t rows, int value, uint32_t d, uint32_t tag, bool near) {
    if (near)
        __builtin_amdgcn_raw_buffer_store_b64(v2u{d, tag}, rows, value * 4, 0, 0);
    else
        hand_over(rows, value, d, tag);
}
// (The check of the limit on its own, before the spins: with first_spin of step_one.hip.h in its place, which is right as
// well, a nine-row step of the 1.7B shape takes 643 us instead of 612.  A one-token step has it the other way round: 396
// with first_spin, 401 with this.)
__device__ __forceinline__ bool timed_out(int spins, uint32_t &since, uint32_t limit) {
    if (limit == 0) return true;
    return step_one::timed_out(spins, since, limit);
}
// Looks until good(x), two looks under way, half of one's time apart: for what few look at.
template <class T, class Ask, class Good>
__device__ __forceinline__ bool look(T &x, uint32_t limit, Ask ask, Good good) {
    T y;
    uint32_t since = 0;
    ask(x);
    for (int spins = 1;; ++spins) {
        __builtin_amdgcn_s_sleep(kNap);
        asm volatile("" ::: "memory");   // a look is a new one
        ask(y);
        __builtin_amdgcn_sched_barrier(0);
        if (good(x)) return true;
        __builtin_amdgcn_s_sleep(kNap);
        asm volatile("" ::: "memory");
        ask(x);
        __builtin_amdgcn_sched_barrier(0);
        if (good(y)) {
            x = y;
            return true;
        }
        if (timed_out(spins, since, limit)) return false;
    }
}
// .. and one, for what takes many registers.
template <class T, class Ask, class Good>
__device__ __forceinline__ bool look_singly(T &x, uint32_t limit, Ask ask, Good good) {
    uint32_t since = 0;
    for (int spins = 1;; ++spins) {
        asm volatile("" ::: "memory");
        ask(x);
        __builtin_amdgcn_sched_barrier(0);
        if (good(x)) return true;
        if (timed_out(spins, since, limit)) return false;
    }
}
// Words of eight values of a row: word tid + 256 i into v[i] (zero past the end).
template <int U>
__device__ __forceinline__ bool receive(const uint8_t *row, int words, uint32_t tag, v4u *v, uint32_t limit) {
    const int tid = afresh((int)threadIdx.x);
    const __amdgpu_buffer_rsrc_t r = rsrc_of(row, words * 32);
    for (int z = 0; z < kPause; ++z) __builtin_amdgcn_s_sleep(1);
    struct Both {
        v4u x[U], y[U];
    } both;
    const auto ask = [&](Both &b) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int off = wanted(tid + i * kFront < words, (tid + i * kFront) * 32);
            b.x[i] = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kDeviceScope);
            b.y[i] = __builtin_amdgcn_raw_buffer_load_b128(r, off, 16, kDeviceScope);
        }
    };
    const auto good = [&](const Both &b) {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < U; ++i)
            ok = ok & ((tid + i * kFront >= words) | ((b.x[i].y == tag) & (b.x[i].w == tag) & (b.y[i].y == tag) & (b.y[i].w == tag)));
        return (bool)__all(ok);
    };
    const bool ok = U == 1 ? look(both, limit, ask, good) : look_singly(both, limit, ask, good);
#pragma unroll
    for (int i = 0; i < U; ++i) v[i] = v4u{both.x[i].x, both.x[i].z, both.y[i].x, both.y[i].z};
    return ok;
}

// ---- int8 rows --------------------------------------------------------------------------------
// Eight neighbouring values, quantised with s, at word w of the row, in the order in which unpacked weights meet them: 16
// (sign: 32) values form 16-byte pieces whose dword j holds values j, 4 + j, 8 + j, 12 + j (sign: j, 8 + j, ..; second piece
// 4 + j, ..).
template <int BITS>
__device__ __forceinline__ void put_word(const __amdgpu_buffer_rsrc_t row, int w, const float *x, float s, bool ok) {
    uint32_t t[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)   // 1.5 2^23: rounds to nearest even, the integer is the low byte
        t[i] = __float_as_uint(__builtin_amdgcn_fmed3f(x[i] * s, -127.0f, 127.0f) + 12582912.0f);
    const auto pack = [&t](int i) {
        return __builtin_amdgcn_perm(t[i + 1], t[i], 0x0c0c0400u) | __builtin_amdgcn_perm(t[i + 3], t[i + 2], 0x04000c0cu);
    };
    const uint32_t w0 = pack(0), w1 = pack(4);
    const auto from = [](uint32_t v, auto ctrl) {
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xf, 0xf, true);
    };
    using Xor1 = std::integral_constant<int, bonsai_wave::kXor1>;
    using Xor2 = std::integral_constant<int, bonsai_wave::kXor2>;
    const bool odd = w & 1;
    if constexpr (BITS == 2) {
        // bytes j of both halves: this lane's are rows 2 (w & 1), + 1 of the piece's columns
        const uint32_t p01 = __builtin_amdgcn_perm(w1, w0, 0x05010400u), p23 = __builtin_amdgcn_perm(w1, w0, 0x07030602u);
        const uint32_t got = from(odd ? p01 : p23, Xor1{}), keep = odd ? p23 : p01;
        const uint32_t lo = odd ? got : keep, hi = odd ? keep : got;
        __builtin_amdgcn_raw_buffer_store_b64(v2u{__builtin_amdgcn_perm(hi, lo, 0x05040100u), __builtin_amdgcn_perm(hi, lo, 0x07060302u)}, row,
                                              wanted(ok, w * 8), 0, kDeviceScope);
    } else {
        const auto transpose = [&](uint32_t v) {   // 4 x 4 bytes over four lanes
            const uint32_t o = from(v, Xor1{});
            const uint32_t r = odd ? __builtin_amdgcn_perm(v, o, 0x07030501u) : __builtin_amdgcn_perm(o, v, 0x06020400u);
            const uint32_t u = from(r, Xor2{});
            return w & 2 ? __builtin_amdgcn_perm(r, u, 0x07060302u) : __builtin_amdgcn_perm(u, r, 0x05040100u);
        };
        const uint32_t a = transpose(w0), b = transpose(w1);
        // four lanes' first pieces, then their second ones, eight neighbouring bytes a lane: a line is written at once
        using First = std::integral_constant<int, 0x88>;    // quad_perm [0, 2, 0, 2]
        using Second = std::integral_constant<int, 0xDD>;   // quad_perm [1, 3, 1, 3]
        const uint32_t a0 = from(a, First{}), a1 = from(a, Second{}), b0 = from(b, First{}), b1 = from(b, Second{});
        __builtin_amdgcn_raw_buffer_store_b64(w & 2 ? v2u{b0, b1} : v2u{a0, a1}, row, wanted(ok, w * 8), 0, kDeviceScope);
    }
}

// ---- weights ------------------------------------------------------------------------------------
template <int BITS>
struct Piece;   // a lane's weights of one group: 32 of its row
template <>
struct Piece<2> {
    v2u w;
    __device__ __forceinline__ void read(const uint8_t *row, int g, int kb, int key) {   // piece of row `row`, group g
        w = *reinterpret_cast<const v2u *>(row + (g >> 2) * 2048 + ((((2 * g & 7) + (kb >> 1)) ^ key) * 16) + (kb & 1) * 8);
    }
    __device__ __forceinline__ v4i half(int i) const {
        const uint32_t p = i ? w.y : w.x;
        return v4i{(int)(p & 0x03030303u), (int)((p >> 2) & 0x03030303u), (int)((p >> 4) & 0x03030303u), (int)((p >> 6) & 0x03030303u)};
    }
    static constexpr int kOffset = (int)0xfefefefeu;   // what the codes are too large by, as weights
};
template <>
struct Piece<1> {
    uint32_t w;
    __device__ __forceinline__ void read(const uint8_t *row, int g, int kb, int key) {
        w = *reinterpret_cast<const uint32_t *>(row + (g >> 3) * 2048 + (((g & 7) ^ key) * 16) + kb * 4);
    }
    __device__ __forceinline__ v4i half(int i) const {   // bits as 0 and 2
        const uint32_t p = i ? w >> 3 : w << 1, q = i ? w >> 4 : w;
        return v4i{(int)(p & 0x02020202u), (int)(q & 0x02020202u), (int)((q >> 1) & 0x02020202u), (int)((q >> 2) & 0x02020202u)};
    }
    static constexpr int kOffset = (int)0xffffffffu;
};
template <int BITS, int S, int T>
struct Taken {   // weights of a wave's stretch: S groups of T row tiles
    static constexpr int kGroups = S, kTiles = T;
    Piece<BITS> w[S][T];
    uint32_t s[S][T];
};
// Sixteen rows of 128 bytes lie in 2 KB of LDS, row after row, the 16-byte pieces of row r at (piece ^ key_of(r)): sixteen
// rows' pieces fall into different banks.
__device__ __forceinline__ int key_of(int row) { return (row >> 1) & 7; }

// From memory to LDS without registers: lane i's `BYTES` at `off` go to lds + BYTES i.  In assembly because the compiler would
// wait for them before the next read of any LDS; who reads what has come waits by vmcnt and a barrier.  (m0 is read when the
// load is issued, and is left as it was.)
template <int BYTES>
__device__ __forceinline__ void fetch(const v4u from, int off, uint32_t lds) {
    uint32_t m0;
    if constexpr (BYTES == 16)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
                     : "=&s"(m0) : "s"(lds), "v"(off), "s"(from) : "memory");
    else
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dword %2, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
                     : "=&s"(m0) : "s"(lds), "v"(off), "s"(from) : "memory");
}
__device__ __forceinline__ v4u words_of(uintptr_t p, int bytes) {   // a buffer resource for it
    return v4u{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)p), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(p >> 32) & 0xffffu)),
               (uint32_t)__builtin_amdgcn_readfirstlane(bytes), 0x00020000u};
}
// A workgroup's weights and scales of a projection to `lds`, whole lines by eight lanes a row.  (Each lane its own row's pieces,
// into registers, takes the compute unit's address path 27 ns a request instead of 7, and everything else waited: 5 us a
// layer.)
// Row i of the share is row place(i) of n; the scales of its first `run` rows are those of neighbouring rows, of the others as
// well (pairs: of the gate rows, of the up rows).
template <class Place>
__device__ __forceinline__ void fetch_share(uintptr_t weights, uintptr_t scales, const Share &sh, int bw, int rows, int run, int n, Place place, int on,
                                            uint32_t lds) {
    if (!on || rows <= 0) return;
    const int lane = afresh((int)threadIdx.x & 63);
    const int row_bytes = sh.chunks * 16;
    const v4u rw = words_of(weights, n * row_bytes), rs = words_of(scales, n * sh.groups * 2);
    const int recip = 65536 / sh.blocks + 1;
    for (int i = bw; i < sh.tiles * sh.blocks * 2; i += kBackWaves) {
        const int tile = ((i >> 1) * recip) >> 16, block = (i >> 1) - tile * sh.blocks;
        const int r = (i & 1) * 8 + (lane >> 3), row = tile * 16 + r, chunk = block * 8 + ((lane & 7) ^ key_of(r));
        fetch<16>(rw, wanted(row < rows && chunk < sh.chunks, place(row) * row_bytes + chunk * 16), (uint32_t)__builtin_amdgcn_readfirstlane((int)lds + i * 1024));
    }
    const int row_scales = sh.groups * 2, bytes = (sh.pairs ? rows >> 1 : rows) * row_scales, parts = sh.part_bytes >> 8;
    const int from[2] = {place(0) * row_scales, place(sh.pairs ? 1 : run) * row_scales}, next = run * row_scales;
    for (int i = bw; i < (sh.pairs ? 2 * parts : parts); i += kBackWaves) {
        const int up = i >= parts, at = (i - up * parts) * 256 + lane * 4;
        const bool behind = !sh.pairs && at >= next;
        fetch<4>(rs, wanted(at < bytes, (up || behind ? from[1] : from[0]) + (behind ? at - next : at)),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)lds + sh.weight_bytes + i * 256));
    }
}

struct Common {
    const Args &a;
    int wg, lane, gqa, q_dim, n_qkv, m_rows;
    Share sq, so, sg, sd;
    int rows_q, rows_o, rows_g, rows_d;
    uint32_t epoch;
    bool attends, is_row, near;
    int n, hide, kvh, unit, split, head, per, splits, room;
    HeadOrder order;
    int head_row0;   // of the kv head's rows of q|k|v, the workgroup's first
    uint8_t *smem;
    int wave_bytes;
    const uint8_t *once, *gate;
    uint16_t *raw;
    float *resid, *mult;
    Meet &meet;
    uint8_t *h, *h2, *qkv, *inner, *parts, *q8, *q8_next;
    int layer8, o8, g8, d8, s8;
};

// ---- all waves: head rows of the attention ---------------------------------------------------
// Two rows a wave, a query's by lanes 0 - 31 and the key's by 32 - 63; lane i has dims 2 i, 2 i + 1 and, 64 further, their
// partners.
struct Rope {
    uint32_t c0, c1, s0, s1;   // of the wave's token
    uint32_t w0, w1;           // norm weights of the layer
    __device__ __forceinline__ void ask(const v2u &table) {
        const int lane = afresh((int)threadIdx.x & 63);
        const __amdgpu_buffer_rsrc_t q = rsrc_of(reinterpret_cast<const void *>(address(table, 10)), 2 * kHd);
        const __amdgpu_buffer_rsrc_t k = rsrc_of(reinterpret_cast<const void *>(address(table, 11)), 2 * kHd);
        const int i = 4 * (lane & 31), iq = wanted(lane < 32, i), ik = wanted(lane >= 32, i);
        w0 = __builtin_amdgcn_raw_buffer_load_b32(q, iq, 0, 0) | __builtin_amdgcn_raw_buffer_load_b32(k, ik, 0, 0);
        w1 = __builtin_amdgcn_raw_buffer_load_b32(q, iq, 128, 0) | __builtin_amdgcn_raw_buffer_load_b32(k, ik, 128, 0);
    }
};
__device__ __forceinline__ double sum32(double v) {
    using bonsai_wave::partner;
    v += partner<bonsai_wave::kXor1>(v);
    v += partner<bonsai_wave::kXor2>(v);
    v += partner<bonsai_wave::kHalfMirror>(v);
    v += partner<bonsai_wave::kMirror>(v);
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)b, (uint32_t)b, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    return __longlong_as_double((long long)(((uint64_t)hi[0] << 32) | lo[0])) + __longlong_as_double((long long)(((uint64_t)hi[1] << 32) | lo[1]));
}
// Wave `wave` of the workgroup brings row `wave` of the block: the query, normed and rotated, and where the part holds rows
// of the block itself, key and value, which the first query head's workgroup also stores to the workspace.
__device__ __forceinline__ bool head_rows(const Common &c, int l, int wave, const Rope &rope, uint32_t tag, uint32_t limit) {
    uint32_t *q_lds = reinterpret_cast<uint32_t *>(c.smem), *k_lds = q_lds + kRows * kHd / 2, *v_lds = k_lds + kRows * kHd / 2;
    if (wave >= c.m_rows) return true;
    const int lane = c.lane, word = lane & 31;
    const bool key = lane >= 32, own = (c.split + 1) * c.per > c.n;
    const __amdgpu_buffer_rsrc_t r = rsrc_of(c.qkv + (size_t)wave * c.n_qkv * 4, c.n_qkv * 4);
    const int of_head = c.kvh * c.order.rows() * 4;
    const int at = of_head + (key ? c.gqa : c.head - c.kvh * c.gqa) * 512 + word * 8;
    struct In {
        v2u lo, hi, v;
    } in;
    if (!look(in, limit, [&](In &t) {
            t.lo = __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, kDeviceScope);
            t.hi = __builtin_amdgcn_raw_buffer_load_b64(r, at, 256, kDeviceScope);
            t.v = __builtin_amdgcn_raw_buffer_load_b64(r, lane * 8, of_head + (c.gqa + 1) * 512, kDeviceScope);
        }, [&](const In &t) { return (bool)__all(((t.lo.y == tag) & (t.hi.y == tag) & (t.v.y == tag)) | (!own & (key | ((t.lo.y == tag) & (t.hi.y == tag))))); }))
        return false;
    const auto lo_of = [](uint32_t p) { return __uint_as_float(p << 16); };
    const auto hi_of = [](uint32_t p) { return __uint_as_float(p & 0xffff0000u); };
    const float f0 = lo_of(in.lo.x), f1 = hi_of(in.lo.x), g0 = lo_of(in.hi.x), g1 = hi_of(in.hi.x);
    const double ss = sum32(((double)(f0 * f0) + (double)(g0 * g0)) + ((double)(f1 * f1) + (double)(g1 * g1)));
    const float var = (float)ss / (float)kHd;
    const float rs = 1.0f / sqrtf(var + c.a.eps);
    const uint32_t t0 = pack_bf16(f0 * rs, f1 * rs), t1 = pack_bf16(g0 * rs, g1 * rs);
    const uint32_t n0 = pack_bf16(lo_of(rope.w0) * lo_of(t0), hi_of(rope.w0) * hi_of(t0));
    const uint32_t n1 = pack_bf16(lo_of(rope.w1) * lo_of(t1), hi_of(rope.w1) * hi_of(t1));
    // rotate_half(n) = [-n1, n0]
    const uint32_t a0 = pack_bf16(lo_of(n0) * lo_of(rope.c0), hi_of(n0) * hi_of(rope.c0)), b0 = pack_bf16(-lo_of(n1) * lo_of(rope.s0), -hi_of(n1) * hi_of(rope.s0));
    const uint32_t a1 = pack_bf16(lo_of(n1) * lo_of(rope.c1), hi_of(n1) * hi_of(rope.c1)), b1 = pack_bf16(lo_of(n0) * lo_of(rope.s1), hi_of(n0) * hi_of(rope.s1));
    const uint32_t o0 = pack_bf16(lo_of(a0) + lo_of(b0), hi_of(a0) + hi_of(b0)), o1 = pack_bf16(lo_of(a1) + lo_of(b1), hi_of(a1) + hi_of(b1));
    uint32_t *to = (key ? k_lds : q_lds) + wave * (kHd / 2) + word;
    to[0] = o0;
    to[32] = o1;
    if (own) {
        v_lds[wave * (kHd / 2) + lane] = in.v.x;
        const int slot = c.n + wave;   // its place among the slots
        if (slot >= c.split * c.per && slot < (c.split + 1) * c.per && c.unit == c.split * c.gqa) {
            uint32_t *kv = reinterpret_cast<uint32_t *>(c.a.kv + ((size_t)l * c.a.n_kv + c.kvh) * c.a.slots * kHd + (size_t)(c.a.sigma + wave) * kHd);
            if (key) {
                kv[word] = o0;
                kv[word + 32] = o1;
            }
            kv[(size_t)c.a.n_layers * c.a.n_kv * c.a.slots * (kHd / 2) + lane] = in.v.x;
        }
    }
    return true;
}
__device__ __forceinline__ float *att_out(const Common &c) {
    return reinterpret_cast<float *>(c.smem + 3 * kRows * kHd * 2 + kFrontWaves * 16 * kVPitch);
}
// The four front waves' sums of a (head, part) together, a thread two dims of a row, into the parts.
__device__ __forceinline__ void store_part(const Common &c, uint32_t tag) {
    const int tid = afresh((int)threadIdx.x);
    const int row = tid >> 6, d = (tid & 63) * 2;
    if (row >= c.m_rows) return;
    const float *o = att_out(c), *ml = o + kFrontWaves * kRows * kOPitch;
    float m = -INFINITY, sum = 0.0f, o0 = 0.0f, o1 = 0.0f;
#pragma unroll
    for (int w = 0; w < kFrontWaves; ++w) m = fmaxf(m, ml[(w * kRows + row) * 2]);
    const float base = m == -INFINITY ? 0.0f : m;
#pragma unroll
    for (int w = 0; w < kFrontWaves; ++w) {
        const float f = __builtin_amdgcn_exp2f(ml[(w * kRows + row) * 2] - base);
        sum += f * ml[(w * kRows + row) * 2 + 1];
        o0 += f * o[(w * kRows + row) * kOPitch + d];
        o1 += f * o[(w * kRows + row) * kOPitch + d + 1];
    }
    const __amdgpu_buffer_rsrc_t r = rsrc_of(c.parts + (size_t)(c.head * c.room + c.split) * kRows * kPartBytes, kRows * kPartBytes);
    __builtin_amdgcn_raw_buffer_store_b128(v4u{__float_as_uint(o0), tag, __float_as_uint(o1), tag}, r, row * kPartBytes + d * 8, 0, kDeviceScope);
    if (d == 0)
        __builtin_amdgcn_raw_buffer_store_b128(v4u{__float_as_uint(m), tag, __float_as_uint(sum), tag}, r, row * kPartBytes + kHd * 8, 0, kDeviceScope);
}
// Row workgroup: beside the row's int8 values its multiplier ..
__device__ __forceinline__ void raise(const Common &c, int phase, uint8_t *rows8, float s) {
    const int tid = afresh((int)threadIdx.x);
    if (tid < kCopies)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s), rsrc_of(rows8 + c.s8 + phase * kCopies * 128, kCopies * 128), tid * 128 + c.wg * 4,
                                              0, kDeviceScope);
}
// .. and, half a microsecond or more before it, that the row is about to come.  The back waves look for the rows from then on:
// all 256 workgroups' looking from the start takes the memory's bandwidth from what they look for, and looking only behind
// the multipliers costs a look.
__device__ __forceinline__ void announce(const Common &c, int phase, uint8_t *rows8) { raise(c, 4 + phase, rows8, 0.0f); }

// The parts of row `wg`, all heads, into the raw row.
__device__ __forceinline__ bool merge_parts(const Common &c, uint32_t tag, uint32_t limit) {
    const int tid = afresh((int)threadIdx.x);
    const int d = (tid & 63) * 2;
    const size_t part = (size_t)kRows * kPartBytes;
    for (int head = __builtin_amdgcn_readfirstlane(tid >> 6); head < c.a.n_heads; head += kThreads / 64) {
        const __amdgpu_buffer_rsrc_t r = rsrc_of(c.parts + (size_t)head * c.room * part + (size_t)c.wg * kPartBytes, (int)(c.room * part));
        float m = -INFINITY, sum = 0.0f, o0 = 0.0f, o1 = 0.0f;
        const auto add = [&](int p, auto parts_c) -> bool {   // parts p ..
            constexpr int N = decltype(parts_c)::value;
            struct Parts {
                v4u x[N], y[N];
            } in;
            const auto ask = [&](Parts &t) {
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const int at = (p + i) * (int)part;
                    t.x[i] = __builtin_amdgcn_raw_buffer_load_b128(r, at + d * 8, 0, kDeviceScope);
                    t.y[i] = __builtin_amdgcn_raw_buffer_load_b128(r, at + kHd * 8, 0, kDeviceScope);
                }
            };
            const auto good = [&](const Parts &t) {
                bool ok = true;
#pragma unroll
                for (int i = 0; i < N; ++i) ok = ok & ((t.x[i].y == tag) & (t.x[i].w == tag) & (t.y[i].y == tag) & (t.y[i].w == tag));
                return (bool)__all(ok);
            };
            if (!(N == 1 ? look(in, limit, ask, good) : look_singly(in, limit, ask, good))) return false;
            float top = m;
#pragma unroll
            for (int i = 0; i < N; ++i) top = fmaxf(top, __uint_as_float(in.y[i].x));
            const float base = top == -INFINITY ? 0.0f : top;
            const float keep = __builtin_amdgcn_exp2f(m - base);
            m = top;
            sum *= keep;
            o0 *= keep;
            o1 *= keep;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const float f = __builtin_amdgcn_exp2f(__uint_as_float(in.y[i].x) - base);
                sum += f * __uint_as_float(in.y[i].z);
                o0 += f * __uint_as_float(in.x[i].x);
                o1 += f * __uint_as_float(in.x[i].z);
            }
            return true;
        };
        int p = 0;
        for (; p + 4 <= c.splits; p += 4)
            if (!add(p, std::integral_constant<int, 4>{})) return false;
        if (p + 2 <= c.splits) {
            if (!add(p, std::integral_constant<int, 2>{})) return false;
            p += 2;
        }
        if (p < c.splits && !add(p, std::integral_constant<int, 1>{})) return false;
        const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
        *reinterpret_cast<uint32_t *>(c.raw + head * kHd + d) = pack_bf16(o0 * inv, o1 * inv);
    }
    return true;
}

// Int8 rows' lines of N groups: lanes 8 r .. 8 r + 7 have rows r and r + 8.
template <int N>
struct Lines {
    v4u v[N][2];
    __device__ __forceinline__ bool look_for(const __amdgpu_buffer_rsrc_t rows, int k, int m_rows, int group, int groups, uint32_t limit) {
        const int lane = afresh((int)threadIdx.x & 63);
        return look_singly(*this, limit, [&](Lines &t) {
#pragma unroll
            for (int j = 0; j < N; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int row = (lane >> 3) + 8 * h;
                    t.v[j][h] = __builtin_amdgcn_raw_buffer_load_b128(rows, wanted(row < m_rows && j < groups, row * k + (group + j) * 128 + (lane & 7) * 16),
                                                                      0, kDeviceScope);
                }
        }, [](const Lines &t) {
            uint32_t least = ~0u;
#pragma unroll
            for (int j = 0; j < N; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    least = min(min(least, t.v[j][h].x ^ kEmpty), t.v[j][h].y ^ kEmpty);
                    least = min(min(least, t.v[j][h].z ^ kEmpty), t.v[j][h].w ^ kEmpty);
                }
            return (bool)__all(least != 0u);
        });
    }
};

// ---- back waves ---------------------------------------------------------------------------------
__device__ __forceinline__ float silu_mul(float g, float u) { return step_one::silu_mul(g, u); }

template <int BITS, int SQ, int TQ, int SO, int SG, int TG, int SD>
__device__ __forceinline__ bool back(const Common &c, int bw, Rope rope) {
    const Args &a = c.a;
    const auto lds_of = [](const uint8_t *p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t *)p; };
    const auto from = [&](const Share &sh) { return [&](int row) { return (c.wg - sh.first) * sh.rows + row; }; };
    const auto head_row = [&](int row) { return c.order.row_of(c.kvh, c.head_row0 + row); };
    const auto in_turn = [&](int row) { return c.wg * c.sg.rows / 2 + (row & 1) * a.ffn + (row >> 1); };   // gate, up
    const auto fetch_q = [&](const v2u &t, int on) { fetch_share(address(t, 0), address(t, 4), c.sq, bw, c.rows_q, kHd - c.head_row0 % kHd, c.n_qkv, head_row, on, lds_of(c.once)); };
    const auto fetch_o = [&](const v2u &t) { fetch_share(address(t, 1), address(t, 5), c.so, bw, c.rows_o, c.rows_o, a.dim, from(c.so), 1, lds_of(c.once)); };
    const auto fetch_g = [&](const v2u &t) { fetch_share(address(t, 2), address(t, 6), c.sg, bw, c.rows_g, c.rows_g, 2 * a.ffn, in_turn, 1, lds_of(c.gate)); };
    const auto fetch_d = [&](const v2u &t) { fetch_share(address(t, 3), address(t, 7), c.sd, bw, c.rows_d, c.rows_d, a.dim, from(c.sd), 1, lds_of(c.once)); };
    v2u cur = ask_layer(a, 0);
    fetch_q(cur, 1);
    rope.ask(cur);

    // The wave's stretch of K.  The weights of it go from LDS into registers while the rows are waited for.
    const auto take = [&](auto &wt, const Share &sh, const uint8_t *w) {
        constexpr int S = std::decay_t<decltype(wt)>::kGroups, T = std::decay_t<decltype(wt)>::kTiles;
        const int lane = afresh(c.lane), row = lane & 15, kb = lane >> 4;
#pragma unroll
        for (int i = 0; i < S; ++i) {
            const int g = bw * sh.stretch + i;
            if (i >= sh.stretch || g >= sh.groups) break;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int n = t * 16 + row;   // its row of the share
                wt.w[i][t].read(w + t * sh.blocks * 2048 + row * 128, g, kb, key_of(row));
                wt.s[i][t] = *reinterpret_cast<const uint16_t *>(
                    w + sh.weight_bytes + (sh.pairs ? (n & 1) * sh.part_bytes + ((n >> 1) * sh.groups + g) * 2 : (n * sh.groups + g) * 2));
            }
        }
    };
    // The tokens come from the int8 rows at `rows8` as whole lines and go by the wave's own LDS into the matrix cores' order (lane
    // by lane each row's piece took 0.8 us at K = 2048 and 1.9 us at 6144, whatever cache they came from), the results to
    // the same LDS, [wave][tile][token][row].
    const auto multiply = [&](const auto &wt, const Share &sh, const uint8_t *rows8, uint32_t limit) {
        constexpr int S = std::decay_t<decltype(wt)>::kGroups, T = std::decay_t<decltype(wt)>::kTiles;
        constexpr int kAhead = S < 4 ? (S + 1) / 2 * 2 : 4;   // groups requested together
        const int lane = afresh(c.lane);
        uint8_t *const mine = c.smem + bw * c.wave_bytes;
        const __amdgpu_buffer_rsrc_t ra = rsrc_of(rows8, c.m_rows * sh.k);
        const v4i acc_zero = v4i{0, 0, 0, 0}, ones = v4i{Piece<BITS>::kOffset, Piece<BITS>::kOffset, Piece<BITS>::kOffset, Piece<BITS>::kOffset};
        float acc[T][4];
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][i] = 0.0f;
        const int row = lane & 15, kb = lane >> 4, key = key_of(row), put_row = lane >> 3;
        const int first = bw * sh.stretch, groups = sh.groups - first < sh.stretch ? sh.groups - first : sh.stretch;
#pragma unroll
        for (int from = 0; from < S; from += kAhead) {
            if (from >= groups) break;
            Lines<kAhead> x;
            if (!x.look_for(ra, sh.k, c.m_rows, first + from, groups - from, limit) && lane == 0) c.meet.bad = 1;
#pragma unroll
            for (int two = 0; two < kAhead; two += 2) {
                if (from + two >= groups) break;
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int r = put_row + 8 * h;
                        *reinterpret_cast<v4u *>(mine + j * 2048 + r * 128 + ((lane & 7) ^ key_of(r)) * 16) = x.v[two + j][h];
                    }
                v4i a0[2], a1[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const uint8_t *at = mine + j * 2048 + row * 128;
                    a0[j] = *reinterpret_cast<const v4i *>(at + ((2 * kb) ^ key) * 16);
                    a1[j] = *reinterpret_cast<const v4i *>(at + ((2 * kb + 1) ^ key) * 16);
                }
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int i = from + two + j;
                    if (i >= S || i >= groups) break;
                    v4i less = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0[j], ones, acc_zero, 0, 0, 0);
                    less = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1[j], ones, less, 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0[j], wt.w[i][t].half(0), less, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1[j], wt.w[i][t].half(1), d, 0, 0, 0);
                        const float ws = __uint_as_float(wt.s[i][t] << 16);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[t][e] += (float)d[e] * ws;
                    }
                }
            }
        }
        float *const out = reinterpret_cast<float *>(mine);
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) out[(t * 16 + kb * 4 + e) * 16 + row] = acc[t][e];
    };
    // A projection of the int8 rows `rows8`: W neighbouring rows of a token, added up over the waves, are one thread's,
    // done(token, row, values, the token's multiplier).
    const auto project = [&](auto wt_c, auto w_c, const Share &sh, int rows, const uint8_t *rows8, const uint8_t *w, uint32_t limit,
                             auto done) -> bool {
        constexpr int W = decltype(w_c)::value;
        typedef float Vec __attribute__((ext_vector_type(W)));
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the wave's part of the weights is there
        __syncthreads();                                  // all of them are
        std::decay_t<decltype(wt_c)> wt;
        take(wt, sh, w);
        __syncthreads();   // the rows' multipliers are there
        if (given_up(c.meet)) return false;
        multiply(wt, sh, rows8, limit);
        const int t = afresh((int)threadIdx.x) - kFront;
        const int per_token = rows / W, total = per_token * c.m_rows;
        const int recip = 65536 / per_token + 1;
        __syncthreads();
        if (given_up(c.meet)) return false;
        for (int e = t; e < total; e += kBack) {
            const int token = (e * recip) >> 16, row = (e - token * per_token) * W;
            const float *p = reinterpret_cast<const float *>(c.smem) + ((row >> 4) * 16 + token) * 16 + (row & 15);
            constexpr int kAtOnce = 12 / W * 2;   // reads under way
            const float s = c.mult[token];
            Vec v;
#pragma unroll
            for (int from = 0; from < kBackWaves; from += kAtOnce) {
                Vec part[kAtOnce];
#pragma unroll
                for (int w = 0; w < kAtOnce && from + w < kBackWaves; ++w) part[w] = *reinterpret_cast<const Vec *>(p + (from + w) * (c.wave_bytes >> 2));
#pragma unroll
                for (int w = 0; w < kAtOnce && from + w < kBackWaves; ++w) v = from + w == 0 ? part[0] : v + part[w];
                __builtin_amdgcn_sched_barrier(0);
            }
            done(token, row, v, s);
        }
        __syncthreads();   // the results are on their way
        return true;
    };
    // the next step's place of int8 row `wg`, multiplier included
    const auto empty_row = [&](int l) {
        const int t = afresh((int)threadIdx.x) - kFront;
        const auto fill = [&](int at, int bytes) {
            const __amdgpu_buffer_rsrc_t r = rsrc_of(c.q8_next + (size_t)l * c.layer8 + at + c.wg * bytes, bytes);
            for (int i = t * 16; i < bytes; i += kBack * 16)
                __builtin_amdgcn_raw_buffer_store_b128(v4u{kEmpty, kEmpty, kEmpty, kEmpty}, r, i, 0, kDeviceScope);
        };
        fill(0, a.dim);
        fill(c.o8, c.q_dim);
        fill(c.g8, a.dim);
        fill(c.d8, a.ffn);
        if (t < 8 * kCopies)
            __builtin_amdgcn_raw_buffer_store_b32(kEmpty, rsrc_of(c.q8_next + (size_t)l * c.layer8 + c.s8, 8 * kCopies * 128), t * 128 + c.wg * 4, 0, kDeviceScope);
    };
    for (int layer = 0; layer < a.n_layers; ++layer) {
        const int l = afresh_scalar(layer);
        const uint32_t limit = l == 0 ? a.first_wait : a.later_wait;
        const int more = l + 1 < a.n_layers;
        const v2u nxt = ask_layer(a, more ? l + 1 : l);
        const uint32_t tag = c.epoch * (uint32_t)a.n_layers + (uint32_t)l + 1u;
        uint8_t *const rows8 = c.q8 + (size_t)l * c.layer8;
        typedef std::integral_constant<int, 2> Two;

        if (c.is_row) {   // norm + quantise: sums, maximum
            __syncthreads();
            if (given_up(c.meet)) return false;
            __syncthreads();
        }
        if (c.rows_q) {
            const __amdgpu_buffer_rsrc_t to = rsrc_of(c.qkv, kRows * c.n_qkv * 4);
            const int at_q = c.kvh * c.order.rows() + c.head_row0;
            if (!project(Taken<BITS, SQ, TQ>{}, Two{}, c.sq, c.rows_q, rows8, c.once, limit,
                         [&](int token, int row, auto v, float s) {
                             hand_over_near(to, token * c.n_qkv + at_q + row, pack_bf16(v[0] / s, v[1] / s), tag, c.near);
                         }))
                return false;
        }
        if (c.wg < kRows) empty_row(l);

        if (c.attends) {
            if (!head_rows(c, l, kFrontWaves + bw, rope, tag, limit) && c.lane == 0) c.meet.bad = 1;
            __syncthreads();   // the rows are in LDS
            if (given_up(c.meet)) return false;
            __syncthreads();   // the front waves' sums
            store_part(c, tag);
        }
        fetch_o(cur);
        fetch_g(cur);
        if (c.is_row) {
            if (!merge_parts(c, tag, limit) && c.lane == 0) c.meet.bad = 1;
            __syncthreads();   // the raw row
            if (given_up(c.meet)) return false;
            __syncthreads();   // maximum
        }
        const auto add = [&](const Share &sh, uint8_t *rows_to, bool last, uint32_t new_tag) {
            const __amdgpu_buffer_rsrc_t to = rsrc_of(rows_to, kRows * a.dim * 4);
            return [&, to, last, new_tag](int token, int row, auto v, float s) {
                float *res = c.resid + token * c.so.rows + row;
                const float h0 = bf16_round(bf16_round(v[0] / s) + res[0]), h1 = bf16_round(bf16_round(v[1] / s) + res[1]);
                res[0] = h0;
                res[1] = h1;
                const int at = token * a.dim + (c.wg - sh.first) * sh.rows + row;
                if (last)
                    *reinterpret_cast<uint32_t *>(a.h_out + at) = pack_bf16(h0, h1);
                else
                    hand_over(to, at, pack_bf16(h0, h1), new_tag);
            };
        };
        if (c.rows_o && !project(Taken<BITS, SO, 1>{}, Two{}, c.so, c.rows_o, rows8 + c.o8, c.once, limit,
                                 add(c.so, c.h2, false, tag)))
            return false;
        fetch_d(cur);

        if (c.is_row) {
            __syncthreads();
            if (given_up(c.meet)) return false;
            __syncthreads();
        }
        if (c.rows_g) {
            const __amdgpu_buffer_rsrc_t to = rsrc_of(c.inner, kRows * a.ffn * 4);
            if (!project(Taken<BITS, SG, TG>{}, std::integral_constant<int, 4>{}, c.sg, c.rows_g, rows8 + c.g8, c.gate, limit, [&](int token, int row, auto v, float s) {
                             const float i0 = silu_mul(bf16_round(v[0] / s), bf16_round(v[1] / s));
                             const float i1 = silu_mul(bf16_round(v[2] / s), bf16_round(v[3] / s));
                             hand_over(to, token * a.ffn + (c.wg * c.sg.rows + row) / 2, pack_bf16(i0, i1), tag);
                         }))
                return false;
        }
        rope.ask(nxt);

        if (c.is_row) {
            __syncthreads();   // maximum
            if (given_up(c.meet)) return false;
        }
        if (c.rows_d && !project(Taken<BITS, SD, 1>{}, Two{}, c.sd, c.rows_d, rows8 + c.d8, c.once, limit,
                                 add(c.sd, c.h, !more, tag + 1u)))
            return false;
        fetch_q(nxt, more);
        cur = nxt;
    }
    return true;
}

// ---- front waves --------------------------------------------------------------------------------
// ROW: of a row's workgroup, which has no part of the attention.
template <int BITS, int UD, int UQ, int UF, bool ROW>
__device__ __forceinline__ bool front(const Common &c, int wave, Rope rope) {
    const Args &a = c.a;
    const int tid = threadIdx.x, lane = c.lane, n = c.n;
    v2u cur = ask_layer(a, 0);
    v4u ln1[UD], ln2[UD];
    const auto ask_norm = [&](v4u *v, const v2u &t, int which) {
        const __amdgpu_buffer_rsrc_t r = rsrc_of(reinterpret_cast<const void *>(address(t, 8 + which)), 2 * a.dim);
        const int at = afresh(tid);
#pragma unroll
        for (int i = 0; i < UD; ++i)
            v[i] = __builtin_amdgcn_raw_buffer_load_b128(r, wanted(at + i * kFront < (a.dim >> 3), (at + i * kFront) * 16), 0, 0);
    };
    // Keys and values of the wave's sixteen slots of a chunk of 64: keys as rows of A, sixteen slots by eight dims of 32 a
    // lane; values four slots a load, sixteen lanes a slot.
    const int slot0 = c.split * c.per + wave * 16;
    v4u keys[4], vals[4];
    const auto ask_history = [&](int l, int at, int on) {
        const size_t plane = (size_t)a.n_kv * a.slots * kHd;
        const uint16_t *k = a.kv + (size_t)l * plane + (size_t)c.kvh * a.slots * kHd;
        const int bytes = on ? n * 256 : 0;
        const __amdgpu_buffer_rsrc_t rk = rsrc_of(k, bytes), rv = rsrc_of(k + (size_t)a.n_layers * plane, bytes);
        const int i = afresh(lane);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            keys[j] = __builtin_amdgcn_raw_buffer_load_b128(rk, (at + (i & 15)) * 256 + j * 64 + (i >> 4) * 16, 0, 0);
            vals[j] = __builtin_amdgcn_raw_buffer_load_b128(rv, (at + (i >> 4) + 4 * j) * 256 + (i & 15) * 16, 0, 0);
        }
    };
    if constexpr (ROW) {
        ask_norm(ln1, cur, 0);
    } else {
        rope.ask(cur);
        if (c.attends) ask_history(0, slot0, 1);
    }
    // what row (lane & 15) sees of the block
    const auto in = (const __attribute__((address_space(1))) int32_t *)(uintptr_t)a.step_in;
    const uint32_t sees = (lane & 15) < c.m_rows ? (uint32_t)in[2 + (lane & 15)] : 0u;

    const auto norm_row = [&](const v4u *v, const v4u *w, bool ok, uint8_t *rows8, int at8, int phase) -> bool {
        float f[UD][8];
        if (!step_one::norm<UD>(c.meet, v, w, a.dim, a.eps, wave, lane, ok, f)) return false;
        const float s = multiplier(c.meet);
        const int t = afresh(tid);
#pragma unroll
        for (int i = 0; i < UD; ++i)
            put_word<BITS>(rsrc_of(rows8 + at8 + c.wg * a.dim, a.dim), t + i * kFront, f[i], s, t + i * kFront < (a.dim >> 3));
        raise(c, phase, rows8, s);
        return true;
    };
    const auto quant_row = [&](const v4u *v, auto units_c, int k, bool ok, uint8_t *rows8, int at8, int phase) -> bool {
        const float top = top_of<decltype(units_c)::value>(v);
        if (lane == 0) {
            c.meet.top[wave] = top;
            if (!ok) c.meet.bad = 1;
        }
        __syncthreads();
        if (given_up(c.meet)) return false;
        const float s = multiplier(c.meet);
        const int t = afresh(tid);
#pragma unroll
        for (int i = 0; i < decltype(units_c)::value; ++i) {
            float f[8];
            unpack_word(v[i], f);
            put_word<BITS>(rsrc_of(rows8 + at8 + c.wg * k, k), t + i * kFront, f, s, t + i * kFront < (k >> 3));
        }
        raise(c, phase, rows8, s);
        return true;
    };
    // all rows' multipliers
    const auto wait_rows = [&](int phase, const uint8_t *rows8, uint32_t &x, uint32_t limit) -> bool {
        const __amdgpu_buffer_rsrc_t r = rsrc_of(rows8 + c.s8 + (phase * kCopies + c.wg % kCopies) * 128, kRows * 4);
        return look(x, limit, [&](uint32_t &t) { t = __builtin_amdgcn_raw_buffer_load_b32(r, wanted(lane < c.m_rows, lane * 4), 0, kDeviceScope); },
                    [](const uint32_t &t) { return (bool)__all(t != kEmpty); });
    };
    const auto project = [&](int phase, const uint8_t *rows8, uint32_t limit, auto meanwhile) -> bool {
        uint32_t x;
        __syncthreads();   // the weights are there
        if (!ROW && wave == 0 && !wait_rows(4 + phase, rows8, x, limit) && lane == 0) c.meet.bad = 1;
        __syncthreads();
        if (given_up(c.meet)) return false;
        if (wave == 0) {
            if (!wait_rows(phase, rows8, x, limit) && lane == 0) c.meet.bad = 1;
            if (lane < kRows) c.mult[lane] = __uint_as_float(x);
        }
        meanwhile();
        __syncthreads();   // the back waves' units
        if (given_up(c.meet)) return false;
        __syncthreads();   // and results
        return true;
    };

    for (int layer = 0; layer < a.n_layers; ++layer) {
        const int l = afresh_scalar(layer);
        const uint32_t limit = l == 0 ? a.first_wait : a.later_wait;
        const int more = l + 1 < a.n_layers;
        const v2u nxt = ask_layer(a, more ? l + 1 : l);
        const uint32_t tag = c.epoch * (uint32_t)a.n_layers + (uint32_t)l + 1u;
        uint8_t *const rows8 = c.q8 + (size_t)l * c.layer8;

        if constexpr (ROW) {
            v4u row[UD];
            bool ok = true;
            if (l == 0) {
                const uint32_t token = (uint32_t)in[2 + 2 * c.m_rows + c.wg];
                const __amdgpu_buffer_rsrc_t r = rsrc_of(a.embed + (size_t)(token < (uint32_t)a.vocab ? token : (uint32_t)a.vocab - 1) * a.dim, 2 * a.dim);
#pragma unroll
                for (int i = 0; i < UD; ++i) row[i] = __builtin_amdgcn_raw_buffer_load_b128(r, wanted(tid + i * kFront < (a.dim >> 3), (tid + i * kFront) * 16), 0, 0);
            } else {
                ok = receive<UD>(c.h + (size_t)c.wg * a.dim * 4, a.dim >> 3, tag, row, limit);
            }
            announce(c, 0, rows8);
            if (!norm_row(row, ln1, ok, rows8, 0, 0)) return false;
            ask_norm(ln2, cur, 1);
        }
        if (c.rows_q && !project(0, rows8, limit, [] {})) return false;

        // ---- attention of the block's rows to one head's slots, or a part of them; S^T = K Q^T and O^T = V^T P^T, so that
        // a lane owns one row and the probabilities go from the softmax into the next product
        if (!ROW && c.attends) {
            if (!head_rows(c, l, wave, rope, tag, limit) && lane == 0) c.meet.bad = 1;
            __syncthreads();
            if (given_up(c.meet)) return false;
            const uint16_t *q_lds = reinterpret_cast<const uint16_t *>(c.smem), *k_lds = q_lds + kRows * kHd, *v_lds = k_lds + kRows * kHd;
            uint8_t *v_tile = c.smem + 3 * kRows * kHd * 2 + wave * 16 * kVPitch;
            const int al = afresh(lane), row = al & 15, kb = al >> 4;
            float m_run = -INFINITY, l_run = 0.0f;
            v4f o[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) o[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            const float to_log2 = a.scale * 1.44269504088896341f;
            for (int at = 0; at < c.per && c.split * c.per + at < n + c.m_rows; at += 64) {
                if (at) ask_history(l, slot0 + at, 1);
                const int first = slot0 + at;
                if (first + 16 > n) {   // rows of the block itself
                    const int own = first + row - n;
                    if (own >= 0)
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            keys[j] = own < c.m_rows ? *reinterpret_cast<const v4u *>(k_lds + own * kHd + j * 32 + kb * 8) : v4u{0, 0, 0, 0};
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int mine = first + kb + 4 * j - n;
                        if (mine >= 0) vals[j] = mine < c.m_rows ? *reinterpret_cast<const v4u *>(v_lds + mine * kHd + row * 8) : v4u{0, 0, 0, 0};
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) *reinterpret_cast<v4u *>(v_tile + (kb + 4 * j) * kVPitch + row * 16) = vals[j];
                v4f sc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(attn_as_bf16x8(uint4{keys[j].x, keys[j].y, keys[j].z, keys[j].w}),
                                                                 attn_as_bf16x8(*reinterpret_cast<const uint4 *>(q_lds + row * kHd + j * 32 + kb * 8)), sc, 0, 0, 0);
                float m = -INFINITY;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int slot = first + kb * 4 + r, own = slot - n;
                    const bool see = own < 0 ? slot != c.hide : (own < c.m_rows && ((sees >> own) & 1u));
                    sc[r] = see ? sc[r] * to_log2 : -INFINITY;
                    m = fmaxf(m, sc[r]);
                }
                step_one::Pair p = pair16(m);
                p = pair32(fmaxf(p.a, p.b));
                m = fmaxf(m_run, fmaxf(p.a, p.b));
                const float base = m == -INFINITY ? 0.0f : m;
                const float keep = __builtin_amdgcn_exp2f(m_run - base);
                m_run = m;
                float w[4];
                l_run *= keep;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    w[r] = __builtin_amdgcn_exp2f(sc[r] - base);
                    l_run += w[r];
                }
                const v2u pw = v2u{pack_bf16(w[0], w[1]), pack_bf16(w[2], w[3])};
                v4s pv;
                __builtin_memcpy(&pv, &pw, 8);
                bonsai_wave::order_lds();
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    uint16_t e[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) e[r] = *reinterpret_cast<const uint16_t *>(v_tile + (kb * 4 + r) * kVPitch + (t * 16 + row) * 2);
                    v4s vt;
                    __builtin_memcpy(&vt, e, 8);
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[t][r] *= keep;
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(vt, pv, o[t], 0, 0, 0);
                }
                bonsai_wave::order_lds();
            }
            step_one::Pair lp = pair16(l_run);
            lp = pair32(lp.a + lp.b);
            float *out = att_out(c), *ml = out + kFrontWaves * kRows * kOPitch;
#pragma unroll
            for (int t = 0; t < 8; ++t) *reinterpret_cast<v4f *>(out + (wave * kRows + row) * kOPitch + t * 16 + kb * 4) = o[t];
            if (kb == 0) {
                ml[(wave * kRows + row) * 2] = m_run;
                ml[(wave * kRows + row) * 2 + 1] = lp.a + lp.b;
            }
            __syncthreads();
            store_part(c, tag);
        }
        if constexpr (ROW) {
            if (!merge_parts(c, tag, limit) && lane == 0) c.meet.bad = 1;
            announce(c, 1, rows8);
            __syncthreads();   // the raw row
            if (given_up(c.meet)) return false;
            v4u row[UQ];
            const int t = afresh(tid);
#pragma unroll
            for (int i = 0; i < UQ; ++i)
                row[i] = t + i * kFront < (c.q_dim >> 3) ? *reinterpret_cast<const v4u *>(c.raw + (t + i * kFront) * 8) : v4u{0, 0, 0, 0};
            if (!quant_row(row, std::integral_constant<int, UQ>{}, c.q_dim, true, rows8, c.o8, 1)) return false;
        }
        if (c.rows_o && !project(1, rows8, limit, [] {})) return false;

        if constexpr (ROW) {
            v4u row[UD];
            const bool ok = receive<UD>(c.h2 + (size_t)c.wg * a.dim * 4, a.dim >> 3, tag, row, limit);
            announce(c, 2, rows8);
            if (!norm_row(row, ln2, ok, rows8, c.g8, 2)) return false;
        }
        const auto ahead = [&] {   // what the next layer needs
            if constexpr (ROW) {
                ask_norm(ln1, nxt, 0);
            } else {
                rope.ask(nxt);
                if (c.attends) ask_history(more ? l + 1 : l, slot0, more);
            }
        };
        if (!c.rows_g)
            ahead();
        else if (!project(2, rows8, limit, ahead))
            return false;

        if constexpr (ROW) {
            v4u row[UF];
            const bool ok = receive<UF>(c.inner + (size_t)c.wg * a.ffn * 4, a.ffn >> 3, tag, row, limit);
            announce(c, 3, rows8);
            if (!quant_row(row, std::integral_constant<int, UF>{}, a.ffn, ok, rows8, c.d8, 3)) return false;
        }
        if (c.rows_d && !project(3, rows8, limit, [] {})) return false;
        cur = nxt;
    }
    return true;
}

template <int BITS, int SQ, int TQ, int SO, int SG, int TG, int SD, int UD, int UQ, int UF>
__global__ void __launch_bounds__(kThreads)
step_block_kernel(const Args a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wg = blockIdx.x;
    __shared__ Meet meet;
    const int groups = a.groups, gqa = a.n_heads / a.n_kv;
    const int q_dim = a.n_heads * kHd, n_qkv = (a.n_heads + 2 * a.n_kv) * kHd;
    const HeadOrder order{a.n_heads, a.n_kv, gqa};
    const Share sq(BITS, a.dim, order.rows(), groups / a.n_kv, false, false), so(BITS, q_dim, a.dim, groups, false, true),
        sg(BITS, a.dim, 2 * a.ffn, groups, true, false), sd(BITS, a.ffn, a.dim, groups, false, true);
    const auto part = [](const Share &s, int n, int i) {
        const int left = n - i * s.rows;
        return left < 0 ? 0 : (left < s.rows ? left : s.rows);
    };
    const auto mine = [wg, part](const Share &s, int n) { return wg < s.first ? 0 : part(s, n, wg - s.first); };
    const int back_wg = groups - 1 - wg;   // the rows' workgroups have no part of the attention
    const int kvh = back_wg % a.n_kv, unit = back_wg / a.n_kv, split = unit / gqa;
    const int rows_q = part(sq, order.rows(), unit), rows_o = mine(so, a.dim), rows_g = mine(sg, 2 * a.ffn), rows_d = mine(sd, a.dim);
    const auto in = (const __attribute__((address_space(4))) int32_t *)(uintptr_t)a.step_in;
    const int n = in[0] < 0 ? 0 : (in[0] < a.sigma ? in[0] : a.sigma);   // as everywhere: a history within its slots
    // a head's slots: the history and, behind it, the block's rows, in parts of at least 64
    const int head = kvh * gqa + unit - split * gqa;
    const int room = room_of(groups, a.n_heads);
    const int total = n + a.rows;
    const int per = 64 * ((total + 64 * room - 1) / (64 * room));
    const int splits = (total + per - 1) / per;
    const bool attends = split < splits, is_row = wg < a.rows;
    if (rows_q + rows_o + rows_g + rows_d == 0 && !attends && wg >= kRows) return;

    uint32_t *control = reinterpret_cast<uint32_t *>(a.exchange);
    const auto state = (const __attribute__((address_space(4))) uint32_t *)(uintptr_t)control;
    const uint32_t epoch = state[0];
    if (state[1]) {
        if (wg == 0 && tid == 0) *a.status = 1;
        return;
    }
    const Places at(a.n_layers, a.dim, a.ffn, a.n_heads, a.n_kv, groups);
    const Lds lds(sq, so, sg, sd, q_dim, TQ > TG ? TQ : TG);
    const size_t set8 = (size_t)a.n_layers * at.layer8;
    const Common c{a, wg, tid & 63, gqa, q_dim, n_qkv, a.rows, sq, so, sg, sd, rows_q, rows_o, rows_g, rows_d, epoch, attends, is_row,
                   step_one::near_heads(state, wg), n, in[1], kvh, unit, split, head, per, splits, room, order, unit * sq.rows, smem, lds.wave, smem + lds.once, smem + lds.gate, reinterpret_cast<uint16_t *>(smem),
                   reinterpret_cast<float *>(smem + lds.resid), reinterpret_cast<float *>(smem + lds.mult), meet, a.exchange + at.h, a.exchange + at.h2,
                   a.exchange + at.qkv, a.exchange + at.inner, a.exchange + at.parts, a.exchange + at.q8 + (epoch & 1) * set8, a.exchange + at.q8 + (~epoch & 1) * set8, at.layer8, at.o8, at.g8, at.d8, at.s8};
    if (tid == 0) meet.bad = 0;
    // the residual stream of the workgroup's columns
    for (int e = tid; e < a.rows * rows_o; e += kThreads) {
        const int token = e / rows_o, col = e - token * rows_o;
        const uint32_t id = (uint32_t)a.step_in[2 + 2 * a.rows + token];
        c.resid[token * so.rows + col] = bf16_bits_to_f32(a.embed[(size_t)(id < (uint32_t)a.vocab ? id : (uint32_t)a.vocab - 1) * a.dim + (wg - so.first) * so.rows + col]);
    }
    Rope rope{};
    if (wave < a.rows) {
        const int p = a.step_in[2 + a.rows + wave];
        const size_t row = (size_t)(p < 0 ? 0 : (p >= a.max_pos ? a.max_pos - 1 : p)) * (kHd / 2) + (tid & 31);
        const uint32_t *cos_t = reinterpret_cast<const uint32_t *>(a.cos_t), *sin_t = reinterpret_cast<const uint32_t *>(a.sin_t);
        rope.c0 = cos_t[row];
        rope.c1 = cos_t[row + 32];
        rope.s0 = sin_t[row];
        rope.s1 = sin_t[row + 32];
    }
    __syncthreads();
    const bool done = wave < kFrontWaves ? (is_row ? front<BITS, UD, UQ, UF, true>(c, wave, rope) : front<BITS, UD, UQ, UF, false>(c, wave, rope))
                                         : back<BITS, SQ, TQ, SO, SG, TG, SD>(c, wave - kFrontWaves, rope);
    if (tid == 0) {
        if (!done) {
            *a.status = 1;
            control[1] = 1;
        } else if (wg == 0) {
            control[0] = epoch + 1;
        }
    }
}

__global__ void __launch_bounds__(256) reset_kernel(v4u *p, size_t words, size_t tags) {   // tags: words that are cleared

    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < words; i += (size_t)gridDim.x * 256) {
        const uint32_t v = i < tags ? 0u : kEmpty;
        p[i] = v4u{v, v, v, v};
    }
}

// ---- host ---------------------------------------------------------------------------------------
struct Build {
    int bits, sq, tq, so, sg, tg, sd, ud, uq, uf;
};
constexpr Build kBuilds[] = {
    {2, 2, 1, 2, 2, 3, 4, 1, 1, 3},   // the 1.7B shape and below
    {2, 2, 2, 3, 2, 5, 7, 2, 2, 5},   // the 4B shape
    {1, 2, 1, 2, 2, 3, 4, 1, 1, 3},
    {1, 2, 2, 3, 2, 5, 7, 2, 2, 5},
};
struct Fit {
    int build = -1, lds = 0;
    int64_t bytes = 0, clear = 0, marked = 0;   // exchange memory; cleared up to `clear`, from there to `marked` (its end) empty rows
};
inline Fit fit(int bits, int n_layers, int dim, int ffn, int n_heads, int n_kv, int groups) {
    Fit f;
    const int q_dim = n_heads * kHd;
    // (One layer: workgroup 0 may be done, and advance the counter, before every other one has read it.)
    if ((bits != 1 && bits != 2) || n_layers < 2 || n_kv < 1 || n_heads < 1 || n_heads % n_kv != 0 || (groups - kRows) / n_heads < 1 ||
        groups > 65535 || dim < 128 || ffn < 128 || dim % 128 != 0 || ffn % 128 != 0)
        return f;
    const int64_t n_qkv = (int64_t)(n_heads + 2 * n_kv) * kHd;
    if (2 * (int64_t)ffn * dim >= kOob || n_qkv * dim >= kOob) return f;   // 32-bit offsets into a matrix
    const HeadOrder order{n_heads, n_kv, n_heads / n_kv};
    const Share sq(bits, dim, order.rows(), groups / n_kv, false, false), so(bits, q_dim, dim, groups, false, true), sg(bits, dim, 2 * ffn, groups, true, false),
        sd(bits, ffn, dim, groups, false, true);
    const Places at(n_layers, dim, ffn, n_heads, n_kv, groups);
    const auto words = [](int k) { return (k / 8 + kFront - 1) / kFront; };
    for (int i = 0; i < (int)(sizeof kBuilds / sizeof kBuilds[0]); ++i) {
        const Build &b = kBuilds[i];
        if (b.bits == bits && sq.stretch <= b.sq && sq.tiles <= b.tq && so.stretch <= b.so && so.tiles <= 1 && sg.stretch <= b.sg &&
            sg.tiles <= b.tg && sd.stretch <= b.sd && words(dim) <= b.ud && words(q_dim) <= b.uq && words(ffn) <= b.uf) {
            f.build = i;
            f.lds = Lds(sq, so, sg, sd, q_dim, b.tq > b.tg ? b.tq : b.tg).size;
            break;
        }
    }
    if (f.build >= 0 && f.lds > kMostLds) f.build = -1;
    f.bytes = f.marked = at.size;
    f.clear = at.q8;   // control and tags
    return f;
}
inline const void *kernel_of(int build) {
    switch (build) {
        case 0: return reinterpret_cast<const void *>(&step_block_kernel<2, 2, 1, 2, 2, 3, 4, 1, 1, 3>);
        case 1: return reinterpret_cast<const void *>(&step_block_kernel<2, 2, 2, 3, 2, 5, 7, 2, 2, 5>);
        case 2: return reinterpret_cast<const void *>(&step_block_kernel<1, 2, 1, 2, 2, 3, 4, 1, 1, 3>);
        default: return reinterpret_cast<const void *>(&step_block_kernel<1, 2, 2, 3, 2, 5, 7, 2, 2, 5>);
    }
}

}  // namespace step_block
#endif  // BONSAI_STEP_BLOCK_HIP_H
