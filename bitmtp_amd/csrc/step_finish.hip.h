// What follows a step in one launch (step_one.hip.h, step_block.hip.h): the final norm of the rows that are projected onto
// the vocabulary or, first, the step once more.
//
// Those launches need every compute unit at once and give up where they don't get them.  What is queued behind a step reads
// its results in stream order, without the host in between, so they have to be right by the time the stream goes on: where
// this launch finds the mark of a step that gave up, it does the whole step again and puts the exchange memory back into
// its first state.  It needs no number of workgroups at once.  The step is cut into tasks in the order of their
// dependencies; a workgroup draws the next task's number and waits for tasks of earlier phases only, whose numbers were
// drawn by workgroups that are running, so the lowest number never waits and all of them end, with one workgroup on the
// device as with all.
//
// It is the slow way, with a fence over the device at either end of a task: a one-token step of the 1.7B shape takes 5.1 ms,
// of nine rows 6.8 ms, sixteen rows of the 4B shape 12.8 ms, where separate launches take 0.7 to 1.6; a caller that sees
// `*status` keeps to those for a while.  (One workgroup, without tasks and fences: 58, 77 and 208 ms.)  Without a mark the
// launch is the final norm that separate launches have as well, and takes as long (4.6 us); the check as a launch of its own
// took 5 us more.
//
// Rounding points and exact group sums of the separate launches; fp32 sums over K in one order, fp32 probabilities.
#ifndef BONSAI_STEP_FINISH_HIP_H
#define BONSAI_STEP_FINISH_HIP_H

namespace step_finish {

using step_one::Layer;
using step_one::unpack_word;
using step_one::v2u;
using step_one::v4u;

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kThreads = kWaves * 64;
constexpr int kGroups = 64;                    // workgroups: the rows of a norm, the tasks of a repeated step
constexpr int kRows = 16;
constexpr uint32_t kLongest = 2000000000;      // 20 s, which no task waits unless an earlier one is lost
constexpr uint32_t kLost = 2;                  // the mark and the status then: the tasks' numbers are of no use to later steps
enum { kEpoch, kGaveUp, kDrawn, kDone, kLeft, kControlWords };   // words of the exchange memory, with those of the step's launch

struct Places {   // byte offsets of the rows of a repeated step, behind the exchange memory (its residual stream is h_out)
    int64_t att, gu, q8, s8, size;   // q|k|v at 0
    __host__ __device__ Places(int rows, int dim, int ffn, int n_heads, int n_kv) {
        const int q_dim = n_heads * kHd;
        const int64_t r = rows;
        att = r * (q_dim + 2 * n_kv * kHd) * 2;
        gu = att + r * q_dim * 2;
        q8 = gu + r * ffn * 4;
        s8 = q8 + r * (ffn > q_dim ? (ffn > dim ? ffn : dim) : (q_dim > dim ? q_dim : dim));
        size = s8 + 4 * kRows;
    }
};

struct Args {
    const Layer *layers;
    const uint16_t *embed;
    const int32_t *step_in;
    uint16_t *kv;
    const uint16_t *cos_t, *sin_t;
    uint8_t *exchange, *rows_at;        // `words` 16-byte words; rows of a repeated step
    uint16_t *h_out;
    int32_t *status;
    const uint16_t *norm_w;             // final norm of rows norm_first ..: int8 and multipliers, or bf16
    int8_t *norm_q;
    float *norm_s;
    uint16_t *norm_out;
    uint32_t words, mark_from, mark_to; // the exchange memory's first state: these words hold `mark`, the others 0
    uint32_t mark;
    int norm_first, norm_rows, rows, n_layers, dim, ffn, n_heads, n_kv, slots, sigma, max_pos, vocab;
    float eps, scale;
};

struct Meet {   // LDS where the waves meet
    double sum[kWaves];
    float top[kWaves];
    uint32_t drawn;
    int lost;
};

// ---- rows, by a workgroup ------------------------------------------------------------------
__device__ __forceinline__ void put_int8(int8_t *row, int word, const float *f, float s) {   // eight neighbouring values
    uint32_t d[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i)
        d[i >> 2] |= ((uint32_t)(int)fminf(fmaxf(__builtin_rintf(f[i] * s), -128.0f), 127.0f) & 0xffu) << (8 * (i & 3));
    *reinterpret_cast<v2u *>(row + word * 8) = v2u{d[0], d[1]};
}
// .. in the order of `codes`: of sixteen values, byte 4 j + i is value 4 i + j
__device__ __forceinline__ void put_turned(int8_t *row, int word, const float *f, float s) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const auto byte = [&](float x) { return (uint32_t)(int)fminf(fmaxf(__builtin_rintf(x * s), -128.0f), 127.0f) & 0xffu; };
        *reinterpret_cast<uint16_t *>(row + (word >> 1) * 16 + j * 4 + (word & 1) * 2) = (uint16_t)(byte(f[j]) | byte(f[4 + j]) << 8);
    }
}
// Words tid + 512 i of a row, value(word, values); put(word, values, multiplier), which is returned.
template <int U, class Value, class Put>
__device__ __forceinline__ float quantise(Meet &meet, int words, Value value, Put put) {
    const int tid = threadIdx.x;
    float f[U][8], top = 0.0f;
#pragma unroll
    for (int i = 0; i < U; ++i)
        if (tid + i * kThreads < words) {
            value(tid + i * kThreads, f[i]);
#pragma unroll
            for (int j = 0; j < 8; ++j) top = fmaxf(top, fabsf(f[i][j]));
        }
    top = bonsai_wave::max64(top);
    if ((tid & 63) == 0) meet.top[tid >> 6] = top;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kWaves; ++i) top = fmaxf(top, meet.top[i]);
    const float recip = 1.0f / fmaxf(top, 1e-5f);
    const float s = recip * 127.0f;
#pragma unroll
    for (int i = 0; i < U; ++i)
        if (tid + i * kThreads < words) put(tid + i * kThreads, f[i], s);
    return s;
}
// Values of the thread's word of a row of dim (at most 4096), normed.
__device__ __forceinline__ void norm_word(Meet &meet, const v4u x, const v4u w, bool there, int dim, float eps, float *f) {
    const int tid = threadIdx.x;
    float wf[8];
    unpack_word(x, f);
    unpack_word(w, wf);
    double ss = 0.0;
    if (there)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float sq = f[i] * f[i];
            ss += (double)sq;
        }
    ss = bonsai_wave::sum64(ss);
    if ((tid & 63) == 0) meet.sum[tid >> 6] = ss;
    __syncthreads();
    double total = 0.0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) total += meet.sum[i];
    const float var = (float)total / (float)dim;
    const float rs = 1.0f / sqrtf(var + eps);
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = bf16_round(wf[i] * bf16_round(f[i] * rs));
}
__device__ __forceinline__ v4u word_of(const uint16_t *row, int word) { return reinterpret_cast<const v4u *>(row)[word]; }

// Row `row` of those projected onto the vocabulary.
__device__ __forceinline__ void final_norm(const Args &a, Meet &meet, int row, const v4u x, const v4u w) {
    const int word = threadIdx.x;
    const bool there = word < (a.dim >> 3);
    float f[8];
    norm_word(meet, x, w, there, a.dim, a.eps, f);
    if (a.norm_out != nullptr) {
        if (there)
            reinterpret_cast<v4u *>(a.norm_out + (size_t)row * a.dim)[word] =
                v4u{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7])};
        return;
    }
    const float s = quantise<1>(meet, a.dim >> 3, [&](int, float *v) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = f[i];
    }, [&](int at, const float *v, float mult) { put_int8(a.norm_q + (size_t)row * a.dim, at, v, mult); });
    if (word == 0) a.norm_s[row] = s;
}

// ---- the step again ------------------------------------------------------------------------
// 16 codes, as dwords of signed bytes in the order of put_turned.
template <int BITS>
__device__ __forceinline__ v4i codes(uint32_t p) {
    v4i w;
    if constexpr (BITS == 1) p = (p & 0xfu) | (p & 0xf0u) << 4 | (p & 0xf00u) << 8 | (p & 0xf000u) << 12;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t c = BITS == 2 ? (p >> (2 * j)) & 0x03030303u : ((p >> j) & 0x01010101u) << 1;
        w[j] = (int)(((c | 0x80808080u) - (BITS == 2 ? 0x02020202u : 0x01010101u)) ^ 0x80808080u);   // code - 2, 2 bit - 1
    }
    return w;
}
// Rows tile * 16 .. of a projection, by a wave: done(token, row, result as bf16).
template <int BITS, class Done>
__device__ __forceinline__ void project(const int8_t *q8, const float *s8, int rows, const uint8_t *w, const uint16_t *ws, int k, int tile, Done done) {
    const int lane = (int)(threadIdx.x & 63), kb = lane >> 4, row = tile * 16 + (lane & 15);
    const int groups = k / 128, token = (lane & 15) < rows ? lane & 15 : rows - 1;
    const int8_t *const x = q8 + (size_t)token * k + kb * 32;
    const uint8_t *const wr = w + (size_t)row * groups * (16 * BITS) + kb * (4 * BITS);
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int g = 0; g < groups; ++g) {
        uint32_t p0, p1;
        if constexpr (BITS == 2) {
            const v2u p = *reinterpret_cast<const v2u *>(wr + g * 32);
            p0 = p.x;
            p1 = p.y;
        } else {
            const uint32_t p = *reinterpret_cast<const uint32_t *>(wr + g * 16);
            p0 = p & 0xffffu;
            p1 = p >> 16;
        }
        const v4i x0 = *reinterpret_cast<const v4i *>(x + g * 128), x1 = *reinterpret_cast<const v4i *>(x + g * 128 + 16);
        v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(x0, codes<BITS>(p0), v4i{0, 0, 0, 0}, 0, 0, 0);
        d = __builtin_amdgcn_mfma_i32_16x16x64_i8(x1, codes<BITS>(p1), d, 0, 0, 0);
        const float s = bf16_bits_to_f32(ws[(size_t)row * groups + g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += (float)d[e] * s;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (kb * 4 + e < rows) done(kb * 4 + e, row, bf16_round(acc[e] / s8[kb * 4 + e]));
}
// A query head of a row, by a wave: a lane a slot, then two of the dims.  In bf16 to `out`.
__device__ __forceinline__ void attend(const uint16_t *query, const uint16_t *k_head, const uint16_t *v_head, int n, int hide, uint32_t sees, int rows,
                                       int sigma, float scale, uint16_t *out) {
    const int lane = (int)(threadIdx.x & 63), total = n + rows;
    const v4u *q = reinterpret_cast<const v4u *>(query);
    const auto slot_of = [&](int j) { return (size_t)(j < n ? j : sigma + j - n) * kHd; };
    float m_run = -INFINITY, sum = 0.0f, o0 = 0.0f, o1 = 0.0f;
    for (int base = 0; base < total; base += 64) {
        const int j = base + lane;
        const bool see = j < n ? j != hide : j < total && ((sees >> (j - n)) & 1u);
        const v4u *k = reinterpret_cast<const v4u *>(k_head + slot_of(j < total ? j : total - 1));
        float d = 0.0f;
#pragma unroll 8
        for (int e = 0; e < kHd / 8; ++e) {
            const v4u x = k[e], y = q[e];
            d = dot2_bf16(x.x, y.x, d);
            d = dot2_bf16(x.y, y.y, d);
            d = dot2_bf16(x.z, y.z, d);
            d = dot2_bf16(x.w, y.w, d);
        }
        d = see ? d * (scale * 1.44269504088896341f) : -INFINITY;
        const float m = fmaxf(m_run, wave_max(d)), from = m == -INFINITY ? 0.0f : m;
        const float keep = __builtin_amdgcn_exp2f(m_run - from), p = __builtin_amdgcn_exp2f(d - from);
        m_run = m;
        sum = sum * keep + wave_sum(p);
        o0 *= keep;
        o1 *= keep;
        for (int e = 0; e < 64; ++e) {   // (behind the last slot the last one, with a probability of 0)
            const float pe = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(p), e));
            const uint32_t v = *reinterpret_cast<const uint32_t *>(v_head + slot_of(base + e < total ? base + e : total - 1) + 2 * lane);
            o0 += pe * __uint_as_float(v << 16);
            o1 += pe * __uint_as_float(v & 0xffff0000u);
        }
    }
    const float y0 = sum > 0.0f ? o0 / sum : 0.0f, y1 = sum > 0.0f ? o1 / sum : 0.0f;
    *reinterpret_cast<uint32_t *>(out + 2 * lane) = pack_bf16(y0, y1);
}

struct Task {
    int phase, layer, index;
    uint32_t after;   // tasks that have to be done
};
enum { kNorm1, kQkv, kHeads, kAttend, kQuantAtt, kO, kNorm2, kGateUp, kQuantInner, kDown, kPhases, kEmbed = kPhases, kFinal, kReset };
// The tasks in order: embedding rows, the phases of every layer, final norm, exchange memory.
struct Plan {
    int count[kPhases], rows, n_layers, norm_rows;
    uint32_t layer, total;
    __host__ __device__ Plan(int rows_, int n_layers_, int dim, int ffn, int n_heads, int n_kv, int norm_rows_) {
        rows = rows_;
        n_layers = n_layers_;
        norm_rows = norm_rows_;
        const int heads = n_heads + 2 * n_kv;
        // a row a workgroup; a tile of sixteen weight rows, a head's row a wave
        const int c[kPhases] = {rows, heads * kHd / (16 * kWaves), (heads * rows + kWaves - 1) / kWaves, (n_heads * rows + kWaves - 1) / kWaves, rows,
                                dim / (16 * kWaves), rows, 2 * ffn / (16 * kWaves), rows, dim / (16 * kWaves)};
        layer = 0;
        for (int i = 0; i < kPhases; ++i) {
            count[i] = c[i];
            layer += (uint32_t)c[i];
        }
        total = (uint32_t)rows + (uint32_t)n_layers * layer + (uint32_t)norm_rows + kGroups;
    }
    __host__ __device__ Task task(uint32_t number) const {
        if (number < (uint32_t)rows) return Task{kEmbed, 0, (int)number, 0u};
        uint32_t left = number - (uint32_t)rows;
        const int l = (int)(left / layer);
        if (l < n_layers) {
            left -= (uint32_t)l * layer;
            int phase = 0;
            uint32_t after = number - left;
            while (left >= (uint32_t)count[phase]) {
                left -= (uint32_t)count[phase];
                after += (uint32_t)count[phase];
                ++phase;
            }
            return Task{phase, l, (int)left, after};
        }
        left -= (uint32_t)n_layers * layer;
        const uint32_t after = number - left;
        if (left < (uint32_t)norm_rows) return Task{kFinal, 0, (int)left, after};
        return Task{kReset, 0, (int)(left - (uint32_t)norm_rows), after};
    }
};

template <int BITS>
__device__ __forceinline__ void do_task(const Args &a, Meet &meet, const Task &t) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q_dim = a.n_heads * kHd, heads = a.n_heads + 2 * a.n_kv, n_qkv = heads * kHd;
    const Places at(a.rows, a.dim, a.ffn, a.n_heads, a.n_kv);
    uint16_t *const qkv = reinterpret_cast<uint16_t *>(a.rows_at), *const att = reinterpret_cast<uint16_t *>(a.rows_at + at.att),
                   *const gu = reinterpret_cast<uint16_t *>(a.rows_at + at.gu);
    int8_t *const q8 = reinterpret_cast<int8_t *>(a.rows_at + at.q8);
    float *const s8 = reinterpret_cast<float *>(a.rows_at + at.s8);
    const Layer &w = a.layers[t.layer];
    uint16_t *const keys = a.kv + (size_t)t.layer * a.n_kv * a.slots * kHd, *const vals = keys + (size_t)a.n_layers * a.n_kv * a.slots * kHd;
    const auto add = [&](int token, int row, float y) {
        uint16_t *p = a.h_out + (size_t)token * a.dim + row;
        *p = (uint16_t)f32_to_bf16_bits(y + bf16_bits_to_f32(*p));
    };
    const int tile = t.index * kWaves + wave;

    switch (t.phase) {
        case kEmbed: {
            const uint32_t id = (uint32_t)a.step_in[2 + 2 * a.rows + t.index];
            const uint16_t *e = a.embed + (size_t)(id < (uint32_t)a.vocab ? id : (uint32_t)a.vocab - 1) * a.dim;
            for (int i = tid; i < a.dim >> 3; i += kThreads) reinterpret_cast<v4u *>(a.h_out + (size_t)t.index * a.dim)[i] = word_of(e, i);
            break;
        }
        case kNorm1:
        case kNorm2: {
            const bool there = tid < (a.dim >> 3);
            const int word = there ? tid : 0;
            float f[8];
            norm_word(meet, word_of(a.h_out + (size_t)t.index * a.dim, word), word_of(t.phase == kNorm1 ? w.ln1 : w.ln2, word), there, a.dim, a.eps, f);
            const float s = quantise<1>(meet, a.dim >> 3, [&](int, float *v) {
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = f[i];
            }, [&](int at8, const float *v, float mult) { put_turned(q8 + (size_t)t.index * a.dim, at8, v, mult); });
            if (tid == 0) s8[t.index] = s;
            break;
        }
        case kQkv:
            project<BITS>(q8, s8, a.rows, w.w[0], w.s[0], a.dim, tile,
                          [&](int token, int row, float y) { qkv[(size_t)token * n_qkv + row] = (uint16_t)f32_to_bf16_bits(y); });
            break;
        case kHeads: {   // queries stay, keys and values go to their slots
            if (tile >= heads * a.rows) break;
            const int row = tile / heads, head = tile - row * heads;
            uint16_t *x = qkv + ((size_t)row * heads + head) * kHd;
            const int kvh = head < a.n_heads ? 0 : (head - a.n_heads) % a.n_kv;
            const size_t slot = ((size_t)kvh * a.slots + a.sigma + row) * kHd;
            if (head < a.n_heads + a.n_kv) {
                const bool query = head < a.n_heads;
                uint32_t o0, o1;
                rope_row_math(rope_row_load(x, query ? w.qn : w.kn, a.cos_t, a.sin_t, a.step_in[2 + a.rows + row], a.max_pos, lane), a.eps, o0, o1);
                uint16_t *to = query ? x : keys + slot;
                to[lane] = (uint16_t)o0;
                to[lane + 64] = (uint16_t)o1;
            } else {
                vals[slot + lane] = x[lane];
                vals[slot + lane + 64] = x[lane + 64];
            }
            break;
        }
        case kAttend: {
            if (tile >= a.n_heads * a.rows) break;
            const int row = tile / a.n_heads, head = tile - row * a.n_heads, kvh = head / (a.n_heads / a.n_kv);
            const int n = a.step_in[0] < 0 ? 0 : (a.step_in[0] < a.sigma ? a.step_in[0] : a.sigma);
            attend(qkv + ((size_t)row * heads + head) * kHd, keys + (size_t)kvh * a.slots * kHd, vals + (size_t)kvh * a.slots * kHd, n, a.step_in[1],
                   (uint32_t)a.step_in[2 + row], a.rows, a.sigma, a.scale, att + (size_t)row * q_dim + head * kHd);
            break;
        }
        case kQuantAtt: {
            const float s = quantise<1>(meet, q_dim >> 3, [&](int at8, float *v) { unpack_word(word_of(att + (size_t)t.index * q_dim, at8), v); },
                                        [&](int at8, const float *v, float mult) { put_turned(q8 + (size_t)t.index * q_dim, at8, v, mult); });
            if (tid == 0) s8[t.index] = s;
            break;
        }
        case kO:
            project<BITS>(q8, s8, a.rows, w.w[1], w.s[1], q_dim, tile, add);
            break;
        case kGateUp:
            project<BITS>(q8, s8, a.rows, w.w[2], w.s[2], a.dim, tile,
                          [&](int token, int row, float y) { gu[(size_t)token * 2 * a.ffn + row] = (uint16_t)f32_to_bf16_bits(y); });
            break;
        case kQuantInner: {
            const uint16_t *g = gu + (size_t)t.index * 2 * a.ffn, *u = g + a.ffn;
            const float s = quantise<3>(meet, a.ffn >> 3, [&](int at8, float *v) {
                float y[8];
                unpack_word(word_of(g, at8), v);
                unpack_word(word_of(u, at8), y);
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = step_one::silu_mul(v[i], y[i]);
            }, [&](int at8, const float *v, float mult) { put_turned(q8 + (size_t)t.index * a.ffn, at8, v, mult); });
            if (tid == 0) s8[t.index] = s;
            break;
        }
        case kDown:
            project<BITS>(q8, s8, a.rows, w.w[3], w.s[3], a.ffn, tile, add);
            break;
        case kFinal: {
            const int word = tid < (a.dim >> 3) ? tid : 0;
            final_norm(a, meet, t.index, word_of(a.h_out + (size_t)(a.norm_first + t.index) * a.dim, word), word_of(a.norm_w, word));
            break;
        }
        default:   // (all but the control words: others still look at the first ones, and where the dies are stays)
            for (uint32_t i = (uint32_t)(t.index * kThreads + tid); i < a.words; i += kGroups * kThreads) {
                const uint32_t v = i >= a.mark_from && i < a.mark_to ? a.mark : 0u;
                if (i >= step_one::kControlBytes / 16) reinterpret_cast<v4u *>(a.exchange)[i] = v4u{v, v, v, v};
            }
    }
}

template <int BITS>
__device__ __forceinline__ void step_again(const Args &a, Meet &meet) {
    const int tid = threadIdx.x;
    uint32_t *const control = reinterpret_cast<uint32_t *>(a.exchange);
    const Plan plan(a.rows, a.n_layers, a.dim, a.ffn, a.n_heads, a.n_kv, a.norm_rows);
    if (tid == 0) meet.lost = 0;
    for (;;) {
        if (tid == 0) meet.drawn = __hip_atomic_fetch_add(control + kDrawn, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const uint32_t number = (uint32_t)__builtin_amdgcn_readfirstlane((int)meet.drawn);
        if (number >= plan.total) break;
        const Task t = plan.task(number);
        if (tid == 0) {
            const uint32_t since = (uint32_t)wall_clock64();
            while (__hip_atomic_load(control + kDone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < t.after) {
                __builtin_amdgcn_s_sleep(2);
                if ((uint32_t)wall_clock64() - since > kLongest) {
                    meet.lost = 1;
                    break;
                }
            }
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(meet.lost)) {
            if (tid == 0) {
                control[kGaveUp] = kLost;
                *a.status = (int32_t)kLost;
            }
            return;
        }
        __threadfence();   // what earlier tasks stored, wherever they ran
        do_task<BITS>(a, meet, t);
        __threadfence();   // .. and what this one did, for the later ones
        __syncthreads();
        if (tid == 0) __hip_atomic_fetch_add(control + kDone, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // The mark stays until every workgroup has seen it.
    if (tid == 0 && __hip_atomic_fetch_add(control + kLeft, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1)
        for (int i = 0; i < kControlWords; ++i) control[i] = 0;
}

template <int BITS>
__global__ void __launch_bounds__(kThreads)
finish_kernel(const Args a) {
    __shared__ Meet meet;
    const int row = blockIdx.x;
    const auto control = (const __attribute__((address_space(4))) uint32_t *)(uintptr_t)a.exchange;
    v4u x = v4u{0, 0, 0, 0}, w = x;
    if (row < a.norm_rows && (int)threadIdx.x < (a.dim >> 3)) {
        x = word_of(a.h_out + (size_t)(a.norm_first + row) * a.dim, threadIdx.x);
        w = word_of(a.norm_w, threadIdx.x);
    }
    const uint32_t mark = control[kGaveUp];
    if (mark == 0) {
        if (row < a.norm_rows) final_norm(a, meet, row, x, w);
        return;
    }
    if (mark == kLost) {
        if (row == 0 && threadIdx.x == 0) *a.status = (int32_t)kLost;   // (over the 1 of the step's own launch)
        return;
    }
    step_again<BITS>(a, meet);
}

}  // namespace step_finish
#endif  // BONSAI_STEP_FINISH_HIP_H
