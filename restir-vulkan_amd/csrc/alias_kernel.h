// alias_kernel.h — the body of the device alias-table build (createAliasTable, src/misc.cpp:418-497),
// written once over a workgroup policy G so that the same code runs as k_alias_build (one
// 1024-lane workgroup, alias_build.hip) and in a CPU build with one thread per lane
// (tests/cpu_kernels/alias_build_cpu.cpp), where ThreadSanitizer and AddressSanitizer watch
// every access between the barriers.
//
// G provides: tid() (lane in the workgroup), sync() (workgroup barrier that also orders memory)
// and shfl_up(v, d) (the value of lane tid - d of the caller's 64-lane wave; every lane of the
// wave calls it together). The includer defines AK_FN (the function qualifiers) before
// including this file.
//
// The reference sums the light powers in index order in float, normalises them to mean 1, queues
// the items >= 1 ("large") and < 1 ("small") in index order, then repeatedly pairs the front large
// g with the front small l: column l = (scaled[l], alias g), scaled[g] = (scaled[g] + scaled[l]) -
// 1, and g goes to the back of the small or the large queue. Taken one round of the large queue at
// a time (the larges queued when the round starts, in order), the pairs of a round are
// independent: the k-th large of the round meets the k-th small still queued. A round's pairs are
// therefore formed in parallel, and the larges that stay large (turn small) are appended in pair
// order through a workgroup scan. When fewer smalls are queued than the round has larges, the
// round goes in steps, each pairing as many as are queued; what a step appends to the small queue
// serves the next step.
//
// One workgroup waits for memory more than it computes, so each lane takes kPer consecutive items
// per step (their loads are in flight together), and once no more than kTail items are left, they
// move into LDS. Past kStep lights the launcher spreads the power sum, the normalisation and the
// large rounds over the device (alias_build.hip); the body then takes over for the rest.
#pragma once

#include <cstdint>

#include "../../include/restir_abi.h"

// AK_WAVE_SYNC(g): what the wave's lanes stored before it, its other lanes read after it. The
// includer may define it (the device's has to keep the compiler from moving accesses past it); an
// exchange does it where each exchange is a barrier of the wave.
#ifndef AK_WAVE_SYNC
#define AK_WAVE_SYNC(g) (void)(g).shfl_up(0u, 1u)
#endif

namespace ak {

constexpr uint32_t kLanes = 1024;  // one workgroup of 16 waves
constexpr uint32_t kWaves = kLanes / 64;
constexpr uint32_t kPer = 8;       // consecutive items per lane and step
constexpr uint32_t kStep = kLanes * kPer;
constexpr uint32_t kTail = 4096;   // items paired in LDS
// counts of a scan step packed in one word: smalls in the low 16 bits, larges in the high 16
constexpr uint32_t kSmall = 1u, kLarge = 1u << 16;
static_assert(kStep < (1u << 16), "a step's counts fit 16 bits");

struct Shared {
    float staged[kLanes];
    uint32_t waveTotal[kWaves];
    float sum;
    uint32_t state[6];                 // the queues after few_rounds
    // the last items: their values, light indices and queues (of positions here)
    float scaled[kTail];
    uint32_t ids[kTail], under[kTail], overA[kTail], overB[kTail];
};

template <class G>
AK_FN uint32_t wave_inclusive(G &g, uint32_t v) {
    const uint32_t lane = g.tid() & 63u;
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t o = g.shfl_up(v, d);
        if (lane >= d) v += o;
    }
    return v;
}

// exclusive scan of v over the workgroup; *total gets the sum
template <class G>
AK_FN uint32_t group_exclusive(G &g, Shared &sh, uint32_t v, uint32_t *total) {
    const uint32_t incl = wave_inclusive(g, v);
    const uint32_t w = g.tid() >> 6;
    if ((g.tid() & 63u) == 63u) sh.waveTotal[w] = incl;
    g.sync();
    uint32_t off = 0, tot = 0;
    for (uint32_t k = 0; k < kWaves; ++k) {
        const uint32_t t = sh.waveTotal[k];
        off += k < w ? t : 0u;
        tot += t;
    }
    g.sync();  // waveTotal is reused by the next call
    *total = tot;
    return off + incl - v;
}

AK_FN uint32_t float_bits(float v) { return __builtin_bit_cast(uint32_t, v); }
AK_FN float bits_float(uint32_t v) { return __builtin_bit_cast(float, v); }

// The power sum in index order, without adding one by one. While a sum stays in one binade, a whole
// multiple k of its ulp, adding w >= 0 adds to k the integer nearest to w / ulp, whatever k is,
// except for a tie, which goes to the even neighbour and so depends only on the parity of k. A run
// of additions is therefore a map from the parity of k to an increment; such maps compose.
// kOver: not known, or the sum may leave its binade.
constexpr uint32_t kOver = 1u << 24;
struct Inc {
    uint32_t even, odd;
};
AK_FN uint32_t inc_then(uint32_t first, uint32_t parity, const Inc &second) {
    if (first >= kOver) return kOver;
    const uint32_t s = first + (((first + parity) & 1u) ? second.odd : second.even);
    return s < kOver ? s : kOver;
}
AK_FN Inc compose(const Inc &first, const Inc &second) {
    return Inc{inc_then(first.even, 0u, second), inc_then(first.odd, 1u, second)};
}
// Adding w to a sum whose exponent field is e
AK_FN Inc inc_of(float w, uint32_t e) {
    const uint32_t u = float_bits(w);
    if (u & 0x80000000u) return (u << 1) ? Inc{kOver, kOver} : Inc{0u, 0u};
    const uint32_t field = u >> 23;
    if (field == 255u) return Inc{kOver, kOver};
    const uint32_t m = field ? ((u & 0x7fffffu) | 0x800000u) : u;
    const int32_t shift = static_cast<int32_t>(e) - static_cast<int32_t>(field ? field : 1u);  // w = m 2^-shift ulps
    if (shift <= 0) {
        if (m == 0u) return Inc{0u, 0u};
        if (shift < -24 || m >= (kOver >> -shift)) return Inc{kOver, kOver};
        return Inc{m << -shift, m << -shift};
    }
    if (shift > 24) return Inc{0u, 0u};  // below half an ulp
    const uint32_t f = m >> shift, rem = m & ((1u << shift) - 1u), half = 1u << (shift - 1);
    if (rem == half) return Inc{f + (f & 1u), f + ((f + 1u) & 1u)};
    const uint32_t r = f + (rem > half ? 1u : 0u);
    return Inc{r, r};
}

// The light power of light i (misc.cpp:426-442).
AK_FN float power_of(const restir_point_light *points, const restir_tri_light *triLights, uint32_t i) {
    return points ? points[i].color_luminance[3] : triLights[i].emission_luminance[3] * triLights[i].normalArea[3];
}

// Column i before the pairing, and its scaled power (misc.cpp:446-456).
AK_FN float normalised(restir_alias_table_column *cols, uint32_t i, float w, float powerSum, float count) {
    restir_alias_table_column c;
    c.prob = 0.0f;
    c.alias = -1;
    c.oriProb = w / powerSum;
    c.aliasOriProb = 0.0f;
    cols[i] = c;
    return count * w / powerSum;
}

AK_FN void settle(restir_alias_table_column *cols, uint32_t i) {  // prob 1, alias itself
    cols[i].prob = 1.0f;
    cols[i].alias = static_cast<int32_t>(i);
}

// The queues of the pairing: smalls under[head, tail), larges cur[0, m), of which the first k0 have
// had their pair of this round; nxt[0, mNext): those of them that stay large.
struct Queues {
    float *scaled;
    uint32_t *under, *cur, *nxt;
    const uint32_t *ids;  // light of an item; null: the item is the light
    uint32_t head, tail, m, k0, mNext;
};
AK_FN uint32_t light_of(const Queues &q, uint32_t item) { return q.ids ? q.ids[item] : item; }

AK_FN void next_round(Queues &q) {
    uint32_t *t = q.cur;
    q.cur = q.nxt;
    q.nxt = t;
    q.m = q.mNext;
    q.k0 = q.mNext = 0;
}
// What stays when a queue is empty: larges left (misc.cpp:479-484; of a round that the smalls did not
// last for, the rest of the round and its survivors), smalls left (486-491).
template <class G>
AK_FN void settle_rest(G &g, restir_alias_table_column *cols, const Queues &q) {
    for (uint32_t j = q.k0 + g.tid(); j < q.m; j += kLanes) settle(cols, light_of(q, q.cur[j]));
    for (uint32_t j = g.tid(); j < q.mNext; j += kLanes) settle(cols, light_of(q, q.nxt[j]));
    for (uint32_t j = q.head + g.tid(); j < q.tail; j += kLanes) settle(cols, light_of(q, q.under[j]));
}

// Pairing (misc.cpp:459-477), one round of the large queue at a time, until a queue is empty (the
// rest is then settled) or, at the end of a round, no more than `stop` items or kFew larges are left.
enum class Left { nothing, few, some };
constexpr uint32_t kFew = 64;
template <class G>
AK_FN Left pair(G &g, Shared &sh, restir_alias_table_column *cols, Queues &q, uint32_t stop) {
    const uint32_t tid = g.tid();
    for (;;) {
        if (q.k0 == 0) {
            if (q.m == 0 || q.head == q.tail) break;
            if (q.m + (q.tail - q.head) <= stop) return Left::some;
            if (q.m <= kFew) return Left::few;
        }
        while (q.k0 < q.m && q.head < q.tail) {
            const uint32_t c = q.m - q.k0 < q.tail - q.head ? q.m - q.k0 : q.tail - q.head;
            // items per lane: one when the lanes suffice
            const uint32_t per = c <= kLanes ? 1u : kPer;
            for (uint32_t b = 0; b < c; b += kLanes * per) {
                const uint32_t j0 = b + tid * per;
                const uint32_t cnt = j0 < c ? (c - j0 < per ? c - j0 : per) : 0u;
                uint32_t gl[kPer], l[kPer], kind = 0, large = 0;
                float sg[kPer], sl[kPer];
                for (uint32_t k = 0; k < kPer; ++k) {
                    gl[k] = l[k] = 0u;
                    if (k < cnt) {
                        gl[k] = q.cur[q.k0 + j0 + k];
                        l[k] = q.under[q.head + j0 + k];
                    }
                }
                for (uint32_t k = 0; k < kPer; ++k) {
                    sg[k] = sl[k] = 0.0f;
                    if (k < cnt) {
                        sg[k] = q.scaled[gl[k]];
                        sl[k] = q.scaled[l[k]];
                    }
                }
                for (uint32_t k = 0; k < kPer; ++k)
                    if (k < cnt) {
                        restir_alias_table_column &col = cols[light_of(q, l[k])];
                        col.prob = sl[k];
                        col.alias = static_cast<int32_t>(light_of(q, gl[k]));
                        const float v = (sg[k] + sl[k]) - 1.0f;
                        q.scaled[gl[k]] = v;
                        if (v < 1.0f) {
                            kind += kSmall;
                        } else {
                            kind += kLarge;
                            large |= 1u << k;
                        }
                    }
                uint32_t tot;
                const uint32_t ex = group_exclusive(g, sh, kind, &tot);
                uint32_t toSmall = q.tail + (ex & 0xffffu), toLarge = q.mNext + (ex >> 16);
                for (uint32_t k = 0; k < kPer; ++k)
                    if (k < cnt) {
                        if (large & (1u << k)) q.nxt[toLarge++] = gl[k];
                        else q.under[toSmall++] = gl[k];
                    }
                q.tail += tot & 0xffffu;
                q.mNext += tot >> 16;
            }
            q.head += c;
            q.k0 += c;
            g.sync();  // appended queue entries and new weights visible to the next step
        }
        if (q.k0 < q.m) break;  // the small queue ran dry inside the round
        next_round(q);
    }
    settle_rest(g, cols, q);
    return Left::nothing;
}

// The rounds of at most kFew larges, by the workgroup's first wave without barriers, until a queue is
// empty. A large that becomes small goes to the back of q's smalls, or (all: q is a copy of the
// front of a longer queue) of all's, with its value. For queues in LDS: a round then takes a fraction
// of the workgroup's 1.5 us, and a light as bright as many takes as many rounds.
template <class G>
AK_FN void few_rounds(G &g, Shared &sh, restir_alias_table_column *cols, Queues &q, Queues *all) {
    const uint32_t tid = g.tid();
    if (tid < 64u) {
        while (q.m > 0 && q.head < q.tail) {
            const uint32_t c = q.m - q.k0 < q.tail - q.head ? q.m - q.k0 : q.tail - q.head;
            uint32_t kind = 0, gl = 0;
            float v = 0.0f;
            if (tid < c) {
                gl = q.cur[q.k0 + tid];
                const uint32_t l = q.under[q.head + tid];
                const float sl = q.scaled[l];
                restir_alias_table_column &col = cols[light_of(q, l)];
                col.prob = sl;
                col.alias = static_cast<int32_t>(light_of(q, gl));
                v = (q.scaled[gl] + sl) - 1.0f;
                q.scaled[gl] = v;
                kind = v < 1.0f ? kSmall : kLarge;
            }
            const uint32_t incl = wave_inclusive(g, kind);
            if (tid == 63u) sh.waveTotal[0] = incl;
            AK_WAVE_SYNC(g);
            const uint32_t tot = sh.waveTotal[0], ex = incl - kind;
            if (kind == kLarge) {
                q.nxt[q.mNext + (ex >> 16)] = gl;
            } else if (kind == kSmall && all) {
                const uint32_t light = light_of(q, gl);
                all->under[all->tail + (ex & 0xffffu)] = light;
                all->scaled[light] = v;
            } else if (kind == kSmall) {
                q.under[q.tail + (ex & 0xffffu)] = gl;
            }
            (all ? all->tail : q.tail) += tot & 0xffffu;
            q.mNext += tot >> 16;
            q.head += c;
            q.k0 += c;
            if (q.k0 == q.m) next_round(q);
            AK_WAVE_SYNC(g);  // queue entries, values and the total's slot are used again
        }
        if (tid == 0) {
            sh.state[0] = q.head;
            sh.state[1] = all ? all->tail : q.tail;
            sh.state[2] = q.m;
            sh.state[3] = q.k0;
            sh.state[4] = q.mNext;
            sh.state[5] = q.cur == sh.overB ? 1u : 0u;
        }
    }
    g.sync();
    q.head = sh.state[0];
    (all ? all->tail : q.tail) = sh.state[1];
    q.m = sh.state[2];
    q.k0 = sh.state[3];
    q.mNext = sh.state[4];
    q.cur = sh.state[5] ? sh.overB : sh.overA;
    q.nxt = sh.state[5] ? sh.overA : sh.overB;
}

// aliasOriProb of column i (misc.cpp:493-495)
AK_FN void finish(restir_alias_table_column *cols, uint32_t i) {
    cols[i].aliasOriProb = cols[cols[i].alias].oriProb;
}

// The pairing from q on: the last kTail items in LDS; where few larges face more smalls than that,
// the larges and one window of the smalls after another.
template <class G>
AK_FN void pair_all(G &g, Shared &sh, restir_alias_table_column *cols, Queues &q) {
    const Left left = pair(g, sh, cols, q, kTail);
    if (left == Left::nothing) return;
    const uint32_t smalls = q.tail - q.head, in = left == Left::some ? smalls : 0u;
    // larges first, then the queued smalls, in their order
    for (uint32_t j = g.tid(); j < q.m + in; j += kLanes) {
        const uint32_t l = j < q.m ? q.cur[j] : q.under[q.head + (j - q.m)];
        sh.ids[j] = l;
        sh.scaled[j] = q.scaled[l];
        if (j < q.m) sh.overA[j] = j;
        else sh.under[j - q.m] = j;
    }
    Queues t{sh.scaled, sh.under, sh.overA, sh.overB, sh.ids, 0u, in, q.m, 0u, 0u};
    g.sync();
    if (left == Left::some) {
        if (pair(g, sh, cols, t, 0u) == Left::nothing) return;
        few_rounds(g, sh, cols, t, static_cast<Queues *>(nullptr));
        settle_rest(g, cols, t);
        return;
    }
    while (t.m > 0 && q.head < q.tail) {
        const uint32_t len = q.tail - q.head < kTail - kFew ? q.tail - q.head : kTail - kFew;
        for (uint32_t j = g.tid(); j < len; j += kLanes) {
            const uint32_t l = q.under[q.head + j];
            sh.ids[kFew + j] = l;
            sh.scaled[kFew + j] = q.scaled[l];
            sh.under[j] = kFew + j;
        }
        t.head = 0;
        t.tail = len;
        g.sync();
        few_rounds(g, sh, cols, t, &q);
        q.head += t.head;
        g.sync();  // the window is rewritten, and what was appended to q's smalls is read
    }
    t.tail = t.head;  // its smalls left are q's
    settle_rest(g, cols, t);
    for (uint32_t j = q.head + g.tid(); j < q.tail; j += kLanes) settle(cols, q.under[j]);
}

template <class G>
AK_FN void build(G &g, Shared &sh, const restir_point_light *points, const restir_tri_light *triLights, uint32_t n,
                 restir_alias_table_column *cols, float *power, float *scaled, uint32_t *under, uint32_t *overA,
                 uint32_t *overB) {
    const uint32_t tid = g.tid();

    // light powers and their sum in index order
    float sum = 0.0f;
    for (uint32_t base = 0; base < n; base += kLanes) {
        const uint32_t i = base + tid;
        float w = 0.0f;
        if (i < n) {
            w = power_of(points, triLights, i);
            power[i] = w;
        }
        sh.staged[tid] = w;
        g.sync();
        if (tid == 0) {
            const uint32_t m = n - base < kLanes ? n - base : kLanes;
            for (uint32_t k = 0; k < m; ++k) sum += sh.staged[k];
        }
        g.sync();
    }
    if (tid == 0) sh.sum = sum;
    g.sync();
    const float powerSum = sh.sum;
    const float count = static_cast<float>(n);

    // normalise; queue larges and smalls in index order
    uint32_t nLarge = 0, nSmall = 0;
    for (uint32_t base = 0; base < n; base += kLanes) {
        const uint32_t i = base + tid;
        uint32_t kind = 0;
        if (i < n) {
            const float s = normalised(cols, i, power[i], powerSum, count);
            scaled[i] = s;
            kind = s >= 1.0f ? kLarge : kSmall;
        }
        uint32_t tot;
        const uint32_t ex = group_exclusive(g, sh, kind, &tot);
        if (kind == kLarge) overA[nLarge + (ex >> 16)] = i;
        else if (kind == kSmall) under[nSmall + (ex & 0xffffu)] = i;
        nLarge += tot >> 16;
        nSmall += tot & 0xffffu;
    }

    // The queues, scaled[] and cols[] written above must be visible before any lane pairs: the
    // lane that pairs large k reads the queue entry another lane wrote after the scan's last
    // barrier (without this barrier, lane 0 could read overA[0] before its writer had stored it).
    g.sync();

    Queues q{scaled, under, overA, overB, nullptr, 0u, nSmall, nLarge, 0u, 0u};
    pair_all(g, sh, cols, q);
    g.sync();
    for (uint32_t i = tid; i < n; i += kLanes) finish(cols, i);
}

}  // namespace ak
