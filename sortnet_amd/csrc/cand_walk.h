// What the kernels that walk the marked inputs of a row (sort_cols.hip, row_cands.hip, bound_cols.hip) share: the list of
// marks of a wavefront, how the list is cut before it is walked, and the walk.
//
// A table marks an input when its term could reach a bound that holds for every row of a tile.  Once a few strong marks
// have been walked the wavefront knows its own rows' results so far, and the smallest of them over its lanes is a far
// better bound: a mark whose largest possible term stays below it changes nothing in any row and is dropped before its
// operands are fetched.  Selecting and testing costs two gathers per 64 marks; it saves a term for every row of the tile.
// Marks per row before and after, 128 rows of the other operand (512 x 5120 x 5120 unless noted): sort neuron on centred
// activations of spread 0.3 against unit weights 605 -> 176 and, layer by layer of an evaluated network, 123 -> 58,
// 48 -> 32; interval bounds of a 10240-wide network 516 -> 106, 154 -> 64, of its images (12288 inputs, per batch row)
// 543 -> 238; l-inf of images against small weights 328 -> 138.
#pragma once
#include "fwd_tile.h"

namespace sd {

constexpr int kWalkListCap = 2048; // entries of a wavefront's list (16-bit input numbers): the marks of 64 full table words
constexpr int kWalkGroups = 32;    // strong marks that are walked first
// Forms with lists of the K largest: marks of a list of up to 64 that are walked first (an insertion is K instructions per output row
// and list: what a better bound drops pays sooner than for the maxima); lists of up to eight more are walked as they are.
constexpr int walk_short(int K) { return K == 1 ? 0 : K + 6; }
constexpr int kWalkShortMore = 8;
constexpr int kWalkCutMin = 64;    // lists of at most this many marks are walked as they are

// smallest value over the wavefront of a float whose sign bit is clear, as its bit pattern (wave-uniform)
__device__ __forceinline__ float wave_min_nonneg(float f) {
    int v = __builtin_bit_cast(int, f);
    constexpr int none = 0x7fffffff;
    v = min(v, __builtin_amdgcn_update_dpp(none, v, 0x111, 0xf, 0xf, false));   // row_shr:1
    v = min(v, __builtin_amdgcn_update_dpp(none, v, 0x112, 0xf, 0xf, false));   // row_shr:2
    v = min(v, __builtin_amdgcn_update_dpp(none, v, 0x114, 0xf, 0xf, false));   // row_shr:4
    v = min(v, __builtin_amdgcn_update_dpp(none, v, 0x118, 0xf, 0xf, false));   // row_shr:8
    v = min(v, __builtin_amdgcn_update_dpp(none, v, 0x142, 0xa, 0xf, false));   // row_bcast:15 into rows 1 and 3
    v = min(v, __builtin_amdgcn_update_dpp(none, v, 0x143, 0xc, 0xf, false));   // row_bcast:31 into rows 2 and 3
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(v, 63));
}

// sum over this lane and the lanes before it (adds within rows of 16 lanes, then the rows' totals across: no LDS)
__device__ __forceinline__ int wave_prefix_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);    // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);    // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);    // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);    // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2 and 3
    return v;
}

// Lists the marked inputs of a row in ascending order and hands them over, as many at a time as the list holds: at least
// once, also when there are none.  word(c): table word of inputs 32 c .. 32 c + 31, for c < NCH.  use(count, first): walks
// the list.  ready: the number of marks when they are all listed already (of a list that was handed over whole).
// Returns the number of marks when they were handed over whole, otherwise -1.
template <class Word, class Use>
__device__ __forceinline__ int for_marks(uint16_t* list, int NCH, int lane, Word&& word, Use&& use, int ready = -1) {
    int c0 = ready >= 0 ? NCH : 0;
    uint32_t next = ready < 0 && lane < NCH ? word(lane) : 0u;
    bool first = true;
    while (true) {
        int cnt = ready >= 0 ? ready : 0;
        while (c0 < NCH) {
            uint32_t bits = next;
            const int mine = __builtin_popcount(bits), incl = wave_prefix_sum(mine);
            const int total = __builtin_amdgcn_readlane(incl, 63);
            if (cnt + total > kWalkListCap) break;   // (64 words alone always fit)
            if (c0 + 64 < NCH) next = c0 + 64 + lane < NCH ? word(c0 + 64 + lane) : 0u;
            // every lane appends the marks of its word behind those of the lanes before it
            int at = cnt + incl - mine;
            cnt += total;
            while (bits) {
                const int i = __builtin_ctz(bits);
                bits &= bits - 1;
                list[at++] = (uint16_t)(((c0 + lane) << 5) | i);   // (rows of at most 65536 inputs)
            }
            c0 += 64;
        }
        __builtin_amdgcn_wave_barrier();
        use(cnt, first);
        __builtin_amdgcn_wave_barrier();   // the reads of the list come before the next marks
        if (c0 >= NCH) return first ? cnt : -1;
        first = false;
    }
}

__device__ __forceinline__ float lane_value(float v, int k) {   // of lane k, as a scalar operand
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
}

// What a mark brings along from the row that is walked: its weight, or its input (a) and the input's upper bound (b).
struct Own { float a, b; };

// Walks up to 64 marks, one per lane (`n`: the input, `o`; cnt of them), four at a time with the loads of the next four
// in flight.  load(buffer, i, input): issues the loads of mark i of a group, input wave-uniform; use(buffer, i, k, input, o):
// the mark that lane k holds.  Every load is issued unconditionally (groups past the end repeat the last mark and are not
// used), so that the waits the compiler places cover exactly the group that is used next.
template <class Load, class Use>
__device__ __forceinline__ void walk_block(int n, const Own& o, int cnt, Load&& load, Use&& use) {
    auto issue = [&](int buf, int k0) __attribute__((always_inline)) {
        #pragma unroll
        for (int i = 0; i < 4; i++) load(buf, i, __builtin_amdgcn_readlane(n, k0 + i < cnt ? k0 + i : cnt - 1));
    };
    auto spend = [&](int buf, int k0) __attribute__((always_inline)) {
        #pragma unroll
        for (int i = 0; i < 4; i++)
            if (k0 + i < cnt) use(buf, i, k0 + i, __builtin_amdgcn_readlane(n, k0 + i), o);
    };
    issue(0, 0);
    for (int k0 = 0; k0 < cnt; k0 += 8) {
        issue(1, k0 + 4);
        spend(0, k0);
        issue(0, k0 + 8);
        spend(1, k0 + 4);
    }
}

// Walks the listed marks of a row (`total` of them).  Of a long list the first SAMPLE form 32 groups (positions equal modulo
// 32), whose strongest (`excess`, the larger the stronger) are walked first.  Against tiles of batch rows 640 (two gathers per 64
// marks that cost little: positions at 128 x 5120 x 5120, 605 marks, 168 us with 128, 160 with 256, 149; interval bounds of 256 x
// 10240 x 10240 243 -> 235), against tiles of weight rows 128 (their rows come from beyond the die's cache: 256 x 12288 x
// 10240 438 us, 481 with 256, 590).  Then the list goes by 64 marks at a time, and
// of these only those are walked that keep() says can matter now.
//   SHORT: of a list of up to 64 marks, a mark per lane, about so many of the strongest go first and the others by keep(), as in a long
//   list (0: such lists are walked as they are).  Most rows of an evaluated network's later layers have such lists: certification of
//   6 x 5120 at batch 512 1347 -> 1312 us (13 strongest 1324, lists of up to 40 as they are 1318); 16 instead of 32 of the long
//   lists' strongest marks first: 1347 -> 1360.  Not in the values' walk of the sort neuron with positions, which another walk follows: 512 x 5120 x
//   5120 at spreads 0.05 and 0.3 168.3 and 520.2 us without, 170.4 and 521.9 with, 64 x 2048 x 2048 at 0.3 73.3 and 74.2.
//   own(input) -> Own: a gather;  load / use: see walk_block;
//   threshold(strong): brings what keep() compares with up to date, after the strong marks and after every 64;
//   ORDERED: forms for which the order of the inputs counts.  The strong marks are then walked for their values alone, by
//   value(): restart() clears the state behind them, and they go by again with the others, in order; what threshold() has made
//   of their values must not fall again (l-inf of 512 x 5120 x 5120 with positions, everything marked: 521 us when it did, 500;
//   bounds of 250 x 3072 x 1021, forward and backward, 91 and 89).  Only at the first
//   call for a row (`first`): later parts of a long list are cut by what the row has reached.
template <bool ORDERED, bool PAIR, int SAMPLE, int SHORT, class OwnOf, class Excess, class Load, class Value, class Use, class Threshold, class Keep, class Restart>
__device__ __forceinline__ void walk_marks(const uint16_t* list, int total, bool first, int lane, OwnOf&& own, Excess&& excess,
                                           Load&& load, Value&& value, Use&& use, Threshold&& threshold, Keep&& keep,
                                           Restart&& restart) {
    static_assert(kWalkCutMin >= 64, "the strong marks of a long list are taken from one mark per lane at least");
    static_assert(!ORDERED || SHORT == 0, "short lists of ordered forms are walked as they are");
    const bool cut = total > (SHORT ? SHORT + kWalkShortMore : kWalkCutMin);
    int won = -1;
    // marks that are kept move to the first lanes, in their order
    auto gather = [&](bool k, int& n, Own& o) __attribute__((always_inline)) {   // -> how many
        const unsigned long long m = __builtin_amdgcn_ballot_w64(k);
        const int at = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
        const int cnt = __builtin_popcountll(m);
        const int to = (k ? at : cnt + lane - at) << 2;
        n = __builtin_amdgcn_ds_permute(to, n);
        o.a = __builtin_bit_cast(float, __builtin_amdgcn_ds_permute(to, __builtin_bit_cast(int, o.a)));
        if (PAIR) o.b = __builtin_bit_cast(float, __builtin_amdgcn_ds_permute(to, __builtin_bit_cast(int, o.b)));
        return cnt;
    };
    auto strongest = [&](int& n, Own& o) __attribute__((always_inline)) {   // -> how many
        if (SHORT && total <= 64) {   // a mark per lane: the SHORT strongest, and those that are about as strong
            n = (int)list[lane < total ? lane : total - 1];
            o = own(n);
            const int v = lane < total ? __builtin_bit_cast(int, excess(n, o)) : -1;
            int kth = 0;
            #pragma unroll 1
            for (int bit = 30; bit > 17; bit--) {
                const int c = kth | (1 << bit);
                kth = __builtin_popcountll(__builtin_amdgcn_ballot_w64(v >= c)) >= SHORT ? c : kth;
            }
            won = v >= kth ? lane : -1;
            return gather(v >= kth, n, o);
        }
        const int e1 = 64 + lane < total ? 64 + lane : total - 1;
        n = (int)list[lane];
        const int n1 = (int)list[e1];
        o = own(n);
        const Own o1 = own(n1);
        float x = excess(n, o);
        const float x1 = excess(n1, o1);
        won = lane;
        if (x1 > x && 64 + lane < total) { x = x1; n = n1; o = o1; won = e1; }
        for (int e0 = 128; e0 < (total < SAMPLE ? total : SAMPLE); e0 += 64) {
            const int e2 = e0 + lane < total ? e0 + lane : total - 1, n2 = (int)list[e2];
            const Own o2 = own(n2);
            const float x2 = excess(n2, o2);
            if (x2 > x && e0 + lane < total) { x = x2; n = n2; o = o2; won = e2; }
        }
        // the two lanes of a group agree on the stronger of their marks
        const float ox = __shfl_xor(x, 32);
        const int on = __shfl_xor(n, 32), ow = __shfl_xor(won, 32);
        const float oa = __shfl_xor(o.a, 32), ob = PAIR ? __shfl_xor(o.b, 32) : oa;
        if (ox > x || (!(x > ox) && ow < won)) { n = on; o.a = oa; o.b = ob; won = ow; }
        return kWalkGroups;
    };
    auto block = [&](int b, int& n, Own& o) __attribute__((always_inline)) {   // -> how many are left
        const int e = b + lane;
        n = (int)list[e < total ? e : total - 1];
        o = own(n);
        if (!cut) return total - b < 64 ? total - b : 64;
        return gather(e < total && keep(n, o) && (ORDERED || e != won), n, o);
    };
    int n = 0;
    Own o{};
    if constexpr (ORDERED) {
        if (cut && first) {
            strongest(n, o);
            walk_block(n, o, kWalkGroups, load, value);
            threshold(true);
            restart();
        } else if (cut) threshold(false);
        for (int b = 0; b < total; b += 64) {
            const int cnt = block(b, n, o);
            walk_block(n, o, cnt, load, use);
            if (cut && b + 64 < total) threshold(false);
        }
    } else {
        // one loop for both, so that the walk is expanded once (and without a branch round it: that would cost a copy of
        // the state)
        for (int b = cut ? -64 : 0; b < total; b += 64) {
            const int cnt = b < 0 ? strongest(n, o) : block(b, n, o);
            walk_block(n, o, cnt, load, use);
            if (cut && b + 64 < total) threshold(b < 0);
        }
    }
}

// Top-K lists are kept as the bit patterns of their values (all >= 0, where signed integers order like the floats), ascending:
// new[k] = max(res[k], min(res[k+1], v)) (core/cuda/sort_neuron.cu:76-77) = the median of the three, one integer instruction
// per slot.  A negative v (sign bit set: a negative integer) is below every entry and changes nothing; an undefined v with a
// clear sign bit would order above every number, so callers hand over defined values only.
__device__ __forceinline__ int imed3(int a, int b, int c) {
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
template <int K>
__device__ __forceinline__ void insert_bits(int (&res)[K], float value) {
    const int v = __builtin_bit_cast(int, value);
    #pragma unroll
    for (int k = 0; k < K - 1; k++) res[k] = imed3(res[k], v, res[k + 1]);
    res[K - 1] = max(res[K - 1], v);
}
// One value for each of two lists.  An insertion that would change neither list in any lane is left out: of 123 marks per
// row (K = 10) 83 change one when they go by in the order of the inputs, 36 with the strong ones first.
template <int K>
__device__ __forceinline__ void insert_pair(int (&ra)[K], float a, int (&rb)[K], float b) {
    if constexpr (K > 2) {
        if (__builtin_amdgcn_ballot_w64(__builtin_bit_cast(int, a) > ra[0] || __builtin_bit_cast(int, b) > rb[0]) == 0ull) return;
    }
    insert_bits<K>(ra, a);
    insert_bits<K>(rb, b);
}

template <int K>
__device__ __forceinline__ float geo_sum_bits(const int (&res)[K], float q) {
    float f[K];
    #pragma unroll
    for (int k = 0; k < K; k++) f[k] = __builtin_bit_cast(float, res[k]);
    return geo_sum<K>(f, q);
}

}  // namespace sd
