// How the grouped matrix product for prompts (moe_prefill.hip) is cut into workgroups: host arithmetic, and a step of the
// grouping kernel that the host can run as well.
#pragma once

#include <cmath>
#include <cstdint>
#include <initializer_list>

constexpr uint32_t kPfChain = 32;   // blocks of a row from which on its sums are folded: more

struct pf_shape {
    uint32_t cus, hidden, inter, experts, top_k, tokens;
};

// The forms of the product: one chain of sums a row; folded sums with twelve, eight or four waves a workgroup; folded sums of
// items of at most 32 pairs with eight.
enum pf_form : uint32_t { kChain, kTwelve, kEight, kFour, kNarrow };

// Items that runs of at most `cols` pairs make of the experts' lists, each about Poisson.
inline double pf_items(const pf_shape &a, uint32_t cols) {
    const double mean = (double)a.tokens * a.top_k / a.experts, six = 6.0 * std::sqrt(mean);
    const double sure = std::floor(std::fmax(mean - six, 0.0) / cols);   // that every list is longer than
    double items = 1.0 - std::exp(-mean) + sure;
    for (double k = (sure + 1.0) * cols; k < mean + six; k += cols) items += 0.5 * std::erfc((k + 0.5 - mean) / std::sqrt(2.0 * mean));
    return a.experts * items;
}

// What a form takes, for rows of more than kPfChain blocks: rounds of its workgroups, half of a last one that is not full, times
// what a round takes (relative; measured a step of 64 at 16 shapes of 1024 .. 4096 / 256 .. 1536, 32 .. 256 experts of 13 .. 225
// pairs).  Twelve waves read the activations least often, four make the finest rounds and share a CU with another
// workgroup from half a round on; the narrow form's items are of 32 pairs, four waves a SIMD.  us of gate/up, twelve, eight, four, narrow:
// 2816 / 704, top-8 of 128, 1000 tokens 208, 226, 225, 248; 2304 / 1280, top-2 of 32, 1000 tokens 90, 78, 87, 92;
// 4096 / 448, top-4 of 32, 300 tokens 76, 55, 48, 47; 1920 / 896, top-4 of 256, 1000 tokens 191, 204, 203, 170.
inline double pf_estimate(const pf_shape &a, pf_form form, double items, uint32_t rows, uint32_t rows_a_wave) {
    const uint32_t waves = form == kTwelve ? 12u : form == kFour ? 4u : 8u, per_cu = form == kTwelve || form == kEight ? 1u : 2u;
    const double r = items * ((rows + waves * rows_a_wave - 1u) / (waves * rows_a_wave)) / (per_cu * a.cus);
    const double whole = std::fmax(1.0, std::ceil(r - 0.05));
    const double cost = form == kTwelve ? 1.85 : form == kEight ? 1.34 : form == kFour ? (r <= 0.5 ? 1.15 : r < 1.0 ? 1.3 : 1.45) : r < 1.0 ? 1.5 : 2.27;
    return cost * 0.5 * (whole + r);
}

// One chain a row (up to kPfChain blocks): always eight waves, four a SIMD.  (2048 / 512, top-8 of 256, 1000 tokens, down: 78 us;
// with three activation buffers and two waves a SIMD 95.)
inline pf_form pf_form_of(const pf_shape &a, bool paired, double items, bool narrow) {
    if ((paired ? a.hidden : a.inter) <= 32u * kPfChain) return kChain;
    const uint32_t rows = paired ? a.inter : a.hidden, rows_a_wave = paired ? 16u : 32u;
    pf_form best = kTwelve;
    double least = pf_estimate(a, best, items, rows, rows_a_wave);
    for (pf_form f : {kEight, kFour, kNarrow}) {
        const double t = pf_estimate(a, f, items, rows, rows_a_wave);
        if ((f != kNarrow || narrow) && t < least) best = f, least = t;
    }
    return best;
}

struct pf_plan {
    uint32_t cols;   // pairs of an item at most
    pf_form gate_up, down;
};
// Items are cut for both products: to 32 pairs if the gate/up product is the faster for it, in the narrow form.
inline pf_plan pf_plan_of(const pf_shape &a) {
    const double wide = pf_items(a, 64u), narrow = pf_items(a, 32u);
    const pf_form gu = pf_form_of(a, true, wide, false);
    if (gu != kChain && pf_estimate(a, kNarrow, narrow, a.inter, 16u) < pf_estimate(a, gu, wide, a.inter, 16u))
        return pf_plan{32u, kNarrow, pf_form_of(a, false, narrow, true)};
    return pf_plan{64u, gu, pf_form_of(a, false, wide, false)};
}

// Ranks of a token's pairs k0 .. k0 + 7 among their experts' (rank[u], of own[u]; -1 for a pair that is dropped): add(w) adds one to
// word w of the counts and returns what it held.  A dropped pair counts in word 2 * experts: with no lane's branch around each,
// a token's atomics are in flight together.  Slots past top_k add nowhere (how many there are is the same for the whole workgroup):
// 64 lanes that add to one word take the LDS 64 turns.  The grouping kernel, 1000 tokens of 128 experts, us with eight adds a token
// and with top_k: top-2 10.8 and 7.6, top-4 10.3 and 8.8; top-2 of 32, 4000 tokens 33.0 and 22.7.
template <uint32_t N, class ADD>
constexpr void pf_rank_first(const int32_t (&own)[8], const bool (&ok)[8], uint32_t experts, ADD add, int32_t (&rank)[8]) {
    for (uint32_t u = 0; u < N; ++u) rank[u] = add(ok[u] ? (uint32_t)own[u] : 2u * experts);
    for (uint32_t u = 0; u < 8u; ++u) rank[u] = u < N && ok[u] ? rank[u] : -1;
}
template <class ADD>
constexpr void pf_rank_pairs(const int32_t (&own)[8], const bool (&ok)[8], uint32_t k0, uint32_t top_k, uint32_t experts, ADD add,
                             int32_t (&rank)[8]) {
    switch (top_k - k0) {
        case 1: return pf_rank_first<1>(own, ok, experts, add, rank);
        case 2: return pf_rank_first<2>(own, ok, experts, add, rank);
        case 3: return pf_rank_first<3>(own, ok, experts, add, rank);
        case 4: return pf_rank_first<4>(own, ok, experts, add, rank);
        case 5: return pf_rank_first<5>(own, ok, experts, add, rank);
        case 6: return pf_rank_first<6>(own, ok, experts, add, rank);
        case 7: return pf_rank_first<7>(own, ok, experts, add, rank);
        default: return pf_rank_first<8>(own, ok, experts, add, rank);
    }
}
