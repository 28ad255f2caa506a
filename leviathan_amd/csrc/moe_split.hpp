// How the rows of the few-token expert kernels are cut into workgroups: plain arithmetic, without the device.
#pragma once

#include <cstdint>

// The schedule field that stands for the rule below; any other one is a number of workgroups a CU.
constexpr uint32_t kGateUpPerCu = 2;

// Rows of a gate/up workgroup (moe_gate_up_mfma).  A group is 16 rows.  `most` workgroups of one group fit a CU at once:
// while three rounds of them hold all rows, a workgroup takes one group, as small as the same number of workgroups a
// CU allows (3968 / 1472, top-6, one token: 18 rows a workgroup are two groups, the second of two rows); beyond, several
// whole groups with the next one's weights in flight.  At least two workgroups a CU.
inline uint32_t moe_gate_up_rows(uint32_t cus, uint32_t hidden, uint32_t inter, uint32_t pairs, uint32_t per_cu) {
    if (per_cu != kGateUpPerCu) {
        const uint64_t chunks = ((uint64_t)cus * per_cu + pairs - 1u) / pairs;   // of a pair's rows
        return (uint32_t)((inter + chunks - 1u) / chunks);
    }
    const uint64_t rows = (uint64_t)inter * pairs, most = hidden <= 2048u ? 4u : 2u;
    uint64_t per = (rows + 16u * cus - 1u) / (16u * cus);                        // groups a CU
    if (per > most) per = (per + most - 1u) / most * most;                       // whole rounds
    if (per < 2u) per = 2u;
    const uint64_t want = per <= 3u * most && (most == 2u || per <= most) ? (rows + per * cus - 1u) / (per * cus)
                                                                          : 16u * ((rows + 32u * cus - 1u) / (32u * cus));
    return want < inter ? (uint32_t)want : inter;
}
