// dm_plan.h -- launch arithmetic that a kernel and its host code share, or
// that decides which kernel takes a call.  Plain constexpr functions without
// any HIP, so that a CPU program can check them over every size.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace dm {

// The grouped-experts launch of `pairs` (token, selection) pairs: its entries
// (an expert and up to 8 of its tokens) are found on the device, and each
// workgroup works on one entry.  Two workgroups per CU, and never fewer than
// the entries, of which there are at most as many as pairs: a partition of 32
// CUs has 64 workgroups where 16 tokens can make 128 entries.
constexpr uint32_t experts_grid(uint32_t cus, uint32_t pairs) { return 2 * cus > pairs ? 2 * cus : pairs; }
// Workgroups per entry; workgroup b works on entry b / share, if there is one.
constexpr uint32_t experts_share(uint32_t grid, uint32_t entries) { return grid > entries ? grid / entries : 1u; }

// Whether a resident layer call's tokens are grouped by expert on the device
// (each selected expert streamed once for all its tokens by the fp16 kernel)
// rather than run as one int8 job per pair of token and selection.
//  * One token shares nothing: never.
//  * More than 8 tokens or max_jobs pairs: always (else the host forms the
//    launches after a round trip: 10 tokens of 1024 x 512, 60 experts top 2,
//    47 against 61 us).
//  * Otherwise where the pairs' experts come to 140 MB and grouping is expected
//    to save 20 MB of them (selections spread evenly over the experts).  In us,
//    per pair / grouped, with the MB saved:
//      4096 x 1536, 32 experts top 4: 2 tokens 51 / 63 (6), 3 65 / 69 (18),
//      4 75 / 75 (34), 5 90 / 78 (54);
//      4096 x 1536, 64 experts top 2: 7 tokens 69 / 74 (15), 8 78 / 77 (21);
//      2048 x 768, 128 experts top 8: 4 tokens 63 / 64 (9), 6 78 / 73 (21);
//      4096 x 1024, 64 experts top 8: 2 tokens 61 / 67 (8), 3 80 / 76 (24);
//      6144 x 2048, 16 experts top 8: 1 token 71 / 84 (0), 2 107 / 105 (98),
//      3 143 / 115; 1024 x 512, 32 experts top 8 (65 MB in all): 8 47 / 48 (35).
constexpr bool moe_groups_by_expert(uint64_t batch, uint64_t k, uint64_t experts, uint64_t expert_bytes, uint64_t max_jobs) {
    if (batch < 2) return false;
    const uint64_t pairs = batch * k;
    if (batch > 8 || pairs > max_jobs) return true;
    double none = 1.0;  // chance that no token selects a given expert
    for (uint64_t t = 0; t < batch; t++) none *= 1.0 - (double)k / (double)experts;
    const double shared = (double)pairs - (double)experts * (1.0 - none);
    return (double)pairs * (double)expert_bytes >= 140.0 * (1 << 20) && shared * (double)expert_bytes >= 20e6;
}

// ---- decode matvecs of Q4_K and Q6_K: the int8 kernel or the fp16 one ----
// The int8 kernel (kernels_qmv8.hip) takes each token's records through the
// matrix cores apart and lets every wave build those of its columns, so its
// work per block grows with the tokens and its prologue with the columns; it
// splits K so that a launch has at least 4096 waves, 16 per CU, and a launch
// of more than that and less than twice as many leaves part of its second
// round empty.  The fp16 kernel (kernels_qmv.hip) costs as much for 1 token as
// for 8, and its prologue about 2 us more.  One token: always int8; four or
// more, and three of Q6_K: always fp16.  Between them, int8 / fp16 in us over
// rotating matrices:
//   Q4_K, 2 tokens
//     up to 4096 rows, by columns: 1024 x 5120 6.1 / 6.3, x 6144 6.5 / 6.4,
//     x 8192 8.2 / 6.5; 1536 x 7168 7.5 / 7.8, x 8192 8.3 / 7.8; 2048 x 7168
//     7.5 / 7.9, x 8192 8.3 / 7.9; 4096 x 8192 9.3 / 11.2, x 10240 10.1 / 11.1,
//     x 12288 12.3 / 11.6
//     above, short rows: 12288 x 2048 6.9 / 8.5, 40960 x 1024 8.8 / 9.6, 65536
//     x 2048 16.2 / 16.8, 6144 x 3072 7.0 / 7.6; 10240 x 3072 9.3 / 8.7
//     4096 waves: 8192 x 5120 10.0 / 10.8, x 6144 11.9 / 11.0; 16384 x 4096
//     10.8 / 11.4; 32768 x 6144 26.1 / 26.6, x 8192 40.1 / 33.7; beside them
//     7168 x 5120 11.3 / 10.7, 12288 x 4096 11.4 / 10.2, 20480 x 4096 15.5 / 12.8
//     persistent waves (above 65536 rows): 98304 x 5120 59.0 / 60.6, 151936 x
//     6144 98.3 / 109.7, x 8192 140 / 135
//   Q6_K, 2 tokens
//     up to 4096 rows: 1024 x 3072 6.5 / 6.8, x 4096 7.0 / 5.7; 2048 x 5120
//     7.9 / 9.2, x 6144 8.5 / 7.7; 4096 x 7168 10.6 / 11.5, x 8192 12.1 / 11.6,
//     1024 x 16384 93.8 / 8.9
//     above: 8192 x 2048 7.3 / 8.0, 12288 x 2048 9.7 / 9.8, 24576 x 1024 9.0 /
//     9.7, 7168 x 3072 9.3 / 8.4; 28672 x 1024 11.1 / 9.6, 14336 x 2048 11.8 /
//     9.9; of 4096 waves 16384 x 2048 9.4 / 9.9, 32768 x 1024 9.4 / 9.8, 32768
//     x 2048 14.5 / 14.2
//     heads: 98304 x 4096 70.5 / 69.5, 151936 x 4096 107 / 109, x 5120 131 / 137
//   Q4_K, 3 tokens: 1024 x 2048 5.1 / 5.5, 1536 x 4096 6.9 / 7.4, x 3072 7.0 /
//     6.4, x 1536 5.9 / 5.5, 1024 x 4096 6.9 / 5.9; 2048 x 5120 7.5 / 8.8, x 6144
//     8.3 / 7.2; 4096 x 6144 9.1 / 9.6, x 8192 11.6 / 11.1; 8192 x 2048 7.2 / 7.3,
//     10240 x 2048 9.5 / 8.5, 8192 x 3072 9.2 / 7.7
constexpr bool qmv8_faster(bool q6_k, uint64_t rows, uint64_t columns, uint64_t batch) {
    if (batch == 1) return true;
    if (batch > 3 || (batch == 3 && q6_k)) return false;
    // (three tokens of few rows: only where the split leaves each wave one block)
    if (batch == 3 && rows < 2048) return (columns == 2048 && rows >= 1024) || (columns == 4096 && rows >= 1536);
    const bool q4_pair = !q6_k && batch == 2;
    if (rows <= 4096) return q4_pair ? columns < 4608 + 7 * rows / 4 : columns < 8192 && columns < 2304 + 7 * rows / 4;
    const uint64_t tiles = (rows + 15) / 16, weights = rows * columns, m = 1u << 20;
    const bool whole = tiles > 4096 || 4096 % tiles == 0;  // whole rounds of waves
    if (q4_pair)
        return columns <= 2048 || (columns <= 3072 && rows <= 8192) || (whole && columns <= (rows > 16384 ? 6144 : 5120));
    if (batch == 3) return columns <= 2048 && weights <= 16 * m;
    return (columns <= 2048 && weights <= (whole ? 32 : 24) * m) || (columns <= 8192 && weights > 300 * m);
}

// ---- the fp16 matvec (kernels_qmv.hip) ----
struct QmvPlan {
    uint32_t kb, waves, wave_k, k_parts, row_groups, phases;
};

// The K split.  A workgroup of 16 waves of up to 128 registers holds the
// fragments of 8 tokens of up to 32 blocks (2 per wave; a gate/up pair, which
// needs more registers besides, 16), one of 8 waves of 256 those of 16
// tokens of 16 blocks, or of 8 tokens of a pair's 24.  Longer rows, and
// matrices with fewer tiles than CUs, are split over k_parts workgroups;
// gate/up pairs, whose epilogue needs whole sums, go through longer rows in
// phases instead.  The split minimises the largest workgroup's share of the
// weights; within it, the most waves share K.
constexpr QmvPlan qmv_split(uint32_t parts, uint32_t tiles, uint32_t blocks, uint32_t batch, int mode, uint32_t cus) {
    QmvPlan p{};
    p.k_parts = parts;
    const uint32_t part_blocks = (blocks + parts - 1) / parts;
    p.phases = 1;
    if (batch <= 8 && part_blocks <= (mode == 2 ? 16u : 32u)) {
        p.waves = 16;
    } else {
        p.waves = 8;
        if (part_blocks > (batch <= 8 ? 24u : 16u)) p.phases = (part_blocks + 15) / 16;
    }
    p.row_groups = cus / parts < tiles ? cus / parts : tiles;
    const uint32_t phase_blocks = (part_blocks + p.phases - 1) / p.phases;
    p.kb = (phase_blocks + p.waves - 1) / p.waves;
    p.wave_k = (phase_blocks + p.kb - 1) / p.kb;
    return p;
}

constexpr QmvPlan qmv_plan(uint32_t rows, uint32_t blocks, uint32_t batch, int mode, uint32_t cus, uint32_t meet_words) {
    const uint32_t tiles = (rows + 15) / 16;
    QmvPlan best{};
    double best_cost = 0.0;
    for (uint32_t parts = 1; parts <= 8 && parts <= blocks && parts <= cus; parts *= 2) {
        if (parts > 1 &&
            (mode == 2 || (uint64_t)tiles * (parts - 1) * ((batch + 1) / 2) * 16 > meet_words))
            break;
        const QmvPlan p = qmv_split(parts, tiles, blocks, batch, mode, cus);
        const uint32_t part_blocks = (blocks + parts - 1) / parts;
        const uint32_t per = (tiles + p.row_groups - 1) / p.row_groups;
        // tile blocks the busiest workgroup streams, plus the cost of a
        // meeting (a round trip of an atomic, as long as about ten tile
        // blocks) and of rebuilding the fragments of every pass
        const double cost =
            (double)per * part_blocks + (parts > 1 ? 10.0 : 0.0) + (p.phases > 1 ? 8.0 * p.phases * per : 0.0);
        if (best.k_parts == 0 || cost < best_cost) {
            best = p;
            best_cost = cost;
        }
    }
    return best;
}

// First block of run u of `units` (a run is one wave's blocks in one phase of
// one part; u = units: the end).  In 32 bits: the kernels work it out in their
// loops, where a wider division, or a second one for the remainder, costs 3 to
// 16% of a call.
constexpr uint32_t run_begin(uint32_t u, uint32_t units, uint32_t blocks) { return u * blocks / units; }
// Whether that product stays within 32 bits whatever split the plan takes.  A
// wave holds at most 3 blocks, so every split has more than blocks / 3 runs, and
// rows from 92682 blocks (23.7 million columns) on do not fit; shorter ones from
// 65536 blocks on are looked at split by split.
constexpr bool qmv_runs_fit(uint32_t blocks, uint32_t batch, int mode) {
    for (uint32_t parts = 1; parts <= (mode == 2 ? 1u : 8u); parts *= 2) {
        const QmvPlan p = qmv_split(parts, 1, blocks, batch, mode, parts);
        if ((uint64_t)p.wave_k * p.k_parts * p.phases * blocks > 0xffffffffull) return false;
    }
    return true;
}

// ---- the prefill GEMM (kernels_gemm.hip) ----
constexpr uint32_t kGemmRows = 128;   // tile height, to which the workspace rows are padded
constexpr uint32_t kGemmWaves = 4;    // waves of a workgroup, each with a quarter of K
constexpr uint64_t gemm_padded_rows(uint64_t m) { return (m + kGemmRows - 1) / kGemmRows * kGemmRows; }
// LDS of the A preparation: 8 rows of the largest quarter's columns as bf16.
constexpr uint64_t gemm_prep_lds(uint64_t k) {
    const uint64_t blocks = k / 256, quarter = (blocks + kGemmWaves - 1) / kGemmWaves;
    return 8 * (quarter * 128 + 4) * 4;
}
// Whether the MFMA path takes a product of m x k activations with n encoded
// rows of w_bytes in all: more than 16 tokens (fewer stream W faster through
// the decode matvec), whole 256-column blocks, offsets that fit the 31-bit
// buffer range, and a quarter of K that the preparation can stage in the 160
// KiB of LDS (up to 39936 columns; longer rows go to the decode matvec, 16
// tokens at a time).  The stores of the rows past m in the last tile rely on
// their offsets lying past the end of C, so those offsets may not wrap at 32
// bits: at 17 rows (padded to 128) n stops at 8388608.
constexpr bool gemm_fits_mfma(uint64_t m, uint64_t n, uint64_t k, uint64_t w_bytes) {
    return m > 16 && k % 256 == 0 && gemm_prep_lds(k) <= 160 * 1024 && w_bytes + 1024 < 0x7fffffffull &&
           gemm_padded_rows(m) * k * 2 < 0x7fffffffull && m * n * 4 < 0x7fffffffull &&
           gemm_padded_rows(m) * n * 4 <= 0x100000000ull;
}

}  // namespace dm
