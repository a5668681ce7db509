"""CPU checks of the launch arithmetic that kernels and host code share
(diskmule_amd/csrc/dm_plan.h): the header is compiled with the host compiler
and its functions are run over whole ranges of sizes."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include "dm_plan.h"
extern "C" {
uint32_t experts_grid(uint32_t cus, uint32_t pairs) { return dm::experts_grid(cus, pairs); }
uint32_t experts_share(uint32_t grid, uint32_t entries) { return dm::experts_share(grid, entries); }
void qmv_plan(uint32_t rows, uint32_t blocks, uint32_t batch, int mode, uint32_t cus, uint32_t *out) {
    const dm::QmvPlan p = dm::qmv_plan(rows, blocks, batch, mode, cus, 512 * 1024);
    const uint32_t v[6] = {p.kb, p.waves, p.wave_k, p.k_parts, p.row_groups, p.phases};
    for (int i = 0; i < 6; i++) out[i] = v[i];
}
int moe_groups_by_expert(uint64_t batch, uint64_t k, uint64_t experts, uint64_t bytes) {
    return dm::moe_groups_by_expert(batch, k, experts, bytes, 64);
}
int qmv8_faster(int q6_k, uint64_t rows, uint64_t columns, uint64_t batch) {
    return dm::qmv8_faster(q6_k, rows, columns, batch);
}
uint64_t gemm_prep_lds(uint64_t k) { return dm::gemm_prep_lds(k); }
int gemm_fits_mfma(uint64_t m, uint64_t n, uint64_t k, uint64_t w_bytes) { return dm::gemm_fits_mfma(m, n, k, w_bytes); }
int qmv_runs_fit(uint32_t blocks, uint32_t batch, int mode) { return dm::qmv_runs_fit(blocks, batch, mode); }
// Whether the runs are consecutive, cover all blocks and hold at most `most` each.
int runs_cover(uint32_t units, uint32_t blocks, uint32_t most) {
    uint64_t at = 0;
    for (uint32_t u = 0; u < units; u++) {
        const uint64_t lo = dm::run_begin(u, units, blocks), hi = dm::run_begin(u + 1, units, blocks);
        if (lo != at || hi < lo || hi - lo > most) return 0;
        at = hi;
    }
    return at == blocks;
}
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plans")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "diskmule_amd", "csrc"), str(d / "shim.cpp"), "-o", str(d / "shim.so")],
                   check=True)
    lib = ctypes.CDLL(str(d / "shim.so"))
    for name in ("experts_grid", "experts_share"):
        getattr(lib, name).restype = ctypes.c_uint32
    lib.qmv8_faster.argtypes = [ctypes.c_int] + [ctypes.c_uint64] * 3
    lib.gemm_prep_lds.restype = ctypes.c_uint64
    lib.gemm_prep_lds.argtypes = [ctypes.c_uint64]
    lib.moe_groups_by_expert.argtypes = [ctypes.c_uint64] * 4
    lib.gemm_fits_mfma.argtypes = [ctypes.c_uint64] * 4
    return lib


def test_every_grouped_expert_entry_has_workgroups(plan):
    """Whatever the CU count (a partition may show 32 or fewer) and however
    the pairs fall on experts (1 to `pairs` entries), every entry is some
    workgroup's, each entry's workgroups are numbered 0 .. share - 1, and a
    whole MI355X keeps two workgroups per CU."""
    for cus in (1, 4, 16, 31, 32, 38, 64, 80, 128, 256, 304):
        for pairs in range(1, 129):
            grid = plan.experts_grid(cus, pairs)
            assert grid >= 2 * cus
            for entries in range(1, pairs + 1):
                share = plan.experts_share(grid, entries)
                assert share >= 1 and (entries - 1) * share + share - 1 < grid, (cus, pairs, entries)
    assert all(plan.experts_grid(256, pairs) == 512 for pairs in range(1, 129))


def test_tokens_are_grouped_by_expert_only_where_they_share(plan):
    """One token, or tokens that can hardly share an expert, never; calls that
    the one-job-per-pair launches do not take, always; between them only
    where enough bytes are saved (the measured calls on either side)."""
    mb = 1 << 20
    for k, experts in ((1, 1), (8, 8), (8, 16), (8, 128), (64, 64), (100, 128)):
        assert not plan.moe_groups_by_expert(1, k, experts, 1000 * mb)
        assert plan.moe_groups_by_expert(9, k, experts, mb) and plan.moe_groups_by_expert(16, k, experts, mb)
    assert plan.moe_groups_by_expert(2, 33, 128, mb)  # 66 pairs
    size = {(2048, 768): 3059712, (4096, 1536): 12238848, (4096, 1024): 8159232, (6144, 2048): 24477696, (1024, 512): 1019904}
    for shape, experts, k, batch, grouped in (
            ((2048, 768), 128, 8, 4, False), ((2048, 768), 128, 8, 6, True), ((4096, 1536), 32, 4, 3, False),
            ((4096, 1536), 32, 4, 5, True), ((4096, 1536), 64, 2, 7, False), ((4096, 1024), 64, 8, 2, False),
            ((4096, 1024), 64, 8, 3, True), ((6144, 2048), 16, 8, 1, False), ((6144, 2048), 16, 8, 3, True),
            ((1024, 512), 32, 8, 8, False)):
        assert bool(plan.moe_groups_by_expert(batch, k, experts, size[shape])) == grouped, (shape, experts, k, batch)


def test_matvecs_of_two_and_three_tokens_take_the_faster_kernel(plan):
    """Shapes measured on both kernels, on either side of every line of the
    rule: long rows leave the int8 kernel also where the matrix is small, short
    rows keep it also where it is large."""
    q4, q6 = 0, 1
    int8 = [(q4, 1024, 5120, 2), (q4, 1536, 7168, 2), (q4, 2048, 7168, 2), (q4, 4096, 8192, 2),
            (q4, 12288, 2048, 2), (q4, 32768, 1024, 2), (q4, 6144, 3072, 2), (q4, 8192, 5120, 2), (q4, 32768, 6144, 2), (q4, 151936, 4096, 2),
            (q6, 1024, 3072, 2), (q6, 2048, 5120, 2), (q6, 4096, 7168, 2), (q6, 24576, 1024, 2), (q6, 16384, 2048, 2),
            (q6, 151936, 5120, 2), (q4, 1024, 2048, 3), (q4, 1536, 4096, 3),
            (q4, 2048, 5120, 3), (q4, 4096, 6144, 3), (q4, 8192, 2048, 3)]
    fp16 = [(q4, 1024, 8192, 2), (q4, 2048, 8192, 2), (q4, 4096, 12288, 2), (q4, 6144, 4096, 2), (q4, 12288, 4096, 2),
            (q4, 8192, 8192, 2), (q4, 32768, 8192, 2), (q6, 1024, 4096, 2), (q6, 4096, 8192, 2), (q6, 1024, 16384, 2),
            (q6, 7168, 3072, 2), (q6, 32768, 2048, 2), (q6, 32768, 16384, 2), (q4, 1024, 4096, 3), (q4, 1536, 3072, 3),
            (q4, 4096, 8192, 3), (q4, 8192, 3072, 3), (q6, 4096, 4096, 3), (q4, 4096, 4096, 4), (q6, 4096, 4096, 4)]
    assert all(plan.qmv8_faster(*case) for case in int8), [c for c in int8 if not plan.qmv8_faster(*c)]
    assert not any(plan.qmv8_faster(*case) for case in fp16), [c for c in fp16 if plan.qmv8_faster(*c)]
    assert all(plan.qmv8_faster(q, rows, columns, 1) for q in (q4, q6) for rows in (1, 16, 5000, 151936)
               for columns in (256, 4096, 65536))


BLOCKS = [*range(1, 70), 95, 96, 97, 112, 127, 128, 129, 208, 256, 257, 512, 1000, 4096, 65535, 65536, 92681, 92682,
          131072, 1000003, (1 << 24) - 1]


@pytest.mark.parametrize("mode", [0, 2])
def test_fp16_matvec_plans_give_every_block_to_a_wave(plan, mode):
    """Every plan of the fp16 matvec: it is one of the compiled forms, and the
    runs of its waves, parts and phases are consecutive, cover all blocks of
    K and are no longer than the blocks a wave holds fragments for; the rows
    of so many blocks that a run's start passes 32 bits are not taken."""
    assert all(plan.qmv_runs_fit(blocks, batch, mode) for batch in (1, 16) for blocks in range(1, 65536, 7))
    assert not any(plan.qmv_runs_fit(blocks, batch, mode) for batch in (1, 16) for blocks in range(92682, 1 << 24, 9973))
    out = (ctypes.c_uint32 * 6)()
    for cus in (32, 256):
        for rows in (1, 16, 17, 300, 4096, 20000, 151936):
            for batch in (1, 2, 8, 9, 16):
                for blocks in BLOCKS:
                    plan.qmv_plan(rows, blocks, batch, mode, cus, out)
                    kb, waves, wave_k, parts, row_groups, phases = out
                    case = (cus, rows, batch, blocks, list(out))
                    assert 1 <= wave_k <= waves and parts * row_groups <= cus and (parts == 1 or mode == 0), case
                    tiles = -(-rows // 16)
                    assert parts == 1 or tiles * (parts - 1) * ((batch + 1) // 2) * 16 <= 512 * 1024, case
                    if phases > 1 or batch > 8:
                        assert waves == 8 and 1 <= kb <= 2, case
                    elif waves == 8:
                        assert mode == 2 and kb == 3, case
                    else:
                        assert waves == 16 and 1 <= kb <= (2 if mode == 0 else 1), case
                    if plan.qmv_runs_fit(blocks, batch, mode):
                        assert plan.runs_cover(wave_k * parts * phases, blocks, kb), case
                    else:
                        assert blocks > 0xffff, case


def test_prefill_gemm_stages_a_quarter_of_k_in_lds(plan):
    """The preparation's LDS never passes a workgroup's 160 KiB on a shape that
    the MFMA path takes; 39936 columns are its last."""
    for k in range(256, 200000, 256):
        taken = plan.gemm_fits_mfma(17, 64, k, 64 * (k // 256) * 210)
        assert bool(taken) == (k <= 39936) and (not taken or plan.gemm_prep_lds(k) <= 160 * 1024), k


def test_prefill_gemm_stores_of_padding_rows_stay_past_the_end(plan):
    """No store of a row past m reaches C: the 32-bit offset of every padding
    row's columns is past C's end, also at the most columns that fit."""
    for m in (17, 40, 127, 129, 200, 1000, 2049):
        padded = -(-m // 128) * 128
        edge = (1 << 32) // (4 * padded)  # the last n whose padded rows end within 2^32 bytes
        for n in sorted({64, 5000, edge - 1, edge, edge + 1, 2 * edge, ((1 << 31) - 4) // (4 * m)}):
            if not plan.gemm_fits_mfma(m, n, 256, 144 * n):
                assert n > edge or 144 * n + 1024 >= 0x7fffffff or m * n * 4 >= 0x7fffffff, (m, n)
                continue
            assert ((padded - 1) * n + n - 1) * 4 < 1 << 32, (m, n)  # (they start at m * n * 4, C's end)
