"""Which kernel and tile a bf16 or fp32 product takes (gemm_choice.hpp), on the
256 compute units of an MI355X, the cases of the ring kernel's GPU tests among
them."""

from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import pytest

from conftest import ROOT
from test_gemm_ring_gpu import CASES, F32_CASES

UNITS = 256
RING = ["64x32 alone", "64x64", "64x64 alone", "64x64 deep", "128x64", "128x128", "128x128 deep"]


@pytest.fixture(scope="module")
def rules():
    library = Path(ROOT) / "tests" / "cpp" / "bin" / "libinternals.so"
    if not library.exists():
        subprocess.run(["make", "-s", "-C", str(library.parents[1])], check=True)
    return ctypes.CDLL(str(library))


def bf16(rules, m, n, k, gelu=False, count=1, persistent_fits=None):
    fits = n % 256 == 0 and k >= 256 and count == 1 if persistent_fits is None else persistent_fits
    choice = rules.bf16_choice(m, n, k, count, int(gelu), int(fits), UNITS)
    return RING[choice] if choice < 100 else f"persistent {choice - 100}"


@pytest.mark.parametrize("m,n,k,gelu,expected", [
    # 63 of an XCD's 64 slots: 15.8 to 22.8 us by card on 128 x 128 tiles.
    (3152, 2304, 768, False, "persistent 192"),
    # 70 tiles for the 64 slots of one XCD, though 500 for 512 over the chip: 28.1 against 24.4 us.
    (3200, 2560, 640, True, "persistent 192"),
    (3152, 2560, 640, True, "persistent 192"),
    # Three rounds: 24 to 32 us by where the operands come from, against 21 to 24.
    (4616, 2304, 768, False, "persistent 256"),
    # 60 and 54 of 64 slots: the ring, 14.0 against 17.4 and 16.6 against 21.3 us.
    (4616, 1536, 384, True, "128x128"),
    (8224, 768, 768, False, "128x128"),
    # Short K: the ring only by more.
    (9232, 768, 256, False, "persistent 192"),
    (6304, 1024, 256, True, "128x128"),
    # 128 x 64 tiles would fill every CU but leave none over.
    (394, 4096, 1024, True, "64x64 deep"),
    (12608, 3072, 768, True, "persistent 320"),
    (12608, 2304, 768, False, "persistent 256"),
    (12608, 768, 3072, False, "persistent 192"),
])
def test_ring_or_persistent(rules, m, n, k, gelu, expected):
    assert bf16(rules, m, n, k, gelu) == expected


@pytest.mark.parametrize("m,n,k,count,expected", [
    (6504, 240, 3072, 1, "64x64 deep"),
    (4888, 232, 1536, 1, "64x64 deep"),
    (1283, 1256, 768, 1, "128x64"),
])
def test_gelu_of_one_round(rules, m, n, k, count, expected):
    """128 x 64 tiles alone on their CUs: 30.8 us against 21.9 of the first; the
    last one's K has no use for three stages."""
    assert bf16(rules, m, n, k, True, count) == expected


@pytest.mark.parametrize("case", CASES, ids=str)
def test_each_ring_case_reaches_its_tile(rules, case):
    m, n, k, _, gelu, _, _, pad, tile = case
    fits = n % 256 == 0 and k >= 256 and (n + pad) % 8 == 0
    assert bf16(rules, m, n, k, gelu, persistent_fits=fits) == tile


RING_F32 = ["32x16 alone", "32x32", "32x32 deep", "64x32", "64x64", "tiled"]


@pytest.mark.parametrize("m,n,k,count,expected", [
    (197, 192, 768, 1, "32x16 alone"),
    # Operands from HBM: three stages (90 us on 64 x 32 tiles, 66 on these).
    (9182, 96, 3072, 1, "32x32 deep"),
    (3152, 384, 384, 1, "32x32 deep"),
    # More tiles a CU than three stages leave workgroups for.
    (1576, 2304, 768, 1, "32x32"),
    (12608, 320, 384, 1, "32x32"),
    # A long K and many tiles, and a short K: the cheapest tile.
    (10602, 744, 3072, 1, "64x64"),
    (11603, 248, 128, 1, "64x64"),
    # More work than that in one piece.
    (12507, 1928, 512, 1, "tiled"),
    (577, 608, 192, 27, "tiled"),
    # Batches whose entries go to the XCDs whole.
    (196, 200, 384, 192, "32x32"),
    (54, 24, 768, 136, "32x32 deep"),
    (577, 577, 64, 24, "64x32"),
])
def test_fp32_ring(rules, m, n, k, count, expected):
    assert RING_F32[rules.f32_choice(m, n, k, count, UNITS, 0)] == expected


@pytest.mark.parametrize("rows,expected", [(196, "64x32"), (256, "tiled")])
def test_fp32_entries_run_as_one_problem(rules, rows, expected):
    """64 images' patches of 14 x 14 pixels: 126 us on the ring and 151 tiled, 149 and 136."""
    assert RING_F32[rules.f32_choice(64 * rows, 768, 588, 1, UNITS, rows)] == expected


@pytest.mark.parametrize("case", F32_CASES, ids=str)
def test_each_fp32_ring_case_reaches_its_tile(rules, case):
    assert RING_F32[rules.f32_choice(*case[:3], 1, UNITS, 0)] == case[-1]


@pytest.mark.parametrize("count,whole", [(1, False), (3, False), (8, True), (9, False), (12, False), (24, True),
                                         (27, False), (72, True), (73, True), (75, True), (192, True),
                                         (65537, True)])
def test_entries_go_to_the_xcds_whole_where_they_divide_evenly(rules, count, whole):
    assert rules.whole_entries(count, 64) == int(whole)
    assert rules.whole_entries(count, 16384) == 0  # past a grid


@pytest.mark.parametrize("count,launches", [(1, 1), (65528, 1), (65529, 2), (2 ** 31 - 65529, 32772),
                                            (2 ** 31 - 65528, 32772), (2 ** 31 - 1, 32773)])
def test_large_batches_end(rules, count, launches):
    """Also where the last first entry plus a grid's extent is past an int."""
    assert rules.batch_launches(count) == launches
