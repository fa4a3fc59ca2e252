"""Rules on pass geometry (ffsim_amd/csrc/pass_rules.hpp), evaluated on the CPU."""

import ctypes
import subprocess
from math import comb
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
C128, C64 = 0, 1


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    out = tmp_path_factory.mktemp("rules") / "pass_rules.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC",
                    str(ROOT / "tests/native/pass_rules_check.cpp"),
                    str(ROOT / "ffsim_amd/csrc/host_core.cpp"), "-o", str(out)], check=True)
    return ctypes.CDLL(str(out))


NONE, AS_ROWS, SLABS, COLUMNS = range(4)


@pytest.mark.parametrize("dtype", [C128, C64])
@pytest.mark.parametrize("norb,nelec,form", [
    (12, (6, 6), SLABS), (14, (7, 6), SLABS), (16, (8, 8), SLABS), (18, (9, 9), SLABS),
    (20, (5, 1), SLABS),
    # no electrons to reduce over: nothing is transposed
    (16, (8, 0), NONE), (24, (12, 0), NONE),
    # one row or one column is its own transpose
    (24, (12, 24), AS_ROWS), (24, (0, 12), AS_ROWS), (1, (1, 1), AS_ROWS),
    # few rows of very many columns
    (24, (1, 8), COLUMNS), (24, (1, 12), COLUMNS), (22, (2, 9), COLUMNS), (20, (2, 7), None),
])
def test_transition_rdm_layout(rules, dtype, norb, nelec, form):
    da, db = (comb(norb, n) for n in nelec)
    slab = ctypes.c_long()
    got = rules.trdm_layout(dtype, ctypes.c_long(da), ctypes.c_long(db), nelec[1],
                            ctypes.byref(slab))
    if form is not None:
        assert got == form
    if got == SLABS:
        elem = 16 if dtype == C128 else 8
        assert 1 <= slab.value <= da
        assert 2 * slab.value * db * elem <= 96 << 20
        # 64 lanes of a dot product have work, and the transposition's grid fits
        assert slab.value == da or slab.value >= 64
        assert (slab.value + 31) // 32 <= 65535


def _small(rules, dtype, norb, nocc, n_batch, n_states=1, on_columns=0):
    out = (ctypes.c_int * 4)()
    rules.small_pass(dtype, norb, nocc, ctypes.c_long(n_batch), n_states, on_columns, out)
    return out


@pytest.mark.parametrize("dtype", [C128, C64])
@pytest.mark.parametrize("norb", range(6, 13))
def test_every_sector_up_to_norb_12_runs_in_place(rules, dtype, norb):
    """Whatever the other sector: empty and full ones leave a single column."""
    for nocc in range(norb + 1):
        for other in range(norb + 1):
            n_batch = comb(norb, other)
            for on_columns in (0, 1):
                units, cols, sweeps, _ = _small(rules, dtype, norb, nocc, n_batch, 2, on_columns)
                assert units and 256 // units * sweeps >= comb(norb, nocc)
                # with strings on rows a 16-byte unit must not reach past the columns
                assert cols or n_batch >= (1 if dtype == C128 else 2)


@pytest.mark.parametrize("dtype", [C128, C64])
@pytest.mark.parametrize("norb", range(6, 13))
@pytest.mark.parametrize("n_states", [1, 2, 3, 8, 32, 256])
def test_small_tiles_hold_their_sector(rules, dtype, norb, n_states):
    """A compiled geometry whose tile has a row for every string."""
    compiled = {(4, 15, 1), (8, 8, 1), (8, 15, 1), (8, 29, 1), (16, 16, 1), (16, 29, 1)}
    if dtype == C64:
        compiled |= {(8, 29, 2), (16, 29, 2)}
    for nocc in range(norb + 1):
        for other in range(norb + 1):
            units, _, sweeps, cols = _small(rules, dtype, norb, nocc, comb(norb, other), n_states)
            assert (units, sweeps, cols) in compiled
            assert 256 // units * sweeps >= comb(norb, nocc)


@pytest.mark.parametrize("dtype,nocc,n_states,units", [
    # one round of 64-byte rows; two states of complex128 are one round of 128-byte rows
    (C128, 6, 1, 4), (C128, 6, 2, 8), (C128, 5, 2, 8), (C128, 6, 32, 8),
    (C64, 6, 2, 4), (C64, 6, 3, 8), (C64, 6, 5, 4), (C64, 6, 8, 8), (C64, 4, 6, 8),
])
def test_small_tile_width_norb_12(rules, dtype, nocc, n_states, units):
    assert _small(rules, dtype, 12, nocc, comb(12, nocc), n_states)[0] == units


def _sector(rules, dtype, norb, nocc, other):
    """(window, units, whole sector in a tile, last pass pipelined)"""
    out = (ctypes.c_int * 3)()
    piped = rules.sector_pass(dtype, norb, nocc, ctypes.c_long(comb(norb, other)), out)
    return out[0], out[1], bool(out[2]), bool(piped)


@pytest.mark.parametrize("dtype", [C128, C64])
@pytest.mark.parametrize("norb", range(13, 19))
def test_single_string_sectors_run_plain(rules, dtype, norb):
    """Nothing to rotate: one plain pass, no tile of hundreds of rows for one."""
    for nocc in (0, norb):
        for other in range(norb + 1):
            w, _, whole, piped = _sector(rules, dtype, norb, nocc, other)
            assert w == 12 and not whole and not piped


@pytest.mark.parametrize("dtype", [C128, C64])
def test_sectors_of_norb_13_to_16_run_whole(rules, dtype):
    for norb, nocc in [(13, 6), (14, 7), (15, 7), (16, 5), (16, 1), (13, 12)]:
        assert _sector(rules, dtype, norb, nocc, nocc) == (norb, _sector(
            rules, dtype, norb, nocc, nocc)[1], True, True)
    assert _sector(rules, dtype, 16, 8, 8)[:3] == (12, 8, False)


@pytest.mark.parametrize("dtype", [C128, C64])
@pytest.mark.parametrize("norb,nocc,other", [(17, 2, 3), (17, 3, 2), (18, 3, 3), (16, 8, 1),
                                             (18, 0, 3), (18, 3, 0), (18, 3, 18), (18, 18, 3)])
def test_passes_that_run_plain(rules, dtype, norb, nocc, other):
    """The shapes that tests/test_gpu_plain_passes.py takes for plain ones."""
    assert not _sector(rules, dtype, norb, nocc, other)[3]


@pytest.mark.parametrize("dtype", [C128, C64])
@pytest.mark.parametrize("norb,nocc,other", [(16, 8, 8), (18, 9, 9), (17, 8, 4), (14, 2, 7)])
def test_passes_that_run_pipelined(rules, dtype, norb, nocc, other):
    assert _sector(rules, dtype, norb, nocc, other)[3]
