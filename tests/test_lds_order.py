"""Lanes of a wave that exchange values through LDS without a block barrier: the compiler sees one lane's accesses only, so the source has to order
one lane's stores against another lane's loads.  Read from the source, on the CPU: a violation shows on a GPU only if a compiler uses its freedom."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "livecc_amd", "csrc")


def body(src, name):
    at = re.search(r"LCC_DEVICE void " + name + r"\(", src).start()
    i = src.index("{\n", at)
    depth, j = 0, i
    while True:
        depth += {"{": 1, "}": -1}.get(src[j], 0)
        j += 1
        if depth == 0:
            return re.sub(r"//.*", "", src[i:j])


@pytest.mark.parametrize("name,store,load", [
    ("tile_epilogue_wide", r"st8\(lds ", r"ld16\(lds "),
    ("tile_slab_wide", r"reinterpret_cast<f32x4\*>\(lds ", r"reinterpret_cast<const f32x4\*>\(lds ")])
def test_rows_through_lds_are_ordered_between_lanes(name, store, load):
    """Per group of rows: order (the last group's loads are done), stores, order, loads."""
    text = body(open(os.path.join(CSRC, "gemm.hip")).read(), name)
    seen = sorted([(m.start(), "O") for m in re.finditer(r"wave_lds_order\(\)", text)] + [(m.start(), "S") for m in re.finditer(store, text)] +
                  [(m.start(), "L") for m in re.finditer(load, text)])
    assert "".join(k for _, k in seen) == "OSOL"


def test_the_order_is_a_fence_on_both_sides_of_the_exchange():
    text = body(open(os.path.join(CSRC, "common.h")).read(), "wave_lds_order")
    assert re.search(r'fence\(__ATOMIC_ACQ_REL, "wavefront"\)', text) and "wave_barrier" in text


def test_no_requested_residual_piece_is_left_unused():
    """A row group that is skipped leaves its residual pieces in flight; the compiler then waits for all memory in every k-step of the next tile."""
    text = body(open(os.path.join(CSRC, "gemm.hip")).read(), "tile_epilogue_wide")
    skips = re.findall(r"if \((.*?>= M)\) break;", text)
    assert skips and all(s.startswith("EPI != EPI_RESIDUAL && ") for s in skips)


def test_a_stage_row_of_the_walking_tiles_belongs_to_one_phase_whatever_the_height():
    """A block that goes from a tile of 17 row fragments to one of 18 copies the next tile's first phase into the stage whose second phase is being read: no row
    of the stage may be in the first phase of one height and in the second of another."""
    text = body(open(os.path.join(CSRC, "gemm.hip")).read(), "gemm_walk_body")
    struct = re.search(r"struct Walk \{(.*?)\n\};", open(os.path.join(CSRC, "gemm.hip")).read(), re.S).group(1)
    places = re.search(r"const int row = p < n_first \? from \+ p \* 8 : p < n_first \+ n_second \? (\S+) \+ from \+ \(p - n_first\) \* 8 : -1;", text)
    assert "dst = row >= 0 ? (unsigned)row * 128u" in text
    reads = re.search(r"aoff\[kk\] = \(\(wm \? (\S+) : 0\) \+ li\) \* 8", text)
    assert places and reads and places.group(1) == reads.group(1)
    at = {"row1": lambda f: (f >> 1) * 16, "S::ROW1": lambda f: {"16 * MTX": 16 * 9}[re.search(r"ROW1 = VH \? (.*?) : BM / 2;", struct).group(1)]}[places.group(1)]
    of_phase = ([set(), set()])
    for f in (16, 17, 18):
        first, second = f >> 1, f - (f >> 1)          # row fragments of the two wave rows, four of each in the first phase
        for start, n in ((0, first), (at(f), second)):
            for i in range(n):
                of_phase[i >= 4] |= set(range(start + 16 * i, start + 16 * i + 16))
    assert not of_phase[0] & of_phase[1]
    assert max(of_phase[1]) < 288
