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
