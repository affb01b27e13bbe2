"""Host-side routing of the GEMM entry point at the engine's shapes (lcc_debug_gemm_plan: no launch, no GPU): which kernel family serves a
call and how many split-K slabs the engine's prefill asks for.  Pins the round-5 table of DESIGN section 4 so that a change of a tile
score, of a predicate or of the split rule shows up here before it shows up as a slower bench line."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
H, I, QKV = 3584, 18944, 4608


@pytest.fixture(scope="module")
def ops(built_lib):          # conftest: builds the git-ignored library when this file runs alone / on a fresh checkout
    from livecc_amd import ops as o
    return o


def test_eight_chunks_take_the_big_tiles(ops):
    assert ops.gemm_plan(3088, 2 * I, H, ops.EPI_SWIGLU)[0] == 272          # variable-height tiles: 12 x 148 blocks instead of 13 x 148
    assert ops.gemm_plan(3088, H, I, ops.EPI_RESIDUAL)[0] == 192            # 17 x 14 = 238 blocks fill one round
    assert ops.gemm_plan(3088, H, H, ops.EPI_RESIDUAL)[0] == 192
    assert ops.gemm_plan(3088, QKV, H, ops.EPI_NONE)[0] == 256
    assert ops.gemm_plan(9048, 2 * I, H, ops.EPI_SWIGLU)[0] in (256, 272)
    assert ops.gemm_plan(24058, 2 * I, H, ops.EPI_SWIGLU)[0] == 256         # 1504 fragments = 94 x 16: the 256-row tiles are the same thing


def test_one_chunk_takes_the_tall_kernel_and_the_small_variable_height_slabs(ops):
    assert ops.gemm_plan(386, 2 * I, H, ops.EPI_SWIGLU) == (448, 1)         # gate/up: one block row, 237 blocks
    for n, k, want in ((H, H, 6), (H, I, 6), (QKV, H, 4)):                  # o, down, q|k|v: 3 row tiles x 14 / 14 / 18 column tiles
        tile, splits = ops.gemm_plan(386, n, k, ops.EPI_NONE)
        assert splits == want, (n, k, splits)
        assert ops.gemm_plan(386, n, k, ops.EPI_NONE, nsplit=splits)[0] == 144
    assert ops.gemm_plan(386, H, I, ops.EPI_NONE, nsplit=4)[0] == 128       # with four slabs the 128-row tiles keep the call (224 blocks beat 168)
    assert ops.gemm_plan(386, H, I, ops.EPI_NONE, w_fp8=True) == (0, 4)     # fp8 weights: the round-4 split counts


def test_decode_batches_stream_the_weights(ops):
    for m in (1, 8, 16, 32, 64):
        assert ops.gemm_plan(m, 2 * I, H, ops.EPI_SWIGLU)[0] == 16
    assert ops.gemm_plan(65, 2 * I, H, ops.EPI_SWIGLU)[0] != 16


def test_other_row_counts_keep_their_round_4_routes(ops):
    assert ops.gemm_plan(1131, 2 * I, H, ops.EPI_SWIGLU)[0] == 256          # the first turn: 5 row tiles, the last half skipped
    assert ops.gemm_plan(122, H, I, ops.EPI_NONE)[1] >= 1                   # 8 fragments: no small class (a multiple of 8), any split count is legal
    assert ops.gemm_plan(122, H, I, ops.EPI_NONE, nsplit=4)[0] != 144
    assert ops.gemm_plan(1456, 1280, 5120, ops.EPI_RESIDUAL)[0] == 64       # one-stream vision fc2: the 4-wave 64 x 128 tiles (230 blocks)
    assert ops.gemm_plan(11648, 5120, 1280, ops.EPI_QUICK_GELU)[0] in (256, 272)


def test_the_switch_restores_the_128_row_slabs(built_lib):
    code = ("import sys; sys.path.insert(0, %r)\nfrom livecc_amd import ops\n"
            "s = ops.gemm_plan(386, 3584, 18944, ops.EPI_NONE)[1]\nprint(s, ops.gemm_plan(386, 3584, 18944, ops.EPI_NONE, nsplit=s)[0])" % ROOT)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env=dict(os.environ, LCC_GEMM_VH_SMALL="0"), timeout=120)
    assert r.returncode == 0, r.stderr[-400:]
    assert r.stdout.strip() == "4 128", r.stdout      # four slabs on the 128-row tiles: the round-4 form


def test_several_weight_tiles_a_block_where_they_save_more_than_they_cost(ops):
    """10 to 16 rows: products whose blocks pull much take what 17 rows take, short ones (measured up to 18 % slower so) one tile, as up to nine rows do."""
    slabs = lambda N, K: ops.gemv_num_splits(N, K)      # noqa: E731
    for M in (10, 12, 16):
        for N, K in ((3584, 18944), (8192, 29568), (3584, 22528)):
            assert ops.gemv_plan(M, N, K, nsplit=slabs(N, K)) > 1, (M, N, K)
        for N, K in ((2304, 1536), (2560, 2560), (1408, 3072), (1024, 4096), (2816, 1536)):
            assert ops.gemv_plan(M, N, K, nsplit=slabs(N, K)) == 1, (M, N, K)
        for N, K in ((152064, 3584), (151936, 1536), (32000, 4096)):
            assert ops.gemv_plan(M, N, K) > 1, (M, N, K)
        assert ops.gemv_plan(M, 3584, 3584) == 1
        assert ops.gemv_plan(M, 17920, 1536, ops.EPI_SWIGLU) == 6
    assert ops.gemv_plan(14, 4096, 4096, nsplit=4) == ops.gemv_plan(10, 5120, 5120, nsplit=4) == ops.gemv_plan(10, H, H, nsplit=4) == 1 and ops.gemv_plan(10, QKV, H, nsplit=4) == 1 and ops.gemv_plan(16, QKV, H, nsplit=4) == 1
    for N, K in ((3584, 18944), (2304, 1536)):
        assert ops.gemv_plan(9, N, K, nsplit=slabs(N, K)) == 1 and ops.gemv_plan(17, N, K, nsplit=slabs(N, K)) > 1
    assert ops.gemv_plan(16, 3584, 18944 + 32) == 1 and ops.gemv_plan(17, 3584, 18944 + 32) == 0 and ops.gemv_plan(65, 3584, 18944) == 0


@pytest.mark.parametrize("M", [1, 8, 9, 13, 16, 17, 40, 64, 65])
def test_input_and_gate_up_projections_in_one_launch_take_whole_64_k_chunks(built_lib, M):
    """9 to 64 rows (lcc_debug_gemv_pair_plan).  The kernel reads whole 64-k chunks of the activations: at K = 64 n + 32 the last one would run into the next row
    (behind the last one past the buffer) and meet the last 32 weights twice."""
    from livecc_amd import ops
    for K in (64, 192, 1536, 3584):
        assert ops.gemv_pair_plan(M, 1296, 2 * 1024, K, 1) == (9 <= M <= 64)
        assert not ops.gemv_pair_plan(M, 1296, 2 * 1024, K + 32, 1)
        assert not ops.gemv_pair_plan(M, 1296, 2 * 1024, K + 16, 1)


def test_prefill_attention_plan_at_the_engines_shapes(built_lib):
    """Tile height x key-split count of the LLM prefill attention (lcc_debug_attn_plan: the function lcc_llm_prefill itself calls, no launch):
    one block per CU and (tile, KV head, split), relative time = rounds of blocks x keys per block; measured in
    profiles/r06/attn_tall_tiles_ab.jsonl and attn_tall_tiles_splits_probe.jsonl."""
    from livecc_amd import _lib, ops
    assert ops.attn_tile_rows(28, 4) == 36 and ops.attn_tile_rows(64, 8) == 32 and ops.attn_tile_rows(12, 2) == 42 and ops.attn_tile_rows(16, 1) == 32
    plan = lambda n_new, kv, hq=28, hkv=4, cus=256: ops.attn_plan(n_new, kv, hq, hkv, cus)      # noqa: E731
    assert plan([386], 6586) == (36, 5)              # one streaming chunk: 11 tiles x 4 KV heads x 5 splits = 220 blocks, one round (65 us; (32, 4): 73)
    assert plan([386] * 2, 6586) == (32, 2)          # 208 blocks, one round: 113.7 us ((36, 8) 126, (32, 7) 129: what "fill the last round" chose)
    assert plan([386] * 3, 6586) == (32, 1)          # 1,158 rows: no split above 1,024 rows (the partial buffers); 156 / 132 blocks: one round, a tie
    assert plan([386] * 4, 6586) == (32, 1)          # 208 blocks unsplit, a tie with the tall tile
    assert plan([386] * 5, 6586) == (36, 1)          # 260 blocks = two rounds, 220 tall ones = one
    assert plan([300] * 3, 6586) == (32, 2)          # 900 rows may split: 30 tiles x 4 x 2 = 240 blocks of half the keys, one round
    assert plan([386] * 8, 6586) == (32, 1)          # 416 / 352 blocks: two rounds either way
    assert plan([1131] * 8, 1131) == (36, 1)         # 1152 -> 1024 blocks: five rounds -> four
    assert plan([4096], 12288) == (32, 1)            # a one-shot piece: 512 / 456 blocks, two rounds either way
    assert plan([386], 200) == (32, 1)               # too few keys to split (>= 8 key tiles per split): 52 / 44 blocks, one round: a tie
    assert plan([386], 26000) == (36, 5)             # a long history changes nothing for one chunk
    assert plan([386], 6586, 64, 8) == (32, 2)       # 72B heads (G = 8): the tall tile does not exist; 13 x 8 x 2 = 208 blocks
    assert plan([386], 6586, 32, 2) == (0, 0)        # 16 query heads per KV head: another kernel family
    with pytest.raises(_lib.LccError):
        plan([386, 0], 6586)
    with pytest.raises(_lib.LccError):
        plan([386], 6586, 28, 5)


def test_short_products_of_129_to_192_rows_take_the_64_row_tiles(ops):
    """One round of 128 x 256 tiles whose last row tile is at most half full, with few k-steps a block: two 64-row tiles a compute unit."""
    assert [ops.gemm_plan(M, 17920, 1536, e)[0] for M in (129, 160, 192) for e in (ops.EPI_NONE, ops.EPI_SWIGLU)] == [64] * 6
    assert [ops.gemm_plan(M, 17920, 1536, ops.EPI_SWIGLU)[0] for M in (193, 256)] == [128, 128]
    assert [ops.gemm_plan(M, QKV, H, 0, 4)[0] for M in (150, 192)] == [64, 64]
    assert ops.gemm_plan(137, H, I, 0, 6)[0] == 128


def test_decode_attention_splits_over_streams(built_lib):
    """Key splits of the decode attention, as lcc_llm_decode asks for them: one stream as many as its tiles give (one tile up to 24 of them, two
    beyond, up to 64 splits, 128 from 16k keys on, none without a tile); batches of one length stop at 768 blocks, two splits at least, so that 64 streams do
    not write and merge the partials of 64 splits each; a long cache beside short ones keeps more, so that the launch does not wait for its chain of tiles."""
    import numpy as np

    def f(keys, heads=4):
        a = np.asarray(keys, dtype=np.int32)
        return built_lib.lcc_debug_attn_decode_splits(a.ctypes.data, len(a), heads)

    assert [f([k]) for k in (1, 32, 33, 500, 768, 769, 2000, 6500, 16384, 16385, 24000)] == [1, 1, 2, 16, 24, 13, 32, 51, 64, 103, 125]
    assert [f([4000] * n) for n in (1, 2, 3, 4, 8, 12, 16, 17, 32, 48, 64)] == [63, 63, 63, 42, 21, 16, 12, 11, 6, 4, 3]
    assert f([6000] * 64, 8) == 2 and f([40] * 64, 8) == 2 and f([20] * 64, 8) == 1
    for heads in (2, 4, 8):
        for streams in range(1, 65):
            for k in (1, 100, 700, 3000, 9000, 30000):
                n, tiles = f([k] * streams, heads), (k + 31) // 32
                assert 1 <= n <= 128 and (n <= 2 or n * streams * heads <= 768) and (n - 1) * -(-tiles // n) < tiles          # no split without a tile
    # one long cache: its chain is a few tiles a split, whatever its place; more short ones beside it make a split dearer, never fewer splits than one length has
    for streams, most in ((8, 12), (16, 16), (64, 32)):
        mixed = [f(([500] * i + [20000] + [500] * (streams - 1 - i))) for i in (0, streams // 2, streams - 1)]
        assert len(set(mixed)) == 1 and f([20000] * streams) <= mixed[0] <= 128 and -(-625 // mixed[0]) <= most
    assert f([6000] * 7 + [5000]) == f([6000] * 8) < f([6000, 6000] + [1000] * 6)
    assert f([]) < 0 and f([0]) < 0 and f([5, 0]) < 0 and f([5], 0) < 0 and built_lib.lcc_debug_attn_decode_splits(None, 1, 4) < 0


@pytest.mark.parametrize("preset,fp8,last", [("livecc-7b", 0, 16), ("livecc-7b", 1, 16), ("qwen2vl-2b", 0, 8), ("qwen2vl-2b", 1, 8), ("qwen2vl-72b", 0, 4), ("qwen2vl-72b", 1, 9)])
def test_decode_batches_that_take_the_row_scaled_products(built_lib, preset, fp8, last):
    """From three streams on while a layer's weight bytes x rows are below 8e9, 16 streams at most (8 at 2,048 channels and below)."""
    import ctypes
    from livecc_amd import _lib
    from livecc_amd.config import PRESETS
    c = PRESETS[preset]()
    cfg = _lib.ModelConfig(c.vocab_size, c.hidden_size, c.intermediate_size, c.num_hidden_layers, c.num_attention_heads, c.num_key_value_heads, 128, 1e-6, 16, 24, 24,
                           c.vit_depth, c.vit_embed_dim, c.vit_num_heads, c.vit_mlp_dim, 1176, 2)
    cfg.llm_fp8 = fp8
    lim = _lib.EngineLimits(64, 1024, 256, 1024, 16)
    e = built_lib.lcc_engine_create(ctypes.byref(cfg), ctypes.byref(lim))
    try:
        assert [n for n in range(1, 65) if built_lib.lcc_debug_decode_row_scaled(e, n)] == list(range(3, last + 1))
        assert built_lib.lcc_debug_decode_row_scaled(e, 0) < 0 and built_lib.lcc_debug_decode_row_scaled(None, 3) < 0
    finally:
        built_lib.lcc_engine_destroy(e)


def test_long_contractions_of_a_few_hundred_to_a_few_thousand_rows_are_split(built_lib):
    """Between one chunk's rows and a piece of 4,096: two to six splits where a tenth is saved, never more than the slab buffer holds (six), each split
    of several k-tiles; one where the tiles fill the chip, on a short K, for fp8 weights."""
    from livecc_amd import ops
    plan = lambda M, N, K, **kw: ops.gemm_plan(M, N, K, ops.EPI_NONE, **kw)[1]
    assert all(2 <= plan(M, N, K) <= 6 for M, N, K in ((449, 3584, 18944), (600, 3584, 18944), (1000, 3584, 22528), (1131, 3584, 18944), (1000, 1536, 8960), (2104, 1536, 10496)))
    assert plan(4096, 3584, 18944) == plan(3088, 3584, 18944) == plan(2000, 3584, 18944) == plan(5000, 3584, 18944) == 1
    assert plan(1000, 3584, 18944, w_fp8=True) == 1 and plan(1000, 3584, 6080) == 1
    for M in range(449, 4097, 37):
        for N, K in ((3584, 18944), (1536, 8960), (272, 6144)):
            assert 1 <= plan(M, N, K) <= 6


@pytest.mark.parametrize("M,N", [(90, 256), (100, 1024), (386, 3584), (600, 4608)])
def test_narrow_fp8_products_refuse_a_result_they_cannot_store_aligned(built_lib, M, N):
    """Shapes of the 64 x 128 and 128 x 128 tiles: rows of C at an odd multiple of four bytes, or C itself at 8 bytes, are refused before anything is launched (host
    memory stands in for the device's)."""
    import ctypes as C
    from livecc_amd import _lib
    buf = C.create_string_buffer(4096)
    p = (C.addressof(buf) + 15) // 16 * 16
    call = lambda c, ldc: built_lib.lcc_gemm_w8_bf16(p, 256, p, C.cast(p, C.POINTER(C.c_float)), None, None, 0, c, ldc, M, N, 256, 0, None, 0, p, None)
    assert call(p, N + 2) == call(p, N + 1) == -2 and call(p + 8, N) == -3


@pytest.mark.parametrize("m,n,k,splits", [(1000, 3584, 22528, 3), (1000, 3584, 18944, 3), (500, 3584, 18944, 6), (1200, 3584, 22528, 5), (2500, 3584, 22528, 2),
                                          (514, 4608, 6144, 4), (1227, 1280, 6144, 5), (496, 37888, 22528, 1), (1000, 1536, 8960, 5), (2104, 1536, 10496, 3)])
def test_split_counts_of_long_contractions_do_not_follow_the_tiles_weights(ops, m, n, k, splits):
    """The count decides into how many fp32 sums a contraction is cut, and so a result's bits; which tile runs a product does not."""
    assert ops.gemm_plan(m, n, k, ops.EPI_NONE)[1] == splits


@pytest.mark.parametrize("m", [65, 128, 129, 192, 193, 256, 257, 320, 385, 448])
@pytest.mark.parametrize("n", [32800, 37888, 40960])
def test_the_tall_tile_of_few_rows_is_swiglu_alone(ops, m, n):
    """Its heights of 2 to 4 fragments a quarter exist for that epilogue; another product of up to 256 rows would multiply 448."""
    for epi in (ops.EPI_NONE, ops.EPI_QUICK_GELU, ops.EPI_GELU_ERF, ops.EPI_RESIDUAL):
        assert (ops.gemm_plan(m, n, H, epi)[0] == 448) == (m > 256), epi
    assert ops.gemm_plan(m, n, H, ops.EPI_SWIGLU)[0] == 448
