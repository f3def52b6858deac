"""The launcher's choice of tile shape for large half-precision products (host logic, no GPU): held to the measured
time of every shape on 92 problem sizes (tests/golden/gemm_variant_timings.txt, written on an MI355X by
tests/golden/make_gemm_variant_timings.py)."""
import os

import numpy as np

from lc0_amd import kernels as K

COLUMN = {"gemm_dma_256x256x64": 0, "gemm_dma_256x192x64": 1, "gemm_dma_256x128x32": 2, "gemm_dma_128x128x64": 3,
          "gemm_dma_128x64x64": 4}


def _table():
    path = os.path.join(os.path.dirname(__file__), "golden", "gemm_variant_timings.txt")
    rows = [line.split() for line in open(path) if line.strip() and not line.startswith("#")]
    return [(int(r[0]), int(r[1]), int(r[2]), [float(t) for t in r[3:8]]) for r in rows]


def _time_of_choice(m, n, k, table):
    """Measured time of what the launcher does for this problem; None for a product cut along its rows into parts
    the table does not hold."""
    name = K.gemm_variant_name(m, n, k)
    if not name.endswith("+rest"):
        return table[(m, n, k)][COLUMN[name]]
    m1 = K.gemm_row_split(m, n, k)
    assert 0 < m1 < m and m1 % 256 == 0, (m, n, k, m1)
    if (m1, n, k) not in table or (m - m1, n, k) not in table:
        return None
    return table[(m1, n, k)][COLUMN[name[:-5]]] + _time_of_choice(m - m1, n, k, table)


def test_chosen_tile_shape_is_close_to_the_fastest_measured_one():
    table = {(m, n, k): times for m, n, k, times in _table()}
    regrets, cut = [], 0
    for (m, n, k), times in table.items():
        t = _time_of_choice(m, n, k, table)
        cut += K.gemm_row_split(m, n, k) > 0
        if t is not None:
            regrets.append(t / min(times) - 1.0)   # (below zero where two launches beat every single shape)
    print("%d of %d problems are cut along their rows" % (cut, len(table)))
    regrets = np.array(regrets)
    print("mean %.4f max %.4f over %d problems" % (regrets.mean(), regrets.max(), len(regrets)))
    assert len(regrets) >= 85
    assert regrets.mean() <= 0.012
    assert regrets.max() <= 0.10


def test_choices_for_the_encoder_layers_at_batch_256():
    """The four projections of a 15x1024 layer at 256 positions: whole rounds of 256 tiles on the 256 CUs."""
    assert K.gemm_variant_name(16384, 3072, 1024) == "gemm_dma_256x256x64"   # 768 tiles
    assert K.gemm_variant_name(16384, 1024, 1024) == "gemm_dma_256x256x64"   # 256 tiles
    assert K.gemm_variant_name(16384, 1536, 1024) == "gemm_dma_256x192x64"   # 512 tiles
    assert K.gemm_variant_name(16384, 1024, 1536) == "gemm_dma_256x256x64"


def test_products_that_leave_a_partial_round_are_cut_along_their_rows():
    """Whole rounds of large tiles first, the rest on whatever suits it; products that fill their rounds stay whole."""
    assert K.gemm_row_split(20480, 1024, 1536) == 16384
    assert K.gemm_variant_name(20480, 1024, 1536) == "gemm_dma_256x256x64+rest"
    assert K.gemm_row_split(24576, 1024, 1024) == 16384
    for m, n, k in ((16384, 3072, 1024), (16384, 1024, 1024), (16384, 1536, 1024), (32768, 1024, 1536), (4096, 1024, 1024),
                    (65536, 3072, 1024)):
        assert K.gemm_row_split(m, n, k) == 0, (m, n, k)
    assert K.gemm_row_split(20480, 64, 1024) == 0 and K.gemm_row_split(1 << 20, 1024, 256) == 0   # outside the model


def test_the_rest_of_a_cut_product_runs_on_the_shape_it_is_priced_with():
    """4416 rows of 2048 columns would get 128x128 tiles as a product of their own (55 us; 256x192 tiles, by which the cut is priced, 46.5):
    with them the pair is slower than one launch. A shape priced as high as the cheapest stays."""
    assert K.gemm_variant_name(4416, 2048, 2048) == "gemm_dma_128x128x64"
    for m, n, k, m1, rest in ((12608, 2048, 2048, 8192, "256x192"), (12416, 1984, 1856, 8192, "256x192"), (11648, 2176, 1792, 7168, "256x192"),
                              (14848, 1088, 1728, 10752, "128x128"), (13312, 1792, 1024, 9216, "128x128")):
        assert K.gemm_row_split(m, n, k) == m1
        assert K.gemm_rest_variant_name(m, n, k) == "gemm_dma_%sx64" % rest, (m, n, k)
    assert K.gemm_rest_variant_name(20480, 1024, 1536) == K.gemm_variant_name(4096, 1024, 1536)   # (the model of 16384 rows and more)
    assert K.gemm_rest_variant_name(16384, 1024, 1024) == ""


def test_small_and_batched_products_keep_their_kernels():
    assert K.gemm_variant_name(1, 3072, 1024) == "gemm_rowpanel"
    assert K.gemm_variant_name(64, 64, 1024, batch=256) == "gemm_64x64x64"    # policy logits, one product per position
    assert K.gemm_variant_name(16384, 32, 1024) == "gemm_64x64x64"            # smolgen compression beside the projection
    assert K.gemm_variant_name(16384, 32, 1024, latency_first=True) == "gemm_rowpanel"


def test_few_rows_with_many_columns_or_products():
    """33 to 128 rows (smolgen's second dense layer, the policy logits): direct-to-LDS tiles or panels, not the tiles that walk
    the whole reduction in one workgroup per 64x64 outputs."""
    for latency_first in (False, True):
        for m in (33, 48, 63, 64):
            assert K.gemm_variant_name(m, 8192, 256, latency_first=latency_first) == "gemm_dma_64x64x64"
            assert K.gemm_variant_name(m, 8192, 264, latency_first=latency_first) == "gemm_rowpanel"
        assert K.gemm_variant_name(128, 3072, 256, latency_first=latency_first) == "gemm_dma_64x64x64"
    for batch in (65, 77, 128):
        assert K.gemm_variant_name(64, 64, 1024, batch=batch) == "gemm_dma_64x64x64"
    assert K.gemm_variant_name(64, 64, 1024, batch=129) == "gemm_64x64x64"
    assert K.gemm_variant_name(32, 8192, 256) == "gemm_rowpanel"
    # few products with a short reduction: panels as long as one workgroup per CU covers them
    assert K.gemm_variant_name(64, 64, 256, batch=16) == "gemm_rowpanel"
    assert K.gemm_variant_name(4, 256, 256, batch=20) == "gemm_rowpanel"
    assert K.gemm_variant_name(64, 64, 256, batch=77) == "gemm_dma_64x64x64"


def test_the_smolgen_chain_leaves_the_projection_where_that_has_more_than_one_round_of_tiles():
    """256x256 tiles over the 64 rows of every position and the 3 d_model columns of the projection, whatever the width of the body; in
    e4m3 that of the narrower of the two."""
    for emb in (384, 512, 1024):
        for d_model in (384, 512, 768, 1024, 1088):
            batch = K.smolgen_overlap_min_batch(emb, d_model)
            tiles = 64 * batch / 256 * 3 * d_model / 256
            assert batch == 80 or 255 <= tiles <= 258, (emb, d_model, batch)
    assert [K.smolgen_overlap_min_batch(d, d) for d in (384, 512, 768, 1024, 1536)] == [227, 170, 114, 85, 80]
    assert [K.smolgen_overlap_min_batch(e, d, f8=True) for e, d in ((512, 1024), (1024, 512), (1024, 1024))] == [170, 170, 85]
    assert K.smolgen_overlap_min_batch(512, 512, f32=True) == 80
    for emb, d_model in ((0, 0), (1024, 0), (0, 1024), (-1, 512)):
        assert K.smolgen_overlap_min_batch(emb, d_model, f8=True) == 0


def test_e4m3_products_of_few_rows_with_large_weights():
    """More than one 64x64 tile per CU and weights beyond an XCD's 4 MiB of L2: 128x64 tiles; otherwise 64x64."""
    for m, n, k in ((512, 3072, 1536), (256, 8192, 2048), (300, 8192, 1024), (640, 3072, 2048)):
        assert K.gemm_f8_variant_name(m, n, k) == "gemm_f8_128x64x128", (m, n, k)
    for m, n, k in ((256, 3072, 2048), (256, 8192, 512), (832, 1536, 1024), (832, 3072, 1024), (1024, 3072, 1536)):
        assert K.gemm_f8_variant_name(m, n, k) == "gemm_f8_64x64x128", (m, n, k)
    assert K.gemm_f8_variant_name(64, 1024, 1024) == "gemm_f8_rowpanel"
