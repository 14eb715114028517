"""Which prompt GEMM kernel a launch takes (host arithmetic, 256 CUs; without a
device the library assumes those of an MI355X). CPU only."""
import pytest

from helpers import PAIR, RESIDUAL, STORE, qmm_route

QKV, GDN, WIDE = [8192, 1024, 1024], [8192, 4096, 32, 32], [12288, 12288]


@pytest.fixture(autouse=True)
def _no_override(monkeypatch):
    monkeypatch.delenv("PEREGRINE_GEMM_DMA", raising=False)


# rows: forms of q / k / v, the Gated DeltaNet input projections, the output projections, gate / up and
# down of the 9B widths with prepared copies
@pytest.mark.parametrize("rows,routes", [
    (1, (41, 41, 11, 81, 11)), (16, (41, 41, 11, 81, 11)), (64, (41, 41, 11, 81, 11)),
    (65, (42, 42, 21, 82, 21)), (128, (42, 42, 21, 82, 21)), (129, (41, 192, 41, 192, 41)),
    (300, (192, 192, 42, 192, 42)), (1600, (1320, 1320, 256, 1320, 256)), (2048, (256, 1256, 256, 1256, 256)),
])
def test_model_widths(rows, routes):
    got = (qmm_route(STORE, rows, QKV, 4096, True), qmm_route(STORE, rows, GDN, 4096, True),
           qmm_route(STORE, rows, [4096], 4096, True), qmm_route(PAIR, rows, WIDE, 4096, True),
           qmm_route(RESIDUAL, rows, [4096], 12288, True))
    assert got == routes


# where the column tiles leave the 32- and 64-row forms a nearly empty round; the two-round launch of
# 16 x 128 rows costs more than one of 64 x 128
@pytest.mark.parametrize("epilogue,rows,outs,route", [
    (STORE, 384, 1360, 12), (STORE, 640, 816, 12), (STORE, 322, 2720, 22), (STORE, 640, 1632, 22),
    (STORE, 889, 1168, 42), (RESIDUAL, 889, 1168, 42), (PAIR, 322, 2720, 41), (PAIR, 384, 2720, 41),
])
def test_ragged_rounds(epilogue, rows, outs, route):
    assert qmm_route(epilogue, rows, [outs] * (2 if epilogue == PAIR else 1), 4096) == route


def test_k_steps_and_refused_sizes():
    assert qmm_route(STORE, 43, [4096], 320) == 192  # the few-row kernel takes k in steps of 256
    assert qmm_route(STORE, 0, [4096], 4096) == 0
    assert qmm_route(STORE, 43, [4096, 0], 4096) == 0
    assert qmm_route(STORE, 43, [16] * 5, 4096) == 0
    assert qmm_route(3, 43, [4096], 4096) == 0


@pytest.mark.parametrize("force,prepared,want", [("0", True, 192), ("0", False, 192), ("256", True, 1256),
                                                 ("320", True, 1320), ("320", False, 192), ("", True, 81)])
def test_override(monkeypatch, force, prepared, want):
    monkeypatch.setenv("PEREGRINE_GEMM_DMA", force)
    assert qmm_route(PAIR, 43, WIDE, 4096, prepared) == want
