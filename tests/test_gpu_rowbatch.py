"""The row-batch kernels at the row counts where their tiles, K splits and dispatch rules change: a
prompt prefilled at once against the same positions decoded one by one (other kernels, themselves
checked against the oracle), at the 270M block shape with a small vocabulary."""
import os

import numpy as np
import pytest

import synth
import vrt

pytestmark = pytest.mark.gpu

# Both paths hold activations to 22 bits or better and sum in fp32: 2^-22 per block and projection, a few
# times that after the two blocks' norms; a lost low half or a dropped tile shows as 1e-4 or more.
TOL = 5e-6
SHAPE = dict(n_layers=2, d_model=640, n_heads=4, head_dim=256, ffn=2048, vocab=1000, context=8800, window=512)
ROWS = (1, 2, 15, 16, 17, 33, 64, 65, 129, 255, 300, 513, 700, 1025, 1500, 2047, 2049, 4200, 8192, 8193, 8700)   # past 8192: a second segment, over the first one's cache


def _rel(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b.astype(np.float64)))


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    path = os.path.join(str(tmp_path_factory.mktemp("rowbatch")), "two_blocks.gguf")
    synth.write_gemma3_gguf(path, seed=21, **SHAPE)
    return path


@pytest.fixture(scope="module")
def narrow(tmp_path_factory):
    """Three heads of 96: key ranges shared by the heads of two query tiles, a short last group."""
    path = os.path.join(str(tmp_path_factory.mktemp("rowbatch")), "narrow.gguf")
    synth.write_gemma3_gguf(path, seed=22, **dict(SHAPE, n_layers=6, d_model=288, n_heads=3, head_dim=96, ffn=160, window=70,
                                                  context=1200))
    return path


@pytest.mark.parametrize("rows", ROWS)
def test_prefill_matches_decode(ctx, model, rows):
    _compare(ctx, model, rows, TOL)


@pytest.mark.parametrize("rows", (1, 31, 32, 33, 100, 333, 1187))
def test_prefill_matches_decode_three_heads(ctx, narrow, rows):
    _compare(ctx, narrow, rows, TOL)


def _compare(ctx, path, rows, tol):
    g = vrt.Gemma3(ctx, path)
    try:
        ids = synth.uniform_ids(900 + rows, rows, 2, 1000)
        print(f"[rowbatch] {rows} rows", flush=True)
        _, hp = g.prefill(ids, top_k=2, hidden=True)
        lp = g.logits()
        g.reset()
        if rows > 1:
            g.forced(ids[:-1], 0)
        _, hd = g.decode(int(ids[-1]), rows - 1, top_k=2, hidden=True)
        ld = g.logits()
        assert _rel(hp, hd) <= tol
        assert _rel(lp, ld) <= tol
    finally:
        g.close()
