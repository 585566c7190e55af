"""GPU parity of the matrix-core matmul that streams a row's blocks in order
(mmw_kernel, mmq.hip): bit-exact against per-vector oracle matvecs at the edges
of its row tiles (16 rows, 64 per work group), token sets (8) and groups (16,
32), block counts (odd and even, with the tokens' rows staged in LDS up to
2048 columns and not beyond), and at the extreme integers of its f16 mins and
two-digit scales.  Runs on the MI355X box only."""
import numpy as np
import pytest

import npref

pytestmark = pytest.mark.gpu

Q4_K, Q6_K = 12, 14


@pytest.fixture(scope="module")
def be(oracle):
    import loom_amd
    from loom_amd import backend

    loom_amd.init(0)
    yield backend
    backend.clearWeightCache()


def _check(be, oracle, t, raw, xs, rows, cols):
    be.clearWeightCache()
    n = xs.shape[0]
    got = np.empty((n, rows), np.float32)
    assert be.matmul(t, got, raw, xs, n, rows, cols)
    want = np.stack([oracle.matvec(t, raw, xs[k], rows, cols) for k in range(n)])
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


# (row tiles) x (groups of 16 vectors) >= 1024 takes the streamed kernel
@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("rows,cols,n", [(16384 + 1, 256, 16), (8192 + 15, 768, 17), (8192 + 49, 512, 25),
                                         (8192, 2048, 32), (8192 + 16, 2304, 24), (16384 + 33, 2816, 16)])
def test_streamed_matmul_edges(be, oracle, t, rows, cols, n):
    rng = np.random.default_rng(rows + cols + n + t)
    raw = npref.pinned_scale_blocks(t, rows, cols, rng)
    xs = np.stack([oracle.normal(cols, 100 * n + k, 0.0, float(k % 5 + 1)) for k in range(n)])
    _check(be, oracle, t, raw, xs, rows, cols)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
def test_streamed_matmul_extreme_integers(be, oracle, t):
    """Every quant, scale and min at an end of its range against activations of
    one sign: the largest block integers (Q4_K 8 * 63 * 15 * 32 * 127 and the
    mins' 16 * 63 * 2032, Q6_K 128 * 32 * 256 * 127) through every exact step."""
    rows, cols, n = 16384, 512, 16
    rng = np.random.default_rng(5 + t)
    raw = npref.pinned_scale_blocks(t, rows, cols, rng)
    b = raw.reshape(-1, 144 if t == Q4_K else 210)
    if t == Q4_K:
        b[0::3, 4:] = 0xFF
        b[1::3, 16:] = 0x00
        b[1::3, 4:16] = 0xFF
    else:
        b[0::4, :192], b[0::4, 192:208] = 0xFF, 0x7F  # q - 32 = 31, scale 127
        b[1::4, :192], b[1::4, 192:208] = 0x00, 0x80  # -32, -128
        b[2::4, :192], b[2::4, 192:208] = 0x00, 0x7F
        b[3::4, :192], b[3::4, 192:208] = 0xFF, 0x80
    xs = np.ones((n, cols), np.float32)
    xs[1::2] = -3.0
    xs[2::4, ::2] = -1.0
    _check(be, oracle, t, raw, xs, rows, cols)


@pytest.mark.parametrize("n", [16, 33])
def test_dense_ffn_frame_on_matrix_cores(oracle, n):
    """A llama-architecture model in Q4_K / Q6_K: from 16 lanes its dense
    FFN's gate/up and down run on the matrix cores (frame_layer).  PARITY
    per-lane logits bit-identical to lo_decode_batch on identical state."""
    import dataclasses

    import loom_amd
    from loom_amd import frame as lh
    from oracle.model import OracleModel
    from test_gpu_frame import _batch_steps

    loom_amd.init(0)
    spec = dataclasses.replace(lh.stories15m(ctx_len=96), dim=512, n_layers=2, vocab=1024, n_heads=8, n_kv_heads=4,
                               head_dim=64, rope_dim=64, ffn=1280, embed_t=Q4_K, output_t=Q6_K, wq_t=Q4_K, wk_t=Q4_K,
                               wv_t=Q6_K, wo_t=Q4_K, ffn_gate_t=Q4_K, ffn_down_t=Q6_K)
    dm = lh.DeviceModel.synth(spec, seed=17, keep_ggml=True)
    rels, same = _batch_steps(lh, OracleModel(oracle, dm), dm, n, 2, 60, seed=n)
    assert rels.max() == 0.0 and same
