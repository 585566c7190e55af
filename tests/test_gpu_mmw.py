"""GPU parity of the matrix-core matmuls that stream a row's blocks in order
(mmw_kernel and, for 32-value blocks, mmw32_kernel, mmq.hip), of the one with 64
x 128 tiles (mmp_kernel) and of the one-shot kernels beside them: bit-exact
against per-vector oracle matvecs at the edges of their row tiles (16 rows, 64
per work group), token sets (8) and groups (16, 32), block counts (odd and even,
with the tokens' rows staged in LDS up to 2048 columns and not beyond), at the
extreme integers of the f16 mins and two-digit scales, and on either side of the
lines between the kernels.  Needs the GPU."""
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


# (row tiles) x (groups of 16 vectors) >= 768 takes the streamed kernel
@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("rows,cols,n", [(16384 + 1, 256, 16), (8192 + 15, 768, 17), (8192 + 49, 512, 25),
                                         (8192, 2048, 32), (8192 + 16, 2304, 24), (16384 + 33, 2816, 16)])
def test_streamed_matmul_edges(be, oracle, t, rows, cols, n):
    rng = np.random.default_rng(rows + cols + n + t)
    raw = npref.pinned_scale_blocks(t, rows, cols, rng)
    xs = np.stack([oracle.normal(cols, 100 * n + k, 0.0, float(k % 5 + 1)) for k in range(n)])
    _check(be, oracle, t, raw, xs, rows, cols)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("n", [16, 128])
def test_streamed_matmul_extreme_integers(be, oracle, t, n):
    """Every quant, scale and min at an end of its range against activations of
    one sign: the largest block integers (Q4_K 8 * 63 * 15 * 32 * 127 and the
    mins' 16 * 63 * 2032, Q6_K 128 * 32 * 256 * 127) through every exact step."""
    rows, cols = 16384, 512
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


# tiles of 64 rows x 128 vectors that fill a round of 256 CUs: full tiles, one row
# and one vector short of / past an edge, one to three blocks, a partial second round
@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("rows,cols,n", [(8192, 512, 256), (8192 - 65, 768, 255), (4096 - 63, 256, 511),
                                         (14000, 512, 255), (16384 + 8192, 256, 257 - 4)])
def test_tiled_matmul_edges(be, oracle, t, rows, cols, n):
    rng = np.random.default_rng(rows + cols + n + t)
    raw = npref.pinned_scale_blocks(t, rows, cols, rng)
    xs = np.stack([oracle.normal(cols, 100 * n + k, 0.0, float(k % 5 + 1)) for k in range(n)])
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


Q4_0, Q8_0 = 2, 8


# lane groups of 32-value blocks that stream: at least 768 (row tile, 16 vectors)
# pairs, or a shape the one-shot kernel does not hold with enough rows x vectors
# (1100 x 1952 from 58 vectors, the dot4 matvec below)
@pytest.mark.parametrize("t", [Q4_0, Q8_0])
@pytest.mark.parametrize("rows,cols,n", [(8192 + 5, 288, 16), (8192 + 17, 2080, 20), (12288 + 1, 2048, 9),
                                         (12288 + 15, 4096, 16), (16384, 32, 65), (8192 + 33, 4384, 33),
                                         (1100, 1952, 8), (1100, 1952, 58)])
def test_streamed_32_block_matmul_edges(be, oracle, t, rows, cols, n):
    """Odd block counts (9, 65, 137, 61), units of fewer than 8 blocks, one
    block per row, partial token sets and groups, rows staged whole and not."""
    rng = np.random.default_rng(rows + cols + n + t)
    raw = npref.pinned_scale_blocks(t, rows, cols, rng)
    xs = np.stack([oracle.normal(cols, 100 * n + k, 0.0, float(k % 5 + 1)) for k in range(n)])
    _check(be, oracle, t, raw, xs, rows, cols)


# either side of each line by which a Q8_0 / Q4_0 matmul is routed: rows on and off the 128-byte line (multiples
# of 128 columns in Q8_0, 256 in Q4_0), widths of 1024, 1536 and 2048, one round of one-shot work groups and two
@pytest.mark.parametrize("t", [Q4_0, Q8_0])
@pytest.mark.parametrize("rows,cols,n", [(200, 4096, 16), (300, 3072, 7), (300, 3072, 8), (257, 1088, 8),
                                         (300, 1280, 9), (768, 1024, 48), (768, 1024, 63), (1000, 960, 24), (2048, 512, 8),
                                         (8192, 512, 12), (2500, 1536, 32), (2500, 1984, 32), (2500, 1984, 47),
                                         (1500, 2016, 16), (6000, 2016, 12), (4096, 288, 8), (512, 160, 8),
                                         (512, 256, 9)])
def test_32_block_routes(be, oracle, t, rows, cols, n):
    rng = np.random.default_rng(rows + cols + n + t)
    raw = npref.pinned_scale_blocks(t, rows, cols, rng)
    xs = np.stack([oracle.normal(cols, 100 * n + k, 0.0, float(k % 5 + 1)) for k in range(n)])
    _check(be, oracle, t, raw, xs, rows, cols)


# the same for the K-quants under 16 vectors: rows of one and two blocks, rows of 20 to 24 around 2048 rows
@pytest.mark.parametrize("t,rows,cols,n", [(Q6_K, 1004, 512, 11), (Q6_K, 2500, 512, 12), (Q6_K, 7168, 256, 8),
                                           (Q6_K, 2047, 5120, 8), (Q6_K, 300, 4864, 8), (Q6_K, 2048, 6144, 8), (Q6_K, 300, 5120, 16),
                                           (Q4_K, 1000, 6144, 7), (Q4_K, 1000, 6144, 8), (Q4_K, 300, 5632, 5)])
def test_k_quant_routes(be, oracle, t, rows, cols, n):
    rng = np.random.default_rng(rows + cols + n + t)
    raw = npref.pinned_scale_blocks(t, rows, cols, rng)
    xs = np.stack([oracle.normal(cols, 100 * n + k, 0.0, float(k % 5 + 1)) for k in range(n)])
    _check(be, oracle, t, raw, xs, rows, cols)


# five to fifteen vectors on the matrix cores (one-shot; 1100 x 1024 Q4_0 on the dot4 matvec), rows too wide for
# 32 lanes a wave
@pytest.mark.parametrize("t,rows,cols,n", [(Q4_K, 300, 2048, 5), (Q4_K, 77, 8192, 17), (Q6_K, 300, 768, 8),
                                           (Q6_K, 130, 8192, 9), (Q8_0, 2100, 4096, 5), (Q4_0, 1100, 1024, 11), (Q4_0, 1100, 1088, 11),
                                           (Q4_K, 4100, 11008, 32), (Q6_K, 8200, 8448, 16)])
def test_matmul_from_five_vectors(be, oracle, t, rows, cols, n):
    rng = np.random.default_rng(rows + cols + n + t)
    raw = npref.pinned_scale_blocks(t, rows, cols, rng)
    xs = np.stack([oracle.normal(cols, 100 * n + k, 0.0, float(k % 5 + 1)) for k in range(n)])
    _check(be, oracle, t, raw, xs, rows, cols)


@pytest.mark.parametrize("t,dim,ffn,n", [(Q8_0, 288, 96, 21), (Q4_0, 544, 288, 40), (Q8_0, 2080, 768, 12),
                                         (Q4_0, 1024, 1536, 13), (Q4_K, 512, 256, 10), (Q4_K, 2304, 768, 5),
                                         (Q4_K, 2304, 3072, 17), (Q4_K, 4352, 1536, 17), (Q4_K, 2304, 768, 9), (Q4_K, 2304, 768, 10)])
def test_moe_layer_streamed_experts(be, oracle, t, dim, ffn, n):
    """The routed layer with its expert matmuls in groups of 16 for every type
    (streamed; Q4_K gate/up streamed from 2304 x 3072 on, down from 4352 x
    1536, one-shot below; 2304 x 768 from 10 tokens, the dot4 matvec before):
    ids, gates and output bits against lo_moe_batch_union."""
    _moe_layer(be, oracle, t, dim, ffn, 6, 3, n)


# small Q8_0 / Q4_0 experts: 20 tokens and either 100 pairs or more than three per expert
@pytest.mark.parametrize("t", [Q4_0, Q8_0])
@pytest.mark.parametrize("E,k,n", [(32, 4, 24), (32, 4, 25), (16, 4, 19), (16, 4, 20)])
def test_moe_layer_small_experts(be, oracle, t, E, k, n):
    _moe_layer(be, oracle, t, 768, 384, E, k, n)


def _moe_layer(be, oracle, t, dim, ffn, E, k, n):
    import torch
    from test_gpu_moe import _dev_layer, make_layer

    w = make_layer(oracle, dim, ffn, E, k, seed=dim + n, gate_t=t, down_t=t)
    layer = _dev_layer(be, w)
    xs = np.stack([oracle.normal(dim, 700 + i, 0.0, 1.0) for i in range(n)])
    resid = np.stack([oracle.normal(dim, 900 + i, 0.0, 1.0) for i in range(n)])
    out, ids = torch.from_numpy(resid.copy()).cuda(), torch.empty((n, k), dtype=torch.int32, device="cuda")
    layer(torch.from_numpy(xs).cuda(), out, combine=be.COMBINE_EXPERT_ASC, ids=ids)
    want, wid, _ = oracle.moe_batch_union(w, xs, resid)
    torch.cuda.synchronize()
    assert np.array_equal(ids.cpu().numpy().astype(np.uint32), wid)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))


# the widest rows whose block scales fit the LDS, and one block more, which no kernel serves
@pytest.mark.parametrize("t,cols,served", [(Q6_K, 2076 * 256, True), (Q6_K, 2077 * 256, False), (Q4_K, 2080 * 256, True),
                                           (Q4_K, 2081 * 256, False)])
def test_widest_streamed_rows(be, oracle, t, cols, served):
    import torch

    import loom_amd

    rows, n = 512, 256
    rng = np.random.default_rng(cols)
    raw = npref.pinned_scale_blocks(t, rows, cols, rng)
    w = be.repack_dev(t, torch.from_numpy(raw).cuda(), rows, cols, 1)
    x = torch.randn(n, cols, generator=torch.Generator(device="cuda").manual_seed(t), device="cuda")
    out = torch.full((n, rows), 7.0, device="cuda")
    rc = be.matvec_dev(t, out, w, x, n, rows, cols)
    torch.cuda.synchronize()
    if not served:
        assert rc == loom_amd.DECLINED and bool((out == 7.0).all())
        return
    assert rc == loom_amd.OK
    for k in (0, 100, n - 1):
        want = oracle.matvec(t, raw, x[k].cpu().numpy(), rows, cols)
        assert np.array_equal(out[k].cpu().numpy().view(np.uint32), want.view(np.uint32)), k


# the shared expert's matmuls add to the routed sum (accumulate) and run as one matrix each
@pytest.mark.parametrize("gt,dt,dim,sffn,n", [
    (Q8_0, Q8_0, 2048, 288, 17), (Q4_0, Q4_0, 2048, 288, 17),   # down streamed, 32-value blocks
    (Q8_0, Q8_0, 288, 4096, 32), (Q4_0, Q4_0, 288, 4096, 32),   # gate/up streamed as a pair, rows staged; down one-shot
    (Q8_0, Q8_0, 2080, 4096, 33), (Q4_0, Q4_0, 2080, 4096, 33),  # the same, rows not staged
    (Q4_K, Q4_K, 8192, 256, 16), (Q4_K, Q6_K, 8192, 256, 16),   # down one-shot
    (Q4_K, Q4_K, 8192, 256, 24), (Q4_K, Q6_K, 8192, 256, 24),   # down streamed, in groups of 16 and 32
    (Q4_K, Q4_K, 8192, 256, 250), (Q4_K, Q6_K, 8192, 256, 250),  # down on 64 x 128 tiles
])
def test_shared_expert_adds_on_matrix_cores(be, oracle, gt, dt, dim, sffn, n):
    """Bits of the whole layer against lo_moe_batch_union (EXPERT_ASC adds the
    routed sum to what out holds, then the shared expert's)."""
    import torch
    from test_gpu_moe import make_layer

    ffn, E, k = 256 if gt == Q4_K else 96, 4, 1
    w = make_layer(oracle, dim, ffn, E, k, seed=dim + n, gate_t=gt, down_t=dt)
    rng = np.random.default_rng(dim + sffn + n)
    sg, su = (npref.pinned_scale_blocks(gt, sffn, dim, rng) for _ in range(2))
    sd = npref.pinned_scale_blocks(dt, dim, sffn, rng)
    w.shexp = (sg, su, sd, gt, gt, dt, sffn)

    def dev(t, raw, rows, cols, planes=1):
        return be.repack_dev(t, torch.from_numpy(raw).cuda(), rows, cols, planes)

    layer = be.MoeLayer(dim, ffn, E, k, torch.from_numpy(w.router).cuda(), dev(gt, w.gate, ffn, dim, E),
                        dev(gt, w.up, ffn, dim, E), dev(dt, w.down, dim, ffn, E), gt, gt, dt,
                        shexp=(dev(gt, sg, sffn, dim), dev(gt, su, sffn, dim), dev(dt, sd, dim, sffn), gt, gt, dt, sffn))
    xs = np.stack([oracle.normal(dim, 700 + i, 0.0, 1.0) for i in range(n)])
    resid = np.stack([oracle.normal(dim, 900 + i, 0.0, 1.0) for i in range(n)])
    out = torch.from_numpy(resid.copy()).cuda()
    layer(torch.from_numpy(xs).cuda(), out, combine=be.COMBINE_EXPERT_ASC)
    want, _, _ = oracle.moe_batch_union(w, xs, resid)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))
