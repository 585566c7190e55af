"""GPU parity of the one-vector matvec whose work groups quantize the vector
themselves (dmmv_self_kernel): loomhip_matvec_dev against the oracle's
matvec, bit for bit, at the edges of its block counts, row tiles and limits
(2048 columns, 512 work groups).  Runs on the MI355X box only."""
import numpy as np
import pytest

import npref

pytestmark = pytest.mark.gpu

Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14


@pytest.mark.parametrize("t,cols", [(Q4_0, 32), (Q4_0, 288), (Q4_0, 2048), (Q8_0, 96), (Q8_0, 2048), (Q8_0, 2080),
                                    (Q4_K, 256), (Q4_K, 2048), (Q4_K, 2304), (Q6_K, 768), (Q6_K, 2048)])
@pytest.mark.parametrize("rows", [1, 33, 768, 4097])
def test_one_vector_matvec_dev(oracle, t, rows, cols):
    import torch

    import loom_amd
    from loom_amd import backend as be

    loom_amd.init(0)
    raw = npref.pinned_scale_blocks(t, rows, cols, np.random.default_rng(rows + cols + t))
    w = be.repack_dev(t, torch.from_numpy(raw).cuda(), rows, cols, 1)
    x = oracle.normal(cols, rows + cols, 0.0, 1.0)
    x[0], x[cols // 2] = np.nan, np.inf  # quantize to zero, as everywhere
    out = torch.full((rows,), 7.0, device="cuda")
    assert be.matvec_dev(t, out, w, torch.from_numpy(x).cuda(), 1, rows, cols) == loom_amd.OK
    torch.cuda.synchronize()
    want = oracle.matvec(t, raw, x, rows, cols)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("t,rows,cols", [(Q4_0, 768, 768), (Q8_0, 2048, 2048), (Q4_K, 2048, 2048), (Q6_K, 2304, 768),
                                         (Q4_0, 96, 2048)])
@pytest.mark.parametrize("place", ["same", "tail", "head", "behind"])
def test_one_vector_matvec_dev_over_its_input(oracle, t, rows, cols, place):
    """out over x: at the same address, by x's last four elements, by out's
    last four, and right behind x without overlap.  The launches tell the route:
    two where the ranges meet (all of x is read before the first store), one
    where they do not."""
    import torch

    import loom_amd
    from loom_amd import backend as be

    loom_amd.init(0)
    raw = npref.pinned_scale_blocks(t, rows, cols, np.random.default_rng(rows + cols + t))
    w = be.repack_dev(t, torch.from_numpy(raw).cuda(), rows, cols, 1)
    x = oracle.normal(cols, rows + cols, 0.0, 1.0)
    ox, oo = {"same": (0, 0), "tail": (0, cols - 4), "head": (rows - 4, 0), "behind": (0, cols)}[place]
    buf = torch.zeros(rows + 2 * cols, device="cuda")
    buf[ox:ox + cols] = torch.from_numpy(x).cuda()
    out = buf[oo:oo + rows]
    loom_amd.take_launch_count()
    assert be.matvec_dev(t, out, w, buf[ox:ox + cols], 1, rows, cols) == loom_amd.OK
    assert loom_amd.take_launch_count() == (1 if place == "behind" else 2)
    torch.cuda.synchronize()
    want = oracle.matvec(t, raw, x, rows, cols)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("t,rows,cols,n", [(Q4_0, 768, 2048, 1), (Q4_K, 4096, 4096, 1), (Q8_0, 4097, 2048, 1),
                                           (Q8_0, 64, 2080, 1), (Q4_K, 768, 2048, 3), (Q6_K, 300, 2048, 9)])
def test_one_timing_record_per_matvec(oracle, t, rows, cols, n):
    """A call that declines the one-launch form (wider rows, more work groups)
    before it runs the two adds one sample to the matvec's timing, not two."""
    import torch

    import loom_amd
    from loom_amd import backend as be

    loom_amd.init(0)
    w = torch.zeros(loom_amd.plane_bytes(t, rows, cols), dtype=torch.uint8, device="cuda")
    x, out = torch.zeros(n, cols, device="cuda"), torch.empty(n, rows, device="cuda")
    be.profileKernels(True)
    try:
        for _ in range(3):
            assert be.matvec_dev(t, out, w, x, n, rows, cols) == loom_amd.OK
        torch.cuda.synchronize()
        assert be.kernelStats()["dense"]["count"] == 3
    finally:
        be.profileKernels(False)


@pytest.mark.parametrize("n", [1, 6])
def test_one_timing_record_per_frame_stage(n):
    """The same inside the frame: q, k and v in Q8_0 decline the matrix-core
    launch at 6 lanes; at one lane wo and the dense down decline the one-launch
    matvec where their rows are wider than 2048."""
    import dataclasses

    import torch

    import loom_amd
    from loom_amd import backend as be
    from loom_amd import frame as lh

    loom_amd.init(0)
    layers = 3
    spec = dataclasses.replace(lh.stories15m(ctx_len=32), dim=512, n_layers=layers, vocab=512, n_heads=40,
                               n_kv_heads=8, head_dim=64, rope_dim=64, ffn=2080, embed_t=Q8_0, output_t=Q8_0,
                               wq_t=Q8_0, wk_t=Q8_0, wv_t=Q8_0, wo_t=Q8_0, ffn_gate_t=Q8_0, ffn_down_t=Q8_0)
    dec = lh.Decoder(lh.DeviceModel.synth(spec, seed=3), n)
    be.profileKernels(True)
    try:
        assert dec.step() == loom_amd.OK
        torch.cuda.synchronize()
        st = be.kernelStats()
        assert [st[k]["count"] for k in ("qkv", "wo", "dense")] == [layers] * 3
    finally:
        be.profileKernels(False)


@pytest.mark.parametrize("dim,ffn,launches", [(2048, 5120, 0), (2048, 5152, 1), (2304, 4096, 0), (2304, 4128, 1)])
def test_ffn_norm_with_gate_up_at_its_limits(oracle, dim, ffn, launches):
    """One lane, PARITY: the FFN norm inside the gate/up launch up to 640 work
    groups over 2048 columns and 512 over more, in a launch of its own beyond
    (one more per layer).  Logits bit-identical to the oracle's step."""
    import dataclasses

    import loom_amd
    from loom_amd import frame as lh
    from oracle.model import OracleModel
    from test_gpu_frame import _batch_steps

    loom_amd.init(0)
    layers = 2
    spec = dataclasses.replace(lh.stories15m(ctx_len=32), dim=dim, n_layers=layers, vocab=512, n_heads=4,
                               n_kv_heads=4, head_dim=64, rope_dim=64, ffn=ffn)
    dm = lh.DeviceModel.synth(spec, seed=5, keep_ggml=True)
    rels, same = _batch_steps(lh, OracleModel(oracle, dm), dm, 1, 2, 8, seed=3)
    assert rels.max() == 0.0 and same
    count = []
    for f in (4096, ffn):
        dec = lh.Decoder(lh.DeviceModel.synth(dataclasses.replace(spec, ffn=f), seed=5), 1)
        loom_amd.take_launch_count()
        assert dec.step() == loom_amd.OK
        count.append(loom_amd.take_launch_count())
    assert count[1] - count[0] == launches * layers
