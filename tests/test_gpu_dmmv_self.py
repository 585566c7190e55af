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
