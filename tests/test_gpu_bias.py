"""The bias that goes with a call, on every route the call can take."""
import numpy as np
import pytest

from test_gpu_parity import assert_within_tolerance, make, say, truth_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,n,q,g,offset", [(512, 40, 3, 128, False), (4096, 70, 2, 64, True), (1024, 1001, 5, 32, False)])
def test_bias_on_every_kernel(lutgemm, oracle, device, k, n, q, g, offset):
    """One row, two rows, the batch kernel and the kernel for many rows, with and without splits along k.  With weights
    of zero the result is the bias bit for bit.  Otherwise one row and more than 16 are within the tolerance of the
    path around sum + bias, which are rounded once; 2 to 16 rows are the result without bias plus the bias in fp16."""
    import torch
    from lutgemm import synth
    w, W = make(lutgemm, synth, k, n, q, g, offset=offset, seed=k + n)
    zero = lutgemm.BCQWeight(w["bW"], w["alpha"] * 0, k, n, q, k // g, None)
    x = synth.make_x(40, k, seed=n)
    b = (np.random.default_rng(n).standard_normal(n) * 3).astype(np.float16)
    truth = truth_of(oracle, w, x) + b.astype(np.float64)
    xd, bd = torch.from_numpy(x).to(device), torch.from_numpy(b).to(device)
    st = torch.cuda.current_stream().cuda_stream
    for m in (1, 2, 3, 16, 17, 40):
        for splits in (1, min(4, (k + 511) // 512)):
            say("case bias", k, n, q, "m", m, "splits", splits)
            W.set_plan(4, splits)
            W.set_batch_plan(8, splits)
            y = torch.full((m, n), float("nan"), dtype=torch.float16, device=device)
            W.matvec_bias(xd.data_ptr(), y.data_ptr(), bd.data_ptr(), m, st)
            torch.cuda.synchronize()
            want = torch.full_like(y, float("nan"))
            W.matvec(xd.data_ptr(), want.data_ptr(), m, st)
            if 2 <= m <= 16:
                assert torch.equal(y, want + bd), m
            else:
                assert_within_tolerance(y.cpu().numpy(), truth[:m], "m=%d splits=%d" % (m, splits))
            zero.set_plan(4, splits)
            zero.set_batch_plan(8, splits)
            zero.matvec_bias(xd.data_ptr(), y.data_ptr(), bd.data_ptr(), m, st)
            assert torch.equal(y, bd.expand(m, n)), m
            # no bias: lutgemm_matvec
            W.matvec_bias(xd.data_ptr(), y.data_ptr(), 0, m, st)
            assert torch.equal(y.view(torch.int16), want.view(torch.int16)), m
    W.close()
    zero.close()


@pytest.mark.parametrize("rows", [1, 5, 20, 100])
def test_layer_bias(lutgemm, oracle, device, rows):
    """LutLinear with the bias it was built with, with leading dimensions, and with one that cannot join the sums."""
    import torch
    from lutgemm import synth, torch_ops
    k, n, q, g = 1024, 200, 3, 128
    w = synth.make_weight(k, n, q, g, seed=9)
    b = torch.randn(n, generator=torch.Generator().manual_seed(1)).half()
    layer = torch_ops.LutLinear(dict(bW=w["bW"], alpha=w["alpha"], q_bias=None, k=k, n=n, q=q, num_groups=k // g), bias=b)
    x = torch.from_numpy(synth.make_x(rows, k, seed=9)).to(device)
    truth = truth_of(oracle, w, x.cpu().numpy()) + b.double().numpy()
    say("case layer bias", rows)
    y = layer(x)
    assert y.shape == (rows, n) and y.dtype == torch.float16
    rel = np.linalg.norm(y.cpu().double().numpy() - truth) / np.linalg.norm(truth)
    assert rel <= 1e-3, rel
    assert torch.equal(layer(x.view(1, rows, k)), y.view(1, rows, n))
    assert torch.equal(layer(x.t().contiguous().t()), y)          # another order in memory
    if rows == 1:
        assert torch.equal(layer(x[0]), y[0])
    layer.bias = layer.bias.float()                               # what module.float() makes of it: a float32 sum
    wide = layer(x)
    assert wide.dtype == torch.float32
    assert np.linalg.norm(wide.cpu().double().numpy() - truth) / np.linalg.norm(truth) <= 1e-3
    with pytest.raises(Exception):
        torch.ops.lutgemm.matvec_bias(x, layer.handle, layer.bias)
    with pytest.raises(Exception):
        torch.ops.lutgemm.matvec_bias(x, layer.handle, b.to(device)[:-1])
    layer.weight.close()
