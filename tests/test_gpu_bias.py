"""The bias that goes with a call, on every route the call can take."""
import numpy as np
import pytest

from test_gpu_parity import make, say, truth_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,n,q,g,offset", [(512, 40, 3, 128, False), (4096, 70, 2, 64, True), (1024, 1001, 5, 32, False)])
def test_bias_on_every_kernel(lutgemm, oracle, device, k, n, q, g, offset):
    """One row, two rows, the kernels for few and for many rows, and the batch kernel for all from 3 rows on where its plan is
    set, with and without splits along k: the result without bias plus the bias in fp16, bit for bit; with weights of zero, the bias."""
    import torch
    from lutgemm import synth
    w, W = make(lutgemm, synth, k, n, q, g, offset=offset, seed=k + n)
    zero = lutgemm.BCQWeight(w["bW"], w["alpha"] * 0, k, n, q, k // g, None)
    x = synth.make_x(40, k, seed=n)
    b = (np.random.default_rng(n).standard_normal(n) * 3).astype(np.float16)
    xd, bd = torch.from_numpy(x).to(device), torch.from_numpy(b).to(device)
    st = torch.cuda.current_stream().cuda_stream
    for m in (1, 2, 3, 16, 17, 40):
        for splits in (0, 1, min(4, (k + 511) // 512)):   # 0: the automatic plans
            say("case bias", k, n, q, "m", m, "splits", splits, W.plan(m))
            W.set_plan(4 if splits else 0, splits)
            W.set_batch_plan(8 if splits else 0, splits)
            if m > 16 and not splits:
                assert (W.plan(m)["k_splits"] > 1) == (k > 1024)
            y = torch.full((m, n), float("nan"), dtype=torch.float16, device=device)
            W.matvec_bias(xd.data_ptr(), y.data_ptr(), bd.data_ptr(), m, st)
            torch.cuda.synchronize()
            want = torch.full_like(y, float("nan"))
            W.matvec(xd.data_ptr(), want.data_ptr(), m, st)
            assert torch.equal(y.view(torch.int16), (want + bd).view(torch.int16)), m
            zero.set_plan(4 if splits else 0, splits)
            zero.set_batch_plan(8 if splits else 0, splits)
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


@pytest.mark.parametrize("rows", [1, 2, 16, 17, 40, 600])
def test_layer_bias_has_the_bits_of_an_addition(lutgemm, device, rows):
    """Whether the bias goes with the call or not, on the packed route and on the dense one."""
    import torch
    from lutgemm import synth, torch_ops
    k, n, q, g = 1024, 200, 3, 128
    w = synth.make_weight(k, n, q, g, seed=10)
    c = dict(bW=w["bW"], alpha=w["alpha"], q_bias=None, k=k, n=n, q=q, num_groups=k // g)
    b = torch.randn(n, generator=torch.Generator().manual_seed(2)).half().to(device)
    layer, plain = torch_ops.LutLinear(c, bias=b), torch_ops.LutLinear(c)
    x = torch.from_numpy(synth.make_x(rows, k, seed=10)).to(device)
    say("case layer bias bits", rows)
    assert torch.equal(layer(x).view(torch.int16), (plain(x) + b).view(torch.int16))
    layer.weight.close()
    plain.weight.close()


@pytest.mark.parametrize("transform", ["vmap", "vmap last", "jvp", "forward mode", "grad", "vmap of grad", "backward"])
def test_layer_bias_is_transformed_like_an_addition(lutgemm, device, transform):
    """A bias that is mapped over or differentiated is added to the result, whose derivative in it is one."""
    import torch
    import torch.autograd.forward_ad as forward_ad
    from lutgemm import synth, torch_ops
    k, n, q, g, m = 512, 40, 3, 128, 3
    w = synth.make_weight(k, n, q, g, seed=11)
    layer = torch_ops.LutLinear(dict(bW=w["bW"], alpha=w["alpha"], q_bias=None, k=k, n=n, q=q, num_groups=k // g), bias=torch.zeros(n))
    x = torch.from_numpy(synth.make_x(m, k, seed=11)).to(device)
    y = torch.ops.lutgemm.matvec(x, layer.handle)
    some = torch.randn(4, n, generator=torch.Generator().manual_seed(3)).half().to(device)
    ones = torch.ones(n, dtype=torch.float16, device=device)

    def call(bias):
        return torch.func.functional_call(layer, {"bias": bias}, (x,))

    say("case layer bias transform", transform)
    if transform == "vmap":
        assert torch.equal(torch.vmap(call)(some), y + some[:, None])
    elif transform == "vmap last":
        assert torch.equal(torch.vmap(call, in_dims=1)(some.t().contiguous()), y + some[:, None])
    elif transform == "jvp":
        value, tangent = torch.func.jvp(call, (some[0],), (ones,))
        assert torch.equal(value, y + some[0]) and torch.equal(tangent, ones.expand(m, n))
    elif transform == "forward mode":
        with forward_ad.dual_level():
            value, tangent = forward_ad.unpack_dual(call(forward_ad.make_dual(some[0], ones)))
            assert torch.equal(value, y + some[0]) and torch.equal(tangent, ones.expand(m, n))
    elif transform == "grad":
        assert torch.equal(torch.func.grad(lambda b: call(b).sum())(some[0]), ones * m)
    elif transform == "vmap of grad":
        assert torch.equal(torch.vmap(torch.func.grad(lambda b: call(b).sum()))(some), (ones * m).expand(4, n))
    else:
        leaf = some[0].clone().requires_grad_()
        call(leaf).sum().backward()
        assert torch.equal(leaf.grad, ones * m)
    layer.weight.close()
