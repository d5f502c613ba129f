"""GPU parity of the kernel for 3 to 16 activation rows: the plans and routes that
the library takes (rows, columns read as they are and gathered, sums by atomics and through memory), and every instance
through its launch interface."""
import os
import subprocess
import sys

import numpy as np
import pytest

from gpu_util import assert_within_tolerance, run_matvec
from test_gpu_parity import make, say, truth_of

pytestmark = pytest.mark.gpu

CASES = [  # k, n, q, g, offset: plans of 8 and of more wavefronts, sums by atomics and through memory
    (128, 1, 1, 128, False), (640, 33, 2, 640, True), (8192, 512, 3, 128, False), (2048, 8200, 2, 256, False),
    (4096, 8192, 4, 128, True), (12288, 1536, 1, 128, False), (3072, 264, 8, 128, True), (1024, 12290, 5, 512, False),
    (32, 40, 2, 32, False), (7168, 1024, 3, 32, False), (4160, 4104, 2, 64, True), (2080, 12288, 4, 32, True), (1536, 96, 7, 64, False),
]


@pytest.mark.parametrize("k,n,q,g,offset", CASES)
def test_few_rows_kernel(lutgemm, oracle, device, k, n, q, g, offset):
    from lutgemm import synth
    w, W = make(lutgemm, synth, k, n, q, g, offset=offset, seed=k + n)
    x = synth.make_x(16, k, seed=n)
    truth = truth_of(oracle, w, x)
    for m in (3, 8, 9, 16):
        say("case few rows", k, n, q, g, offset, "m", m, W.plan(m))
        y = run_matvec(lutgemm, W, x[:m], device)
        assert_within_tolerance(y, truth[:m], "m=%d plan=%s" % (m, W.plan(m)))
        # the same launch again, and the column form, bit for bit (the words for the splits are back at zero)
        assert np.array_equal(y.view(np.uint16), run_matvec(lutgemm, W, x[:m], device).view(np.uint16))
        assert np.array_equal(y.view(np.uint16), run_matvec(lutgemm, W, x[:m], device, cols=True).view(np.uint16))
        # the batch kernel, which other weights take, agrees
        W.set_batch_plan(8, 1)
        assert_within_tolerance(run_matvec(lutgemm, W, x[:m], device), truth[:m], "batch kernel, m=%d" % m)
        W.set_batch_plan()
    W.close()


@pytest.mark.parametrize("q,g,offset", [(1, 128, False), (3, 128, False), (2, 128, True), (3, 64, False), (2, 32, True)])
def test_few_rows_non_finite_activations(lutgemm, device, q, g, offset):
    """The pattern of infinities and NaNs is that of the batch kernel, and stays in the rows it belongs to."""
    from lutgemm import synth
    k, n, m = 4096, 96, 9
    w, W = make(lutgemm, synth, k, n, q, g, offset=offset, seed=5)
    x = synth.make_x(m, k, seed=5)
    clean = run_matvec(lutgemm, W, x, device)
    bad = x.copy()
    bad[1, 700] = np.nan
    bad[4, 5] = np.inf
    bad[8, 5], bad[8, 3000] = np.inf, -np.inf
    say("case few rows non-finite", q, g, offset, W.plan(m))
    y = run_matvec(lutgemm, W, bad, device)
    W.set_batch_plan(8, 2)
    batch = run_matvec(lutgemm, W, bad, device)
    for r in (1, 4, 8):
        assert np.array_equal(np.isnan(y[r]), np.isnan(batch[r])) and not np.isfinite(y[r]).any(), r
        inf = np.isinf(batch[r])
        assert np.array_equal(y[r][inf], batch[r][inf]), r
    rest = [r for r in range(m) if r not in (1, 4, 8)]
    assert np.array_equal(y[rest].view(np.uint16), clean[rest].view(np.uint16))
    W.close()


@pytest.mark.parametrize("k,n,q,g,offset", [(1120, 4104, 2, 32, True), (640, 300, 3, 128, False), (4160, 96, 4, 64, False), (32, 40, 6, 32, True)])
def test_few_columns_end_at_k(lutgemm, device, k, n, q, g, offset):
    """k ends within a k-block and NaNs follow the last column of x: they must not be read, neither as part of the block nor as what
    the zero scales of the tile's padding are multiplied with."""
    import torch
    from lutgemm import synth
    _, W = make(lutgemm, synth, k, n, q, g, offset=offset, seed=k)
    x = synth.make_x(16, k, seed=n)
    for m in (3, 7, 8, 12, 16):
        say("case few columns end at k", k, n, q, g, offset, "m", m, W.plan(m))
        assert W.plan(m)["waves"] == 8   # read as they are
        rows = run_matvec(lutgemm, W, x[:m], device)
        xd = torch.full((k * m + 16384,), float("nan"), dtype=torch.float16, device=device)
        xd[:k * m] = torch.from_numpy(np.ascontiguousarray(x[:m].T).reshape(-1)).to(device)
        yd = torch.zeros((n, m), dtype=torch.float16, device=device)
        W.matvec_cols(xd.data_ptr(), yd.data_ptr(), m, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert np.array_equal(yd.cpu().numpy().T.view(np.uint16), rows.view(np.uint16))
    W.close()


@pytest.mark.parametrize("k,n,q,g,offset", [(4096, 4096, 3, 128, False), (2048, 8192, 2, 64, True), (7168, 1024, 4, 32, False)])
def test_columns_in_place(lutgemm, device, k, n, q, g, offset):
    """y over x: the results of a call into another buffer, bit for bit, however the two overlap."""
    import torch
    from lutgemm import synth
    _, W = make(lutgemm, synth, k, n, q, g, offset=offset, seed=k)
    st = torch.cuda.current_stream().cuda_stream
    direct = 0
    for m in (2, 3, 8, 16, 20):
        direct += 3 <= m <= 16 and W.plan(m)["waves"] == 8   # read where they lie into another buffer
        x = torch.from_numpy(np.ascontiguousarray(synth.make_x(m, k, seed=m).T)).to(device).reshape(-1)
        apart = torch.zeros(n * m, dtype=torch.float16, device=device)
        W.matvec_cols(x.data_ptr(), apart.data_ptr(), m, st)
        for x_at, y_at in ((0, 0), (0, 128 * m), (64 * m, 0), (0, (k - 1) * m + m - 1), ((n - 8) * m, 0)):
            say("case columns in place", k, n, q, g, offset, "m", m, "x at", x_at, "y at", y_at, W.plan(m))
            both = torch.zeros(max(x_at + k * m, y_at + n * m), dtype=torch.float16, device=device)
            xv, yv = both[x_at:x_at + k * m], both[y_at:y_at + n * m]
            assert xv.data_ptr() % 16 == 0
            xv.copy_(x)
            W.matvec_cols(xv.data_ptr(), yv.data_ptr(), m, st)
            torch.cuda.synchronize()
            assert torch.equal(yv.view(torch.int16), apart.view(torch.int16))
    assert direct
    W.close()


@pytest.mark.parametrize("k,n,q,g", [(12288, 32768, 4, 128), (12288, 32768, 3, 128), (12288, 32768, 4, 64), (12288, 32768, 4, 32),
                                     (12288, 16384, 6, 128)])
def test_few_rows_planes_that_cancel(lutgemm, device, k, n, q, g):
    """Every code is the weight zero (uniform codes around an offset), the activations have a mean: the planes' sums are large and
    cancel exactly, so a result is the rounding of the sums.  A matrix instruction rounds its 64 products and the sum so far,
    which is at most what all planes add up to between two cancellations: a step of 64 k, or a k-block of 512 where five
    planes and more take two passes over it.  A rounding is within half a unit in the last place (2^-24 of that), its deviation
    1 / sqrt(3) of it, and 1 / 3 as the sum grows from nothing; independent ones add up by the root of their number.  The bound is
    six of these deviations, for 16 n results."""
    step, code = 2.0 ** -7, 4
    signs = [code >> b & 1 for b in range(q)]
    alpha = np.array([step * 2 ** b / 2 for b in range(q)], dtype=np.float32)
    offset = -sum(a if s else -a for a, s in zip(alpha, signs))
    bW = np.empty((k // 32, q, n), dtype=np.uint32)
    for b in range(q):
        bW[:, b] = 0xffffffff if signs[b] else 0
    W = lutgemm.BCQWeight(bW, np.broadcast_to(alpha[None, :, None], (k // g, q, n)).copy(), k, n, q, k // g,
                          np.full((k // g, n), offset, dtype=np.float32))
    x = (np.random.default_rng(k + q).standard_normal((16, k)) + 1).astype(np.float16)
    window = 64 if q + 1 <= 4 else 512
    most = float(alpha.sum() + abs(offset)) * np.abs(x.astype(np.float64)).reshape(16, -1, window).sum(2).max()
    bound = 2 * 2.0 ** -24 * most * np.sqrt(k / 64 * (q + 1))
    for m in (8, 16):
        say("case few rows planes that cancel", k, n, q, g, "m", m, W.plan(m), "bound", bound)
        worst = float(np.abs(run_matvec(lutgemm, W, x[:m], device).astype(np.float64)).max())
        say("largest", worst)
        assert worst <= bound, (m, worst, bound)
    W.close()


@pytest.mark.parametrize("q,g,offset,rows", [(1, 128, False, (3, 8, 5)), (2, 256, True, (16, 3, 9)), (3, 32, False, (8, 7, 4)),
                                             (6, 64, True, (4, 16, 12)), (8, 128, False, (9, 16, 3))])
def test_few_rows_work_list(lutgemm, oracle, device, q, g, offset, rows):
    """Independent batches in one launch, with and without splits along k, one of odd width; a weight with an infinite scale
    among them, which the batch kernel keeps, divides the list and has the results of its own call."""
    import torch
    from lutgemm import synth
    shapes = [(1024, 300), (3072, 96), (512, 2049)]
    made = [make(lutgemm, synth, k, n, q, g, offset=offset, seed=k + i) for i, (k, n) in enumerate(shapes)]
    w_inf, _ = made[0]
    alpha = np.array(w_inf["alpha"], dtype=np.float32)
    alpha[0, 0, 5] = np.inf
    W_inf = lutgemm.BCQWeight(w_inf["bW"], alpha, 1024, 300, q, 1024 // g, w_inf["q_bias"])
    xs = [synth.make_x(m, k, seed=m) for (k, n), m in zip(shapes, rows)]
    for with_inf in (False, True):
        items = list(zip([W for _, W in made], xs, [n for _, n in shapes]))
        if with_inf:
            items.insert(1, (W_inf, xs[0], 300))
        xd = [torch.from_numpy(x).to(device) for _, x, _ in items]
        yd = [torch.zeros((x.shape[0], n), dtype=torch.float16, device=device) for _, x, n in items]
        seq = lutgemm.MatvecSequence([(W, x.data_ptr(), y.data_ptr(), x.shape[0]) for (W, _, _), x, y in zip(items, xd, yd)])
        say("case few rows list", q, g, offset, rows, "inf", with_inf, seq.fused_plan())
        assert seq.fused_plan()["entries"] == (1 if with_inf else 3)
        for _ in range(2):
            seq.launch(torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            got = [y.cpu().numpy() for y in yd]
            if with_inf:
                assert np.array_equal(got[1].view(np.uint16), run_matvec(lutgemm, W_inf, xs[0], device).view(np.uint16))
                del got[1]
            for (w, _), x, y in zip(made, xs, got):
                assert_within_tolerance(y, truth_of(oracle, w, x), "list, m=%d" % x.shape[0])
    for W in [W for _, W in made] + [W_inf]:
        W.close()


@pytest.mark.parametrize("infinite", [False, True])
@pytest.mark.parametrize("q,g,offset,rows", [(1, 128, True, (3, 8, 16)), (2, 64, False, (16, 5, 9)), (3, 32, False, (8, 9, 4)), (4, 32, True, (4, 16, 12)),
                                             (6, 128, True, (9, 3, 16)), (8, 64, False, (12, 4, 7)), (5, 32, True, (3, 16, 8))])
def test_work_list_of_the_batch_kernel(lutgemm, oracle, device, q, g, offset, rows, infinite):
    """Weights with a plan set for the batch kernel, and weights with infinite scales, share launches of it: results are those of
    single calls with the list's split along k bit for bit, so that a NaN or an infinity stays with its output."""
    import torch
    from lutgemm import synth
    st = torch.cuda.current_stream().cuda_stream
    items = []
    for i, ((k, n), m) in enumerate(zip([(1024, 300), (4096, 96), (512, 2049)], rows)):
        w = synth.make_weight(k, n, q, g, offset=offset, seed=k + i)
        alpha = np.array(w["alpha"], dtype=np.float32)
        if infinite:
            alpha[0, q - 1, 5] = np.inf if i else -np.inf
        W = lutgemm.BCQWeight(w["bW"], alpha, k, n, q, k // g, w["q_bias"])
        if not infinite:
            W.set_batch_plan(8, 1)
        x = synth.make_x(m, k, seed=m)
        items.append((w, W, x, torch.from_numpy(x).to(device), torch.zeros((m, n), dtype=torch.float16, device=device)))
    seq = lutgemm.MatvecSequence([(W, xd.data_ptr(), yd.data_ptr(), xd.shape[0]) for _, W, _, xd, yd in items])
    plan = seq.fused_plan()
    say("case list of the batch kernel", q, g, offset, rows, infinite, plan)
    assert plan["entries"] == 3
    seq.launch(st)
    torch.cuda.synchronize()
    first = [yd.cpu().numpy() for *_, yd in items]
    seq.launch(st)
    torch.cuda.synchronize()
    for (w, W, x, _, yd), y in zip(items, first):
        n = y.shape[1]
        assert np.array_equal(yd.cpu().numpy().view(np.uint16), y.view(np.uint16))
        blocks = -(-W.kSize // 512)
        per_split = min(plan["k_blocks"], blocks)
        splits = -(-blocks // per_split)
        assert -(-blocks // splits) == per_split, "a split that single calls can be given"
        W.set_batch_plan(8, splits)
        single = run_matvec(lutgemm, W, x, device)
        finite = np.delete(np.arange(n), 5) if infinite else np.arange(n)
        assert np.array_equal(y[:, finite].view(np.uint16), single[:, finite].view(np.uint16))
        assert_within_tolerance(y[:, finite], truth_of(oracle, w, x)[:, finite], "list, m=%d" % x.shape[0])
        if infinite:
            assert not np.isfinite(y[:, 5]).any()
            assert np.array_equal(np.isnan(y[:, 5]), np.isnan(single[:, 5]))
            whole = ~np.isnan(single[:, 5])
            assert np.array_equal(y[whole, 5], single[whole, 5])
        W.close()


def test_every_few_rows_instance(lutgemm):
    """Planes, inputs, wavefronts, splits along k and their sums that the plans of the sizes above do not reach."""
    program = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "few_test")
    assert os.path.exists(program), "build the C++ tests first (make -C tests/cpp, or __graft_entry__.build())"
    r = subprocess.run([program], capture_output=True, text=True, timeout=110)
    sys.stdout.write(r.stdout)
    sys.stderr.write(r.stderr)
    assert r.returncode == 0 and "FEW OK 960" in r.stdout


def test_without_memory_for_partial_sums(lutgemm):
    """Handles whose device refuses the room for the partial sums of 3 to 16 rows (room_test.cpp)."""
    program = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "room_test")
    assert os.path.exists(program), "build the C++ tests first (make -C tests/cpp, or __graft_entry__.build())"
    r = subprocess.run([program], capture_output=True, text=True, timeout=110)
    sys.stdout.write(r.stdout)
    sys.stderr.write(r.stderr)
    assert r.returncode == 0 and "ROOM OK" in r.stdout
