"""GPU parity of the kernel for more than 16 activation rows: the edges of its tiles (rows, outputs, k-blocks),
every plane count with and without an offset, every scale layout, splits along k, both forms of the call (plans of two
row tiles, by their sizes; test_every_instance has them all)."""
import os
import subprocess
import sys

import numpy as np
import pytest

from gpu_util import assert_within_tolerance, run_matvec
from test_gpu_parity import make, say, truth_of

pytestmark = pytest.mark.gpu

CASES = [  # k, n, q, g, offset, rows
    (32, 1, 1, 32, False, (17,)), (512, 31, 2, 512, True, (17, 32, 33)), (544, 33, 3, 32, True, (48, 49)),
    (1056, 257, 4, 96, False, (64, 65)), (2048, 264, 5, 64, False, (31, 100)), (1536, 130, 5, 512, True, (50, 130)),
    (1024, 512, 6, 128, True, (16 * 6 + 1,)), (4096, 100, 7, 32, False, (20, 64)), (2560, 70, 8, 128, True, (17, 40)),
    (3072, 96, 8, 64, False, (80,)), (49152, 40, 3, 128, False, (18, 63)), (512, 8200, 1, 256, True, (24, 200)),
]


@pytest.mark.parametrize("k,n,q,g,offset,rows", CASES)
def test_many_rows_kernel(lutgemm, oracle, device, k, n, q, g, offset, rows):
    from lutgemm import synth
    w, W = make(lutgemm, synth, k, n, q, g, offset=offset, seed=k + n)
    x = synth.make_x(max(rows), k, seed=n)
    truth = truth_of(oracle, w, x)
    for m in rows:
        say("case rows", k, n, q, g, offset, "m", m, W.plan(m))
        y = run_matvec(lutgemm, W, x[:m], device)
        assert_within_tolerance(y, truth[:m], "m=%d plan=%s" % (m, W.plan(m)))
        # the same launch again, and the column form, bit for bit (the split-k counts are back at zero)
        assert np.array_equal(y.view(np.uint16), run_matvec(lutgemm, W, x[:m], device).view(np.uint16))
        assert np.array_equal(y.view(np.uint16), run_matvec(lutgemm, W, x[:m], device, cols=True).view(np.uint16))
        # a call of up to 16 rows afterwards finds its split-k words at zero
        assert_within_tolerance(run_matvec(lutgemm, W, x[:9], device), truth[:9], "9 rows after %d" % m)
    W.close()


@pytest.mark.parametrize("q,g", [(1, 128), (3, 128), (2, 32)])
def test_many_rows_non_finite_activations(lutgemm, device, q, g):
    """The pattern of infinities and NaNs is that of the batch kernel, and stays in the rows it belongs to."""
    from lutgemm import synth
    k, n, m = 4096, 96, 40
    w, W = make(lutgemm, synth, k, n, q, g, seed=5)
    x = synth.make_x(m, k, seed=5)
    clean = run_matvec(lutgemm, W, x, device)
    bad = x.copy()
    bad[3, 700] = np.nan
    bad[9, 5] = np.inf
    bad[12, 5], bad[12, 3000] = np.inf, -np.inf
    say("case rows non-finite", q, g, W.plan(m))
    y = run_matvec(lutgemm, W, bad, device)
    few = run_matvec(lutgemm, W, bad[:16], device)
    for r in (3, 9, 12):
        assert np.array_equal(np.isnan(y[r]), np.isnan(few[r])), r
        inf = np.isinf(few[r])
        assert np.array_equal(y[r][inf], few[r][inf]) and not np.isfinite(y[r]).any(), r
    rest = [r for r in range(m) if r not in (3, 9, 12)]
    assert np.array_equal(y[rest].view(np.uint16), clean[rest].view(np.uint16))
    W.close()


def test_many_rows_under_capture_and_on_two_streams(lutgemm, oracle, device):
    """Whether the stream's set has room for partial sums already or gets it under capture: eager launches, replays and a
    second stream give the same bits."""
    import torch
    from lutgemm import synth
    k, n, q, g, m = 8192, 512, 3, 128, 40
    w, W = make(lutgemm, synth, k, n, q, g, seed=6)
    assert W.plan(m)["k_splits"] > 1
    xs = [torch.from_numpy(synth.make_x(m, k, seed=s)).to(device) for s in (6, 7)]
    truth = [truth_of(oracle, w, x.cpu().numpy()) for x in xs]
    static_x, out = xs[0].clone(), torch.zeros((m, n), dtype=torch.float16, device=device)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    for room in (False, True):
        say("case rows capture", "after an eager call" if room else "first")
        with torch.cuda.stream(side):
            W.matvec(static_x.data_ptr(), out.data_ptr(), m if room else 1, side.cuda_stream)
            side.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                W.matvec(static_x.data_ptr(), out.data_ptr(), m, side.cuda_stream)
        for rep in range(2):
            for x, t in zip(xs, truth):
                static_x.copy_(x)
                out.zero_()
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
                assert_within_tolerance(out.cpu().numpy(), t, "replay %d" % rep)
                eager = run_matvec(lutgemm, W, x.cpu().numpy(), device)
                assert np.array_equal(out.cpu().numpy().view(np.uint16), eager.view(np.uint16)), (room, rep)
    W.close()


@pytest.mark.parametrize("q,g,offset,value", [(1, 128, False, np.inf), (3, 512, False, -np.inf), (2, 64, True, np.inf),
                                              (2, 32, False, np.inf), (3, 128, True, np.nan), (2, 128, False, 65520.0)])
def test_many_rows_non_finite_scales(lutgemm, device, tmp_path, q, g, offset, value):
    """Non-finite scales (or offsets: the last group's) give the bits of 16 rows at a time, whichever way the weight was
    made; an infinite scale of a group that is one sum (64 or 128 activations) gives infinities, not NaN."""
    from lutgemm import synth
    k, n, m = 2048, 70, 40
    w = synth.make_weight(k, n, q, g, offset=offset, seed=q + g)
    alpha, z = w["alpha"].copy(), None if w["q_bias"] is None else w["q_bias"].copy()
    alpha[1, 0, 5] = value
    if z is not None:
        z[-1, 64] = value
    x = synth.make_x(m, k, seed=12)
    W = lutgemm.BCQWeight(w["bW"], alpha, k, n, q, k // g, z)
    W.save(str(tmp_path / "w.lutw"))
    made = [W, lutgemm.BCQWeight.load(str(tmp_path / "w.lutw")), W.clone()]
    say("case rows non-finite scales", q, g, offset, value)
    want = np.concatenate([run_matvec(lutgemm, W, x[:16], device), run_matvec(lutgemm, W, x[16:32], device),
                           run_matvec(lutgemm, W, x[24:], device)[8:]])
    for V in made:
        for cols in (False, True):
            y = run_matvec(lutgemm, V, x, device, cols=cols)
            assert np.array_equal(y.view(np.uint16), want.view(np.uint16))
    assert not np.isfinite(want[:, 5]).any() and (g not in (64, 128) or np.isnan(value) or np.isinf(want[:, 5]).all())
    assert np.isfinite(np.delete(want, [5, 64], axis=1)).all()
    for V in made:
        V.close()


def test_many_rows_beside_a_capture(lutgemm, device):
    """A launch that needs room for partial sums, made by another host thread while a stream is being captured in global
    mode, neither spoils the capture nor takes another plan."""
    import threading

    import torch
    from lutgemm import synth
    k, n, q, g, m = 8192, 512, 3, 128, 40
    w, W = make(lutgemm, synth, k, n, q, g, seed=13)
    assert W.plan(m)["k_splits"] > 1
    x = torch.from_numpy(synth.make_x(m, k, seed=13)).to(device)
    want = run_matvec(lutgemm, W, x.cpu().numpy(), device)
    y, z = (torch.zeros((m, n), dtype=torch.float16, device=device) for _ in range(2))
    mine, other = torch.cuda.Stream(), torch.cuda.Stream()
    W.matvec(x.data_ptr(), y.data_ptr(), 1, other.cuda_stream)          # the stream's set, without room for partial sums
    torch.cuda.synchronize()
    errors = []

    def work():
        try:
            W.matvec(x.data_ptr(), y.data_ptr(), m, other.cuda_stream)
        except Exception as e:   # reported by the main thread
            errors.append(repr(e))

    say("case rows beside a capture")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(mine):
        z.add_(0.0)
        mine.synchronize()
        with torch.cuda.graph(graph, stream=mine):
            z.add_(1.0)
            thread = threading.Thread(target=work)
            thread.start()
            thread.join()
    torch.cuda.synchronize()
    assert not errors, errors
    assert np.array_equal(y.cpu().numpy().view(np.uint16), want.view(np.uint16))
    for rep in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, torch.full_like(z, rep + 1.0)), rep
    W.close()


def test_room_for_partial_sums_is_what_the_plan_needs(lutgemm, device):
    """A handle's device memory grows by less than twice what the plan of a call exchanges, once for calls that need as
    much, and not at all by calls that do not split k."""
    from lutgemm import synth
    k, n, q, g = 4096, 1024, 4, 128
    w, W = make(lutgemm, synth, k, n, q, g, seed=14)
    x = synth.make_x(512, k, seed=14)
    before, largest = W.info().device_bytes, 0
    for m in (512, 20, 32, 100, 64):
        plan = W.plan(m)
        say("case room", m, plan)
        run_matvec(lutgemm, W, x[:m], device)
        grown = W.info().device_bytes - before
        if plan["k_splits"] == 1:
            assert grown == 0, m
            continue
        # fp32 sums of whole tiles of 16 rows (up to 4 of them in a workgroup) and 32 outputs
        largest = max(largest, plan["k_splits"] * 4 * (n + 31) // 32 * 32 * -(-m // 64) * 64)
        assert 0 < grown < 4 * largest, (m, grown, largest)
        run_matvec(lutgemm, W, x[:m], device)
        assert W.info().device_bytes - before == grown
    assert largest
    W.close()


def test_a_batch_plan_that_is_set_holds_for_many_rows(lutgemm, oracle, device):
    """lutgemm_weight_set_batch_plan acts on calls of more than 16 rows, which take passes of 16 with it, until it is reset
    or replaced by a measurement; clones have it too."""
    from lutgemm import synth
    k, n, q, g, m = 4096, 600, 3, 128, 40
    w, W = make(lutgemm, synth, k, n, q, g, seed=15)
    x = synth.make_x(m, k, seed=15)
    auto, y_auto = W.plan(m), run_matvec(lutgemm, W, x, device)
    W.set_batch_plan(9, 4)
    V = W.clone()
    for handle in (W, V):
        say("case rows set batch plan", handle.plan(m))
        assert handle.plan(m) == handle.plan(16) and handle.plan(m)["waves"] == 9 and handle.plan(m)["k_splits"] == 4
        y = run_matvec(lutgemm, handle, x, device)
        passes = [run_matvec(lutgemm, handle, x[r:r + 16], device) for r in (0, 16, 32)]
        assert np.array_equal(y.view(np.uint16), np.concatenate(passes).view(np.uint16))
        assert_within_tolerance(y, truth_of(oracle, w, x), "passes")
    W.set_batch_plan()
    V.autotune()
    for handle in (W, V):
        assert handle.plan(m) == auto
        assert np.array_equal(run_matvec(lutgemm, handle, x, device).view(np.uint16), y_auto.view(np.uint16))
        handle.close()


def test_every_instance(lutgemm):
    """Planes, row tiles, k groups and splits along k that the plans of the sizes above do not reach (rows_test.cpp)."""
    program = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "rows_test")
    assert os.path.exists(program), "build the C++ tests first (make -C tests/cpp, or __graft_entry__.build())"
    r = subprocess.run([program], capture_output=True, text=True, timeout=110)
    sys.stdout.write(r.stdout)
    sys.stderr.write(r.stderr)
    assert r.returncode == 0 and "ROWS OK 288" in r.stdout
