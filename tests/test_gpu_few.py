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


def test_every_few_rows_instance(lutgemm):
    """Planes, inputs, wavefronts, splits along k and their sums that the plans of the sizes above do not reach."""
    program = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "few_test")
    assert os.path.exists(program), "build the C++ tests first (make -C tests/cpp, or __graft_entry__.build())"
    r = subprocess.run([program], capture_output=True, text=True, timeout=110)
    sys.stdout.write(r.stdout)
    sys.stderr.write(r.stderr)
    assert r.returncode == 0 and "FEW OK 960" in r.stdout
