"""Weights re-tiled on the device against the host packer, byte for byte (padding included)."""
import numpy as np
import pytest

from test_packer import SHAPES, problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,q,g,offset", SHAPES + [(544, 4099, 4, 544, True), (8192, 257, 3, 32, True), (512, 36, 7, 64, False)])
def test_device_tiles_equal_host_tiles(lutgemm, device, tmp_path, K, N, q, g, offset):
    print("case pack", K, N, q, g, offset, flush=True)
    rng = np.random.default_rng(K + N)
    bW, alpha, z = problem(rng, K, N, q, g, offset)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, -np.nan, 65504, 65519.9, 65520, 1e30, 2.0 ** -24, 2.0 ** -25,
                        2.0 ** -25 * 1.0001, 3 * 2.0 ** -25, 1 + 2.0 ** -11, 1 + 3 * 2.0 ** -11, -1e-9, 1e-40, 6.1e-5], np.float32)
    wide = rng.normal(0, 1, size=alpha.shape).astype(np.float32)
    wide.reshape(-1)[:special.size] = special[:wide.size]
    wide_z = None if z is None else rng.normal(0, 1, size=z.shape).astype(np.float32)
    for a, o in ((alpha.view(np.float16), None if z is None else z.view(np.float16)), (wide, wide_z)):
        lutgemm.pack_file(str(tmp_path / "host.lutw"), bW, a, K, N, q, K // g, o)
        W = lutgemm.BCQWeight(bW, a, K, N, q, K // g, o)
        W.save(str(tmp_path / "device.lutw"))
        W.close()
        assert (tmp_path / "device.lutw").read_bytes() == (tmp_path / "host.lutw").read_bytes(), a.dtype
