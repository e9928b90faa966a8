"""The arrays of a step arrive whole and in order from one copy."""
import numpy as np
import torch

from xllm_service_amd.engine.staging import Staging, upload


def test_upload():
    rng = np.random.default_rng(0)
    for shapes in ([(1,), (3, 5), (7,)], [(3, 1), (0,), (2, 0), (5,)],
                   [(2, 3), (4, 4), (9,), (1, 1)]):
        arrays = [rng.integers(-2 ** 31, 2 ** 31 - 1, s).astype(d)
                  for s in shapes for d in (np.int32, np.int64)]
        arrays.append((rng.integers(0, 9, (3, 8)) + 2 ** 40)[:, ::2])
        for a, t in zip(arrays, upload(arrays, "cpu")):
            assert t.shape == a.shape and t.is_contiguous()
            assert t.numpy().dtype == a.dtype and (t.numpy() == a).all()


def test_staging_sections():
    s = Staging([("a", (3,), np.int64, np.arange(3)), ("b", (5,), np.int32, -1),
                 ("t", (4, 6), np.int32, 0)], "cpu")
    assert s.dev["a"].tolist() == [0, 1, 2] and s.dev["b"].tolist() == [-1] * 5
    assert s.dev["t"].shape == (4, 6)
    s.host["a"][:] = 9
    s.host["t"][:] = np.arange(24).reshape(4, 6)
    assert s._last % 4 == 0 and s._row == 6
    s.wait()                           # nothing is on its way yet
    s.flush(2)
    s.wait()
    assert s.dev["a"].tolist() == [9] * 3
    assert s.dev["t"].flatten().tolist() == list(range(12)) + [0] * 12
    s.host["b"][:] = 4
    s.flush(4)
    assert s.dev["b"].tolist() == [4] * 5
    assert s.dev["t"].flatten().tolist() == list(range(24))
