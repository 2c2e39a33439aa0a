"""LinearBackend results around the blocks they come back in: one value, one block less and more by a value, two and
several blocks, resident and temporary weights, two backends at once. Against exact float64 products."""
import sys
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BLOCK = (512 << 10) // 8  # values per block


@pytest.mark.parametrize("rows,out", [(1, 1), (1, BLOCK - 1), (1, BLOCK), (1, BLOCK + 1), (2, BLOCK), (3, BLOCK - 7),
                                      (64, 4864)])
@pytest.mark.parametrize("keyed", [True, False])
def test_blocks(torch_dev, rows, out, keyed):
    import tritify_amd as T

    print(f"case: backend blocks rows={rows} out={out} keyed={keyed}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(rows + out)
    k = 5
    x = rng.integers(-265720, 265721, size=(rows, k)).astype(np.int32)
    w = rng.integers(-265720, 265721, size=(out, k)).astype(np.int32)
    want = (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.int64).reshape(-1)
    b = T.HipBackend(0)
    wt = T.Weights(T.weight_id_fresh(), w.reshape(-1))
    for _ in range(2):
        y = b.linear_weights(x.reshape(-1), wt, rows, out, k) if keyed else b.linear(x.reshape(-1), w.reshape(-1), rows, out, k)
        assert np.array_equal(y, want)
    b.close()


def test_two_backends_in_two_threads(torch_dev):
    import tritify_amd as T

    def work(seed):
        rng = np.random.default_rng(seed)
        b = T.HipBackend(0)
        wrong = []
        for i in range(8):
            rows, out, k = int(rng.integers(1, 40)), int(rng.integers(1, 9000)), int(rng.integers(1, 60))
            x = rng.integers(-1000, 1000, size=(rows, k)).astype(np.int32)
            w = rng.integers(-265720, 265721, size=(out, k)).astype(np.int32)
            y = b.linear(x.reshape(-1), w.reshape(-1), rows, out, k).reshape(rows, out)
            wrong.append(not np.array_equal(y, (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.int64)))
        b.close()
        return wrong

    with ThreadPoolExecutor(2) as pool:
        for done in [pool.submit(work, s) for s in (1, 2)]:
            assert done.result() == [False] * 8  # an exception of the thread is raised here
