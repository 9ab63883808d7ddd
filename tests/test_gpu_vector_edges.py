"""Fr vector operations at the edges of their kernels' tiles and chunks, against
the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one block up to 256 (an element a thread) and 1024, tiles of 1024 up to 2^20, chunks of 8 in tiles above
@pytest.mark.parametrize("n", [2, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2048, 2049, 200001, 1 << 20, (1 << 20) + 1, (1 << 20) + 8199])
@pytest.mark.parametrize("in_place", [False, True])
def test_grand_product_at_tile_edges(bellman, oracle, n, in_place):
    B, dev = bellman
    x = oracle.random_fr(n + 11, n)
    dx = dev.upload(x)
    dy = dx if in_place else dev.malloc(n * 32)
    B.call("ff_grand_product", B.ff_grand_product_configuration(dev.pool, dev.stream, dx, dy, n))
    dev.sync()
    assert np.array_equal(dev.download(dy, (n, 8)), oracle.grand_product(x))
    dev.free(dx)
    if not in_place:
        dev.free(dy)
