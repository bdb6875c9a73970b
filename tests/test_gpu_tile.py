"""The row-major -> tiled fragment layout (whole 16-byte pieces, or element by element for a matrix
that is not aligned to them) against the layout's definition: element (n, k) of K-wide rows lies in
the 8 KiB tile (n / 16, k / 256) at ((step * 4 + group) * 16 + n % 16) * 8 + k % 8 with step = k / 8 % 8
and group = k % 256 / 64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from qwen35 import Engine
    e = Engine(max_rows=16, max_ctx=256, seed=0)
    yield e
    e.close()


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("N,K", [(16, 256), (48, 1024), (112, 512), (2000, 1024), (1024, 3584)])
def test_tiles(eng, N, K, shift):
    import torch
    rng = np.random.default_rng(N + K)
    src = rng.integers(0, 1 << 15, N * K).astype(np.int16)
    rows = (N + 15) // 16 * 16
    x = torch.zeros(N * K + 8, dtype=torch.int16, device="cuda")
    x[shift:shift + N * K] = torch.from_numpy(src).cuda()
    y = torch.full((rows * K,), -1, dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    eng.op_tile_weight(x.data_ptr() + 2 * shift, N, K, y.data_ptr())
    eng.sync()
    n, k = np.meshgrid(np.arange(N), np.arange(K), indexing="ij")
    at = ((n // 16) * (K // 256) + k // 256) * 4096 + (((k // 8 % 8) * 4 + k % 256 // 64) * 16 + n % 16) * 8 + k % 8
    want = np.full(rows * K, -1, np.int16)
    want[at.reshape(-1)] = src
    assert np.array_equal(y.cpu().numpy(), want)
