"""The f32 gather at the edges of its workgroups (one wave of a tile's pieces): heads whose pieces
do not fill whole workgroups, one position, partial last tiles, blocks larger than a tile."""
import numpy as np
import pytest

from helpers import F16, Q8_0, rng
from test_gpu_kernels import cu32, cu64, fill_items, layout, new_pool

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dtype,G,D,B", [(Q8_0, 1, 64, 16), (Q8_0, 3, 64, 48), (Q8_0, 1, 128, 16), (Q8_0, 5, 128, 32),
                                         (Q8_0, 2, 256, 16), (F16, 1, 8, 16), (F16, 3, 64, 32), (F16, 5, 128, 16)])
def test_gather_f32_bit_exact(hip, dtype, G, D, B):
    print(f"gather parts {dtype} G={G} D={D} B={B}", flush=True)
    r = rng(G * D + B)
    L, lens = layout(dtype, G, D, B), [1, 15, 16, 17, 100]
    N = sum(-(-n // B) for n in lens) + 2
    pool = new_pool(L, N, fill=3)
    blocks, table_at, sim = fill_items(hip, L, pool, N, lens, r, outliers=0.01 if dtype == Q8_0 else 0)
    n = np.array(lens)
    at = np.concatenate([[3], 3 + np.cumsum(n)[:-1]])  # 3 positions in front stay untouched
    out = [torch.full(((int(n.sum()) + 3) * G * D,), -7.0, device="cuda") for _ in range(2)]
    hip.gather(L, pool, N, cu32(blocks), cu32(table_at), cu32(n), cu64(at), max(lens), *out)
    hip.check()
    for got, isv in zip((x.cpu().numpy() for x in out), (False, True)):
        assert (got[:3 * G * D] == -7.0).all()
        for t, (a, m) in enumerate(zip(at, lens)):
            want = sim.gather(blocks, table_at, t, m)[isv]
            assert np.array_equal(got[a * G * D:(a + m) * G * D].view(np.uint32),
                                  np.asarray(want, np.float32).reshape(-1).view(np.uint32))
