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


def uneven(hip, dtype, G, D, lens, max_len, seed=3):
    """Items of `lens` positions through tables into one small pool, gathered in one launch bounded
    by max_len and, as the reference, one item at a time bounded by its own length."""
    print(f"gather walk {dtype} G={G} D={D} items={len(lens)} max_len={max_len}", flush=True)
    r = rng(seed)
    L, N = layout(dtype, G, D, 16), 32
    pool = new_pool(L, N, fill=seed)
    k, v = (torch.randn((N * 16, G * D), device="cuda") for _ in range(2))
    hip.append(L, pool, N, k, v, cu32(np.arange(N * 16)))
    n, need = np.array(lens), -(-np.array(lens) // 16)
    blocks = cu32(r.integers(0, N, int(need.sum())))
    table_at = np.concatenate([[0], np.cumsum(need)[:-1]])
    at = np.concatenate([[0], np.cumsum(n)[:-1]])
    T = int(n.sum())

    def gather(items, bound, out):
        hip.gather(L, pool, N, blocks, cu32(table_at[items]), cu32(n[items]), cu64(at[items]), bound, *out)

    got, want = ([torch.full((T * G * D,), -7.0, device="cuda") for _ in range(2)] for _ in range(2))
    gather(np.arange(len(lens)), max_len, got)
    for i in range(0, len(lens), max(1, len(lens) // 40)):
        gather(np.array([i]), int(n[i]), want)
        s = slice(int(at[i]) * G * D, int(at[i] + n[i]) * G * D)
        for a, b in zip(got, want):
            assert torch.equal(a[s].view(torch.int32), b[s].view(torch.int32)), i
    assert not any((x == -7.0).any() for x in got)
    hip.check()


@pytest.mark.parametrize("dtype,G,D", [(Q8_0, 8, 128), (Q8_0, 1, 64), (Q8_0, 3, 256), (F16, 8, 128), (F16, 3, 64)])
def test_gather_of_uneven_items(hip, dtype, G, D):
    """One item far longer than the rest (units tile by tile), and batches of many pieces (units item
    by item)."""
    uneven(hip, dtype, G, D, [9001] + [1 + i % 40 for i in range(150)], 9001)
    uneven(hip, dtype, G, D, [17] * 70 + [20000], 20000)
    if G == 8:
        uneven(hip, dtype, G, D, [1 + (i * 37) % 1024 for i in range(160)], 1024)


@pytest.mark.parametrize("D", [64, 128, 256])
def test_gather_of_many_even_items(hip, D):
    """More than 16384 units, their number not a multiple of 8 (d = 128, 256: one XCD each)."""
    uneven(hip, Q8_0, 1, D, [200 + i % 61 for i in range(1101)], 260)


def test_gather_of_more_units_than_a_launch_holds(hip):
    """4096 items bounded by 16384 positions, 32 heads of 128, run (2^22 units); 65536 items bounded
    by 262160 positions (2^30 units) are refused, not cut short."""
    from qubivex_amd._lib import DeviceError

    uneven(hip, Q8_0, 32, 128, [1 + i % 20 for i in range(4096)], 16384)
    with pytest.raises(DeviceError):
        uneven(hip, Q8_0, 32, 128, [1] * 65536, 262160)
