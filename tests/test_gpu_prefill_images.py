"""q8_0 prefill from tile images: the same operands as the form that converts its own tiles, so the
same outputs bit for bit, whatever the segments, blocks and splits."""
import numpy as np
import pytest

from helpers import Q8_0, normal, rng
from test_gpu_kernels import cf32, cu32, layout, new_pool

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def prefill(hip, knobs, L, pool, N, blocks, table_at, lens, n_tok, H, q, images, chunks=1):
    knobs("prefill_images", images)
    knobs("prefill_chunks", chunks)
    n_tok = np.array(n_tok)
    pos0, q_at = np.array(lens) - n_tok, np.concatenate([[0], np.cumsum(n_tok)[:-1]])
    out = torch.full_like(q, float("nan"))
    hip.prefill_attention(L, pool, N, q, cu32(blocks), cu32(table_at), cu32(pos0), cu32(q_at), cu32(n_tok), H,
                          max(lens) - 1, int(n_tok.max()), out)
    return out


def filled(hip, G, B, lens, seed):
    L = layout(Q8_0, G, 128, B)
    need = [-(-n // B) for n in lens]
    N = sum(need) + 3
    blocks = rng(seed).permutation(N)[:sum(need)]
    table_at = np.concatenate([[0], np.cumsum(need)[:-1]])
    pool = new_pool(L, N, fill=seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    for t, n in enumerate(lens):
        p = np.arange(n)
        slots = blocks[table_at[t] + p // B] * B + p % B
        k, v = (torch.randn((n, G * 128), generator=g, device="cuda") for _ in range(2))
        hip.append(L, pool, N, k, v, cu32(slots))
    return L, pool, N, blocks, table_at


@pytest.mark.parametrize("chunks", [1, 3])
@pytest.mark.parametrize("G,GS,B,lens,n_tok", [
    (2, 4, 16, [33, 64, 1, 300, 31, 20], [33, 10, 1, 70, 31, 0]),   # partial tiles, an empty segment
    (1, 7, 48, [200, 97], [64, 97]),
    (8, 8, 256, [500, 17], [20, 17]),
    (8, 1, 16, [8000] * 12, [5] * 12),                              # more images than are held at once
])
def test_images_give_the_same_bits(hip, knobs, G, GS, B, lens, n_tok, chunks):
    print(f"q8_0 images G={G} GS={GS} B={B} lens={lens} chunks={chunks}", flush=True)
    L, pool, N, blocks, table_at = filled(hip, G, B, lens, 5 + G)
    q = cf32(normal(rng(3), (sum(n_tok), G * GS, 128)))
    a, b = (prefill(hip, knobs, L, pool, N, blocks, table_at, lens, n_tok, G * GS, q, i, chunks) for i in (0, 1))
    hip.check()
    assert torch.isfinite(a).all() and torch.equal(a, b)


def test_images_report_what_the_other_form_reports(hip, knobs):
    from qubivex_amd._lib import ShapeError, UnsupportedError

    lens, n_tok = [100, 60], [40, 60]
    L, pool, N, blocks, table_at = filled(hip, 2, 16, lens, 9)
    q = cf32(normal(rng(3), (100, 8, 128)))
    bad = blocks.copy()
    bad[table_at[1] + 1] = N
    prefill(hip, knobs, L, pool, N, bad, table_at, lens, n_tok, 8, q, 1)
    with pytest.raises(ShapeError):
        hip.check()
    big = torch.full((1, 256), 1e5, device="cuda")  # a value scale of 787
    hip.append(L, pool, N, big, big, cu32([int(blocks[table_at[0]]) * 16 + 3]))
    prefill(hip, knobs, L, pool, N, blocks, table_at, lens, n_tok, 8, q, 1)
    with pytest.raises(UnsupportedError):
        hip.check()
