"""The decode forms of few units: one wide workgroup per unit (k_attn_wide), and the split by
work whose waves take their shares on their own, at the sizes where they can go wrong."""
import numpy as np
import pytest

from helpers import F16, MAX_ABS, Q8_0, REL_L2, attn_errors, normal, rng
from test_gpu_append_attention import run_case
from test_gpu_kernels import cf32, cu32, fill_items, layout, new_pool

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# tiles per workgroup around the wave count (12 at d = 128, 16 at d = 64), partial last tiles,
# fewer tiles than waves, one position; more than 64 tiles per wave (a second fetch of ids)
LENS = {128: [1, 16, 191, 192, 193, 384, 400], 64: [1, 255, 256, 257, 512, 529]}
FORMS = [{"attn_wide": 1 << 20}, {"attn_stream_wg": 3}, {"attn_stream_wg": 40}]


def check_against_oracle(hip, dtype, G, H, D, B, lens):
    r, L = rng(D + G + H), layout(dtype, G, D, B)
    N = sum(-(-n // B) for n in lens) + 3
    pool = new_pool(L, N, fill=7)
    blocks, table_at, sim = fill_items(hip, L, pool, N, lens, r, outliers=0.01 if dtype == Q8_0 else 0)
    q, pos = normal(r, (len(lens), H, D)), np.array(lens, np.uint32) - 1
    out = torch.full((len(lens) * H * D,), float("nan"), dtype=torch.float32, device="cuda")
    hip.attention(L, pool, N, cf32(q), cu32(blocks), cu32(table_at), cu32(pos), H, int(pos.max()), out)
    hip.check()
    max_abs, rel = attn_errors(out.cpu().numpy().reshape(q.shape), sim.attention(q, H, blocks, table_at, pos))
    print(f"  max_abs={max_abs:.2e} rel_l2={rel:.2e}", flush=True)
    assert max_abs <= MAX_ABS and rel <= REL_L2


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("dtype,G,H,D,B", [(F16, 4, 16, 128, 16), (F16, 2, 32, 64, 32), (Q8_0, 4, 16, 128, 16),
                                           (Q8_0, 1, 7, 128, 48), (Q8_0, 2, 8, 64, 16)])
def test_forms_of_few_units_match_the_oracle(hip, knobs, dtype, G, H, D, B, form):
    print(f"few units {dtype} G={G} H={H} D={D} B={B} {form}", flush=True)
    for k, v in form.items():
        knobs(k, v)
    check_against_oracle(hip, dtype, G, H, D, B, LENS[D])


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("dtype", [F16, Q8_0])
@pytest.mark.parametrize("D,lens", [(128, [190, 191, 12300, 1, 15]), (64, [254, 256, 16500, 31])])
def test_fused_append_in_the_forms_of_few_units(hip, knobs, dtype, D, lens, form):
    run_case(hip, dtype, 2, 8, D, 16, lens, form, knobs)


@pytest.mark.parametrize("dtype,G,H", [(F16, 4, 16), (F16, 1, 16), (Q8_0, 4, 16), (Q8_0, 2, 16)])
def test_waves_on_their_own_at_d256(hip, knobs, dtype, G, H):
    """More than 8192 (unit, tile) pairs at d = 256, packed and with more than 4 query heads per KV
    head (2 head chunks at 16), beside units of one tile; few pairs, by workgroup, too."""
    lens = [8200, 33, 600, 1] + [255, 256, 257] * 3
    print(f"d=256 {dtype} G={G} H={H}", flush=True)
    check_against_oracle(hip, dtype, G, H, 256, 16, lens)
    check_against_oracle(hip, dtype, G, H, 256, 16, lens[1:4])
    run_case(hip, dtype, G, H, 256, 16, lens, {}, knobs)
