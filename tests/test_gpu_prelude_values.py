"""The prelude's value rows: left alone without a bias or a clip, else as before, in each of its
kernels (registers, full-row, LDS)."""
import numpy as np
import pytest

import oracle
from helpers import normal, rng
from test_gpu_prelude import rope_rows

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("extra", ["none", "v_bias", "clip"])
@pytest.mark.parametrize("norm,heads,kvh,d", [("per_head", 6, 3, 128), ("none", 4, 2, 64), ("full", 6, 2, 128),
                                              ("full", 8, 1, 64), ("per_head", 3, 3, 96)])
@pytest.mark.parametrize("s", [1, 7])
def test_value_rows(hip, norm, heads, kvh, d, s, extra):
    from qubivex_amd import KvLayout

    print(f"prelude values {norm} heads={heads} kvh={kvh} d={d} s={s} {extra}", flush=True)
    r = rng(d + s)
    q, k, v = (normal(r, (s, n * d)) for n in (heads, kvh, kvh))
    v[0, 0], v[-1, -1] = np.nan, -0.0
    rope = rope_rows(r.integers(0, 900, s), d)
    code = {"none": 0, "full": 1, "per_head": 2}[norm]
    nq, nk = {"none": (0, 0), "full": (heads * d, kvh * d), "per_head": (d, d)}[norm]
    qn, kn = (normal(r, n) if n else None for n in (nq, nk))
    vb = normal(r, kvh * d) if extra == "v_bias" else None
    clip = 0.5 if extra == "clip" else None
    want = oracle.prelude(q, k, v, heads, kvh, d, rope, None, None, vb, clip, code, qn, kn, 1e-6)
    dev = lambda a: None if a is None else torch.from_numpy(a).cuda()  # noqa: E731
    got = [dev(x) for x in (q, k, v)]
    hip.prelude(KvLayout("f16", kvh, d, 16), heads, *got, dev(rope), norm=norm, clip=clip, eps=1e-6,
                v_bias=dev(vb), q_norm=dev(qn), k_norm=dev(kn))
    hip.check()
    for g, w in zip(got, want):
        assert np.array_equal(g.cpu().numpy().view(np.uint32), np.asarray(w, np.float32).reshape(g.shape).view(np.uint32))
