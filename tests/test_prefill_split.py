"""Prefill launches whose row blocks share their context out to several workgroups
(k_prefill_f16 / k_prefill_q8 with n_ch chunks and k_prefill_merge): the workgroup mapping
restated on the CPU, and on the GPU every chunk count against the oracle."""
import random

import numpy as np
import pytest

from helpers import F16, MAX_ABS, Q8_0, REL_L2, attn_errors, normal, rng
from test_gpu_prefill import expand

torch = pytest.importorskip("torch")


def launch(groups_seg, n_ch, n_qb):
    """The host's n_sub and grid (launch_prefill)."""
    groups, n_sub = groups_seg * n_ch, 1
    while groups < 128 and groups * n_sub % 8 and n_sub * 2 <= n_qb:
        n_sub *= 2
    return n_sub, -(-groups * n_sub // 8) * 8 * -(-n_qb // n_sub)


def row_block(bid, n_cb, n_ch, n_sub, n_il, xcd_map):
    per = -(-n_cb // n_sub)
    i = bid // 8 if xcd_map else bid
    q, b = (i % n_il, i // n_il) if n_il else (i // per, i % per)
    part = q * 8 + bid % 8 if xcd_map else q
    return (n_cb - 1 - (b * n_sub + part % n_sub)) % 2**32, part // n_sub % n_ch, part // n_sub // n_ch


@pytest.mark.parametrize("xcd_map", [True, False])
def test_every_row_block_and_chunk_has_one_workgroup(xcd_map):
    r = random.Random(3)
    for _ in range(300):
        sg, n_ch, n_qb = r.randint(1, 70), r.randint(1, 16), r.choice([1, 2, 3, 5, 8, 33, 64])
        n_sub, grid = launch(sg, n_ch, n_qb)
        parts = -(-sg * n_ch * n_sub // 8) * 8
        for n_il in (0, parts // 8 if xcd_map else parts):
            seen = [b for b in (row_block(x, n_qb, n_ch, n_sub, n_il, xcd_map) for x in range(grid))
                    if b[0] < n_qb and b[2] < sg]
            assert len(seen) == len(set(seen)) == sg * n_ch * n_qb, (sg, n_ch, n_qb, n_il)


@pytest.mark.gpu
@pytest.mark.parametrize("chunks", [2, 3, 16])
@pytest.mark.parametrize("dtype,H,G,D,B", [(F16, 32, 8, 128, 16), (F16, 8, 2, 64, 48), (Q8_0, 32, 8, 128, 32),
                                           (F16, 14, 2, 128, 256)])
def test_split_prefill_matches_the_oracle(hip, knobs, dtype, H, G, D, B, chunks):
    """Segments of fewer tiles than chunks, of whole and partial tiles, a single token, an empty
    one and rows that see none of a chunk's positions; the refused segment writes nothing."""
    from test_gpu_kernels import cf32, cu32, fill_items, layout, new_pool

    print(f"split prefill {dtype} H={H} G={G} D={D} B={B} chunks={chunks}", flush=True)
    knobs("prefill_chunks", chunks)
    r = rng(40 + D + B + chunks)
    L = layout(dtype, G, D, B)
    lens, n_tok = [33, 320, 7, 1, 641, 16, 50], np.array([33, 70, 7, 1, 40, 0, 20], np.uint32)
    N = sum(-(-n // B) for n in lens) + 5
    pool = new_pool(L, N, fill=9)
    blocks, table_at, sim = fill_items(hip, L, pool, N, lens, r, outliers=0.01 if dtype == Q8_0 else 0)
    T = int(n_tok.sum())
    q_at = np.concatenate([[0], np.cumsum(n_tok)[:-1]]).astype(np.uint32)
    pos0 = (np.array(lens) - n_tok).astype(np.uint32)
    q = normal(r, (T, H, D))

    def attend(nt):
        out = torch.full((T * H * D,), float("nan"), dtype=torch.float32, device="cuda")
        hip.prefill_attention(L, pool, N, cf32(q), cu32(blocks), cu32(table_at), cu32(pos0), cu32(q_at),
                              cu32(nt), H, max(lens) - 1, 70, out)
        return out

    out = attend(n_tok)
    hip.check()
    got = out.cpu().numpy().reshape(T, H, D)
    ta, pos, rows = expand(table_at, lens, n_tok, q_at)
    max_abs, rel = attn_errors(got[rows], sim.attention(q[rows], H, blocks, ta, pos))
    print(f"  max_abs={max_abs:.2e} rel_l2={rel:.2e}", flush=True)
    assert max_abs <= MAX_ABS and rel <= REL_L2
    from qubivex_amd._lib import ShapeError

    bad = n_tok.copy()
    bad[1] = 71  # more tokens than max_tok
    out = attend(bad)
    with pytest.raises(ShapeError):
        hip.check()
    assert torch.isnan(out.reshape(T, H * D)[33:103]).all() and torch.isfinite(out.reshape(T, H * D)[103:]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("knob", [{"prefill_dma": 0}, {"prefill_dma": 0, "prefill_exact_p": 1},
                                  {"prefill_exact_p": 1}, {"prefill_v2": 0}], ids=str)
@pytest.mark.parametrize("chunks", [1, 3])
@pytest.mark.parametrize("H,G,D,B", [(32, 8, 128, 16), (8, 2, 64, 48)])
def test_other_f16_builds_match_the_oracle(hip, knobs, H, G, D, B, chunks, knob):
    """The register-staged builds, those that carry P exactly, and the form without a split (which
    takes no chunks), on the same segments."""
    print(f"{knob}", flush=True)
    for k, v in knob.items():
        knobs(k, v)
    test_split_prefill_matches_the_oracle(hip, knobs, F16, H, G, D, B, chunks)


@pytest.mark.gpu
def test_captured_split_prefill_survives_a_larger_launch(hip, knobs):
    """A launch captured on a stream with a workspace, and on one without, allocates nothing and
    replays right after a later launch that outgrew the workspace."""
    from test_gpu_kernels import cf32, cu32, fill_items, layout, new_pool

    knobs("prefill_chunks", 4)
    r, H, G, D = rng(5), 16, 4, 128
    L = layout(F16, G, D)
    lens = [600] * 40
    N = 40 * 38 + 3
    pool = new_pool(L, N, fill=2)
    blocks, table_at, _ = fill_items(hip, L, pool, N, lens, r)
    q, b, ta = cf32(normal(r, (40 * 64, H, D))), cu32(blocks), cu32(table_at)

    def attend(n, out):
        p0, qa, nt = (cu32(x) for x in (np.full(n, 536), np.arange(n) * 64, np.full(n, 64)))
        return lambda: hip.prefill_attention(L, pool, N, q, b, ta, p0, qa, nt, H, 599, 64, out)

    outs = [torch.empty(40 * 64 * H * D, device="cuda") for _ in range(2)]
    small, large = attend(2, outs[0]), attend(40, outs[1])
    for warm in (True, False):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            if warm:
                small()
            else:
                hip.append(L, pool, N, q[:0], q[:0], b[:0])
                hip.check(s)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        used = hip.usage()["used"]
        with torch.cuda.graph(g, stream=s):
            small()
        assert hip.usage()["used"] == used
        g.replay()
        torch.cuda.synchronize()
        ref = outs[0].clone()
        for _ in range(3):
            outs[0].zero_()
            with torch.cuda.stream(s):
                large()
            s.synchronize()
            g.replay()
            torch.cuda.synchronize()
            n = 2 * 64 * H * D
            assert torch.equal(outs[0][:n], ref[:n])
        assert attn_errors(outs[0][:n].cpu().numpy(), outs[1][:n].cpu().numpy())[1] <= REL_L2
        hip.check(s)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F16, Q8_0])
def test_captured_prefill_shares_no_workspace(hip, knobs, dtype):
    """A launch captured on a warmed stream is the unsplit form without images, bit for bit, and
    replays on another stream beside that stream's own split launches and a second graph
    captured there, none of them waiting for another."""
    from test_gpu_kernels import cf32, cu32, fill_items, layout, new_pool

    knobs("prefill_images", 1)
    r, H, G, D, n = rng(6), 16, 4, 128, 4
    L = layout(dtype, G, D)
    N = n * 38 + 3
    pool = new_pool(L, N, fill=2)
    blocks, table_at, _ = fill_items(hip, L, pool, N, [600] * n, r)
    b, ta = cu32(blocks), cu32(table_at)
    p0, qa, nt = (cu32(x) for x in (np.full(n, 536), np.arange(n) * 64, np.full(n, 64)))
    qs = [cf32(normal(r, (n * 64, H, D))) for _ in range(3)]
    outs = [torch.empty(n * 64 * H * D, device="cuda") for _ in range(3)]

    def attend(i):
        hip.prefill_attention(L, pool, N, qs[i], b, ta, p0, qa, nt, H, 599, 64, outs[i])

    knobs("prefill_images", 0)
    knobs("prefill_chunks", 1)
    plain = []
    for i in range(2):
        attend(i)
        plain.append(outs[i].clone())
    knobs("prefill_images", 1)
    knobs("prefill_chunks", 4)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        attend(2)
        split = outs[2].clone()
    s.synchronize()
    graphs = []
    for i in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            attend(i)
        graphs.append(g)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for _ in range(4):
        for o in outs:
            o.zero_()
        torch.cuda.synchronize()
        for g, t in zip(graphs, streams):
            with torch.cuda.stream(t):
                g.replay()
        with torch.cuda.stream(s):
            attend(2)
        torch.cuda.synchronize()
        assert torch.equal(outs[0], plain[0]) and torch.equal(outs[1], plain[1])
        assert torch.equal(outs[2], split)
    hip.check(s)


@pytest.mark.gpu
def test_workspace_grows_while_another_stream_is_captured(hip, knobs):
    """Split launches that allocate and replace their stream's workspace leave a capture that is
    under way on another stream whole."""
    from test_gpu_kernels import cf32, cu32, fill_items, layout, new_pool

    knobs("prefill_chunks", 4)
    r, H, G, D = rng(7), 16, 4, 128
    L = layout(F16, G, D)
    N = 40 * 38 + 3
    pool = new_pool(L, N, fill=2)
    blocks, table_at, _ = fill_items(hip, L, pool, N, [600] * 40, r)
    q, b, ta = cf32(normal(r, (40 * 64, H, D))), cu32(blocks), cu32(table_at)
    args = {n: [cu32(x) for x in (np.full(n, 536), np.arange(n) * 64, np.full(n, 64))] for n in (2, 40)}
    outs = [torch.zeros(40 * 64 * H * D, device="cuda") for _ in range(3)]

    def attend(n, out):
        p0, qa, nt = args[n]
        hip.prefill_attention(L, pool, N, q, b, ta, p0, qa, nt, H, 599, 64, out)

    a, s = torch.cuda.Stream(), torch.cuda.Stream()
    for t in (a, s):  # the streams' state, without a workspace
        with torch.cuda.stream(t):
            hip.append(L, pool, N, q[:0], q[:0], b[:0])
        hip.check(t)
    torch.cuda.synchronize()
    used = hip.usage()["used"]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=a):
        attend(2, outs[0])
        with torch.cuda.stream(s):
            attend(2, outs[1])
            attend(40, outs[2])
        attend(2, outs[0])
    assert hip.usage()["used"] > used
    for _ in range(3):
        outs[0].zero_()
        g.replay()
        torch.cuda.synchronize()
        n = 2 * 64 * H * D
        for o in outs[:2]:
            assert attn_errors(o[:n].cpu().numpy(), outs[2][:n].cpu().numpy())[1] <= REL_L2
    hip.check(s)
    hip.check(a)
