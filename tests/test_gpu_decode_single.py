"""Short caches decode in one launch, one workgroup per query head
(decode_single_kernel): the edges of its rounds of rows (480 / 240 / 120 cached
keys at head_dim 64 / 128 / 256), empty caches, windows, the most heads it
takes, and the key count past which the split form takes over, against the
oracle; appended rows bitwise."""
import numpy as np
import pytest

import oracle as o
import spissa_amd as sa
from spissa_amd.device import plan_attention
from spissa_amd.synth import normal_f32, seed_for
from tests.helpers import assert_bitwise, rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-4


@pytest.mark.parametrize("hq,hkv,d,past,window,single", [
    (32, 8, 64, [0], 0, True),
    (32, 8, 64, [1, 15, 280, 281, 0, 17, 3, 120], 0, True),  # 256 heads: every CU one workgroup
    (32, 8, 64, [1, 15, 512, 481, 0, 17, 3, 120], 0, False),  # 67 MB fetched by the XCDs in all
    (32, 8, 64, [480, 481, 17, 0], 0, True),
    (64, 64, 64, [585, 480, 481, 1], 0, True),  # a KV head per query head: fetched once either way
    (32, 8, 64, [585], 0, True),
    (32, 8, 64, [586], 0, False),
    (32, 8, 64, [1] * 9, 0, False),      # 288 heads
    (24, 8, 128, [239, 240, 241], 0, True),
    (4, 1, 256, [146, 120, 121], 0, True),
    (4, 1, 256, [147], 0, False),
    (8, 4, 256, [900, 40], 100, True),   # only the window counts
    (3, 3, 128, [60], 7, True),
])
def test_fused_step(gpu, hq, hkv, d, past, window, single):
    import torch

    from spissa_amd.device import Session

    cfg = sa.KvAttentionConfig(1, hq, hkv, d, True, window)
    plan = plan_attention(cfg, past)
    assert (plan["splits"] == 1 and plan["heads_per_block"] == 1 and plan["workgroups"] == len(past) * hq) == single
    st = torch.cuda.Stream()
    s = Session(0, stream=st)
    w, base = hkv * d, 500000.0
    table = s.rope_table(0, d, base, max_positions=max(past) + 1)
    caches, refs = [], []
    r = lambda tag, n, b: normal_f32(seed_for(72, d, b, tag, n), n)
    for b, p in enumerate(past):
        c, rc = s.kv_cache(hkv, d, p + 1), o.KvCache(hkv, d, p + 1)
        if p:
            k, v = r("k", p * w, b), r("v", p * w, b)
            c.append(k.copy(), v.copy(), p)
            rc.append(k.copy(), v.copy(), p)
        caches.append(c)
        refs.append(rc)
    B = len(past)
    q, k, v = r("q", B * hq * d, 99), r("k", B * w, 98), r("v", B * w, 97)
    dq, dk, dv = (torch.from_numpy(t).cuda() for t in (q, k, v))
    out = torch.empty(B * hq * d, device="cuda")
    torch.cuda.synchronize()
    s.decode_step(table, dq, dk, dv, caches, cfg, out)
    s.sync()
    got = out.cpu().numpy().reshape(B, -1)
    for b, p in enumerate(past):
        qb, kb, vb = q.reshape(B, -1)[b].copy(), k.reshape(B, -1)[b].copy(), v.reshape(B, -1)[b].copy()
        o.apply_llama_rotary_inplace(qb, kb, hq, hkv, 1, d, d, base, p)
        ref = o.sdpa_with_cache(qb, kb, vb, refs[b], 1, hq, hkv, d, True, window)
        err = rel_err(got[b], ref)
        print(f"[single] {hq}/{hkv} x {d}, {p} keys, window {window}: {err:.1e}", flush=True)
        assert err <= TOL
        assert_bitwise(caches[b].keys()[p * w:], kb, "appended key")
        assert_bitwise(caches[b].values()[p * w:], vb, "appended value")


def test_a_step_past_the_limit_can_be_captured_after_one_below_it(gpu):
    """A call that takes one launch still prepares the partials' workspace: the
    next token's, the first that needs it, may be captured. And a first call in
    one launch can itself be captured."""
    import torch

    from spissa_amd.device import Session

    hq, hkv, d, past = 32, 8, 64, 585
    cfg = sa.KvAttentionConfig(1, hq, hkv, d, True)
    w = hkv * d
    r = lambda tag, n: normal_f32(seed_for(74, d, 0, tag, n), n)
    k, v = r("k", (past + 1) * w), r("v", (past + 1) * w)
    q, kc, vc = r("q", hq * d), r("k", w), r("v", w)

    def session(p):
        st = torch.cuda.Stream()
        s = Session(0, stream=st)
        c = s.kv_cache(hkv, d, past + 1)
        c.append(k[:p * w].copy(), v[:p * w].copy(), p)
        return s, st, c, [torch.from_numpy(t).cuda() for t in (q, kc, vc)], torch.zeros(hq * d, device="cuda")

    def replays(s, st, c, dev, out):
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            s.attention_decode_batch(*dev, [c], cfg, out)
        for _ in range(3):
            out.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            yield out.cpu().numpy()

    def reference(p):
        rc = o.KvCache(hkv, d, past + 1)
        rc.append(k[:p * w].copy(), v[:p * w].copy(), p)
        return o.sdpa_with_cache(q, kc, vc, rc, 1, hq, hkv, d, True, 0)

    s, st, c, dev, out = session(past)
    torch.cuda.synchronize()
    s.attention_decode_batch(*dev, [c], cfg, out)  # 585 keys: one launch
    s.sync()
    assert rel_err(out.cpu().numpy(), reference(past)) <= TOL
    c.append(k[past * w:].copy(), v[past * w:].copy(), 1)
    for got in replays(s, st, c, dev, out):  # 586: split
        assert rel_err(got, reference(past + 1)) <= TOL
    s.sync()

    s, st, c, dev, out = session(past)
    for got in replays(s, st, c, dev, out):  # the session's first call
        assert rel_err(got, reference(past)) <= TOL
    s.sync()
