"""Prompt attention over long spans (forward.hip, fw_attn_prompt_split_kernel:
f32 products as three f16 ones) at the edges of its rule (spans from 2048
positions), token blocks (32) and tiles (32 positions), with cached rows of
very different size, and with infinities and NaN, against the oracle.

Bar: 1e-5, as the decode tests: chunks of up to 16 tokens keep every matvec
in f32 (rope is left out, whose last bit shows at late positions). A longer
chunk rounds its matrices to f16 (5e-3, the prompt tests' bar).
"""
import numpy as np
import pytest

from test_gpu_attention import fill, views
from test_gpu_forward import CFG, build, rel_l2

pytestmark = pytest.mark.gpu

BASE = dict(CFG, head_dim=256, max_ctx=2400, sliding_window=40, rope_full_partial=0.0, rope_slide_partial=0.0)


def run(model, oracle, dev, cfg, pos, n):
    import torch
    toks = [int(t) for t in np.random.default_rng(n).integers(0, cfg["vocab"], n)]
    out = torch.full((cfg["vocab"],), float("nan"), device=dev)
    model.forward_batch(toks, pos, out)
    torch.cuda.synchronize()
    for i, t in enumerate(toks):
        want = oracle.forward(t, pos + i)
    return out.cpu().numpy(), want


@pytest.mark.parametrize("heads,kvh", [(4, 1), (8, 2)])
@pytest.mark.parametrize("pos,n", [(2045, 3), (2032, 16), (2047, 9), (2100, 32), (2011, 70), (2301, 33)])
def test_span_block_and_tile_edges(sm, ref, dev, heads, kvh, pos, n):
    cfg = dict(BASE, heads=heads, kv_heads=kvh)
    model, oracle = build(sm, ref, dev, "q8_0", sm.X_F32, cfg)
    fill(model, oracle, dev, cfg, pos, pos)
    got, want = run(model, oracle, dev, cfg, pos, n)
    assert rel_l2(got, want) <= (1e-5 if n <= 16 else 5e-3)


@pytest.mark.parametrize("kexp,vexp", [(-60, 30), (20, -100), (4, 0)])
def test_rows_of_very_different_size(sm, ref, dev, kexp, vexp):
    """Every key and value scaled far from 1, then some rows by 2^-9 .. 2^6 of that."""
    import torch
    cfg = dict(BASE, heads=4, kv_heads=1)
    model, oracle = build(sm, ref, dev, "q8_0", sm.X_F32, cfg)
    pos, n = 2100, 7
    fill(model, oracle, dev, cfg, pos, 5)
    e = np.random.default_rng(6).integers(-9, 7, (pos, 1))
    for li, kv in enumerate(views(model, dev, cfg)):
        for t, host, x in zip(kv, (oracle.kv_k[li], oracle.kv_v[li]), (kexp, vexp)):
            host[:pos] = np.ldexp(host[:pos], np.minimum(e, 0) + x if x == kexp else e + x)
            t[:pos] = torch.from_numpy(host[:pos]).to(dev)
    got, want = run(model, oracle, dev, cfg, pos, n)
    assert rel_l2(got, want) <= 1e-5


@pytest.mark.parametrize("which,bad", [(1, float("nan")), (1, float("inf")), (0, float("nan")), (0, float("inf")),
                                       (0, -float("inf"))])
def test_infinities_and_nan(sm, ref, dev, which, bad):
    """One element of one cached row of the full layers: logits are finite
    exactly where the oracle's are, and equal there."""
    import torch
    cfg = dict(BASE, heads=4, kv_heads=1)
    model, oracle = build(sm, ref, dev, "q8_0", sm.X_F32, cfg)
    pos, n = 2060, 6
    fill(model, oracle, dev, cfg, pos, 8)
    for li, kv in enumerate(views(model, dev, cfg)):
        host = (oracle.kv_k, oracle.kv_v)[which][li]
        host[77, 3] = bad
        kv[which][77, 3] = bad
    with np.errstate(all="ignore"):
        got, want = run(model, oracle, dev, cfg, pos, n)
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    ok = np.isfinite(want)
    assert not ok.any() or rel_l2(got[ok], want[ok]) <= 1e-5


def test_reservations_grow(sm, ref, dev):
    """Chunks past a reservation replace the block buffers, the K-split slices
    with them: 17 tokens reserved and run, then 130, then 20 again."""
    cfg = dict(BASE, heads=4, kv_heads=1, max_ctx=256)
    model, oracle = build(sm, ref, dev, "q8_0", sm.X_F32, cfg)
    model.reserve(17)
    pos = 0
    for n in (17, 130, 20):
        got, want = run(model, oracle, dev, cfg, pos, n)
        assert rel_l2(got, want) <= 5e-3
        pos += n
