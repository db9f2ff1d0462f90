"""The split attention of decode tokens and verify blocks (forward.hip,
fw_attn_split_kernel) at the edges of its tiles (16 positions) and splits (64
per head: one tile each up to 1024 positions, several past that), for every
head size and group size, against the oracle over the same random cache.

Bar: 1e-5, as the decode tests (f32 arithmetic throughout; rope is left out
past the first positions, where the last bit of powf shows in the angles)."""
import numpy as np
import pytest

from test_gpu_forward import CFG, FULL, build, rel_l2

pytestmark = pytest.mark.gpu


class Rows:
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


def views(model, dev, cfg):
    import torch
    shape = (cfg["max_ctx"], cfg["kv_heads"] * cfg["head_dim"])
    return [[torch.as_tensor(Rows(p, shape), device=dev) for p in model.kv(li)] for li in range(cfg["layers"])]


def fill(model, oracle, dev, cfg, n, seed):
    import torch
    rng = np.random.default_rng(seed)
    for li, kv in enumerate(views(model, dev, cfg)):
        for t, host in zip(kv, (oracle.kv_k[li], oracle.kv_v[li])):
            host[:n] = rng.standard_normal((n, host.shape[1])).astype(np.float32)
            t[:n] = torch.from_numpy(host[:n]).to(dev)
            t[n:] = float("nan")     # rows not written yet


@pytest.mark.parametrize("hd,heads,kv_heads", [(64, 4, 2), (64, 3, 3), (128, 6, 2), (256, 4, 1), (256, 8, 4)])
@pytest.mark.parametrize("pos,window", [(0, 40), (14, 40), (15, 16), (1008, 512), (1023, 40), (1024, 700),
                                        (2111, 1500)])
def test_tile_and_split_edges(sm, ref, dev, hd, heads, kv_heads, pos, window):
    import torch
    cfg = dict(CFG, head_dim=hd, heads=heads, kv_heads=kv_heads, max_ctx=2144, sliding_window=window, layers=2)
    if pos > 100:
        cfg.update(rope_full_partial=0.0, rope_slide_partial=0.0)
    model, oracle = build(sm, ref, dev, "q8_0", sm.X_F32, cfg)
    fill(model, oracle, dev, cfg, pos, pos + hd)
    toks = [int(t) for t in np.random.default_rng(3).integers(0, cfg["vocab"], 9)]
    one = torch.zeros(cfg["vocab"], device=dev)
    model.forward(toks[0], pos, one)
    torch.cuda.synchronize()
    assert rel_l2(one.cpu().numpy(), oracle.forward(toks[0], pos)) <= 1e-5
    for n in (3, 8):
        out = torch.zeros(n, cfg["vocab"], device=dev)
        model.verify(toks[1:1 + n], pos + 1, out)
        torch.cuda.synchronize()
        for i in range(n):
            err = rel_l2(out[i].cpu().numpy(), oracle.forward(toks[1 + i], pos + 1 + i))
            assert err <= 1e-5, (n, i, err)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_hidden_rows_do_not_leak(sm, ref, dev, bad):
    """A cached row that only a block's first token still sees (the sliding
    window's start) holds NaN or infinity in the last, sliding layer: that
    token's logits are not finite, the others' are what they are without it."""
    import torch
    cfg = dict(CFG, head_dim=256, heads=4, kv_heads=1, max_ctx=256, sliding_window=40)
    assert not FULL[cfg["layers"] - 1]
    model, oracle = build(sm, ref, dev, "q8_0", sm.X_F32, cfg)
    pos = 100
    fill(model, oracle, dev, cfg, pos, 7)
    toks = list(range(1, 9))
    want, got = torch.zeros(8, cfg["vocab"], device=dev), torch.zeros(8, cfg["vocab"], device=dev)
    model.verify(toks, pos, want)
    views(model, dev, cfg)[-1][1][pos - 39, 5] = bad
    model.verify(toks, pos, got)
    torch.cuda.synchronize()
    assert not torch.isfinite(got[0]).any()
    assert rel_l2(got[1:].cpu().numpy(), want[1:].cpu().numpy()) <= 1e-5
