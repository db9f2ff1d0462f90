"""Prompt attention over long spans (forward.hip, fw_attn_prompt_split_kernel:
f32 products as three f16 ones) at the edges of its rule (spans from 2048
positions), token blocks (32) and tiles (32 positions), with cached rows of
very different size, and with infinities and NaN, against the oracle; and
every token's attention against 64 bits where rows are zero, tiny, or much
smaller than rows beside them that the token does not see or weighs little.

Bar: 1e-5, as the decode tests: chunks of up to 16 tokens keep every matvec
in f32 (rope is left out, whose last bit shows at late positions). A longer
chunk rounds its matrices to f16 (5e-3, the prompt tests' bar).
"""
import numpy as np
import pytest

from test_gpu_attention import fill, views
from test_gpu_forward import CFG, build, rel_l2

pytestmark = pytest.mark.gpu

# an FFN wide enough for the partials of eight span splits at four heads: a chunk whose partials do not fit in the
# FFN's buffers runs the f32 kernel
BASE = dict(CFG, head_dim=256, intermediate=4608, max_ctx=2400, sliding_window=40, rope_full_partial=0.0,
            rope_slide_partial=0.0)


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


def one_layer(sm, ref, dev, heads=4, kvh=1, eps=1e-20, gain=1.0, zero=(), loud=(), inter=BASE["intermediate"]):
    """A full layer whose attention output reaches the next layer's input
    unmixed: its MLP adds nothing (a zero norm) and the embedding is faint,
    2^-18, or zero for tokens of `zero` (no query, key, value or residual) and
    of order 16 for those of `loud`. gain scales the normed input: queries,
    keys and values are of its order, or, where eps outweighs the squared
    embedding, of that of gain * 2^-18 / sqrt(eps). Returns the model, which
    captures that input at slot 1, and the same in f64."""
    import torch
    c = dict(BASE, heads=heads, kv_heads=kvh, eps=eps, layers=2, intermediate=inter)
    hid, hd = c["hidden"], c["head_dim"]
    qd, kvd = heads * hd, kvh * hd
    shapes = dict(qkv=(qd + 2 * kvd, hid), attn_gate=(heads, hid), out=(hid, qd), gate=(inter, hid), up=(inter, hid),
                  down=(hid, inter))
    data = {k: sm.synth_container(50 + i, *s) for i, (k, s) in enumerate(shapes.items())}
    W = {k: ref.decode(d).astype(np.float64) for k, d in data.items()}
    norm, none = torch.full((hid,), gain, device=dev), torch.zeros(hid, device=dev)
    mats = {k: sm.DeviceContainer(d, dev) for k, d in data.items()}
    layers = [dict(mats, in_norm=norm, post_norm=none, full=f) for f in (True, False)]
    blocks = sm.synth_q8_0(77, c["vocab"], hid).reshape(c["vocab"], hid // 32, 34)
    for at, d in ((slice(None), 2.0 ** -24), (list(zero), 0.0), (list(loud), 0.25)):
        blocks[at, :, :2] = np.array([d], np.float16).view(np.uint8)
    blocks = blocks.reshape(-1)
    embed = ref.q8_0_dequant(blocks, c["vocab"], hid).astype(np.float64)
    model = sm.Model(dict(c, x_dtype=sm.X_F32, dim=4, nc=4096, nstages=2, v3=1), layers,
                     torch.from_numpy(blocks).to(dev), norm)
    model.enable_capture([0, 1])

    def want(toks, pos=0, K=None, V=None):
        """The next layer's input of every token after the cached rows K, V
        [pos][kvd]; without rows, the queries."""
        h = embed[toks]
        x = gain * h / np.sqrt((h * h).mean(-1, keepdims=True) + float(np.float32(eps)))
        qkv = x @ W["qkv"].T
        gate = 1 / (1 + np.exp(-(x @ W["attn_gate"].T)))
        q = qkv[:, :qd].reshape(len(toks), heads, hd)
        if K is None:
            return q
        K, V = np.concatenate([K, qkv[:, qd:qd + kvd]]), np.concatenate([V, qkv[:, qd + kvd:]])
        out = np.empty((len(toks), heads, hd))
        for t in range(len(toks)):
            n = pos + t + 1
            for i in range(heads):
                at = slice(i * kvh // heads * hd, (i * kvh // heads + 1) * hd)
                s = K[:n, at] @ q[t, i] / np.sqrt(hd)
                w = np.exp(s - s.max())
                out[t, i] = gate[t, i] * (w @ V[:n, at]) / w.sum()
        return h + out.reshape(len(toks), qd) @ W["out"].T
    return model, c, want


def every_token(model, cfg, want, dev, toks, pos, K, V):
    """Each token's row of the next layer's input against the f64 one: the distances."""
    import torch
    for t, host in zip(views(model, dev, dict(cfg, layers=1))[0], (K, V)):
        t[:pos] = torch.from_numpy(host).to(dev)
        t[pos:] = float("nan")
    model.forward_batch(toks, pos)
    torch.cuda.synchronize()
    got, exact = model.captured(1)[pos:].cpu().numpy(), want(toks, pos, K.astype(np.float64), V.astype(np.float64))
    assert got.shape == exact.shape
    return [rel_l2(g, e) for g, e in zip(got, exact)]


def rows(rng, pos, exp, mean=0.0):
    return np.ldexp(mean + rng.standard_normal((pos, 256)), exp).astype(np.float32)


@pytest.mark.parametrize("vexp", [0, -5, -10])
@pytest.mark.parametrize("every", [False, True], ids=["first", "every-tile"])
def test_zero_value_rows(sm, ref, dev, vexp, every):
    """Four value rows that share a lane group are zero, once or in every
    tile: the rows beside them keep their bits."""
    model, cfg, want = one_layer(sm, ref, dev, gain=2.0 ** vexp)
    rng, pos = np.random.default_rng(1), 2070
    K, V = rows(rng, pos, -vexp), rows(rng, pos, vexp, 1.0)
    V[np.arange(pos) % (32 if every else 4096) < 4] = 0
    err = every_token(model, cfg, want, dev, list(range(9)), pos, K, V)
    assert max(err) <= 1e-5, err


@pytest.mark.parametrize("pos", [2070, 2046, 2079])
@pytest.mark.parametrize("vexp", [-6, -14, -18])
def test_hidden_rows_leave_no_trace(sm, ref, dev, vexp, pos):
    """The chunk's last token has values 2^6 .. 2^18 times the size of all
    others, the rows just before it have nearly all of the weight: the tokens
    before it, which do not see it, keep their bits."""
    model, cfg, want = one_layer(sm, ref, dev, eps=2.0 ** (-36 - 2 * vexp), loud=[100])
    rng, q = np.random.default_rng(2), want([5])[0].mean(0)
    K, V = rows(rng, pos, -7 - vexp), rows(rng, pos, vexp, 1.0)
    K[-14:] += 12 * 16 * q / (q * q).sum()
    err = every_token(model, cfg, want, dev, [5] * 7 + [100], pos, K, V)
    assert max(err[:-1]) <= 1e-5, err


@pytest.mark.parametrize("vexp,loud", [(-16, 1), (-26, 1), (-30, 0), (-90, 0), (-112, 0), (-114, 0)])
def test_tiny_values(sm, ref, dev, vexp, loud):
    """Cached values down to 2^-114, equal weights (no queries), beside zero
    rows of the chunk and, with loud, a last token's hidden row of order 1."""
    zero = list(range(6))
    model, cfg, want = one_layer(sm, ref, dev, zero=zero, loud=[100])
    rng, pos = np.random.default_rng(3), 2070
    K, V = rows(rng, pos, 0), rows(rng, pos, vexp, 1.0)
    err = every_token(model, cfg, want, dev, zero + [100] * loud, pos, K, V)
    assert max(err[:6]) <= 1e-5, err


@pytest.mark.parametrize("vexp", [-8, -16, -40])
def test_small_rows_with_the_weight(sm, ref, dev, vexp):
    """Four rows take nearly all of every token's weight and are 2^-8 .. 2^-40 of
    the rows beside them, whose weight is down to where both count."""
    model, cfg, want = one_layer(sm, ref, dev)
    toks, pos, rng = [100] * 6, 2070, np.random.default_rng(4)
    q = want([100])[0].mean(0)
    K, V = rows(rng, pos, -7), rows(rng, pos, 0, 1.0)
    K[64:68] += (-vexp * 0.7 + 8) * 16 * q / (q * q).sum()
    V[64:68] = np.ldexp(V[64:68], vexp)
    err = every_token(model, cfg, want, dev, toks, pos, K, V)
    assert max(err) <= 1e-5, err


@pytest.mark.parametrize("kexp", [20, 100, 109, 114])
def test_large_keys_and_small_queries(sm, ref, dev, kexp):
    """Scores of order 1 to 8 whose keys alone, times the query's scaled halves, pass f32's range."""
    model, cfg, want = one_layer(sm, ref, dev, gain=2.0 ** (3 - kexp))
    rng, pos = np.random.default_rng(5), 2070
    err = every_token(model, cfg, want, dev, list(range(9)), pos, rows(rng, pos, kexp), rows(rng, pos, 0, 1.0))
    assert max(err) <= 1e-5, err


@pytest.mark.parametrize("width,mean", [(0.5, 0.0), (6, 0.0), (12, 0.0), (12, 1.0)])
def test_no_further_from_64_bits_than_the_f32_kernel(sm, ref, dev, width, mean):
    """Chunks of 16 tokens through this kernel and, under an FFN too narrow
    for its partials, through the f32 one, over scores of deviation `width`
    (sharp ones show their last bits in the weights)."""
    pos, err = 2070, []
    for inter in (BASE["intermediate"], 512):
        model, cfg, want = one_layer(sm, ref, dev, inter=inter)
        total = 0.0
        for seed in range(6):
            rng = np.random.default_rng(seed)
            K, V = rows(rng, pos, 0) * np.float32(width / 0.47), rows(rng, pos, 0, mean)
            total += sum(every_token(model, cfg, want, dev, rng.integers(0, cfg["vocab"], 16).tolist(), pos, K, V))
        err.append(total)
    assert err[0] <= err[1], err
