"""Attention of prompt passes (more than 8 rows of one sequence): the cache
and the next forward after one tall pass equal those after passes of at most
8 rows, which run the other attention kernels (pinned to the oracle), bit for
bit.  Heights and starts around the 32-row tile, the 64-entry sub-chunk and
the 256-entry chunk, passes that end at the last position before the window
is full and one past it, and sink sizes the prefix rule accepts and not."""
import numpy as np
import pytest

import pocketforge_amd as pf
from pocketforge_amd import weights as W

pytestmark = pytest.mark.gpu

CFG = {64: dict(n_layers=2, n_embd=1024, n_heads=16, head_dim=64, n_ff=512, n_vocab=1024, n_mtp=1),
       128: dict(n_layers=2, n_embd=2048, n_heads=16, head_dim=128, n_ff=512, n_vocab=1024, n_mtp=1)}
WIDE = dict(sink_size=4, window_size=2048, pool_block=16, max_context=2048)
EDGE = dict(sink_size=4, window_size=500, pool_block=6, max_context=1024)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("kv,start,rows", [
    (WIDE, 0, 9), (WIDE, 0, 97), (WIDE, 3, 128), (WIDE, 0, 256), (WIDE, 225, 97), (WIDE, 250, 256),
    (WIDE, 1030, 16), (WIDE, 1030, 17), (WIDE, 1030, 31), (WIDE, 1055, 33), (WIDE, 1279, 65),
    (EDGE, 400, 105), (EDGE, 400, 106), (dict(EDGE, sink_size=0), 0, 100), (dict(EDGE, sink_size=8), 1, 100),
    (dict(EDGE, sink_size=9), 0, 100), (dict(EDGE, max_context=128), 29, 100), (dict(EDGE, max_context=128), 30, 100)])
def test_tall_pass_equals_short_passes(gpu, hd, kv, start, rows):
    cfg = CFG[hd]
    m = pf.Model(gpu, cfg, W.make_weights(cfg, seed=5))
    tall, short = pf.Engine(m, **kv), pf.Engine(m, **kv)
    toks = W.prompt_ids(start + rows + 1, cfg["n_vocab"], seed=77)
    for i in range(0, start, 8):
        tall.prefill(toks[i:min(i + 8, start)])
    tall.prefill(toks[start:start + rows])
    for i in range(0, start + rows, 8):
        short.prefill(toks[i:min(i + 8, start + rows)])
    for head in range(cfg["n_heads"]):
        a, b = (e.kv_export(0, 1, head, start + rows + 64) for e in (tall, short))
        assert a[4] == b[4]
        for x, y in zip(a[:4], b[:4]):
            np.testing.assert_array_equal(x, y)
    (la, ha), (lb, hb) = (e.forward(toks[start + rows:]) for e in (tall, short))
    np.testing.assert_array_equal(ha, hb)
    np.testing.assert_array_equal(la, lb)
    tall.close()
    short.close()
    m.close()


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("kv,n", [(WIDE, 1100), (EDGE, 504), (EDGE, 505), (EDGE, 506), (EDGE, 900),
                                  (dict(EDGE, sink_size=9), 600), (dict(EDGE, max_context=520), 515),
                                  (dict(EDGE, window_size=64), 300), (dict(EDGE, window_size=512, max_context=1600), 1530),
                                  (dict(EDGE, window_size=300, max_context=1600), 1100),
                                  (dict(WIDE, window_size=700, pool_block=1), 1900)])
def test_prompt_equals_short_passes(gpu, hd, kv, n):
    """A whole prompt in passes as tall as the pass memory allows, in one or
    several attention groups, cut or not where the window fills, leaves the
    cache and the next logits as passes of 8 rows do."""
    cfg = CFG[hd]
    m = pf.Model(gpu, cfg, W.make_weights(cfg, seed=6))
    b, short = pf.BatchEngine(m, 1, **kv), pf.Engine(m, **kv)
    toks = W.prompt_ids(n + 1, cfg["n_vocab"], seed=78)
    b.prefill_seq(0, toks[:n])
    for i in range(0, n, 8):
        short.prefill(toks[i:min(i + 8, n)])
    for head in (0, cfg["n_heads"] - 1):
        x, y = (e.kv_export(0, 1, head, n + 64) for e in (b, short))
        assert x[4] == y[4]
        for p, q in zip(x[:4], y[:4]):
            np.testing.assert_array_equal(p, q)
    lb, hb = b.forward_batch([0], toks[None, n:])
    ls, hs = short.forward(toks[n:])
    np.testing.assert_array_equal(hb[0], hs)
    np.testing.assert_array_equal(lb[0], ls)
    b.close()
    short.close()
    m.close()


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("at,rows", [(40, 128), (63, 128), (95, 97), (130, 256), (300, 400)])
def test_overflowed_value_stays_out_of_earlier_rows(gpu, hd, at, rows):
    """A token whose values overflow (infinite V scale) leaves every row
    before it as it is without that token: layer 1's cache of those rows,
    which holds layer 0's attention, is the same bit for bit."""
    cfg = CFG[hd]
    w = W.make_weights(cfg, seed=9)
    big, usual = 7, 8
    # channel 4 is 0 in every table row but `big`'s, where the first norm takes
    # it to about 1e38, and the V matrix on to infinity
    fmt, codes, scales = w["emb"]
    codes = codes.copy()
    codes[:, 0, 2] = (codes[:, 0, 2] & 0xF0) | 8
    codes[big, 0, 2] |= 15
    w["emb"] = (fmt, codes, scales)
    w["attn_norm"] = w["attn_norm"].copy()
    w["attn_norm"][0, 4] = 5e37
    fmt, codes, scales = w["layers"][0]["wv"]
    w["layers"][0]["wv"] = (fmt, codes, (scales.view(np.float16) * np.float16(1024)).view(np.uint16))
    m = pf.Model(gpu, cfg, w)
    toks = W.prompt_ids(rows, cfg["n_vocab"], seed=79)
    toks[toks == big] = usual
    planes = []
    for t in (usual, big):
        e = pf.BatchEngine(m, 1, **WIDE)
        toks[at] = t
        e.prefill_seq(0, toks)
        planes.append([[e.kv_export(0, layer, head, rows + 64)[:4] for head in (0, cfg["n_heads"] - 1)] for layer in (0, 1)])
        e.close()
    m.close()
    for head in range(2):
        assert np.isfinite(planes[0][1][head][3]).all() and not np.isfinite(planes[1][0][head][3][at])
        for x, y in zip(planes[0][1][head], planes[1][1][head]):
            np.testing.assert_array_equal(x[:at], y[:at])


def _engine_bytes(cfg, kv, n_seq):
    """An engine with 256 rows (or a verify pass's) of every pass buffer and of
    ring slack: what the budget of a program is laid out for."""
    L, D, F, V, H, hd = (cfg[k] for k in ("n_layers", "n_embd", "n_ff", "n_vocab", "n_heads", "head_dim"))
    R = cfg["n_mtp"] + 1
    window = min(kv["window_size"], kv["max_context"])
    pool_cap = max(0, kv["max_context"] - kv["sink_size"] - window) // kv["pool_block"] + 1
    rows = max(256, -(-R * n_seq // 32) * 32)
    chunks = (8 + pool_cap + window + 1 + 255) // 256
    cache = n_seq * L * H * (8 + window + kv["pool_block"] + 256 + pool_cap) * (2 * hd + 8)
    rope = (kv["max_context"] + 2 * rows) * hd * 4
    passes = rows * (4 * (4 * D + F) + max(D, F) + 16 + 4 * H * (2 * chunks + 8) + 4 * D * (chunks + 1))
    outputs = 4 * (max(8, n_seq) + max(8, R * n_seq)) * (V + D)
    heads = 4 * (max(n_seq, R - 1) * D + n_seq * D + (R - 1) * V + n_seq * V)
    words = 8 * (8 * 3 * D + 8 * (2 * D + F) + H * (2 * chunks + 8 + (chunks + 1) * hd))
    return cache + rope + passes + outputs + heads + words + 4 * 8 * 2 * F // 32 + 65536   # + descriptors


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("kv,n_seq", [(dict(EDGE, window_size=64), 1), (EDGE, 1), (WIDE, 1), (dict(WIDE, max_context=700), 3),
                                      (dict(EDGE, window_size=64), 64), (EDGE, 60)])
def test_memory_of_an_engine(gpu, hd, kv, n_seq):
    """Taller prompt passes take no memory that 256 rows would not, so a limit
    (pf_engine_set_max_memory) stops generation no earlier for them, and they
    move no bound on positions or pass heights."""
    cfg = CFG[hd]
    m = pf.Model(gpu, cfg, W.make_weights(cfg, seed=5))
    before = gpu.device_bytes
    e = pf.BatchEngine(m, n_seq, **kv)
    assert gpu.device_bytes - before <= _engine_bytes(cfg, kv, n_seq)
    rows = max(256, -(-2 * n_seq // 32) * 32)
    toks = W.prompt_ids(kv["max_context"] + 2 * rows + 1, cfg["n_vocab"], seed=80)
    with pytest.raises(pf.PFError):
        e.prefill_seq(n_seq - 1, toks)
    f = pf.lib().pf_batch_forward
    row = np.ascontiguousarray(toks[:rows + 1])
    seq = np.array([n_seq - 1], np.uint32)
    assert f(e.h, pf.P(seq, pf.u32p), 1, rows + 1, pf.P(row, pf.i32p), None, None) != 0
    e.close()
    m.close()


@pytest.mark.parametrize("heads,hd", [(4, 64), (12, 64), (4, 128), (12, 128)])
@pytest.mark.parametrize("n", [200, 256, 600])
def test_prompt_of_another_sequence(gpu, heads, hd, n):
    """Heads x chunks that do not fill the XCDs (the last launches of a row
    tile return at once) and a sequence other than the first."""
    cfg = dict(n_layers=2, n_embd=heads * hd, n_heads=heads, head_dim=hd, n_ff=512, n_vocab=1024, n_mtp=1)
    m = pf.Model(gpu, cfg, W.make_weights(cfg, seed=7))
    b, short = pf.BatchEngine(m, 3, **WIDE), pf.Engine(m, **WIDE)
    toks = [W.prompt_ids(n + 1, cfg["n_vocab"], seed=81 + s) for s in range(3)]
    for s in (1, 0, 2):
        b.prefill_seq(s, toks[s][:n])
    for s in range(3):
        short.reset()
        for i in range(0, n, 8):
            short.prefill(toks[s][i:min(i + 8, n)])
        for head in range(heads):
            x, y = b.kv_export(s, 1, head, n + 64), short.kv_export(0, 1, head, n + 64)
            assert x[4] == y[4]
            for p, q in zip(x[:4], y[:4]):
                np.testing.assert_array_equal(p, q)
        lb, hb = b.forward_batch([s], toks[s][None, n:])
        ls, hs = short.forward(toks[s][n:])
        np.testing.assert_array_equal(hb[0], hs)
        np.testing.assert_array_equal(lb[0], ls)
    b.close()
    short.close()
    m.close()


def test_long_batched_pass_of_one_sequence(gpu):
    """320 rows of one sequence past its window in one call (more than the
    ring's slack: two passes) equal short passes."""
    cfg = dict(CFG[64], n_vocab=512, n_mtp=4)
    kv = dict(sink_size=4, window_size=400, pool_block=6, max_context=1600)
    m = pf.Model(gpu, cfg, W.make_weights(cfg, seed=8))
    b, short = pf.BatchEngine(m, 64, **kv), pf.Engine(m, **kv)   # verify passes of 320 rows
    n, rows = 900, 320
    toks = W.prompt_ids(n + rows + 1, cfg["n_vocab"], seed=90)
    b.prefill_seq(5, toks[:n])
    logits, hidden = b.forward_batch([5], toks[None, n:n + rows])
    for i in range(0, n, 8):
        short.prefill(toks[i:min(i + 8, n)])
    for i in range(n, n + rows, 8):
        ls, hs = short.forward(toks[i:i + 8])
        np.testing.assert_array_equal(hidden[0, i - n:i - n + 8], hs)
        np.testing.assert_array_equal(logits[0, i - n:i - n + 8], ls)
    b.close()
    short.close()
    m.close()
