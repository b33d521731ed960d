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
                                  (dict(EDGE, window_size=64), 300)])
def test_prompt_equals_short_passes(gpu, hd, kv, n):
    """A whole prompt in passes of up to 512 rows, cut where the window fills,
    leaves the cache and the next logits as passes of 8 rows do."""
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
