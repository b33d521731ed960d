"""Kernel-level parity of the gfx950 path against the oracle (bit-exact)."""
import ctypes as C
import os

import os
import subprocess

import numpy as np
import pytest

import oracle as O
import pocketforge_amd as pf
from golden_cfg import KV_CFGS

pytestmark = pytest.mark.gpu

G = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


_CTX = []


def _t(a):
    return pf.DeviceArray.from_numpy(_CTX[0], a)


@pytest.fixture(autouse=True)
def _ctx(gpu):
    _CTX[:] = [gpu]
    yield


def test_quantize_activation_rows(gpu):
    rng = np.random.default_rng(0)
    x = (rng.standard_normal((6, 2048)) * 0.9).astype(np.float32)
    x[1] = 0.0
    x[2, :] = np.arange(2048, dtype=np.float32) / 16.0 - 64.0    # exact .5 ties after scaling
    q, s = gpu.quantize_activation_rows(_t(x))
    q, s = q.numpy(), s.numpy()
    for m in range(6):
        q2, s2 = O.quantize_activation_row(x[m])
        np.testing.assert_array_equal(q[m], q2)
        assert s[m] == np.float32(s2)


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (3, 33, 15), (1, 40, 16), (2, 31, 31), (33, 32, 33), (5, 77, 0),
                                   (64, 65, 255), (31, 1000, 1100), (129, 4100, 47), (300, 4097, 130), (1, 3, 5),
                                   (2, 3, 8), (40, 70, 4), (33, 65, 12), (5, 129, 17), (65, 33, 28),
                                   (520, 4100, 100), (4100, 520, 5)])
def test_matmul_i8_ragged(gpu, M, N, K):
    """The MFMA int8 matmul at tile, step and row-tail edges (matrices of fewer
    than 16 bytes among them), K over a workgroup's waves and a tile per wave:
    integer sums equal, the scaled outputs bit for bit."""
    rng = np.random.default_rng(M * 1000 + K)
    A = rng.integers(-128, 128, (M, K), dtype=np.int8)
    B = rng.integers(-128, 128, (N, K), dtype=np.int8)
    pad = lambda a: a if a.size else np.zeros(1, a.dtype)   # a buffer to point at
    C = pf.DeviceArray.from_numpy(gpu, np.full((M, N), 7, np.int32))
    a, b = _t(pad(A)), _t(pad(B))
    gpu.check(pf.lib().pf_matmul_int8(gpu.h, a.ptr, b.ptr, C.ptr, M, N, K), "pf_matmul_int8")
    gpu.synchronize()
    np.testing.assert_array_equal(C.numpy(), A.astype(np.int32) @ B.astype(np.int32).T)
    if K == 0:
        return
    Af = (rng.standard_normal((M, K)) * 0.5).astype(np.float32)
    ws = (rng.random(N) * 0.02 + 0.001).astype(np.float32)
    for act in (None, (np.abs(Af).max(1) / 120.0).astype(np.float32)):
        ref = np.zeros((M, N), np.float32)
        O.lib().orc_matmul_quantized(O.ptr(Af, O.f32p), O.ptr(B, O.i8p), O.ptr(ref, O.f32p), M, N, K,
                                     O.ptr(ws, O.f32p), O.ptr(act, O.f32p) if act is not None else None)
        got = gpu.matmul_quantized(_t(Af), _t(B), _t(ws), _t(act) if act is not None else None).numpy()
        np.testing.assert_array_equal(got, ref)


def test_matmul_int8_beyond_one_launch(gpu):
    """More columns than one grid's threads cover (a tile per wave needs 2
    threads per column, K over the waves 16)."""
    N = (1 << 28) + 70
    B = np.resize(np.arange(-128, 123, dtype=np.int8), N)
    b, a, c = (pf.DeviceArray.from_numpy(gpu, x) for x in (B, np.array([3], np.int8), np.zeros(N, np.int32)))
    gpu.check(pf.lib().pf_matmul_int8(gpu.h, a.ptr, b.ptr, c.ptr, 1, N, 1), "pf_matmul_int8")
    gpu.synchronize()
    assert (c.numpy() == np.multiply(B, 3, dtype=np.int32)).all()
    for x in (a, b, c):
        x.free()


@pytest.mark.parametrize("where", ["B", "act_scales", "A"])
def test_matmul_quantized_over_its_inputs(gpu, where):
    """Outputs that take the place of an input the call still reads."""
    M, N, K = 200, 1000, 300
    rng = np.random.default_rng(4)
    A = (rng.standard_normal((M, K)) * 0.5).astype(np.float32)
    B = rng.integers(-127, 128, (N, K), dtype=np.int8)
    ws = (rng.random(N) * 0.02 + 0.001).astype(np.float32)
    act = (np.abs(A).max(1) / 120.0).astype(np.float32)
    ref = np.zeros((M, N), np.float32)
    O.lib().orc_matmul_quantized(O.ptr(A, O.f32p), O.ptr(B, O.i8p), O.ptr(ref, O.f32p), M, N, K, O.ptr(ws, O.f32p),
                                 O.ptr(act, O.f32p))
    a, b, w, s = _t(A), _t(B), _t(ws), _t(act)
    host = np.zeros(M * N, np.float32)
    src = {"B": B, "act_scales": act, "A": A}[where].reshape(-1).view(np.uint8)
    host.view(np.uint8)[: src.size] = src
    C = pf.DeviceArray.from_numpy(gpu, host)
    ptr = {"A": a.ptr, "B": b.ptr, "act_scales": s.ptr, where: C.ptr}
    gpu.check(pf.lib().pf_matmul_quantized(gpu.h, ptr["A"], ptr["B"], C.ptr, M, N, K, w.ptr, ptr["act_scales"]),
              "pf_matmul_quantized")
    gpu.synchronize()
    np.testing.assert_array_equal(C.numpy().reshape(M, N), ref)


def test_matmul_int8_and_quantized(gpu):
    rng = np.random.default_rng(1)
    M, N, K = 5, 77, 300
    A = rng.integers(-127, 128, (M, K), dtype=np.int8)
    B = rng.integers(-8, 8, (N, K), dtype=np.int8)
    Cm = gpu.matmul_int8(_t(A), _t(B)).numpy()
    np.testing.assert_array_equal(Cm, A.astype(np.int32) @ B.astype(np.int32).T)
    Af = (rng.standard_normal((M, K)) * 0.5).astype(np.float32)
    ws = (rng.random(N) * 0.02 + 0.001).astype(np.float32)
    asc = (rng.random(M) * 0.01 + 0.001).astype(np.float32)
    L = O.lib()
    for act in (None, asc):
        ref = np.zeros((M, N), np.float32)
        L.orc_matmul_quantized(O.ptr(Af, O.f32p), O.ptr(B, O.i8p), O.ptr(ref, O.f32p), M, N, K,
                               O.ptr(ws, O.f32p), O.ptr(act, O.f32p) if act is not None else None)
        got = gpu.matmul_quantized(_t(Af), _t(B), _t(ws), _t(act) if act is not None else None).numpy()
        np.testing.assert_array_equal(got, ref)


def test_matmul_reference_golden(gpu):
    K = dict(np.load(os.path.join(G, "ref_kernels.npz")))
    got = gpu.matmul_int8(_t(K["mm_A"]), _t(K["mm_B"])).numpy()
    np.testing.assert_array_equal(got, K["mm_C_fma"])
    got = gpu.matmul_quantized(_t(K["mq_A"]), _t(K["mm_B"]), _t(K["mq_ws"])).numpy()
    np.testing.assert_array_equal(got, K["mq_C_fma"])
    got = gpu.matmul_quantized(_t(K["mq_A"]), _t(K["mm_B"]), _t(K["mq_ws"]), _t(K["mq_as"])).numpy()
    np.testing.assert_array_equal(got, K["mq_Cas_fma"])


@pytest.mark.parametrize("fmt", [pf.FMT_Q4, pf.FMT_Q2, pf.FMT_Q15, pf.FMT_Q8])
@pytest.mark.parametrize("shape", [(128, 512), (320, 2048), (64, 1792)])
def test_gemv_int8_block(gpu, fmt, shape):
    N, K = shape
    codes, scales = pf.gen_matrix(99, fmt * 7 + N, 0.02, N, K, fmt)
    W = gpu.upload_matrix(fmt, codes, scales)
    rng = np.random.default_rng(N + K)
    for M in (1, 5, 8):
        x = (rng.standard_normal((M, K)) * 0.5).astype(np.float32)
        y = gpu.gemv_q(W, _t(x)).numpy()
        for m in range(M):
            a8, s = O.quantize_activation_row(x[m])
            ref = O.gemv_i8(fmt, codes, scales, a8, s)
            np.testing.assert_array_equal(y[m], ref, err_msg=f"fmt {fmt} M {M} row {m}")
    W.close()


@pytest.mark.parametrize("fmt", [pf.FMT_Q4, pf.FMT_Q8])
@pytest.mark.parametrize("N,K", [(64, 256), (4032, 512), (4160, 768), (8192, 1024), (16384, 2048)])
def test_gemv_f32_row_counts(gpu, N, K, fmt):
    """1 to 8 activation rows (one slice of up to 6, else slices of 4) over
    matrices on either side of the rows-per-wave thresholds."""
    codes, scales = pf.gen_matrix(8, N, 0.02, N, K, fmt)
    W = gpu.upload_matrix(fmt, codes, scales, rowmajor=True)
    h = np.random.default_rng(N + K).standard_normal((8, K)).astype(np.float32)
    ref = [O.gemv_f32(fmt, codes, scales, x) for x in h]
    for M in range(1, 9):
        y = gpu.gemv_f32(W, _t(h[:M])).numpy()
        for m in range(M):
            np.testing.assert_array_equal(y[m], ref[m], err_msg=f"{M} rows, row {m}")
    W.close()


def test_gemv_rejects_out_of_range_scales(gpu):
    codes, scales = pf.gen_matrix(5, 1, 0.02, 64, 256, pf.FMT_Q4)
    scales = scales.copy()
    scales[3, 0] = np.float16(1e-7).view(np.uint16)     # 2^-23 next to ~2^-7 scales
    scales[3, 1] = np.float16(1000.0).view(np.uint16)
    with pytest.raises(pf.PFError, match="binades"):
        gpu.upload_matrix(pf.FMT_Q4, codes, scales)
    codes, scales = pf.gen_matrix(5, 1, 0.02, 64, 256, pf.FMT_Q15)
    codes = codes.copy()
    codes[0, 0, 0] |= 3
    with pytest.raises(pf.PFError, match="code 3"):
        gpu.upload_matrix(pf.FMT_Q15, codes, scales)


@pytest.mark.parametrize("fmt", [pf.FMT_Q4, pf.FMT_Q8])
@pytest.mark.parametrize("K", [256, 768, 2048])
def test_gemv_f32(gpu, K, fmt):
    N = 640
    codes, scales = pf.gen_matrix(7, K, 0.02, N, K, fmt)
    W = gpu.upload_matrix(fmt, codes, scales, rowmajor=True)
    rng = np.random.default_rng(K)
    for M in (1, 5):
        h = (rng.standard_normal((M, K))).astype(np.float32)
        y = gpu.gemv_f32(W, _t(h)).numpy()
        for m in range(M):
            np.testing.assert_array_equal(y[m], O.gemv_f32(fmt, codes, scales, h[m]))
    W.close()


@pytest.mark.parametrize("key", sorted(KV_CFGS))
def test_kv_cache_api(gpu, key):
    """KVCache store / attention_scores / attention_weighted_sum on the GPU
    against the oracle and the reference's own outputs."""
    KV = dict(np.load(os.path.join(G, "ref_kv.npz")))
    Ln, H, hd, sink, win, pool, maxc, n = KV_CFGS[key]
    kv = pf.KVCache(gpu, Ln, H, hd, sink, win, pool, maxc)
    L = O.lib()
    ok = L.orc_kv_create(Ln, H, hd, sink, win, pool, maxc)
    keys, vals, qs = KV[f"{key}_keys"], KV[f"{key}_vals"], KV[f"{key}_qs"]
    stored = 0
    for c in KV[f"{key}_ckpt"]:
        while stored < c:
            for l in range(Ln):
                for h in range(H):
                    kv.store(l, h, stored, keys[stored, l, h], vals[stored, l, h])
                    L.orc_kv_store(ok, l, h, stored, O.ptr(keys[stored, l, h], O.f32p),
                                   O.ptr(vals[stored, l, h], O.f32p))
            stored += 1
        assert kv.size() == KV[f"{key}_c{c}_size"]
        for l in range(Ln):
            for h in range(H):
                for qi in range(8):
                    sc = kv.attention_scores(l, h, qs[qi])
                    assert len(sc) == KV[f"{key}_c{c}_count"][l, h]
                    np.testing.assert_array_equal(sc, KV[f"{key}_c{c}_scores_fma"][l, h, qi, :len(sc)])
                    p = np.exp(sc - sc.max()).astype(np.float32)
                    p = (p / p.sum()).astype(np.float32)
                    ws = kv.attention_weighted_sum(l, h, p)
                    ref = np.zeros(hd, np.float32)
                    L.orc_kv_attention_weighted_sum(ok, l, h, O.ptr(p, O.f32p), O.ptr(ref, O.f32p), len(p))
                    np.testing.assert_array_equal(ws, ref)
                    np.testing.assert_allclose(ws, KV[f"{key}_c{c}_wsum_fma"][l, h, qi], rtol=1e-5, atol=1e-6)
    kv.clear()
    assert kv.size() == 0
    assert len(kv.attention_scores(0, 0, qs[0])) == 0
    L.orc_kv_destroy(ok)
    kv.close()


SAMPLERS = {
    "greedy": pf.Sampling(0.8, 0.95, 40, 1),
    "temp0": pf.Sampling(0.0, 0.95, 40, 0),
    "top_p": pf.Sampling(0.8, 0.95, 40, 0),
    "top_k": pf.Sampling(0.8, 1.0, 40, 0),
    "temperature": pf.Sampling(1.3, 1.0, 0, 0),
}


@pytest.fixture(scope="module")
def engine_v16k(gpu):
    """A one-layer model with the benchmark vocabulary (16384), for the
    sampler at the size where its radix sort holds 16 keys per thread."""
    from pocketforge_amd import weights as W
    cfg = dict(n_layers=1, n_embd=256, n_heads=4, head_dim=64, n_ff=512, n_vocab=16384, n_mtp=4)
    m = pf.Model(gpu, cfg, W.make_weights(cfg, seed=1234))
    e = pf.Engine(m, sink_size=4, window_size=64, pool_block=6, max_context=256)
    yield e
    e.close()
    m.close()


@pytest.mark.parametrize("name", sorted(SAMPLERS))
@pytest.mark.parametrize("V", [1024, 16384])
def test_sampler(gpu, tiny_engine, engine_v16k, name, V):
    eng = tiny_engine if V == 1024 else engine_v16k
    assert eng.cfg["n_vocab"] == V
    cfg = SAMPLERS[name]
    ocfg = O.Sampling(cfg.temperature, cfg.top_p, cfg.top_k, cfg.greedy)
    rng = np.random.default_rng(V)
    for trial in range(12):
        logits = (rng.standard_normal(V) * (0.5 + trial)).astype(np.float32)
        if trial == 3:
            logits[::7] = logits.max()           # ties at the maximum
        draw = trial * 3
        t, d = eng.sample(logits, cfg, 7, draw)
        t2, d2 = O.sample(logits, ocfg, 7, draw)
        assert (t, d) == (t2, d2), (name, trial)


def test_dot_softmax_rmsnorm_argmax(gpu):
    """matmul_neon.hpp helpers on the device against the oracle's canonical
    orders (bit-exact), the reference's known answers
    (tests/test_matmul.cpp:103-153) and closed forms."""
    L = O.lib()
    rng = np.random.default_rng(5)
    for n in (1, 6, 255, 256, 300, 2048, 5000):
        a = rng.standard_normal(n).astype(np.float32)
        b = rng.standard_normal(n).astype(np.float32)
        assert np.float32(gpu.dot_product(_t(a), _t(b))) == np.float32(L.orc_dot_canon(O.ptr(a, O.f32p),
                                                                                         O.ptr(b, O.f32p), n))
        v = (a * 3).astype(np.float32)
        dv = _t(v)
        gpu.softmax(dv)
        ref = v.copy()
        L.orc_softmax(O.ptr(ref, O.f32p), n)
        np.testing.assert_array_equal(dv.numpy(), ref)
        w = rng.standard_normal(n).astype(np.float32)
        got = gpu.rmsnorm(_t(a), _t(w)).numpy()
        ref = np.zeros(n, np.float32)
        L.orc_rmsnorm(O.ptr(ref, O.f32p), O.ptr(a, O.f32p), O.ptr(w, O.f32p), n)
        np.testing.assert_array_equal(got, ref)
        x = a.copy()
        x[n // 2] = x.max() + 1.0
        if n > 3:
            x[n // 3] = x[n // 2]                       # tie: the first index wins
        assert gpu.argmax(_t(x)) == int(np.argmax(x))
    # reference known answers
    assert gpu.dot_product(_t(np.arange(1, 7, dtype=np.float32)), _t(np.arange(6, 0, -1, dtype=np.float32))) == 56.0
    sm = _t(np.array([2.0, 1.0, 0.1, 0.5, 3.0], np.float32))
    gpu.softmax(sm)
    s = sm.numpy()
    assert abs(s.sum() - 1.0) < 1e-3 and s[4] > s[0] > s[1] > s[3] > s[2]
    rn = gpu.rmsnorm(_t(np.array([1, 2, 3, 4], np.float32)), _t(np.array([0.5, 1, 1.5, 2], np.float32))).numpy()
    assert abs(rn[0] - 0.5 / np.sqrt(7.5)) < 0.01 and abs(rn[3] - 8 / np.sqrt(7.5)) < 0.01
    assert gpu.argmax(_t(np.array([-1.0, 3.0, 0.5, -0.2, 2.0], np.float32))) == 1


@pytest.mark.parametrize("with_table", [True, False])
def test_mtp_heads_standalone(gpu, with_table):
    """MTPHeads::forward outside an engine: 4 chained heads, fp32 tied table
    or the placeholder logits, bit-exact against the oracle."""
    d, V, H = 256, 1024, 4
    heads = []
    m = pf.MTPHeads(gpu, H, d, V)
    for k in range(H):
        trip = []
        for w in range(3):
            codes, scales = pf.gen_matrix(77, 100 + 3 * k + w, 0.02, d, d, pf.FMT_Q4)
            m.set_head(k, w, codes, scales)
            trip.append((O.Q4, codes, scales))
        heads.append(trip)
    rng = np.random.default_rng(3)
    table = (rng.standard_normal((V, d)) * 0.02).astype(np.float32) if with_table else None
    m.set_table(table)
    hidden = rng.standard_normal(d).astype(np.float32)
    got = m.forward(hidden)
    ref = O.mtp_heads_forward(heads, d, V, table, hidden)
    np.testing.assert_array_equal(got, ref)
    if not with_table:
        v = np.arange(V, dtype=np.uint64)
        np.testing.assert_array_equal(got[2], ((v * np.uint64(2654435761) + np.uint64(2)) % np.uint64(V))
                                      .astype(np.float32) / np.float32(V))
    assert m.memory_usage() > 0
    m.close()


@pytest.mark.parametrize("fmt", [pf.FMT_Q4, pf.FMT_Q2, pf.FMT_Q15, pf.FMT_Q8])
@pytest.mark.parametrize("N,K", [(64, 256), (64, 3840), (128, 5632), (64, 8192)])
def test_gemv_rows_held(gpu, fmt, N, K):
    """pf_gemv_q at every row count a launch holds (1, up to 5, up to 8) and
    one to four chunks per wave."""
    codes, scales = pf.gen_matrix(96, fmt * 17 + K, 0.02, N, K, fmt)
    W = gpu.upload_matrix(fmt, codes, scales)
    x = (np.random.default_rng(K).standard_normal((8, K)) * 0.5).astype(np.float32)
    ref = []
    for row in x:
        a8, s = O.quantize_activation_row(row)
        ref.append(O.gemv_i8(fmt, codes, scales, a8, s))
    for M in (1, 2, 4, 5, 6, 8):
        y = gpu.gemv_q(W, _t(x[:M])).numpy()
        for m in range(M):
            np.testing.assert_array_equal(y[m], ref[m], err_msg=f"{M} rows, row {m}")
    W.close()


@pytest.mark.parametrize("heads,d,V", [(1, 256, 1024), (2, 768, 515), (3, 512, 2049), (5, 2048, 777), (6, 256, 64)])
def test_mtp_heads_counts(gpu, heads, d, V):
    """Every slice height of the dense table pass (four heads, then the rest)
    and vocabularies that do not fill its waves, bit-exact."""
    m = pf.MTPHeads(gpu, heads, d, V)
    ws = []
    for k in range(heads):
        trip = []
        for w in range(3):
            codes, scales = pf.gen_matrix(78, 100 + 3 * k + w, 0.02, d, d, pf.FMT_Q4)
            m.set_head(k, w, codes, scales)
            trip.append((O.Q4, codes, scales))
        ws.append(trip)
    rng = np.random.default_rng(heads + d)
    table = (rng.standard_normal((V, d)) * 0.02).astype(np.float32)
    m.set_table(table)
    hidden = rng.standard_normal(d).astype(np.float32)
    np.testing.assert_array_equal(m.forward(hidden), O.mtp_heads_forward(ws, d, V, table, hidden))
    m.close()


@pytest.mark.parametrize("fmt", [pf.FMT_Q4, pf.FMT_Q2, pf.FMT_Q15, pf.FMT_Q8])
@pytest.mark.parametrize("M,N,K", [(9, 64, 256), (33, 2112, 768), (320, 4096, 512), (257, 4160, 256), (9, 64, 1024),
                                   (33, 2112, 1280), (161, 128, 1024), (16, 192, 8192)])
def test_gemm_splits(gpu, fmt, M, N, K):
    """Both K splits of the GEMM (eight and four waves) and both row
    quantizations (256 and 1024 threads), few and uneven steps per wave, a last
    row tile of one row and groups that do not fill the XCDs."""
    codes, scales = pf.gen_matrix(97, fmt * 13 + N, 0.02, N, K, fmt)
    W = gpu.upload_matrix(fmt, codes, scales)
    x = (np.random.default_rng(M + K).standard_normal((M, K)) * 0.5).astype(np.float32)
    y = gpu.gemv_q(W, _t(x)).numpy()
    for m in sorted({0, 8, M // 2, M - 2, M - 1}):
        a8, s = O.quantize_activation_row(x[m])
        np.testing.assert_array_equal(y[m], O.gemv_i8(fmt, codes, scales, a8, s), err_msg=f"row {m}")
    W.close()


@pytest.mark.parametrize("fmt", [pf.FMT_Q4, pf.FMT_Q2, pf.FMT_Q15, pf.FMT_Q8])
@pytest.mark.parametrize("M,N", [(33, 64), (512, 2112)])
def test_gemm_exact_at_its_limits(gpu, fmt, M, N):
    """The GEMM's integer sums at the limits the upload admits, for both K
    splits: 8192 columns, block scales over exactly 15 binades from subnormal
    on (negative and zero ones among them), the codes of largest magnitude and
    activations at their row's maximum: sums of up to 0.987 x 2^53 (Q4, Q8)."""
    K = 8192
    nb = K // 32
    rng = np.random.default_rng(fmt * 100 + M)
    e = rng.integers(0, 17, (N, nb))                      # biased exponents 0 (subnormal) .. 16
    scales = (e << 10 | rng.integers(0, 1024, (N, nb)) | rng.integers(0, 2, (N, nb)) << 15).astype(np.uint16)
    scales[rng.random((N, nb)) < 0.05] = 0
    width, low, top = {pf.FMT_Q4: (16, 0x00, 0xFF), pf.FMT_Q2: (8, 0x00, 0xFF), pf.FMT_Q15: (8, 0x00, 0xAA),
                       pf.FMT_Q8: (32, 0x80, 0x7F)}[fmt]
    codes = np.where(rng.random((N, nb, width)) < 0.5, low, top).astype(np.uint8)
    x = np.where(rng.random((M, K)) < 0.5, -1.0, 1.0).astype(np.float32)
    scales[:4] = 16 << 10 | 1023                          # every term of one sign, as large as any
    scales[:4, 0] = 1                                     # and the smallest scale: a unit of 2^-24
    scales[2:4, 1:] |= 0x8000
    codes[:4] = low
    x[0], x[M - 1] = 1.0, -1.0
    W = gpu.upload_matrix(fmt, codes, scales)
    y = gpu.gemv_q(W, _t(x)).numpy()
    for m in (0, 8, M // 2, M - 1):
        a8, s = O.quantize_activation_row(x[m])
        np.testing.assert_array_equal(y[m], O.gemv_i8(fmt, codes, scales, a8, s), err_msg=f"row {m}")
    W.close()


@pytest.mark.parametrize("fmt", [pf.FMT_Q4, pf.FMT_Q2, pf.FMT_Q15, pf.FMT_Q8])
@pytest.mark.parametrize("shape", [(128, 512), (320, 2048), (64, 1792)])
def test_gemm_int8_block(gpu, fmt, shape):
    """The int8 MFMA GEMM (M > 8 rows: many-sequence verify, batched prefill)
    equals the oracle's exact block GEMV row by row, bit for bit, including
    M not a multiple of 32 and the 10 tiles of 320 rows."""
    N, K = shape
    codes, scales = pf.gen_matrix(98, fmt * 11 + N, 0.02, N, K, fmt)
    W = gpu.upload_matrix(fmt, codes, scales)
    rng = np.random.default_rng(N * 3 + K)
    for M in (9, 32, 45, 320):
        x = (rng.standard_normal((M, K)) * 0.5).astype(np.float32)
        x[M // 2] = 0.0                                   # an all-zero row (scale 1, codes 0)
        y = gpu.gemv_q(W, _t(x)).numpy()
        for m in range(M):
            a8, s = O.quantize_activation_row(x[m])
            np.testing.assert_array_equal(y[m], O.gemv_i8(fmt, codes, scales, a8, s), err_msg=f"fmt {fmt} M {M} row {m}")
    W.close()


def test_fp32_products_of_many_rows():
    """k_mm_f32 with a head's gate and up in one launch, and with a residual,
    against the few-row kernels bit for bit (tests/cpp/test_mm_f32.hip: no call
    returns these products)."""
    exe = os.path.join(os.path.dirname(pf.__file__), "_lib", "tests", "test_mm_f32")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0
