"""Norms, RoPE, KV append, element-wise ops and the argmax tail: HIP vs oracle (needs an MI355X)."""
import numpy as np
import pytest

import oracle
from adam_amd import adamah as A
from adam_amd import quant
from gpu_util import note, up, f32map, put, read, rel_l2, load_qtensor, device_free_bytes

pytestmark = pytest.mark.gpu
TOL = 1e-3


def pair(hip):
    return [hip, oracle.init()]


@pytest.mark.parametrize("dim,rows", [(1152, 1), (4096, 1), (256, 5), (100, 3)])
def test_rmsnorm_family(hip, dim, rows):
    rng = np.random.default_rng(dim + rows)
    x = rng.standard_normal(rows * dim).astype(np.float32) * 3
    w = rng.uniform(0.5, 1.5, dim).astype(np.float32)
    r = rng.standard_normal(rows * dim).astype(np.float32)
    outs = []
    for g in pair(hip):
        note(f"rmsnorm dim={dim} rows={rows}")
        f32map(g, 0, 4 * rows * dim + dim, np.concatenate([x, r, w]))
        f32map(g, 3, dim, w)
        base = lambda o: up(g, [o + i * dim for i in range(rows)])
        s, rr, d1, d2 = base(0), base(rows * dim), base(2 * rows * dim + dim), base(3 * rows * dim + dim)
        wt = up(g, [2 * rows * dim] * rows)
        g.map_rmsnorm_dev(0, s, wt, d1, rows, dim, 1e-6)
        a = read(g, 0, 2 * rows * dim + dim, rows * dim)
        g.map_rmsnorm_x_dev(0, 3, s, up(g, [0] * rows), d1, rows, dim, 1e-5)
        b = read(g, 0, 2 * rows * dim + dim, rows * dim)
        g.map_rmsnorm_add_dev(0, s, wt, rr, d2, rows, dim, 1e-6)
        c = read(g, 0, 3 * rows * dim + dim, rows * dim)
        g.map_rmsnorm_add_dev(0, s, wt, rr, rr, rows, dim, 1e-6)          # in place on the residual
        d = read(g, 0, rows * dim, rows * dim)
        outs.append((a, b, c, d))
    for u, v in zip(*outs):
        assert rel_l2(u, v) < 1e-5


@pytest.mark.parametrize("dim,add", [(256, False), (1152, True)])
def test_rmsnorm_rows_at_irregular_places(hip, dim, add):
    """Several rows whose sources, destinations (and residuals) are NOT evenly spaced, in another order than they lie
    in memory, and a weight vector of their own per row: the multi-row kernel takes the rows' places from the tables
    on the device (evenly spaced rows get them by value) and gives the oracle's rows."""
    rng = np.random.default_rng(dim)
    rows = 5
    src = [7 * dim + 3, 0, 3 * dim + 1, 11 * dim, 5 * dim + 2]
    res = [20 * dim + o for o in (4 * dim, 0, 9 * dim + 5, 2 * dim, 6 * dim + 1)]
    dst = [40 * dim + o for o in (3 * dim, 8 * dim + 2, 0, 5 * dim + 7, dim + 1)]
    wts = [60 * dim + o for o in (2 * dim, 0, dim, 4 * dim, 3 * dim)]
    total = 66 * dim
    data = rng.standard_normal(total).astype(np.float32)
    outs = []
    for g in pair(hip):
        note(f"rmsnorm rows at irregular places dim={dim} add={add}")
        f32map(g, 0, total, data)
        hs, hr, hd, hw = up(g, src), up(g, res), up(g, dst), up(g, wts)
        if add:
            g.map_rmsnorm_add_dev(0, hs, hw, hr, hd, rows, dim, 1e-6)
        else:
            g.map_rmsnorm_dev(0, hs, hw, hd, rows, dim, 1e-6)
        outs.append(read(g, 0, 0, total))
    assert rel_l2(outs[0], outs[1]) < 1e-5
    for i in range(rows):                      # every row by the closed form as well
        x = data[src[i]:src[i] + dim].astype(np.float64)
        y = x / np.sqrt(np.mean(x * x) + 1e-6) * data[wts[i]:wts[i] + dim]
        if add:
            y = y + data[res[i]:res[i] + dim]
        assert rel_l2(outs[0][dst[i]:dst[i] + dim], y) < 1e-5, i


@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("dim", [1, 100, 1001, 1152, 4096, 5000, 8191])
def test_rmsnorm_of_several_rows_has_the_bits_of_one(hip, monkeypatch, dim, add):
    """Rows held in registers, of any width, whole words or not: the sums of the one-row kernel (ADAMAH_RMSNORM_ROWS=0: a workgroup of
    it a row) in its order."""
    rng = np.random.default_rng(dim)
    n = 24
    x = rng.standard_normal(dim * (2 * n + 2)).astype(np.float32) * np.float32(3)
    src, wt, res = dim * np.arange(n), np.full(n, n * dim), np.full(n, (n + 1) * dim)
    dst = (n + 2) * dim + src
    got = []
    for rows in ("1", "0"):
        monkeypatch.setenv("ADAMAH_RMSNORM_ROWS", rows)
        note(f"rmsnorm dim={dim} add={add} rows={rows}")
        f32map(hip, 0, x.size, x)
        h = [up(hip, v) for v in (src, wt, res, dst)]
        if add:
            hip.map_rmsnorm_add_dev(0, h[0], h[1], h[2], h[3], n, dim, 1e-5)
        else:
            hip.map_rmsnorm_dev(0, h[0], h[1], h[3], n, dim, 1e-5)
        got.append(read(hip, 0, 0, x.size))
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    y = x[:n * dim].reshape(n, dim).astype(np.float64)
    want = y / np.sqrt((y * y).mean(1, keepdims=True) + 1e-5) * x[n * dim:][:dim] + (x[(n + 1) * dim:][:dim] if add else 0)
    assert rel_l2(got[0][(n + 2) * dim:], want.reshape(-1)) < 1e-5


@pytest.mark.parametrize("heads,dim,pos,base", [(32, 128, 0, 500000.0), (8, 128, 4095, 500000.0),
                                               (4, 256, 639, 1e6), (1, 256, 16383, 1e4)])
def test_rope(hip, heads, dim, pos, base):
    rng = np.random.default_rng(pos + heads)
    x = rng.standard_normal(heads * dim).astype(np.float32)
    outs = []
    for g in pair(hip):
        note(f"rope heads={heads} dim={dim} pos={pos}")
        f32map(g, 0, 2 * heads * dim, x)
        g.map_rope_dev(0, up(g, [0]), up(g, [heads * dim]), 1, heads, dim, pos, base)
        outs.append(read(g, 0, heads * dim, heads * dim))
    if pos == 0:
        assert np.array_equal(outs[0], x)
    assert rel_l2(outs[0], outs[1]) < 1e-5


def test_qk_norm_rope_gemma_shape(hip):
    Hq, Hk, D = 4, 1, 256
    rng = np.random.default_rng(5)
    q = rng.standard_normal(Hq * D).astype(np.float32); k = rng.standard_normal(Hk * D).astype(np.float32)
    wq = rng.uniform(0.5, 1.5, D).astype(np.float32); wk = rng.uniform(0.5, 1.5, D).astype(np.float32)
    outs = []
    for g in pair(hip):
        note("qk_norm_rope 4+1 x 256")
        f32map(g, 0, 4096, np.concatenate([q, k, wq, wk]))
        g.map_qk_norm_rope_x_dev(0, 0, up(g, [i * D for i in range(Hq)]), up(g, [(Hq + Hk) * D] * Hq),
                                 up(g, [Hq * D]), up(g, [(Hq + Hk + 1) * D]), up(g, [2048]),
                                 Hq, D, Hk, D, 611, 1e6)
        outs.append(read(g, 0, 2048, (Hq + Hk) * D))
    assert rel_l2(outs[0], outs[1]) < 1e-5


def test_qk_norm_rope_rows_entry_point_equals_per_token_calls(hip):
    """adamah_qk_norm_rope_rows_dev (an extension: m tokens at pos0, pos0 + 1, ... in one native call) leaves the
    words the m calls of map_qk_norm_rope_x_dev leave, inside a batch and outside; the oracle's form agrees."""
    Hq, Hk, D, m, pos0 = 4, 1, 256, 9, 300
    per = (Hq + Hk) * D
    rng = np.random.default_rng(15)
    x = rng.standard_normal(m * per).astype(np.float32)
    w = rng.uniform(0.5, 1.5, 2 * D).astype(np.float32)
    w0, dst0 = m * per, m * per + 2 * D

    def go(g, one_call, batch):
        f32map(g, 0, dst0 + m * per, np.concatenate([x, w]))
        qs = [up(g, [t * per + i * D for i in range(Hq)]) for t in range(m)]
        ks = [up(g, [t * per + Hq * D]) for t in range(m)]
        ds = [up(g, [dst0 + t * per]) for t in range(m)]
        qw, kw = up(g, [w0] * Hq), up(g, [w0 + D])
        if batch:
            g.batch_begin()
        if one_call:
            g.qk_norm_rope_rows_dev(0, 0, qs, qw, ks, kw, ds, Hq, D, Hk, D, pos0, 1e6)
        else:
            for t in range(m):
                g.map_qk_norm_rope_x_dev(0, 0, qs[t], qw, ks[t], kw, ds[t], Hq, D, Hk, D, pos0 + t, 1e6)
        if batch:
            g.batch_end()
        return read(g, 0, dst0, m * per)

    note("qk_norm_rope rows entry point")
    base = go(hip, False, False)
    for batch in (False, True):
        assert np.array_equal(go(hip, True, batch).view(np.uint32), base.view(np.uint32))
    assert rel_l2(base, go(oracle.init(), True, False)) < 1e-5
    with pytest.raises(RuntimeError):
        hip.qk_norm_rope_rows_dev(0, 0, [987654], 1, [987655], 1, [987656], Hq, D, Hk, D, pos0, 1e6)


@pytest.mark.parametrize("m,Hq,Hk,D,case", [
    (13, 4, 1, 256, "apart"), (64, 1, 0, 2, "apart"), (65, 1, 0, 2, "apart"), (2, 30, 20, 6, "apart"), (2, 40, 30, 6, "apart"),
    (40, 3, 2, 64, "in place"), (40, 3, 2, 64, "one astray"), (33, 2, 2, 34, "backwards")])
def test_qk_norm_rope_of_many_rows(hip, m, Hq, Hk, D, case):
    """One launch for all tokens where the rows step evenly and clear of each other; where they do not (results over the
    sources, a row elsewhere, results laid down in reverse) and where they fit one list of row tasks, token by token.  The
    same words either way."""
    n = Hq + Hk
    rng = np.random.default_rng(m)
    x = rng.standard_normal(m * n * D + D).astype(np.float32)
    w = rng.uniform(0.5, 1.5, 2 * D).astype(np.float32)
    w0, dst0 = x.size, x.size + 2 * D

    def go(one_call):
        f32map(hip, 0, dst0 + (m + 1) * n * D, np.concatenate([x, w]))
        src = lambda t: t * n * D + (D if case == "one astray" and t == m // 2 else 0)
        dst = lambda t: src(t) if case == "in place" else dst0 + (m - 1 - t if case == "backwards" else t) * n * D
        qs = [up(hip, src(t) + np.arange(Hq) * D) for t in range(m)]
        ks = [up(hip, src(t) + (Hq + np.arange(max(Hk, 1))) * D) for t in range(m)]
        ds = [up(hip, [dst(t)]) for t in range(m)]
        qw, kw = up(hip, [w0] * Hq), up(hip, [w0 + D] * max(Hk, 1))
        hip.batch_begin()
        if one_call:
            hip.qk_norm_rope_rows_dev(0, 0, qs, qw, ks, kw, ds, Hq, D, Hk, D, 7, 1e4)
        else:
            for t in range(m):
                hip.map_qk_norm_rope_x_dev(0, 0, qs[t], qw, ks[t], kw, ds[t], Hq, D, Hk, D, 7 + t, 1e4)
        hip.batch_end()
        return read(hip, 0, 0, dst0 + (m + 1) * n * D), hip.get_last_barrier_count()

    note(f"qk_norm_rope of many rows m={m} {Hq}+{Hk}x{D} {case}")
    (a, la), (b, _) = go(True), go(False)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert la == 1 or case != "apart" or n > 64


def test_kv_append_rounds_to_fp16_and_mirrors(hip):
    Hkv, d, cap = 2, 64, 8
    rng = np.random.default_rng(6)
    kv = rng.standard_normal(2 * Hkv * d).astype(np.float32)
    kv_start = 1024
    outs = []
    for g in pair(hip):
        note("kv append fp16")
        f32map(g, 0, kv_start + 2 * Hkv * cap * d, kv)
        g.kv_cache_fp16(0, kv_start, 2 * Hkv * cap * d)
        spec = []
        for gi in range(Hkv):
            spec += [gi, kv_start // d + gi * cap, gi + Hkv, kv_start // d + (Hkv + gi) * cap]
        for pos in (0, 3):
            g.map_row_copy_offset_dev(0, up(g, spec), up(g, [0]), pos, 2 * Hkv, d)
        outs.append(read(g, 0, kv_start, 2 * Hkv * cap * d))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    rows = outs[0].reshape(2 * Hkv, cap, d)
    want = kv.astype(np.float16).astype(np.float32).reshape(2 * Hkv, d)
    assert np.array_equal(rows[:, 0], want) and np.array_equal(rows[:, 3], want) and not rows[:, 1].any()


@pytest.mark.parametrize("op", [A.OP_ADD, A.OP_GEGLU, A.OP_SWIGLU, A.OP_MUL, A.OP_SUB, A.OP_MAX])
def test_op2(hip, op):
    n = 6912
    rng = np.random.default_rng(op)
    a = rng.standard_normal(n).astype(np.float32) * 4; b = rng.standard_normal(n).astype(np.float32)
    outs = []
    for g in pair(hip):
        note(f"op2 code {op}")
        f32map(g, 0, 3 * n, np.concatenate([a, b]))
        g.map_op2_dev(0, op, up(g, np.arange(n)), up(g, np.arange(n, 2 * n)), up(g, np.arange(2 * n, 3 * n)), n)
        outs.append(read(g, 0, 2 * n, n))
    if op in (A.OP_ADD, A.OP_MUL, A.OP_SUB, A.OP_MAX):
        assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    assert rel_l2(outs[0], outs[1]) < 1e-6


def test_op1_broadcast_fma_reduce_layernorm_softmax(hip):
    n = 1000
    rng = np.random.default_rng(9)
    a = rng.standard_normal(n).astype(np.float32) * 3
    res = []
    for g in pair(hip):
        note("op1 / broadcast / fma / softmax / layernorm / reduce")
        f32map(g, 0, 8 * n, np.concatenate([a, a[::-1], np.full(n, 0.5, np.float32)]))
        src, src2, src3, dst = (up(g, np.arange(i * n, (i + 1) * n)) for i in (0, 1, 2, 4))
        out = []
        for code in (A.OP_TANH, A.OP_NEG, A.OP_EXP, A.OP_SIGMOID, A.OP_GELU, A.OP_SQUARE):
            g.map_op1_dev(0, code, src, dst, n); out.append(read(g, 0, 4 * n, n))
        g.map_broadcast_dev(0, A.OP_MUL, src, up(g, np.full(n, 2 * n)), dst, n); out.append(read(g, 0, 4 * n, n))
        g.map_broadcast_dev(0, A.OP_DIV, src, up(g, np.full(n, 2 * n)), dst, n); out.append(read(g, 0, 4 * n, n))
        g.map_fma_dev(0, src, src2, src3, dst, n); out.append(read(g, 0, 4 * n, n))
        g.map_softmax_abs_dev(0, up(g, [0, 500]), up(g, [4 * n, 4 * n + 500]), 500, 2); out.append(read(g, 0, 4 * n, n))
        g.map_attn_softmax_abs_dev(0, up(g, [0]), up(g, [4 * n]), n, 1, 0.25, 30.0); out.append(read(g, 0, 4 * n, n))
        g.map_softmax_dev(0, up(g, [0, 1]), up(g, [8, 9]), 500, 2); out.append(read(g, 0, 4 * n, n))
        g.map_layernorm_dev(0, up(g, [0, 1]), up(g, [8, 9]), up(g, [2 * n, 2 * n]), up(g, [n, n + 500]), 500, 1e-5, 2)
        out.append(read(g, 0, 4 * n, n))
        res.append(out)
    for i, (u, v) in enumerate(zip(*res)):
        assert rel_l2(u, v) < 2e-6, i


def test_embedding_fetch_paths(hip):
    """Tied Q4 embedding: gather_dev (dequantised) -> scatter_dev -> broadcast MUL; Q8 row gather."""
    V, E = 300, 1152
    rng = np.random.default_rng(12)
    w = (rng.standard_normal((V, E)) * 0.02).astype(np.float32)
    q4, q8 = quant.quantize_q4_0(w), quant.quantize_q8_0(w)
    tok, scale = 137, float(np.sqrt(E))
    outs = []
    for g in pair(hip):
        note("embedding fetch")
        load_qtensor(g, 1, q4); load_qtensor(g, 2, q8)
        f32map(g, 0, 3 * E + 8, None)
        g.scatter(0, np.array([3 * E], np.uint32), np.array([scale], np.float32))
        hid = up(g, np.arange(E))
        g.batch_begin()
        src, _, n, _ = g.map_gather_dev(1, up(g, tok * E + np.arange(E)), E)
        g.map_scatter_dev(0, hid, E, src)
        g.map_broadcast_dev(0, A.OP_MUL, hid, up(g, np.full(E, 3 * E)), hid, E)
        g.map_row_gather_xq8_dev(0, 2, 0, E, tok, E, scale)
        g.batch_end()
        outs.append((read(g, 0, 0, E), read(g, 0, E, E)))
    assert np.array_equal(outs[0][0].view(np.uint32), outs[1][0].view(np.uint32))
    assert np.array_equal(outs[0][0], q4.dequant()[tok] * np.float32(scale))
    assert np.array_equal(outs[0][1].view(np.uint32), outs[1][1].view(np.uint32))


@pytest.mark.parametrize("kind,N,K,rpg", [("q4", 5000, 1152, 256), ("q8", 3001, 4096, 256), ("q4", 700, 64, 64),
                                          ("q4", 48, 40, 16)])
def test_matvec_argmax_tail(hip, kind, N, K, rpg):
    """Fused LM-head GEMV + argmax: token id, per-group partial values and indices.  K = 40 makes
    rows start inside blocks, which must take the element-wise path."""
    rng = np.random.default_rng(N)
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    if K % 32 == 0:
        w[N // 2 + 3] = w[7]; w[N - 1] = w[7]                   # exact ties between rows
    qt = (quant.quantize_q4_0 if kind == "q4" else quant.quantize_q8_0)(w.reshape(-1, 32))
    x = rng.standard_normal(K).astype(np.float32)
    ng = (N + rpg - 1) // rpg
    mid = 1 if kind == "q4" else 2
    res = []
    for g in pair(hip):
        note(f"matvec_argmax {kind} {N}x{K} rpg={rpg}")
        load_qtensor(g, mid, qt)
        f32map(g, 0, K + 2 * ng + 8, x)
        fn = g.map_matvec_argmax_t_xq4_dev if kind == "q4" else g.map_matvec_argmax_t_xq8_dev
        fn(0, mid, up(g, [0]), up(g, [0]), up(g, np.arange(K, K + ng)),
           up(g, np.arange(K + ng, K + 2 * ng)), up(g, [K + 2 * ng]), K, N, rpg)
        res.append((int(read(g, 0, K + 2 * ng, 1)[0]), read(g, 0, K, ng), read(g, 0, K + ng, ng)))
    o = res[1]
    # token id: exact unless the oracle's own top-2 gap is at float32 rounding level
    top2 = np.sort(o[2])[-2:]
    if res[0][0] != o[0]:
        assert top2[1] - top2[0] <= 4e-6 * abs(top2[1]), (res[0][0], o[0])
    assert rel_l2(res[0][2], o[2]) < TOL
    agree = (res[0][1] == o[1]).mean()
    assert agree > 0.97, agree


@pytest.mark.parametrize("kind,N,K,rpg", [("q4", 100, 32, 7), ("q8", 513, 64, 256), ("q4", 512, 128, 256), ("q8", 300, 96, 64), ("q8", 999, 512, 100),
                                          ("q4", 70, 1024, 70), ("q8", 130, 1056, 33), ("q4", 64, 2048, 64)])
def test_matvec_argmax_of_short_rows(hip, kind, N, K, rpg):
    """Rows of 1 .. 64 blocks (several rows of a wave at once up to 32), groups that end inside a wave's rows."""
    test_matvec_argmax_tail(hip, kind, N, K, rpg)


def test_argmax_plain_ties_nan(hip):
    vals = np.full(5000, -1.0, np.float32)
    vals[[4097, 77, 3000]] = 9.5; vals[5] = np.nan
    f32map(hip, 0, 5008, vals)
    hip.map_argmax_dev(0, up(hip, np.arange(5000)), up(hip, [5004]), 5000)
    assert read(hip, 0, 5004, 1)[0] == 77.0


@pytest.mark.parametrize("kind,N,K,rpg,m", [("q8", 3001, 4096, 256, 16), ("q4", 5000, 1152, 256, 5), ("q8", 700, 128, 64, 19),
                                            ("q4", 4096, 256, 1000, 2)])
def test_matvec_argmax_of_consecutive_rows_in_one_pass(hip, kind, N, K, rpg, m):
    """The LM head of a lockstep batch: m GEMV + argmax ops over one matrix and consecutive activation
    rows in one batch read the matrix once (fp16 matrix-core GEMM + two ranking launches per 16 rows).
    Tokens equal the oracle's unless its own top two logits are closer than the fp16 operand rounding;
    the partial lists left behind are the last op's, values within 1e-3 relative L2."""
    rng = np.random.default_rng(N + m)
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    qt = (quant.quantize_q4_0 if kind == "q4" else quant.quantize_q8_0)(w)
    x = rng.standard_normal((m, K)).astype(np.float32)
    x[m - 1] *= 100.0
    ng = (N + rpg - 1) // rpg
    mid = 1 if kind == "q4" else 2
    base = m * K
    res = []
    for g in pair(hip):
        note(f"matvec_argmax run {kind} {N}x{K} rpg={rpg} m={m}")
        load_qtensor(g, mid, qt)
        f32map(g, 0, base + 2 * ng + m + 8, x.reshape(-1))
        fn = g.map_matvec_argmax_t_xq4_dev if kind == "q4" else g.map_matvec_argmax_t_xq8_dev
        b, li, lv = up(g, [0]), up(g, np.arange(base, base + ng)), up(g, np.arange(base + ng, base + 2 * ng))
        rows, dsts = [up(g, [j * K]) for j in range(m)], [up(g, [base + 2 * ng + j]) for j in range(m)]
        g.batch_begin()
        for j in range(m):
            fn(0, mid, rows[j], b, li, lv, dsts[j], K, N, rpg)
        g.batch_end()
        if g is hip:
            assert hip.get_last_barrier_count() == 4 * ((m + 15) // 16)   # conversion, GEMM, two ranking launches
        res.append((read(g, 0, base + 2 * ng, m).astype(np.int64), read(g, 0, base, ng), read(g, 0, base + ng, ng)))
    logits = x.astype(np.float64) @ qt.dequant().astype(np.float64).T
    for j in range(m):
        if res[0][0][j] != res[1][0][j]:
            top2 = np.sort(logits[j])[-2:]
            assert top2[1] - top2[0] <= 2e-3 * abs(top2[1]), (j, res[0][0][j], res[1][0][j])
            assert logits[j, res[0][0][j]] >= top2[0] - 1e-9
    assert rel_l2(res[0][2], res[1][2]) < 1e-3
    assert (res[0][1] == res[1][1]).mean() > 0.95


def test_gather_dev_results_stop_consuming_handles(hip):
    """map_gather_dev returns a new result handle per call (a decode loop makes one per token); the library keeps
    the latest few thousand and hands the oldest out again, so ids stay bounded while recent results stay valid."""
    note("gather_dev handle ring")
    n = 64
    f32map(hip, 0, 4 * n, np.arange(4 * n, dtype=np.float32))
    locs = [up(hip, np.arange(lo, lo + n)) for lo in (0, n, 2 * n)]
    h0 = hip.map_gather_dev(0, locs[0], n)[0]
    h1 = hip.map_gather_dev(0, locs[1], n)[0]
    assert h0 != 0 and h1 != 0 and h0 != h1
    assert np.array_equal(hip.download_dev(h0, n), np.arange(0, n, dtype=np.float32))      # an older result is intact
    assert np.array_equal(hip.download_dev(h1, n), np.arange(n, 2 * n, dtype=np.float32))
    ids = set()
    for i in range(6000):
        ids.add(hip.map_gather_dev(0, locs[i % 3], n)[0])
    assert 0 not in ids and len(ids) <= 4200
    last = hip.map_gather_dev(0, locs[2], n)[0]
    assert np.array_equal(hip.download_dev(last, n), np.arange(2 * n, 3 * n, dtype=np.float32))


def test_gather_dev_results_of_alternating_sizes_stay_bounded(hip):
    """A small result (one embedding row) and a large one (a prefill chunk's rows) asked for in turn, far past the
    limits of the result rings: every size class hands its own oldest result out again, so neither the ids nor the
    device memory behind them keep growing, and the results stay right."""
    note("gather_dev size-class rings")
    small, large = 64, 65536
    f32map(hip, 0, large, np.arange(large, dtype=np.float32))
    ls, ll = up(hip, np.arange(small)), up(hip, np.arange(large))
    ids_s, ids_l = set(), set()
    free_mid = None
    for i in range(9000):
        ids_s.add(hip.map_gather_dev(0, ls, small)[0])
        if i % 2 == 0:
            ids_l.add(hip.map_gather_dev(0, ll, large)[0])
        if i == 6000:
            hip.sync()
            free_mid = device_free_bytes()       # both classes are past their limits here
    hip.sync()
    assert 0 not in ids_s and 0 not in ids_l and not (ids_s & ids_l)
    assert len(ids_s) <= 4096 and len(ids_l) <= 256, (len(ids_s), len(ids_l))
    assert device_free_bytes() >= free_mid, "the arena grew after both rings were full"
    hs, hl = hip.map_gather_dev(0, ls, small)[0], hip.map_gather_dev(0, ll, large)[0]
    assert np.array_equal(hip.download_dev(hs, small), np.arange(small, dtype=np.float32))
    assert np.array_equal(hip.download_dev(hl, large), np.arange(large, dtype=np.float32))


@pytest.mark.parametrize("M,K,N,n_ops", [(1, 256, 300, 1), (3, 70, 33, 2), (1, 4096, 512, 1)])
def test_plain_float_matmuls(hip, M, K, N, n_ops):
    """map_matmul_dev, map_matmul_t_x_dev and map_matmul_x_dev (float32 operands; the second and third read B
    from another map -- the path a model with float weight matrices takes) against the oracle."""
    rng = np.random.default_rng(M + K + N)
    Aop = rng.standard_normal((n_ops, M, K)).astype(np.float32)
    B = rng.standard_normal((n_ops, K, N)).astype(np.float32)
    a_sz, b_sz, c_sz = M * K, K * N, M * N
    a0, b0, c0 = 0, n_ops * a_sz + 3, n_ops * (a_sz + b_sz) + 7
    out = {}
    for name, g in (("hip", hip), ("oracle", oracle.init())):
        note(f"plain matmuls {M}x{K}x{N} ops={n_ops} on {name}")
        f32map(g, 0, c0 + 3 * n_ops * c_sz)
        put(g, 0, a0, Aop); put(g, 0, b0, B)
        f32map(g, 3, 2 * n_ops * b_sz + 8)
        put(g, 3, 4, B); put(g, 3, 4 + n_ops * b_sz, B.transpose(0, 2, 1))
        la = up(g, a0 + np.arange(n_ops) * a_sz)
        lc = [up(g, c0 + v * n_ops * c_sz + np.arange(n_ops) * c_sz) for v in range(3)]
        g.map_matmul_dev(0, la, up(g, b0 + np.arange(n_ops) * b_sz), lc[0], M, K, N, n_ops)
        g.map_matmul_x_dev(0, 3, la, up(g, 4 + np.arange(n_ops) * b_sz), lc[1], M, K, N, n_ops)
        g.map_matmul_t_x_dev(0, 3, la, up(g, 4 + n_ops * b_sz + np.arange(n_ops) * b_sz), lc[2], M, K, N, n_ops)
        out[name] = read(g, 0, c0, 3 * n_ops * c_sz).reshape(3, -1)
    want = np.stack([Aop[o].astype(np.float64) @ B[o].astype(np.float64) for o in range(n_ops)]).reshape(-1)
    for v in range(3):
        assert rel_l2(out["hip"][v], out["oracle"][v]) < 1e-5
        assert rel_l2(out["hip"][v], want) < 1e-5


@pytest.mark.parametrize("n_tok,n_seq,Hq,Hk,D,pos0,rotate,kv16", [(1, 1, 4, 1, 64, 0, True, True), (5, 3, 6, 2, 128, 0, True, True),
                                                                  (33, 1, 32, 8, 128, 100, True, True), (3, 40, 2, 2, 64, 7, True, False),
                                                                  (4, 2, 4, 2, 256, 9, False, True)])
def test_rope_append_rows_equals_rotations_and_row_copies(hip, n_tok, n_seq, Hq, Hk, D, pos0, rotate, kv16):
    """adamah_hip_rope_append_rows_dev (an extension) leaves, bit for bit, the words of map_rope_dev over the Q and K rows of every
    sequence and map_row_copy_offset_dev of the results; rows have padding between them, and nothing else is written."""
    rng = np.random.default_rng(n_tok * 100 + n_seq)
    cap, rows, qs, ks, vs = pos0 + n_tok + 3, n_tok * n_seq, Hq * D + 8, Hk * D + 4, Hk * D + 12
    q0 = 16
    k0, v0 = q0 + rows * qs, q0 + rows * (qs + ks)
    c0 = -(-(v0 + rows * vs) // D) * D
    per = 2 * Hk * cap * D
    total = c0 + n_seq * per + 8
    x = rng.standard_normal(total).astype(np.float32)
    kb = [c0 + s * per for s in range(n_seq)]
    vb = [k + Hk * cap * D for k in kb]
    got = []
    for one_call in (False, True):
        note(f"rope append n_tok={n_tok} n_seq={n_seq} one_call={one_call}")
        f32map(hip, 0, total, x)
        if kv16:
            hip.kv_cache_fp16(0, c0, n_seq * per)
        if one_call:
            hip.rope_append_rows_dev(0, q0, qs, Hq, k0, ks, Hk, v0, vs, D, n_tok, kb, vb, cap * D, pos0, 1e4, rotate=rotate)
        else:
            for s in range(n_seq):
                r = s * n_tok + np.arange(n_tok)
                if rotate:
                    for at, step, H in ((q0, qs, Hq), (k0, ks, Hk)):
                        h = up(hip, at + r * step)
                        hip.map_rope_dev(0, h, h, n_tok, H, D, pos0, 1e4)
            data = read(hip, 0, 0, total)
            for s in range(n_seq):
                for t in range(n_tok):
                    for at, step, cache in ((k0, ks, kb[s]), (v0, vs, vb[s])):
                        row = data[at + (s * n_tok + t) * step:][:Hk * D].reshape(Hk, D)
                        row = row.astype(np.float16).astype(np.float32) if kv16 else row
                        for h in range(Hk):
                            put(hip, 0, cache + h * cap * D + (pos0 + t) * D, row[h])
        got.append(read(hip, 0, 0, total))
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    bad = dict(q=q0, qs=qs, k=k0, v=v0, kb=kb, vb=vb, step=cap * D)
    for change in (dict(v=k0), dict(kb=vb), dict(vb=[total - 8] * n_seq), dict(k=total - Hk * D + 1), dict(qs=D) if rotate and Hq > 1 else dict(kb=[k0] * n_seq)):
        a = {**bad, **change}
        with pytest.raises(RuntimeError):
            hip.rope_append_rows_dev(0, a["q"], a["qs"], Hq, a["k"], ks, Hk, a["v"], vs, D, n_tok, a["kb"], a["vb"], a["step"], pos0, 1e4, rotate=rotate)
    assert np.array_equal(read(hip, 0, 0, total).view(np.uint32), got[1].view(np.uint32))


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n_tok,n_seq,Hq,Hk,D,pos0", [(3, 2, 32, 8, 256, 5), (2, 1, 3, 1, 6, 0), (1, 33, 5, 2, 8, 1), (2, 1, 1, 1, 2, 3), (4, 1, 40, 12, 72, 2)])
def test_rope_append_rows_of_any_start(hip, n_tok, n_seq, Hq, Hk, D, pos0, shift):
    """Rows that start on four values and rows that do not, more pairs than a workgroup takes at once and fewer than it has threads."""
    rng = np.random.default_rng(D)
    cap, rows = pos0 + n_tok + 1, n_tok * n_seq
    qs, ks, vs = Hq * D, Hk * D + 4, Hk * D
    q0 = shift
    k0, v0 = q0 + rows * qs, q0 + rows * (qs + ks)
    c0, per = v0 + rows * vs, 2 * Hk * cap * D
    x = rng.standard_normal(c0 + n_seq * per).astype(np.float32)
    kb = [c0 + s * per for s in range(n_seq)]
    out = []
    for g in (hip, oracle.init()):
        note(f"rope append {n_tok} x {n_seq}, {Hq} + {Hk} heads of {D}, shift {shift}")
        f32map(g, 0, x.size, x)
        g.kv_cache_fp16(0, c0, n_seq * per)
        g.rope_append_rows_dev(0, q0, qs, Hq, k0, ks, Hk, v0, vs, D, n_tok, kb, [k + Hk * cap * D for k in kb], cap * D, pos0, 1e4, rotate=True)
        out.append(read(g, 0, 0, x.size))
    assert rel_l2(out[0][:c0], out[1][:c0]) < 1e-6
    assert np.array_equal(out[0][k0 + rows * ks:c0], x[k0 + rows * ks:c0])
    assert np.abs(out[0][c0:] - out[1][c0:]).max() <= 2.0 ** -10 * np.abs(x).max() * 1.5 + 1e-7     # one fp16 step where the rotations round apart


def test_rope_append_rows_of_sequences_beyond_2_to_the_32_elements(hip):
    """The 33rd sequence, where a second launch begins, with its Q row at element 2^32 of the map (17 GB, two elements a pack)."""
    note("rope append across 2^32 elements")
    n_seq, D, cap = 35, 8, 4
    k0, v0 = 1024, 2048
    kb = [4096 + s * 2 * cap * D for s in range(n_seq)]
    top = 1 << 32
    rng = np.random.default_rng(4)
    q, kv = rng.standard_normal((n_seq, D)).astype(np.float32), rng.standard_normal((2, n_seq, D)).astype(np.float32)
    got = []
    try:
        for packs, q0 in ((top // 2 + 64, top - 32 * D), (1 << 13, 12288)):
            hip.map_create_typed(0, A.DTYPE_F32, 2, packs)
            hip.set_dtype(A.DTYPE_F32)
            for at, x in ((q0, q), (k0, kv[0]), (v0, kv[1])):
                assert hip.scatter_contiguous(0, at // 2, x.reshape(-1), n_locs=x.size // 2) == 0
            hip.rope_append_rows_dev(0, q0, D, 1, k0, D, 1, v0, D, D, 1, kb, [k + cap * D for k in kb], cap * D, 3, 1e4, rotate=True)
            part = lambda at, n: hip.gather(0, np.arange(at // 2, (at + n) // 2, dtype=np.uint32)).view(np.float32).copy()
            got.append((part(q0, q.size), part(0, 4096 + n_seq * 2 * cap * D)))
    finally:
        f32map(hip, 0, 64)
    assert not np.array_equal(got[0][0], q.reshape(-1))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("B,Hq,Hk,D", [(8, 32, 8, 128), (5, 16, 2, 64), (3, 32, 8, 128)])
def test_wide_rotation_takes_few_key_rows_and_copies_along(hip, monkeypatch, B, Hq, Hk, D):
    """One token of B sequences: more than 64 Q rows beside at most 64 K rows and copies still rotate and append in one launch, and
    leave the words of separate ones (ADAMAH_ROWS_WIDE=0)."""
    rng = np.random.default_rng(B * Hq)
    cap, pos = 9, 4
    q0, k0 = 0, B * Hq * D
    v0 = k0 + B * Hk * D
    c0 = v0 + B * Hk * D
    per = 2 * Hk * cap * D
    x = rng.standard_normal(c0 + B * per).astype(np.float32)
    spec = np.empty((B, 2 * Hk, 2), np.uint32)
    for s in range(B):
        for h in range(Hk):
            spec[s, 2 * h] = ((k0 // D) + s * Hk + h, (c0 + s * per) // D + h * cap)
            spec[s, 2 * h + 1] = ((v0 // D) + s * Hk + h, (c0 + s * per) // D + (Hk + h) * cap)
    got = []
    for wide in ("0", "1"):
        monkeypatch.setenv("ADAMAH_ROWS_WIDE", wide)
        note(f"wide rotation B={B} wide={wide}")
        f32map(hip, 0, x.size, x)
        hip.kv_cache_fp16(0, c0, B * per)
        hq, hk, hs, hz = up(hip, [q0]), up(hip, [k0]), up(hip, spec.reshape(-1)), up(hip, [0])
        hip.batch_begin()
        hip.map_rope_dev(0, hq, hq, 1, B * Hq, D, pos, 1e4)
        hip.map_rope_dev(0, hk, hk, 1, B * Hk, D, pos, 1e4)
        hip.map_row_copy_offset_dev(0, hs, hz, pos, 2 * Hk * B, D)
        hip.batch_end()
        got.append((read(hip, 0, 0, x.size), hip.get_last_barrier_count()))
    assert got[1][1] == 1 and got[0][1] > 1
    assert np.array_equal(got[0][0].view(np.uint32), got[1][0].view(np.uint32))
