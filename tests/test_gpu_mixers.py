"""Layered mixer models on the GPU: every op against the NumPy op surface, whole models against the plain statement of
the mechanisms, in one piece, in portions, token by token, in lockstep, and through generation and trace replay."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from adam_amd import adamah as A
from adam_amd.engine import GenerationConfig
from adam_amd.mixer_engine import MixerEngine
from adam_amd.models import load_engine, vomotar_config
from adam_amd.safetensors_file import bf16_to_f32, f32_to_bf16
from gpu_util import f32map, note, read, rel_l2, up
from mixer_cases import CONFIGS, config, delta, floats, par, rel, weights, write_model
from mixer_pair import CA, OP, ST, WS, WT, Pair
from oracle import mixers_np as M

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL = {"float32": 2e-5, "bfloat16": 6e-2}      # bfloat16: the worst row; the NumPy surface with the same rounding reaches 3.3e-2


# ---- products --------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows,n,k,groups,epi", [
    (1, 70, 33, 3, 0), (1, 96, 640, 0, 2), (1, 51, 1100, 1, 1), (1, 33, 1536, 32, 0), (2, 70, 33, 3, 0), (5, 64, 200, 5, 2),
    (16, 129, 64, 1, 1), (17, 64, 320, 2, 2), (31, 45, 96, 0, 0), (33, 96, 130, 13, 2), (64, 200, 256, 4, 1), (65, 130, 72, 0, 0),
    (200, 1000, 192, 3, 0), (300, 8224, 64, 1, 2), (300, 8200, 128, 1, 1),
    (1, 10, 20000, 4, 0), (3, 37, 16000, 4, 0)])
def test_linear(hip, dtype, rows, n, k, groups, epi):
    note(f"linear {dtype} rows {rows} n {n} k {k} groups {groups} epi {epi}")
    rng = np.random.default_rng(rows * 1000 + n)
    ks, src_rows = (k + 63) // 64 * 64, rows + 3
    out_w = n // 2 if epi == 2 else n
    wt_len = 0 if not groups else (k if groups % 2 else k // groups)
    act = int(rng.integers(0, 3)) if groups else 0
    src, gate, wt, out = 5, 5 + src_rows * k, 5 + 2 * src_rows * k, 5 + 2 * src_rows * k + k
    total = out + rows * (out_w + 3)
    opnd, oo = 64, 64 + rows * ks
    p = Pair(hip, total + 64, wt=n * ks + 8, opnd=oo + rows * ((out_w + 63) // 64 * 64 + 64), dtype=dtype)
    W = np.zeros((n, ks), np.uint16)
    W[:, :k] = f32_to_bf16((rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32))
    p.put(WT, 8, W)
    p.put(WS, 0, rng.standard_normal(total))
    spec = A.LinearSpec(w=8, n=n, k=k, k_stride=ks, src=src, src_stride=k, groups=groups, eps=1e-4, wt=wt, wt_len=wt_len, gate=gate,
                        gate_stride=k, gate_act=act, opnd=opnd, ready=0, out=out, out_stride=out_w + 3, epi=epi, out_opnd=oo,
                        out_opnd_stride=(out_w + 63) // 64 * 64)
    h = p.up(spec.words())
    pick = p.up(rng.integers(0, src_rows, rows))
    tol = 2e-5 if dtype == "float32" or rows == 1 else 4e-2        # bfloat16: an operand may round the other way
    p.call("linear_dev", WS, OP, WT, h, pick, rows)
    if epi == 2 and rows > 1:
        # the pairs went to the operand rows: a product with the identity brings them out, its operand ready
        w2 = (out_w + 63) // 64 * 64
        eye = np.zeros((out_w, w2), np.float32)
        eye[np.arange(out_w), np.arange(out_w)] = 1
        for g in p.g:
            g.map_create_typed(WT, A.DTYPE_BF16, 1, eye.size)
        p.put(WT, 0, f32_to_bf16(eye))
        s2 = A.LinearSpec(w=0, n=out_w, k=out_w, k_stride=w2, opnd=oo, ready=1, out=out, out_stride=out_w + 3)
        p.call("linear_dev", WS, OP, WT, p.up(s2.words()), 0, rows)
    p.same(WS, out, rows * (out_w + 3) - 3, tol, "out")


@pytest.mark.parametrize("n,k,groups,epi,branched,act", [
    (1, 1088, 1, 0, 0, 0), (2047, 1024, 0, 1, 0, 0), (2048, 2048, 1, 0, 2, 0), (2049, 2048, 4, 0, 0, 2), (2048, 2112, 1, 1, 1, 0),
    (130, 4096, 1024, 0, 0, 3), (7, 4104, 1, 0, 2, 0), (2051, 4160, 1, 1, 0, 1), (67, 2048, 1, 2, 2, 0), (2050, 4096, 1, 0, 1, 0), (9, 8192, 2, 1, 0, 0),
    (5, 32768, 1, 0, 0, 0), (3, 9000, 0, 0, 0, 0), (40, 960, 1, 0, 2, 0), (4131, 2048, 1, 2, 2, 0)])
@pytest.mark.parametrize("listed,shift", [(False, 0), (True, 1)])
def test_one_row_products(hip, n, k, groups, epi, branched, act, listed, shift):
    """A wave has one row up to 2048 of them and two beyond, eight steps in flight beyond 2048 columns, some a second task just beyond a
    workgroup a CU; rows on four floats (shift 0) and off."""
    note(f"one row n {n} k {k} groups {groups} epi {epi} branched {branched} act {act} listed {listed} shift {shift}")
    rng = np.random.default_rng(n + k)
    ks, st, at, pos = (k + 63) // 64 * 64, (k + 3) // 4 * 4 + 4 + shift, {}, 4 + shift
    tail = 3 if epi == 2 else 0
    for name, sz in (("x", 3 * st), ("br", 3 * st), ("gate", 3 * st), ("wt", k), ("bw", k), ("res", 3 * st), ("keep", 3 * st), ("bias", n), ("out", n), ("tail", n)):
        at[name] = pos
        pos += (sz + 3) // 4 * 4 + (4 if shift == 0 else 3)
    p = Pair(hip, pos, wt=n * ks)
    W = np.zeros((n, ks), np.uint16)
    W[:, :k] = f32_to_bf16((rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32))
    p.put(WT, 0, W)
    p.put(WS, 0, rng.standard_normal(pos))
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=ks, src=at["x"], src_stride=st, groups=groups, eps=1e-4, wt=at["wt"], wt_len=k if groups else 0, wt_add=0.5,
                        gate=at["gate"], gate_stride=st, gate_act=act, branched=branched, branch=at["br"], branch_stride=st, branch_wt=at["bw"],
                        res_out=at["res"], res_stride=st, keep=at["keep"], keep_stride=st, kept=1, bias=at["bias"], biased=int(epi == 0), out=at["out"],
                        out_stride=n, epi=epi, tail=tail, tail_out=at["tail"], tail_stride=n)
    p.call("linear_dev", WS, OP, WT, p.up(spec.words()), p.up([2]) if listed else 0, 1)
    # float32 throughout: as for the operands above
    for name, sz in (("out", (n - tail) // 2 if epi == 2 else n), ("keep", 3 * st), ("res", 3 * st), ("tail", max(tail, 1))):
        p.same(WS, at[name], sz, 2e-5, name)


@pytest.mark.parametrize("rows,n,k,biased,add", [
    (2000, 8170, 64, 0, 0), (2048, 4096, 128, 1, 1), (1999, 4090, 192, 1, 0), (600, 12600, 64, 0, 1), (300, 10300, 128, 1, 0),
    (300, 6001, 320, 0, 0), (40, 300, 256, 1, 1), (33, 64, 64, 0, 0), (100, 131, 1024, 0, 1)])
def test_linear_tiles(hip, rows, n, k, biased, add):
    """Every tile of the many-row product (256 x 256 down to 64 x 64 on 256 CUs), rings shorter and longer than K, ragged ends."""
    note(f"linear tiles rows {rows} n {n} k {k}")
    rng = np.random.default_rng(n)
    st = n + (0 if n % 4 == 0 else 3)
    W = f32_to_bf16(rng.standard_normal((n, k)).astype(np.float32))
    x = f32_to_bf16(rng.standard_normal((rows, k)).astype(np.float32))
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, W.size)
    hip.scatter_contiguous(WT, 0, W.reshape(-1))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, x.size)
    hip.scatter_contiguous(OP, 0, x.reshape(-1))
    old = rng.standard_normal((rows + 1) * st).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    f32map(hip, WS, old.size + n, np.concatenate([old, bias]))
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=k, opnd=0, ready=1, out=0, out_stride=st, epi=add, bias=old.size, biased=biased)
    hip.linear_dev(WS, OP, WT, up(hip, spec.words()), 0, rows)
    got = read(hip, WS, 0, old.size).reshape(rows + 1, st)
    f64 = lambda b: (b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    old = old.reshape(rows + 1, st)
    want = f64(x) @ f64(W).T + (bias if biased else 0.0) + (old[:rows, :n] if add else 0.0)
    # exact products, float32 sums of at most 1026 terms: 1026 * 2^-24 relative to the terms' root sum of squares at most
    assert rel_l2(got[:rows, :n], want) < 6.2e-5
    assert np.array_equal(got[:rows, n:], old[:rows, n:]) and np.array_equal(got[rows], old[rows])       # nothing beyond


@pytest.mark.parametrize("rows,n,k,epi,tail", [
    (2, 1, 1088, 0, 0), (16, 4095, 1536, 1, 0), (17, 4097, 2048, 0, 0), (32, 8195, 1600, 1, 0), (12, 12300, 2048, 0, 0), (3, 16390, 1088, 1, 0),
    (31, 36901, 1088, 0, 0), (5, 70003, 1088, 1, 0), (16, 8200, 2560, 0, 0), (32, 300, 2624, 1, 0), (9, 4100, 3072, 0, 0), (20, 515, 3520, 1, 0),
    (16, 8208, 4096, 0, 0), (29, 4099, 4032, 0, 0), (12, 32, 1088, 2, 0), (32, 8227, 2048, 2, 35), (2, 8257, 4096, 2, 1), (18, 16448, 1216, 2, 64),
    (13, 34000, 1344, 2, 16), (7, 3601, 2112, 0, 0),
    # columns read twice in passes behind one another; sums of gate and up that LDS does not hold at once
    (31, 36901, 1216, 0, 0), (5, 70003, 1344, 1, 0), (32, 12300, 1600, 0, 0), (20, 33859, 1152, 2, 35), (32, 40000, 1280, 2, 64), (9, 9222, 2624, 0, 0),
    (3, 1500, 1216, 0, 0)])
def test_products_of_few_rows(hip, rows, n, k, epi, tail):
    """One pass of 16 matrix rows a workgroup up to more than LDS holds the sums of, rows of every count of steps, whole and ragged; an
    infinite value of a token whose columns a wave reads twice."""
    note(f"few rows {rows} n {n} k {k} epi {epi} tail {tail}")
    rng = np.random.default_rng(n + k)
    f64 = lambda b: (b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    W = f32_to_bf16(rng.standard_normal((n, k), dtype=np.float32) / np.float32(np.sqrt(k)))
    x = rng.standard_normal((rows, k), dtype=np.float32)
    x[rows - 1, 5] = np.inf
    xb = f32_to_bf16(x)
    pair_w, st, op_at = (n - tail) // 2 if epi == 2 else 0, max(tail, 1) + 2 if epi == 2 else n + 3, (rows * k + 7) // 8 * 8
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, W.size)
    hip.scatter_contiguous(WT, 0, W.reshape(-1))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, op_at + rows * (pair_w + 1) + 8)
    hip.scatter_contiguous(OP, 0, xb.reshape(-1))
    old = rng.standard_normal((rows + 1, st)).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    f32map(hip, WS, old.size + n, np.concatenate([old.reshape(-1), bias]))
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=k, opnd=0, ready=1, out=0, out_stride=st, epi=epi, out_opnd=op_at, out_opnd_stride=pair_w + 1,
                        tail=tail, tail_out=0, tail_stride=st, bias=old.size, biased=int(epi == 0))
    hip.linear_dev(WS, OP, WT, up(hip, spec.words()), 0, rows)
    got = read(hip, WS, 0, old.size).reshape(rows + 1, st)
    y = f64(xb[:-1]) @ f64(W).T
    tol = k * 2.0 ** -24                          # exact products, float32 sums of k terms: relative to the terms' root sum of squares
    held = n if epi < 2 else tail
    assert np.array_equal(got[:, held:], old[:, held:]) and np.array_equal(got[rows], old[rows])             # nothing beyond
    inf = np.sign(f64(W[:, 5])) * np.inf          # (a weight of 0 meets it: no number)
    with np.errstate(invalid="ignore"):
        inf[f64(W[:, 5]) == 0.0] = np.nan
    if epi < 2:
        want = y + (old[:rows - 1, :n] if epi else bias)
        assert rel_l2(got[:rows - 1, :n], want) < tol and np.array_equal(got[rows - 1, :n], inf.astype(np.float32), equal_nan=True)
        return
    if tail:
        assert rel_l2(got[:rows - 1, :tail], y[:, n - tail:]) < tol
        assert np.array_equal(got[rows - 1, :tail], inf[n - tail:].astype(np.float32), equal_nan=True)
    head = y[:, :n - tail].reshape(rows - 1, -1, 2, 16)
    want = (head[:, :, 0] / (1.0 + np.exp(-head[:, :, 0])) * head[:, :, 1]).reshape(rows - 1, pair_w)
    raw = hip.gather(OP, np.arange(op_at, op_at + rows * (pair_w + 1), dtype=np.uint32))
    pairs = f64(raw.view(np.uint16)[:raw.size]).reshape(rows, -1)[:-1, :pair_w]
    assert rel_l2(pairs, want) < 4 * tol + 2.0 ** -8


@pytest.mark.parametrize("rows,k,groups,act,per_group", [
    (1, 2048, 1, 1, 0), (1, 8192, 32, 2, 1), (2, 8196, 1, 0, 0), (3, 4096, 64, 3, 1), (3, 16384, 16, 1, 0), (2, 16640, 1, 2, 0), (5, 768, 3, 3, 0),
    (5, 768, 1, 0, 1), (7, 256, 64, 1, 1), (4, 1200, 25, 2, 0), (530, 4096, 4, 1, 1), (520, 4352, 1, 3, 0), (515, 36, 0, 0, 0),
    (4, 256, 1, 2, 0), (4, 260, 1, 1, 0), (4, 260, 5, 0, 1), (6, 1024, 8, 1, 1), (6, 1028, 1, 3, 0), (1, 1152, 1, 0, 0), (1, 1022, 1, 2, 0),
    (1, 1028, 0, 0, 0), (9, 1300, 0, 0, 0), (9, 1302, 0, 0, 0), (600, 1100, 0, 0, 0), (3, 20000, 0, 0, 0)])
def test_operand_rows_in_one_trip(hip, rows, k, groups, act, per_group):
    """Rows and groups that a workgroup's registers hold (and just do not), groups of lanes and of waves, every gate."""
    note(f"operand rows {rows} k {k} groups {groups} act {act}")
    rng = np.random.default_rng(k + rows)
    n, ks = 40, (k + 63) // 64 * 64
    wt_len = 0 if not groups else k // groups if per_group else k
    gate, wt, keep = rows * k, 2 * rows * k, 2 * rows * k + k
    out = keep + rows * k
    p = Pair(hip, out + rows * n + 64, wt=n * ks, opnd=rows * ks, dtype="float32")
    W = np.zeros((n, ks), np.uint16)
    W[:, :k] = f32_to_bf16((rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32))
    p.put(WT, 0, W)
    p.put(WS, 0, rng.standard_normal(keep))
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=ks, src=0, src_stride=k, groups=groups, eps=1e-4, wt=wt, wt_len=wt_len, wt_add=0.5, gate=gate,
                        gate_stride=k, gate_act=act if groups else 0, opnd=0, ready=0, keep=keep, keep_stride=k, kept=1, out=out, out_stride=n)
    p.call("linear_dev", WS, OP, WT, p.up(spec.words()), 0, rows)
    # float32 throughout; a group's sum of at most 16640 squares: 2e-5 as for every operand above
    p.same(WS, keep, rows * k, 2e-5, "operand")
    p.same(WS, out, rows * n, 2e-5, "out")


@pytest.mark.parametrize("rows,n", [(33, 70), (100, 1001), (300, 515), (700, 2048), (2050, 2100)])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6])
def test_linear_of_few_steps(hip, rows, n, steps):
    """Products of as many 64-column steps as the ring of tiles has buffers, one more, one and two fewer, on small and large tiles."""
    k = 64 * steps
    note(f"linear rows {rows} n {n} k {k}")
    rng = np.random.default_rng(rows + k)
    f64 = lambda b: (b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    W, x = (f32_to_bf16(rng.standard_normal(s).astype(np.float32)) for s in ((n, k), (rows, k)))
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, W.size)
    hip.scatter_contiguous(WT, 0, W.reshape(-1))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, x.size)
    hip.scatter_contiguous(OP, 0, x.reshape(-1))
    f32map(hip, WS, rows * n)
    hip.linear_dev(WS, OP, WT, up(hip, A.LinearSpec(w=0, n=n, k=k, k_stride=k, opnd=0, ready=1, out=0, out_stride=n).words()), 0, rows)
    got, want = read(hip, WS, 0, rows * n).reshape(rows, n), f64(x) @ f64(W).T
    # exact products, float32 sums: k 2^-24 relative to the terms' root sum of squares at most
    assert max(rel_l2(a, b) for a, b in zip(got, want)) < k * 2.0 ** -24


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows,n,k,epi,tail", [
    (33, 70, 320, 0, 0), (40, 131, 4096, 1, 0), (64, 96, 1088, 2, 0), (65, 201, 2048, 2, 41), (190, 2050, 1024, 0, 0), (300, 515, 3008, 1, 0),
    (257, 1000, 576, 2, 8), (3, 45, 512, 0, 0), (512, 2048, 2048, 0, 0)])
def test_linear_shares_and_pieces(hip, dtype, rows, n, k, epi, tail):
    """Long rows over shares of K, float32 rows in their bfloat16 pieces (one of them infinite, one huge, one tiny)."""
    note(f"linear shares {dtype} rows {rows} n {n} k {k} epi {epi}")
    rng = np.random.default_rng(n + k)
    f64 = lambda b: (b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    W = f32_to_bf16(rng.standard_normal((n, k)).astype(np.float32) / np.float32(np.sqrt(k)))
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[0] *= np.float32(2.0 ** 100)
    x[1] *= np.float32(2.0 ** -80)
    wide = dtype == "float32"
    if not wide:
        x = f64(f32_to_bf16(x)).astype(np.float32)
    x[rows - 1, 5] = np.inf
    pair_w = (n - tail) // 2 if epi == 2 else 0
    st, op_at = n + 3, (rows * k + 7) // 8 * 8
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, W.size)
    hip.scatter_contiguous(WT, 0, W.reshape(-1))
    hip.map_create_typed(OP, A.DTYPE_F32 if wide else A.DTYPE_BF16, 1, op_at + rows * (pair_w + 1) + 8)
    hip.scatter_contiguous(OP, 0, x.reshape(-1) if wide else f32_to_bf16(x.reshape(-1)))
    old = rng.standard_normal((rows, st)).astype(np.float32)
    f32map(hip, WS, old.size, old.reshape(-1))
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=k, opnd=0, ready=1, out=0, out_stride=st, epi=epi, out_opnd=op_at, out_opnd_stride=pair_w + 1,
                        tail=tail, tail_out=0, tail_stride=st)
    hip.linear_dev(WS, OP, WT, up(hip, spec.words()), 0, rows)
    got = read(hip, WS, 0, old.size).reshape(rows, st)
    with np.errstate(invalid="ignore"):
        y = x.astype(np.float64) @ f64(W).T
    body = y[:-1]
    # exact products; float32 sums of 3 k terms and shares at most: 3 k 2^-24 relative to the terms' root sum of squares.  float32
    # rows: the roundings of a sum are independent, so twice sqrt(3 k) 2^-24 (without the lowest piece: 1.1e-5, seen up to k = 2048)
    tol = 2 * np.sqrt(3 * k) * 2.0 ** -24 if wide else 3 * k * 2.0 ** -24
    each = lambda g, w: max(rel_l2(a, b) for a, b in zip(g, w))
    if epi < 2:
        want = body + (old[:-1, :n] if epi else 0.0)
        assert each(got[:-1, :n], want) < tol
        assert not np.isfinite(got[-1, :n]).any() and np.array_equal(got[:, n:], old[:, n:])
        return
    if tail:
        assert each(got[:-1, :tail], body[:, n - tail:]) < tol
    assert np.array_equal(got[:, tail:], old[:, tail:])
    head = body[1:, :n - tail].reshape(rows - 2, -1, 2, 16)
    want = (head[:, :, 0] / (1.0 + np.exp(-head[:, :, 0])) * head[:, :, 1]).reshape(rows - 2, pair_w)
    raw = hip.gather(OP, np.arange(op_at, op_at + rows * (pair_w + 1), dtype=np.uint32))
    pairs = raw.view(np.float32) if wide else f64(raw.view(np.uint16)[:raw.size])          # (a 16-bit map's values lie packed)
    pairs = pairs.reshape(rows, -1)[1:-1, :pair_w]
    # (a row of 2^-80: its pairs are products of two tiny numbers, 2^-161)
    assert each(pairs[1:], want[1:]) < (4 * tol if wide else 4 * tol + 2.0 ** -8)


@pytest.mark.parametrize("rows,n,k", [(1, 45, 320), (3, 45, 192), (3, 45, 320), (88, 131, 512), (40, 131, 4096), (300, 515, 3008)])
def test_infinite_weights_and_rows_in_float32(hip, rows, n, k):
    """Infinite weights meet values that one bfloat16 piece holds, that two do and that three do, zero and an infinity; in one
    launch, over shares of K, by the float32 instruction and in the one-row kernel: infinities keep their sign, and no number
    comes out exactly where float32 has none."""
    note(f"linear with infinities rows {rows} n {n} k {k}")
    rng = np.random.default_rng(n + k)
    W = rng.standard_normal((n, k)).astype(np.float32)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[:, 7], x[:, 8], x[:, 9], x[:, k - 1] = 1.0, -1.0 - 2.0 ** -12, 1.0 + 2.0 ** -20, -3.0
    x[rows // 2, 8] = 0.0
    x[rows - 1, 11] = -np.inf
    for j, col, v in ((0, 7, np.inf), (1, 7, -np.inf), (2, 8, np.inf), (3, 9, -np.inf), (4, 7, np.nan), (5, 7, np.inf), (n - 1, k - 1, np.inf), (6, 11, np.inf),
                      (7, 11, 0.0)):
        W[j, col] = v
    W[5, 9] = -np.inf
    W = f32_to_bf16(W)
    W[4, 7] = 0x7FC0
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, W.size)
    hip.scatter_contiguous(WT, 0, W.reshape(-1))
    hip.map_create_typed(OP, A.DTYPE_F32, 1, x.size)
    f32map(hip, WS, x.size + rows * n, x.reshape(-1))
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=k, src=0, src_stride=k, opnd=0, out=x.size, out_stride=n)
    hip.linear_dev(WS, OP, WT, up(hip, spec.words()), 0, rows)
    got = read(hip, WS, x.size, rows * n).reshape(rows, n)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ (W.astype(np.uint32) << 16).view(np.float32).astype(np.float64).T
    assert np.isinf(want).any() and np.isnan(want).any()
    for what in (np.isposinf, np.isneginf, np.isnan):
        assert np.array_equal(what(got), what(want)), what
    ok = np.isfinite(want)
    assert rel_l2(got[ok], want[ok]) < 3 * k * 2.0 ** -24


@pytest.mark.parametrize("rows,n,k", [(3, 33, 320), (88, 40, 4096), (40, 131, 8192), (300, 515, 1024)])
def test_the_lowest_piece_counts(hip, rows, n, k):
    """float32 rows whose products cancel down to their last bit: neighbouring columns hold 1 + 2^-23 and 1 under weights of
    1 and -1.  Every sum on the way is exact in float32, and so is the result."""
    note(f"linear lowest piece rows {rows} n {n} k {k}")
    rng = np.random.default_rng(k)
    x = np.ones((rows, k), np.float32)
    x[:, 0::2] += np.float32(2.0 ** -23) * rng.integers(0, 2, (rows, k // 2)).astype(np.float32)
    W = np.ones((n, k), np.float32)
    W[:, 1::2] = -1.0
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, W.size)
    hip.scatter_contiguous(WT, 0, f32_to_bf16(W).reshape(-1))
    hip.map_create_typed(OP, A.DTYPE_F32, 1, x.size)
    f32map(hip, WS, x.size + rows * n, x.reshape(-1))
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=k, src=0, src_stride=k, opnd=0, out=x.size, out_stride=n)
    hip.linear_dev(WS, OP, WT, up(hip, spec.words()), 0, rows)
    got = read(hip, WS, x.size, rows * n).reshape(rows, n)
    assert np.array_equal(got, np.repeat((x.astype(np.float64) @ W[0].astype(np.float64))[:, None], n, axis=1).astype(np.float32))


@pytest.mark.parametrize("rows", [1, 3])
def test_linear_argmax_takes_the_first_of_equals(hip, rows):
    note(f"linear argmax rows {rows}")
    n, k = 5003, 64
    rng = np.random.default_rng(2)
    p = Pair(hip, rows * k + rows * n + 64, wt=n * k, opnd=rows * k)
    W = f32_to_bf16(rng.standard_normal((n, k)).astype(np.float32))
    W[4001] = W[2003] = W[2002] = f32_to_bf16(np.full(k, 4.0, np.float32))
    p.put(WT, 0, W)
    x = np.abs(rng.standard_normal((rows, k)))
    p.put(WS, 0, x)
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=k, src=0, src_stride=k, out=rows * k, out_stride=n)
    p.call("linear_argmax_dev", WS, OP, WT, p.up(spec.words()), p.up(rows * (k + n) + np.arange(rows)), rows)
    a, b = p.read(WS, rows * (k + n), rows)
    assert a.tolist() == b.tolist() == [2002.0] * rows


@pytest.mark.parametrize("n", [1, 5, 255, 256, 257, 1000, 1023, 1024, 1025, 1028, 2051, 4096, 5000])
def test_linear_argmax_of_short_rows(hip, n):
    """Rows around what one float a thread covers, of 256 and of 1024 threads; two equals a wave apart."""
    note(f"linear argmax n {n}")
    rng = np.random.default_rng(n)
    W = f32_to_bf16(rng.uniform(-1, 1, (n, 64)).astype(np.float32))
    at = (n - 1, max(n - 66, 0))
    W[list(at)] = f32_to_bf16(np.ones(64, np.float32))
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, W.size)
    hip.scatter_contiguous(WT, 0, W.reshape(-1))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, 128)
    f32map(hip, WS, 128 + 2 * n + 2, np.ones(128, np.float32))
    spec = A.LinearSpec(w=0, n=n, k=64, k_stride=64, src=0, src_stride=64, out=128, out_stride=n)
    hip.linear_argmax_dev(WS, OP, WT, up(hip, spec.words()), up(hip, 128 + 2 * n + np.arange(2)), 2)
    assert read(hip, WS, 128 + 2 * n, 2).tolist() == [float(min(at))] * 2


@pytest.mark.parametrize("n,st", [(16384, 16384), (16385, 16388), (40000, 40001), (49152, 49152), (12296, 12300)])
def test_linear_argmax_of_long_rows(hip, n, st):
    """Runs that are read four floats at a time, their remainder, rows that do not start on sixteen bytes; equals far apart."""
    note(f"linear argmax n {n}")
    rows, k = 3, 64
    rng = np.random.default_rng(n)
    W = f32_to_bf16(rng.standard_normal((n, k)).astype(np.float32))
    big = f32_to_bf16(np.full(k, 4.0, np.float32))
    at = {0: [n - 1, 5000], 1: [n - 1], 2: [12288 + 7, 3, 9000]}
    x = np.zeros((rows, k), np.float32)
    for r, places in at.items():                  # row r sees only its own columns
        x[r, 16 * r:16 * r + 16] = 1.0
        for p in places:
            W[p, 16 * r:16 * r + 16] = big[:16]
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, W.size)
    hip.scatter_contiguous(WT, 0, W.reshape(-1))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, rows * k)
    f32map(hip, WS, rows * (k + st) + 16, x)
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=k, src=0, src_stride=k, out=rows * k, out_stride=st)
    tok = rows * (k + st) + np.arange(rows)
    hip.linear_argmax_dev(WS, OP, WT, up(hip, spec.words()), up(hip, tok), rows)
    assert read(hip, WS, int(tok[0]), rows).tolist() == [float(min(at[r])) for r in range(rows)]


def test_merge_norm(hip):
    note("merge norm")
    rows, dim, st = 5, 77, 80
    p = Pair(hip, 3 * rows * st + 2 * dim + 9)
    p.put(WS, 0, np.random.default_rng(0).standard_normal(p.n))
    spec = A.MergeSpec(a=0, b=rows * st, stride=st, wa=3 * rows * st, wb=3 * rows * st + dim, dst=2 * rows * st, dst_stride=st, dim=dim,
                       eps=1e-3, scale=0.5)
    p.call("merge_norm_dev", WS, p.up(spec.words()), rows)
    p.same(WS, 2 * rows * st, rows * st, 1e-5)


# ---- recurrences -----------------------------------------------------------------------------------------------------
def delta_pair(hip, H, KH, D, V, taps, rank, rows, seqs, strong, seed, off=1, pad=5):
    rng = np.random.default_rng(seed)
    n_ch = 2 * KH * D + H * V
    xs = n_ch + H + 2 * rank + 1
    at, pos = {}, 3
    for n, sz in (("x", rows * xs), ("a", rows * H * D), ("g", rows * H * V), ("o", rows * H * V), ("conv", n_ch * taps), ("A", H), ("dt", H * D)):
        at[n] = pos
        pos += sz
    ks = (rank + 63) // 64 * 64
    state = H * D * V + taps * n_ch + pad
    p = Pair(hip, pos + 16, wt=(H * D + H * V) * ks, opnd=2 * rows * ks, state=seqs * state)
    W = np.zeros((H * D + H * V, ks), np.uint16)
    W[:, :rank] = f32_to_bf16((rng.standard_normal((H * D + H * V, rank)) / np.sqrt(rank)).astype(np.float32))
    p.put(WT, 0, W)
    p.put(WS, at["conv"], rng.standard_normal(n_ch * taps) * 0.7)
    p.put(WS, at["A"], np.linspace(-3.0, 3.0 if strong else 0.5, H))
    p.put(WS, at["dt"], rng.uniform(-4, 2 if strong else 0, H * D))
    p.put(ST, 0, np.full(seqs * state, 7.0))        # what another sequence left behind
    low = lambda w, n, col, out: p.up(A.LinearSpec(w=w, n=n, k=rank, k_stride=ks, src=at["x"] + n_ch + H + col, src_stride=xs, opnd=0,
                                                   out=at[out], out_stride=n).words())
    dec, gate = low(0, H * D, 0, "a"), low(H * D * ks, H * V, rank, "g")
    c = at["conv"]
    spec = p.up(A.DeltaSpec(heads=H, kv_heads=KH, dim=D, vdim=V, taps=taps, x=at["x"], x_stride=xs, x_b=n_ch, cq=c, ck=c + KH * D * taps,
                            cv=c + 2 * KH * D * taps, a_log=at["A"], dt_bias=at["dt"], out=at["o"], out_stride=H * V, state_map=ST,
                            s_off=off, conv_off=off + H * D * V, seq_stride=state).words())
    fresh = lambda n: p.put(WS, at["x"], rng.standard_normal((n, xs)))

    def run(n_seq, m, seq0, pos0):
        fresh(n_seq * m)
        p.call("delta_rule_dev", WS, OP, WT, spec, dec, gate, n_seq, m, seq0, pos0)
        p.same(WS, at["o"], n_seq * m * H * V, 2e-5, f"outputs {n_seq}x{m} at {pos0}")
        p.same(WS, at["g"], n_seq * m * H * V, 2e-5, "gate")
        for i in range(n_seq):
            p.same(ST, (seq0 + i) * state + off, H * D * V, 2e-5, f"state of sequence {i} after {pos0 + m}")
    return run


@pytest.mark.parametrize("H,KH,D,V,taps,rank,strong", [
    (4, 2, 24, 20, 4, 11, False), (3, 3, 17, 33, 3, 5, True), (1, 1, 1, 1, 1, 1, False), (2, 1, 64, 16, 2, 70, True),
    (2, 2, 128, 144, 5, 16, False), (2, 1, 200, 40, 4, 128, True), (2, 1, 256, 64, 8, 30, False),
    (1, 1, 256, 250, 16, 20, False)])
def test_delta_rule(hip, H, KH, D, V, taps, rank, strong):
    note(f"delta rule H {H} KH {KH} D {D} V {V} taps {taps} rank {rank}")
    run = delta_pair(hip, H, KH, D, V, taps, rank, 40, 3, strong, seed=D)
    pos = 0
    for m in (2, 1, 17, 1, 1, 40, 16, 3):            # one sequence in slot 1, portions and single tokens in turn
        run(1, m, 1, pos)
        pos += m
    run(1, 33, 1, 0)                                 # the slot again, another sequence
    for i in range(3):
        run(1, 5, i, 0)
    for t in range(3):                               # one token of each of three sequences
        run(3, 1, 0, 5 + t)
    run(1, 1, 2, 0)                                  # a sequence that starts with a single token
    run(1, 2, 2, 1)


@pytest.mark.parametrize("H,KH,D,V,taps,rank,seqs", [
    (8, 8, 128, 128, 4, 128, 17), (8, 4, 128, 96, 3, 20, 17), (4, 2, 100, 132, 4, 140, 17), (9, 3, 17, 68, 4, 16, 16), (2, 1, 64, 256, 1, 64, 33),
    (8, 8, 129, 128, 4, 8, 17), (8, 8, 64, 128, 5, 8, 17)])
def test_delta_rule_steps_of_many_sequences(hip, H, KH, D, V, taps, rank, seqs):
    """Enough heads for four columns a thread, rows of state on 16 bytes; one column where dim or taps are beyond its registers."""
    note(f"delta rule of {seqs} sequences, H {H} KH {KH} D {D} V {V} taps {taps} rank {rank}")
    n_ch = 2 * KH * D + H * V
    run = delta_pair(hip, H, KH, D, V, taps, rank, seqs, seqs, False, seed=V, off=4, pad=8 + -(taps * n_ch) % 4)
    for pos in (0, 1, 2, 3, 9):
        run(seqs, 1, 0, pos)


def test_delta_rule_keeps_a_key_over_a_long_gap(hip):
    """A channel that does not decay holds a value through 300 tokens beside channels that forget within one."""
    note("delta rule, long gap")
    H, D, V, taps = 1, 16, 8, 1
    n_ch, rank = 2 * D + V, 1
    xs = n_ch + 1 + 2
    N = 300
    p = Pair(hip, N * xs + N * (D + 2 * V) + n_ch + 1 + D + 8, wt=(D + V) * 64, opnd=N * 64, state=D * V + n_ch)
    ao, go, oo = N * xs, N * (xs + D), N * (xs + D + V)
    cv = N * (xs + D + 2 * V)
    p.put(WS, cv, np.ones(n_ch))
    p.put(WS, cv + n_ch, [0.0])
    p.put(WS, cv + n_ch + 1, np.where(np.arange(D) < 4, -40.0, 6.0))       # decay 1 - e^-40, and e^-6 per token
    x = np.zeros((N, xs), np.float32)
    x[:, D + 8] = 9.0                                # filler keys: one of the channels that forget
    x[:, 2 * D:2 * D + V] = np.random.default_rng(0).standard_normal((N, V))
    x[:, n_ch] = 6.0
    x[0, D:2 * D] = 0
    x[0, D + 1] = 9.0                                # token 0 writes under channel 1
    x[-1, 1] = 9.0                                   # the last token asks for it
    p.put(WS, 0, x)
    low = lambda w, n, out: p.up(A.LinearSpec(w=w, n=n, k=1, k_stride=64, src=n_ch + 1, src_stride=xs, out=out, out_stride=n).words())
    spec = p.up(A.DeltaSpec(heads=1, kv_heads=1, dim=D, vdim=V, taps=taps, x=0, x_stride=xs, x_b=n_ch, cq=cv, ck=cv + D, cv=cv + 2 * D,
                            a_log=cv + n_ch, dt_bias=cv + n_ch + 1, out=oo, out_stride=V, state_map=ST, s_off=0, conv_off=D * V,
                            seq_stride=D * V + n_ch).words())
    p.call("delta_rule_dev", WS, OP, WT, spec, low(0, D, ao), low(D * 64, V, go), 1, N, 0, 0)
    p.same(WS, oo, N * V, 2e-5)
    got = p.read(WS, oo + (N - 1) * V, V)[0]
    v0 = x[0, 2 * D:2 * D + V]
    want = M.silu(v0.astype(float)) * M.sigmoid(6.0) * D ** -0.5
    assert np.abs(got - want).max() < 2e-3 * np.abs(want).max() + 1e-4


@pytest.mark.parametrize("H,D,V,rot", [(3, 20, 12, 12), (1, 8, 5, 8), (2, 64, 64, 0), (2, 192, 80, 64), (4, 128, 130, 128), (1, 256, 16, 2)])
def test_retention(hip, H, D, V, rot):
    note(f"retention H {H} D {D} V {V} rot {rot}")
    rng = np.random.default_rng(D + V)
    rows, xs = 40, H * (2 * D + V) + 7
    state = H * D * V + 3
    xo, oo = 2, 2 + rows * xs
    fr = oo + rows * H * V
    p = Pair(hip, fr + rot // 2 + H + 4, state=3 * state)
    p.put(ST, 0, np.full(3 * state, -3.0))
    p.put(WS, fr, 3000.0 ** (-2.0 * np.arange(rot // 2) / max(rot, 1)))
    p.put(WS, fr + rot // 2, 1.0 - 2.0 ** -np.linspace(1, 10, H))
    spec = p.up(A.RetentionSpec(heads=H, dim=D, vdim=V, rot_dims=rot, freq=fr, decay=fr + rot // 2, x=xo, x_stride=xs, x_q=1, x_k=1 + H * D,
                                x_v=1 + 2 * H * D, out=oo, out_stride=H * V, state_map=ST, s_off=2, seq_stride=state).words())

    def run(n_seq, m, seq0, pos):
        p.put(WS, xo, rng.standard_normal((n_seq * m, xs)))
        p.call("retention_dev", WS, spec, n_seq, m, seq0, pos)
        p.same(WS, oo, n_seq * m * H * V, 5e-5, f"outputs {n_seq}x{m} at {pos}")
        p.same(ST, seq0 * state + 2, H * D * V, 5e-5, f"state after {pos + m}")
    pos = 0
    for m in (1, 2, 16, 1, 33, 15, 40):
        run(1, m, 1, pos)
        pos += m
    run(1, 7, 1, 0)
    for i in (0, 2):
        run(1, 7, i, 0)
    run(3, 1, 0, 7)


CHUNK_ROWS = (16, 17, 33, 48, 64, 65, 96, 7)      # 1, 2, 3, 3, 4, 5, 6 and 1 chunks: two kernels, and every remainder of three


@pytest.mark.parametrize("D,V", [(24, 20), (100, 16), (180, 33)])
def test_walk_of_few_and_of_many_chunks(hip, D, V):
    note(f"walk over the chunks, D {D} V {V}")
    run = delta_pair(hip, 2, 1, D, V, 3, 9, 96, 2, False, seed=D)
    pos = 0
    for m in CHUNK_ROWS:
        run(1, m, 1, pos)
        pos += m
    rng = np.random.default_rng(V)
    H, xs = 2, 2 * (2 * D + V)
    state, oo = H * D * V, 96 * xs
    p = Pair(hip, oo + 96 * H * V + H, state=state)
    p.put(ST, 0, np.zeros(state))
    p.put(WS, oo + 96 * H * V, [0.9, 0.999])
    spec = p.up(A.RetentionSpec(heads=H, dim=D, vdim=V, rot_dims=0, freq=0, decay=oo + 96 * H * V, x=0, x_stride=xs, x_q=0, x_k=H * D,
                                x_v=2 * H * D, out=oo, out_stride=H * V, state_map=ST, s_off=0, seq_stride=state).words())
    pos = 0
    for m in CHUNK_ROWS:
        p.put(WS, 0, rng.standard_normal((m, xs)))
        p.call("retention_dev", WS, spec, 1, m, 0, pos)
        p.same(WS, oo, m * H * V, 5e-5, f"outputs of {m} at {pos}")
        p.same(ST, 0, state, 5e-5, f"state after {pos + m}")
        pos += m


# ---- attention -------------------------------------------------------------------------------------------------------
def attention_pair(hip, H, G, D, V, C, dtype, rows, seqs, seed, scale=0.25):
    rng = np.random.default_rng(seed)
    r8 = lambda n: (n + 7) // 8 * 8
    xs = H * D + G * (D + V) + 3
    oo = 4 + rows * xs
    ro = oo + rows * H * V
    kc, vc = G * C * r8(D), G * C * r8(V)
    p = Pair(hip, ro + 2 * H + 4, cache=seqs * (kc + vc + 8), dtype=dtype)
    p.put(WS, ro, np.concatenate([np.linspace(0.02, 1.5, H), rng.uniform(0.05, 0.6, H)]))
    spec = p.up(A.ChunkAttnSpec(heads=H, kv_heads=G, dim=D, vdim=V, chunk=C, x=4, x_stride=xs, x_q=1, x_k=1 + H * D, x_v=1 + (H + G) * D,
                                r1=ro, r2=ro + H, scale=scale, eps=1e-4, out=oo, out_stride=H * V, cache_map=CA, k_off=0, v_off=kc,
                                seq_stride=kc + vc + 8).words())
    tol = 3e-5 if dtype == "float32" else 2e-2

    def run(n_seq, m, seq0, pos, x=None):
        x = rng.standard_normal((n_seq * m, xs)) if x is None else x
        p.put(WS, 4, x)
        p.call("chunk_attention_dev", WS, spec, n_seq, m, seq0, pos)
        p.same(WS, oo, n_seq * m * H * V, tol, f"{n_seq}x{m} at {pos}")
        return p.read(WS, oo, n_seq * m * H * V)[0].reshape(n_seq * m, H, V)
    return run, xs, rng


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("H,G,D,V,C", [(4, 2, 16, 24, 10), (3, 3, 33, 7, 16), (1, 1, 1, 1, 1), (4, 1, 64, 48, 37), (2, 1, 136, 128, 70),
                                       (2, 2, 160, 200, 5), (2, 1, 256, 256, 100), (6, 3, 8, 80, 1000)])
def test_chunk_attention(hip, H, G, D, V, C, dtype):
    note(f"chunk attention H {H} G {G} D {D} V {V} chunk {C} {dtype}")
    run, _, _ = attention_pair(hip, H, G, D, V, C, dtype, 100, 3, seed=D + C)
    pos = 0
    for m in (2, 1, 3, 64, 1, 1, 100, 7, 33, 1):      # through chunk edges in portions and alone
        run(1, m, 1, pos)
        pos += m
    run(1, 13, 1, 0)                                  # the slot again
    for i in (0, 2):
        run(1, 13, i, 0)
    for t in range(4):
        run(3, 1, 0, 13 + t)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_chunk_attention_over_several_spans_of_keys(hip, dtype):
    """A chunk of 1500 tokens: a decoded token reads its keys in three spans; the edge to the next chunk comes after."""
    note(f"chunk attention, long chunk {dtype}")
    C = 1500
    run, _, _ = attention_pair(hip, 4, 2, 32, 40, C, dtype, 300, 1, seed=5, scale=0.6)
    pos = 0
    while pos < 1491:
        m = min(300, 1491 - pos)
        run(1, m, 0, pos)
        pos += m
        if pos in (300, 600, 1200):
            run(1, 1, 0, pos)
            pos += 1
    for pos in range(1491, 1504):
        run(1, 1, 0, pos)


def test_chunk_attention_of_sequences_beyond_2_to_the_32_elements(hip):
    """Two portions whose border lies at element 2^32 of the activation map (17 GB, two elements a pack): the second sequence's rows
    are read there and not at the map's start."""
    note("chunk attention across 2^32 elements")
    H, G, D, V, C, rows = 2, 1, 16, 16, 32, 5
    xs, top = H * D + G * (D + V), 1 << 32
    kv = G * C * D
    x = np.random.default_rng(3).standard_normal((2 * rows, xs)).astype(np.float32)
    x0 = top - rows * xs
    hip.map_create_typed(CA, A.DTYPE_F32, 1, 4 * kv)
    spec = lambda at: up(hip, A.ChunkAttnSpec(heads=H, kv_heads=G, dim=D, vdim=V, chunk=C, x=at, x_stride=xs, x_q=0, x_k=H * D, x_v=H * D + G * D, r1=8, r2=8,
                                              scale=0.25, eps=1e-4, out=64, out_stride=H * V, cache_map=CA, k_off=0, v_off=kv, seq_stride=2 * kv).words())
    got = []
    try:
        for packs, at in ((top // 2 + rows * xs, x0), (1 << 12, 2048)):
            hip.map_create_typed(WS, A.DTYPE_F32, 2, packs)
            hip.set_dtype(A.DTYPE_F32)
            assert hip.scatter_contiguous(WS, 4, np.full(4, 0.1, np.float32), n_locs=2) == 0
            assert hip.scatter_contiguous(WS, at // 2, x.reshape(-1), n_locs=x.size // 2) == 0
            hip.chunk_attention_seqs_dev(WS, spec(at), 2, rows, 0, 0)
            got.append(hip.gather(WS, np.arange(32, 32 + rows * H * V, dtype=np.uint32)).view(np.float32).copy())
    finally:
        f32map(hip, WS, 64)
    assert np.abs(got[1]).max() > 0.1 and np.array_equal(got[0], got[1])


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("cut", ["whole", "pairs", "alone"])
def test_a_standing_out_key_is_seen_inside_its_chunk_only(hip, dtype, cut):
    """Token j's key and token i's query are made to match strongly: i takes j's value when both lie in one chunk, and
    nothing of it when j is the last token ahead of i's chunk."""
    C, H, D, V = 12, 2, 16, 8
    note(f"standing-out key {dtype} {cut}")
    for j, i, seen in ((0, 11, True), (12, 23, True), (12, 12, True), (11, 12, False), (23, 24, False), (24, 30, True), (22, 24, False)):
        run, xs, rng = attention_pair(hip, H, H, D, V, C, dtype, 36, 1, seed=9, scale=1.0)
        x = rng.standard_normal((36, xs)) * 0.1
        v = rng.standard_normal((36, H, V))
        x[:, 1 + 2 * H * D:1 + 2 * H * D + H * V] = v.reshape(36, -1)
        x[i, 1:1 + H * D] = x[j, 1 + H * D:1 + 2 * H * D] = np.tile(np.eye(D)[3] * 6.0, H)
        step = {"whole": 36, "pairs": 2, "alone": 1}[cut]
        out = np.concatenate([run(1, step, 0, lo, x[lo:lo + step]) for lo in range(0, 36, step)])
        vn = v[j] / np.sqrt(np.mean(v[j] ** 2, axis=-1, keepdims=True) + 1e-4)
        assert (np.abs(out[i] - vn).max() < 0.05) == seen, (j, i)


# ---- models ----------------------------------------------------------------------------------------------------------
def tokens(cfg, n, seed=1):
    return [int(t) for t in np.random.default_rng(seed).integers(0, cfg["vocab"], n)]


def engine(hip, cfg, W, dtype="float32", **kw):
    return MixerEngine(hip, vomotar_config(cfg), W, A=A, dtype=dtype, **kw)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_model_whole_in_portions_and_token_by_token(hip, name, dtype):
    cfg = CONFIGS[name]
    W, n = weights(cfg, seed=2), 90
    toks = tokens(cfg, n)
    want = M.forward(cfg, floats(W), toks)
    for chunk in (256, 17, 1):
        note(f"model {name} {dtype} portions of {chunk}")
        eng = engine(hip, cfg, W, dtype, prefill_chunk=chunk)
        assert rel(eng.score("a", toks, range(n)), want) < TOL[dtype], chunk
    note(f"model {name} {dtype} uneven portions, slots freed and used again")
    eng = engine(hip, cfg, W, dtype, prefill_chunk=64, batch=2)
    rng = np.random.default_rng(4)
    for r in range(3):
        seq = {f"{r}{s}": tokens(cfg, 60, seed=30 + 2 * r + s) for s in range(2)}
        ref = {s: M.forward(cfg, floats(W), t) for s, t in seq.items()}
        at = dict.fromkeys(seq, 0)
        while any(a < 60 for a in at.values()):
            s = rng.choice([s for s in seq if at[s] < 60])
            m = int(min(rng.choice([1, 2, 3, 16, 25]), 60 - at[s]))
            assert rel(eng.score(s, seq[s][at[s]:at[s] + m], range(m)), ref[s][at[s]:at[s] + m]) < TOL[dtype], (r, s, at)
            at[s] += m
        for s in seq:
            eng.release(s)


def test_residual_after_every_layer(hip):
    """Each prefix of the stack as a model of its own: the residual rows after its last layer."""
    cfg = CONFIGS["odd"]
    W, toks = weights(cfg, seed=8), tokens(CONFIGS["odd"], 30)
    per_layer = []
    M.forward(cfg, floats(W), toks, per_layer)
    for n in range(1, len(cfg["layers"]) + 1):
        note(f"residual after {n} layers")
        eng = engine(hip, {**cfg, "layers": cfg["layers"][:n]}, W, prefill_chunk=30)
        eng.score("a", toks)
        assert rel(eng.read_rows("hidden", 30, cfg["width"]), per_layer[n - 1]) < 1e-5


@pytest.mark.parametrize("plan", [True, False])
def test_long_decoding_across_many_chunk_edges(hip, plan):
    cfg = config([delta(), par(size=7), par(size=50)], width=40, groups=2, vocab=64)
    W, toks = weights(cfg, seed=12), tokens(config([delta()], vocab=64), 400)
    note(f"long decoding plan={plan}")
    want = M.forward(cfg, floats(W), toks)
    eng = engine(hip, cfg, W, prefill_chunk=64, decode_plan=plan)
    got = [eng.score("a", toks[:5], range(5))] + [eng.score("a", [t], [0]) for t in toks[5:]]
    assert rel(np.concatenate(got), want) < 5e-5


def test_generation(hip):
    """Greedy tokens of the framework's loop, one step ahead of the read-back, equal those of the plain model; so do
    lockstep sequences; a prefix the state holds is reused."""
    cfg = CONFIGS["odd"]
    W, prompt = weights(cfg, seed=4), tokens(CONFIGS["odd"], 11)
    toks = list(prompt)
    for _ in range(40):
        toks.append(int(np.argmax(M.forward(cfg, floats(W), toks)[-1])))
    note("greedy generation")
    for kw in (dict(), dict(lookahead=False), dict(decode_plan=False), dict(sampling_mode="gpu_argmax")):
        eng = engine(hip, cfg, W, prefill_chunk=8, **kw)
        out, stats = eng.generate(prompt, GenerationConfig(max_tokens=40))
        assert out == toks[11:], kw
    assert stats["sampling_mode"] == "gpu_argmax"
    eng = engine(hip, cfg, W, prefill_chunk=8)
    eng.generate(prompt, GenerationConfig(max_tokens=40))
    follow = toks + tokens(cfg, 4, seed=8)
    more, st = eng.generate(follow, GenerationConfig(max_tokens=5), reuse_prefix=51)
    assert st["n_prompt_reused"] == 51
    assert more == engine(hip, cfg, W, prefill_chunk=8).generate(follow, GenerationConfig(max_tokens=5))[0]
    note("stop token")
    out, _ = eng.generate(prompt, GenerationConfig(max_tokens=40, eos_token_ids=(toks[20],)))
    assert out == toks[11:11 + toks[11:].index(toks[20])]
    note("lockstep")
    prompts = [tokens(cfg, 9, seed=20 + i) for i in range(4)]
    alone = [engine(hip, cfg, W, prefill_chunk=8).generate(p, GenerationConfig(max_tokens=30))[0] for p in prompts]
    out, _ = engine(hip, cfg, W, prefill_chunk=8, batch=4).generate_batch(prompts, 30)
    assert out == alone
    note("sampling")
    for kw in (dict(temperature=0.8, top_k=8, top_p=0.9, repeat_penalty=1.2, seed=3), dict(temperature=0.7, top_k=0, seed=3)):
        ref = MixerEngine(oracle.init(), vomotar_config(cfg), W, A=A, dtype="float32", prefill_chunk=8)
        want, _ = ref.generate(prompt, GenerationConfig(max_tokens=12, **kw))
        assert engine(hip, cfg, W, prefill_chunk=8).generate(prompt, GenerationConfig(max_tokens=12, **kw))[0] == want


@pytest.mark.parametrize("name,dtype,P,B", [("odd", "float32", 2, 3), ("odd", "float32", 17, 4), ("odd", "bfloat16", 16, 2),
                                            ("ones", "float32", 5, 4), ("wide", "bfloat16", 33, 3), ("wide", "float32", 34, 2)])
def test_prompts_that_share_the_weights(hip, name, dtype, P, B):
    """Several prompts in one pass (as many as 70 rows hold: all, some and one left over) and one by one."""
    note(f"prompts together {name} {dtype} {B} x {P}")
    cfg, got = CONFIGS[name], []
    prompts = [[int(t) for t in tokens(cfg, P, seed=40 + i)] for i in range(B)]
    for together in (True, False):
        eng = engine(hip, cfg, weights(cfg, seed=5), dtype=dtype, prefill_chunk=70, batch=B)
        assert eng._takes_portions()
        if not together:
            eng._takes_portions = lambda: False
        eng.reset()
        first = eng._prefill_each(prompts)
        eng._forward_chunk([1] * B, P, lockstep=True)           # what the states hold shows in the step that follows
        got.append((first, eng.read_rows("hidden", B)))
    assert got[0][0] == got[1][0] or dtype == "bfloat16"
    # (bfloat16: two best may change places, so each token's logit in float64 lies within the two roundings of the best one's, four
    # times a row's typical error for the largest of a few hundred)
    W = floats(weights(cfg, seed=5))
    for i, p in enumerate(prompts):
        z = M.forward(cfg, W, p)[-1]
        for first, _ in got:
            assert z.max() - z[first[i]] <= 2 * 4 * TOL[dtype] * np.sqrt(np.mean(z * z)), (i, first[i])
    # a pass of more rows takes other tiles, so float32 sums in another order, and bfloat16 operands that round the other way
    assert rel(got[0][1], got[1][1]) < TOL[dtype]


def test_trace_replay_and_command_line(hip, tmp_path):
    """The programs, each in a process of its own, on a model folder."""
    cfg = CONFIGS["odd"]
    W, toks = weights(cfg, seed=5), tokens(CONFIGS["odd"], 50)
    write_model(tmp_path, cfg, W)
    want = M.forward(cfg, floats(W), toks)
    steps = [([0, 33], [32, 4]), ([33, 35], []), ([35, 36], [0]), ([36, 50], [13])]
    lines = [json.dumps({"step": i, "entries": [{"id": "q", "tokens": toks[a:b], "want": w}], "end": ["q"] if b == 50 else []})
             for i, ((a, b), w) in enumerate(steps)]
    for dtype in ("bfloat16", "float32"):
        note(f"trace_run {dtype}")
        r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", str(tmp_path), "--dtype", dtype, "--out", str(tmp_path),
                            "--max-tokens", "64"], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=90)
        assert r.returncode == 0, r.stderr[-2000:]
        assert [ln for ln in r.stdout.splitlines() if ln.startswith("done")] == [f"done {i}" for i in range(4)]
        assert not os.path.exists(tmp_path / "1.f32")
        for i, ((a, b), w) in enumerate(steps):
            if w:
                got = np.fromfile(tmp_path / f"{i}.f32", "<f4").reshape(len(w), -1)
                assert rel(got, want[[a + k for k in w]]) < TOL[dtype]
    note("python -m adam_amd")
    r = subprocess.run([sys.executable, "-m", "adam_amd", str(tmp_path), "--tokens", ",".join(map(str, toks[:9])), "--max-tokens", "6",
                        "--dtype", "float32"], capture_output=True, text=True, timeout=90, cwd=ROOT)
    assert r.returncode == 0, r.stderr[-2000:]
    seq = list(toks[:9])
    for _ in range(6):
        seq.append(int(np.argmax(M.forward(cfg, floats(W), seq)[-1])))
    assert json.loads(r.stdout.splitlines()[-1])["tokens"] == seq[9:]


def test_calls_with_impossible_operands_are_refused(hip):
    """Ranges and sizes are checked on the host before anything is launched."""
    note("refused calls")
    eng = engine(hip, CONFIGS["ones"], weights(CONFIGS["ones"]))
    up = lambda s: hip.upload_dev(s.words())[0]
    mid, off, n, k, stride = eng._stacks[('head',)]
    good = dict(w=off, n=n, k=k, k_stride=stride, src=0, src_stride=k, out=0, out_stride=n)
    for bad in (dict(w=1 << 30), dict(k_stride=stride + 8), dict(groups=2), dict(epi=2), dict(out=(1 << 32) - 2), dict(n=0)):
        with pytest.raises(RuntimeError, match="-3"):
            hip.linear_dev(0, 2, mid, up(A.LinearSpec(**{**good, **bad})), 0, 1)
    with pytest.raises(RuntimeError, match="-3"):
        hip.linear_dev(0, 2, mid, hip.upload_dev(np.zeros(4, np.uint32))[0], 0, 1)       # not a spec
    r = dict(heads=1, dim=8, vdim=8, rot_dims=8, freq=0, decay=0, x=0, x_stride=32, x_q=0, x_k=8, x_v=16, out=0, out_stride=8, state_map=3,
             s_off=0, seq_stride=64)
    for bad in (dict(dim=300), dict(rot_dims=9), dict(seq_stride=63), dict(x_v=30), dict(state_map=9)):
        with pytest.raises(RuntimeError, match="-3"):
            hip.retention_dev(0, up(A.RetentionSpec(**{**r, **bad})), 1, 1, 0, 0)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("H,G,D,V,C,ms", [(64, 8, 40, 24, 900, (520, 260, 31, 200)), (6, 2, 128, 128, 290, (250, 33, 300)), (3, 1, 200, 72, 700, (300, 300))])
def test_chunk_attention_with_the_keys_parted_among_waves(hip, H, G, D, V, C, ms, dtype):
    """Portions that give every compute unit a workgroup of queries and ones that do not (the waves of a workgroup part the keys, some of
    them with none), across a chunk's edge as well."""
    note(f"chunk attention, keys parted, H {H} D {D} chunk {C} {dtype}")
    run, _, _ = attention_pair(hip, H, G, D, V, C, dtype, 520, 1, seed=C)
    pos = 0
    for m in ms:
        run(1, m, 0, pos)
        pos += m


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("H,G,D,V,C,rows,n_seq", [(16, 4, 64, 64, 400, 150, 9), (40, 8, 32, 48, 600, 290, 3)])
def test_a_portion_has_the_same_sums_beside_others(hip, H, G, D, V, C, rows, n_seq, dtype):
    """Portions that by themselves leave compute units idle (the waves of a workgroup part the keys) and together do not: outputs and
    caches are, bit for bit, those of each sequence alone."""
    note(f"chunk attention of {n_seq} sequences, H {H} D {D} chunk {C} {dtype}")
    rng = np.random.default_rng(C)
    xs, kc, vc = H * D + G * (D + V), G * C * D, G * C * V
    oo = n_seq * rows * xs
    ro = oo + n_seq * rows * H * V
    ss = kc + vc
    x = [rng.standard_normal(oo).astype(np.float32) for _ in range(2)]
    spec = lambda i: up(hip, A.ChunkAttnSpec(heads=H, kv_heads=G, dim=D, vdim=V, chunk=C, x=i * rows * xs, x_stride=xs, x_q=0, x_k=H * D, x_v=(H + G) * D, r1=ro,
                                             r2=ro + H, scale=0.25, eps=1e-4, out=oo + i * rows * H * V, out_stride=H * V, cache_map=CA, k_off=0, v_off=kc,
                                             seq_stride=ss).words())
    specs = [spec(i) for i in range(n_seq)]
    got = []
    for together in (False, True):
        hip.map_create_typed(CA, A.DTYPE_F32 if dtype == "float32" else A.DTYPE_BF16, 1, n_seq * ss)
        f32map(hip, WS, ro + 2 * H, np.concatenate([np.zeros(ro, np.float32), np.linspace(0.02, 1.5, H), np.full(H, 0.3)]).astype(np.float32))
        words = []
        for i, xi in enumerate(x):
            hip.scatter_contiguous(WS, 0, xi)
            if together:
                hip.chunk_attention_seqs_dev(WS, specs[0], n_seq, rows, 0, i * rows)
            else:
                for q in range(n_seq):
                    hip.chunk_attention_dev(WS, specs[q], 1, rows, q, i * rows)
            words.append(read(hip, WS, oo, n_seq * rows * H * V).view(np.uint32).copy())
        got.append(words)
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("k,n,rows,listed,branched", [(64, 40, 2, False, False), (200, 1003, 5, True, False), (4096, 517, 9, True, True), (4608, 70, 16, False, False),
                                                      (4672, 33, 6, True, False), (9216, 66, 3, True, True), (20000, 21, 2, True, False), (1000, 8, 1, True, False)])
def test_heads_of_several_rows_are_the_one_row_head(hip, k, n, rows, listed, branched):
    """adamah_hip_linear_argmax_rows_dev, at every number of rows a workgroup takes at a time (k bounds it): the best columns and the
    logits left behind are, but for the order of the norm's sums, those of the one-row head called for each row."""
    rng = np.random.default_rng(k + n)
    ks = -(-k // 64) * 64
    src_rows = rows + 3
    at = rng.permutation(src_rows)[:rows] if listed else np.arange(rows)
    w = np.zeros((n, ks), np.float32)
    w[:, :k] = rng.standard_normal((n, k)) / np.sqrt(k)
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, n * ks)
    hip.scatter_contiguous(WT, 0, f32_to_bf16(w.reshape(-1)))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, 8)
    x0, b0, wt, bw, bias, out, tok = np.cumsum([0] + [src_rows * k] * 2 + [k, k, n, n]).tolist()
    f32map(hip, WS, tok + src_rows, rng.standard_normal(tok + src_rows).astype(np.float32))
    s = dict(n=n, k=k, k_stride=ks, w=0, src=x0, src_stride=k, out=out, out_stride=n, groups=1, eps=1e-5, wt=wt, wt_len=k, wt_add=0.5, bias=bias, biased=1)
    if branched:
        s.update(branched=1, branch=b0, branch_stride=k, branch_wt=bw)
    note(f"heads of several rows k={k} n={n} rows={rows}")
    want, last = [], None
    for r in at:
        one = dict(s, src=x0 + int(r) * k)
        if branched:
            one["branch"] = b0 + int(r) * k
        hip.linear_argmax_dev(WS, OP, WT, up(hip, A.LinearSpec(**one).words()), up(hip, [tok]), 1)
        want.append(int(read(hip, WS, tok, 1)[0]))
        last = read(hip, WS, out, n)
    hip.scatter_contiguous(WS, out, np.zeros(n, np.float32))
    hip.linear_argmax_rows_dev(WS, OP, WT, up(hip, A.LinearSpec(**s).words()), up(hip, at) if listed else 0, up(hip, tok + 1 + np.arange(rows)), rows)
    assert [int(t) for t in read(hip, WS, tok + 1, rows)] == want
    got = read(hip, WS, out, n)
    assert np.abs(got - last).max() < 64 * 2.0 ** -24 * np.abs(last).max()
    with pytest.raises(RuntimeError):
        hip.linear_argmax_rows_dev(WS, OP, WT, up(hip, A.LinearSpec(**dict(s, src=tok)).words()), up(hip, at) if listed else 0, up(hip, tok + 1 + np.arange(rows)), rows)


def test_heads_of_rows_beyond_2_to_the_32_elements(hip):
    """Rows too long to go several at a time, the second one at element 2^32 of the activation map (17 GB, two elements a pack), with no
    list of rows."""
    note("heads of rows across 2^32 elements")
    k, ks, n, top = 20000, 20032, 40, 1 << 32
    rng = np.random.default_rng(6)
    w = np.zeros((n, ks), np.float32)
    w[:, :k] = rng.standard_normal((n, k))
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, n * ks)
    hip.scatter_contiguous(WT, 0, f32_to_bf16(w.reshape(-1)))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, 8)
    x = rng.standard_normal((2, k)).astype(np.float32)
    got = []
    try:
        for packs, at in ((top // 2 + k, top - k), (1 << 16, 4096)):
            hip.map_create_typed(WS, A.DTYPE_F32, 2, packs)
            hip.set_dtype(A.DTYPE_F32)
            assert hip.scatter_contiguous(WS, at // 2, x.reshape(-1), n_locs=x.size // 2) == 0
            s = A.LinearSpec(n=n, k=k, k_stride=ks, w=0, src=at, src_stride=k, out=64, out_stride=n, groups=1, eps=1e-5)
            hip.linear_argmax_rows_dev(WS, OP, WT, up(hip, s.words()), 0, up(hip, [0, 1]), 2)
            got.append(hip.gather(WS, np.arange(0, 32 + n // 2, dtype=np.uint32)).view(np.float32).copy())
    finally:
        f32map(hip, WS, 64)
    want = (x / np.sqrt((x.astype(np.float64) ** 2).mean(1, keepdims=True) + 1e-5)) @ bf16_to_f32(f32_to_bf16(w[:, :k].reshape(-1))).reshape(n, k).T.astype(np.float64)
    assert got[0][:2].tolist() == want.argmax(1).tolist() == got[1][:2].tolist()
    assert np.array_equal(got[0], got[1]) and rel_l2(got[0][64:64 + n], want[1]) < 1e-5
