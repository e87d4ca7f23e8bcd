"""Results that keep their words.  Ahead of a router a sum in another order is another choice of experts: 1e-6 in one layer's output moved
the logits of a mixture's prompt by 3e-2.  What these kernels add up in which order is therefore part of what they promise."""
import zlib

import numpy as np
import pytest

from adam_amd import adamah as A
from adam_amd.safetensors_file import f32_to_bf16
from gpu_util import note, up, f32map, read

pytestmark = pytest.mark.gpu

WS, OP, WT, ST = 0, 2, 1, 3


def places(first, **sizes):
    """Offsets of regions one behind the other, each on four floats; the last entry is the end."""
    at, pos = {}, first
    for name, n in sizes.items():
        at[name] = pos
        pos += (n + 3) // 4 * 4
    return at, pos


# ---- walks over the chunks ---------------------------------------------------------------------------------------------
def walk(hip, kind, H, G, D, V, seqs, rows):
    """CRC of the outputs and of the states behind a portion of `rows` tokens of each sequence, from a state that is not empty."""
    rng = np.random.default_rng(H * 1000 + D + rows)
    n, taps = seqs * rows, 4
    if kind == "delta":
        ch = 2 * G * D + H * V
        xs, state, rank = ch + H + 2 * 16, H * D * V + taps * ch, 16
        at, end = places(4, x=n * xs, a=n * H * D, g=n * H * V, o=n * H * V, conv=ch * taps, A=H, dt=H * D)
        hip.map_create_typed(WT, A.DTYPE_BF16, 1, (H * D + H * V) * 64)
        W = np.zeros((H * D + H * V, 64), np.float32)
        W[:, :rank] = rng.standard_normal((H * D + H * V, rank)) / 4
        hip.scatter_contiguous(WT, 0, f32_to_bf16(W).reshape(-1))
        hip.map_create_typed(OP, A.DTYPE_BF16, 1, 2 * n * 64)
    elif kind == "retention":
        xs, state = H * (2 * D + V), H * D * V
        at, end = places(4, x=n * xs, o=n * H * V, decay=H)
    else:
        ch = H * V + 2 * G * D
        xs, state = H * V + ch + H, H * D * V + taps * ch
        at, end = places(4, x=n * xs, o=n * H * V, conv=ch * taps, b=ch, dt=H, A=H, D=H)
    hip.set_dtype(A.DTYPE_F32)
    put = lambda m, off, v: hip.scatter_contiguous(m, off, np.ascontiguousarray(v, np.float32).reshape(-1))
    hip.map_create(WS, 1, end + 4)
    hip.map_create(ST, 1, seqs * state)
    put(WS, at["x"], rng.standard_normal(n * xs, dtype=np.float32))
    put(ST, 0, rng.standard_normal(seqs * state, dtype=np.float32))
    if "conv" in at:
        put(WS, at["conv"], rng.standard_normal(ch * taps, dtype=np.float32) * np.float32(0.7))
        put(WS, at["A"], np.linspace(-3.0, 0.5, H))
        put(WS, at["dt"], rng.standard_normal(H * D if kind == "delta" else H, dtype=np.float32))
    if kind == "delta":
        low = lambda w, m, col, out: up(hip, A.LinearSpec(w=w, n=m, k=rank, k_stride=64, src=at["x"] + ch + H + col, src_stride=xs, opnd=0,
                                                          out=at[out], out_stride=m).words())
        dec, gate, c = low(0, H * D, 0, "a"), low(H * D * 64, H * V, rank, "g"), at["conv"]
        spec = A.DeltaSpec(heads=H, kv_heads=G, dim=D, vdim=V, taps=taps, x=at["x"], x_stride=xs, x_b=ch, cq=c, ck=c + G * D * taps,
                           cv=c + 2 * G * D * taps, a_log=at["A"], dt_bias=at["dt"], out=at["o"], out_stride=H * V, state_map=ST, s_off=0,
                           conv_off=H * D * V, seq_stride=state)
        hip.delta_rule_seqs_dev(WS, OP, WT, up(hip, spec.words()), dec, gate, seqs, rows, 0, 9)
    elif kind == "retention":
        put(WS, at["decay"], 1.0 - 2.0 ** -np.linspace(3, 9, H))
        spec = A.RetentionSpec(heads=H, dim=D, vdim=V, rot_dims=0, freq=0, decay=at["decay"], x=at["x"], x_stride=xs, x_q=0, x_k=H * D,
                               x_v=2 * H * D, out=at["o"], out_stride=H * V, state_map=ST, s_off=0, seq_stride=state)
        hip.retention_seqs_dev(WS, up(hip, spec.words()), seqs, rows, 0, 9)
    else:
        put(WS, at["b"], rng.standard_normal(ch, dtype=np.float32))
        put(WS, at["D"], rng.standard_normal(H, dtype=np.float32))
        spec = A.StateSpaceSpec(heads=H, groups=G, state=D, vdim=V, taps=taps, x=at["x"], x_stride=xs, x_c=H * V, x_dt=H * V + ch, conv=at["conv"],
                                conv_b=at["b"], dt_bias=at["dt"], a_log=at["A"], skip=at["D"], out=at["o"], out_stride=H * V, state_map=ST,
                                s_off=0, conv_off=H * D * V, seq_stride=state)
        hip.state_space_dev(WS, up(hip, spec.words()), seqs, rows, 0, 9)
    return [f"{zlib.crc32(read(hip, m, off, size).tobytes()):08x}" for m, off, size in ((WS, at["o"], n * H * V), (ST, 0, seqs * state))]


# Recorded with this library's walks of four waves (W S and Q S one product behind the other by wave, the waves' parts added as
# (0 + 1) + (2 + 3), the chunk's own products behind that sum, in order) and ROCm 7.2's expf and exp2f.
WALKS = {
    ("delta", 2, 1, 24, 20, 1, 7): "98665651 5837517d",
    ("delta", 3, 3, 100, 33, 2, 77): "7b2191fd f986b388",
    ("delta", 2, 2, 128, 16, 1, 170): "76175282 56bba8ef",
    ("delta", 4, 2, 180, 40, 1, 65): "a5a30d12 b19d4695",
    ("delta", 1, 1, 256, 64, 1, 50): "387a19e7 42e9a6b8",
    ("delta", 16, 16, 64, 64, 5, 40): "493b53b8 b70306d0",
    ("delta", 16, 8, 64, 64, 9, 150): "dbd6aaa7 f7dfe3cb",
    ("delta", 16, 16, 128, 100, 3, 150): "049324e3 55f86e0d",
    ("delta", 20, 20, 192, 100, 2, 90): "83ab5318 3183c87b",
    ("delta", 20, 20, 256, 100, 2, 90): "202dd06b ffd35d1a",
    ("retention", 2, 0, 24, 20, 1, 7): "0fb25b32 c4b37fec",
    ("retention", 3, 0, 100, 33, 2, 77): "aea11587 7cbdea86",
    ("retention", 2, 0, 180, 40, 1, 65): "5fe31224 6db0836f",
    ("retention", 1, 0, 256, 64, 1, 50): "ff24d1bc 2825e1d2",
    ("retention", 16, 0, 64, 64, 9, 150): "2a6fe897 cd358e76",
    ("retention", 16, 0, 128, 100, 5, 150): "8367e4e7 6f540275",
    ("retention", 20, 0, 192, 100, 2, 90): "cc94d0f8 bd48135c",
    ("retention", 20, 0, 250, 100, 2, 90): "175f578f d42d027b",
    ("space", 2, 1, 24, 20, 1, 7): "e1e179c3 23146a8a",
    ("space", 4, 2, 100, 33, 1, 77): "b600b15f 33b552db",
    ("space", 4, 4, 180, 40, 1, 65): "6e7f7d9b 4d4ec6db",
    ("space", 2, 1, 256, 64, 1, 50): "a40188e0 b260f797",
    ("space", 130, 10, 64, 100, 1, 150): "a9b6b790 e153d87c",
    ("space", 130, 10, 128, 100, 1, 150): "46180f9e 57ce785f",
    ("space", 64, 8, 192, 100, 1, 90): "db1be02e 968e6ca1",
    ("space", 64, 8, 250, 100, 1, 90): "a74b3f51 e9cf6a5c",
}


@pytest.mark.parametrize("case", WALKS, ids=lambda c: "-".join(map(str, c)))
def test_walk_keeps_its_words(hip, case):
    """One chunk to ten, one head to more workgroups than two a compute unit, every tile count, ragged in all directions."""
    note(f"words of a walk {case}")
    assert walk(hip, *case) == WALKS[case].split()


# ---- norms of operand rows -------------------------------------------------------------------------------------------------
fma = lambda a, b, c: (np.float64(1) * a * b + c).astype(np.float32)


def wave_sum(v):
    """[..., 64] lanes -> [...]: lane ^ 32, ^ 16, ... ^ 1."""
    while v.shape[-1] > 1:
        v = v[..., :v.shape[-1] // 2] + v[..., v.shape[-1] // 2:]
    return v[..., 0]


def in_turn(v):
    """Along the last axis, one behind the other."""
    t = np.zeros(v.shape[:-1], np.float32)
    for i in range(v.shape[-1]):
        t = t + v[..., i]
    return t


def inverse(total, n, eps):
    return np.float32(1) / np.sqrt(total / np.float32(n) + np.float32(eps))


def normed(x, groups, eps):
    """Rows by groups of whole waves' worth (four columns a lane) or one: 256 columns a wave, the waves' sums in turn."""
    y = np.empty_like(x)
    gs = x.shape[1] // groups
    for i, row in enumerate(x):
        g = np.zeros((groups, (gs + 255) // 256 * 256), np.float32)
        g[:, :gs] = row.reshape(groups, gs)
        q, ss = g.reshape(groups, -1, 64, 4), np.float32(0)
        for e in range(4):
            ss = fma(q[..., e], q[..., e], ss)
        y[i] = (row.reshape(groups, gs) * inverse(in_turn(wave_sum(ss)), gs, eps)[:, None]).reshape(-1)
    return y


@pytest.mark.parametrize("rows,k,groups", [(rows, *shape) for rows in (1, 3, 600) for shape in
                                           [(1024, 1), (2048, 1), (4096, 1), (4096, 2), (4096, 4), (2052, 1), (8192, 1), (8192, 8), (4100, 1)]
                                           if rows < 512 or shape[0] <= 4096])             # (many longer rows: another form)
def test_norm_adds_up_in_turn(hip, rows, k, groups):
    """What the product keeps of its normed row, to the bit."""
    note(f"words of a norm, rows {rows} k {k} groups {groups}")
    rng = np.random.default_rng(k + groups)
    ks, n = (k + 63) // 64 * 64, 40
    at, end = places(4, x=rows * k, keep=rows * k, out=rows * n)
    x = rng.standard_normal((rows, k), dtype=np.float32)
    f32map(hip, WS, end, x, at["x"])
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, n * ks)
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, rows * ks)
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=ks, src=at["x"], src_stride=k, groups=groups, eps=1e-6, keep=at["keep"], keep_stride=k, kept=1,
                        opnd=0, out=at["out"], out_stride=n)
    hip.linear_dev(WS, OP, WT, up(hip, spec.words()), 0, rows)
    at_most = min(rows, 20)
    got = read(hip, WS, at["keep"], rows * k).reshape(rows, k)[-at_most:]
    assert np.array_equal(got.view(np.uint32), normed(x[-at_most:], groups, 1e-6).view(np.uint32))


@pytest.mark.parametrize("k,shift,twice", [(1024, 0, True), (2048, 0, True), (2048, 1, False), (1501, 3, True), (4096, 0, True), (4095, 0, False)])
def test_branched_norms_of_one_row_add_up_by_thread(hip, k, shift, twice):
    """x + the branch's row behind a norm of its own, then a norm: 512 threads, each its columns in turn, then wave by wave."""
    note(f"words of a branched norm, k {k} shift {shift} twice {twice}")
    rng = np.random.default_rng(k)
    ks, n, eps = (k + 63) // 64 * 64, 24, np.float32(1e-5)
    at, end = places(4, **{name: k + 4 for name in ("x", "b", "bw", "wt", "res", "keep")}, out=n)
    at = {name: off + (shift if name != "out" else 0) for name, off in at.items()}
    x, b, bw, wt = (rng.standard_normal(k, dtype=np.float32) for _ in range(4))
    f32map(hip, WS, end + 4)
    for name, v in (("out", np.zeros(n)), ("keep", np.zeros(k)), ("res", np.zeros(k)), ("wt", wt), ("bw", bw), ("b", b), ("x", x)):
        hip.scatter_contiguous(WS, at[name], np.ascontiguousarray(v, np.float32))
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, n * ks)
    spec = A.LinearSpec(w=0, n=n, k=k, k_stride=ks, src=at["x"], src_stride=k, groups=1, eps=eps, wt=at["wt"], wt_len=k if twice else 0, wt_add=0.5,
                        branched=2, branch=at["b"], branch_stride=k, branch_wt=at["bw"], res_out=at["res"], res_stride=k,
                        keep=at["keep"], keep_stride=k, kept=1, out=at["out"], out_stride=n)
    hip.linear_dev(WS, OP, WT, up(hip, spec.words()), 0, 1)

    def norm(v):
        ss = np.zeros(512, np.float32)
        for c in np.pad(v, (0, -k % 512)).reshape(-1, 512):
            ss = fma(c, c, ss)
        return inverse(in_turn(wave_sum(ss.reshape(8, 64))), k, eps)
    half = np.float32(0.5)
    res = fma(b * norm(b), half + bw, x)
    kept = res * norm(res) * (half + wt if twice else np.float32(1))
    for name, want in (("res", res), ("keep", kept)):
        assert np.array_equal(read(hip, WS, at[name], k).view(np.uint32), want.view(np.uint32)), name


# ---- products of few rows ----------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("k", [2112, 2560, 3008, 4096])
@pytest.mark.parametrize("rows,epi", [(2, 0), (16, 1), (19, 0), (32, 0)])
def test_a_narrow_product_does_not_hang_on_its_width(hip, rows, epi, k):
    """Up to 16 matrix rows a compute unit the sums are those of sixteen waves, whichever kernel takes the width: 13 of them, 15 of them and
    a few rows of the same matrix, the same words."""
    note(f"words of a narrow product, rows {rows} k {k} epi {epi}")
    rng = np.random.default_rng(k + rows)
    cu = 256
    widths = (15 * cu, 13 * cu, 6 * cu + 5, 33)
    n = widths[0]
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, n * k)
    hip.scatter_contiguous(WT, 0, f32_to_bf16(rng.standard_normal(n * k, dtype=np.float32)))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, rows * k)
    hip.scatter_contiguous(OP, 0, f32_to_bf16(rng.standard_normal(rows * k, dtype=np.float32)))
    old = rng.standard_normal((rows, n), dtype=np.float32)
    got = []
    for w in widths:
        f32map(hip, WS, rows * n, old)
        spec = A.LinearSpec(w=0, n=w, k=k, k_stride=k, opnd=0, ready=1, out=0, out_stride=n, epi=epi)
        hip.linear_dev(WS, OP, WT, up(hip, spec.words()), 0, rows)
        got.append(read(hip, WS, 0, rows * n).reshape(rows, n))
    for w, y in zip(widths[1:], got[1:]):
        assert np.array_equal(y[:, :w].view(np.uint32), got[0][:, :w].view(np.uint32)), w
        assert np.array_equal(y[:, w:], old[:, w:])


@pytest.mark.parametrize("rows,k", [(2, 1152), (16, 1216), (19, 2112), (32, 2624), (12, 3072), (17, 3648), (9, 1472)])
def test_a_wide_product_does_not_hang_on_its_width(hip, rows, k):
    """Beyond 16 matrix rows a compute unit the sums are those of eight waves: two kernels share the widths, the same words."""
    note(f"words of a wide product, rows {rows} k {k}")
    rng = np.random.default_rng(k + rows)
    widths = tuple(256 * w + 5 for w in (36, 31, 24, 16))
    n = widths[0]
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, n * k)
    hip.scatter_contiguous(WT, 0, f32_to_bf16(rng.standard_normal(n * k, dtype=np.float32)))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, rows * k)
    hip.scatter_contiguous(OP, 0, f32_to_bf16(rng.standard_normal(rows * k, dtype=np.float32)))
    f32map(hip, WS, rows * n)
    got = []
    for w in widths:
        hip.linear_dev(WS, OP, WT, up(hip, A.LinearSpec(w=0, n=w, k=k, k_stride=k, opnd=0, ready=1, out=0, out_stride=n).words()), 0, rows)
        got.append(read(hip, WS, 0, rows * n).reshape(rows, n))
    for w, y in zip(widths[1:], got[1:]):
        assert np.array_equal(y[:, :w].view(np.uint32), got[0][:, :w].view(np.uint32)), w


# ---- products of one row -------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("k", [960, 1024, 2100, 4096, 4160])
@pytest.mark.parametrize("kind", ["norm", "branch", "pairs"])
def test_one_row_does_not_hang_on_the_workgroups(hip, kind, k):
    """A few workgroups beyond one a compute unit, more of them, and none: what a matrix row gives is the same word, whether its wave has it
    as its first task or its second."""
    note(f"words of one row, {kind} k {k}")
    rng = np.random.default_rng(k)
    ks = (k + 63) // 64 * 64
    widths = [2 * 8 * w for w in (300, 290, 288, 264, 258, 256, 140)]          # rows: two a wave, eight waves
    n = widths[0]
    at, end = places(4, x=k, wt=k, b=k, bw=k, res=k, out=n)
    W = f32_to_bf16(rng.standard_normal((n, ks), dtype=np.float32))
    W[:, k:] = 0
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, n * ks)
    hip.scatter_contiguous(WT, 0, W.reshape(-1))
    hip.map_create_typed(OP, A.DTYPE_BF16, 1, ks)
    f32map(hip, WS, end, rng.standard_normal(end, dtype=np.float32))
    got = []
    for w in widths:
        spec = dict(w=0, n=w, k=k, k_stride=ks, src=at["x"], src_stride=k, groups=1, eps=1e-5, wt=at["wt"], wt_len=k, opnd=0, out=at["out"], out_stride=w)
        if kind != "norm":
            spec.update(branched=2, branch=at["b"], branch_stride=k, branch_wt=at["bw"], res_out=at["res"], res_stride=k)
        if kind == "pairs":
            spec.update(epi=2, out_opnd=0, out_opnd_stride=w // 2)
        hip.linear_dev(WS, OP, WT, up(hip, A.LinearSpec(**spec).words()), 0, 1)
        got.append(read(hip, WS, at["out"], w // 2 if kind == "pairs" else w))
    x, b, bw, wt = (read(hip, WS, at[name], k).astype(np.float64) for name in ("x", "b", "bw", "wt"))
    if kind != "norm":
        x = x + b / np.sqrt(np.mean(b * b) + 1e-5) * bw
    y = (W.astype(np.uint32) << 16).view(np.float32)[:, :k].astype(np.float64) @ (x / np.sqrt(np.mean(x * x) + 1e-5) * wt)
    if kind == "pairs":
        g, u = y.reshape(-1, 2, 16).transpose(1, 0, 2).reshape(2, -1)
        y = g / (1 + np.exp(-g)) * u
    assert np.linalg.norm(got[0] - y) < 1e-5 * np.linalg.norm(y)               # sums of k terms in float32, by 64 lanes: about 1e-6
    for w, v in zip(widths[1:], got[1:]):
        assert np.array_equal(v.view(np.uint32), got[0][:len(v)].view(np.uint32)), w


# ---- one row through the experts -----------------------------------------------------------------------------------------------
@pytest.mark.parametrize("E,I,top,ff,shared,width,epi", [(4, 0, 4, 1024, 2048, 300, 0), (3, 1, 4, 1000, 2500, 2070, 1), (2, 2, 4, 512, 0, 70, 0),
                                                         (7, 1, 8, 576, 2048, 33, 1), (4, 4, 2, 448, 2112, 50, 0), (1, 1, 2, 2048, 4096, 4200, 0),
                                                         (2, 6, 2, 1536, 2048, 100, 1), (8, 0, 1, 64, 128, 40, 0)])
def test_one_row_of_the_experts_adds_up_in_the_order_of_its_columns(hip, E, I, top, ff, shared, width, epi):
    """Equal logits, so that every weight is a power of two; the correction decides who is chosen and in which order.  A lane has columns
    8 lane .. of every 512 of the chosen experts' activations (weighted) and the shared expert's behind them, in turn."""
    note(f"words of the experts, {E} + {I} top {top} ff {ff} shared {shared} width {width} epi {epi}")
    rng = np.random.default_rng(E * ff + width)
    n, ks, F, F16, S = E + I, (width + 63) // 64 * 64, (ff + 63) // 64 * 64, (ff + 15) // 16 * 16, (shared + 63) // 64 * 64
    assert n & (n - 1) == 0
    at, end = places(4, h=width, log=n + 1, corr=n, out=width, act=top * F, sact=max(S, 4))
    gu, dn, sd = 0, E * 2 * F16 * ks, E * 2 * F16 * ks + E * width * F
    bf = lambda w: (w.astype(np.uint32) << 16).view(np.float32)
    W = f32_to_bf16(rng.standard_normal((E, 2 * F16, ks), dtype=np.float32) / np.float32(np.sqrt(width)))
    W[:, :, width:] = 0
    D = f32_to_bf16(rng.standard_normal((E, width, F), dtype=np.float32))
    sh = f32_to_bf16(rng.standard_normal((width, S), dtype=np.float32))
    hip.map_create_typed(WT, A.DTYPE_BF16, 1, sd + width * S + 8)
    for off, w in ((gu, W), (dn, D)) + (((sd, sh),) if shared else ()):
        hip.scatter_contiguous(WT, off, w.reshape(-1))
    x, old = rng.standard_normal(width, dtype=np.float32), rng.standard_normal(width, dtype=np.float32)
    corr, sact = rng.permutation(n).astype(np.float32), rng.standard_normal(max(S, 4), dtype=np.float32)
    f32map(hip, WS, end + 4)
    log = np.zeros(n + 1)
    log[n] = 120.0                                             # the shared expert's gate: exactly one
    for name, v in (("h", x), ("log", log), ("corr", corr), ("out", old), ("sact", sact)):
        hip.scatter_contiguous(WS, at[name], np.ascontiguousarray(v, np.float32))
    spec = A.ExpertsSpec(experts=E, identity=I, top=top, ff=ff, ff_stride=F, width=width, k_stride=ks, gate_up=gu, gate_up_step=2 * F16 * ks,
                         down=dn, down_step=width * F, logits=at["log"], logits_stride=n + 1, correction=at["corr"], x=at["h"], x_stride=width,
                         act=at["act"], shared_ff=shared, shared_ff_stride=S, shared_down=sd, shared_act=at["sact"], out=at["out"],
                         out_stride=width, epi=epi)
    hip.experts_dev(WS, OP, WT, up(hip, spec.words()), 0, 1)
    first = [int(e) for e in np.argsort(-corr)[:top]]
    chosen, p = [e for e in first if e < E], np.float32(1.0 / n)
    act = read(hip, WS, at["act"], top * F).reshape(top, F)
    cols = [np.where(np.arange(F) < ff, act[j] * p, np.float32(0)) for j in range(len(chosen))]
    mats = [bf(D[e]) for e in chosen]
    if shared:
        cols.append(np.where(np.arange(S) < shared, sact[:S], np.float32(0)))
        mats.append(bf(sh))
    a = np.zeros((width, 64), np.float32)
    if cols:
        v, m = np.concatenate(cols), np.concatenate(mats, axis=1)
        pad = -len(v) % 512
        for b, w in zip(np.pad(v, (0, pad)).reshape(-1, 64, 8), np.pad(m, ((0, 0), (0, pad))).reshape(width, -1, 64, 8).transpose(1, 0, 2, 3)):
            for e in range(8):
                a = fma(w[..., e], b[:, e], a)
    back = np.float32(p * (top - len(chosen)))
    want = fma(np.broadcast_to(back, x.shape), x, wave_sum(a))
    want = old + want if epi else want
    assert np.array_equal(read(hip, WS, at["out"], width).view(np.uint32), want.view(np.uint32))
