"""The fused attention launches against float64 where fewer bits of P, or of
its exponent, would show: a heavy key without a value, scores far from zero,
and every accepted tile shape with a tolerance of the output's rounding."""
import numpy as np
import pytest

from ktir_cpu_amd import configs
from ktir_cpu_amd import runtime as rt
from oracle.interp import bf16_bits, bf16_from_bits
from tests.test_oracle_example_pins import PA_FN

pytestmark = pytest.mark.gpu

# rows, keys, columns of the dense kernel's tiles of 64 or 128
SHAPES = [(m, n, d) for m in (64, 128) for n in (64, 128) for d in (64, 128) if (m, n, d) != (128, 128, 128)]
# half a unit of the output type, relative; half the spacing of its smallest values
HALF = {"f16": (2.0 ** -11, 2.0 ** -25), "bf16": (2.0 ** -8, 0.0), "f32": (2.0 ** -24, 0.0)}


def _bits(x, dt):
    return bf16_bits(np.asarray(x, np.float32)) if dt == "bf16" else np.asarray(x, np.float16)


def _f64(x):
    return (bf16_from_bits(x) if x.dtype == np.uint16 else x).astype(np.float64)


def _prepare(src, fn, kw):
    from ktir_cpu_amd.interpreter import KTIRInterpreter
    it = KTIRInterpreter()
    it.load(src)
    prep = it.prepare(fn, **kw)
    (d,) = [x[1] for x in prep.plan.launches if x[0] in ("attn", "pattn")]
    return prep, d


def _device(ptr, n):
    out = np.empty(n, np.float32)
    rt.check(rt.lib().ktir_memcpy_d2h(out.ctypes.data, ptr, out.nbytes), "ktir_memcpy_d2h")
    return out.astype(np.float64)


def _dense(q, k, v, scale, causal):
    """float64 attention, and the sum of P |V| that a relative error of P acts on."""
    s = np.einsum("bhid,bhjd->bhij", q, k) * scale
    if causal:
        s = np.where(np.tril(np.ones(s.shape[-2:])) > 0, s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    return p @ v, p @ np.abs(v)


def _near(got, want, dt, spread, p_err=2.0 ** -21):
    """One rounding to `dt`, after errors of `p_err` of every P (f32
    exponentials and sums of them: a few units each)."""
    half, tiny = HALF[dt]
    assert (np.abs(got - want) <= half * np.abs(want) * 1.001 + tiny + p_err * spread).all(), \
        (np.abs(got - want) / (half * np.abs(want) + tiny + p_err * spread)).max()


def _exp_err(gap):
    """Of an f32 exponential of -gap: its argument times log2 e is off by up to
    2^-24 of itself, the hardware's exp2 by a unit; the same again for l."""
    return gap * 2.0 ** -23 + 2.0 ** -21


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("causal,S", [(True, 384), (False, 256), (True, 128)])
@pytest.mark.parametrize("M,N,D", SHAPES)
def test_tiles_of_every_shape(M, N, D, causal, S, dt):
    rng = np.random.default_rng(M + N + D)
    q, k, v = (_bits(rng.standard_normal((1, 3, S, D)), dt) for _ in range(3))
    prep, d = _prepare(configs.flash_attention(1, 3, S, D, M, dt, causal, N), "flash_attention",
                       dict(q_ptr=q, k_ptr=k, v_ptr=v, o_ptr=np.zeros_like(q), scale=D ** -0.5))
    assert (d.M, d.N, d.D) == (M, N, D) and dict(prep.plan.counts()) == {"attn": 1}
    want, spread = _dense(_f64(q), _f64(k), _f64(v), D ** -0.5, causal)
    _near(_f64(prep.outputs()["o_ptr"]), want, dt, spread)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,D", [(64, 128, 64), (128, 64, 128)])
def test_tiles_of_wider_rows(M, N, D, dt):
    """Q, K, V and O as columns of wider arrays: rows 8 elements further apart."""
    rng = np.random.default_rng(5)
    S, W = 2 * max(M, N), D + 8
    wide = [_bits(rng.standard_normal((1, 2, S, W)), dt) for _ in range(3)]
    src = configs.flash_attention(1, 2, S, D, M, dt, False, N)
    old, new = f"sizes: [1, 2, {S}, {D}], strides: [{2 * S * D}, {S * D}, {D}, 1]", \
        f"sizes: [1, 2, {S}, {D}], strides: [{2 * S * W}, {S * W}, {W}, 1]"
    assert src.count(old) == 4
    prep, d = _prepare(src.replace(old, new), "flash_attention",
                       dict(zip(("q_ptr", "k_ptr", "v_ptr"), wide), o_ptr=np.zeros_like(wide[0]), scale=D ** -0.5))
    assert (d.q_row, d.k_row, d.v_row, d.o_row) == (W,) * 4
    got = _f64(prep.outputs()["o_ptr"])
    want, spread = _dense(*(_f64(x)[..., :D] for x in wide), D ** -0.5, False)
    _near(got[..., :D], want, dt, spread)
    assert (got[..., D:] == 0).all()


def _sink(S, D, at, gap, value):
    """q, k, v of one head: key `at` scores `gap` more than the others and has V = 0."""
    q, k = np.zeros((S, D)), np.zeros((S, D))
    q[:, 0] = 8.0
    k[at, 0] = gap / 8.0
    v = np.broadcast_to(value * (1.0 + np.arange(D) / 128.0), (S, D)).copy()
    v[at] = 0.0
    return q, k, v


@pytest.mark.parametrize("out_dt", ["own", "f32"])
@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("gap", [9.0, 14.0, 16.5, 24.0])
@pytest.mark.parametrize("at", [3, 500])
@pytest.mark.parametrize("M,N,D", [(64, 64, 64), (128, 128, 64), (64, 64, 128)])
def test_tiles_heavy_key_without_value(M, N, D, at, gap, dt, out_dt):
    """Every result is made of keys that weigh e^-gap: their P has to hold its
    bits there, not only next to 1."""
    S = 512
    q, k, v = (_bits(x[None, None], dt) for x in _sink(S, D, at, gap, 250.0))
    src = configs.flash_attention(1, 1, S, D, M, dt, False, N)
    o = np.zeros_like(q)
    if out_dt == "f32":
        tail = src[src.index("%o_init"):]
        f32 = tail.replace("    %ob = arith.truncf", "    %unused = arith.truncf").replace("%ob [[", "%of [[") \
            .replace(f"tensor<{M}x{D}x{dt}> into", f"tensor<{M}x{D}xf32> into").replace(f"1x1x{M}x{D}x{dt}>", f"1x1x{M}x{D}xf32>") \
            .replace(f"{S}x{D}x{dt}>", f"{S}x{D}xf32>")
        head = src[:src.index("%o_init")]
        i = head.index("%o_view =")
        head = head[:i] + head[i:].replace(f"x{dt}>", "xf32>", 1)
        src, o = head + f32, np.zeros(q.shape, np.float32)
    prep, d = _prepare(src, "flash_attention", dict(q_ptr=q, k_ptr=k, v_ptr=v, o_ptr=o, scale=1.0))
    assert (d.M, d.N, d.D) == (M, N, D)
    want, spread = _dense(_f64(q), _f64(k), _f64(v), 1.0, False)
    _near(_f64(prep.outputs()["o_ptr"]), want, dt if out_dt == "own" else "f32", spread, _exp_err(gap))


# finite fills of a mask: the score of a masked key, and the running maximum of a
# row while all its keys are masked
FILLS = {"-1.0e4": -1e4, "-1.0e6": -1e6, "-1.0e7": -1e7, "-1.0e9": -1e9, "0xFF7FFFFF": float(np.finfo(np.float32).min)}


def _filled(src, fill):
    """`src` with `fill` for masked scores, and keys kept from beyond the row's
    position on: rows whose first tiles are masked whole, and a last row that
    is masked throughout (whose weights are then all equal)."""
    name = "%mv" if "%mv = arith.select" in src else "%r"
    old = f"{name} = arith.select %keep, %sv, %neg_inf : f32"
    head = "    %c1 = arith.constant 1 : index\n"
    assert src.count(old) == src.count(head) == 1 and "arith.cmpi ule" in src
    return src.replace(old, old.replace("%neg_inf", "%fill")).replace("arith.cmpi ule", "arith.cmpi ugt") \
        .replace(head, head + f"    %fill = arith.constant {fill} : f32\n")


def _filled_want(s, keep, v, fill):
    s = np.where(keep, s, FILLS[fill])
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    return p @ v, p @ np.abs(v)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("fill", list(FILLS))
@pytest.mark.parametrize("M,N,D", [(64, 64, 64), (128, 64, 128), (128, 128, 64)])
@pytest.mark.parametrize("H", [2, 140])
def test_tiles_of_finite_fills(M, N, D, fill, dt, H):
    S = 256
    rng = np.random.default_rng(M + N)
    q, k, v = (_bits(rng.standard_normal((1, H, S, D)), dt) for _ in range(3))
    src = _filled(configs.flash_attention(1, H, S, D, M, dt, True, N), fill)
    old = f"arith.divui %q_end, %KBLK : index" if M != N else "%n_kv = arith.addi %qb, %c1 : index"
    assert src.count(old) == 1
    src = src.replace(old, old[:old.index("arith")] + f"arith.constant {S // N} : index")
    prep, d = _prepare(src, "flash_attention", dict(q_ptr=q, k_ptr=k, v_ptr=v, o_ptr=np.zeros_like(q), scale=D ** -0.5))
    assert (d.M, d.N, d.D) == (M, N, D)
    s = np.einsum("bhid,bhjd->bhij", _f64(q), _f64(k)) * D ** -0.5
    pos = np.arange(S)
    want, spread = _filled_want(s, pos[None, :] > pos[:, None], _f64(v), fill)
    _near(_f64(prep.outputs()["o_ptr"]), want, dt, spread)


def _far_scores(S, D, steps):
    """q and k of exact scores near 7600 that rise by 3/4 from step to step of `steps` keys."""
    q, k = np.zeros((S, D)), np.zeros((S, D))
    q[:, 0], q[:, 1] = 4.0, 1.0
    k[:, 0] = 1900.0
    j = np.arange(S)
    k[:, 1] = (j // steps) * 0.75 - (j * 7 % 13) / 8.0
    return q, k


@pytest.mark.parametrize("M,N,D", [(64, 64, 64), (128, 64, 128), (128, 128, 64)])
def test_tiles_row_sum_of_far_scores(M, N, D):
    """exp(S - m) of scores near 7600: the row sum as exact as of scores near 0,
    also across the rows' moves of the base."""
    S = 512
    q, k = _far_scores(S, D, N)
    rng = np.random.default_rng(1)
    q, k, v = (_bits(x[None, None], "f16") for x in (q, k, rng.standard_normal((S, D))))
    prep, d = _prepare(configs.flash_attention(1, 1, S, D, M, "f16", False, N), "flash_attention",
                       dict(q_ptr=q, k_ptr=k, v_ptr=v, o_ptr=np.zeros_like(q), scale=1.0))
    s = (_f64(q)[0, 0] @ _f64(k)[0, 0].T)[0]
    np.testing.assert_array_equal(_device(d.m_out, S), np.full(S, s.max()))
    np.testing.assert_allclose(_device(d.l_out, S), np.full(S, np.exp(s - s.max()).sum()), rtol=4e-6)


# ---- paged ---------------------------------------------------------------------

def _paged(dt, tokens, block_q, head, q, k, v, context, scale):
    """One KV head: q [tokens, 4, head], k and v [keys, head] in order of position."""
    n = k.shape[0] // 16
    gen = dict(tokens=tokens, block_q=block_q, head=head, q_heads=4, kv_heads=1, blocks=n, max_pages=n)
    order = np.random.default_rng(2).permutation(n)
    pages = lambda x: _bits(x, dt).reshape(n, 16, 1, head)[np.argsort(order)]
    kw = dict(output_ptr=_bits(np.zeros(q.shape), dt), query_ptr=_bits(q, dt), key_cache_ptr=pages(k),
              value_cache_ptr=pages(v), block_tables_ptr=order.astype(np.int32)[None], cur_batch_start_index=0,
              block_table_offset=0, num_tiles=n, context_len=context, scale=scale)
    prep, d = _prepare(configs.paged_attention(dt=dt, **gen), PA_FN, kw)
    assert d.n_items > 0
    return prep, d


def _paged_want(q, k, v, context, scale, dt):
    q, k, v = (_f64(_bits(x, dt)) for x in (q, k, v))
    s = np.einsum("thd,jd->thj", q, k) * scale
    late = np.arange(k.shape[0])[None, None] > context + np.arange(q.shape[0])[:, None, None]
    s = np.where(late, -np.inf, s)
    m = s.max(-1, keepdims=True)
    p = np.exp(s - m)
    l = p.sum(-1, keepdims=True)
    return p @ v / l, p @ np.abs(v) / l, m[..., 0], l[..., 0]


# half a unit of what P is rounded to: a lane of at most 16 rows carries one
# f16 term or two bf16 ones
P_ERR = {(8, "f16"): 2.0 ** -12, (8, "bf16"): 2.0 ** -17, (32, "f16"): 0.0, (32, "bf16"): 0.0}
ROWS = {8: dict(tokens=8, block_q=2), 32: dict(tokens=16, block_q=8)}


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("rows", list(ROWS))
def test_paged_within_its_roundings(rows, head, dt, splits, monkeypatch):
    from ktir_cpu_amd import fusion
    monkeypatch.setattr(fusion, "_pattn_splits", lambda *a: splits)
    rng = np.random.default_rng(rows + head)
    t, S = ROWS[rows]["tokens"], 336
    q, k, v = (rng.standard_normal(x) for x in ((t, 4, head), (S, head), (S, head)))
    args = (q, k, v, S - t, head ** -0.5)
    prep, d = _paged(dt, t, ROWS[rows]["block_q"], head, *args)
    want, spread, _, _ = _paged_want(*args, dt)
    _near(_f64(prep.outputs()["output_ptr"]), want, dt, spread, P_ERR[rows, dt] + 2.0 ** -21)


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("gap", [9.0, 14.0, 16.5, 24.0])
@pytest.mark.parametrize("at", [3, 300])
@pytest.mark.parametrize("rows", list(ROWS))
def test_paged_heavy_key_without_value(rows, at, gap, dt, splits, monkeypatch):
    from ktir_cpu_amd import fusion
    monkeypatch.setattr(fusion, "_pattn_splits", lambda *a: splits)
    t, S, head = ROWS[rows]["tokens"], 512, 128
    if rows == 8 and dt == "f16":
        gap = min(gap, 17.0)                     # below, one f16 term is subnormal
    q, k, v = _sink(S, head, at, gap, 250.0)
    args = (np.broadcast_to(q[0], (t, 4, head)), k, v, S - t, 1.0)
    prep, d = _paged(dt, t, ROWS[rows]["block_q"], head, *args)
    want, spread, _, _ = _paged_want(*args, dt)
    _near(_f64(prep.outputs()["output_ptr"]), want, dt, spread, P_ERR[rows, dt] + _exp_err(gap))


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("rows", list(ROWS))
def test_paged_row_sum_of_far_scores(rows, splits, monkeypatch):
    """As for the dense tiles, across wavefronts and workgroups whose keys
    have other maxima."""
    from ktir_cpu_amd import fusion
    monkeypatch.setattr(fusion, "_pattn_splits", lambda *a: splits)
    t, S, head = ROWS[rows]["tokens"], 512, 128
    q, k = _far_scores(S, head, 32)
    args = (np.broadcast_to(q[0], (t, 4, head)), k, np.random.default_rng(1).standard_normal((S, head)), S - t, 1.0)
    prep, d = _paged("f16", t, ROWS[rows]["block_q"], head, *args)
    _, _, m, l = _paged_want(*args, "f16")
    np.testing.assert_array_equal(_device(d.m_out, 4 * t), m.reshape(-1))
    np.testing.assert_allclose(_device(d.l_out, 4 * t), l.reshape(-1), rtol=4e-6)


@pytest.mark.parametrize("splits,waves", [(1, 4), (3, 4), (1, 1)])
@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("fill", list(FILLS))
@pytest.mark.parametrize("rows", list(ROWS))
def test_paged_finite_fills(rows, fill, dt, splits, waves, monkeypatch):
    """Tokens near the end of the keys: most pages of a row masked whole, the
    last token's all."""
    from ktir_cpu_amd import fusion
    monkeypatch.setattr(fusion, "_pattn_splits", lambda *a: splits)
    monkeypatch.setattr(fusion, "_pattn_waves", lambda *a: waves)
    real = configs.paged_attention
    monkeypatch.setattr(configs, "paged_attention", lambda **k: _filled(real(**k), fill))
    t, S, head = ROWS[rows]["tokens"], 256, 64
    rng = np.random.default_rng(rows)
    q, k, v = (rng.standard_normal(x) for x in ((t, 4, head), (S, head), (S, head)))
    prep, d = _paged(dt, t, ROWS[rows]["block_q"], head, q, k, v, S - t, head ** -0.5)
    q, k, v = (_f64(_bits(x, dt)) for x in (q, k, v))
    s = np.einsum("thd,jd->thj", q, k) * head ** -0.5
    keep = np.arange(S)[None, None] > S - t + np.arange(t)[:, None, None]
    want, spread = _filled_want(s, keep, v, fill)
    # (f16 on one wavefront: P relative to a base that lags by up to 8)
    _near(_f64(prep.outputs()["output_ptr"]), want, dt, spread, P_ERR[rows, dt] + 2.0 ** -21)
