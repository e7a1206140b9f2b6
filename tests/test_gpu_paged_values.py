"""Paged attention on values that its matrix-core kernels could lose: NaN and
infinities in Q, K and V, for lanes whose P is one or several terms of the
operand type; and lanes that are sequences of their own, which share no pages."""
import numpy as np
import pytest

from ktir_cpu_amd import configs
from oracle.interp import OracleInterpreter, bf16_bits, bf16_from_bits
from tests.test_oracle_example_pins import PA_ARGS, PA_FN, paged_inputs

pytestmark = pytest.mark.gpu

# rows per lane: 8 and 32 (2 and 8 tokens of 4 query heads each)
ROWS = {8: dict(tokens=8, block_q=2), 32: dict(tokens=16, block_q=8)}


def _bits(x, dt):
    return bf16_bits(x.astype(np.float32)) if dt == "bf16" else x.astype(np.float16)


def _f32(x, dt):
    return bf16_from_bits(x) if dt == "bf16" else x.astype(np.float32)


def _run(src, kw, oracle=True):
    from ktir_cpu_amd.interpreter import KTIRInterpreter
    ref = None
    if oracle:
        o = OracleInterpreter()
        o.load(src)
        ref = o.execute_function(PA_FN, **{k: (v.copy() if isinstance(v, np.ndarray) else v) for k, v in kw.items()})
    g = KTIRInterpreter()
    g.load(src)
    got = g.execute_function(PA_FN, **kw)
    d = g.last_plan.launches[-1][1]
    assert g.last_plan.counts().get("pattn") == 1 and d.n_items > 0
    return got["output_ptr"], None if ref is None else ref["output_ptr"]


@pytest.mark.parametrize("splits,waves", [(1, 4), (2, 4), (1, 8), (1, 1)])
@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("rows", list(ROWS))
def test_non_finite_inputs(rows, head, dt, splits, waves, monkeypatch):
    """NaN in a query row, an infinity in a key, infinities of both signs and
    a NaN in V: NaN and infinities exactly where the oracle has them."""
    from ktir_cpu_amd import fusion
    monkeypatch.setattr(fusion, "_pattn_splits", lambda *a: splits)
    monkeypatch.setattr(fusion, "_pattn_waves", lambda *a: waves)
    gen = dict(ROWS[rows], head=head)
    kw = paged_inputs(tokens=gen["tokens"], head=head, seed=11)
    pages = kw["block_tables_ptr"][0]
    pages[:9] = np.arange(3, 12)                 # every page once
    q, k, v = (kw[n].astype(np.float32) for n in ("query_ptr", "key_cache_ptr", "value_cache_ptr"))
    q[1, 6, 7] = np.nan                          # KV head 1
    k[pages[2], 5, 2, 3] = np.inf                # KV head 2
    v[pages[0], 4, 3, 5] = np.inf
    v[pages[3], 9, 3, 9], v[pages[5], 2, 3, 11] = -np.inf, np.nan
    v[pages[1], 1, 4, 17], v[pages[6], 1, 4, 17] = np.inf, -np.inf
    kw.update({n: _bits(x, dt) for n, x in zip(("query_ptr", "key_cache_ptr", "value_cache_ptr"), (q, k, v))},
              output_ptr=_bits(kw["output_ptr"], dt), **dict(PA_ARGS, num_tiles=9, context_len=125))
    got, ref = _run(configs.paged_attention(dt=dt, **gen), kw)
    got, ref = _f32(got, dt), _f32(ref, dt)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    assert np.isnan(ref).any() and np.isposinf(ref).any() and np.isneginf(ref).any()
    ok = ~np.isnan(ref)
    np.testing.assert_allclose(got[ok], ref[ok], rtol=1e-2, atol=1e-3)


def _sequences(n, pages, dt, head=64):
    """n tokens of 4 query heads, each a sequence with its own `pages` pages."""
    rng = np.random.default_rng(n + pages)
    gen = dict(tokens=n, block_q=1, q_heads=8, kv_heads=2, head=head, blocks=96, max_pages=n * pages)
    src = configs.paged_attention(dt=dt, **gen)
    old = "%bt_col = arith.addi %block_table_offset, %j : index"
    assert old in src
    src = src.replace(old, "%bt_col = arith.addi %own, %j : index")
    one = "    %c1 = arith.constant 1 : index\n"
    src = src.replace(one, one + f"    %per = arith.constant {pages} : index\n    %own = arith.muli %p0, %per : index\n", 1)
    kw = paged_inputs(tokens=n, q_heads=8, kv_heads=2, head=head, blocks=96, max_pages=n * pages, seed=n)
    kw = {k: (v if k == "block_tables_ptr" else _bits(v, dt)) for k, v in kw.items()}
    return src, dict(kw, **dict(PA_ARGS, num_tiles=pages, context_len=16 * pages - n // 2))


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("n,pages,waves", [(40, 3, 1), (40, 24, 4)])
def test_sequences_of_their_own(n, pages, waves, dt):
    """Few pages each: one wavefront per lane; more: four per item of one lane."""
    from ktir_cpu_amd.interpreter import KTIRInterpreter
    src, kw = _sequences(n, pages, dt)
    o = OracleInterpreter()
    o.load(src)
    ref = o.execute_function(PA_FN, **{k: (v.copy() if isinstance(v, np.ndarray) else v) for k, v in kw.items()})
    g = KTIRInterpreter()
    g.load(src)
    got = g.execute_function(PA_FN, **kw)
    d = g.last_plan.launches[-1][1]
    assert (d.lanes, d.n_items, d.splits, d.waves) == (2 * n, 2 * n, 1, waves)
    # P in one f16 term or two bf16 terms, one rounding of the result
    np.testing.assert_allclose(_f32(got["output_ptr"], dt), _f32(ref["output_ptr"], dt),
                               rtol=2.0 ** (-7 if dt == "bf16" else -10), atol=2.0 ** -10 if dt == "f16" else 2.0 ** -14)
