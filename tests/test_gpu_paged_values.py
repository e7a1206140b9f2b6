"""Paged attention on values that its matrix-core kernels could lose: NaN and
infinities in Q, K and V, for lanes whose P is one or several terms of the
operand type."""
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


@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("rows", list(ROWS))
def test_non_finite_inputs(rows, head, dt, splits, monkeypatch):
    """NaN in a query row, an infinity in a key, infinities of both signs and
    a NaN in V: NaN and infinities exactly where the oracle has them."""
    from ktir_cpu_amd import fusion
    monkeypatch.setattr(fusion, "_pattn_splits", lambda *a: splits)
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
