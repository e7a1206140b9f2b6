"""Attention results that are used again after they have been stored: the
fused launch then still writes the accumulator that the later use is computed
from, and leaves it out only where nothing reads it.  The plans are checked on
the CPU with a library that does nothing, the results on the GPU against the
oracle."""
import ctypes as C

import numpy as np
import pytest

from ktir_cpu_amd import configs
from ktir_cpu_amd import runtime as rt
from ktir_cpu_amd.interpreter import KTIRInterpreter
from oracle.interp import OracleInterpreter, bf16_from_bits
from tests import _cases
from tests.test_oracle_example_pins import PA_ARGS, PA_FN, paged_inputs


class _NoDevice:
    """Stands in for the library: addresses are handed out, nothing runs."""

    def __init__(self):
        self.next = 1 << 32

    def ktir_malloc(self, n, out):
        C.cast(out, C.POINTER(C.c_uint64))[0] = self.next
        self.next += (int(n) + 511) // 256 * 256
        return 0

    def __getattr__(self, name):
        return lambda *a: 0


@pytest.fixture
def no_device(monkeypatch):
    lib = _NoDevice()
    monkeypatch.setattr(rt, "lib", lambda: lib)


# what follows the first store, by the names of the result's tile ({o}, of the
# tensor type {T}), of its f32 form %of ({Tf}) and of the second output's access
AGAIN = {
    "stored": "    ktdp.store {o}, %again_acc : {T}, {at}",
    "added_to": "    %again = arith.addf {o}, {o} : {T}\n    ktdp.store %again, %again_acc : {T}, {at}",
    # a loop's iter_args go out of scope with it: their names are free again
    "named_as_iter_arg": "    ktdp.store %acc, %again_acc : {T}, {at}",
    "one_element": "    %again = tensor.splat %elem : {T}\n    ktdp.store %again, %again_acc : {T}, {at}",
}
# what stands before the first store
BEFORE = {
    "named_as_iter_arg": "    %acc = arith.addf {o}, {o} : {T}\n",
    "one_element": "    %elem = tensor.extract {flat}[%c0, %c0] : {Tflat}\n",
}


def _again(src, how, old_ptr, old_view, old_acc, o, T, at, flat, Tflat):
    """`src` with a second output, an argument after `old_ptr`, laid out as the first."""
    src = src.replace(f"%{old_ptr}: index", f"%{old_ptr}: index, %again_ptr: index", 1)
    lines = src.split("\n")
    i = next(k for k, x in enumerate(lines) if x.lstrip().startswith(f"%{old_view} ="))
    j = next(k for k in range(i + 1, len(lines)) if lines[k].lstrip().startswith("%"))
    lines[j:j] = [x.replace(old_view, "again_view").replace(old_ptr, "again_ptr") for x in lines[i:j]]
    i = next(k for k, x in enumerate(lines) if x.lstrip().startswith(f"%{old_acc} ="))
    j = next(k for k, x in enumerate(lines) if x.lstrip().startswith(f"ktdp.store {o}, %{old_acc}"))
    acc = [x.replace(f"%{old_acc}", "%again_acc").replace(f"%{old_view}", "%again_view") for x in lines[i:j]]
    f = dict(o=o, T=T, at=at, flat=flat, Tflat=Tflat)
    lines[i:j + 1] = BEFORE.get(how, "").format(**f).split("\n")[:-1] + lines[i:j] + acc + [lines[j], AGAIN[how].format(**f)]
    return "\n".join(lines)


def _paged(how, dt="f16", **gen):
    gen = dict(dict(tokens=8, block_q=2, head=128), **gen)
    src = configs.paged_attention(dt=dt, **gen)
    g, bq, D = 4, gen["block_q"], gen["head"]
    kw = dict(paged_inputs(tokens=gen["tokens"], head=D, seed=3), **PA_ARGS)
    if how is not None:
        src = _again(src, how, "output_ptr", "o_view", "o_acc", "%o3", f"tensor<{bq}x{g}x{D}x{dt}>",
                     f"!ktdp.access_tile<{bq}x{g}x{D}xindex>", "%oh", f"tensor<{bq * g}x{D}x{dt}>")
        args, kw = kw, {}
        for k, v in args.items():
            kw[k] = v
            if k == "output_ptr":
                kw["again_ptr"] = np.zeros_like(v)
    return src, PA_FN, kw


def _flash(how, blk, D, dt="f16", S=None):
    src, fn, args = _cases.flash_attention(B=1, H=2, S=S or 2 * blk, D=D, blk=blk, dt=dt)
    if how is None:
        return src, fn, args
    src = _again(src, how, "o_ptr", "o_view", "o_acc", "%o4", f"tensor<1x1x{blk}x{D}x{dt}>",
                 f"!ktdp.access_tile<1x1x{blk}x{D}xindex>", "%ob", f"tensor<{blk}x{D}x{dt}>")
    kw = {}
    for k, v in args.items():
        kw[k] = v
        if k == "o_ptr":
            kw["again_ptr"] = np.zeros_like(v)
    return src, fn, kw


CASES = {
    "paged_8_rows": lambda how, dt: _paged(how, dt),
    "paged_32_rows": lambda how, dt: _paged(how, dt, tokens=16, block_q=8),
    "tiles_64": lambda how, dt: _flash(how, 64, 64, dt),
    "tiles_128_by_64": lambda how, dt: _flash(how, 128, 64, dt),
    "tiles_64_by_128": lambda how, dt: _flash(how, 64, 128, dt),
    "tiles_128": lambda how, dt: _flash(how, 128, 128, dt),
}


@pytest.mark.parametrize("how", [None] + list(AGAIN), ids=["once"] + list(AGAIN))
@pytest.mark.parametrize("case", list(CASES))
def test_plan_writes_the_accumulator_where_it_is_read(case, how, no_device):
    src, fn, kw = CASES[case](how, "f16")
    it = KTIRInterpreter()
    it.load(src)
    plan = it.prepare(fn, **kw).plan
    assert plan.mode == "lockstep"
    (d,) = [x[1] for x in plan.launches if x[0] in ("attn", "pattn")]
    assert (d.acc_out != 0) == (how is not None)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("how", list(AGAIN))
@pytest.mark.parametrize("case", list(CASES))
def test_result_used_after_its_store(case, how, dt):
    """The second output within the rounding of the first (two units of the
    type: the sum of two results doubles their difference)."""
    if dt == "bf16" and case.startswith("paged"):
        src, fn, kw = CASES[case](how, dt)
        from oracle.interp import bf16_bits
        kw = {k: (bf16_bits(v.astype(np.float32)) if getattr(v, "dtype", None) == np.float16 else v) for k, v in kw.items()}
    else:
        src, fn, kw = CASES[case](how, dt)
    o = OracleInterpreter()
    o.load(src)
    ref = o.execute_function(fn, **{k: (v.copy() if isinstance(v, np.ndarray) else v) for k, v in kw.items()})
    g = KTIRInterpreter()
    g.load(src)
    out = g.execute_function(fn, **kw)
    counts = g.last_plan.counts()
    assert counts.get("attn", 0) + counts.get("pattn", 0) == 1
    f = bf16_from_bits if dt == "bf16" else (lambda x: x.astype(np.float32))
    assert np.abs(f(ref["again_ptr"])).max() > 0
    for k in ("again_ptr", "output_ptr" if "output_ptr" in out else "o_ptr"):
        np.testing.assert_allclose(f(out[k]), f(ref[k]), rtol=2.0 ** (-6 if dt == "bf16" else -9), atol=1e-3)
