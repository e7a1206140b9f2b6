"""Sums and differences of two products, alone and as the pair of a rotation
(a*b +- c*d and a*d +- c*b in one launch): every form that may or may not
share a launch gives the bits of the op-by-op oracle, and `disjoint`, which
decides whether two stores may, never says so of tiles that share an element."""
import itertools

import numpy as np
import pytest

from ktir_cpu_amd import configs
from ktir_cpu_amd.program import LaneOff, LeafSpec, disjoint


def test_disjoint_tiles_never_share_an_element():
    rng = np.random.default_rng(5)
    said = 0
    for _ in range(400):
        shape = tuple(int(rng.integers(1, 4)) for _ in range(2)) + (int(rng.integers(1, 6)),)
        st = (int(rng.integers(1, 5)) * 6, int(rng.integers(1, 4)) * 4, 1)
        la = rng.integers(0, 4, 3) * int(rng.choice([4, 6, 12]))
        lb = la + int(rng.integers(-9, 10)) + (rng.integers(0, 2, 3) if rng.random() < 0.2 else 0)
        a = LeafSpec(0, "f32", LaneOff.from_array(la), st, 0, 1000)
        b = LeafSpec(0, "f32", LaneOff.from_array(lb), st, 0, 1000)

        def cells(base):
            return {int(x) + sum(i * s for i, s in zip(c, st)) for x in base for c in itertools.product(*map(range, shape))}

        if disjoint(a, la, b, lb, shape):
            said += 1
            assert not cells(la) & cells(lb), (shape, st, la, lb)
    assert said > 20
    z = np.zeros(2, np.int64)
    far = LeafSpec(4000, "f32", LaneOff(0, 0), (1,), 0, 10)
    assert disjoint(LeafSpec(0, "f32", LaneOff(0, 0), (1,), 0, 1000), z, far, z, (8,))


def _source(dt, cols, rows, tile, second, op1, op2, col2, view_rows, width):
    """y1 = a*b op1 c*d at column 0, y2 = the products `second` joined by op2
    at column col2 of an output `width` columns wide."""
    T = configs._t([tile, cols], dt)
    at = f"!ktdp.access_tile<{tile}x{cols}xindex>"
    ins = "abcd"
    views = "\n".join(configs._view(f"{n}_view", f"{n}_ptr", [view_rows, cols], [cols, 1], dt) for n in ins)
    body = []
    for n in ins:
        body.append(configs._tile(f"{n}_acc", f"{n}_view", ["%row", "%c0"], [tile, cols], [view_rows, cols], dt))
        body.append(f"    %{n} = ktdp.load %{n}_acc : {at} -> {T}")
    for k, (prods, op, col) in enumerate(((("ab", "cd"), op1, "%c0"), (second, op2, "%cW"))):
        for j, p in enumerate(prods):
            body.append(f"    %m{k}{j} = arith.mulf %{p[0]}, %{p[1]} : {T}")
        body.append(f"    %y{k} = arith.{op} %m{k}0, %m{k}1 : {T}")
        body.append(configs._tile(f"y{k}_acc", "o_view", ["%row", col], [tile, cols], [view_rows, width], dt))
        body.append(f"    ktdp.store %y{k}, %y{k}_acc : {T}, {at}")
    nl = "\n"
    return f"""module {{
  func.func @k(%a_ptr: index, %b_ptr: index, %c_ptr: index, %d_ptr: index, %o_ptr: index)
      attributes {{grid = [{rows // tile}]}} {{
    %p = ktdp.get_compute_tile_id : index
    %c0 = arith.constant 0 : index
    %cW = arith.constant {col2} : index
    %cT = arith.constant {tile} : index
    %row = arith.muli %p, %cT : index
{views}
{configs._view("o_view", "o_ptr", [view_rows, width], [width, 1], dt)}
{nl.join(body)}
    return
  }}
}}"""


# id: dtype, columns, rows, tile rows, second sum's products, ops, column of the second store, launches
FORMS = [
    ("f16", "f16", 64, 24, 8, ("ad", "cb"), "subf", "addf", 64, 1),
    ("bf16_swapped", "bf16", 32, 12, 4, ("bc", "da"), "addf", "subf", 32, 1),
    ("f32", "f32", 8, 6, 2, ("ac", "bd"), "subf", "subf", 8, 1),
    ("f16_many_chunks", "f16", 264, 40, 20, ("ad", "cb"), "addf", "addf", 264, 1),
    ("columns_not_8", "f16", 20, 8, 4, ("ad", "cb"), "subf", "addf", 20, 2),
    ("stores_overlap", "f16", 64, 8, 4, ("ad", "cb"), "subf", "addf", 32, 2),
    ("same_products", "f16", 64, 8, 4, ("ab", "dc"), "subf", "addf", 64, 2),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dt,cols,rows,tile,second,op1,op2,col2,n", [f[1:] for f in FORMS], ids=[f[0] for f in FORMS])
@pytest.mark.parametrize("short", [0, 3], ids=["whole", "past_end"])
def test_sums_of_products_bit_exact(dt, cols, rows, tile, second, op1, op2, col2, n, short):
    """`short` rows at the end of every array are missing: reads past the
    end give 0 and writes past it are dropped (a tile with no row inside is
    an error, so at least one of the last tile's rows is there)."""
    short = min(short, tile - 1)
    from ktir_cpu_amd.interpreter import KTIRInterpreter
    from oracle.interp import OracleInterpreter
    rng = np.random.default_rng(cols + rows)

    def arr(r, c):
        x = rng.standard_normal((r, c)).astype(np.float32)
        x[rng.random((r, c)) < 0.1] *= 0.0           # zeros of both signs
        if dt == "bf16":
            return (x.view(np.uint32) >> 16).astype(np.uint16)
        return x.astype(np.float16 if dt == "f16" else np.float32)

    width = 2 * cols
    kw = {f"{k}_ptr": arr(rows - short, cols) for k in "abcd"}
    kw["o_ptr"] = arr(rows - short, width)
    src = _source(dt, cols, rows, tile, second, op1, op2, col2, rows, width)
    o = OracleInterpreter()
    o.load(src)
    ref = o.execute_function("k", **{k: v.copy() for k, v in kw.items()})["o_ptr"]
    g = KTIRInterpreter()
    g.load(src)
    got = g.execute_function("k", **kw)["o_ptr"]
    assert g.last_plan.mode == "lockstep" and g.last_plan.counts() == {"prog": n}
    np.testing.assert_array_equal(got.view(np.uint8), ref.view(np.uint8))
