"""Cases that time the framework's main path on one GPU.

A case is one KTIR kernel of a family that the generators in
``ktir_cpu_amd/configs.py`` write, at one size.  Its pass is what a program
does once its arguments are in HBM: replay the prepared launch plan
(``KTIRInterpreter.prepare`` / ``Prepared.run``), or, for the smallest kernel,
one whole ``execute_function`` call on host arrays.  Outputs are torch views
of the arrays in the device arena (the host arrays that ``execute_function``
returns, for the whole call).

``exact`` computes the same function in float64 with torch alone.
"""

import math
import sys

import numpy as np
import torch

from ktir_cpu_amd import configs
from ktir_cpu_amd.interpreter import KTIRInterpreter

_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # the reference's vector_add example, whole call: copies in, walk, one launch, copies out
        dict(name="add_call_4096", family="add", cores=32, block=128, per_core=1, whole=True),
        # embedding-style update: gather 262 144 rows of a 1 Mi x 128 table, add them into an f32 table
        dict(name="gather_scatter_1m", family="gather", rows=1 << 20, dim=128, cores=64, chunk=128, per_core=32,
             unique=0.9),
        # attention-probability sized softmax over a power-of-two row, f16
        dict(name="softmax_f16_4096", family="softmax", cores=512, per_core=8, rblk=8, cols=4096, dt="f16"),
        # softmax over a ragged row (a sequence length that is no power of two), bf16
        dict(name="softmax_bf16_3000", family="softmax", cores=256, per_core=8, rblk=4, cols=3000, dt="bf16"),
        # RMSNorm over a 40-head x 128 hidden size (the rotary example's 40 heads)
        dict(name="rmsnorm_f16_5120", family="rmsnorm", cores=512, per_core=4, rblk=4, cols=5120, dt="f16"),
        # the large square product, 128 x 128 tiles
        dict(name="gemm_8192", family="gemm", M=8192, N=8192, K=8192, tile=128, bk=64, gm=8, gn=8, dt="f16"),
        # a projection of 512 tokens in the small tiles of the reference's matmul examples
        dict(name="gemm_512_tile64", family="gemm", M=512, N=4096, K=4096, tile=64, bk=32, gm=8, gn=8, dt="f16"),
        # causal prefill attention over a long sequence, bf16
        dict(name="attn_bf16_8192", family="attn", B=1, H=32, S=8192, D=128, blk=128, dt="bf16", causal=True),
        # full (encoder) attention with 64-wide heads and 64-row tiles, f16
        dict(name="attn_f16_d64", family="attn", B=1, H=16, S=2048, D=64, blk=64, dt="f16", causal=False),
        # a chunk of prefill over a paged KV cache: 256 tokens after 1024
        dict(name="paged_prefill_256", family="paged", tokens=256, block_q=2, hq=32, hk=8, D=128, page=16, ctx=1024,
             dt="f16"),
        # one decode step over a paged KV cache of 8192 keys
        dict(name="paged_decode_8192", family="paged", tokens=1, block_q=1, hq=32, hk=8, D=128, page=16, ctx=8191,
             dt="f16"),
        # rotary embedding of 40 heads x 4096 positions
        dict(name="rope_40x4096", family="rope", H=40, S=4096, D=128, gs=4, gh=2, tile=256),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    family = rng.choice(["add", "gather", "softmax", "softmax", "rmsnorm", "gemm", "gemm", "attn", "attn", "paged",
                         "paged", "rope"])
    if family == "add":
        cores, block = _log(rng, 1, 2048), _log(rng, 64, 32768)
        per = _log(rng, 1, max(1, min(16, (1 << 26) // (cores * block))))
        return dict(family=family, cores=cores, block=block, per_core=per, whole=cores * block * per <= 65536)
    if family == "gather":
        dim = rng.choice([32, 64, 96, 128, 256])
        rows = _log(rng, 4096, (1 << 27) // dim)
        chunk = rng.choice([16, 32, 50, 64, 128, 200])
        cores = _log(rng, 1, 64)
        per = max(1, min(32, (rows // 4) // (cores * chunk)))
        return dict(family=family, rows=rows, dim=dim, cores=cores, chunk=chunk, per_core=per, unique=0.9)
    if family in ("softmax", "rmsnorm"):
        cols = _log(rng, 64, 16384)
        if rng.random() < 0.5:
            cols = -(-cols // 64) * 64
        rblk = max(1, min(8, 32768 // cols))
        cores = _log(rng, 4, 512)
        per = _log(rng, 1, max(1, min(16, (1 << 27) // (cores * rblk * cols))))
        return dict(family=family, cores=cores, per_core=per, rblk=rblk, cols=cols, dt=rng.choice(["f16", "bf16"]))
    if family == "gemm":
        tile, bk = rng.choice([(128, 64), (128, 64), (64, 32), (64, 64)])
        most = 1 << (12 if tile == 128 else 11)
        gm, gn = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 8])
        M = tile * gm * _log(rng, 1, max(1, most // (tile * gm)))
        N = tile * gn * _log(rng, 1, max(1, most // (tile * gn)))
        return dict(family=family, M=M, N=N, K=bk * _log(rng, 4, 4096 // bk), tile=tile, bk=bk, gm=gm, gn=gn,
                    dt=rng.choice(["f16", "bf16"]))
    if family == "attn":
        D, blk = rng.choice([(128, 128), (128, 128), (64, 64), (64, 128), (128, 64)])
        fused = (D, blk) == (128, 128)
        S = blk * _log(rng, 2, (4096 if fused else 1024) // blk)
        return dict(family=family, B=rng.choice([1, 2]), H=_log(rng, 1, 32 if fused else 16), S=S, D=D, blk=blk,
                    dt=rng.choice(["bf16", "f16"]), causal=rng.random() < 0.6)
    if family == "paged":
        hk = rng.choice([1, 2, 4, 8])
        g = rng.choice([1, 2, 4, 8])
        D = rng.choice([64, 128, 128])
        dt = rng.choice(["f16", "f16", "bf16"])
        if rng.random() < 0.5:
            return dict(family=family, tokens=1, block_q=1, hq=hk * g, hk=hk, D=D, page=16, ctx=_log(rng, 16, 8191),
                        dt=dt)
        bq = rng.choice([1, 2, 4])
        return dict(family=family, tokens=bq * _log(rng, 2, 256 // bq), block_q=bq, hq=hk * g, hk=hk, D=D, page=16,
                    ctx=_log(rng, 1, 2048) - 1, dt=dt)
    gs, gh = rng.choice([1, 2, 4]), rng.choice([1, 2, 4])
    tile = rng.choice([32, 64, 128, 256])
    return dict(family="rope", H=gh * _log(rng, 1, 40 // gh), S=gs * tile * _log(rng, 1, 4096 // (gs * tile)),
                D=rng.choice([64, 128]), gs=gs, gh=gh, tile=tile)


# ---- inputs --------------------------------------------------------------------

def _inputs(c, seed):
    """The arguments of the case's kernel in order: torch tensors for arrays
    (on the GPU when there is one), numbers for scalars."""
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)

    def normal(shape, dt, scale=1.0):
        return (torch.randn(shape, generator=g, device=_DEV) * scale).to(_TORCH[dt])

    f = c["family"]
    if f == "add":
        n = c["cores"] * c["block"] * c["per_core"]
        return dict(x_ptr=normal((n,), "f16"), y_ptr=normal((n,), "f16"),
                    output_ptr=torch.zeros(n, dtype=torch.float16, device=_DEV), BLOCK_SIZE=c["block"])
    if f == "gather":
        n = c["cores"] * c["chunk"] * c["per_core"]
        uniq = torch.randperm(c["rows"], generator=g, device=_DEV)[:max(1, int(n * c["unique"]))]
        dup = uniq[torch.randint(0, uniq.numel(), (n - uniq.numel(),), generator=g, device=_DEV)]
        idx = torch.cat([uniq, dup])[torch.randperm(n, generator=g, device=_DEV)]
        return dict(table_ptr=normal((c["rows"], c["dim"]), "f16"), idx_ptr=idx.to(torch.int32),
                    out_ptr=torch.zeros((c["rows"], c["dim"]), device=_DEV))
    if f in ("softmax", "rmsnorm"):
        rows = c["cores"] * c["per_core"] * c["rblk"]
        x = normal((rows, c["cols"]), c["dt"], 2.0)
        if f == "softmax":
            return dict(x_ptr=x, y_ptr=torch.zeros_like(x))
        w = (torch.rand(c["cols"], generator=g, device=_DEV) + 0.5).to(_TORCH[c["dt"]])
        return dict(x_ptr=x, w_ptr=w, y_ptr=torch.zeros_like(x), eps=1e-6)
    if f == "gemm":
        s = c["K"] ** -0.5
        return dict(a_ptr=normal((c["M"], c["K"]), c["dt"], s), b_ptr=normal((c["K"], c["N"]), c["dt"], s),
                    c_ptr=torch.zeros((c["M"], c["N"]), dtype=_TORCH[c["dt"]], device=_DEV))
    if f == "attn":
        q, k, v = (normal((c["B"], c["H"], c["S"], c["D"]), c["dt"]) for _ in range(3))
        return dict(q_ptr=q, k_ptr=k, v_ptr=v, o_ptr=torch.zeros_like(q), scale=c["D"] ** -0.5)
    if f == "paged":
        nt = _pages(c)
        cache = (2 * nt, c["page"], c["hk"], c["D"])
        q = normal((c["tokens"], c["hq"], c["D"]), c["dt"])
        table = torch.randperm(2 * nt, generator=g, device=_DEV)[:nt].to(torch.int32).reshape(1, nt)
        return dict(output_ptr=torch.zeros_like(q), query_ptr=q, key_cache_ptr=normal(cache, c["dt"]),
                    value_cache_ptr=normal(cache, c["dt"]), block_tables_ptr=table, cur_batch_start_index=0,
                    block_table_offset=0, num_tiles=nt, context_len=c["ctx"], scale=c["D"] ** -0.5)
    x = normal((c["H"] * c["S"], c["D"]), "f16")
    half = c["D"] // 2
    freq = 10000.0 ** (-torch.arange(half, dtype=torch.float64, device=_DEV) * 2.0 / c["D"])
    ang = torch.outer(torch.arange(c["S"], dtype=torch.float64, device=_DEV), freq)
    return dict(x_ptr=x, cos_ptr=ang.cos().to(torch.float16), sin_ptr=ang.sin().to(torch.float16),
                out_ptr=torch.zeros_like(x))


def _pages(c):
    return -(-(c["ctx"] + c["tokens"]) // c["page"])


def _host(v):
    """The host array a KTIR argument is given as (bf16 travels as uint16 bits)."""
    if not isinstance(v, torch.Tensor):
        return v
    if v.dtype == torch.bfloat16:
        return v.view(torch.int16).cpu().numpy().view(np.uint16)
    return v.cpu().numpy()


def _kernel(c):
    """(KTIR text, function name, output argument)."""
    f = c["family"]
    if f == "add":
        return (configs.vector_add(c["cores"] * c["block"] * c["per_core"], c["block"], c["cores"]), "add_kernel",
                "output_ptr")
    if f == "gather":
        n = c["cores"] * c["chunk"] * c["per_core"]
        return (configs.gather_scatter_add(c["rows"], c["dim"], n, c["cores"], c["chunk"]), "gather_scatter_add",
                "out_ptr")
    if f in ("softmax", "rmsnorm"):
        rows = c["cores"] * c["per_core"] * c["rblk"]
        return getattr(configs, f)(rows, c["cols"], c["cores"], c["rblk"], c["dt"]), f + "_kernel", "y_ptr"
    if f == "gemm":
        src = configs.gemm(c["M"], c["N"], c["K"], c["tile"], c["tile"], c["bk"], c["gm"], c["gn"])
        return src.replace("f16", "bf16") if c["dt"] == "bf16" else src, "gemm_kernel", "c_ptr"
    if f == "attn":
        return (configs.flash_attention(c["B"], c["H"], c["S"], c["D"], c["blk"], c["dt"], c["causal"]),
                "flash_attention", "o_ptr")
    if f == "paged":
        nt = _pages(c)
        return (configs.paged_attention(c["tokens"], c["hq"], c["hk"], c["D"], c["page"], 2 * nt, nt, c["block_q"],
                                        dt=c["dt"]), "kernel_unified_attention_spyre_2d", "output_ptr")
    return configs.rope(c["H"], c["S"], c["D"], c["gs"], c["gh"], c["tile"]), "rope_fwd_kernel", "out_ptr"


class _Held:
    """A prepared function and its device memory, given back with the last
    tensor that looks into it."""

    def __init__(self, interp, prep):
        self.interp, self.prep = interp, prep

    def __del__(self):
        if sys.is_finalizing():
            return
        self.prep.arena.buf.free()
        self.interp._pool.free_all()


class _View:
    """One array argument in the arena, for torch.as_tensor."""

    def __init__(self, held, name):
        a = next(x for x in held.prep.arena.allocs if x.name == name)
        kind = {"f16": "<f2", "bf16": "<i2", "f32": "<f4", "i32": "<i4"}[a.dtype]
        self.held = held
        self.__cuda_array_interface__ = dict(shape=a.shape, typestr=kind, version=2, strides=None,
                                             data=(held.prep.arena.ptr_of(a), False))


def prepare(case, seed):
    src, fn, out = _kernel(case)
    args = {k: _host(v) for k, v in _inputs(case, seed).items()}
    it = KTIRInterpreter()
    it.load(src)
    if case.get("whole"):
        return dict(interp=it, fn=fn, args=args, out=out)
    held = _Held(it, it.prepare(fn, **args))
    y = torch.as_tensor(_View(held, out), device="cuda")
    if case.get("dt") == "bf16":
        y = y.view(torch.bfloat16)
    return dict(prep=held.prep, y=y)


def run(state):
    if "interp" in state:
        return state["interp"].execute_function(state["fn"], **state["args"])[state["out"]]
    # attention: V counts as new on every pass, so its f16 copy is made again
    state["prep"].plan.run(reuse_v16=False)
    return state["y"]


# ---- work, tolerance, exact results -----------------------------------------------

def work(case):
    c, f = case, case["family"]
    if f == "add":
        n = c["cores"] * c["block"] * c["per_core"]
        return dict(bytes=6 * n, flops=n)
    if f == "gather":
        n = c["cores"] * c["chunk"] * c["per_core"]
        uniq = max(1, int(n * c["unique"]))
        return dict(bytes=4 * n + (2 + 8) * c["dim"] * uniq, flops=n * c["dim"])
    if f in ("softmax", "rmsnorm"):
        n = c["cores"] * c["per_core"] * c["rblk"] * c["cols"]
        return dict(bytes=4 * n + (2 * c["cols"] if f == "rmsnorm" else 0), flops=5 * n)
    if f == "gemm":
        return dict(bytes=2 * (c["M"] * c["K"] + c["K"] * c["N"] + c["M"] * c["N"]), flops=2 * c["M"] * c["N"] * c["K"])
    if f == "attn":
        pairs = c["S"] * (c["S"] + 1) // 2 if c["causal"] else c["S"] ** 2
        return dict(bytes=8 * c["B"] * c["H"] * c["S"] * c["D"], flops=4 * c["B"] * c["H"] * pairs * c["D"])
    if f == "paged":
        keys = sum(c["ctx"] + t + 1 for t in range(c["tokens"]))
        return dict(bytes=4 * c["tokens"] * c["hq"] * c["D"] + 4 * (c["ctx"] + c["tokens"]) * c["hk"] * c["D"]
                    + 4 * _pages(c), flops=4 * c["hq"] * keys * c["D"])
    n = c["H"] * c["S"] * c["D"]
    return dict(bytes=4 * n + 2 * c["S"] * c["D"], flops=3 * n)


def tolerance(case):
    f, bf = case["family"], case.get("dt") == "bf16"
    # one f16 rounding of an exact sum; f32 adds in the reference's order
    if f in ("add", "gather"):
        return "exact"
    # f16 products and sums, each rounded, none reordered
    if f == "rope":
        return "exact"
    # one rounding of the result to 8 (bf16) or 11 (f16) bits moves it by at
    # most 2^-9 or 2^-12 of itself where f32 sums differ in their last bits;
    # attention also rounds its probabilities to 16 bits
    return dict(rel=8e-3, max=4e-2) if bf else dict(rel=1e-3, max=6e-3)


def exact(case, seed):
    c, f = case, case["family"]
    a = _inputs(case, seed)
    d = {k: v.double() for k, v in a.items() if isinstance(v, torch.Tensor) and v.is_floating_point()}
    if f == "add":
        y = d["x_ptr"] + d["y_ptr"]
        return y.cpu().numpy() if c["whole"] else y
    if f == "gather":
        # an index repeated inside a chunk keeps its last writer: one add per
        # (chunk, row); prepare() has launched the kernel once before the pass
        idx = a["idx_ptr"].long()
        chunk = torch.arange(idx.numel(), device=idx.device) // c["chunk"]
        rows = torch.unique(chunk * c["rows"] + idx) % c["rows"]
        return d["table_ptr"] * (2.0 * torch.bincount(rows, minlength=c["rows"]))[:, None]
    if f == "softmax":
        return torch.softmax(d["x_ptr"], 1)
    if f == "rmsnorm":
        x = d["x_ptr"]
        return x * torch.rsqrt((x * x).mean(1, keepdim=True) + a["eps"]) * d["w_ptr"]
    if f == "gemm":
        return d["a_ptr"] @ d["b_ptr"]
    if f == "attn":
        o, S = torch.empty_like(d["q_ptr"]), c["S"]
        pos = torch.arange(S, device=o.device)
        for b in range(c["B"]):
            for h in range(c["H"]):
                kt, v = d["k_ptr"][b, h].t().contiguous(), d["v_ptr"][b, h]
                for r in range(0, S, 2048):
                    s = (d["q_ptr"][b, h, r:r + 2048] @ kt) * a["scale"]
                    if c["causal"]:
                        s = s.masked_fill(pos[None, :] > pos[r:r + 2048, None], -math.inf)
                    o[b, h, r:r + 2048] = torch.softmax(s, 1) @ v
        return o
    if f == "paged":
        n, grp = c["ctx"] + c["tokens"], c["hq"] // c["hk"]
        pages = a["block_tables_ptr"][0].long()
        k = d["key_cache_ptr"][pages].reshape(-1, c["hk"], c["D"])[:n]
        v = d["value_cache_ptr"][pages].reshape(-1, c["hk"], c["D"])[:n]
        pos = torch.arange(n, device=k.device)
        late = pos[None, :] > c["ctx"] + torch.arange(c["tokens"], device=k.device)[:, None]
        o = torch.empty_like(d["query_ptr"])
        for h in range(c["hq"]):
            s = (d["query_ptr"][:, h] @ k[:, h // grp].t().contiguous()) * a["scale"]
            o[:, h] = torch.softmax(s.masked_fill(late, -math.inf), 1) @ v[:, h // grp].contiguous()
        return o
    x = d["x_ptr"].reshape(c["H"], c["S"], c["D"])
    x1, x2 = x[..., :c["D"] // 2], x[..., c["D"] // 2:]
    cos, sin = d["cos_ptr"], d["sin_ptr"]
    return torch.cat([x1 * cos - x2 * sin, x1 * sin + x2 * cos], -1).reshape(-1, c["D"])
