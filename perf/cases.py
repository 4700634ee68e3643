"""Performance cases of the EXL3 layer and codec, through the Python binding's public calls.

A case is a dict of plain values; `listed()` gives the fixed ones, `draw()` another
of the same ranges.  Weights are random trellis words (a quantised stream is close
to uniform), su = +-1 and sv = +-U(0.5, 1.5) / sqrt(k), activations N(0, sigma).
"""
import importlib.util
import math
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]
CODEBOOKS = ("3inst", "mcg", "mul1")
DTYPES = {"f16": torch.float16, "f32": torch.float32}


def _binding():
    name = "exl3_amd_perf"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, ROOT / "xiaomi-hexagon-exl3_amd" / "exl3_amd.py")
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ------------------------------------------------------------------ cases
def listed():
    return [
        # the smallest call: one MLP projection for one token, called eagerly
        dict(name="layer_small_b1", kind="layer", k=2048, n=6144, bits=4, cb="mul1", rows=1, x="f16", y="f16",
             residual=False),
        # one wide down projection for one token (the benchmark's headline layer)
        dict(name="layer_down_b1", kind="layer", k=14336, n=4096, bits=4, cb="mul1", rows=1, x="f16", y="f16",
             residual=False),
        # the vocabulary head for one token
        dict(name="head_b1", kind="layer", k=2048, n=151936, bits=6, cb="mul1", rows=1, x="f16", y="f32",
             residual=False),
        # the decode step of a serving loop, captured once and replayed per token: the projections of
        # four decoder layers (q/k/v, o, gate/up, down at 6/6/4/3 bits), one and eight sequences
        dict(name="decode_step_b1", kind="step", layers=4, hidden=2048, kv=512, ffn=6144, rows=1, cb="mul1"),
        dict(name="decode_step_b8", kind="step", layers=4, hidden=2048, kv=512, ffn=6144, rows=8, cb="mul1"),
        # a short ragged prompt with ggml's F32 tensors and the residual ADD in the call
        dict(name="layer_resid_r37", kind="layer", k=6144, n=2048, bits=3, cb="mcg", rows=37, x="f32", y="f32",
             residual=True),
        # prefill of 512 tokens through the wide down projection
        dict(name="prefill_512", kind="layer", k=14336, n=4096, bits=4, cb="mul1", rows=512, x="f16", y="f16",
             residual=False),
        # prefill of a long prompt: gate and up of a large MLP in one grouped call (the largest case)
        dict(name="prefill_group_4096", kind="group", k=4096, n0=14336, n1=14336, bits=4, cb="mul1", rows=4096,
             x="f16", y="f16"),
        # the DSP service's layer: upstream tiles and separate scales, fp32 in and out, batch 8
        dict(name="service_b8", kind="iface", k=2048, n=6144, bits=5, cb="3inst", rows=8),
        # the embedding rows of a 512-token prompt from the tied 6-bit head (GET_ROWS)
        dict(name="embed_512", kind="rows", k=2048, n=151936, bits=6, cb="mul1", ids=512, y="f32"),
        # dequantising the projections of one decoder layer into fp16 (load time)
        dict(name="dequant_layer", kind="dequant", hidden=2048, kv=512, ffn=6144, cb="mul1"),
        # one matrix back in the original basis, fp16 (checking or converting a model)
        dict(name="reconstruct", kind="reconstruct", k=2048, n=6144, bits=4, cb="mul1"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dim(rng, lo, hi):
    """A multiple of 128, spread over the logarithm of the range, odd multiples among them."""
    return 128 * _log_int(rng, lo // 128, hi // 128)


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "step", "group", "iface", "rows", "dequant", "reconstruct"))
    cb = rng.choice(("mul1", "mul1", "mcg", "3inst"))
    bits = rng.choice((2, 3, 4, 4, 5, 6, 8))
    f = lambda: rng.choice(("f16", "f32"))  # noqa: E731
    if kind == "layer":
        rows = rng.choice((1, rng.randint(2, 14), _log_int(rng, 15, 128), _log_int(rng, 129, 2048)))
        return dict(kind=kind, k=_dim(rng, 2048, 14336), n=_dim(rng, 512, 14336), bits=bits, cb=cb, rows=rows, x=f(),
                    y=f(), residual=rng.random() < 0.3)
    if kind == "step":
        return dict(kind=kind, layers=rng.randint(2, 4), hidden=_dim(rng, 1024, 4096), kv=_dim(rng, 256, 1024),
                    ffn=_dim(rng, 3072, 14336), rows=_log_int(rng, 1, 16), cb=cb)
    if kind == "group":
        return dict(kind=kind, k=_dim(rng, 1024, 4096), n0=_dim(rng, 512, 14336), n1=_dim(rng, 512, 14336), bits=bits,
                    cb=cb, rows=_log_int(rng, 1, 4096), x=f(), y=f())
    if kind == "iface":
        return dict(kind=kind, k=_dim(rng, 1024, 6144), n=_dim(rng, 512, 6144), bits=bits, cb=cb,
                    rows=rng.randint(1, 8))
    if kind == "rows":
        return dict(kind=kind, k=_dim(rng, 1024, 4096), n=_dim(rng, 8192, 151936), bits=bits, cb=cb,
                    ids=_log_int(rng, 1, 2048), y=f())
    if kind == "dequant":
        return dict(kind=kind, hidden=_dim(rng, 1024, 4096), kv=_dim(rng, 256, 1024), ffn=_dim(rng, 3072, 14336),
                    cb=cb)
    return dict(kind="reconstruct", k=_dim(rng, 1024, 6144), n=_dim(rng, 512, 14336), bits=bits, cb=cb)


# ------------------------------------------------------------------ inputs
class _Inputs:
    """Seeded inputs on the GPU, drawn in a fixed order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, rows, k, dtype, sigma=1.0):
        return (torch.randn((rows, k), generator=self.g, device="cuda") * sigma).to(DTYPES[dtype])

    def signs(self, count):
        return torch.randint(0, 2, (count,), generator=self.g, device="cuda").float() * 2 - 1

    def words(self, shape):  # uniform bytes, eight at a time
        count = math.prod(shape)
        raw = torch.empty(count // 8, dtype=torch.int64, device="cuda")
        raw.random_(-(1 << 63), None, generator=self.g)
        return raw.view(torch.uint8).view(shape)

    def scales(self, k, n):
        su = self.signs(k).to(torch.float16)
        mag = 0.5 + torch.rand(n, generator=self.g, device="cuda")
        return su, (self.signs(n) * mag / math.sqrt(k)).to(torch.float16)

    def tiles(self, k, n, bits):
        """Upstream tile grid [k / 16, n / 16, 16 bits] u16 (as int16)."""
        return self.words((k // 16, n // 16, 32 * bits)).view(torch.int16)

    def records(self, k, n, bits):
        """Group records [n / 128][k / 128]: 64 tiles, su, sv (uint8, flat)."""
        su, sv = self.scales(k, n)
        rec = torch.empty((n // 128, k // 128, 2048 * bits + 512), dtype=torch.uint8, device="cuda")
        rec[:, :, : 2048 * bits] = self.words((n // 128, k // 128, 2048 * bits))
        rec[:, :, 2048 * bits : 2048 * bits + 256] = su.view(torch.uint8).view(1, k // 128, 256)
        rec[:, :, 2048 * bits + 256 :] = sv.view(torch.uint8).view(n // 128, 1, 256)
        return rec.view(-1)


def _step_projections(case):
    """(k, ns, bits) of the calls of one decoder layer: q/k/v, o, gate/up, down."""
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return [(h, (h, kv, kv), 6), (h, (h,), 6), (h, (f, f), 4), (f, (h,), 3)]


def _inputs(case, seed):
    """What the caller has: everything here is made from the seed, on the GPU."""
    g, kind = _Inputs(seed), case["kind"]
    if kind == "layer":
        k, n, rows = case["k"], case["n"], case["rows"]
        return dict(rec=g.records(k, n, case["bits"]), x=g.normal(rows, k, case["x"]),
                    res=g.normal(rows, n, case["y"]) if case["residual"] else None)
    if kind == "group":
        k = case["k"]
        return dict(recs=[g.records(k, n, case["bits"]) for n in (case["n0"], case["n1"])],
                    x=g.normal(case["rows"], k, case["x"]))
    if kind == "step":
        calls = []
        for _ in range(case["layers"]):
            for k, ns, bits in _step_projections(case):
                calls.append(dict(k=k, ns=ns, bits=bits, recs=[g.records(k, n, bits) for n in ns],
                                  x=g.normal(case["rows"], k, "f16", 0.5)))
        return dict(calls=calls)
    if kind == "iface":
        k, n = case["k"], case["n"]
        su, sv = g.scales(k, n)
        return dict(tiles=g.tiles(k, n, case["bits"]), su=su, sv=sv, x=g.normal(case["rows"], k, "f32"))
    if kind == "rows":
        rec = g.records(case["k"], case["n"], case["bits"])
        ids = torch.randint(0, case["n"], (case["ids"],), generator=g.g, device="cuda", dtype=torch.int32)
        return dict(rec=rec, ids=ids)
    if kind == "dequant":
        return dict(mats=[(g.tiles(k, n, bits), bits, k, n) for k, ns, bits in _step_projections(case) for n in ns])
    k, n = case["k"], case["n"]
    su, sv = g.scales(k, n)
    return dict(tiles=g.tiles(k, n, case["bits"]), su=su, sv=sv)


def prepare(case, seed):
    amd = _binding()
    s = _inputs(case, seed)
    s.update(case=case, cb=CODEBOOKS.index(case["cb"]))
    kind = case["kind"]

    def out(rows, n, dtype):
        return torch.empty((rows, n), dtype=DTYPES[dtype], device="cuda")

    if kind == "layer":
        k, n, rows = case["k"], case["n"], case["rows"]
        s.update(y=out(rows, n, case["y"]), ws=amd.new_workspace(k, n, rows))
    elif kind == "group":
        k, ns, rows = case["k"], (case["n0"], case["n1"]), case["rows"]
        s.update(mats=[(r, n, out(rows, n, case["y"])) for r, n in zip(s["recs"], ns)],
                 ws=amd.new_workspace(k, ns[0], rows, nbytes=amd.group_workspace_bytes(k, ns, rows)))
    elif kind == "step":
        rows, calls = case["rows"], s["calls"]
        need = max(amd.group_workspace_bytes(c["k"], c["ns"], rows) for c in calls)
        s["ws"] = amd.new_workspace(calls[0]["k"], calls[0]["ns"][0], rows, nbytes=need)
        for c in calls:
            c["ys"] = [out(rows, n, "f16") for n in c["ns"]]
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            for c in calls:
                mats = list(zip(c["recs"], c["ns"], c["ys"]))
                if len(mats) == 1:
                    amd.mul_mat(c["recs"][0], c["bits"], c["k"], c["ns"][0], c["x"], codebook=s["cb"], y=c["ys"][0],
                                workspace=s["ws"])
                else:
                    amd.mul_mat_group(mats, c["bits"], c["k"], c["x"], codebook=s["cb"], workspace=s["ws"])
    elif kind == "iface":
        s.update(y=out(case["rows"], case["n"], "f32"),
                 ws=amd.new_iface_workspace(case["bits"], case["k"], case["n"], case["rows"]))
    elif kind == "rows":
        s["y"] = out(case["ids"], case["k"], case["y"])
    elif kind == "dequant":
        s["items"] = [(t, bits, k, n, torch.empty((k, n), dtype=torch.int16, device="cuda"))
                      for t, bits, k, n in s["mats"]]
    else:
        s["y"] = torch.empty((case["k"], case["n"]), dtype=torch.int16, device="cuda")
    return s


def run(s):
    amd, case, cb = _binding(), s["case"], s["cb"]
    kind = case["kind"]
    if kind == "layer":
        return amd.mul_mat(s["rec"], case["bits"], case["k"], case["n"], s["x"], codebook=cb, y=s["y"],
                           workspace=s["ws"], residual=s["res"])
    if kind == "group":
        return amd.mul_mat_group(s["mats"], case["bits"], case["k"], s["x"], codebook=cb, workspace=s["ws"])
    if kind == "step":
        s["graph"].replay()
        return [y for c in s["calls"] for y in c["ys"]]
    if kind == "iface":
        return amd.iface_matmul(s["tiles"], s["su"], s["sv"], s["x"], case["bits"], case["k"], case["n"], codebook=cb,
                                y=s["y"], workspace=s["ws"])
    if kind == "rows":
        return amd.get_rows(s["rec"], case["bits"], case["k"], case["n"], s["ids"], codebook=cb, out=s["y"])
    if kind == "dequant":
        return [o.view(torch.float16) for o in amd.decode_batch(s["items"], codebook=cb)]
    return amd.reconstruct(s["tiles"], case["bits"], case["k"], case["n"], su=s["su"], sv=s["sv"], codebook=cb,
                           out=s["y"]).view(torch.float16)


# ------------------------------------------------------------------ work and tolerance
def work(case):
    """Each input byte read once, each output byte written once; the layer's products."""
    size = {"f16": 2, "f32": 4}

    def layer(k, ns, bits, rows, xs, ys):
        return (k * sum(ns) * bits // 8 + 2 * k * len(ns) + 2 * sum(ns) + xs * k * rows + ys * sum(ns) * rows,
                2 * rows * k * sum(ns))

    kind = case["kind"]
    if kind == "layer":
        b, f = layer(case["k"], (case["n"],), case["bits"], case["rows"], size[case["x"]], size[case["y"]])
        b += size[case["y"]] * case["n"] * case["rows"] if case["residual"] else 0
    elif kind == "group":
        b, f = layer(case["k"], (case["n0"], case["n1"]), case["bits"], case["rows"], size[case["x"]],
                     size[case["y"]])
    elif kind == "step":
        each = [layer(k, ns, bits, case["rows"], 2, 2) for k, ns, bits in _step_projections(case)]
        b, f = (case["layers"] * sum(e[i] for e in each) for i in (0, 1))
    elif kind == "iface":
        b, f = layer(case["k"], (case["n"],), case["bits"], case["rows"], 4, 4)
    elif kind == "rows":  # the record column group of each distinct id (at most all of them), the rows written
        groups = min(case["ids"], case["n"] // 128)
        b = groups * (case["k"] // 128) * (2048 * case["bits"] + 512) + case["ids"] * case["k"] * size[case["y"]]
        f = 0
    elif kind == "dequant":
        b = sum(k * n * bits // 8 + 2 * k * n for k, ns, bits in _step_projections(case) for n in ns)
        f = 0
    else:
        k, n = case["k"], case["n"]
        b, f = k * n * case["bits"] // 8 + 2 * k * n + 2 * (k + n), 0
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind in ("rows", "dequant", "reconstruct"):
        return "exact"  # the format fixes every bit
    # measured against exact(): 2e-7 for fp32-level sums and outputs (hi + lo activations, up to 14 rows),
    # 2.1e-4 with fp16 outputs, 3.6e-4 with fp16 activations (above 14 rows); stated about four times larger
    if case["rows"] > 14:
        return {"rel": 1.4e-3, "max": 2e-2}
    if kind == "step" or case.get("y") == "f16":
        return {"rel": 8e-4, "max": 4e-3}
    return {"rel": 1e-6, "max": 1e-5}


# ------------------------------------------------------------------ 64-bit results in plain torch
def _hadamard():
    i = torch.arange(128, device="cuda")
    a = i[:, None] & i[None, :]
    for s in (4, 2, 1):
        a = a ^ (a >> s)
    return (1 - 2 * (a & 1)).double() / math.sqrt(128.0)


def _halves(v):  # 16-bit patterns in int64 -> their fp16 values
    return ((v ^ 0x8000) - 0x8000).to(torch.int16).view(torch.float16)


def _decode_tiles(t, bits, cb):
    """[..., 32 bits] uint8 tile bytes -> [..., 16, 16] fp16 weights, from the format's definition."""
    w = t.contiguous().view(torch.int32).long() & 0xFFFFFFFF
    p = torch.arange(256, device="cuda")
    start = ((p + 1) * bits - 16) % (256 * bits)
    lo, off = start // 32, start % 32
    pair = (w[..., lo] << 16) | (w[..., (lo + 1) % (8 * bits)] >> 16)
    state = (pair >> (32 - off)) & 0xFFFF
    if cb == "mul1":
        h = (state * 0x83DCD12D) & 0xFFFFFFFF
        s = (h & 255) + (h >> 8 & 255) + (h >> 16 & 255) + (h >> 24)
        one = lambda b: float(_halves(torch.tensor([b], device="cuda"))[0])  # noqa: E731
        v = ((1024 + s).double() * one(0x1EEE) + one(0xC931)).float().half()
    else:
        h = state * 0xCBAC1FED if cb == "mcg" else state * 89226354 + 64248484
        h = (h & 0x8FFF8FFF) ^ 0x3B603B60
        v = (_halves(h & 0xFFFF).float() + _halves(h >> 16 & 0xFFFF).float()).half()
    ll, e = p // 8, p % 8
    row, col = 2 * (ll % 4) + (e & 1) + 8 * ((e >> 1) & 1), ll // 4 + 8 * ((e >> 2) & 1)
    out = torch.empty_like(v)
    out[..., row * 16 + col] = v
    return out.view(*v.shape[:-1], 16, 16)


def _column_group(rec, k, bits, cb, nb, count):
    """Inner weights [k, 128 count] (double), su [k] and sv [128 count] of column groups nb .. nb + count - 1."""
    r = rec.view(-1, k // 128, 2048 * bits + 512)[nb : nb + count]
    c = r.shape[0]
    t = r[:, :, : 2048 * bits].reshape(c, k // 128, 8, 8, 32 * bits)
    w = _decode_tiles(t, bits, cb).permute(1, 2, 4, 0, 3, 5).reshape(k, 128 * c).double()
    su = r[0, :, 2048 * bits : 2048 * bits + 256].contiguous().view(torch.float16).reshape(k).double()
    sv = r[:, 0, 2048 * bits + 256 :].contiguous().view(torch.float16).reshape(128 * c).double()
    return w, su, sv


def _upstream(t, k, n, bits, cb):
    return _decode_tiles(t.view(torch.uint8), bits, cb).permute(0, 2, 1, 3).reshape(k, n).double()


def _chunk(k):
    return max(1, (1 << 24) // (128 * k))


def _apply(x, w, su, sv, h):
    rows, k, n = x.shape[0], w.shape[0], w.shape[1]
    xh = ((x.double() * su).view(rows, k // 128, 128) @ h).view(rows, k)
    return ((xh @ w).view(rows, n // 128, 128) @ h).view(rows, n) * sv


def _layer(rec, x, k, n, bits, cb, h):
    step = _chunk(k)
    return torch.cat([_apply(x, *_column_group(rec, k, bits, cb, nb, step), h)
                      for nb in range(0, n // 128, step)], dim=1)


def exact(case, seed):
    s, h, kind, cb = _inputs(case, seed), _hadamard(), case["kind"], case["cb"]
    if kind == "layer":
        y = _layer(s["rec"], s["x"], case["k"], case["n"], case["bits"], cb, h)
        return y + s["res"].double() if s["res"] is not None else y
    if kind == "group":
        return [_layer(r, s["x"], case["k"], n, case["bits"], cb, h)
                for r, n in zip(s["recs"], (case["n0"], case["n1"]))]
    if kind == "step":
        return [_layer(r, c["x"], c["k"], n, c["bits"], cb, h) for c in s["calls"] for r, n in zip(c["recs"], c["ns"])]
    if kind == "iface":
        w = _upstream(s["tiles"], case["k"], case["n"], case["bits"], cb)
        return _apply(s["x"], w, s["su"].double(), s["sv"].double(), h)
    if kind == "rows":
        k, n, ids = case["k"], case["n"], s["ids"].long()
        out, step = torch.empty((ids.numel(), k), dtype=torch.float64, device="cuda"), _chunk(k)
        for nb in range(0, n // 128, step):
            at = torch.nonzero((ids // 128 >= nb) & (ids // 128 < nb + step))[:, 0]
            if at.numel():
                w, su, sv = _column_group(s["rec"], k, case["bits"], cb, nb, step)
                out[at] = _original(w, su, sv, h)[:, ids[at] - 128 * nb].t()
        return out
    if kind == "dequant":
        return [_upstream(t, k, n, bits, cb) for t, bits, k, n in s["mats"]]
    w = _upstream(s["tiles"], case["k"], case["n"], case["bits"], cb)
    return _original(w, s["su"].double(), s["sv"].double(), h)


def _original(w, su, sv, h):
    k, n = w.shape
    w = ((w.view(k, n // 128, 128) @ h).view(k // 128, 128, n).transpose(1, 2) @ h).transpose(1, 2).reshape(k, n)
    return w * su[:, None] * sv[None, :]
