"""The work this library does for a program that serves a model, as cases to time.

Each case goes through the public entry points (soso_amd.dispatch.HipGpu): the
host-buffer calls of GpuDispatch as soso makes them, and the device-pointer
calls of a program that keeps its activations on the card.  Weights are made as
raw soso/GGML blocks, uploaded once and kept, as a server keeps them; each pass
multiplies activations by them.

A case's "kind" says which entry point it times:
  matvec_host  HipGpu.matvec: one token, numpy in and out (soso's drop-in call)
  matmul_host  HipGpu.matmul: a block of prompt tokens, numpy in and out
  matmul       HipGpu.matmul_dev: several tokens, buffers on the card
  moe          HipGpu.moe_ffn_dev: an MoE layer's FFN from router to sum
  gdn          HipGpu.gdn_block_dev: a Gated DeltaNet block
  decode       HipGpu.decode_step_dev: one token through a whole dense model
"""
import itertools
import math

import numpy as np
import torch

from soso_amd import abi
from soso_amd.dispatch import HipGpu

Q4K, Q8, Q6K, F32 = abi.DTYPE_Q4_K, abi.DTYPE_Q8_0, abi.DTYPE_Q6_K, abi.DTYPE_F32
DTYPES = {"q4_k": Q4K, "q8_0": Q8, "q6_k": Q6K}
BLOCK = {"q4_k": (256, 144), "q8_0": (32, 36), "q6_k": (256, 210)}  # elements, bytes
DEV = "cuda"


def listed():
    return [
        # one attention projection of one token, host buffers: what soso's CPU decode loop offloads
        {"name": "matvec_host_q8", "kind": "matvec_host", "dtype": "q8_0", "rows": 4096, "cols": 4096},
        # the gate (or up) projection of a 128-token block of a prompt, host buffers
        {"name": "matmul_host_n128", "kind": "matmul_host", "dtype": "q4_k", "rows": 14336, "cols": 4096, "n": 128},
        # the same projection for eight sequences that decode together
        {"name": "matmul_q4k_n8", "kind": "matmul", "dtype": "q4_k", "rows": 14336, "cols": 4096, "n": 8},
        # the same for a long stretch of a prompt, on the card
        {"name": "matmul_q4k_n512", "kind": "matmul", "dtype": "q4_k", "rows": 14336, "cols": 4096, "n": 512},
        # the FFN down projection for the ragged end of a prompt
        {"name": "matmul_q4k_down_n199", "kind": "matmul", "dtype": "q4_k", "rows": 4096, "cols": 14336, "n": 199},
        # an attention projection of a Q8_0 model for 64 tokens
        {"name": "matmul_q8_n64", "kind": "matmul", "dtype": "q8_0", "rows": 4096, "cols": 4096, "n": 64},
        # mixed Q4_K / Q6_K files keep the down projection in Q6_K
        {"name": "matmul_q6k_down_n256", "kind": "matmul", "dtype": "q6_k", "rows": 4096, "cols": 14336, "n": 256},
        # an MoE layer (hidden 2048, 128 experts of 768, top-8): one decode token, a decode batch, a prompt block
        {"name": "moe_n1", "kind": "moe", "hdim": 2048, "ffn": 768, "n_exp": 128, "top_k": 8, "n": 1},
        {"name": "moe_n32", "kind": "moe", "hdim": 2048, "ffn": 768, "n_exp": 128, "top_k": 8, "n": 32},
        {"name": "moe_n512", "kind": "moe", "hdim": 2048, "ffn": 768, "n_exp": 128, "top_k": 8, "n": 512},
        # a Gated DeltaNet layer (16 q/k heads, 32 value heads) over a prompt block
        {"name": "gdn_n256", "kind": "gdn", "n_k": 16, "n_v": 32, "kernel": 4, "n": 256},
        # one greedy token of an 8B model with 4096 positions of context
        {"name": "decode_8b", "kind": "decode", "layers": 32, "hidden": 4096, "heads": 32, "kv_heads": 8,
         "ffn": 14336, "vocab": 128256, "pos": 4096, "kv_f16": True},
    ]


def _log(rng, lo, hi, step=1):
    """A whole multiple of `step` between lo and hi, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step)))
    return max(lo, min(hi, int(v) // step * step))


def draw(rng):
    kind = rng.choice(["matvec_host", "matmul_host", "matmul", "matmul", "moe", "gdn", "decode"])
    if kind in ("matvec_host", "matmul_host", "matmul"):
        dtype = rng.choice(sorted(DTYPES))
        step = 32 if dtype == "q8_0" else 256
        c = {"kind": kind, "dtype": dtype, "rows": _log(rng, 256, 14336), "cols": _log(rng, 512, 14336, step)}
        if kind == "matmul_host":
            c["n"] = _log(rng, 2, 128)
        elif kind == "matmul":
            most = {"q4_k": 14336 * 4096 * 512, "q8_0": 14336 * 4096 * 256, "q6_k": 4096 * 14336 * 256}[dtype]
            c["n"] = min(_log(rng, 2, 512), max(2, most // (c["rows"] * c["cols"])))
        return c
    if kind == "moe":
        return {"kind": kind, "hdim": rng.choice([1024, 2048]), "ffn": _log(rng, 256, 1536, 256),
                "n_exp": _log(rng, 16, 128), "top_k": rng.choice([2, 4, 8]), "n": _log(rng, 1, 512)}
    if kind == "gdn":
        n_k = rng.choice([2, 4, 8, 16])
        return {"kind": kind, "n_k": n_k, "n_v": n_k * rng.choice([1, 2, 4]) if n_k < 16 else 32,
                "kernel": rng.choice([2, 3, 4]), "n": _log(rng, 1, 256)}
    heads = rng.choice([8, 16, 32])
    return {"kind": kind, "layers": rng.randint(2, 12), "hidden": rng.choice([1024, 2048, 4096]), "heads": heads,
            "kv_heads": heads // rng.choice([1, 4, 8]), "ffn": rng.choice([2048, 3072, 5632, 8192, 14336]),
            "vocab": _log(rng, 8192, 128256), "pos": _log(rng, 1, 4096), "kv_f16": rng.random() < 0.5}


# ---- raw weights --------------------------------------------------------------


def _gen(seed, *what):
    g = torch.Generator(device=DEV)
    h = int(seed) * 1000003 + 12345
    for w in what:
        h = (h * 6364136223846793005 + int(w) * 2 + 1) % (1 << 62)
    g.manual_seed(h)
    return g


def _bytes(g, *shape):
    """Random bytes: whole words are drawn where the last extent allows."""
    if shape[-1] % 4 == 0:
        w = torch.randint(-(1 << 31), 1 << 31, shape[:-1] + (shape[-1] // 4,), generator=g, device=DEV,
                          dtype=torch.int32)
        return w.view(torch.uint8)
    return torch.randint(0, 256, shape, generator=g, device=DEV, dtype=torch.uint8)


def _raw(dtype, rows, cols, g):
    """Raw blocks [rows, blocks, block bytes] of a matrix whose weights have mean
    zero and a standard deviation of about 1 / sqrt(cols), as trained and
    quantized ones do: codes piled up around the middle, block scales within a
    factor of a few of each other."""
    elems, size = BLOCK[dtype]
    nb = cols // elems
    sigma = 1.0 / math.sqrt(cols)
    out = torch.empty(rows, nb, size, dtype=torch.uint8, device=DEV)
    spread = 0.5 + torch.rand(rows, nb, 1, generator=g, device=DEV)
    if dtype == "q4_k":
        # w = d sc q - dmin m: q the sum of two 3-bit numbers (mean 7), m near sc
        d = (spread * (sigma / 140)).to(torch.float16)
        out[..., 0:2] = d.view(torch.uint8)
        out[..., 2:4] = (d.float() * 7).to(torch.float16).view(torch.uint8)
        sc = torch.randint(24, 64, (rows, nb, 8), generator=g, device=DEV, dtype=torch.int16)
        m = (sc + torch.randint(-3, 4, (rows, nb, 8), generator=g, device=DEV, dtype=torch.int16)).clamp_(0, 63)
        out[..., 4:8] = ((sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6)).to(torch.uint8)
        out[..., 8:12] = ((m[..., :4] & 63) | ((m[..., 4:] >> 4) << 6)).to(torch.uint8)
        out[..., 12:16] = ((sc[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)).to(torch.uint8)
        out[..., 16:] = (_bytes(g, rows, nb, 128) & 0x77) + (_bytes(g, rows, nb, 128) & 0x77)
    elif dtype == "q8_0":
        out[..., 0:4] = (spread * (sigma / 52)).to(torch.float16).float().view(torch.uint8)
        out[..., 4:] = (_bytes(g, rows, nb, 32) & 0x7F) + (_bytes(g, rows, nb, 32) & 0x7F) - 127
    else:
        out[..., :192] = _bytes(g, rows, nb, 192)
        sc = torch.randint(32, 128, (rows, nb, 16), generator=g, device=DEV, dtype=torch.int16)
        sign = torch.randint(0, 2, (rows, nb, 16), generator=g, device=DEV, dtype=torch.int16) * 2 - 1
        out[..., 192:208] = (sc * sign).to(torch.int8).view(torch.uint8)
        out[..., 208:210] = (spread * (sigma / 1500)).to(torch.float16).view(torch.uint8)
    return out


def _dequant(dtype, raw):
    """The weights [rows, cols] of raw blocks, in 64 bits."""
    rows, nb = raw.shape[0], raw.shape[1]

    def half(a):
        return a.contiguous().view(torch.float16).double()
    if dtype == "q4_k":
        d, dmin = half(raw[..., 0:2]), half(raw[..., 2:4])
        s = raw[..., 4:16].to(torch.int16)
        lo, hi, both = s[..., 0:4], s[..., 4:8], s[..., 8:12]
        sc = torch.cat([lo & 63, (both & 15) | ((lo >> 6) << 4)], -1).double()
        m = torch.cat([hi & 63, (both >> 4) | ((hi >> 6) << 4)], -1).double()
        q = raw[..., 16:].reshape(rows, nb, 4, 32)
        q = torch.stack([q & 15, q >> 4], 3).reshape(rows, nb, 8, 32).double()
        w = (d * sc).unsqueeze(-1) * q - (dmin * m).unsqueeze(-1)
    elif dtype == "q8_0":
        w = raw[..., 0:4].contiguous().view(torch.float32).double() * raw[..., 4:].contiguous().view(torch.int8).double()
    else:
        ql = raw[..., :128].reshape(rows, nb, 2, 2, 32).to(torch.int16)
        qh = raw[..., 128:192].reshape(rows, nb, 2, 1, 32).to(torch.int16)
        shifts = torch.tensor([0, 2, 4, 6], device=raw.device, dtype=torch.int16).view(1, 1, 1, 4, 1)
        q = torch.cat([ql & 15, ql >> 4], 3) | (((qh >> shifts) & 3) << 4)
        sc = raw[..., 192:208].contiguous().view(torch.int8).double().unsqueeze(-1)
        w = half(raw[..., 208:210]).unsqueeze(-1) * sc * (q.reshape(rows, nb, 16, 16) - 32).double()
    return w.reshape(rows, -1)


def _times(dtype, raw, x):
    """x [n, cols] (64 bits) times the transposed weights, a stretch of rows at a time."""
    step = max(1, (1 << 27) // x.shape[1])
    return torch.cat([x @ _dequant(dtype, raw[r:r + step]).T.contiguous() for r in range(0, raw.shape[0], step)], 1)


def _x(n, cols, g):
    """Activations after a norm: normal, some channels a few times wider than others."""
    wide = torch.exp(0.5 * torch.randn(cols, generator=g, device=DEV))
    return torch.randn(n, cols, generator=g, device=DEV) * wide


# ---- what a program keeps --------------------------------------------------------

_gpu = None
_names = itertools.count()


def _handle():
    global _gpu
    if _gpu is None:
        torch.zeros(1, device=DEV)
        _gpu = HipGpu(0, vram_budget=256 << 30)
    return _gpu


class Kept:
    """Resident weights and registrations of one state, given back with it."""

    def __init__(self):
        self.g, self.name = _handle(), "c%d" % next(_names)
        self.keys, self.models = [], []

    def weight(self, key, raw, dtype, rows, cols):
        key = self.name + "." + key
        if not self.g.weight_from_dev(key, raw.data_ptr(), raw.numel() * raw.element_size(), dtype, rows, cols):
            raise RuntimeError(self.g.last_error())
        self.keys.append(key)
        return key

    def __del__(self):
        for m in self.models:
            self.g.decode_destroy(m)
        for k in self.keys:
            try:
                self.g.weight_drop(k)
            except Exception:  # dropped when a model fused it
                pass


def _dims(case):
    return DTYPES[case["dtype"]], case["rows"], case["cols"]


def _matmul_inputs(case, seed):
    g = _gen(seed, 1)
    raw = _raw(case["dtype"], case["rows"], case["cols"], g)
    return raw, _x(case.get("n", 1), case["cols"], g)


def _moe_inputs(case, seed):
    g = _gen(seed, 2)
    E, H, F = case["n_exp"], case["hdim"], case["ffn"]
    mats = [_raw("q4_k", E * r, c, g) for r, c in ((F, H), (F, H), (H, F))]
    router = torch.randn(E, H, generator=g, device=DEV) * 0.02
    return mats, router, torch.randn(case["n"], H, generator=g, device=DEV)


def _gdn_inputs(case, seed):
    g = _gen(seed, 3)
    n, n_k, n_v, kernel, d = case["n"], case["n_k"], case["n_v"], case["kernel"], 128
    C = (2 * n_k + n_v) * d

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEV)
    return {"hist": normal(kernel - 1 + n, C), "conv": normal(C, kernel) * 0.5, "z": normal(n, n_v * d),
            "decay": torch.exp(-0.3 * normal(n, n_v).abs()), "beta": torch.sigmoid(normal(n, n_v)),
            "norm": 1 + 0.1 * normal(d), "state": normal(n_v, d, d) * 0.05}


def _decode_shapes(case):
    H, q, kv, F = case["hidden"], case["heads"] * 128, case["kv_heads"] * 128, case["ffn"]
    return [("q", q, H), ("k", kv, H), ("v", kv, H), ("o", H, q), ("gate", F, H), ("up", F, H), ("down", H, F)]


def _decode_inputs(case, seed):
    """A layer's tensors at a time: ("layer", l, norms, raws, k rows, v rows), then ("rest", ...)."""
    H, kv, pos = case["hidden"], case["kv_heads"] * 128, case["pos"]
    half = torch.float16 if case["kv_f16"] else torch.float32
    for l in range(case["layers"]):
        g = _gen(seed, 4, l)
        norms = [1 + 0.1 * torch.randn(H, generator=g, device=DEV) for _ in range(2)]
        raws = {k: _raw("q4_k", r, c, g) for k, r, c in _decode_shapes(case)}
        rows = [torch.randn(pos, kv, generator=g, device=DEV).to(half) for _ in range(2)]
        yield "layer", l, norms, raws, rows
    g = _gen(seed, 5)
    yield ("rest", 1 + 0.1 * torch.randn(H, generator=g, device=DEV), _raw("q6_k", case["vocab"], H, g),
           torch.randn(H, generator=g, device=DEV))


EPS = {"gdn": 1e-6, "decode": 1e-5}
THETA = 500000.0


def prepare(case, seed):
    kind, kept = case["kind"], Kept()
    s = {"kind": kind, "kept": kept, "g": kept.g}
    torch.cuda.synchronize()
    if kind in ("matvec_host", "matmul_host", "matmul"):
        dt, rows, cols = _dims(case)
        raw, x = _matmul_inputs(case, seed)
        torch.cuda.synchronize()
        s["key"], s["dims"], s["n"] = kept.weight("w", raw, dt, rows, cols), (dt, rows, cols), case.get("n", 1)
        if kind == "matmul":
            s["x"], s["y"] = x, torch.empty(case["n"], rows, device=DEV)
        else:
            s["x"] = x.cpu().numpy().reshape(-1 if kind == "matvec_host" else (case["n"], cols))
            s["y"] = np.zeros((case.get("n", 1), rows), np.float32)
    elif kind == "moe":
        E, H, F = case["n_exp"], case["hdim"], case["ffn"]
        mats, router, s["x"] = _moe_inputs(case, seed)
        torch.cuda.synchronize()
        keys = [kept.weight("E%d.%d" % (e, j), mats[j][e * r:(e + 1) * r], Q4K, r, c)
                for e in range(E) for j, (r, c) in enumerate(((F, H), (F, H), (H, F)))]
        rk = kept.weight("router", router, F32, E, H)
        s["layer"], s["n"], s["y"] = kept.name, case["n"], torch.empty(case["n"], H, device=DEV)
        if not kept.g.moe_register(kept.name, rk, keys, E, H, F, case["top_k"]):
            raise RuntimeError(kept.g.last_error())
    elif kind == "gdn":
        t = _gdn_inputs(case, seed)
        s.update(t, out=torch.empty_like(t["z"]), case=dict(case))
    else:
        keys, caches = [], []
        for part in _decode_inputs(case, seed):
            torch.cuda.synchronize()
            if part[0] == "layer":
                _, l, norms, raws, rows = part
                k = {j: kept.weight("%d.%s" % (l, j), raws[j], Q4K, r, c) for j, r, c in _decode_shapes(case)}
                n0, n1 = [kept.weight("%d.n%d" % (l, i), w, F32, 1, w.numel()) for i, w in enumerate(norms)]
                keys += [n0, k["q"], k["k"], k["v"], k["o"], n1, k["gate"], k["up"], k["down"]]
                caches.append(rows)
            else:
                _, norm, head, s["x"] = part
                keys += [kept.weight("norm", norm, F32, 1, norm.numel()),
                         kept.weight("head", head, Q6K, case["vocab"], case["hidden"])]
        cfg = dict(n_layers=case["layers"], hidden=case["hidden"], n_heads=case["heads"],
                   n_kv_heads=case["kv_heads"], head_dim=128, ffn=case["ffn"], vocab=case["vocab"],
                   ctx_max=case["pos"] + 1, rope_theta=THETA, rms_eps=EPS["decode"], kv_f16=int(case["kv_f16"]))
        if not kept.g.decode_create(kept.name, cfg, keys, drop_sources=True):
            raise RuntimeError(kept.g.last_error())
        kept.models.append(kept.name)
        for l, (k, v) in enumerate(caches):
            kept.g.decode_kv_upload(kept.name, l, 0, (k.data_ptr(), case["pos"]), (v.data_ptr(), case["pos"]),
                                    rows_f32=not case["kv_f16"])
        s["pos"], s["logits"] = case["pos"], torch.empty(case["vocab"], device=DEV)
        s["token"] = torch.zeros(1, dtype=torch.int32, device=DEV)
        s["kv_rows"] = torch.empty(case["layers"], 2, case["kv_heads"] * 128, device=DEV,
                                   dtype=torch.float16 if case["kv_f16"] else torch.float32)
    torch.cuda.synchronize()
    return s


def run(s):
    g, kind = s["g"], s["kind"]
    if kind == "matvec_host":
        ok = g.matvec(s["key"], None, *s["dims"], s["x"], s["y"])
        out = s["y"]
    elif kind == "matmul_host":
        ok = g.matmul(s["key"], None, *s["dims"], s["n"], s["x"], s["y"])
        out = s["y"]
    elif kind == "matmul":
        ok = g.matmul_dev(s["key"], s["n"], s["x"].data_ptr(), s["y"].data_ptr())
        out = s["y"]
    elif kind == "moe":
        ok = g.moe_ffn_dev(s["layer"], s["x"].data_ptr(), s["n"], s["y"].data_ptr())
        out = s["y"]
    elif kind == "gdn":
        c = s["case"]
        ok = g.gdn_block_dev(*[s[k].data_ptr() for k in ("hist", "conv", "z", "decay", "beta", "norm", "state", "out")],
                             c["n"], c["n_k"], c["n_v"], 128, c["kernel"], EPS["gdn"])
        out = {"out": s["out"], "state": s["state"]}
    else:
        ok = g.decode_step_dev(s["kept"].name, s["x"].data_ptr(), s["pos"], s["logits"].data_ptr(),
                               s["token"].data_ptr(), s["kv_rows"].data_ptr())
        out = {"logits": s["logits"], "token": s["token"], "kv_rows": s["kv_rows"]}
    if not ok:
        raise RuntimeError(g.last_error())
    return out


# ---- what the path cannot do without ----------------------------------------------


def _bytes_of(dtype, rows, cols):
    elems, size = BLOCK[dtype]
    return rows * (cols // elems) * size


def work(case):
    kind = case["kind"]
    if kind in ("matvec_host", "matmul_host", "matmul"):
        r, c, n = case["rows"], case["cols"], case.get("n", 1)
        return {"bytes": _bytes_of(case["dtype"], r, c) + 4 * n * (r + c), "flops": 2.0 * n * r * c}
    if kind == "moe":
        E, H, F, K, n = case["n_exp"], case["hdim"], case["ffn"], case["top_k"], case["n"]
        active = E * (1 - (1 - min(K, E) / E) ** n)  # experts that n tokens are expected to choose
        return {"bytes": 4 * E * H + active * 3 * _bytes_of("q4_k", F, H) + 8 * n * H,
                "flops": 2.0 * n * H * (E + 3 * F * K)}
    if kind == "gdn":
        n, n_k, n_v, d = case["n"], case["n_k"], case["n_v"], 128
        C = (2 * n_k + n_v) * d
        return {"bytes": 4 * ((case["kernel"] - 1 + n) * C + C * case["kernel"] + 2 * n * n_v * (d + 1) + d
                              + 2 * n_v * d * d),
                "flops": n * (7.0 * n_v * d * d + 2.0 * C * case["kernel"])}
    weights = sum(_bytes_of("q4_k", r, c) for _, r, c in _decode_shapes(case)) * case["layers"]
    head = _bytes_of("q6_k", case["vocab"], case["hidden"])
    kv, T = case["kv_heads"] * 128, case["pos"] + 1
    cache = case["layers"] * 2 * T * kv * (2 if case["kv_f16"] else 4)
    flops = 2.0 * case["vocab"] * case["hidden"] + case["layers"] * (
        sum(2.0 * r * c for _, r, c in _decode_shapes(case)) + 4.0 * case["heads"] * 128 * T)
    return {"bytes": weights + head + cache + 4 * (case["vocab"] + case["hidden"] * (1 + 2 * case["layers"])),
            "flops": flops}


def tolerance(case):
    """Products and recurrences in 32 bits; a whole model carries a rounding of
    its f16 KV rows through every layer that follows."""
    if case["kind"] == "decode":
        return {"rel": 2.5e-4, "max": 2e-3}
    return {"rel": 1e-5, "max": 1e-4}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("matvec_host", "matmul_host", "matmul"):
        raw, x = _matmul_inputs(case, seed)
        y = _times(case["dtype"], raw, x.double())
        return y if kind == "matmul" else y.cpu().numpy()
    if kind == "moe":
        E, H, F, K = case["n_exp"], case["hdim"], case["ffn"], case["top_k"]
        mats, router, x = _moe_inputs(case, seed)
        x = x.double()
        p = torch.softmax(x @ router.double().T.contiguous(), -1)
        top, idx = torch.topk(p, K)
        top = top / top.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for e in range(E):
            t, j = (idx == e).nonzero(as_tuple=True)
            if t.numel():
                gate, up = (_times("q4_k", m[e * F:(e + 1) * F], x[t]) for m in mats[:2])
                down = _times("q4_k", mats[2][e * H:(e + 1) * H], torch.nn.functional.silu(gate) * up)
                y.index_add_(0, t, down * top[t, j].unsqueeze(-1))
        return y
    if kind == "gdn":
        return _exact_gdn(case, seed)
    return _exact_decode(case, seed)


def _exact_gdn(case, seed):
    t = {k: v.double() for k, v in _gdn_inputs(case, seed).items()}
    n, n_k, n_v, d = case["n"], case["n_k"], case["n_v"], 128
    u = sum(t["hist"][k:k + n] * t["conv"][:, k] for k in range(case["kernel"]))
    u = torch.nn.functional.silu(u)

    def unit(a):
        return a / torch.sqrt((a * a).sum(-1, keepdim=True) + EPS["gdn"])
    q = unit(u[:, :n_k * d].reshape(n, n_k, d)) / math.sqrt(d)
    k = unit(u[:, n_k * d:2 * n_k * d].reshape(n, n_k, d))
    v = u[:, 2 * n_k * d:].reshape(n, n_v, d)
    head = torch.arange(n_v, device=DEV) % n_k
    S, outs = t["state"], []
    for i in range(n):
        qi, ki, g = q[i, head], k[i, head], t["decay"][i].view(-1, 1, 1)
        delta = (v[i] - g[..., 0] * (S * ki.unsqueeze(-1)).sum(1)) * t["beta"][i].unsqueeze(-1)
        S = g * S + ki.unsqueeze(-1) * delta.unsqueeze(1)
        outs.append((S * qi.unsqueeze(-1)).sum(1))
    o = torch.stack(outs)
    o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + EPS["gdn"]) * t["norm"]
    return {"out": o.reshape(n, n_v * d) * torch.nn.functional.silu(t["z"]), "state": S}


def _exact_decode(case, seed):
    pos, heads, kvh = case["pos"], case["heads"], case["kv_heads"]
    parts = list(p for p in _decode_inputs(case, seed) if p[0] == "rest")
    _, out_norm, head, x = parts[0]
    half = torch.float16 if case["kv_f16"] else torch.float64
    freq = THETA ** (-torch.arange(0, 128, 2, device=DEV, dtype=torch.float64) / 128)
    cos, sin = torch.cos(pos * freq), torch.sin(pos * freq)

    def norm(a, w):
        return a / torch.sqrt((a * a).mean() + EPS["decode"]) * w.double()

    def rope(a):
        a = a.reshape(-1, 64, 2)
        return torch.stack([a[..., 0] * cos - a[..., 1] * sin, a[..., 0] * sin + a[..., 1] * cos], -1).reshape(-1, 128)

    def mv(raw, a):
        return _times("q4_k", raw, a.view(1, -1)).view(-1)
    h, kv_rows = x.double(), []
    for part in _decode_inputs(case, seed):
        if part[0] != "layer":
            break
        _, _, norms, raws, (K, V) = part
        a = norm(h, norms[0])
        q, k, v = rope(mv(raws["q"], a)), rope(mv(raws["k"], a)), mv(raws["v"], a)
        k, v = k.reshape(-1).to(half), v.to(half)
        kv_rows.append(torch.stack([k, v]).double())
        K = torch.cat([K.double(), k.double().view(1, -1)]).reshape(pos + 1, kvh, 128)
        V = torch.cat([V.double(), v.double().view(1, -1)]).reshape(pos + 1, kvh, 128)
        att = torch.empty(heads, 128, device=DEV, dtype=torch.float64)
        for j in range(heads):
            kv = j // (heads // kvh)
            p = torch.softmax((K[:, kv] * q[j]).sum(-1) / math.sqrt(128), 0)
            att[j] = (V[:, kv] * p.unsqueeze(-1)).sum(0)
        h = h + mv(raws["o"], att.reshape(-1))
        a = norm(h, norms[1])
        h = h + mv(raws["down"], torch.nn.functional.silu(mv(raws["gate"], a)) * mv(raws["up"], a))
    logits = _times("q6_k", head, norm(h, out_norm).view(1, -1)).view(-1)
    return {"logits": logits, "token": None, "kv_rows": torch.stack(kv_rows)}
