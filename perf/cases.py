"""What a program that runs its quantized matrices through this package asks of it, as cases to time.

A case names one public path and the sizes it is called with:

  matvec    one decode projection over GGUF rows in device memory (Device.matvec_dev)
  decode    a decoded token's matrices through a few dense blocks: RMSNorm + q/k/v, the output
            projection onto the residual, RMSNorm + gate/up, the gated down projection onto the
            residual (Device.matvec_group_dev); attention itself is not this package's
  layer     a feed-forward block handed over once and run by handle, GGUF or packed planes
            (Device.PrepLayer, layer_ffn_dev): one row with its norm in front, more rows without
  host      nn.Device.MatVec / MatMul over host memory, weights resident after the first call
  matmul    a prompt's (or a few drafted tokens') projection over GGUF rows or packed planes in device
            memory (Device.matmul_dev, matmul_packed_dev)
  moe       a mixture block, router to combine (Device.moe_block_dev), GGUF banks or packed planes
  mxfp4     MXFP4 weights x bf16 activations, GGUF rows or packed planes

Weights are blocks of N(0, 0.02) matrices quantized by this package's quantizers, drawn anew for each
seed from a pool a type; activations are N(0, 1); router logits come out N(0, 1).  The activation
window is the one the package chooses for the types at hand (quant.act_window).
"""
import math

import numpy as np
import torch

from jitllm_amd import quant, synth
from jitllm_amd.device import Device, Packed

TYPES = {"q4_k": quant.Q4_K, "q6_k": quant.Q6_K, "q8_0": quant.Q8_0, "mxfp4": quant.MXFP4}
POOL_BLOCKS = 4096


def listed():
    return [
        # the smallest projection of a small model: the launch and the host path are the whole of it
        dict(name="matvec q8_0 1024x2048", op="matvec", type="q8_0", rows=1024, k=2048),
        # the benchmark's headline matrix
        dict(name="matvec q4_k 4096x4096", op="matvec", type="q4_k", rows=4096, k=4096),
        # a token through two blocks of a mixed k-quant file (v and down in Q6_K, as such files hold them)
        dict(name="decode k-quants 4096/14336", op="decode", layers=2, n_embd=4096, n_kv=1024, n_ffn=14336, type="q4_k",
             type2="q6_k"),
        # the block seam at decode, from a container's packed planes
        dict(name="layer q8_0 planes 1 row", op="layer", packed=True, type="q8_0", down="q8_0", n_embd=4096, n_ffn=14336, rows=1),
        # the drop-in seam over host memory
        dict(name="host matvec q6_k 4096x4096", op="host", packed=False, type="q6_k", rows=4096, k=4096, ntok=1),
        # a handful of tokens: drafted tokens to verify, or small batches decoded together
        dict(name="matmul q6_k 4096x14336 x12", op="matmul", packed=False, window=256, type="q6_k", rows=4096, k=14336, ntok=12),
        # the benchmark's prompt
        dict(name="matmul q4_k 14336x4096 x512", op="matmul", packed=False, window=256, type="q4_k", rows=14336, k=4096, ntok=512),
        # a long prompt of a Q8_0 file: the largest case
        dict(name="matmul q8_0 14336x4096 x2048", op="matmul", packed=False, window=32, type="q8_0", rows=14336, k=4096,
             ntok=2048),
        # the mixture block of the benchmark, decoded in a batch
        dict(name="moe q4_k 64 rows", op="moe", packed=False, type="q4_k", down="q4_k", rows=64, n_expert=128, k_used=8,
             n_ffn=768, n_embd=2048),
        # and a prompt of a ragged length through it, Q6_K down projections
        dict(name="moe q4_k/q6_k 777 rows", op="moe", packed=False, type="q4_k", down="q6_k", rows=777, n_expert=128, k_used=8,
             n_ffn=768, n_embd=2048),
        # MXFP4 experts of the benchmark: a small batch over a container's planes, a prompt over GGUF rows
        dict(name="mxfp4 planes 2880x2880 x64", op="mxfp4", packed=True, rows=2880, k=2880, ntok=64),
        dict(name="mxfp4 rows 2880x2880 x1024", op="mxfp4", packed=False, rows=2880, k=2880, ntok=1024),
    ]


# -- drawn cases ---------------------------------------------------------------

_MOST_FLOPS = 2.0 * 14336 * 4096 * 2048       # the largest listed case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, unit):
    return max(lo, _log(rng, lo, hi) // unit * unit)


def _fit(ntok, rows, k):
    return max(1, min(ntok, int(_MOST_FLOPS / (2.0 * rows * k))))


def draw(rng):
    op = rng.choice(["matvec", "decode", "layer", "host", "matmul", "matmul", "matmul", "moe", "moe", "mxfp4", "mxfp4"])
    t = rng.choice(["q4_k", "q6_k", "q8_0"])
    unit = 32 if t == "q8_0" else 256
    if op == "matvec":
        return dict(op=op, type=t, rows=_log(rng, 256, 14336), k=_mult(rng, 512, 14336, unit))
    if op == "decode":
        n_embd = _mult(rng, 1024, 4096, 256)
        return dict(op=op, layers=rng.randint(1, 3), n_embd=n_embd, n_kv=n_embd // rng.choice([1, 2, 4]),
                    n_ffn=_mult(rng, 2 * n_embd, min(4 * n_embd, 14336), 256), type=t, type2=rng.choice([t, t, "q6_k"]))
    if op == "layer":
        n_embd = _mult(rng, 1024, 4096, 256)
        return dict(op=op, packed=rng.random() < 0.5, type=t, down=rng.choice([t, t, "q6_k"]), n_embd=n_embd,
                    n_ffn=_mult(rng, 2 * n_embd, min(4 * n_embd, 14336), 256), rows=1 if rng.random() < 0.5 else _log(rng, 2, 64))
    if op == "host":
        return dict(op=op, packed=rng.random() < 0.5, type=t, rows=_log(rng, 256, 8192), k=_mult(rng, 512, 8192, unit),
                    ntok=1 if rng.random() < 0.75 else _log(rng, 2, 32))
    if op == "matmul":
        rows, k = _log(rng, 1024, 14336), _mult(rng, 1024, 14336, 128 if t == "q8_0" else 256)
        return dict(op=op, packed=rng.random() < 0.4, window=32 if t == "q8_0" else rng.choice([256, 256, 32]), type=t, rows=rows, k=k,
                    ntok=_fit(_log(rng, 2, 2048), rows, k))
    if op == "moe":
        packed = rng.random() < 0.3
        t = "q4_k" if packed else rng.choice(["q4_k", "q4_k", "q8_0"])     # (plane banks are served in Q4_K)
        e = _log(rng, 8, 128)
        ffn = _mult(rng, 512, 2048, 256)
        return dict(op=op, packed=packed, type=t, down=rng.choice([t, "q6_k"]) if not packed else t, rows=_log(rng, 1, 1024),
                    n_expert=e, k_used=min(e // 2, rng.choice([2, 4, 8])), n_ffn=ffn, n_embd=_mult(rng, 1024, 2880, 256))
    rows, k = _log(rng, 1024, 5760), _mult(rng, 1024, 5760, 32)
    return dict(op=op, packed=rng.random() < 0.5, rows=rows, k=k, ntok=_log(rng, 1, 2048))


# -- inputs --------------------------------------------------------------------

_pools, _devices, _layer_ids = {}, {}, [0]


def _device(window):
    """The program's one device context a window, kept for its whole run."""
    if window not in _devices:
        _devices[window] = Device(device=0, act_window=window)
    return _devices[window]


def _pool(t):
    if t not in _pools:
        be, bb = quant.BLOCK[t]
        w = synth.quantized_weights(t, 64, POOL_BLOCKS * be // 64, seed=1234 + t)
        _pools[t] = torch.from_numpy(w).reshape(POOL_BLOCKS, bb).cuda()
    return _pools[t]


def _weights(t, rows, k, g):
    """GGUF rows of a [rows][k] matrix in device memory: blocks drawn from the type's pool."""
    n = rows * (k // quant.block_elems(t))
    at = torch.randint(0, POOL_BLOCKS, (n,), generator=g, device="cuda", dtype=torch.int32)
    return torch.index_select(_pool(t), 0, at).reshape(-1)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _planes(dev, t, w, rows, k):
    """The packed planes of GGUF rows w, by the package's own packer."""
    out = [torch.zeros(max(n, 4), dtype=torch.int32, device="cuda") for n in quant.packed_words(t, rows, k)]
    assert dev.pack_weights_dev(t, w.data_ptr(), rows, k, *[p.data_ptr() for p in out])
    torch.cuda.synchronize()
    return out


def _window(case):
    op = case["op"]
    if "window" in case:
        return case["window"]
    if op == "mxfp4":
        return 32
    names = {"decode": ("type", "type2"), "layer": ("type", "down"), "moe": ("type", "down")}.get(op, ("type",))
    return quant.act_window([TYPES[case[n]] for n in names])


class _Layer:
    """A block held by handle; its device memory goes with it."""

    def __init__(self, dev, *a, **kw):
        self.dev, self.id = dev, _layer_ids[0]
        _layer_ids[0] += 1
        assert dev.PrepLayer(self.id, *a, **kw)

    def __del__(self):
        self.dev.ReleaseLayers(self.id, self.id + 1)


class _HostWeights:
    """Weights in host memory; the device copy the package made of them goes with them."""

    def __init__(self, dev, arrays):
        self.dev, self.arrays = dev, arrays

    def __del__(self):
        self.dev.forget_range(self.arrays[0].ctypes.data, 4)


def _numpy(t, dtype=np.uint8):
    return np.ascontiguousarray(t.cpu().numpy().view(dtype))


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    dev, op = _device(_window(case)), case["op"]
    s = {"case": case, "op": op, "dev": dev}
    t = TYPES[case["type"]] if "type" in case else quant.MXFP4
    if op == "matvec":
        s["w"], s["x"] = _weights(t, case["rows"], case["k"], g), _normal(g, case["k"])
        s["out"] = torch.zeros(case["rows"], device="cuda")
        s["args"] = (s["out"].data_ptr(), t, s["w"].data_ptr(), s["x"].data_ptr(), case["rows"], case["k"])
    elif op == "decode":
        e, f, kv, t2 = case["n_embd"], case["n_ffn"], case["n_kv"], TYPES[case["type2"]]
        s["x"], s["y"] = _normal(g, e), torch.zeros(e, device="cuda")
        s["att"], s["norm"] = _normal(g, e), 1 + 0.1 * _normal(g, e)
        s["hold"], s["steps"], s["qkv"] = [], [], []
        for _ in range(case["layers"]):
            wq, wk, wv, wo = _weights(t, e, e, g), _weights(t, kv, e, g), _weights(t2, kv, e, g), _weights(t, e, e, g)
            wg, wu, wd = _weights(t, f, e, g), _weights(t, f, e, g), _weights(t2, e, f, g)
            q, k, v = (torch.zeros(n, device="cuda") for n in (e, kv, kv))
            gt, up = torch.zeros(f, device="cuda"), torch.zeros(f, device="cuda")
            s["hold"].append((wq, wk, wv, wo, wg, wu, wd, gt, up))
            s["qkv"] += [q, k, v]
            x, y, norm = s["x"].data_ptr(), s["y"].data_ptr(), s["norm"].data_ptr()
            s["steps"] += [
                (([q.data_ptr(), k.data_ptr(), v.data_ptr()], [t, t, t2], [wq.data_ptr(), wk.data_ptr(), wv.data_ptr()],
                  [e, kv, kv], x, e), dict(norm_w=norm, norm_eps=1e-5)),
                (([y], [t], [wo.data_ptr()], [e], s["att"].data_ptr(), e), dict(resid=x, alpha=1.0)),
                (([gt.data_ptr(), up.data_ptr()], [t, t], [wg.data_ptr(), wu.data_ptr()], [f, f], x, e),
                 dict(norm_w=norm, norm_eps=1e-5)),
                (([y], [t2], [wd.data_ptr()], [e], gt.data_ptr(), f), dict(act_up=up.data_ptr(), resid=x, alpha=1.0)),
            ]
    elif op == "layer":
        e, f, td, n = case["n_embd"], case["n_ffn"], TYPES[case["down"]], case["rows"]
        mats = [(t, f, e), (t, f, e), (td, e, f)]
        ws = [_weights(*m, g) for m in mats]
        if case["packed"]:
            ws = [tuple(_numpy(p, np.uint32) for p in _planes(dev, m[0], w, m[1], m[2])) for m, w in zip(mats, ws)]
            ws = [(p[0], p[1], None if m[0] == quant.Q8_0 else p[2]) for m, p in zip(mats, ws)]
        else:
            ws = [_numpy(w) for w in ws]
        norm = (1 + 0.1 * _normal(g, e)).cpu().numpy() if n == 1 else None
        s["layer"] = _Layer(dev, 0, t, e, f, *ws, down_type=td, norm_w=norm, norm_eps=1e-5)
        s["h"], s["resid"] = _normal(g, n, e), _normal(g, n, e)
        s["args"] = (s["layer"].id, s["h"].data_ptr(), s["resid"].data_ptr(), n)
    elif op == "host":
        rows, k, n = case["rows"], case["k"], case["ntok"]
        w = _weights(t, rows, k, g)
        s["x"], s["out"] = _normal(g, n * k).cpu().numpy(), np.zeros(n * rows, np.float32)
        if case["packed"]:
            p = [_numpy(a, np.uint32) for a in _planes(dev, t, w, rows, k)]
            s["w"] = _HostWeights(dev, p)
            s["p"] = Packed(p[0], p[1], None if t == quant.Q8_0 else p[2], 0, rows)
        else:
            s["w"] = _HostWeights(dev, [_numpy(w)])
        s["type"] = t
    elif op == "matmul":
        rows, k, n = case["rows"], case["k"], case["ntok"]
        s["x"], s["out"] = _normal(g, n, k), torch.zeros(n, rows, device="cuda")
        w = _weights(t, rows, k, g)
        if case["packed"]:
            s["w"] = _planes(dev, t, w, rows, k)
            w = Packed(*[p.data_ptr() for p in s["w"]], 0, rows)
        else:
            s["w"] = w
            w = w.data_ptr()
        s["args"] = (s["out"].data_ptr(), t, w, s["x"].data_ptr(), rows, k, n)
    elif op == "moe":
        n, ne, ku, f, e, td = case["rows"], case["n_expert"], case["k_used"], case["n_ffn"], case["n_embd"], TYPES[case["down"]]
        s["x"], s["resid"], s["router"] = _normal(g, n, e), _normal(g, n, e), _normal(g, ne, e) / math.sqrt(e)
        s["sel"], s["wt"] = torch.zeros(n, ku + 1, dtype=torch.int32, device="cuda"), torch.zeros(n, ku, device="cuda")
        mats = [(t, ne * f, e), (t, ne * f, e), (td, ne * e, f)]
        ws = [_weights(*m, g) for m in mats]
        if case["packed"]:
            s["w"] = [_planes(dev, m[0], w, m[1], m[2]) for m, w in zip(mats, ws)]
            banks = [Device.packed_bank(*[q.data_ptr() for q in p], 0, m[1]) for m, p in zip(mats, s["w"])]
        else:
            s["w"] = ws
            banks = [w.data_ptr() for w in ws]
        s["args"] = (s["resid"].data_ptr(), t, *banks, s["router"].data_ptr(), s["x"].data_ptr(), n, ku, ne, f, e)
        s["kw"] = dict(sel=s["sel"].data_ptr(), wt=s["wt"].data_ptr(), down_type=td)
    else:
        rows, k, n = case["rows"], case["k"], case["ntok"]
        s["x"], s["out"] = _normal(g, n, k).to(torch.bfloat16), torch.zeros(n, rows, device="cuda")
        w = _weights(quant.MXFP4, rows, k, g)
        if case["packed"]:
            s["w"] = _planes(dev, quant.MXFP4, w, rows, k)
            w = Packed(s["w"][0].data_ptr(), s["w"][1].data_ptr(), None, 0, rows)
        else:
            s["w"] = w
            w = w.data_ptr()
        s["args"] = (s["out"].data_ptr(), w, s["x"].data_ptr(), rows, k, n)
    return s


def _served(ok):
    if not ok:
        raise RuntimeError("declined")


def run(s):
    op, dev = s["op"], s["dev"]
    if op == "matvec":
        _served(dev.matvec_dev(*s["args"]))
        return s["out"]
    if op == "decode":
        for a, kw in s["steps"]:
            _served(dev.matvec_group_dev(*a, **kw))
        return [s["x"], s["y"]] + s["qkv"]
    if op == "layer":
        _served(dev.layer_ffn_dev(*s["args"]))
        return s["resid"]
    if op == "host":
        c = s["case"]
        if c["ntok"] == 1:
            _served(dev.MatVecPacked(s["out"], s["type"], s["p"], s["x"], c["rows"], c["k"]) if c["packed"] else
                    dev.MatVec(s["out"], s["type"], s["w"].arrays[0], s["x"], c["rows"], c["k"]))
        else:
            _served(dev.MatMulPacked(s["out"], s["type"], s["p"], s["x"], c["rows"], c["k"], c["ntok"]) if c["packed"] else
                    dev.MatMul(s["out"], s["type"], s["w"].arrays[0], s["x"], c["rows"], c["k"], c["ntok"]))
        return s["out"]
    if op == "matmul":
        _served((dev.matmul_packed_dev if s["case"]["packed"] else dev.matmul_dev)(*s["args"]))
        return s["out"]
    if op == "moe":
        _served(dev.moe_block_dev(*s["args"], **s["kw"]))
        return [s["resid"], s["sel"], s["wt"]]
    _served((dev.matmul_mxfp4_packed_bf16_dev if s["case"]["packed"] else dev.matmul_mxfp4_bf16_dev)(*s["args"]))
    return s["out"]


# -- what a pass cannot do without ----------------------------------------------

def _bytes(t, rows, k):
    return rows * quant.row_bytes(TYPES[t], k)


def work(case):
    op = case["op"]
    if op == "decode":
        e, f, kv, t, t2 = case["n_embd"], case["n_ffn"], case["n_kv"], case["type"], case["type2"]
        w = 2 * _bytes(t, e, e) + _bytes(t, kv, e) + _bytes(t2, kv, e) + 2 * _bytes(t, f, e) + _bytes(t2, e, f)
        n = 2 * e * e + 2 * kv * e + 3 * f * e
        return {"bytes": case["layers"] * (w + 4 * (e + 2 * kv)) + 4 * 4 * e, "flops": 2 * case["layers"] * n}
    if op == "layer":
        e, f, n = case["n_embd"], case["n_ffn"], case["rows"]
        return {"bytes": 2 * _bytes(case["type"], f, e) + _bytes(case["down"], e, f) + 12 * n * e, "flops": 2 * 3 * e * f * n}
    if op == "moe":
        n, ne, ku, f, e = case["rows"], case["n_expert"], case["k_used"], case["n_ffn"], case["n_embd"]
        touched = ne * (1 - (1 - ku / ne) ** n)      # experts that some row selects, on average
        sheet = 2 * _bytes(case["type"], f, e) + _bytes(case["down"], e, f)
        return {"bytes": touched * sheet + 4 * ne * e + 12 * n * e, "flops": 2 * n * (ku * 3 * e * f + ne * e)}
    t, rows, k, n = case.get("type", "mxfp4"), case["rows"], case["k"], case.get("ntok", 1)
    return {"bytes": _bytes(t, rows, k) + n * (k * (2 if op == "mxfp4" else 4) + rows * 4), "flops": 2 * rows * k * n}


def tolerance(case):
    op = case["op"]
    if op in ("decode", "layer", "moe"):
        # a second matrix behind the int8 quantizer: a 32-bit sum on a rounding boundary moves one
        # of its thousands of values by one step in 127
        return {"rel": 1e-3, "max": 0.1, "differ": 0.0}
    return {"rel": 1e-5, "max": 1e-3}
