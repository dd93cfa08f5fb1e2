"""The work this framework is measured on: its public entry points over the
sizes, types and options of the models it serves.

  kernel level  lrs_matvec_* / lrs_gemm_* / lrs_weight_dequant_dev through
                Weight, gemm_group and quantize_q8_0's device form: what a host
                program that keeps its own buffers calls
  model level   ResidentForward / HybridForward: a prompt block
                (decode_batch) and forced decode steps, with their logits

Layers have the shapes of the 32B dense and the 27B hybrid configurations
(model.py QWEN25_32B / QWEN35_27B) or of the 14B layer set; models take a few
such layers and a 32000-word vocabulary, so that a prepared state is quick to
make.  Weights are GGUF blocks drawn from the seed: every sub-block scale and
quant value occurs, minima cancel the quants' mean, Q6_K super-blocks hold a
scale of -128 (as a quantizer that normalises to the largest scale leaves),
and weights have an r.m.s. of 1 / sqrt(n_in).  Activations are normal with a
few channels eight times larger.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
TYPE = {"q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}
DEV = "cuda"

DENSE = dict(n_layer=4, n_embd=5120, n_head=40, n_head_kv=8, head_dim=128, n_ff=27648,
             vocab=32000, rope_dim=128, ctx=4096, rms_eps=1e-6, freq_base=1e6)
HYBRID = dict(n_layer=4, n_embd=5120, n_head=24, n_head_kv=4, head_dim=256, n_ff=17408,
              vocab=32000, rope_dim=64, ctx=4096, rms_eps=1e-6, freq_base=1e7,
              full_attn_interval=4, dn_k_heads=16, dn_v_heads=16, dn_state=128, dn_conv=4)
# the Q4_K_M mix: v, down and the head in Q6_K; the Q5_K_M one likewise
MIX = {"q4_k_m": (Q4_K, Q6_K), "q5_k_m": (Q5_K, Q6_K), "q8_0": (Q8_0, Q8_0)}
WIDE = ("attn_v", "ffn_down", "output")  # the matrices of the mix's second type


def _product():
    """The package (its folder's name is no Python identifier)."""
    if "llama_rs_amd" not in sys.modules:
        pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llama.rs_amd")
        spec = importlib.util.spec_from_file_location(
            "llama_rs_amd", os.path.join(pkg, "__init__.py"), submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["llama_rs_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["llama_rs_amd"]


_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = _product().Context(0)
    return _ctx


class _Buf:
    """A torch tensor as the device buffer that the *_dev calls take."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one Q8_0 projection of a 4096-wide model, called by itself: launch
        # latency counts as much as its 17.9 MB
        dict(name="matvec_q8_0", kind="matvec", type="q8_0", n_in=4096, n_out=4096, cols=1),
        # the GpuMatmul interface: host vector in, host vector out, one call
        # at a time (the smallest case)
        dict(name="matvec_host_q6_k", kind="matvec_host", type="q6_k", n_in=5120, n_out=1024, cols=1),
        # a few sequences side by side through one gate matrix, ragged rows
        dict(name="matvec_q4_k_6_cols", kind="matvec", type="q4_k", n_in=5120, n_out=13800, cols=6),
        # bf16 prompt GEMM of the 14B gate matrix
        dict(name="gemm_bf16_q4_k", kind="gemm", type="q4_k", n_in=5120, n_out=13824, m=512, prec=1),
        # f32-grade prompt GEMM of the 14B down matrix, a ragged prompt
        dict(name="gemm_f32_q6_k", kind="gemm", type="q6_k", n_in=13824, n_out=5120, m=201, prec=3),
        # q / k / v of a short prompt in one call
        dict(name="gemm_qkv_group", kind="group", type="q4_k", type2="q6_k", n_in=5120, n_out=5120,
             n_kv=1024, m=77, prec=3),
        # a resident weight back to f32 (checks, conversion, LoRA merges)
        dict(name="dequant_q5_k", kind="dequant", type="q5_k", n_in=5120, n_out=5120),
        # token-by-token decode of the dense model in a short context
        dict(name="decode_dense", kind="dense", mix="q4_k_m", pos=600, prompt=0, steps=8),
        # ... and near the end of its 4096 positions, where attention counts
        dict(name="decode_dense_long", kind="dense", mix="q4_k_m", pos=3900, prompt=0, steps=4),
        # a whole prompt block of the dense model (the largest case)
        dict(name="prompt_dense", kind="dense", mix="q4_k_m", pos=0, prompt=512, steps=0),
        # a short follow-up turn behind a context that is already there
        dict(name="prompt_dense_short", kind="dense", mix="q4_k_m", pos=333, prompt=19, steps=0),
        # a turn of the hybrid model: its state starts empty, a ragged prompt,
        # then decode steps
        dict(name="turn_hybrid", kind="hybrid", mix="q4_k_m", pos=0, prompt=300, steps=6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "matvec_host", "gemm", "gemm", "gemm", "group", "dequant",
                       "dense", "dense", "dense", "hybrid"])
    t = rng.choice(list(TYPE))
    wide = 256 * _log(rng, 4, 108)  # row lengths from 1024 to the 27648 of the 32B down matrix
    rows = _log(rng, 500, 28000)
    if kind in ("matvec", "matvec_host"):
        if t == "q8_0":
            wide = min(14336, wide) - 32 * rng.choice([0, 1])  # odd block counts too
        return dict(kind=kind, type=t, n_in=wide, n_out=rows,
                    cols=rng.choice([1, 1, 1, 2, 3, 5, 8, 13]) if kind == "matvec" else 1)
    if kind == "gemm":
        # at most the work of 512 tokens through a 27648 x 5120 matrix
        rows = min(rows, 27648 * 5120 // wide)
        return dict(kind=kind, type=t, n_in=wide, n_out=rows, m=_log(rng, 2, 1024), prec=rng.choice([1, 3, 3]))
    if kind == "group":
        t = rng.choice(["q4_k", "q5_k"])
        return dict(kind=kind, type=t, type2="q6_k", n_in=256 * _log(rng, 4, 24), n_out=_log(rng, 500, 6000),
                    n_kv=_log(rng, 250, 2100), m=_log(rng, 2, 512), prec=rng.choice([1, 3]))
    if kind == "dequant":
        return dict(kind=kind, type=t, n_in=min(wide, 8192), n_out=min(rows, 8000))
    if kind == "dense":
        mix = rng.choice(["q4_k_m", "q4_k_m", "q5_k_m", "q8_0"])
        if rng.random() < 0.35:
            return dict(kind=kind, mix=mix, pos=_log(rng, 1, 4000), prompt=0, steps=rng.randrange(2, 7))
        n = _log(rng, 2, 500)
        return dict(kind=kind, mix=mix, pos=rng.choice([0, rng.randrange(1, 3000)]), prompt=n, steps=0)
    return dict(kind="hybrid", mix=rng.choice(["q4_k_m", "q5_k_m"]), pos=0, prompt=_log(rng, 2, 450),
                steps=rng.randrange(0, 5))


# ---------------------------------------------------------------------------
# inputs from a seed
# ---------------------------------------------------------------------------
def _gen(seed, *path):
    """A generator of its own for every tensor of a seed."""
    h = int(seed) & 0xFFFFFFFFFFFF
    for p in path:
        h = (h * 1000003 + p + 1) % (1 << 61)
    g = torch.Generator(device=DEV)
    g.manual_seed(h)
    return g


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _blocks(g, t, n_out, n_in, rms):
    """GGUF blocks [blocks, bytes] (on the GPU) of an n_out x n_in matrix."""
    be, bb = BLOCK[t]
    n = n_out * n_in // be
    b = torch.randint(0, 256, (n, bb), generator=g, device=DEV, dtype=torch.uint8)
    u = 0.7 + 0.6 * torch.rand(n, generator=g, device=DEV)
    if t == Q8_0:
        b[:, 0:2] = _f16_bytes(u * (rms / 74.0))
        return b
    if t == Q6_K:
        at = torch.randint(0, 16, (n, 1), generator=g, device=DEV)
        b[:, 192:208].scatter_(1, at, 128)  # int8 -128
        b[:, 208:210] = _f16_bytes(u * (rms / 1400.0))
        return b
    mid, spread = (7.5, 4.6) if t == Q4_K else (15.5, 9.2)
    d = u * (rms / (37.0 * spread))
    b[:, 0:2] = _f16_bytes(d)
    b[:, 2:4] = _f16_bytes(d * mid)
    sc = torch.randint(0, 64, (n, 8), generator=g, device=DEV, dtype=torch.int32)
    m = (sc + torch.randint(-3, 4, (n, 8), generator=g, device=DEV, dtype=torch.int32)).clamp(0, 63)
    b[:, 4:8] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
    b[:, 8:12] = (m[:, :4] | ((m[:, 4:] >> 4) << 6)).to(torch.uint8)
    b[:, 12:16] = ((sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)).to(torch.uint8)
    return b


def _upload(g, t, n_out, n_in, rms):
    host = _blocks(g, t, n_out, n_in, rms).cpu().numpy().reshape(-1)
    return _product().Weight.upload(_context(), t, host, n_in, n_out)


def _activations(g, m, n):
    x = torch.randn(m, n, generator=g, device=DEV, dtype=torch.float32)
    big = torch.rand(n, generator=g, device=DEV) < 0.01
    return torch.where(big, 8.0 * x, x).contiguous()


def _uniform(g, n, lo, hi):
    return (lo + (hi - lo) * torch.rand(n, generator=g, device=DEV)).to(torch.float32)


def _matrices(cfg, mix, layer):
    """name -> (type, n_out, n_in) of a layer's quantized matrices."""
    first, second = MIX[mix]
    E, F = cfg["n_embd"], cfg["n_ff"]
    q, kv = cfg["n_head"] * cfg["head_dim"], cfg["n_head_kv"] * cfg["head_dim"]
    sh = dict(ffn_gate=(F, E), ffn_up=(F, E), ffn_down=(E, F))
    if "full_attn_interval" not in cfg:
        sh.update(attn_q=(q, E), attn_k=(kv, E), attn_v=(kv, E), attn_output=(E, q))
    elif (layer + 1) % cfg["full_attn_interval"] == 0:
        sh.update(attn_q=(2 * q, E), attn_k=(kv, E), attn_v=(kv, E), attn_output=(E, q))
    else:
        vd = cfg["dn_v_heads"] * cfg["dn_state"]
        sh.update(ssm_qkv=(2 * cfg["dn_k_heads"] * cfg["dn_state"] + vd, E), ssm_gate=(vd, E), ssm_out=(E, vd))
    return {k: (second if k in WIDE else first, *sh[k]) for k in sorted(sh)}


def _vectors(cfg, seed, layer):
    """name -> f32 vector (on the GPU) of a layer."""
    E = cfg["n_embd"]
    q, kv = cfg["n_head"] * cfg["head_dim"], cfg["n_head_kv"] * cfg["head_dim"]
    r = 1.7 / math.sqrt(E)
    if "full_attn_interval" not in cfg:
        want = dict(attn_norm=(E, 0.9, 1.1), ffn_norm=(E, 0.9, 1.1), bq=(q, -0.1, 0.1), bk=(kv, -0.1, 0.1),
                    bv=(kv, -0.1, 0.1))
    else:
        want = dict(attn_norm=(E, 0.9, 1.1), post_norm=(E, 0.9, 1.1))
        if (layer + 1) % cfg["full_attn_interval"] == 0:
            want.update(q_norm=(cfg["head_dim"], 0.9, 1.1), k_norm=(cfg["head_dim"], 0.9, 1.1))
        else:
            nv = cfg["dn_v_heads"]
            cd = (2 * cfg["dn_k_heads"] + nv) * cfg["dn_state"]
            want.update(ssm_alpha=(nv * E, -r, r), ssm_beta=(nv * E, -r, r), ssm_a=(nv, -1.0, -0.1),
                        ssm_dt=(nv, -1.0, 1.0), ssm_conv=(cd * cfg["dn_conv"], -0.5, 0.5),
                        ssm_norm=(cfg["dn_state"], 0.9, 1.1))
    return {k: _uniform(_gen(seed, 2, layer, i), *want[k]) for i, k in enumerate(sorted(want))}


def _ends(cfg, mix):
    return dict(token_embd=(MIX[mix][0], 0.5), output=(MIX[mix][1], 1.0 / math.sqrt(cfg["n_embd"])))


def _cfg(case):
    return DENSE if case["kind"] == "dense" else HYBRID


def _tokens(case, seed):
    n = case["pos"] + case["prompt"] + case["steps"]
    r = np.random.default_rng([seed, 7])
    return r.integers(0, _cfg(case)["vocab"], n).astype(np.uint32)


def prepare(case, seed):
    lrs, k = _product(), case["kind"]
    if k in ("dense", "hybrid"):
        return _prepare_model(case, seed)
    t, n_in, n_out = TYPE[case["type"]], case["n_in"], case["n_out"]
    rms = 1.0 / math.sqrt(n_in)
    s = dict(case=case, w=_upload(_gen(seed, 0), t, n_out, n_in, rms))
    if k == "dequant":
        s["y"] = torch.empty(n_out, n_in, device=DEV)
        s["yb"] = _Buf(s["y"])
    elif k == "group":
        t2, kv = TYPE[case["type2"]], case["n_kv"]
        s["ws"] = [s["w"], _upload(_gen(seed, 1), t, kv, n_in, rms), _upload(_gen(seed, 2), t2, kv, n_in, rms)]
        s["x"] = _activations(_gen(seed, 3), case["m"], n_in)
        s["y"] = [torch.empty(case["m"], w.n_out, device=DEV) for w in s["ws"]]
        import ctypes as C
        s["wa"] = (C.c_void_p * 3)(*[w.h for w in s["ws"]])
        s["ya"] = (C.c_void_p * 3)(*[y.data_ptr() for y in s["y"]])
    else:
        m = case["cols"] if "cols" in case else case["m"]
        s["x"] = _activations(_gen(seed, 3), m, n_in)
        if k == "matvec_host":
            s["x"] = s["x"].cpu().numpy().reshape(-1)
        else:
            s["y"] = torch.empty(m, n_out, device=DEV)
            s["xb"], s["yb"] = _Buf(s["x"]), _Buf(s["y"])
    torch.cuda.synchronize()
    if k in ("gemm", "group"):
        run(s)  # the context's scratch has its size before a program's steady work
        lrs.check(lrs.lib.lrs_ctx_sync(_context().h))
    return s


def _prepare_model(case, seed):
    _product()
    from llama_rs_amd.model import HybridForward, ResidentForward

    cfg, mix, ctx = _cfg(case), case["mix"], _context()
    layers = []
    for l in range(cfg["n_layer"]):
        L = {n: _upload(_gen(seed, 1, l, i), t, o, n_in, 1.0 / math.sqrt(n_in))
             for i, (n, (t, o, n_in)) in enumerate(_matrices(cfg, mix, l).items())}
        L.update({n: v.cpu().numpy() for n, v in _vectors(cfg, seed, l).items()})
        layers.append(L)
    ends = [_upload(_gen(seed, 3, i), t, cfg["vocab"], cfg["n_embd"], rms)
            for i, (t, rms) in enumerate(_ends(cfg, mix).values())]
    norm = _uniform(_gen(seed, 4), cfg["n_embd"], 0.9, 1.1).cpu().numpy()
    m = (ResidentForward if case["kind"] == "dense" else HybridForward)(ctx, cfg, layers, ends[0], norm, ends[1])
    toks = _tokens(case, seed)
    if case["pos"]:  # the context that is there before the call
        m.decode_batch(toks[:case["pos"]], 0)
    return dict(case=case, m=m, toks=toks)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    k = case["kind"]
    if k in ("dense", "hybrid"):
        m, toks, at, out = s["m"], s["toks"], case["pos"], []
        if k == "hybrid":
            m.reset()  # a new conversation: the recurrent state cannot be rewound
        if case["prompt"]:
            out.append(m.decode_batch(toks[at:at + case["prompt"]], at))
            at += case["prompt"]
        for i in range(case["steps"]):
            out.append(m.decode(toks[at + i], at + i))
        return out
    w = s["w"]
    if k == "matvec":
        w.matvec_dev(s["xb"], s["yb"], case["cols"])
    elif k == "matvec_host":
        return w.matvec(s["x"])
    elif k == "gemm":
        w.gemm_dev(s["xb"], s["yb"], case["m"], case["prec"])
    elif k == "group":
        lrs = _product()
        lrs.check(lrs.lib.lrs_gemm_group_dev(_context().h, s["wa"], 3, s["x"].data_ptr(), s["ya"], case["m"],
                                             case["prec"]))
    else:
        w.dequant_dev(s["yb"])
    return s["y"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _bytes(t, n_out, n_in):
    return n_out * n_in // BLOCK[t][0] * BLOCK[t][1]


def work(case):
    k = case["kind"]
    if k in ("dense", "hybrid"):
        return _work_model(case)
    t, n_in, n_out = TYPE[case["type"]], case["n_in"], case["n_out"]
    b = _bytes(t, n_out, n_in)
    if k == "dequant":
        return dict(bytes=b + 4 * n_in * n_out, flops=n_in * n_out)
    m = case["cols"] if "cols" in case else case["m"]
    rows = n_out
    if k == "group":
        rows += 2 * case["n_kv"]
        b += _bytes(t, case["n_kv"], n_in) + _bytes(TYPE[case["type2"]], case["n_kv"], n_in)
    return dict(bytes=b + 4 * m * (n_in + rows), flops=2 * m * n_in * rows)


def _work_model(case):
    cfg, mix = _cfg(case), case["mix"]
    mats = [v for l in range(cfg["n_layer"]) for v in _matrices(cfg, mix, l).values()]
    wb, el = sum(_bytes(*v) for v in mats), sum(v[1] * v[2] for v in mats)
    head = _bytes(MIX[mix][1], cfg["vocab"], cfg["n_embd"])
    every = cfg.get("full_attn_interval", 1)
    na = cfg["n_layer"] // every
    row = 4 * cfg["n_head_kv"] * cfg["head_dim"]  # bytes of a position's K and V
    qd = cfg["n_head"] * cfg["head_dim"]
    state = 0
    if every > 1:
        state = 8 * (cfg["n_layer"] - na) * cfg["dn_v_heads"] * cfg["dn_state"] ** 2  # read and written
    b = f = 0
    at = case["pos"]
    for n in ([case["prompt"]] if case["prompt"] else []) + [1] * case["steps"]:
        b += wb + head + na * row * (at + n) + state + 4 * cfg["vocab"]
        f += 2 * el * n + 2 * cfg["vocab"] * cfg["n_embd"] + na * 4 * qd * n * (at + (n + 1) // 2)
        at += n
    return dict(bytes=b, flops=f)


def tolerance(case):
    # errors against exact() as first measured, times about four: 22-bit
    # activations in the matvec 0.8-1.5e-6, bf16 hi + lo GEMM operands 4e-6,
    # both operands in bf16 2.4e-3; whole models 1e-5-2e-4 (values next to a
    # rounding boundary of the f16 cache fall on its other side)
    k = case["kind"]
    if k == "dequant":
        return "exact"
    if k in ("matvec", "matvec_host"):
        return {"rel": 5e-6, "max": 5e-5}
    if k in ("gemm", "group"):
        return {"rel": 1e-2, "max": 1e-1} if case["prec"] == 1 else {"rel": 2e-5, "max": 2e-4}
    return {"rel": 1e-3, "max": 1e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(t, b, n_out, n_in):
    """GGUF blocks to float64 [n_out, n_in] (ggml block layouts)."""
    n = b.shape[0]
    if t == Q8_0:
        return (b[:, 2:].contiguous().view(torch.int8).double() * _f16(b[:, :2])).reshape(n_out, n_in)
    if t == Q6_K:
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.stack((ql & 15, ql >> 4), 2)  # half, low / high nibble, a / b, 32
        sh = torch.arange(4, device=DEV, dtype=torch.uint8).reshape(1, 1, 2, 2, 1)
        q = (lo | (((qh.reshape(n, 2, 1, 1, 32) >> (2 * sh)) & 3) << 4)).to(torch.int16) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.int16).reshape(n, 2, 2, 2, 2, 1)
        v = (q.reshape(n, 2, 2, 2, 2, 16) * sc).double().reshape(n, 256) * _f16(b[:, 208:210])
        return v.reshape(n_out, n_in)
    s = b[:, 4:16].to(torch.int32)
    sc = torch.cat((s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)), 1).reshape(n, 4, 2, 1)
    mn = torch.cat((s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)), 1).reshape(n, 4, 2, 1)
    qs = b[:, 16 if t == Q4_K else 48:].reshape(n, 4, 32)
    q = torch.stack((qs & 15, qs >> 4), 2)
    if t == Q5_K:
        sh = torch.arange(8, device=DEV, dtype=torch.uint8).reshape(1, 4, 2, 1)
        q = q | (((b[:, 16:48].reshape(n, 1, 1, 32) >> sh) & 1) << 4)
    d, dm = _f16(b[:, :2]).reshape(n, 1, 1, 1), _f16(b[:, 2:4]).reshape(n, 1, 1, 1)
    return (d * (sc * q.to(torch.int32)).double() - dm * mn.double()).reshape(n_out, n_in)


def _mat(g, t, n_out, n_in, rms):
    return _dequant(t, _blocks(g, t, n_out, n_in, rms), n_out, n_in)


def exact(case, seed):
    k = case["kind"]
    if k in ("dense", "hybrid"):
        return _exact_model(case, seed)
    t, n_in, n_out = TYPE[case["type"]], case["n_in"], case["n_out"]
    rms = 1.0 / math.sqrt(n_in)
    w = _mat(_gen(seed, 0), t, n_out, n_in, rms)
    if k == "dequant":
        return w
    x = _activations(_gen(seed, 3), case["cols"] if "cols" in case else case["m"], n_in).double()
    if k == "group":
        kv = case["n_kv"]
        return [x @ w.T, x @ _mat(_gen(seed, 1), t, kv, n_in, rms).T,
                x @ _mat(_gen(seed, 2), TYPE[case["type2"]], kv, n_in, rms).T]
    y = x @ w.T
    return y.reshape(-1) if k == "matvec_host" else y


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _rope(x, cfg):
    """Adjacent-pair rotation of the first rope_dim dims; x [n, heads, head_dim]."""
    half = cfg["rope_dim"] // 2
    i = torch.arange(half, device=DEV, dtype=torch.float64)
    th = torch.arange(x.shape[0], device=DEV, dtype=torch.float64)[:, None] * cfg["freq_base"] ** (
        -2.0 * i / cfg["rope_dim"])
    c, s = torch.cos(th)[:, None], torch.sin(th)[:, None]
    a, b = x[..., 0:2 * half:2].clone(), x[..., 1:2 * half:2].clone()
    x = x.clone()
    x[..., 0:2 * half:2] = a * c - b * s
    x[..., 1:2 * half:2] = a * s + b * c
    return x


def _attend(q, k, v, cfg):
    """Causal attention, q [n, H, D] over the f16 cache's k, v [n, KV, D]."""
    k, v = k.half().double(), v.half().double()  # the cache holds f16
    n, H, D = q.shape
    rep = H // cfg["n_head_kv"]
    out = torch.empty_like(q)
    pos = torch.arange(n, device=DEV)
    for g in range(cfg["n_head_kv"]):
        for a in range(0, n, 512):
            qq = q[a:a + 512, g * rep:(g + 1) * rep].reshape(-1, D)
            s = (qq @ k[:, g].T.contiguous()) / math.sqrt(D)
            at = pos[a:a + 512].repeat_interleave(rep)
            s = torch.where(pos[None] <= at[:, None], s, -math.inf)
            out[a:a + 512, g * rep:(g + 1) * rep] = (torch.softmax(s, -1) @ v[:, g].contiguous()).reshape(-1, rep, D)
    return out


def _delta(h, W, vec, cfg):
    """The gated delta net over normalised rows h [n, E], state empty."""
    n, NK, NV, D, T = h.shape[0], cfg["dn_k_heads"], cfg["dn_v_heads"], cfg["dn_state"], cfg["dn_conv"]
    eps = cfg["rms_eps"]
    x = h @ W("ssm_qkv").T
    z = (h @ W("ssm_gate").T).reshape(n, NV, D)
    taps = vec["ssm_conv"].reshape(-1, T)
    pad = torch.cat((torch.zeros(T - 1, x.shape[1], device=DEV, dtype=torch.float64), x))
    c = _silu(sum(pad[i:i + n] * taps[:, i] for i in range(T)))
    q, k, v = c[:, :NK * D].reshape(n, NK, D), c[:, NK * D:2 * NK * D].reshape(n, NK, D), c[:, 2 * NK * D:].reshape(
        n, NV, D)
    q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + eps)
    k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + eps)
    of = torch.arange(NV, device=DEV) % NK  # the key head a value head reads
    q, k = q[:, of], k[:, of]
    alpha = h @ vec["ssm_alpha"].reshape(NV, -1).T
    beta = torch.sigmoid(h @ vec["ssm_beta"].reshape(NV, -1).T)
    decay = torch.exp(vec["ssm_a"] * torch.log1p(torch.exp(alpha + vec["ssm_dt"])))
    S = torch.zeros(NV, D, D, device=DEV, dtype=torch.float64)
    y = torch.empty(n, NV, D, device=DEV, dtype=torch.float64)
    for t in range(n):
        S = S * decay[t, :, None, None]
        S = S + (beta[t, :, None] * (v[t] - (S * k[t, :, None]).sum(-1)))[:, :, None] * k[t, :, None]
        y[t] = (S * q[t, :, None]).sum(-1) / math.sqrt(D)
    y = _rms(y, vec["ssm_norm"], eps) * _silu(z)
    return y.reshape(n, -1) @ W("ssm_out").T


def _exact_model(case, seed):
    cfg, mix = _cfg(case), case["mix"]
    toks = torch.from_numpy(_tokens(case, seed).astype(np.int64)).to(DEV)
    n, HD = len(toks), cfg["head_dim"]
    E, eps = cfg["n_embd"], cfg["rms_eps"]
    ends = _ends(cfg, mix)
    t, rms = ends["token_embd"]
    x = _mat(_gen(seed, 3, 0), t, cfg["vocab"], E, rms)[toks]
    for l in range(cfg["n_layer"]):
        mats = _matrices(cfg, mix, l)

        def W(name):
            mt, o, i = mats[name]
            return _mat(_gen(seed, 1, l, list(mats).index(name)), mt, o, i, 1.0 / math.sqrt(i))

        vec = {a: b.double() for a, b in _vectors(cfg, seed, l).items()}
        h = _rms(x, vec["attn_norm"], eps)
        if "ssm_qkv" in mats:
            x = x + _delta(h, W, vec, cfg)
        elif case["kind"] == "hybrid":
            qg = (h @ W("attn_q").T).reshape(n, -1, 2, HD)
            q = _rope(_rms(qg[:, :, 0], vec["q_norm"], eps), cfg)
            k = _rope(_rms((h @ W("attn_k").T).reshape(n, -1, HD), vec["k_norm"], eps), cfg)
            v = (h @ W("attn_v").T).reshape(n, -1, HD)
            att = _attend(q, k, v, cfg) * torch.sigmoid(qg[:, :, 1])
            x = x + att.reshape(n, -1) @ W("attn_output").T
        else:
            q = _rope((h @ W("attn_q").T + vec["bq"]).reshape(n, -1, HD), cfg)
            k = _rope((h @ W("attn_k").T + vec["bk"]).reshape(n, -1, HD), cfg)
            v = (h @ W("attn_v").T + vec["bv"]).reshape(n, -1, HD)
            x = x + _attend(q, k, v, cfg).reshape(n, -1) @ W("attn_output").T
        h = _rms(x, vec["post_norm" if case["kind"] == "hybrid" else "ffn_norm"], eps)
        x = x + (_silu(h @ W("ffn_gate").T) * (h @ W("ffn_up").T)) @ W("ffn_down").T
    last = case["pos"] + case["prompt"]
    want = ([last - 1] if case["prompt"] else []) + list(range(last, n))
    t, rms = ends["output"]
    h = _rms(x[want], _uniform(_gen(seed, 4), E, 0.9, 1.1).double(), eps)
    y = h @ _mat(_gen(seed, 3, 1), t, cfg["vocab"], E, rms).T
    return [y[i] for i in range(len(want))]
