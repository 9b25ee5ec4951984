"""The work that programs have this library do, as cases to be timed.

Seven kinds of call, over the sizes, element types and options they are used
with: the fused predictor + sparse FFN step, the sparse FFN over a given list,
the sliding-window decode, the dense FFN, the SwiGLU FFN, the MoE FFN and the
decode of a whole Falcon-architecture model.  `host` cases go through the
synchronous host-buffer calls (what the cgo binding uses), the others through
the device-pointer calls.  Weights are N(0, 0.02) rows quantized to the GGUF
type, inputs N(0, 1), predictors N(0, 0.05) in F32.
"""
import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "llama.go_amd"))
import llg  # noqa: E402

F32, F16, Q4_0, Q8_0 = 0, 1, 2, 8
RELU, GELU, SILU = 0, 1, 2
ROW_BITS = {F32: 32.0, F16: 16.0, Q4_0: 4.5, Q8_0: 8.5}  # bits per element
WINDOW_K = 5
ALL_ACTIVE = -3.0e38  # a threshold below every logit


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest calls: one layer of a small model, a Go program's host buffers
        dict(name="step_small_host", kind="step", host=True, type=Q4_0, h=512, ff=2048, rank=32,
             active=102, act=RELU),
        # the main decode step: a Falcon-7B layer, 5% of its neurons active
        dict(name="step_q4_0", kind="step", host=False, type=Q4_0, h=4544, ff=18176, rank=128,
             active=909, act=RELU),
        # the same step over 8-bit weights of another width and a denser active set
        dict(name="step_q8_0", kind="step", host=False, type=Q8_0, h=4096, ff=14336, rank=256,
             active=1433, act=RELU),
        # a program with its own selection: a given list over unquantized rows, ragged sizes
        dict(name="list_f16", kind="list", host=False, type=F16, h=2080, ff=7001, active=613,
             act=GELU),
        # decode with the sliding window: 16 tokens, 70% of each active set kept
        dict(name="window_q4_0", kind="window", type=Q4_0, h=4544, ff=18176, active=909, tokens=16,
             act=RELU),
        # layers without a predictor: the dense FFN of the Falcon-7B layer
        dict(name="dense_q4_0", kind="dense", type=Q4_0, h=4544, ff=18176, act=RELU),
        # the dense FFN of SiLU models at a LLaMA-7B layer
        dict(name="swiglu_q8_0", kind="swiglu", type=Q8_0, h=4096, ff=11008),
        # MoE decode: one token through a Mixtral layer
        dict(name="moe_one_q4_0", kind="moe", type=Q4_0, h=4096, eff=14336, n_exp=8, k=2, tokens=1),
        # a short prompt, or a few sequences decoded together
        dict(name="moe_few_q4_0", kind="moe", type=Q4_0, h=4096, eff=14336, n_exp=8, k=2, tokens=7),
        # a prompt over 8-bit experts
        dict(name="moe_prompt_q8_0", kind="moe", type=Q8_0, h=4096, eff=14336, n_exp=8, k=2,
             tokens=100),
        # a long prompt (the largest call)
        dict(name="moe_prompt_q4_0", kind="moe", type=Q4_0, h=4096, eff=14336, n_exp=8, k=2,
             tokens=512),
        # a token of the whole 32-layer Falcon-architecture model behind a 200-token prompt
        dict(name="falcon_token", kind="falcon", type=Q4_0, layers=32, h=4544, heads=71, kv=1,
             head_dim=64, ff=18176, rank=128, active=909, vocab=65024, prompt=200),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi // step, max(-(-lo // step), round(v / step)))) * step


def draw(rng):
    kind = rng.choice(["step", "step", "list", "window", "dense", "swiglu", "moe", "moe", "moe",
                       "falcon"])
    t = rng.choice([Q4_0, Q4_0, Q8_0, F16])
    if kind in ("step", "list", "window"):
        h = _log(rng, 512, 6144, 32)
        ff = _log(rng, 2 * h, 4 * h)
        c = dict(kind=kind, type=t, h=h, ff=ff, active=max(1, int(ff * rng.uniform(0.02, 0.15))),
                 act=rng.choice([RELU, RELU, GELU, SILU]))
        if kind == "window":
            return dict(c, tokens=rng.randint(4, 24))
        c["host"] = rng.random() < 0.3
        return dict(c, rank=_log(rng, 16, 256)) if kind == "step" else c
    if kind in ("dense", "swiglu"):
        h = _log(rng, 512, 8192, 32)
        c = dict(kind=kind, type=t, h=h, ff=_log(rng, 2 * h, min(4 * h, 28672), 32))
        return dict(c, act=rng.choice([RELU, GELU])) if kind == "dense" else c
    if kind == "moe":
        n_exp, k = rng.choice([(4, 1), (8, 2), (8, 2), (16, 4), (64, 8)])
        wide = rng.random() < 0.75  # the widths of real models are multiples of 256 and 128
        h = _log(rng, 512, 4096, 256 if wide else 32)
        eff = _log(rng, 512, max(1024, 14336 * 8 // n_exp), 128 if wide else 32)
        return dict(kind=kind, type=t, h=h, eff=eff, n_exp=n_exp, k=k,
                    tokens=_log(rng, 1, min(512, 1024 // k)))
    hd = rng.choice([64, 128])
    heads, kv = rng.choice([(16, 1), (24, 8), (32, 4), (71, 1)]) if hd == 64 else (
        rng.choice([(8, 2), (16, 4), (24, 1)]))
    h = heads * hd
    return dict(kind=kind, type=rng.choice([Q4_0, Q8_0]), layers=rng.randint(1, 6), h=h,
                heads=heads, kv=kv, head_dim=hd, ff=4 * h, rank=rng.choice([32, 64, 128]),
                active=int(4 * h * rng.uniform(0.03, 0.08)), vocab=_log(rng, 1000, 32000),
                prompt=_log(rng, 2, 500))


# ------------------------------------------------------------------ the inputs
def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + part) % (1 << 62))
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda") * std


def _rows(g, rows, cols, t, std=0.02):
    """GGUF bytes [rows x ByteSize(cols)] of N(0, std) rows on the GPU."""
    parts = []
    for r0 in range(0, rows, max(1, (1 << 26) // cols)):
        w = _randn(g, min(rows - r0, max(1, (1 << 26) // cols)), cols, std=std)
        n = w.shape[0]
        if t == F32:
            parts.append(w.view(torch.uint8))
        elif t == F16:
            parts.append(w.half().view(torch.uint8))
        else:
            b = w.view(n, cols // 32, 32)
            d = b.abs().amax(2, keepdim=True) / (8.0 if t == Q4_0 else 127.0)
            q = torch.round(b / d)
            if t == Q4_0:  # element 2i in the low nibble of byte i, 2i + 1 in the high one
                q = (q.clamp_(-8, 7) + 8).to(torch.uint8)
                q = q[..., 0::2] | (q[..., 1::2] << 4)
            else:
                q = q.clamp_(-127, 127).to(torch.int8).view(torch.uint8)
            parts.append(torch.cat([d.half().view(torch.uint8), q], 2).view(n, -1))
    return torch.cat(parts) if len(parts) > 1 else parts[0]


def _f64(raw, t):
    """The values of GGUF rows in 64 bits."""
    if t == F32:
        return raw.view(torch.float32).double()
    if t == F16:
        return raw.view(torch.float16).double()
    b = raw.view(raw.shape[0], -1, 18 if t == Q4_0 else 34)
    d, q = b[..., :2].contiguous().view(torch.float16).double(), b[..., 2:]
    if t == Q4_0:
        q = torch.stack([q & 15, q >> 4], -1).view(*q.shape[:2], 32).double() - 8.0
    else:
        q = q.contiguous().view(torch.int8).double()
    return (q * d).view(raw.shape[0], -1)


def _act64(act, u):
    if act == SILU:
        return u * torch.sigmoid(u)
    if act == GELU:
        return 0.5 * u * (1 + torch.tanh(math.sqrt(2 / math.pi) * (u + 0.044715 * u ** 3)))
    return torch.relu(u)


def _gap(logits, n):
    """A threshold that about n of the logits exceed, in the widest gap near
    the n-th largest, so that no rounding moves a neuron across it."""
    s = torch.sort(logits, descending=True).values
    lo, hi = max(0, int(0.95 * n) - 2), min(s.numel() - 1, int(1.05 * n) + 2)
    i = lo + int(torch.argmax(s[lo:hi] - s[lo + 1:hi + 1]))
    return float(((s[i] + s[i + 1]) / 2).float())


def _sparse_inputs(c, seed):
    """up and down rows, x, and the predictor with its threshold or the lists."""
    g = _gen(seed, 1)
    d = dict(up=_rows(g, c["ff"], c["h"], c["type"]), down=_rows(g, c["ff"], c["h"], c["type"]))
    if c["kind"] == "step":
        d["x"] = _randn(g, c["h"])
        d["wup"] = _randn(g, c["rank"], c["h"], std=0.05)
        d["wout"] = _randn(g, c["ff"], c["rank"], std=0.05)
        # of some predictor inputs, the one whose active set is the clearest
        # cut: no rounding moves a neuron across its threshold
        a = _randn(g, c["h"], 16)
        logits = d["wout"].double() @ torch.relu(d["wup"].double() @ a.double())
        top = torch.topk(logits, c["active"] + 1, dim=0).values[-2:]
        i = int(torch.argmax((top[0] - top[1]) / logits.std(dim=0)))
        d["a"] = a[:, i].contiguous()
        d["thr"] = float(top[:, i].mean().float())
        d["sets"] = [torch.nonzero(logits[:, i] > d["thr"]).flatten()]
        return d
    n, T = c["active"], c.get("tokens", 1)
    d["x"] = _randn(g, T, c["h"])
    sets = [torch.randperm(c["ff"], generator=g, device="cuda")[:n]]
    for _ in range(T - 1):  # each token keeps 70% of the set before
        keep = sets[-1][torch.randperm(n, generator=g, device="cuda")[:int(0.7 * n)]]
        order = torch.randperm(c["ff"], generator=g, device="cuda")
        sets.append(torch.cat([keep, order[~torch.isin(order, sets[-1])][:n - keep.numel()]]))
    d["sets"] = [torch.sort(s).values for s in sets]
    return d


def _ffn_inputs(c, seed):
    g = _gen(seed, 2)
    d = dict(x=_randn(g, c["h"]), up=_rows(g, c["ff"], c["h"], c["type"]),
             down=_rows(g, c["h"], c["ff"], c["type"]))
    if c["kind"] == "swiglu":
        d["gate"] = _rows(g, c["ff"], c["h"], c["type"])
    return d


def _moe_inputs(c, seed):
    g = _gen(seed, 3)
    n = c["n_exp"]
    return dict(x=_randn(g, c["tokens"], c["h"]), router=_randn(g, n, c["h"], std=0.02),
                gate=_rows(g, n * c["eff"], c["h"], c["type"]),
                up=_rows(g, n * c["eff"], c["h"], c["type"]),
                down=_rows(g, n * c["h"], c["eff"], c["type"]))


def _falcon_inputs(c, seed):
    """The model's weights as the library takes them, the tokens, and the
    64-bit pass over them: the prompt with every neuron, then one token whose
    layers' thresholds are placed for it.  Returns (weights, tokens,
    thresholds, logits of the last token)."""
    g = _gen(seed, 4)
    h, hd, nh, nkv, t = c["h"], c["head_dim"], c["heads"], c["kv"], c["type"]
    tok = torch.randint(0, c["vocab"], (c["prompt"] + 1,), generator=g, device="cuda")
    one, zero = np.ones(h, np.float32), np.zeros(h, np.float32)
    w = dict(embed=_rows(g, c["vocab"], h, t), lm_head=_rows(g, c["vocab"], h, t), out_w=one,
             out_b=zero)
    for key in ("norm_w", "norm_b", "wq", "wk", "wv", "wo", "pwup", "pwout", "up", "down_t"):
        w[key] = []
    n = tok.numel()
    pos = torch.arange(n, device="cuda", dtype=torch.float64)
    freq = pos[:, None] / 10000.0 ** (torch.arange(0, hd, 2, device="cuda").double() / hd)
    cos, sin = torch.cos(freq)[:, None], torch.sin(freq)[:, None]

    def norm(v):
        m = v - v.mean(1, keepdim=True)
        return m / torch.sqrt((m * m).mean(1, keepdim=True) + 1e-5)

    def rope(v):
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    x = _f64(w["embed"][tok], t)
    mask = torch.full((n, n), -math.inf, device="cuda", dtype=torch.float64).triu(1)
    thr = []
    for _ in range(c["layers"]):
        lay = dict(norm_w=one, norm_b=zero, wq=_rows(g, nh * hd, h, t), wk=_rows(g, nkv * hd, h, t),
                   wv=_rows(g, nkv * hd, h, t), wo=_rows(g, h, nh * hd, t),
                   pwup=_randn(g, c["rank"], h, std=0.05),
                   pwout=_randn(g, c["ff"], c["rank"], std=0.05),
                   up=_rows(g, c["ff"], h, t), down_t=_rows(g, c["ff"], h, t))
        for key, v in lay.items():
            w[key].append(v)
        y = norm(x)
        q = rope((y @ _f64(lay["wq"], t).T).view(n, nh, hd))
        k = rope((y @ _f64(lay["wk"], t).T).view(n, nkv, hd))
        v = (y @ _f64(lay["wv"], t).T).view(n, nkv, hd)
        att = torch.empty(n, nh, hd, device="cuda", dtype=torch.float64)
        for i in range(nh):
            j = i * nkv // nh
            s = torch.softmax(q[:, i] @ k[:, j].T.contiguous() / math.sqrt(hd) + mask, 1)
            att[:, i] = s @ v[:, j].contiguous()
        att = att.view(n, nh * hd) @ _f64(lay["wo"], t).T
        logits = lay["pwout"].double() @ torch.relu(lay["pwup"].double() @ att[-1])
        thr.append(_gap(logits, c["active"]))
        u = torch.relu(y @ _f64(lay["up"], t).T)
        u[-1] *= logits > thr[-1]
        x = x + att + u @ _f64(lay["down_t"], t)
    logits = _f64(w["lm_head"], t) @ norm(x[-1:])[0]
    return w, tok.int(), thr, logits


# ------------------------------------------------------------------ the calls
_device = []


def _dev():
    """The program's one device handle."""
    if not _device:
        _device.append(llg.Device())
    return _device[0]


class State:
    """What a program holds between calls; its handles go with it."""

    def __init__(self, case):
        self.case, self.dev, self.held = case, _dev(), []

    def keep(self, handle):
        self.held.append(handle)
        return handle

    def matrix(self, raw, t, rows, cols):
        return self.keep(self.dev.upload_matrix(raw, t, rows, cols))

    def __del__(self):
        for handle in reversed(self.held):
            handle.release()


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _prepare_sparse(s, c, seed):
    d = _sparse_inputs(c, seed)
    h, ff = c["h"], c["ff"]
    torch.cuda.synchronize()  # the library's stream does not wait for torch's
    s.bundle = s.keep(s.dev.upload_bundle(d["up"], d["down"], c["type"], h, ff))
    if c["kind"] == "step":
        s.thr = d["thr"]
        if c["host"]:
            s.pred = llg.Predictor(s.dev, d["wup"].cpu().numpy(), d["wout"].cpu().numpy(), None,
                                   s.thr)
            s.held += [s.pred.w_up, s.pred.w_out]
            s.x, s.a = d["x"].cpu().numpy(), d["a"].cpu().numpy()
            return
        s.wup = s.matrix(d["wup"], F32, c["rank"], h)
        s.wout = s.matrix(d["wout"], F32, ff, c["rank"])
        s.x, s.a = d["x"], d["a"]
        s.out = torch.zeros(h, device="cuda")
        s.n = torch.zeros(1, dtype=torch.int32, device="cuda")
        return
    s.sets = [v.int() for v in d["sets"]]
    s.x = d["x"]
    if c["kind"] == "list" and c["host"]:
        s.x, s.sets = s.x[0].cpu().numpy(), [s.sets[0].cpu().numpy()]
        return
    s.n = torch.tensor([c["active"]], dtype=torch.int32, device="cuda")
    s.out = torch.zeros_like(s.x)
    if c["kind"] == "window":
        s.win = llg.NeuronCache(s.dev, s.bundle, WINDOW_K)
        s.keep(s.win.win)


def _prepare_falcon(s, c, seed):
    w, s.tok, thr, _ = _falcon_inputs(c, seed)
    dims = dict(n_layers=c["layers"], hidden=c["h"], n_heads=c["heads"], n_kv=c["kv"],
                head_dim=c["head_dim"], ff=c["ff"], vocab=c["vocab"], max_seq=c["prompt"] + 1,
                rope_base=10000.0, eps=1e-5)
    torch.cuda.synchronize()
    s.model = s.keep(llg.FalconModel(s.dev, dims, w, [ALL_ACTIVE] * c["layers"], c["type"], RELU))
    s.next = torch.zeros(1, dtype=torch.int32, device="cuda")
    s.out = torch.zeros(c["vocab"], device="cuda")
    torch.cuda.synchronize()
    for i in range(c["prompt"]):
        s.model.step_device(s.tok.data_ptr() + 4 * i, i, s.next.data_ptr())
    s.model.set_thresholds(thr)


def prepare(case, seed):
    c, s = case, State(case)
    if c["kind"] in ("step", "list", "window"):
        _prepare_sparse(s, c, seed)
    elif c["kind"] == "falcon":
        _prepare_falcon(s, c, seed)
    elif c["kind"] == "moe":
        d = _moe_inputs(c, seed)
        torch.cuda.synchronize()
        n, h, eff, t = c["n_exp"], c["h"], c["eff"], c["type"]
        s.w = [s.matrix(d["router"], F32, n, h), s.matrix(d["gate"], t, n * eff, h),
               s.matrix(d["up"], t, n * eff, h), s.matrix(d["down"], t, n * h, eff)]
        s.x, s.out = d["x"], torch.zeros_like(d["x"])
        s.ids = torch.zeros((c["tokens"], c["k"]), dtype=torch.int32, device="cuda")
        s.wts = torch.zeros((c["tokens"], c["k"]), device="cuda")
    else:
        d = _ffn_inputs(c, seed)
        torch.cuda.synchronize()
        h, ff, t = c["h"], c["ff"], c["type"]
        s.w = [s.matrix(d[key], t, ff, h) for key in ("gate", "up") if key in d]
        s.w.append(s.matrix(d["down"], t, h, ff))
        s.x, s.out = d["x"], torch.zeros(h, device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    c, dev, lib = s.case, s.dev, s.dev.lib
    if c["kind"] == "step":
        if c["host"]:
            return llg.ffn_predict_sparse(dev, s.pred, s.bundle, s.a, s.x, c["act"])
        dev.check(lib.llg_hipd_ffn_predict_sparse(
            dev.h, s.wup.id, s.wout.id, 0, s.bundle.id, _p(s.a), _p(s.x), s.thr, c["act"],
            _p(s.out), None, _p(s.n)), "step")
        return s.out, s.n
    if c["kind"] == "list":
        if c["host"]:
            return llg.ffn_sparse_load(dev, s.bundle, s.x, s.sets[0], c["act"])
        dev.check(lib.llg_hipd_ffn_sparse(dev.h, s.bundle.id, _p(s.x), _p(s.sets[0]), _p(s.n),
                                          c["act"], _p(s.out)), "list")
        return s.out
    if c["kind"] == "window":
        for i, active in enumerate(s.sets):
            s.win.step_device(s.x[i].data_ptr(), active.data_ptr(), s.n.data_ptr(),
                              s.out[i].data_ptr(), c["act"])
        return s.out
    if c["kind"] == "dense":
        dev.check(lib.llg_hipd_ffn_dense(dev.h, s.w[0].id, s.w[1].id, _p(s.x), c["act"],
                                         _p(s.out)), "dense")
        return s.out
    if c["kind"] == "swiglu":
        dev.check(lib.llg_hipd_ffn_swiglu(dev.h, s.w[0].id, s.w[1].id, s.w[2].id, _p(s.x),
                                          _p(s.out)), "swiglu")
        return s.out
    if c["kind"] == "moe":
        dev.check(lib.llg_hipd_moe_ffn(
            dev.h, s.w[0].id, s.w[1].id, s.w[2].id, s.w[3].id, c["n_exp"], c["k"], _p(s.x),
            c["tokens"], _p(s.out), _p(s.ids), _p(s.wts)), "moe")
        return s.out, s.ids, s.wts
    s.model.step_device(s.tok.data_ptr() + 4 * c["prompt"], c["prompt"], s.next.data_ptr(),
                        s.out.data_ptr())
    return s.out, s.next


# ------------------------------------------------- what each case is held to
def exact(case, seed):
    c = case
    t = c["type"]
    if c["kind"] in ("step", "list", "window"):
        d = _sparse_inputs(c, seed)
        x = d["x"].double().view(-1, c["h"])
        outs = []
        for i, rows in enumerate(d["sets"]):
            u = _act64(c["act"], _f64(d["up"][rows], t) @ x[i])
            outs.append(u @ _f64(d["down"][rows], t))
        out = torch.stack(outs)
        if c["kind"] == "step":
            return out[0], None
        return out[0] if c.get("host") else out
    if c["kind"] in ("dense", "swiglu"):
        d = _ffn_inputs(c, seed)
        x = d["x"].double()
        u = _f64(d["up"], t) @ x
        u = _act64(SILU, _f64(d["gate"], t) @ x) * u if "gate" in d else _act64(c["act"], u)
        return _f64(d["down"], t) @ u
    if c["kind"] == "moe":
        d = _moe_inputs(c, seed)
        x, h, eff = d["x"].double(), c["h"], c["eff"]
        p = torch.softmax(x @ d["router"].double().T, 1)
        w, ids = torch.topk(p, c["k"], 1)
        w = w / w.sum(1, keepdim=True)
        out = torch.zeros_like(x)
        for e in range(c["n_exp"]):
            tok, slot = torch.nonzero(ids == e, as_tuple=True)
            if tok.numel():
                up = x[tok] @ _f64(d["up"][e * eff:(e + 1) * eff], t).T
                u = _act64(SILU, x[tok] @ _f64(d["gate"][e * eff:(e + 1) * eff], t).T) * up
                y = u @ _f64(d["down"][e * h:(e + 1) * h], t).T
                out.index_add_(0, tok, y * w[tok, slot][:, None])
        return out, None, w
    return _falcon_inputs(c, seed)[3], None


def tolerance(case):
    if case["kind"] == "falcon":  # fp32 through all layers
        return {"rel": 5e-5}
    if case["kind"] == "moe" and case["type"] == Q4_0 and case["tokens"] >= 16:
        return {"rel": 2e-3}  # the documented f16 operands of batched Q4_0 prompts
    # fp32 sums; a Q4_0 dot takes its offset of 8 out of the block's sum at the end
    return {"rel": 2.4e-5 if case["type"] == Q4_0 else 4e-6}


def work(case):
    c = case

    def rows(n, cols):
        return n * cols * ROW_BITS[c["type"]] / 8

    if c["kind"] in ("step", "list", "window"):
        T, n, h = c.get("tokens", 1), c["active"], c["h"]
        # a window token reads its set's rows, and writes the 30% that are new to the window
        b = T * (rows(2 * n, h) + 8 * h + 4 * n)
        if c["kind"] == "window":
            b += rows(2 * int(0.3 * n), h) * T
        f = T * 4 * n * h
        if c["kind"] == "step":
            b += 4 * c["rank"] * (h + c["ff"]) + 4 * h
            f += 2 * c["rank"] * (h + c["ff"])
        return {"bytes": b, "flops": f}
    if c["kind"] in ("dense", "swiglu"):
        m = 2 if c["kind"] == "dense" else 3
        return {"bytes": rows(m * c["ff"], c["h"]) + 8 * c["h"], "flops": 2 * m * c["ff"] * c["h"]}
    if c["kind"] == "moe":
        hit = c["n_exp"] * (1 - (1 - c["k"] / c["n_exp"]) ** c["tokens"])  # experts of the batch
        return {"bytes": rows(3 * hit * c["eff"], c["h"]) + 4 * c["h"] * (2 * c["tokens"] + c["n_exp"]),
                "flops": 2 * c["tokens"] * c["h"] * (3 * c["k"] * c["eff"] + c["n_exp"])}
    q, kv, h = c["heads"] * c["head_dim"], c["kv"] * c["head_dim"], c["h"]
    elems = q + 2 * kv + q + 2 * c["active"]  # rows of h elements a layer reads
    pred = c["rank"] * (h + c["ff"])
    cache = 2 * kv * (c["prompt"] + 1)
    return {"bytes": c["layers"] * (rows(elems, h) + 4 * pred + 4 * cache) + rows(c["vocab"] + 1, h)
            + 4 * c["vocab"],
            "flops": 2 * (c["layers"] * (elems * h + pred + 2 * q * (c["prompt"] + 1))
                          + c["vocab"] * h)}
