"""Workloads of the library, as a user's program calls them.

Six kinds of work:

* ``layer``    the seven projections of one transformer layer for one token, each a
               ``ptmi_matvec_dev`` call on device pointers (what a host decode loop does);
* ``matvec``   one ``ptmi_matvec_dev``;
* ``linear``   one linear layer over T positions through ``ptmi_gemm_dev``: the forward
               Y = X W^T, the input gradient dX = dY W, and dW += dY^T X;
* ``train``    a short training run (``ptmi_model_train_step``, a few SGD steps), then the
               updated weights read back into the host blob, as a checkpoint does;
* ``generate`` one ``ptmi_model_generate``: a prompt and the tokens after it, then the logits;
* ``steps``    single ``ptmi_model_forward_step`` calls, the logits read after each (sampling
               on the host).

Everything is fp32, the library's only data type.  torch supplies device memory; it is
imported before the package so that both use one HIP runtime.
"""
import ctypes
import math

import numpy as np
import torch

import pitorch_amd as pa

VOCAB = 32000
LARGEST_FLOPS = 6.0 * 110e6 * 1024 * 8         # a drawn training run costs at most about this


def listed():
    return [
        # One 15M layer's projections called one by one: the smallest calls, launch-bound.
        dict(name="layer_288", kind="layer", dim=288, hidden=768),
        # The 110M classifier for one token: the largest matvec, a pure weight stream.
        dict(name="matvec_classifier", kind="matvec", out=32000, inp=768),
        # The transposed classifier, d_x = W_cls^T d_logits of a per-position backward: few, very long rows.
        dict(name="matvec_long_rows", kind="matvec", out=768, inp=32000),
        # Odd row length: no row but the first starts on a 16-byte boundary.
        dict(name="matvec_ragged", kind="matvec", out=5003, inp=1027),
        # A 15M feed-forward projection over a short sequence: small GEMMs.
        dict(name="linear_small", kind="linear", T=64, out=768, inp=288),
        # A 110M feed-forward projection over the full context: an ordinary training GEMM.
        dict(name="linear_110m", kind="linear", T=1024, out=2048, inp=768),
        # Sizes that divide by nothing.
        dict(name="linear_ragged", kind="linear", T=501, out=1003, inp=517),
        # The 110M classifier over the full context: the largest GEMMs.
        dict(name="linear_classifier", kind="linear", T=1024, out=32000, inp=768),
        # The 15M training run at its configured length.
        dict(name="train_15m", kind="train", dim=288, hidden=768, layers=6, heads=6, vocab=VOCAB, seq=256, T=256, steps=64),
        # The 110M training run over its full context: the largest work.
        dict(name="train_110m", kind="train", dim=768, hidden=2048, layers=12, heads=12, vocab=VOCAB, seq=1024, T=1024, steps=8),
        # 110M: a long prompt (a document to continue) and a short answer.
        dict(name="prompt_110m", kind="generate", dim=768, hidden=2048, layers=12, heads=12, vocab=VOCAB, seq=1024, prompt=700, total=732),
        # 110M: the short prompt of the decode benchmark, then free decoding.
        dict(name="decode_110m", kind="generate", dim=768, hidden=2048, layers=12, heads=12, vocab=VOCAB, seq=1024, prompt=8, total=136),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size over the logarithm of the range; most divide by 4 or more, as layer widths do, some by nothing."""
    n = _log(rng, lo, hi)
    step = rng.choice((1, 4, 16, 32))
    return max(lo, n // step * step)


def _model(rng):
    """A model shape: (head_dim, heads) of small to 110M-sized models."""
    hd = rng.choice((32, 48, 48, 64, 64, 36))
    heads = rng.randint(4, 12)
    dim = hd * heads
    return dict(dim=dim, hidden=_log(rng, 2 * dim, 2 * dim + 512) // 4 * 4, layers=rng.randint(2, 12), heads=heads)


def draw(rng):
    kind = rng.choice(("layer", "matvec", "matvec", "linear", "linear", "linear", "train", "train", "generate", "generate", "steps"))
    if kind == "layer":
        dim = _size(rng, 64, 1024)
        return dict(kind=kind, dim=dim, hidden=min(2304, dim * rng.choice((2, 3)) - rng.choice((0, 0, 4, 32))))
    if kind == "matvec":
        out = _size(rng, 64, 32000)
        return dict(kind=kind, out=out, inp=_size(rng, 64, max(65, min(32000, 32000 * 768 // out))))
    if kind == "linear":
        T, out = _size(rng, 16, 1024), _size(rng, 64, 32000)
        return dict(kind=kind, T=T, out=out, inp=_size(rng, 64, 2048 if out < 8192 else 768))
    c = _model(rng)
    if kind == "train":
        vocab = rng.choice((512, 4096, VOCAB))
        T = _log(rng, 16, 1024)
        n = vocab * c["dim"] + c["layers"] * (4 * c["dim"] ** 2 + 3 * c["dim"] * c["hidden"])
        return dict(kind=kind, **c, vocab=vocab, seq=max(T, 64), T=T, steps=max(1, min(32, int(LARGEST_FLOPS / (6.0 * n * T)))))
    seq = rng.choice((256, 512, 1024))
    if kind == "generate":
        prompt = _log(rng, 1, seq - 8)
        return dict(kind=kind, **c, vocab=VOCAB, seq=seq, prompt=prompt, total=min(seq, prompt + _log(rng, 1, 128)))
    return dict(kind=kind, **c, vocab=VOCAB, seq=seq, count=rng.randint(4, 16))


# ── inputs ───────────────────────────────────────────────────────────────

def _rand(shape, seed, std, device="cuda", mean=0.0):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    t = torch.randn(shape, generator=g, device=device, dtype=torch.float32)
    return t.mul_(std).add_(mean)


def _sizes(case):
    """(name, shape) of the blob's tensors in file order (the embedding is also the classifier)."""
    D, H, L, V, S = case["dim"], case["hidden"], case["layers"], case["vocab"], case["seq"]
    hd = D // case["heads"]
    return [("emb", (V, D)), ("rms_att", (L, D)), ("wq", (L, D, D)), ("wk", (L, D, D)), ("wv", (L, D, D)),
            ("wo", (L, D, D)), ("rms_ffn", (L, D)), ("w1", (L, H, D)), ("w2", (L, D, H)), ("w3", (L, H, D)),
            ("rms_final", (D,)), ("freq", (S * hd,))]


def _weights(case, seed):
    """The model's tensors from the seed: N(0, 0.02) projections, norm weights around 1."""
    out = {}
    for i, (name, shape) in enumerate(_sizes(case)):
        if name.startswith("rms"):
            out[name] = _rand(shape, seed * 64 + i, 0.05, mean=1.0)
        elif name == "freq":                    # not read by the library (the angles are computed)
            out[name] = torch.zeros(shape, device="cuda")
        else:
            out[name] = _rand(shape, seed * 64 + i, 0.02)
    return out


def _blob(case, seed):
    """A llama2.c .bin blob in host memory (28-byte header, then the tensors) as uint8."""
    n = sum(math.prod(shape) for _, shape in _sizes(case))
    blob = np.empty(28 + 4 * n, np.uint8)
    blob[:28] = np.array([case["dim"], case["hidden"], case["layers"], case["heads"], case["heads"], case["vocab"],
                          case["seq"]], np.int32).view(np.uint8)
    flat = torch.from_numpy(blob[28:].view(np.float32))
    at = 0
    for t in _weights(case, seed).values():
        flat[at:at + t.numel()].copy_(t.reshape(-1))
        at += t.numel()
    return blob


def _tokens(case, seed, n):
    """Token ids, none of them 1 or 2 (begin and end of a sequence)."""
    return np.random.default_rng(seed).integers(3, case["vocab"], n).astype(np.int32)


def _layer_shapes(case):
    D, H = case["dim"], case["hidden"]
    return [(D, D)] * 4 + [(H, D), (H, D), (D, H)]


def prepare(case, seed):
    kind, L = case["kind"], pa.load_ptmi()
    s = dict(case=case, L=L)
    if kind in ("layer", "matvec"):
        shapes = _layer_shapes(case) if kind == "layer" else [(case["out"], case["inp"])]
        s["W"] = [_rand(sh, seed * 64 + i, 0.02) for i, sh in enumerate(shapes)]
        s["x"] = [_rand((sh[1],), seed * 64 + 32 + i, 1.0) for i, sh in enumerate(shapes)]
        s["y"] = [torch.empty(sh[0], device="cuda") for sh in shapes]
    elif kind == "linear":
        T, N, K = case["T"], case["out"], case["inp"]
        s["W"], s["X"] = _rand((N, K), seed * 8, 0.02), _rand((T, K), seed * 8 + 1, 1.0)
        s["dY"], s["dW"] = _rand((T, N), seed * 8 + 2, 1e-3), _rand((N, K), seed * 8 + 3, 1e-2)
        s["Y"], s["dX"] = torch.empty((T, N), device="cuda"), torch.empty((T, K), device="cuda")
    else:
        s["model"] = pa.Model(_blob(case, seed), max_T=case["T"] if kind == "train" else 0)
        if kind == "train":
            s["tokens"] = [_tokens(case, seed * 64 + i, case["T"]) for i in range(case["steps"])]
        else:
            s["tokens"] = _tokens(case, seed * 64, case["prompt"] if kind == "generate" else case["count"])
    torch.cuda.synchronize()
    return s


# ── one pass ─────────────────────────────────────────────────────────────

LR = 0.05


def run(s):
    case, L = s["case"], s["L"]
    kind = case["kind"]
    if kind in ("layer", "matvec"):
        for W, x, y in zip(s["W"], s["x"], s["y"]):
            pa._ffi.check(L.ptmi_matvec_dev(W.data_ptr(), W.shape[1], x.data_ptr(), y.data_ptr(), W.shape[0], W.shape[1], None))
        return s["y"]
    if kind == "linear":
        T, N, K = case["T"], case["out"], case["inp"]
        X, W, Y, dY, dX, dW = (s[k].data_ptr() for k in ("X", "W", "Y", "dY", "dX", "dW"))
        pa._ffi.check(L.ptmi_gemm_dev(2, X, K, W, K, Y, N, T, N, K, 0, None))
        pa._ffi.check(L.ptmi_gemm_dev(0, dY, N, W, K, dX, K, T, K, N, 0, None))
        pa._ffi.check(L.ptmi_gemm_dev(1, dY, N, X, K, dW, K, N, K, T, 1, None))
        return dict(Y=s["Y"], dX=s["dX"], dW=s["dW"])
    m = s["model"]
    if kind == "train":
        losses = [m.train_step(t, LR) for t in s["tokens"]]
        blob = m.blob                               # the host blob takes the updated weights in place
        pa._ffi.check(L.ptmi_model_read_weights(m.h, blob.ctypes.data_as(ctypes.c_void_p), blob.nbytes))
        return dict(losses=np.array(losses, np.float32), weights=blob[28:].view(np.float32))
    if kind == "generate":
        tokens = m.generate(s["tokens"], case["total"], stop_on_eos=False)
        return dict(tokens=tokens, logits=m.logits())
    m.reset_kv()
    picked, logits = [], []
    for t in s["tokens"]:
        picked.append(m.forward_step(int(t)))
        logits.append(m.logits())
    return dict(tokens=np.array(picked, np.int32), logits=logits)


# ── what a pass cannot do without, and how far results may lie apart ─────

def _params(case):
    D, H = case["dim"], case["hidden"]
    return case["layers"] * (4 * D * D + 3 * D * H), case["vocab"] * D


def work(case):
    kind = case["kind"]
    if kind in ("layer", "matvec"):
        shapes = _layer_shapes(case) if kind == "layer" else [(case["out"], case["inp"])]
        return dict(bytes=4.0 * sum(d * n + d + n for d, n in shapes), flops=2.0 * sum(d * n for d, n in shapes))
    if kind == "linear":
        T, N, K = case["T"], case["out"], case["inp"]
        # W, X, dY, dW read, Y, dX, dW written
        return dict(bytes=4.0 * (3 * N * K + 2 * T * K + 2 * T * N), flops=6.0 * T * N * K)
    body, emb = _params(case)
    D, L = case["dim"], case["layers"]
    if kind == "train":
        T = case["T"]
        # weights read and written, logits and the layer inputs written and read once
        per = dict(bytes=4.0 * (2 * (body + emb) + 2 * T * case["vocab"] + 2 * T * D * L),
                   flops=6.0 * (body + emb) * T + 6.0 * L * T * T * D)
        return dict(bytes=case["steps"] * per["bytes"] + 4.0 * (body + emb), flops=case["steps"] * per["flops"])
    # the prompt's keys and values in one pass over the weights, then one pass per further token
    n = case["total"] if kind == "generate" else case["count"]
    first = min(case["prompt"], n) if kind == "generate" else 1
    kv = sum(8.0 * L * D * (p + 1) for p in range(first - 1, n))
    return dict(bytes=4.0 * (body + emb) * (n - first + 1) + kv + 8.0 * L * D * n,
                flops=2.0 * body * n + 2.0 * emb * (n - first + 1) + 2.0 * L * D * n * n)


def tolerance(case):
    # About four times the distance to 64 bits measured for each kind: 4.1e-7 for a dot product of
    # 32000 terms, 1.3e-6 for the classifier's dX (sums over 32000), 2.1e-7 for the weights after
    # 64 steps, 7.5e-6 for the logits at position 732 (fp32 rotation angles of several hundred radians).
    kind = case["kind"]
    if kind in ("layer", "matvec"):
        return dict(rel=2e-6)
    if kind == "linear":
        return dict(rel=5e-6)
    if kind == "train":
        return dict(rel=1e-6)
    return dict(rel=3e-5, differ=0.005)


# ── the same results in 64 bits ──────────────────────────────────────────

def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * w


def _rope(x, pos):
    """Rotates the pairs of [T, heads, head_dim] at the positions `pos`."""
    hd = x.shape[-1]
    f = torch.exp(-9.210340372 * torch.arange(0, hd, 2, device=x.device, dtype=torch.float64) / hd)
    a = pos[:, None, None] * f
    c, s = torch.cos(a), torch.sin(a)
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack((u * c - v * s, u * s + v * c), -1).flatten(-2)


def _forward(case, w, tokens, cache=None):
    """Final hidden rows of the new `tokens`, after the `cache`'s positions (lists of keys and values by layer)."""
    D, hd = case["dim"], case["dim"] // case["heads"]
    n, past = len(tokens), 0 if cache is None or not cache["k"] else cache["k"][0].shape[0]
    pos = torch.arange(past, past + n, device="cuda", dtype=torch.float64)
    x = w["emb"][tokens]
    mask = torch.arange(past + n, device="cuda")[None, :] > pos[:, None]
    for i in range(case["layers"]):
        h = _norm(x, w["rms_att"][i])
        q, k, v = ((h @ w[t][i].t()).view(n, -1, hd) for t in ("wq", "wk", "wv"))
        q, k = _rope(q, pos), _rope(k, pos)
        if cache is not None:
            if past:
                k, v = torch.cat((cache["k"][i], k)), torch.cat((cache["v"][i], v))
                cache["k"][i], cache["v"][i] = k, v
            else:
                cache["k"].append(k)
                cache["v"].append(v)
        att = torch.matmul(q.transpose(0, 1).contiguous(), k.permute(1, 2, 0).contiguous()) / math.sqrt(hd)
        att = torch.softmax(att.masked_fill(mask, -math.inf), -1)
        o = torch.matmul(att, v.transpose(0, 1).contiguous()).transpose(0, 1).reshape(n, D)
        x = x + o @ w["wo"][i].t()
        h = _norm(x, w["rms_ffn"][i])
        x = x + (torch.nn.functional.silu(h @ w["w1"][i].t()) * (h @ w["w3"][i].t())) @ w["w2"][i].t()
    return _norm(x, w["rms_final"])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("layer", "matvec", "linear"):
        s = prepare(case, seed)
        if kind != "linear":
            return [W.double() @ x.double() for W, x in zip(s["W"], s["x"])]
        X, W, dY, dW = (s[k].double() for k in ("X", "W", "dY", "dW"))
        return dict(Y=X @ W.t(), dX=dY @ W, dW=dW + dY.t() @ X)
    w = {k: t.double() for k, t in _weights(case, seed).items()}
    if kind == "train":
        for t in w.values():
            t.requires_grad_(True)
        losses = []
        for i in range(case["steps"]):
            tok = torch.from_numpy(_tokens(case, seed * 64 + i, case["T"])).long().cuda()
            logits = _forward(case, w, tok)[:-1] @ w["emb"].t()
            loss = torch.nn.functional.cross_entropy(logits, tok[1:])
            named = [k for k in w if k != "freq"]
            grads = torch.autograd.grad(loss, [w[k] for k in named])
            with torch.no_grad():
                for k, g in zip(named, grads):
                    w[k] -= LR * g
            losses.append(loss.item())
            del logits, loss, grads
        return dict(losses=np.array(losses), weights=torch.cat([t.detach().reshape(-1) for t in w.values()]))
    with torch.no_grad():
        cache = dict(k=[], v=[])
        if kind == "steps":
            tok = torch.from_numpy(_tokens(case, seed * 64, case["count"])).long().cuda()
            logits = _forward(case, w, tok, cache) @ w["emb"].t()
            return dict(tokens=None, logits=list(logits))
        prompt = _tokens(case, seed * 64, case["prompt"])[:case["total"]]
        logits = _forward(case, w, torch.from_numpy(prompt).long().cuda(), cache)[-1:] @ w["emb"].t()
        for _ in range(case["total"] - len(prompt)):
            logits = _forward(case, w, logits.argmax(-1), cache) @ w["emb"].t()
        return dict(tokens=None, logits=logits[0])
