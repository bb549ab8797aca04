"""The work that a user of this library has it do, as timeable cases.

A program of such a user opens one context, loads its encoders once and then
sends batch after batch through them; that is why encoders are kept here per
geometry (their weights are drawn from a fixed seed) and only the inputs come
from the case's seed. Device buffers are torch tensors handed over by address.

Kinds of a case:
  embed    token ids and mask on the GPU -> pooled, L2-normalised rows
           ("wait": the synchronous call of a single request, else queued)
  service  token ids and mask in host memory -> pooled rows in host memory,
           cut into chunks over the service's lanes
  vit      pixels -> class logits
  whisper  mel spectrogram -> encoder hidden state
  gemm     one linear layer (bias, GELU, fp32 residual as asked)
  int8_ffn the FFN half of an int8 layer, op by op: quantise, FFN-up with
           GELU, quantise, FFN-down, residual LayerNorm with quantisation
  attention, norm   one attention layer, one residual LayerNorm
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "npu-embeddings-xdna1_amd")
_DEV = "cuda"

# Geometry of the repository's own configurations.
MODELS = {
    "minilm": dict(kind="bert", layers=6, hidden=384, heads=12, ffn=1536, cls=False, gated=0),
    "bge_base": dict(kind="bert", layers=12, hidden=768, heads=12, ffn=3072, cls=True, gated=0),
    "bge_large": dict(kind="bert", layers=24, hidden=1024, heads=16, ffn=4096, cls=True, gated=0),
    "nomic": dict(kind="bert", layers=12, hidden=768, heads=12, ffn=3072, cls=False, gated=1),
    "gte": dict(kind="bert", layers=12, hidden=768, heads=12, ffn=3072, cls=True, gated=2),
    "vit_base": dict(kind="vit", layers=12, hidden=768, heads=12, ffn=3072, gated=0),
    "whisper_enc": dict(kind="whisper", layers=32, hidden=1280, heads=20, ffn=5120, gated=0),
}
VOCAB, MAX_POS = 30522, 512
MELS, FRAMES = 128, 3000
IMAGE, PATCH, LABELS = 224, 16, 1000
# The share of a padded batch that is real text: lengths are uniform between
# a sixteenth of the batch's width and all of it.
LEN_LO = 1 / 16


def listed():
    return [
        # A single search query, answered at once: latency.
        dict(name="query_minilm", kind="embed", model="minilm", batch=1, seq=19, wait=True),
        # A question to a larger model with its passage, answered at once.
        dict(name="query_bge_base", kind="embed", model="bge_base", batch=3, seq=131, wait=True),
        # The ordinary indexing batch of the small model.
        dict(name="batch_minilm", kind="embed", model="minilm", batch=32, seq=128, wait=False),
        # The ordinary indexing batch of the base model: the benchmark's.
        dict(name="batch_bge_base", kind="embed", model="bge_base", batch=64, seq=512, wait=False),
        # Long passages through the large model, a batch that fills no tile.
        dict(name="batch_bge_large", kind="embed", model="bge_large", batch=7, seq=389,
             wait=False),
        # Rotary positions, gated FFN and mean pooling.
        dict(name="batch_nomic", kind="embed", model="nomic", batch=24, seq=300, wait=False),
        # An embedding server's request from host memory over three lanes.
        dict(name="service_minilm", kind="service", model="minilm", batch=32, seq=128, lanes=3,
             sequences=601),
        # Image classification.
        dict(name="vit_images", kind="vit", model="vit_base", batch=20),
        # Two half-minute windows of speech.
        dict(name="whisper_windows", kind="whisper", model="whisper_enc", batch=2),
        # The FFN half of an int8 layer over a batch's packed rows.
        dict(name="int8_ffn", kind="int8_ffn", rows=4099, hidden=768, ffn=3072),
        # One attention layer over a padded batch, op by op.
        dict(name="attention_padded", kind="attention", batch=17, seq=433, heads=12, head_dim=64),
        # One linear layer with an fp32 residual, as a pre-LN block has it.
        dict(name="linear_residual", kind="gemm", rows=3000, k=1280, n=1280, epi="none",
             c="f32", residual=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["embed", "embed", "embed", "embed", "service", "vit", "whisper", "gemm",
                       "gemm", "int8_ffn", "attention", "norm"])
    if kind == "embed":
        model = rng.choice(["minilm", "bge_base", "bge_large", "nomic", "gte"])
        batch = _log(rng, 1, 12 if model == "bge_large" else 48)
        seq = _log(rng, 6, 512)
        return dict(kind=kind, model=model, batch=batch, seq=seq,
                    wait=batch <= 4 or rng.random() < 0.2)
    if kind == "service":
        return dict(kind=kind, model="minilm", batch=rng.randint(8, 48), seq=_log(rng, 16, 256),
                    lanes=rng.randint(1, 3), sequences=_log(rng, 40, 800))
    if kind == "vit":
        return dict(kind=kind, model="vit_base", batch=_log(rng, 1, 40))
    if kind == "whisper":
        return dict(kind=kind, model="whisper_enc", batch=rng.randint(1, 2))
    width = 64 * rng.randint(6, 20)
    if kind == "gemm":
        c = rng.choice(["bf16", "f32"])
        residual = c == "f32" and rng.random() < 0.7
        wide = rng.choice([1, 3, 4])
        k, n = (width, width * wide) if rng.random() < 0.6 else (width * wide, width)
        epi = "none" if residual else rng.choice(["none", "gelu_poly", "gelu_erf"])
        return dict(kind=kind, rows=_log(rng, 1, 20000), k=k, n=n, epi=epi, c=c,
                    residual=residual)
    if kind == "int8_ffn":
        return dict(kind=kind, rows=_log(rng, 1, 18000), hidden=width, ffn=4 * width)
    if kind == "attention":
        hd = rng.choice([32, 64, 64])
        return dict(kind=kind, batch=_log(rng, 1, 40), seq=_log(rng, 6, 1500),
                    heads=rng.choice([12, 16, 20]), head_dim=hd)
    return dict(kind="norm", rows=_log(rng, 1, 20000), cols=width)


# ---- weights and inputs -----------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(int(seed))


def _randn(g, shape, std):
    return torch.randn(shape, generator=g, device=_DEV, dtype=torch.float32) * std


def _weights(model):
    """The model's tensors on the GPU: GEMM operands [K, N] in bf16, the rest
    fp32. 1/sqrt(head_dim) is folded into Q's columns and bias."""
    c = MODELS[model]
    g = _gen(20260926 + sorted(MODELS).index(model))
    L, d, f, H = c["layers"], c["hidden"], c["ffn"], c["heads"]
    fu = 2 * f if c["gated"] else f
    scale = 1.0 / math.sqrt(d // H)
    w = {}
    for key, k, n in (("qkv", d, 3 * d), ("ao", d, d), ("up", d, fu), ("down", f, d)):
        w["w_" + key] = torch.empty((L, k, n), device=_DEV, dtype=torch.bfloat16)
        b = _randn(g, (L, n), 0.02)
        for layer in range(L):
            t = _randn(g, (k, n), 0.02)
            if key == "qkv":
                t[:, :d] *= scale
            w["w_" + key][layer] = t.to(torch.bfloat16)
        if key == "qkv":
            b[:, :d] *= scale
        w["b_" + key] = b
    for ln in ("ln1", "ln2"):
        w[ln + "_g"] = 1.0 + _randn(g, (L, d), 0.1)
        w[ln + "_b"] = _randn(g, (L, d), 0.05)
    if c["kind"] == "bert":
        w["word"] = _randn(g, (VOCAB, d), 0.02)
        w["pos"] = _randn(g, (MAX_POS, d), 0.02)
        w["type"] = _randn(g, (2, d), 0.02)
        w["emb_ln_g"], w["emb_ln_b"] = 1.0 + _randn(g, (d,), 0.1), _randn(g, (d,), 0.05)
    else:
        w["fin_ln_g"], w["fin_ln_b"] = 1.0 + _randn(g, (d,), 0.1), _randn(g, (d,), 0.05)
    if c["kind"] == "vit":
        w["patch_w"] = _randn(g, (3 * PATCH * PATCH, d), 0.02).to(torch.bfloat16)
        w["patch_b"] = _randn(g, (d,), 0.02)
        w["cls_token"] = _randn(g, (d,), 0.02)
        w["pos"] = _randn(g, ((IMAGE // PATCH) ** 2 + 1, d), 0.02)
        w["head_w"] = _randn(g, (d, LABELS), 0.02).to(torch.bfloat16)
        w["head_b"] = _randn(g, (LABELS,), 0.02)
    if c["kind"] == "whisper":
        for i, cin in ((1, MELS), (2, d)):
            t = _randn(g, (d, cin, 3), 0.02)
            w["conv%d_w" % i] = t.to(torch.bfloat16).float()
            w["conv%d_b" % i] = _randn(g, (d,), 0.02)
        inc = math.log(10000.0) / (d // 2 - 1)
        t = torch.arange(FRAMES // 2, device=_DEV, dtype=torch.float64)[:, None] * torch.exp(
            -inc * torch.arange(d // 2, device=_DEV, dtype=torch.float64))[None, :]
        w["pos"] = torch.cat([t.sin(), t.cos()], 1).float()
    return w


def _inv_freq(model):
    half = MODELS[model]["hidden"] // MODELS[model]["heads"] // 2
    j = np.arange(half, dtype=np.float64)
    if model == "gte":
        return (160000.0 ** (-j / half) / 8.0 ** (1.0 / half)).astype(np.float32)
    return 1000.0 ** (-j / half)


def _text(case, seed, sequences):
    """Token ids, and the 1/0 mask of sequences of uneven length (one
    sequence alone fills its row)."""
    r = np.random.default_rng(int(seed))
    S = case["seq"]
    lens = r.integers(max(1, int(S * LEN_LO)), S + 1, size=sequences)
    lens[0] = S  # the widest sets the batch's width
    ids = r.integers(1000, VOCAB, size=(sequences, S), dtype=np.int32)
    ids[:, 0] = 101
    keep = np.arange(S)[None, :] < lens[:, None]
    return np.where(keep, ids, 0).astype(np.int32), keep.astype(np.float32), lens


_EPILOGUE = {"none": 0, "gelu_poly": 1, "gelu_erf": 2}


def _inputs(case, seed):
    """The tensors of an op-level or picture / speech case."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "vit":
        return dict(pixels=torch.rand((case["batch"], 3, IMAGE, IMAGE), generator=g,
                                      device=_DEV) * 2 - 1)
    if kind == "whisper":
        return dict(mel=_randn(g, (case["batch"], MELS, FRAMES), 1.0))
    if kind == "gemm":
        M, K, N = case["rows"], case["k"], case["n"]
        t = dict(a=_randn(g, (M, K), 1.0).to(torch.bfloat16),
                 w=_randn(g, (N, K), 0.02).to(torch.bfloat16), bias=_randn(g, (N,), 0.02))
        if case["residual"]:
            t["res"] = _randn(g, (M, N), 1.0)
        return t
    if kind == "int8_ffn":
        M, d, f = case["rows"], case["hidden"], case["ffn"]
        t = dict(x=_randn(g, (M, d), 1.0))
        for key, k, n in (("up", d, f), ("down", f, d)):
            w = _randn(g, (n, k), 0.02)
            s = w.abs().amax(1) / 127.0
            t["w_" + key] = (w / s[:, None]).round().clamp(-127, 127).to(torch.int8)
            t["s_" + key] = s
            t["b_" + key] = _randn(g, (n,), 0.02)
            t["ias_" + key] = 1.0 / (0.5 + 1.5 * torch.rand((k,), generator=g, device=_DEV))
        t["ias_next"] = 1.0 / (0.5 + 1.5 * torch.rand((d,), generator=g, device=_DEV))
        t["g"], t["b"] = 1.0 + _randn(g, (d,), 0.1), _randn(g, (d,), 0.05)
        return t
    if kind == "attention":
        B, S, d = case["batch"], case["seq"], case["heads"] * case["head_dim"]
        r = np.random.default_rng(int(seed))
        lens = r.integers(max(1, int(S * LEN_LO)), S + 1, size=B)
        lens[0] = S
        keep = np.arange(S)[None, :] < lens[:, None]
        qkv = _randn(g, (B * S, 3 * d), 1.0)
        qkv[:, :d] /= math.sqrt(case["head_dim"])
        return dict(qkv=qkv.to(torch.bfloat16),
                    mask=torch.from_numpy(np.where(keep, 0.0, -1e30).astype(np.float32)).to(_DEV),
                    kv_len=torch.from_numpy(lens.astype(np.int32)).to(_DEV))
    M, d = case["rows"], case["cols"]
    return dict(x=_randn(g, (M, d), 1.0), y=_randn(g, (M, d), 1.0).to(torch.bfloat16),
                g=1.0 + _randn(g, (d,), 0.1), b=_randn(g, (d,), 0.05))


# ---- what a user's program keeps ----------------------------------------------------

class _Buf:
    """A torch tensor as the binding's device buffer: address, shape, dtype."""
    _NP = {torch.float32: np.float32, torch.bfloat16: np.uint16, torch.int32: np.int32,
           torch.int8: np.int8}

    def __init__(self, t):
        self.t = t
        self.p = ctypes.c_void_p(t.data_ptr())
        self.shape = tuple(t.shape)
        self.dtype = np.dtype(self._NP[t.dtype])


_kept = {}


def _mxenc():
    if _PKG not in sys.path:
        sys.path.insert(0, _PKG)
    import mxenc
    return mxenc


def _ctx():
    if "ctx" not in _kept:
        torch.zeros(1, device=_DEV)
        _kept["ctx"] = _mxenc().Context(0)
    return _kept["ctx"]


def _host(t):
    t = t.cpu().contiguous()
    return t.view(torch.int16).numpy().view(np.uint16) if t.dtype == torch.bfloat16 else t.numpy()


def _encoder(model):
    """The model's encoder, loaded once."""
    if model not in _kept:
        c = MODELS[model]
        m = {k: _host(v) for k, v in _weights(model).items()}
        m.update(kind=c["kind"], layers=c["layers"], hidden=c["hidden"], heads=c["heads"],
                 head_dim=c["hidden"] // c["heads"], ffn=c["ffn"], gated=c["gated"],
                 vocab=VOCAB, max_pos=MAX_POS, image=IMAGE, patch=PATCH, labels=LABELS,
                 mels=MELS, frames=FRAMES, eps=1e-12 if c["kind"] == "vit" else 1e-5,
                 cls_pool=c.get("cls", False), rope=bool(c["gated"]),
                 rope_theta=1000.0 if model == "nomic" else 0.0)
        if model == "gte":
            m["rope_inv_freq"] = _inv_freq(model)
        _kept[model] = _mxenc().Encoder(_ctx(), m)
    return _kept[model]


def _service(case):
    key = ("service", case["lanes"], case["batch"], case["seq"])
    if key not in _kept:
        for old in [k for k in _kept if isinstance(k, tuple)]:
            _kept.pop(old).close()
        _kept[key] = _mxenc().EmbedService(_encoder(case["model"]), case["lanes"], case["batch"],
                                           case["seq"])
    return _kept[key]


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, ctx=_ctx())
    if kind == "service":
        s["service"] = _service(case)
        s["ids"], s["mask"], _ = _text(case, seed, case["sequences"])
        return s
    if kind == "embed":
        ids, mask, _ = _text(case, seed, case["batch"])
        s["enc"] = _encoder(case["model"])
        s["ids"] = _Buf(torch.from_numpy(ids).to(_DEV))
        s["mask"] = _Buf(torch.from_numpy(mask).to(_DEV))
        s["out"] = _Buf(torch.empty((case["batch"], MODELS[case["model"]]["hidden"]),
                                    device=_DEV))
        return s
    t = _inputs(case, seed)
    if kind == "vit":
        s["enc"] = _encoder(case["model"])
        t["out"] = torch.empty((case["batch"], LABELS), device=_DEV)
    elif kind == "whisper":
        s["enc"] = _encoder(case["model"])
        t["out"] = torch.empty((case["batch"], FRAMES // 2, MODELS[case["model"]]["hidden"]),
                               device=_DEV)
    elif kind == "gemm":
        t["out"] = torch.empty((case["rows"], case["n"]), device=_DEV,
                               dtype=torch.float32 if case["c"] == "f32" else torch.bfloat16)
    elif kind == "int8_ffn":
        M, d, f = case["rows"], case["hidden"], case["ffn"]
        for key, shape, dt in (("q1", (M, d), torch.int8), ("a1", (M,), torch.float32),
                               ("h", (M, f), torch.float32), ("q2", (M, f), torch.int8),
                               ("a2", (M,), torch.float32), ("y", (M, d), torch.float32),
                               ("out", (M, d), torch.float32), ("q3", (M, d), torch.int8),
                               ("a3", (M,), torch.float32)):
            t[key] = torch.empty(shape, device=_DEV, dtype=dt)
    elif kind == "attention":
        t["out"] = torch.empty((case["batch"] * case["seq"], case["heads"] * case["head_dim"]),
                               device=_DEV, dtype=torch.bfloat16)
        t["out"].zero_()
    else:
        t["out"] = torch.empty((case["rows"], case["cols"]), device=_DEV)
        t["out_bf16"] = torch.empty((case["rows"], case["cols"]), device=_DEV,
                                    dtype=torch.bfloat16)
    s.update({k: _Buf(v) for k, v in t.items()})
    return s


def run(s):
    c, ctx, mx = s["case"], s["ctx"], sys.modules["mxenc"]
    kind = c["kind"]
    if kind == "service":
        return s["service"].embed(s["ids"], s["mask"])
    if kind == "embed":
        call = s["enc"].embed if c["wait"] else s["enc"].embed_async
        call(s["ids"], s["mask"], c["batch"], c["seq"], s["out"])
        return s["out"].t
    if kind == "vit":
        s["enc"].vit(s["pixels"], c["batch"], s["out"])
        return s["out"].t
    if kind == "whisper":
        s["enc"].whisper(s["mel"], c["batch"], s["out"])
        return s["out"].t
    if kind == "gemm":
        mx.gemm_wt(ctx, s["a"], c["rows"], c["k"], c["k"], s["w"], c["n"], s["bias"],
                   _EPILOGUE[c["epi"]], s.get("res"), s["out"], c["n"])
        return s["out"].t
    if kind == "int8_ffn":
        M, d, f = c["rows"], c["hidden"], c["ffn"]
        mx.quantise_a_int8(ctx, s["x"], M, d, s["ias_up"], s["q1"], s["a1"])
        mx.gemm_i8_wt(ctx, s["q1"], s["a1"], M, d, d, s["w_up"], s["s_up"], f, s["b_up"],
                      mx.MX_EPI_GELU_POLY, None, s["h"], f)
        mx.quantise_a_int8(ctx, s["h"], M, f, s["ias_down"], s["q2"], s["a2"])
        mx.gemm_i8_wt(ctx, s["q2"], s["a2"], M, f, f, s["w_down"], s["s_down"], d, s["b_down"],
                      0, None, s["y"], d)
        mx.layernorm_i8(ctx, s["x"], s["y"], s["g"], s["b"], 1e-12, M, d, s["out"],
                        s["ias_next"], s["q3"], s["a3"])
        return s["out"].t, s["q3"].t, s["a3"].t
    if kind == "attention":
        d = c["heads"] * c["head_dim"]
        mx.attention(ctx, s["qkv"], 3 * d, c["batch"], c["seq"], c["heads"], c["head_dim"], 1.0,
                     s["mask"], s["kv_len"], s["out"], d)
        return s["out"].t
    mx.layernorm(ctx, s["x"], s["y"], s["g"], s["b"], 1e-12, c["rows"], c["cols"], s["out"],
                 s["out_bf16"])
    return s["out"].t, s["out_bf16"].t


# ---- what a pass cannot do without ----------------------------------------------------

def _mean_lens(S, n):
    """Expected sum and sum of squares of n drawn lengths."""
    lo = max(1, int(S * LEN_LO))
    v = np.arange(lo, S + 1, dtype=np.float64)
    return S + (n - 1) * v.mean(), float(S) ** 2 + (n - 1) * (v ** 2).mean()


def _stack_work(c, rows, pairs, batch):
    """Layers over `rows` rows with `pairs` query-key pairs. Where only each
    sequence's first row is read, the last layer's row-wise half needs just
    those. bytes: every weight once."""
    L, d, f = c["layers"], c["hidden"], c["ffn"]
    fu = 2 * f if c["gated"] else f
    per_row = d * d + d * fu + f * d
    first = c.get("cls", c["kind"] == "vit")
    flops = 2.0 * L * (rows * 3 * d * d) + 4.0 * pairs * d * (L - 1 if first else L)
    flops += 2.0 * per_row * (rows * (L - 1) + batch if first else rows * L)
    return flops, 2.0 * L * (3 * d * d + per_row)


def work(case):
    kind = case["kind"]
    if kind in ("embed", "service"):
        c = MODELS[case["model"]]
        n = case["batch"] if kind == "embed" else case["sequences"]
        rows, pairs = _mean_lens(case["seq"], n)
        flops, weights = _stack_work(c, rows, pairs, n)
        d = c["hidden"]
        return dict(flops=flops, bytes=weights + n * case["seq"] * 8 + rows * d * 4 + n * d * 4)
    if kind == "vit":
        c, B = MODELS[case["model"]], case["batch"]
        P, d = (IMAGE // PATCH) ** 2, c["hidden"]
        flops, weights = _stack_work(c, B * (P + 1), B * (P + 1) ** 2, B)
        flops += 2.0 * B * (P * 3 * PATCH * PATCH * d + d * LABELS)
        return dict(flops=flops, bytes=weights + B * (3 * IMAGE * IMAGE + LABELS) * 4 +
                    2.0 * d * (3 * PATCH * PATCH + LABELS))
    if kind == "whisper":
        c, B = MODELS[case["model"]], case["batch"]
        S, d = FRAMES // 2, c["hidden"]
        flops, weights = _stack_work(c, B * S, B * S * S, B)
        flops += 2.0 * B * (FRAMES * 3 * MELS * d + S * 3 * d * d)
        return dict(flops=flops, bytes=weights + B * (MELS * FRAMES + S * d) * 4 +
                    6.0 * d * (MELS + d))
    if kind == "gemm":
        M, K, N = case["rows"], case["k"], case["n"]
        cb = 4 if case["c"] == "f32" else 2
        return dict(flops=2.0 * M * K * N,
                    bytes=2.0 * (M * K + K * N) + N * 4 + M * N * (cb + 4 * case["residual"]))
    if kind == "int8_ffn":
        M, d, f = case["rows"], case["hidden"], case["ffn"]
        return dict(flops=4.0 * M * d * f, bytes=2.0 * d * f + M * d * 9 + M * 4)
    if kind == "attention":
        d = case["heads"] * case["head_dim"]
        rows, pairs = _mean_lens(case["seq"], case["batch"])
        # every padded query is computed over its sequence's own keys
        pairs = case["seq"] * rows
        return dict(flops=4.0 * pairs * d, bytes=2.0 * case["batch"] * case["seq"] * 2 * d +
                    2.0 * rows * 2 * d)
    return dict(flops=0, bytes=case["rows"] * case["cols"] * 12.0)


def tolerance(case):
    """About four times what each shows against exact()."""
    kind = case["kind"]
    if kind in ("embed", "service"):
        # bf16 activations between every op of 6 to 24 layers: 4e-3 of a CLS
        # row, of which mean pooling averages most (5e-4 to 8e-4).
        return {"rel": 1.6e-2 if MODELS[case["model"]]["cls"] else 4e-3}
    if kind == "vit":
        return {"rel": 1.8e-2}
    if kind == "whisper":
        return {"rel": 1.4e-2}
    if kind == "gemm":
        return {"rel": 7e-3} if case["c"] == "bf16" else {"rel": 5e-6}
    if kind == "int8_ffn":
        # a difference in the last bit before a quantiser moves a code by one
        return {"rel": 5e-3, "differ": 2e-2}
    if kind == "attention":
        return {"rel": 9e-3}
    return {"rel": 3e-3}


# ---- the same in 64 bits ------------------------------------------------------------

def _f64(t):
    return t.to(torch.float64)


def _norm64(x, g, b, eps):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + eps) * _f64(g) + _f64(b)


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def _attend64(q, k, v):
    """[H, S, hd] each, a block of queries at a time."""
    out = torch.empty_like(q)
    for at in range(0, q.shape[1], 512):
        p = torch.softmax(q[:, at:at + 512] @ k.transpose(1, 2).contiguous(), -1)
        out[:, at:at + 512] = p @ v
    return out


def _rotate64(x, angle):
    """[H, S, hd]: pairs (j, j + hd/2) by angle [S, hd/2]."""
    h = x.shape[-1] // 2
    c, s = angle.cos(), angle.sin()
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attn_rows64(c, qkv, spans, angle=None):
    """Attention over [rows, 3d]; spans: (first row, length) per sequence."""
    d, H = c["hidden"], c["heads"]
    out = torch.empty_like(qkv[:, :d])
    for at, n in spans:
        q, k, v = (t.reshape(n, H, d // H).transpose(0, 1).contiguous()
                   for t in qkv[at:at + n].split(d, 1))
        if angle is not None:
            q, k = _rotate64(q, angle[:n]), _rotate64(k, angle[:n])
        out[at:at + n] = _attend64(q, k, v).transpose(0, 1).reshape(n, d)
    return out


def _ffn64(c, w, layer, h):
    h = h @ _f64(w["w_up"][layer]) + _f64(w["b_up"][layer])
    if c["gated"]:
        lo, hi = h.split(c["ffn"], 1)
        h = lo * (hi * torch.sigmoid(hi) if c["gated"] == 1 else _gelu64(hi))
    else:
        h = _gelu64(h)
    return h @ _f64(w["w_down"][layer]) + _f64(w["b_down"][layer])


def _bert64(case, seed, sequences):
    c, w = MODELS[case["model"]], _weights(case["model"])
    ids, _, lens = _text(case, seed, sequences)
    flat = torch.from_numpy(np.concatenate([ids[b, :n] for b, n in enumerate(lens)])).to(_DEV)
    at = np.concatenate([[0], np.cumsum(lens)])
    spans = [(int(at[b]), int(n)) for b, n in enumerate(lens)]
    where = torch.from_numpy(np.concatenate([np.arange(n) for n in lens])).to(_DEV)
    angle = None
    if c["gated"]:
        inv = torch.from_numpy(np.asarray(_inv_freq(case["model"]), np.float64)).to(_DEV)
        angle = torch.arange(case["seq"], device=_DEV, dtype=torch.float64)[:, None] * inv
    x = _f64(w["word"])[flat.long()] + _f64(w["pos"])[where.long()] + _f64(w["type"][0])
    x = _norm64(x, w["emb_ln_g"], w["emb_ln_b"], 1e-12)
    for i in range(c["layers"]):
        qkv = x @ _f64(w["w_qkv"][i]) + _f64(w["b_qkv"][i])
        y = _attn_rows64(c, qkv, spans, angle) @ _f64(w["w_ao"][i]) + _f64(w["b_ao"][i])
        x = _norm64(x + y, w["ln1_g"][i], w["ln1_b"][i], 1e-12)
        x = _norm64(x + _ffn64(c, w, i, x), w["ln2_g"][i], w["ln2_b"][i], 1e-12)
    out = torch.stack([x[a] if c["cls"] else x[a:a + n].mean(0) for a, n in spans])
    return out / out.norm(dim=1, keepdim=True)


def _preln64(case, x, eps):
    """x [B, S, d] through the pre-LN stack and its final LayerNorm."""
    c, w = MODELS[case["model"]], _weights(case["model"])
    B, S, d = x.shape
    x = x.reshape(B * S, d)
    spans = [(b * S, S) for b in range(B)]
    for i in range(c["layers"]):
        h = _norm64(x, w["ln1_g"][i], w["ln1_b"][i], eps)
        h = h @ _f64(w["w_qkv"][i]) + _f64(w["b_qkv"][i])
        x = x + _attn_rows64(c, h, spans) @ _f64(w["w_ao"][i]) + _f64(w["b_ao"][i])
        x = x + _ffn64(c, w, i, _norm64(x, w["ln2_g"][i], w["ln2_b"][i], eps))
    return _norm64(x, w["fin_ln_g"], w["fin_ln_b"], eps).reshape(B, S, d)


def exact(case, seed):
    kind = case["kind"]
    if kind == "embed":
        return _bert64(case, seed, case["batch"])
    if kind == "service":
        return _bert64(case, seed, case["sequences"]).cpu().numpy()
    t = _inputs(case, seed)
    if kind == "vit":
        w, B, n = _weights(case["model"]), case["batch"], IMAGE // PATCH
        p = _f64(t["pixels"]).reshape(B, 3, n, PATCH, n, PATCH).permute(0, 2, 4, 1, 3, 5)
        x = p.reshape(B, n * n, -1) @ _f64(w["patch_w"]) + _f64(w["patch_b"])
        x = torch.cat([_f64(w["cls_token"]).expand(B, 1, -1), x], 1) + _f64(w["pos"])
        x = _preln64(case, x, 1e-12)[:, 0].contiguous()
        return x @ _f64(w["head_w"]) + _f64(w["head_b"])
    if kind == "whisper":
        w = _weights(case["model"])
        x = _f64(t["mel"])
        for i, step in ((1, 1), (2, 2)):
            # a convolution of three taps, as three products
            p = torch.nn.functional.pad(x, (1, 1))
            n = x.shape[2] // step
            taps = [p[:, :, k:k + step * (n - 1) + 1:step].contiguous() for k in range(3)]
            k64 = _f64(w["conv%d_w" % i])
            x = torch.stack([sum(k64[:, :, k].contiguous() @ taps[k][b] for k in range(3))
                             for b in range(x.shape[0])])
            x = _gelu64(x + _f64(w["conv%d_b" % i])[:, None])
        return _preln64(case, x.transpose(1, 2).contiguous() + _f64(w["pos"]), 1e-5)
    if kind == "gemm":
        y = _f64(t["a"]) @ _f64(t["w"]).T.contiguous() + _f64(t["bias"])
        if case["epi"] != "none":
            y = _gelu64(y)
        return y + _f64(t["res"]) if case["residual"] else y
    if kind == "int8_ffn":
        h = _f64(t["x"])
        for key in ("up", "down"):
            u = h * _f64(t["ias_" + key])
            a = u.abs().amax(1, keepdim=True) / 127.0
            q = (u / a).round()
            h = (q @ _f64(t["w_" + key]).T.contiguous()) * a * _f64(t["s_" + key]) + _f64(
                t["b_" + key])
            if key == "up":
                h = _gelu64(h)
        out = _norm64(_f64(t["x"]) + h, t["g"], t["b"], 1e-12)
        return out, None, (out * _f64(t["ias_next"])).abs().amax(1) / 127.0
    if kind == "attention":
        B, S, d = case["batch"], case["seq"], case["heads"] * case["head_dim"]
        c = dict(hidden=d, heads=case["heads"])
        out = torch.empty((B * S, d), device=_DEV, dtype=torch.float64)
        H, qkv = case["heads"], _f64(t["qkv"])
        for b, n in enumerate(t["kv_len"].tolist()):
            q, k, v = (u.reshape(S, H, d // H).transpose(0, 1).contiguous()
                       for u in qkv[b * S:(b + 1) * S].split(d, 1))
            o = _attend64(q, k[:, :n].contiguous(), v[:, :n].contiguous())
            out[b * S:(b + 1) * S] = o.transpose(0, 1).reshape(S, c["hidden"])
        return out
    y = _norm64(_f64(t["x"]) + _f64(t["y"]), t["g"], t["b"], 1e-12)
    return y, y
