"""The work that users of this package have it do, as cases that can be timed and compared.

Each case goes through the package's public entry points: ``RWKV7HIP`` /
``RWKV7HIPBF16`` / ``RWKV7HIPInt8`` (``decode``, ``prefill``, ``forward``), the
operators ``kernels.wkv7`` and ``kernels.gemm``, the training operator
``torch.ops.rwkv_tl.fused_dplr_seq`` with its backward, and ``Sampler``.

``listed`` holds the cases, ``draw`` makes more of the same ranges, ``prepare``
builds what a program holds before the call, ``run`` is one pass, ``work`` its
unavoidable bytes and operations, ``tolerance`` how far another correct
implementation may be off, and ``exact`` the same outputs in 64 bits by plain
torch. Weights and inputs are drawn on the GPU from the seed alone.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

for _p in (Path.cwd() / "rwkv-tl_amd", Path(__file__).resolve().parent.parent / "rwkv-tl_amd"):
    if _p.is_dir():
        sys.path.insert(0, str(_p))
        break

from rwkv_tl_amd import RWKV7HIP, RWKV7HIPBF16, RWKV7HIPInt8, RWKV7Weight, SHAPES, State, kernels  # noqa: E402
from rwkv_tl_amd.sampling import Sampler  # noqa: E402

DEV = "cuda"
N = 64  # head size
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "int8": torch.float16, "f32": torch.float32}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def listed() -> list[dict]:
    return [
        # one token of a chat at batch 1: the smallest step, all latency
        {"name": "decode_b1", "kind": "decode", "model": "0.4b", "dtype": "f16", "B": 1},
        # one token of each of 16 conversations served together
        {"name": "decode_b16", "kind": "decode", "model": "0.4b", "dtype": "f16", "B": 16},
        # a wide serving batch of the larger model
        {"name": "decode_b64_1p5b", "kind": "decode", "model": "1.5b", "dtype": "f16", "B": 64},
        # a short user turn appended to a conversation, a ragged length
        {"name": "prefill_1x13", "kind": "prefill", "model": "0.4b", "dtype": "f16", "B": 1, "T": 13},
        # a prompt of 129 tokens and the first answer token's logits
        {"name": "forward_1x129", "kind": "forward", "model": "0.4b", "dtype": "f16", "B": 1, "T": 129},
        # a document of odd length on the bfloat16 model
        {"name": "prefill_1x509_bf16", "kind": "prefill", "model": "0.4b", "dtype": "bf16", "B": 1, "T": 509},
        # nine short prompts of 29 tokens admitted together
        {"name": "prefill_9x29", "kind": "prefill", "model": "0.4b", "dtype": "f16", "B": 9, "T": 29},
        # four long prompts on the larger model: the largest call, matrix-bound
        {"name": "prefill_4x1024_1p5b", "kind": "prefill", "model": "1.5b", "dtype": "f16", "B": 4, "T": 1024},
        # the recurrence alone, as an operator in a caller's own model
        {"name": "wkv7_8x128", "kind": "wkv7", "dtype": "f16", "w_f32": True, "B": 8, "T": 128, "H": 16},
        # the recurrence in training: forward and backward of one layer, f32
        {"name": "wkv7_train_4x512", "kind": "train", "B": 4, "T": 512, "H": 16},
        # the FFN key product with relu^2 as an operator, a ragged row count
        {"name": "gemm_ffn_key_250", "kind": "gemm", "dtype": "f16", "a_f32": False, "M": 250, "N": 8192, "K": 2048,
         "epi": "relu2"},
        # one sampling step of a serving batch: penalty, top-k, top-p, draw
        {"name": "sample_b16", "kind": "sample", "dtype": "f16", "B": 16, "V": 65536, "top_k": 50, "top_p": 0.9},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "wkv7", "train", "gemm", "sample"])
    if kind == "decode":
        model = rng.choice(["0.1b", "0.4b", "0.4b", "1.5b"])
        B = _log(rng, 1, 64 if model == "1.5b" else 128)
        dtypes = ["f16", "f16", "bf16"] + (["int8"] if B == 1 and model != "1.5b" else [])
        return {"kind": kind, "model": model, "dtype": rng.choice(dtypes), "B": B}
    if kind == "prefill":
        model = rng.choice(["0.1b", "0.4b", "0.4b", "1.5b"])
        rows = _log(rng, 2, 3500 if model == "1.5b" else 1800)
        B = _log(rng, 1, min(32, max(1, rows // 2)))
        dtype = rng.choice(["f16", "f16", "bf16"])
        if B == 1 and rng.random() < 0.3:
            return {"kind": "forward", "model": model, "dtype": dtype, "B": 1, "T": max(2, rows)}
        return {"kind": kind, "model": model, "dtype": dtype, "B": B, "T": max(2, rows // B)}
    if kind == "wkv7":
        return {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "w_f32": rng.random() < 0.5, "B": _log(rng, 1, 16),
                "T": _log(rng, 1, 1024), "H": rng.choice([12, 16, 32])}
    if kind == "train":
        return {"kind": kind, "B": _log(rng, 1, 6), "T": _log(rng, 8, 600), "H": rng.choice([12, 16])}
    if kind == "gemm":
        n, k = rng.choice([(1024, 1024), (4096, 1024), (1024, 4096), (8192, 2048), (2048, 8192), (768, 3072)])
        return {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "a_f32": rng.random() < 0.4, "M": _log(rng, 1, 4096),
                "N": n, "K": k, "epi": rng.choice(["f32", "f16", "relu2"])}
    return {"kind": kind, "dtype": rng.choice(["f16", "f16", "bf16", "f32"]), "B": _log(rng, 1, 64), "V": 65536,
            "top_k": rng.choice([0, 20, 50, 100]), "top_p": rng.choice([0.5, 0.9, 0.95, 1.0])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _state_dict(model: str, dtype: torch.dtype, g: torch.Generator) -> dict[str, torch.Tensor]:
    """Random weights of the named shape: N(0, 0.02) matrices, LayerNorms near
    the identity, and per-channel vectors spread as trained models have them
    (mixes in [0, 1], decays from slow to fast, key scales near 1)."""
    s = SHAPES[model]
    C, Fh, V = s.n_embd, s.n_ffn, s.vocab

    def mat(*shape):
        return (torch.randn(*shape, generator=g, device=DEV) * 0.02).to(dtype)

    def uni(lo, hi, *shape):
        return (torch.rand(*shape, generator=g, device=DEV) * (hi - lo) + lo).to(dtype)

    def nor(mean, std, *shape):
        return (torch.randn(*shape, generator=g, device=DEV) * std + mean).to(dtype)

    sd = {"emb.weight": mat(V, C), "head.weight": mat(V, C)}

    def ln(name):
        sd[f"{name}.weight"], sd[f"{name}.bias"] = nor(1.0, 0.05, C), nor(0.0, 0.02, C)

    ln("blocks.0.ln0")
    ln("ln_out")
    for i in range(s.n_layer):
        a, f = f"blocks.{i}.att", f"blocks.{i}.ffn"
        for name in (f"blocks.{i}.ln1", f"blocks.{i}.ln2", f"{a}.ln_x"):
            ln(name)
        for v in ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g"):
            sd[f"{a}.{v}"] = uni(0.0, 1.0, 1, 1, C)
        sd[f"{a}.w0"] = uni(-6.0, 1.0, 1, 1, C)
        for v in ("a0", "v0"):
            sd[f"{a}.{v}"] = nor(0.0, 0.5, 1, 1, C)
        sd[f"{a}.k_k"], sd[f"{a}.k_a"] = uni(0.5, 1.0, 1, 1, C), uni(0.8, 1.1, 1, 1, C)
        sd[f"{a}.r_k"] = nor(0.0, 0.1, s.n_head, N)
        for name, r in (("w", s.rank_w), ("a", s.rank_a), ("v", s.rank_v), ("g", s.rank_g)):
            sd[f"{a}.{name}1"], sd[f"{a}.{name}2"] = mat(C, r), mat(r, C)
        for m in ("receptance", "key", "value", "output"):
            sd[f"{a}.{m}.weight"] = mat(C, C)
        sd[f"{f}.x_k"] = uni(0.0, 1.0, 1, 1, C)
        sd[f"{f}.key.weight"], sd[f"{f}.value.weight"] = mat(Fh, C), mat(C, Fh)
    return sd


def _model_inputs(case: dict, seed: int):
    """Weights, token ids [B, T] and, for decode, a state in mid-conversation."""
    g, s, dt, B = _gen(seed), SHAPES[case["model"]], DTYPES[case["dtype"]], case["B"]
    sd = _state_dict(case["model"], dt, g)
    T = case.get("T", 1)
    tokens = torch.randint(0, s.vocab, (B, T), generator=g, device=DEV)
    start = None
    if case["kind"] == "decode":
        tx = torch.randn(s.n_layer, B, s.n_embd, generator=g, device=DEV).to(dt)
        rnn = torch.randn(s.n_layer, B, s.n_head, N, N, generator=g, device=DEV) * 0.1
        cx = torch.randn(s.n_layer, B, s.n_embd, generator=g, device=DEV).to(dt)
        start = (tx, rnn, cx)
    return sd, tokens, start


def _wkv_inputs(B: int, T: int, H: int, g: torch.Generator):
    """r, w, k, v, a, b, S0 in f32: a the negated normalised key, b = key * rate, decay exp(-exp(N(-0.5, 0.5)))."""
    shape = (B, T, H, N)

    def rn():
        return torch.randn(*shape, generator=g, device=DEV)

    r, k, v = rn(), rn(), rn()
    w = torch.exp(-torch.exp(rn() * 0.5 - 0.5))
    kk = F.normalize(k, dim=-1)
    b = kk * torch.sigmoid(rn())
    S = torch.randn(B, H, N, N, generator=g, device=DEV) * 0.1
    return r, w, k, v, -kk, b, S


def _op_wkv_inputs(case: dict, seed: int):
    r, w, k, v, a, b, S = _wkv_inputs(case["B"], case["T"], case["H"], _gen(seed))
    dt = DTYPES[case["dtype"]]
    return S, r.to(dt), w if case["w_f32"] else w.to(dt), k.to(dt), v.to(dt), a.to(dt), b.to(dt)


def _train_inputs(case: dict, seed: int):
    g = _gen(seed)
    r, w, k, v, a, b, S = _wkv_inputs(case["B"], case["T"], case["H"], g)
    gy = torch.randn(r.shape, generator=g, device=DEV)
    gS = torch.randn(S.shape, generator=g, device=DEV) * 0.1
    return (S, r, w, k, v, a, b), gy, gS


def _gemm_inputs(case: dict, seed: int):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    A = torch.randn(case["M"], case["K"], generator=g, device=DEV)
    W = (torch.randn(case["N"], case["K"], generator=g, device=DEV) * 0.02).to(dt)
    return (A if case["a_f32"] else A.to(dt)), W


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("decode", "prefill", "forward"):
        sd, tokens, start = _model_inputs(case, seed)
        dt = DTYPES[case["dtype"]]
        w = RWKV7Weight.from_state_dict(sd, device=DEV, dtype=dt)
        cls = {"f16": RWKV7HIP, "bf16": RWKV7HIPBF16, "int8": RWKV7HIPInt8}[case["dtype"]]
        model = cls(w, is_torch_compile=False)
        B = case["B"]
        S = State(model.L, model.C, N, device=DEV, dtype=dt, batch=None if B == 1 else B)
        if start is not None:
            for dst, src in zip(S.arenas, start):
                dst.copy_(src)
        toks = tokens[0] if B == 1 else (tokens.reshape(B) if kind == "decode" else tokens)
        return {"kind": kind, "model": model, "S": S, "tokens": toks}
    if kind == "wkv7":
        return {"kind": kind, "args": _op_wkv_inputs(case, seed)}
    if kind == "train":
        xs, gy, gS = _train_inputs(case, seed)
        return {"kind": kind, "xs": [x.requires_grad_(True) for x in xs], "gy": gy, "gS": gS}
    if kind == "gemm":
        A, W = _gemm_inputs(case, seed)
        return {"kind": kind, "A": A, "W": W, "epi": case["epi"]}
    g = _gen(seed)
    logits = (torch.randn(case["B"], case["V"], generator=g, device=DEV) * 2.5).to(DTYPES[case["dtype"]])
    sampler = Sampler(case["V"], DEV, batch=case["B"], temperature=0.8, top_k=case["top_k"], top_p=case["top_p"],
                      repetition_penalty=1.1, seed=seed)
    return {"kind": kind, "logits": logits, "sampler": sampler,
            "out": torch.empty(case["B"], dtype=torch.int64, device=DEV)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(st):
    kind = st["kind"]
    if kind == "decode":
        logits, S = st["model"].decode(st["tokens"], st["S"])
        return [logits, *S.arenas]
    if kind == "prefill":
        S = st["model"].prefill(st["tokens"], st["S"])
        return list(S.arenas)
    if kind == "forward":
        logits, S = st["model"].forward(st["tokens"], st["S"])
        return [logits, *S.arenas]
    if kind == "wkv7":
        S, *rest = st["args"]
        return [kernels.wkv7(S, *rest), S]
    if kind == "train":
        y, S_T = torch.ops.rwkv_tl.fused_dplr_seq(*st["xs"])
        grads = torch.autograd.grad((y, S_T), st["xs"], (st["gy"], st["gS"]))
        return [y, S_T, *grads]
    if kind == "gemm":
        return kernels.gemm(st["A"], st["W"], st["epi"])
    st["sampler"](st["logits"], st["out"])
    return [st["out"], st["sampler"].seen]


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far off it may be
# ---------------------------------------------------------------------------


def _layer_params(model: str) -> int:
    s = SHAPES[model]
    C, SR = s.n_embd, s.rank_w + s.rank_a + s.rank_v + s.rank_g
    return 4 * C * C + 2 * C * s.n_ffn + 2 * C * SR


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("decode", "prefill", "forward"):
        s, B, T = SHAPES[case["model"]], case["B"], case.get("T", 1)
        P, C, M = _layer_params(case["model"]), s.n_embd, B * T
        wb = 1 if case["dtype"] == "int8" else 2
        nbytes = s.n_layer * (wb * P + 19 * C * 4) + 2 * M * C + 8 * M  # weights, embedding rows, token ids
        nbytes += s.n_layer * B * 2 * (s.n_head * N * N * 4 + 2 * 2 * C)  # state, read and written
        flops = s.n_layer * M * (2 * P + 8 * s.n_head * N * N)
        if kind != "prefill":  # the head and its logits
            nbytes += wb * s.vocab * C + 2 * B * s.vocab
            flops += 2 * B * s.vocab * C
        return {"bytes": nbytes, "flops": flops}
    if kind == "wkv7":
        e = case["B"] * case["T"] * case["H"] * N
        S = case["B"] * case["H"] * N * N
        return {"bytes": e * (2 * 6 + (4 if case["w_f32"] else 2)) + 8 * S, "flops": 8 * e * N}
    if kind == "train":
        e = case["B"] * case["T"] * case["H"] * N
        S = case["B"] * case["H"] * N * N
        # six inputs and gy read, y and six gradients written; S0, S_T, gS_T, gS0
        return {"bytes": 4 * (14 * e + 4 * S), "flops": (8 + 20) * e * N}
    if kind == "gemm":
        M, n, k = case["M"], case["N"], case["K"]
        out = 4 if case["epi"] == "f32" else 2
        return {"bytes": (4 if case["a_f32"] else 2) * M * k + 2 * n * k + out * M * n, "flops": 2 * M * n * k}
    size = 4 if case["dtype"] == "f32" else 2
    return {"bytes": case["B"] * (size * case["V"] + case["V"] // 8 + 8), "flops": 0}


# 16-bit operands run from this many rows of the widest layer matrix on (long
# prefills); below, activations keep 32-bit precision
_LONG = {"0.1b": 2689, "0.4b": 1921, "1.5b": 897}


def tolerance(case: dict):
    kind, bf = case["kind"], case.get("dtype") == "bf16"
    if kind == "sample":
        return "exact"
    if kind == "train":  # f32 throughout
        return {"rel": 1e-5}
    if kind == "gemm" and case["epi"] == "f32":  # f32 sums of exact products, over K terms
        return {"rel": 1e-5}
    if kind in ("prefill", "forward") and case["B"] * case["T"] >= _LONG[case["model"]]:
        # 16-bit operands in every product of 24 layers (measured: 9e-4 off 64 bits in f16)
        return {"rel": 3e-2 if bf else 5e-3}
    # the 16-bit outputs' own rounding: half a unit is 2^-12 (f16), 2^-9 (bf16) of a value
    return {"rel": 8e-3 if bf else 1e-3}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------


def _scan64(S, r, w, k, v, a, b, y):
    """The recurrence step by step; every argument f64, y [B, T, H, N] filled; returns the last state."""
    for t in range(r.shape[1]):
        sa = torch.matmul(S, a[:, t].unsqueeze(-1))
        S = S * w[:, t].unsqueeze(-2)
        S = torch.addcmul(S, sa, b[:, t].unsqueeze(-2))
        S = torch.addcmul(S, v[:, t].unsqueeze(-1), k[:, t].unsqueeze(-2))
        y[:, t] = torch.matmul(S, r[:, t].unsqueeze(-1)).squeeze(-1)
    return S


def _dequantised(W):
    """[out, in] weights as symmetric per-row int8 holds them (scale max|row| / 127 in f32)."""
    w = W.float()
    scale = w.abs().amax(dim=1) * torch.tensor(1.0 / 127.0, dtype=torch.float32, device=w.device)
    q = torch.round(w.double() / scale.double()[:, None]).clamp_(-127, 127)
    return q * scale.double()[:, None]


def _exact_model(case: dict, seed: int):
    sd, tokens, start = _model_inputs(case, seed)
    s, B, T = SHAPES[case["model"]], case["B"], tokens.shape[1]
    C, H, M = s.n_embd, s.n_head, B * T
    quant = case["dtype"] == "int8"
    # the embedding is normalised once at load, in the model's 16-bit format
    emb = F.layer_norm(sd["emb.weight"], (C,), sd["blocks.0.ln0.weight"], sd["blocks.0.ln0.bias"])
    x = F.embedding(tokens, emb).double()
    if start is None:
        z = torch.zeros(s.n_layer, B, C, device=DEV, dtype=torch.float64)
        start = (z, torch.zeros(s.n_layer, B, H, N, N, device=DEV, dtype=torch.float64), z)
    tx, rnn, cx = (t.double().clone() for t in start)

    def vec(name):
        return sd[name].double().reshape(-1)

    def lin(z, W):  # W [out, in], streamed as int8 by the int8 decode
        return torch.matmul(z, (_dequantised(W) if quant else W.double()).t())

    def ln(z, name):
        return F.layer_norm(z, (C,), vec(f"{name}.weight"), vec(f"{name}.bias"))

    def shifted(z, last):
        return torch.cat([last.unsqueeze(1), z[:, :-1]], dim=1)

    v_first = None
    for i in range(s.n_layer):
        a_, f_ = f"blocks.{i}.att", f"blocks.{i}.ffn"
        z = ln(x, f"blocks.{i}.ln1")
        d = shifted(z, tx[i]) - z
        tx[i] = z[:, -1]
        m = {c: z + vec(f"{a_}.x_{c}") * d for c in "rwkvag"}
        r = lin(m["r"], sd[f"{a_}.receptance.weight"])
        k = lin(m["k"], sd[f"{a_}.key.weight"])
        v = lin(m["v"], sd[f"{a_}.value.weight"])

        def lora(c, act=lambda q: q):
            h = act(lin(m[c], sd[f"{a_}.{c}1"].t()))
            return torch.matmul(h, sd[f"{a_}.{c}2"].double())

        if v_first is None:
            v_first = v
        else:
            v = v + (v_first - v) * torch.sigmoid(vec(f"{a_}.v0") + lora("v"))
        w = torch.exp(-torch.sigmoid(vec(f"{a_}.w0") + lora("w", torch.tanh)) / math.sqrt(math.e))
        a = torch.sigmoid(vec(f"{a_}.a0") + lora("a"))
        gate = lora("g", torch.sigmoid)
        kk = (k * vec(f"{a_}.k_k")).view(B, T, H, N)
        k = k + (k * a - k) * vec(f"{a_}.k_a")
        kk = kk / kk.norm(dim=-1, keepdim=True).clamp(min=1e-12)
        r, w, k, v4, a = (q.view(B, T, H, N) for q in (r, w, k, v, a))
        y = torch.empty_like(r)
        rnn[i] = _scan64(rnn[i], r, w, k, v4, kk, -kk * a, y)
        y = F.group_norm(y.reshape(M, C), H, vec(f"{a_}.ln_x.weight"), vec(f"{a_}.ln_x.bias"), 64e-5).view(B, T, H, N)
        y = y + (r * k * sd[f"{a_}.r_k"].double()).sum(-1, keepdim=True) * v4
        x = x + lin(y.reshape(B, T, C) * gate, sd[f"{a_}.output.weight"])
        z = ln(x, f"blocks.{i}.ln2")
        zk = z + vec(f"{f_}.x_k") * (shifted(z, cx[i]) - z)
        cx[i] = z[:, -1]
        x = x + lin(torch.relu(lin(zk, sd[f"{f_}.key.weight"])) ** 2, sd[f"{f_}.value.weight"])
    if case["kind"] == "prefill":
        return [tx, rnn, cx]
    logits = lin(ln(x[:, -1], "ln_out"), sd["head.weight"])
    return [logits[0] if B == 1 else logits, tx, rnn, cx]


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("decode", "prefill", "forward"):
        return _exact_model(case, seed)
    if kind == "wkv7":
        S, r, w, k, v, a, b = (t.double() for t in _op_wkv_inputs(case, seed))
        y = torch.empty_like(r)
        S = _scan64(S, r, w, k, v, a, b, y)
        return [y, S]
    if kind == "train":
        xs, gy, gS = _train_inputs(case, seed)
        xs = [x.double().requires_grad_(True) for x in xs]
        S, r, w, k, v, a, b = xs
        ys = []
        for t in range(r.shape[1]):
            sa = torch.matmul(S, a[:, t].unsqueeze(-1))
            S = S * w[:, t].unsqueeze(-2) + sa * b[:, t].unsqueeze(-2) + v[:, t].unsqueeze(-1) * k[:, t].unsqueeze(-2)
            ys.append(torch.matmul(S, r[:, t].unsqueeze(-1)).squeeze(-1))
        y = torch.stack(ys, dim=1)
        grads = torch.autograd.grad((y, S), xs, (gy.double(), gS.double()))
        return [y.detach(), S.detach(), *grads]
    if kind == "gemm":
        A, W = _gemm_inputs(case, seed)
        y = torch.matmul(A.double(), W.double().t())
        return torch.relu(y) ** 2 if case["epi"] == "relu2" else y
    return None  # token ids
