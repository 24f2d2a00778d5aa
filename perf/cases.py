"""What a user of the engine has it do, as measurable cases.

The package decodes and prefills GatedDeltaNet-1.3B (hidden 2048, 8 x 256
heads, MLP 5632, vocabulary 32000) on one GPU.  Its uses, and the cases that
stand for them:

  decode     ``RunState``: one token stream, the checkpoint's latency path, in
             the three arithmetic contracts (REF: BF16 state; BF16W_FP32S:
             FP32 state, the default; FP32: the control arm)
  streams    ``BatchState``: 1..64 independent streams a step, for serving
  prefill    ``BatchState.prefill``: a prompt of 1..4096 tokens through one
             stream's state, in the scan (default, equal to the steps) or the
             chunked form, then either the first decode steps of the answer
             or the export of the state (what a ``.gdnstate`` file holds)
  recurrence ``gdn_recurrence_noalloc``: the gated delta rule alone on the
             caller's own device buffers

The layers of a model are alike, so most cases run a few of them (1, 2 and 24
are the depths the tests use); two run the whole model, as the benchmark does.
"""
from __future__ import annotations

import math
from typing import Dict, Optional, Tuple

import numpy as np
import torch

import gateddeltanet_amd as g
from gateddeltanet_amd import _lib

H, NH, HD, I, V = 2048, 8, 256, 5632, 32000
STATE = NH * HD * HD   # recurrent state of a layer
TAILS = 3 * 3 * H      # conv tails of a layer
LAYER_W = 5 * H * H + 3 * H * I
REF, BF16W, FP32 = g.CONTRACT_REF, g.CONTRACT_BF16W_FP32S, g.CONTRACT_FP32


def listed():
    return [
        # The headline: a chat's next tokens from the whole model, a given
        # token in and the argmax out, with the last step's logits.
        {"name": "decode_24_layers", "kind": "decode", "contract": BF16W, "layers": 24, "steps": 8},
        # The smallest call: two steps of one layer in the reference's own
        # arithmetic (launches and latency).
        {"name": "decode_ref_1_layer", "kind": "decode", "contract": REF, "layers": 1, "steps": 2},
        # The FP32 control arm, as a parity run steps it.
        {"name": "decode_fp32", "kind": "decode", "contract": FP32, "layers": 3, "steps": 5},
        # A small odd number of conversations at a time.
        {"name": "streams_3", "kind": "streams", "layers": 4, "streams": 3, "steps": 8},
        # An ordinary serving batch.
        {"name": "streams_16", "kind": "streams", "layers": 4, "streams": 16, "steps": 8},
        # The full batch over the whole model, the benchmark's serving leg.
        {"name": "streams_64_24_layers", "kind": "streams", "layers": 24, "streams": 64, "steps": 4},
        # A short prompt and the state it leaves, for a .gdnstate file.
        {"name": "prefill_70_export", "kind": "prefill", "mode": "chunked", "layers": 2, "tokens": 70,
         "steps": 0},
        # A short prompt in the default mode, then the answer's first tokens.
        {"name": "prefill_scan_200", "kind": "prefill", "mode": "scan", "layers": 4, "tokens": 200, "steps": 2},
        # An ordinary prompt of no round length.
        {"name": "prefill_1000", "kind": "prefill", "mode": "chunked", "layers": 4, "tokens": 1000, "steps": 2},
        # The benchmark's prompt, in both modes.
        {"name": "prefill_4096", "kind": "prefill", "mode": "chunked", "layers": 4, "tokens": 4096, "steps": 2},
        {"name": "prefill_scan_4096", "kind": "prefill", "mode": "scan", "layers": 2, "tokens": 4096, "steps": 2},
        # A caller's own loop over the recurrence: one sequence's heads.
        {"name": "recurrence_8_heads", "kind": "recurrence", "contract": BF16W, "heads": 8, "steps": 100},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    kind = rng.choice(["decode", "streams", "streams", "prefill", "prefill", "prefill", "recurrence"])
    layers = rng.randint(1, 4)
    if kind == "decode":
        return {"kind": kind, "contract": rng.choice([REF, BF16W, BF16W, FP32]), "layers": layers,
                "steps": _log_int(rng, 2, 24)}
    if kind == "streams":
        return {"kind": kind, "layers": layers, "streams": _log_int(rng, 1, 64), "steps": rng.randint(6, 10)}
    if kind == "prefill":
        return {"kind": kind, "mode": rng.choice(["scan", "chunked"]), "layers": min(layers, 2 + layers % 2),
                "tokens": _log_int(rng, 1, 4096), "steps": rng.choice([0, 2, 3])}
    return {"kind": kind, "contract": rng.choice([REF, BF16W, FP32]), "heads": _log_int(rng, 1, 48),
            "steps": _log_int(rng, 1, 200)}


# ---------------------------------------------------------------- the inputs

_models: Dict[Tuple[int, bool], g.Model] = {}


def _model(layers: int, bf16: bool) -> g.Model:
    """The checkpoint, loaded once by a program: random weights of the
    model's shapes, with the decay and conv parameters in a trained model's
    range (a in [1, 16), time steps of 1e-3 .. 0.1, taps within 0.5)."""
    key = (layers, bf16)
    if key not in _models:
        m = g.Model.synth(num_layers=layers, seed=layers, std=0.02, bf16=bf16)
        rng = np.random.default_rng(layers)
        for i in range(layers):
            w = m.layer(i)
            dt = np.exp(rng.uniform(np.log(1e-3), np.log(0.1), NH))
            new = {"a_log": np.log(rng.uniform(1, 16, NH)), "dt_bias": dt + np.log(-np.expm1(-dt))}
            for n in ("q_conv", "k_conv", "v_conv"):
                new[n] = rng.uniform(-0.5, 0.5, 4 * H)
            for n, x in new.items():
                x = x.astype(np.float32)
                w[n][:] = g.bf16_round(x) if bf16 else x
        _models[key] = m
    return _models[key]


def _decode_inputs(case, seed):
    rng = np.random.default_rng([seed, 1])
    L = case["layers"]
    tokens = rng.integers(0, V, case["steps"]).astype(np.int32)
    state = rng.standard_normal(L * STATE, dtype=np.float32) * np.float32(0.02)
    tails = rng.standard_normal(L * TAILS, dtype=np.float32)
    if case["contract"] != FP32:
        tails = g.bf16_round(tails)
    if case["contract"] == REF:
        state = g.bf16_round(state)
    return tokens, state, tails


def _streams_inputs(case, seed):
    rng = np.random.default_rng([seed, 2])
    tokens = rng.integers(0, V, (case["steps"], case["streams"])).astype(np.int32)
    if case["layers"] > 4:
        return tokens, None, None  # new conversations: zero state
    n = case["streams"]
    base = rng.standard_normal(case["layers"] * STATE, dtype=np.float32) * np.float32(0.02)
    state = np.stack([np.roll(base, 977 * s) for s in range(n)])
    tails = g.bf16_round(rng.standard_normal((n, case["layers"] * TAILS), dtype=np.float32))
    return tokens, state, tails.reshape(n, -1)


def _prefill_inputs(case, seed):
    rng = np.random.default_rng([seed, 3])
    return (rng.integers(0, V, case["tokens"]).astype(np.int32),
            rng.integers(0, V, (case["steps"], 1)).astype(np.int32))


def _recurrence_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n, s = case["heads"], case["steps"]

    def normal(*shape, std=1.0):
        return torch.randn(shape, generator=gen, device="cuda") * std

    def uniform(*shape):
        return torch.rand(shape, generator=gen, device="cuda")

    q, k, v = (torch.nn.functional.silu(normal(s, n, HD)) for _ in range(3))
    a, b = normal(s, n), normal(s, n)
    dt = torch.exp(math.log(1e-3) + uniform(n) * math.log(100.0))
    a_log = torch.log(1 + 15 * uniform(n)).expand(s, n).contiguous()
    dt_bias = (dt + torch.log(-torch.expm1(-dt))).expand(s, n).contiguous()
    S = normal(n, HD, HD, std=0.02)
    if case["contract"] != FP32:
        q, k, v, a, b = (x.bfloat16().float() for x in (q, k, v, a, b))
    if case["contract"] == REF:
        S = S.bfloat16()
    return q, k, v, a, b, a_log, dt_bias, S


def prepare(case, seed):
    kind = case["kind"]
    if kind == "recurrence":
        x = _recurrence_inputs(case, seed)
        out = torch.empty_like(x[0])
        torch.cuda.synchronize()
        return {"case": case, "in": x, "out": out}
    if kind == "decode":
        tokens, state, tails = _decode_inputs(case, seed)
        rs = g.RunState(_model(case["layers"], case["contract"] != FP32), case["contract"])
        rs.load_state(state, tails)
        return {"case": case, "engine": rs, "tokens": tokens}
    if kind == "streams":
        tokens, state, tails = _streams_inputs(case, seed)
        bs = g.BatchState(_model(case["layers"], True), case["streams"])
        for s in range(case["streams"] if state is not None else 0):
            bs.load_stream_state(s, state[s], tails[s])
        return {"case": case, "engine": bs, "tokens": tokens}
    prompt, tokens = _prefill_inputs(case, seed)
    bs = g.BatchState(_model(case["layers"], True), 1)
    bs.set_prefill_mode(g.PREFILL_CHUNKED if case["mode"] == "chunked" else g.PREFILL_SCAN)
    return {"case": case, "engine": bs, "prompt": prompt, "tokens": tokens}


# ------------------------------------------------------------------ one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "recurrence":
        q, k, v, a, b, a_log, dt_bias, S = state["in"]
        ptrs = [x.data_ptr() for x in (q, k, v, a, b, a_log, dt_bias, S, state["out"])]
        rc = _lib.load().gdn_recurrence_noalloc(case["contract"], case["heads"], case["steps"], *ptrs,
                                                torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise RuntimeError("gdn_recurrence_noalloc failed")
        return {"out": state["out"], "state": S}
    e = state["engine"]
    if kind == "decode":
        tokens = np.array([e.decode_step(int(t)) for t in state["tokens"]], np.int32)
        return {"tokens": tokens, "logits": e.logits(), "hidden": e.final_hidden()}
    if kind == "streams":
        tokens, _, _ = e.teacher_forced(state["tokens"], timing=False)
        return {"tokens": tokens, "logits": np.stack([e.logits(s) for s in range(case["streams"])])}
    # a turn of a conversation: the first pass starts from the empty state,
    # each later one continues from what the last left
    e.prefill(0, state["prompt"])
    out = {"logits": e.logits(0), "hidden": e.final_hidden(0)}
    if case["steps"]:
        e.teacher_forced(state["tokens"], timing=False)
        out["next_logits"] = e.logits(0)
    else:
        out["state"], out["tails"] = e.save_stream_state(0)
    return out


# ------------------------------------------------------- what it cannot avoid

def work(case):
    kind = case["kind"]
    if kind == "recurrence":
        n, s = case["heads"], case["steps"]
        state = n * HD * HD * (2 if case["contract"] == REF else 4)
        return {"bytes": 2 * state + s * n * (4 * HD + 4) * 4, "flops": s * n * HD * HD * 7}
    L = case["layers"]
    dense = L * LAYER_W + H * V  # weights of a pass over the model
    aux = L * (16 * H + 12 * H + 2 * H + HD + 16) + H
    if kind == "decode":
        w = 4 if case["contract"] == FP32 else 2
        st = 2 if case["contract"] == REF else 4
        per = dense * w + aux * w + 2 * L * (STATE * st + TAILS * w) + H * w + V * 4
        return {"bytes": case["steps"] * per, "flops": case["steps"] * (2 * dense + L * STATE * 7)}
    if kind == "streams":
        n = case["streams"]
        per = dense * 2 + aux * 4 + n * (2 * L * (STATE * 4 + TAILS * 2) + H * 2 + V * 4)
        return {"bytes": case["steps"] * per, "flops": case["steps"] * n * (2 * dense + L * STATE * 7)}
    t, k = case["tokens"], case["steps"]
    once = dense * 2 + aux * 4 + 2 * L * (STATE * 4 + TAILS * 2) + V * 4
    return {"bytes": (1 + k) * once + (t + k) * (4 + 2 * H),
            "flops": (t + k) * (2 * L * LAYER_W + L * STATE * 7) + (1 + k) * 2 * H * V}


def tolerance(case):
    kind = case["kind"]
    # one stream's decode and the recurrence alone are defined to the bit
    # (products, reduction orders and rounding points of the reference)
    if kind in ("decode", "recurrence"):
        return "exact"
    # the matrix-core projections are defined up to the order of their FP32
    # sums: a sum that moves by its last bit can move a BF16 rounding, which
    # each further layer spreads
    # (against the sums in 64 bits: 8e-3 and 7e-2 at 2 layers, 1.5e-2 and
    # 7e-2 at 4, 4.3e-2 and 0.26 at 24; about four times that)
    if case["layers"] > 4:
        return {"rel": 0.18, "max": 0.9, "differ": 0.25}
    return {"rel": 0.016 * case["layers"], "max": 0.3, "differ": 0.25}


# -------------------------------------------- the same mathematics in 64 bits

def _bf(x):
    return x.float().bfloat16().double()


def _view(a: np.ndarray, *shape):
    return torch.from_numpy(a.reshape(shape)).cuda().double()


class _Exact:
    """The model on [streams, tokens] of token ids in float64, with the
    contract's rounding points (BF16 after every operator; the single-stream
    BF16 contracts also round every weight product)."""

    def __init__(self, model: g.Model, layers: int, contract: int, products: bool) -> None:
        self.m, self.layers, self.contract, self.products = model, layers, contract, products
        self.eps = float(np.float32(1e-6))

    def r(self, x):
        return x if self.contract == FP32 else _bf(x)

    def matmul(self, x, w):
        if not self.products:
            return x @ w.T
        rows = x.reshape(-1, x.shape[-1])
        out = torch.empty(rows.shape[0], w.shape[0], dtype=torch.float64, device="cuda")
        for i in range(rows.shape[0]):
            for j in range(0, w.shape[0], 4096):
                out[i, j:j + 4096] = _bf(w[j:j + 4096] * rows[i]).sum(1)
        return out.reshape(*x.shape[:-1], w.shape[0])

    def norm(self, x, w):
        return self.r(x * torch.rsqrt((x * x).mean(-1, keepdim=True) + self.eps) * w)

    def conv(self, raw, w, tails):  # raw [S, T, H], tails [S, 3, H]
        seq = torch.cat([tails, raw], 1)
        t = raw.shape[1]
        s = sum(seq[:, i:i + t] * w[:, i] for i in range(4))
        return self.r(torch.nn.functional.silu(s)), seq[:, t:]

    def recurrence(self, q, k, v, beta, decay, S):
        """q, k, v [S, T, heads, 256]; beta, decay [S, T, heads]; S in place."""
        o = torch.empty_like(v)
        unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + self.eps)  # noqa: E731
        q, k = unit(q), unit(k)
        for t in range(q.shape[1]):
            S *= decay[:, t, :, None, None]
            d = beta[:, t, :, None] * (v[:, t] - torch.einsum("shkv,shk->shv", S, k[:, t]))
            S += k[:, t, :, :, None] * d[:, :, None, :]
            o[:, t] = torch.einsum("shkv,shk->shv", S, q[:, t]) / 16
            if self.contract == REF:
                S.copy_(_bf(S))
        return self.r(o)

    def __call__(self, tokens: np.ndarray, state: Optional[torch.Tensor], tails: Optional[torch.Tensor]):
        """tokens [S, T] -> hidden [S, T, H], state [S, L, 8, 256, 256], tails [S, L, 3, 3, H]."""
        n, T = tokens.shape
        emb = torch.from_numpy(self.m.embeddings.reshape(V, H)[tokens.reshape(-1)]).cuda().double()
        x = self.r(emb.reshape(n, T, H))
        states, all_tails = [], []
        for i in range(self.layers):
            w = self.m.layer(i)
            S = torch.zeros(n, NH, HD, HD, dtype=torch.float64, device="cuda") if state is None else \
                state[:, i].clone()
            tl = torch.zeros(n, 3, 3, H, dtype=torch.float64, device="cuda") if tails is None else tails[:, i]
            xn = self.norm(x, _view(w["attn_norm"], H))
            proj = lambda name, src, rows: self.r(self.matmul(src, _view(w[name], rows, src.shape[-1])))  # noqa: E731
            small = lambda name: self.r(xn @ _view(w[name], NH, H).T)  # noqa: E731
            a, b = small("a_proj"), small("b_proj")
            qkv, new_tails = [], []
            for j, name in enumerate("qkv"):
                y, nt = self.conv(proj(name + "_proj", xn, H), _view(w[name + "_conv"], H, 4), tl[:, j])
                qkv.append(y.reshape(n, T, NH, HD))
                new_tails.append(nt)
            beta = torch.sigmoid(b)
            decay = torch.exp(-torch.exp(_view(w["a_log"], NH)) *
                              torch.nn.functional.softplus(a + _view(w["dt_bias"], NH)))
            o = self.recurrence(*qkv, beta, decay, S)
            gate = proj("g_proj", xn, H).reshape(n, T, NH, HD)
            o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + self.eps) * _view(w["o_norm"], HD)
            o = self.r(o * gate * torch.sigmoid(gate)).reshape(n, T, H)
            x = self.r(x + proj("o_proj", o, H))
            xn = self.norm(x, _view(w["mlp_norm"], H))
            h = self.r(torch.nn.functional.silu(proj("mlp_gate_proj", xn, I)) * proj("mlp_up_proj", xn, I))
            x = self.r(x + proj("mlp_down_proj", h, H))
            states.append(S)
            all_tails.append(torch.stack(new_tails, 1))
        return self.norm(x, _view(self.m.final_norm, H)), torch.stack(states, 1), torch.stack(all_tails, 1)

    def logits(self, hidden):
        return self.matmul(hidden, _view(self.m.lm_head, V, H))


def _np(x):
    return x.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "recurrence":
            q, k, v, a, b, a_log, dt_bias, S = (x.double() for x in _recurrence_inputs(case, seed))
            ex = _Exact(None, 0, case["contract"], False)
            ex.eps = 1e-6
            S = S[None].clone()
            decay = torch.exp(-torch.exp(a_log) * torch.nn.functional.softplus(a + dt_bias))
            o = ex.recurrence(q[None], k[None], v[None], torch.sigmoid(b)[None], decay[None], S)
            return {"out": o[0], "state": S[0]}
        L = case["layers"]
        if kind == "decode":
            tokens, state, tails = _decode_inputs(case, seed)
            ex = _Exact(_model(L, case["contract"] != FP32), L, case["contract"], case["contract"] != FP32)
            hidden, _, _ = ex(tokens[None], _view(state, 1, L, NH, HD, HD), _view(tails, 1, L, 3, 3, H))
            return {"tokens": None, "logits": _np(ex.logits(hidden[0, -1])), "hidden": _np(hidden[0, -1])}
        ex = _Exact(_model(L, True), L, BF16W, False)
        if kind == "streams":
            tokens, state, tails = _streams_inputs(case, seed)
            n = case["streams"]
            if state is not None:
                state, tails = _view(state, n, L, NH, HD, HD), _view(tails, n, L, 3, 3, H)
            hidden, _, _ = ex(np.ascontiguousarray(tokens.T), state, tails)
            return {"tokens": None, "logits": _np(ex.logits(hidden[:, -1]))}
        prompt, tokens = _prefill_inputs(case, seed)
        t = case["tokens"]
        hidden, state, tails = ex(np.concatenate([prompt, tokens.reshape(-1)])[None], None, None)
        out = {"logits": _np(ex.logits(hidden[0, t - 1])), "hidden": _np(hidden[0, t - 1])}
        if case["steps"]:
            out["next_logits"] = _np(ex.logits(hidden[0, -1]))
        else:
            out["state"], out["tails"] = _np(state.reshape(-1)), _np(tails.reshape(-1))
        return out
