"""The work a program built on this package has it do, as measurable cases: batch-1 fp16 products in both operand orders,
sibling products in one launch, the input projection, LSTM encoders and per-token cells, the attention decoder's step, a
mixture-of-experts block and a transducer's greedy decoding.  Every case goes through the package's public entry points.

    listed()               the cases, each a dict of plain values
    draw(rng)              one more case of the same ranges
    prepare(case, seed)    what a program holds before the call: operands, and the plan it made when it loaded its model
    run(state)             one pass, and its outputs
    work(case)             bytes and floating-point operations one pass cannot do without
    tolerance(case)        how far another correct implementation at the same precision may be off
"""
import math

import torch

import pimaicompiler_amd as P

DEVICE = "cuda"


def listed():
    return [
        # One 1024 x 1024 layer of an interpreted graph: the smallest product of the benchmark configurations, where the call
        # and the launch are the cost.
        {"name": "addmm_1024", "kind": "gemv", "op": "addmm_w_x", "out": 1024, "in": 1024, "bias": True, "relu": False},
        # The last layer of a transducer's joint network (512 features, 29 symbols) as an addmm whose weight lies [in, out], as a
        # graph holds it that no rewrite has touched.
        {"name": "addmm_joint_out", "kind": "gemv", "op": "addmm_x_w", "out": 29, "in": 512, "bias": True, "relu": False},
        # A vocabulary projection of a size that is a multiple of nothing, weight [in, out].
        {"name": "matmul_odd_vocab", "kind": "gemv", "op": "matmul_x_w", "out": 31999, "in": 1024, "bias": False, "relu": False},
        # The widest feed-forward layer of the benchmark's sweep, with its activation: the stream of a matrix far larger than
        # the caches.
        {"name": "linear_16384x4096", "kind": "gemv", "op": "linear", "out": 16384, "in": 4096, "bias": True, "relu": True},
        # A mixture-of-experts block (8 experts, 768 -> 3072 -> 768) over the 13 tokens of a short sentence, one after another.
        {"name": "moe_13_tokens", "kind": "moe", "E": 8, "d_model": 768, "d_ff": 3072, "tokens": 13},
        # q, k, v and o of one attention layer (768 wide): sibling products of one input, issued as one group.
        {"name": "group_qkvo_768", "kind": "group", "count": 4, "out": 768, "in": 768, "bias": False},
        # The gate rows of a layer for a whole utterance (800 frames), the one dense contraction of the path.
        {"name": "projection_800", "kind": "projection", "T": 800, "in": 1024, "out": 4096, "packed": False},
        # The speech encoder: two layers of 1024 over 240 features, an utterance of 341 frames.
        {"name": "lstm_speech_341", "kind": "lstm", "I": 240, "H": 1024, "L": 2, "bidir": False, "T": 341, "first_res": -1},
        # The translation encoder: its bidirectional first layer over a sentence of 50 words.
        {"name": "lstm_bidir_50", "kind": "lstm", "I": 1024, "H": 1024, "L": 1, "bidir": True, "T": 50, "first_res": -1},
        # One cell of a decoding loop, called once a token with the attention context beside the word (2048 wide).
        {"name": "lstm_token", "kind": "lstm", "I": 2048, "H": 1024, "L": 1, "bidir": False, "T": 1, "first_res": -1},
        # The translation decoder: encoder outputs of a 12-word sentence projected once, then 16 steps of four layers with
        # attention, residual sums and the 32000-word classifier.
        {"name": "decoder_sentence", "kind": "decoder", "H": 1024, "L": 4, "S": 12, "vocab": 32000, "steps": 16},
        # The transducer's decoding of an utterance of 341 frames, mostly blanks.
        {"name": "greedy_341", "kind": "greedy", "L": 2, "H": 320, "F": 1024, "J": 512, "V": 29, "T": 341},
    ]


# ---------------------------------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------------------------------
def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / multiple)) * multiple))


def _most(kind):
    """The arithmetic of the largest listed case of a kind: drawn ones stay below it."""
    return max(work(c)["flops"] for c in listed() if c["kind"] == kind)


def _draw_gemv(rng):
    case = {"kind": "gemv", "op": rng.choice(["addmm_w_x", "addmm_x_w", "matmul_x_w", "linear"]), "out": 0, "in": 0,
            "bias": True, "relu": rng.random() < 0.5}
    step_out = rng.choice([1, 8])   # half of the sizes are multiples of eight, half are what they are
    step_in = rng.choice([1, 8])
    case["out"] = _log_int(rng, 16, 32768, step_out)
    case["in"] = _log_int(rng, 16, min(16384, (1 << 26) // case["out"]), step_in)
    if case["op"] == "matmul_x_w":
        case["bias"] = case["relu"] = False
    return case


def _draw_group(rng):
    return {"kind": "group", "count": rng.randint(2, 8), "out": _log_int(rng, 64, 3072), "in": _log_int(rng, 64, 3072, 8),
            "bias": rng.random() < 0.5}


def _draw_projection(rng):
    case = {"kind": "projection", "T": _log_int(rng, 8, 2048), "in": _log_int(rng, 64, 2048, 8), "out": 4 * _log_int(rng, 64, 1024, 8),
            "packed": rng.random() < 0.5}
    case["T"] = max(8, min(case["T"], (800 * 1024 * 4096) // (case["in"] * case["out"])))
    return case


def _draw_lstm(rng):
    bidir = rng.random() < 0.35
    L = rng.randint(1, 2 if bidir else 4)
    H = _log_int(rng, 64, 2048, 8)
    T = 1 if rng.random() < 0.3 else _log_int(rng, 2, 400)
    case = {"kind": "lstm", "I": _log_int(rng, 40, 2048, 8), "H": H, "L": L, "bidir": bidir, "T": T, "first_res": -1}
    if L >= 2 and not bidir and rng.random() < 0.3:
        case["first_res"] = 1
    # no more arithmetic than the speech encoder
    per_step = work(dict(case, T=1))["flops"]
    case["T"] = max(1, min(T, int(_most("lstm") // per_step)))
    return case


def _draw_decoder(rng):
    return {"kind": "decoder", "H": _log_int(rng, 256, 1024, 8), "L": rng.randint(2, 4), "S": _log_int(rng, 3, 128),
            "vocab": _log_int(rng, 1000, 32000), "steps": rng.randint(2, 16)}


def _draw_moe(rng):
    return {"kind": "moe", "E": rng.choice([2, 4, 8, 8, 16, 32]), "d_model": _log_int(rng, 256, 1024, 8),
            "d_ff": _log_int(rng, 512, 4096, 8), "tokens": rng.randint(1, 26)}


def _draw_greedy(rng):
    L = rng.randint(1, 2)
    H = _log_int(rng, 128, 512, 8)
    J = _log_int(rng, 256, 640, 8)
    V = _log_int(rng, 29, min(768, 8 * (250 - (L * H + J) // 8)))
    case = {"kind": "greedy", "L": L, "H": H, "F": _log_int(rng, 256, 1024, 8), "J": J, "V": V, "T": _log_int(rng, 30, 341)}
    per_frame = work(dict(case, T=1))["flops"]
    case["T"] = max(8, min(case["T"], int(_most("greedy") // per_frame)))
    return case


def draw(rng):
    pick = rng.choice([_draw_gemv] * 4 + [_draw_lstm] * 4 + [_draw_group, _draw_projection, _draw_decoder, _draw_moe, _draw_greedy])
    return pick(rng)


# ---------------------------------------------------------------------------------------------------
# inputs and plans
# ---------------------------------------------------------------------------------------------------
class _Source:
    """Random fp16 tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape, scale=1.0):
        return (torch.randn(*shape, generator=self.g, device=DEVICE) * scale).half()

    def uniform(self, *shape, scale=1.0):
        return ((2 * torch.rand(*shape, generator=self.g, device=DEVICE) - 1) * scale).half()

    def lstm(self, in_w, H, L, D):
        k, params = 1.0 / math.sqrt(H), []
        for l in range(L):
            for _ in range(D):
                w = in_w if l == 0 else D * H
                params += [self.uniform(4 * H, w, scale=k), self.uniform(4 * H, H, scale=k), self.uniform(4 * H, scale=k),
                           self.uniform(4 * H, scale=k)]
        return params


def _prepare_gemv(c, r):
    # (a trained layer's weights: small and centred; larger matrices have smaller ones, so that outputs keep their size)
    scale = min(0.02, 1.0 / math.sqrt(c["in"]))
    w = r.normal(c["out"], c["in"], scale=scale) if c["op"] in ("addmm_w_x", "linear") else r.normal(c["in"], c["out"], scale=scale)
    b = r.normal(c["out"], scale=0.01) if c["bias"] else None
    x = r.uniform(1, c["in"])
    return {"w": w, "b": b, "x": x.t() if c["op"] == "addmm_w_x" else x, "act": "aten::relu" if c["relu"] else "none"}


def _prepare_group(c, r):
    x = r.uniform(1, c["in"])
    n = c["count"]
    return {"x": [x] * n, "w": [r.normal(c["out"], c["in"], scale=0.02) for _ in range(n)],
            "b": [r.normal(c["out"], scale=0.01) for _ in range(n)] if c["bias"] else None}


def _prepare_projection(c, r):
    w = r.uniform(c["out"], c["in"], scale=1.0 / math.sqrt(c["out"] // 4))
    s = {"x": r.normal(c["T"], c["in"]), "w": w, "b": r.uniform(c["out"]).float(), "out": c["out"], "packed": None}
    if c["packed"]:
        s["packed"] = P.pack_projection_weight(w)   # once per weight, when the model is loaded
    return s


def _prepare_lstm(c, r):
    D = 2 if c["bidir"] else 1
    params = r.lstm(c["I"], c["H"], c["L"], D)
    if c["first_res"] >= 0 and c["L"] < 2:
        raise ValueError("a residual sum needs a second layer")
    P.prepare_lstm(params, True, c["L"], c["bidir"], max(c["T"], 16))   # at model load, as the model builder does
    return {"params": params, "x": r.normal(c["T"], 1, c["I"]), "h0": r.uniform(c["L"] * D, 1, c["H"], scale=0.3),
            "c0": r.uniform(c["L"] * D, 1, c["H"], scale=0.3), "first_res": c["first_res"] if c["first_res"] >= 0 else None}


def _prepare_decoder(c, r):
    H, L, S = c["H"], c["L"], c["S"]
    params = []
    for l in range(L):
        params += r.lstm(H if l == 0 else 2 * H, H, 1, 1)
    plan = P.DecoderPlan(params, True, L, first_takes_context=False, first_residual_layer=2,
                         classifier=(r.normal(c["vocab"], H, scale=0.02), r.normal(c["vocab"], scale=0.01)))
    enc = r.normal(S, H)
    att = torch.softmax(r.normal(c["steps"], S).float(), -1).half()
    x = r.normal(c["steps"], H)
    h0, c0 = r.uniform(L, H, scale=0.3), r.uniform(L, H, scale=0.3)
    h, cc = torch.empty_like(h0), torch.empty_like(c0)
    logits = torch.empty(c["steps"], c["vocab"], dtype=torch.float16, device=DEVICE)
    plan.set_encoder(enc)
    steps = []
    for i in range(c["steps"]):   # the first step starts from the encoder's state, the others update the decoder's in place
        steps.append(plan.bind(x[i], list((h0 if i == 0 else h).unbind(0)), list((c0 if i == 0 else cc).unbind(0)), att=att[i],
                               hn=list(h.unbind(0)), cn=list(cc.unbind(0)), logits=logits[i]))
    return {"plan": plan, "enc": enc, "steps": steps, "h": h, "c": cc, "logits": logits, "keep": (att, x, h0, c0)}


def _prepare_moe(c, r):
    E, dm, ff = c["E"], c["d_model"], c["d_ff"]
    plan = P.MoePlan((r.normal(E, dm, scale=0.02), None), [r.normal(ff, dm, scale=0.02) for _ in range(E)],
                     [r.normal(dm, ff, scale=0.02) for _ in range(E)])
    x = r.normal(c["tokens"], dm)
    y = torch.empty_like(x)
    logits = torch.empty(c["tokens"], E, dtype=torch.float16, device=DEVICE)
    expert = torch.empty(c["tokens"], 1, dtype=torch.int32, device=DEVICE)
    steps = [plan.bind(x[i], y[i], logits[i], expert[i]) for i in range(c["tokens"])]
    return {"plan": plan, "steps": steps, "y": y, "logits": logits, "expert": expert, "x": x}


def _prepare_greedy(c, r):
    L, H, F, J, V, T = c["L"], c["H"], c["F"], c["J"], c["V"], c["T"]
    params = r.lstm(H, H, L, 1)
    for l in range(1, L):
        params[4 * l] = (6 * params[4 * l].float()).half()   # (h is small beside an embedding)
    for l in range(L):
        params[4 * l + 2][H:2 * H] -= 2.0                    # the prediction is about the last few symbols
    # Both the frame and the prediction count in the joint network, and no symbol is preferred everywhere.
    w1 = torch.cat([r.normal(J, F, scale=0.9 / math.sqrt(F)), r.normal(J, H, scale=6.0 / math.sqrt(H))], 1)
    w2 = r.normal(V, J, scale=1.0 / math.sqrt(J)).float()
    w2 = (w2 - w2.mean(1, keepdim=True)).half()
    b1, b2 = r.normal(J, scale=0.1), r.normal(V, scale=0.02)
    enc, emb = r.normal(T, F), r.normal(V, H)
    # The blank is the last symbol.  Trained transducers emit a symbol in a fraction of their steps: its bias is set so that it
    # wins in about six steps of seven, going by every frame against a prediction after five symbols.
    w2[V - 1] = 0
    h, cell = [torch.zeros(T, H, device=DEVICE)] * L, [torch.zeros(T, H, device=DEVICE)] * L
    for n in range(5):
        g = emb[(torch.arange(T, device=DEVICE) * (n + 1) + n) % V].float()
        for l in range(L):
            w_ih, w_hh, b_ih, b_hh = (p.float() for p in params[4 * l:4 * l + 4])
            i, f, u, o = (g @ w_ih.t() + h[l] @ w_hh.t() + b_ih + b_hh).chunk(4, 1)
            cell[l] = torch.sigmoid(f) * cell[l] + torch.sigmoid(i) * torch.tanh(u)
            h[l] = g = torch.sigmoid(o) * torch.tanh(cell[l])
    hidden = torch.relu(torch.cat([enc.float(), g], 1) @ w1.float().t() + b1.float())
    best = (hidden @ w2[: V - 1].float().t() + b2[: V - 1].float()).max(1).values
    b2[V - 1] = torch.quantile(best, 0.85).half()
    plan = P.RnntPlan(params, True, L, (w1, b1, w2, b2))
    return {"plan": plan, "enc": enc, "emb": emb, "x0": r.normal(H), "blank": V - 1,
            "most": T * 5}


def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, _Source(seed))
    state["case"] = case
    return state


# ---------------------------------------------------------------------------------------------------
# passes
# ---------------------------------------------------------------------------------------------------
def _run_gemv(s):
    op = s["case"]["op"]
    if op == "addmm_w_x":
        return P.custom_aten_addmm(s["act"], s["b"], s["w"], s["x"])
    if op == "addmm_x_w":
        return P.custom_aten_addmm(s["act"], s["b"], s["x"], s["w"])
    if op == "matmul_x_w":
        return P.custom_aten_matmul(s["x"], s["w"])
    return P.aten_linear(s["x"], s["w"], s["b"], s["act"])


def _run_group(s):
    return P.execute_gemv_group(s["x"], s["w"], s["b"])


def _run_projection(s):
    if s["packed"] is not None:
        return P.input_projection_packed(s["x"], s["packed"], s["out"], s["b"])
    return P.input_projection(s["x"], s["w"], s["b"])


def _run_lstm(s):
    c = s["case"]
    return P.aten_lstm1(s["x"], (s["h0"], s["c0"]), s["params"], True, c["L"], 0.0, False, c["bidir"], False,
                        first_residual_layer=s["first_res"])


def _run_decoder(s):
    s["plan"].set_encoder(s["enc"])
    for step in s["steps"]:
        step()
    return s["logits"], s["h"], s["c"]


def _run_moe(s):
    for step in s["steps"]:
        step()
    return s["y"], s["logits"], s["expert"]


def _run_greedy(s):
    symbols, result, hn, cn = s["plan"].greedy_decode(s["enc"], s["emb"], s["x0"], s["blank"], max_symbols_per_frame=5)
    n = int(result[0])   # the transcript is read here, as every program that decodes does
    return torch.nn.functional.pad(symbols[:n], (0, s["most"] - n), value=-1), result, hn, cn


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


# ---------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------
def _work_gemv(c):
    n, k = c["out"], c["in"]
    return {"bytes": 2 * (n * k + k + n * (2 if c["bias"] else 1)), "flops": 2 * n * k}


def _work_group(c):
    n, k, m = c["out"], c["in"], c["count"]
    return {"bytes": 2 * (m * n * k + k + m * n * (2 if c["bias"] else 1)), "flops": 2 * m * n * k}


def _work_projection(c):
    T, K, N = c["T"], c["in"], c["out"]
    return {"bytes": 2 * (T * K + N * K) + 4 * (T * N + N), "flops": 2 * T * K * N}


def _work_lstm(c):
    H, L, T, D = c["H"], c["L"], c["T"], 2 if c["bidir"] else 1
    weights = D * sum(4 * H * ((c["I"] if l == 0 else D * H) + H) for l in range(L))
    state = 4 * L * D * H
    return {"bytes": 2 * (weights + D * L * 8 * H + T * (c["I"] + D * H) + state), "flops": 2 * T * weights}


def _work_decoder(c):
    H, L, S, V, n = c["H"], c["L"], c["S"], c["vocab"], c["steps"]
    # per step: W_hh and the input columns of W_ih of every layer, the classifier, and the projected context of the upper layers
    # (made once per sentence); what a step reads is read again by the next one.
    ctx = (L - 1) * 4 * H * S
    weights = L * 8 * H * H + V * H
    once = (L - 1) * 4 * H * H
    return {"bytes": n * (2 * weights + 4 * ctx + 2 * V) + 2 * once + 4 * ctx, "flops": n * 2 * (weights + ctx) + 2 * once * S}


def _work_moe(c):
    E, dm, ff, n = c["E"], c["d_model"], c["d_ff"], c["tokens"]
    # (an expert that several tokens choose is read once)
    return {"bytes": 2 * (E * dm + min(E, n) * 2 * dm * ff + n * (2 * dm + E)) + 4 * n, "flops": n * 2 * (E * dm + 2 * dm * ff)}


def _work_greedy(c):
    L, H, F, J, V, T = c["L"], c["H"], c["F"], c["J"], c["V"], c["T"]
    cells = L * 8 * H * H
    joint = J * (F + H) + V * J
    # the joint network once per step (a frame ends with a blank; about one symbol in four frames), the cells once per symbol
    return {"bytes": 2 * (cells + joint + T * F + V * H), "flops": 2 * (T * 5 // 4 * joint + max(1, T // 4) * cells)}


def work(case):
    return globals()["_work_" + case["kind"]](case)


# ---------------------------------------------------------------------------------------------------
# how far correct implementations differ
# ---------------------------------------------------------------------------------------------------
# About four times what the path was measured to differ by from the same arithmetic in 64 bits (relative, largest): products and
# cells 2.2e-4 / 5e-4 and speech encoder 2.5e-4 / 8e-4 (the rounding of fp16 results), decoder 4.4e-4 / 1.9e-3, mixture of
# experts 2.9e-4 / 9e-4 (two roundings in a row), projection 8.3e-8 / 7e-7 at 1024 columns (fp32 sums).
_TOLERANCE = {
    "gemv": {"rel": 9e-4, "max": 2e-3},
    "group": {"rel": 9e-4, "max": 2e-3},
    "projection": {"rel": 6e-7, "max": 5e-6},
    "lstm": {"rel": 1e-3, "max": 3.5e-3},
    "decoder": {"rel": 1.8e-3, "max": 8e-3},
    "moe": {"rel": 1.2e-3, "max": 4e-3},
    "greedy": {"rel": 1e-3, "max": 3.5e-3},
}


def tolerance(case):
    return dict(_TOLERANCE[case["kind"]])
