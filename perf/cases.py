"""The work that programs have this engine do, as timed cases.

A case is a dict of plain values; `op` says which entry point it calls:

  gemv     one weight matrix times one row of activations: batch-1 decode, layer by layer
  gemm     the same for 1 to 2048 rows: a step of a batch of sequences, or a pass over a prompt
  step     the gated delta rule, one token for each of 1 to 64 sequences
  chunk    the gated delta rule over the tokens of a prompt
  attn     paged attention of one new token for each of 1 to 64 sequences
  prefill  a whole model over a prompt, up to the last token's logits
  decode   a whole model's greedy decode after a prompt
  batch    steps of a batch of sequences of a whole model, each after its own prompt

Kernel calls go to one stream of the caller's own (the library keeps one scratch area per device for
them), whole-model calls to the model's. `exact` computes each result from the definitions in 64 bits.
"""
import json
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "qwen-native-engine_amd"))
import qne  # noqa: E402
import weights  # noqa: E402

DEV = torch.device("cuda" if torch.cuda.is_available() else "cpu")
EPS = 1e-6
HD, BLOCK, DK = 256, 16, 128  # attention head, cache block, delta-rule head
STORE, ACCUMULATE, SWIGLU = "store", "accumulate", "swiglu"
EPILOGUE = {STORE: qne.EPI_STORE, ACCUMULATE: qne.EPI_ACCUMULATE, SWIGLU: qne.EPI_SWIGLU}
GEMV_K = (512, 1024, 2048, 3072, 3584, 4096, 6144)  # the widths that gemv takes

# The hybrid decoders of weights.CONFIGS as they are deployed: int4 body with f16 embedding and head,
# or f16 throughout.
MODELS = {"small": "q4", "0.8b": "f16", "2b": "q4"}


def listed():
    return [
        # The smallest matrix of a 2B decode step (the mixers' out-projection): launch and latency.
        dict(name="gemv q4 2048x2048", op="gemv", kind="q4", group=64, rows=2048, k=2048, epi=ACCUMULATE, norm=False),
        # A batch of 64 sequences through the widest matrix of a 2B layer.
        dict(name="gemm q4 64 rows gate_up", op="gemm", kind="q4", group=64, m=64, rows=12288, k=2048, epi=SWIGLU, norm=True),
        # The same matrix for a full pass over a prompt.
        dict(name="gemm q4 2048 rows gate_up", op="gemm", kind="q4", group=64, m=2048, rows=12288, k=2048, epi=SWIGLU, norm=True),
        # A short, odd prompt through the narrow, deep matrix of the layer.
        dict(name="gemm q4 333 rows down", op="gemm", kind="q4", group=64, m=333, rows=2048, k=6144, epi=ACCUMULATE, norm=False),
        # The 0.8B model's f16 weights and its 128-token prompt.
        dict(name="gemm f16 128 rows gate_up", op="gemm", kind="f16", group=0, m=128, rows=7168, k=1024, epi=SWIGLU, norm=True),
        # One token for 64 sequences.
        dict(name="step 64", op="step", batch=64, heads=16),
        # Four prompts of 2048 tokens, and a single odd one.
        dict(name="chunk 4x2048", op="chunk", batch=4, tokens=2048, heads=16),
        dict(name="chunk 1x777", op="chunk", batch=1, tokens=777, heads=16),
        # 64 sequences at contexts between 256 and 4096.
        dict(name="attn 64", op="attn", batch=64, nq=16, nkv=4, low=256, high=4096),
        # The 2B model over a 4000-id prompt, its greedy decode there, and 64 sequences at once.
        dict(name="prefill 2b 4000", op="prefill", model="2b", tokens=4000),
        dict(name="decode 2b 4000", op="decode", model="2b", tokens=4000, steps=16),
        dict(name="batch 2b 64", op="batch", model="2b", rows=64, low=256, high=3500, steps=4),
    ]


def _log_int(rng, low, high):
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def draw(rng):
    op = rng.choice(["gemv", "gemm", "gemm", "gemm", "step", "chunk", "chunk", "attn", "prefill", "prefill", "decode", "batch"])
    if op in ("gemv", "gemm"):
        kind = rng.choice(["q4", "q4", "f16"])
        epi = rng.choice([STORE, ACCUMULATE, SWIGLU])
        rows = _log_int(rng, 64, 12288)
        if op == "gemv":
            k = rng.choice(GEMV_K)
            group = rng.choice([32, 64, 128])
        else:
            group = rng.choice([64, 64, 128])
            k = group * _log_int(rng, 512 // group, 6144 // group)
        case = dict(op=op, kind=kind, group=group if kind == "q4" else 0, rows=rows + (rows % 2 if epi == SWIGLU else 0), k=k,
                    epi=epi, norm=rng.random() < 0.5)
        return dict(case, m=_log_int(rng, 1, 2048)) if op == "gemm" else case
    if op == "step":
        return dict(op=op, batch=_log_int(rng, 1, 64), heads=rng.choice([4, 16, 16]))
    if op == "chunk":
        return dict(op=op, batch=_log_int(rng, 1, 4), tokens=_log_int(rng, 16, 2048), heads=rng.choice([4, 16, 16]))
    if op == "attn":
        nq, nkv = rng.choice([(16, 4), (8, 2), (2, 1)])
        high = _log_int(rng, 64, 4096)
        return dict(op=op, batch=_log_int(rng, 1, 64), nq=nq, nkv=nkv, low=max(1, high // 16), high=high)
    model = rng.choice(list(MODELS))
    if op == "prefill":
        return dict(op=op, model=model, tokens=_log_int(rng, 16, 3999))
    if op == "decode":
        return dict(op=op, model=model, tokens=_log_int(rng, 16, 3999), steps=rng.choice([4, 8, 16]))
    high = _log_int(rng, 64, 2000)
    return dict(op=op, model=model, rows=_log_int(rng, 1, 63), low=max(1, high // 8), high=high, steps=rng.choice([2, 4]))


# ---- inputs -------------------------------------------------------------------------------------


def _rng(seed, name=""):
    """A generator for one named input: the same values whoever asks, whatever was drawn before."""
    h = 0xCBF29CE484222325
    for b in f"{seed}/{name}".encode():
        h = ((h ^ b) * 0x100000001B3) % (1 << 64)
    return torch.Generator(DEV).manual_seed(h >> 1)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _matrix(g, kind, rows, k, group):
    """N(0, 0.02) weights in the encoding: f16, or int4 codes with f16 scale and zero per group, w = s (q - z)."""
    w = _normal(g, rows, k) * 0.02
    if kind == "f16":
        return dict(w=w.half())
    w = w.view(rows, k // group, group)
    low, high = w.amin(2, keepdim=True), w.amax(2, keepdim=True)
    s = ((high - low) / 15).half()
    z = (-low / s.float()).half()
    q = (w / s.float() + z.float()).round().clamp(0, 15).to(torch.uint8).view(rows, k)
    return dict(q=q, s=s.view(rows, -1), z=z.view(rows, -1))


def _packed(mat):
    """An int4 matrix's codes two to a byte (column 2 j in the low half)."""
    return mat["q"][:, 0::2] | (mat["q"][:, 1::2] << 4)


def _dense(mat, rows=slice(None)):
    """A matrix's values in 64 bits."""
    if "w" in mat:
        return mat["w"][rows].double()
    q, s, z = mat["q"][rows], mat["s"][rows].double(), mat["z"][rows].double()
    group = q.shape[1] // s.shape[1]
    return ((q.double().view(*s.shape, group) - z[..., None]) * s[..., None]).view(q.shape)


def _matmul_inputs(case, seed):
    """Activations as the layers see them: a residual stream with channels of different size under
    its norm's gain, or gated activations."""
    g = _rng(seed)
    m, k, rows = case.get("m", 1), case["k"], case["rows"]
    if case["norm"]:
        x = _normal(g, m, k) * torch.exp(0.5 * _normal(g, k))
        gain = 1 + 0.1 * _normal(g, k)
    else:
        x, gain = torch.nn.functional.silu(_normal(g, m, k)) * _normal(g, m, k), None
    y = _normal(g, m, rows // 2 if case["epi"] == SWIGLU else rows)
    return x, gain, _matrix(g, case["kind"], rows, k, case["group"]), y


def _delta_inputs(case, seed):
    g = _rng(seed)
    b, t, h = case["batch"], case.get("tokens", 1), case["heads"]
    q, k = (torch.nn.functional.normalize(_normal(g, b, t, h, DK), dim=-1) for _ in range(2))
    v = _normal(g, b, t, h, DK)
    beta = torch.sigmoid(_normal(g, b, t, h))
    decay = torch.exp(-torch.nn.functional.softplus(_normal(g, b, t, h)))
    return q, k, v, beta, decay, 0.1 * _normal(g, b, h, DK, DK)


def _attn_inputs(case, seed):
    g = _rng(seed)
    b, nq, nkv = case["batch"], case["nq"], case["nkv"]
    blocks = case["high"] // BLOCK + 1
    ctx = torch.randint(case["low"], case["high"], (b,), generator=g, device=DEV, dtype=torch.int32)
    table = torch.randperm(b * blocks, generator=g, device=DEV).to(torch.int32).view(b, blocks)
    pools = [_normal(g, b * blocks, nkv, BLOCK, HD).half() for _ in range(2)]
    return _normal(g, b, nq, HD), _normal(g, b, nkv, HD), _normal(g, b, nkv, HD), pools[0], pools[1], table, ctx


def _config(case):
    return weights.full_config(case["model"])


def _model_matrix(cfg, name, kind, seed):
    rows, k = weights.matrix_shapes(cfg)[name]
    return _matrix(_rng(seed, name), "f16" if name in ("embed", "lm_head") else kind, rows, k, 64)


def _model_vector(cfg, name, seed):
    n = weights.vector_shapes(cfg)[name]
    if name.endswith("conv_w"):
        return _normal(_rng(seed, name), n) * 0.02
    if name.endswith("gdn_params"):
        heads = cfg["gdn_heads"]
        return torch.cat([torch.zeros(heads), torch.full((heads,), -0.5), torch.ones(n - 2 * heads)]).to(DEV)
    return 1 + 0.1 * _normal(_rng(seed, name), n)


def _load(case, seed):
    """The model in the file format, loaded."""
    cfg, kind = _config(case), MODELS[case["model"]]
    layout, mats = weights.plan(cfg, body=kind)
    image = torch.zeros(layout.size, dtype=torch.uint8, device=DEV)

    def put(name, t):
        raw = t.contiguous().view(-1).view(torch.uint8)
        at = layout.tensors[name]["offset"]
        image[at:at + raw.numel()] = raw

    for name in mats:
        mat = _model_matrix(cfg, name, kind, seed)
        put(name + ".w", mat["w"] if "w" in mat else _packed(mat))
        if "s" in mat:
            put(name + ".s", mat["s"])
            put(name + ".z", mat["z"])
    for name in weights.vector_shapes(cfg):
        put(name, _model_vector(cfg, name, seed))
    host = image.cpu().numpy()
    del image
    torch.cuda.empty_cache()
    return qne.Model.load(weights.index_json(cfg, layout, mats, f"random, seed {seed}"), host)


def _prompts(case, seed):
    rng = np.random.default_rng(seed)
    vocab = _config(case)["vocab"]
    if case["op"] == "batch":
        return [rng.integers(0, vocab, n) for n in rng.integers(case["low"], case["high"], case["rows"])]
    return [rng.integers(0, vocab, case["tokens"])]


_own_stream = None


def _stream():
    global _own_stream
    if _own_stream is None:
        _own_stream = torch.cuda.Stream()
    return _own_stream.cuda_stream


def prepare(case, seed):
    op = case["op"]
    state = dict(case=case)
    if op in ("gemv", "gemm"):
        x, gain, mat, y = _matmul_inputs(case, seed)
        if "q" in mat:
            w, sz = _packed(mat), torch.stack([mat["s"], mat["z"]], -1).contiguous()
        else:
            w, sz = mat["w"], None
        state.update(x=x, gain=gain, w=w, sz=sz, y=y)
    elif op in ("step", "chunk"):
        state["inputs"] = [t.contiguous() for t in _delta_inputs(case, seed)]
        state["out"] = torch.empty_like(state["inputs"][2])
    elif op == "attn":
        state["inputs"] = _attn_inputs(case, seed)
        state["out"] = torch.empty_like(state["inputs"][0])
    else:
        model = state["model"] = _load(case, seed)
        state["prompts"] = _prompts(case, seed)
        if op == "decode":
            model.prefill_batched(state["prompts"][0][:-1])
            model.snapshot()
        elif op == "batch":
            rng = np.random.default_rng(seed + 1)
            state["tokens"] = rng.integers(0, model.vocab, (case["steps"], case["rows"]))
            state["batch"] = qne.Batch(model, case["rows"], 4096)
            for row, ids in enumerate(state["prompts"]):
                model.reset()
                model.prefill_batched(ids)
                state["batch"].admit(row)
    if op in ("gemv", "gemm", "step", "chunk", "attn"):
        state["stream"] = _stream()
    return state


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "gemv":
        qne.gemv(qne.MAT_Q4 if s["sz"] is not None else qne.MAT_F16, s["w"].data_ptr(), s["sz"].data_ptr() if s["sz"] is not None else 0,
                 case["rows"], case["k"], case["group"], s["x"].data_ptr(), s["y"].data_ptr(), EPILOGUE[case["epi"]],
                 norm=s["gain"].data_ptr() if s["gain"] is not None else 0, eps=EPS, stream=s["stream"])
        return s["y"]
    if op == "gemm":
        qne.gemm(qne.MAT_Q4 if s["sz"] is not None else qne.MAT_F16, s["w"].data_ptr(), s["sz"].data_ptr() if s["sz"] is not None else 0,
                 case["rows"], case["k"], case["group"], s["x"].data_ptr(), case["k"], case["m"], s["y"].data_ptr(),
                 s["y"].shape[1], EPILOGUE[case["epi"]], norm=s["gain"].data_ptr() if s["gain"] is not None else 0, eps=EPS,
                 stream=s["stream"])
        return s["y"]
    if op == "step":
        qne.gdn_step(*[t.data_ptr() for t in s["inputs"]], s["out"].data_ptr(), case["batch"], case["heads"], stream=s["stream"])
        return [s["out"], s["inputs"][5]]
    if op == "chunk":
        qne.gdn_prefill_chunked(*[t.data_ptr() for t in s["inputs"]], s["out"].data_ptr(), case["batch"], case["tokens"],
                                case["heads"], stream=s["stream"])
        return [s["out"], s["inputs"][5]]
    if op == "attn":
        q, k, v, kp, vp, table, ctx = s["inputs"]
        qne.paged_attn_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), kp.data_ptr(), vp.data_ptr(), table.data_ptr(),
                              table.shape[1], ctx.data_ptr(), s["out"].data_ptr(), case["batch"], case["nq"], case["nkv"],
                              stream=s["stream"])
        return s["out"]
    model = s["model"]
    if op == "prefill":  # a new conversation's prompt
        model.reset()
        model.prefill_batched(s["prompts"][0])
        return model.logits()
    if op == "decode":  # an answer after a saved prompt and one id more, then the logits of the step after it
        model.restore()
        model.prefill_from(s["prompts"][0][-1:], case["tokens"] - 1)
        ids = model.decode_ids(case["steps"] + 1, case["steps"])
        return [np.array(ids), model.step(*model.last_token())]
    for tokens in s["tokens"][:-1]:
        s["batch"].step(case["rows"], tokens)
    return s["batch"].step(case["rows"], s["tokens"][-1], logits=True)[1]


# ---- what a pass needs --------------------------------------------------------------------------


def _matrix_bytes(kind, rows, k, group):
    return rows * k * 2 if kind == "f16" else rows * k // 2 + rows * (k // group) * 4


def _model_work(case, tokens, positions, heads_of):
    """`tokens` rows through the layers in one go, attending `positions` in all; logits of `heads_of` rows."""
    cfg, kind = _config(case), MODELS[case["model"]]
    nbytes = flops = 0
    for name, (rows, k) in weights.matrix_shapes(cfg).items():
        if name == "embed":
            nbytes += tokens * k * 2
            continue
        head = name == "lm_head"
        nbytes += _matrix_bytes("f16" if head else kind, rows, k, 64)
        flops += 2 * rows * k * (heads_of if head else tokens)
    attn = sum(weights.is_attn(cfg, i) for i in range(cfg["layers"]))
    flops += attn * positions * cfg["n_q_heads"] * HD * 4
    flops += (cfg["layers"] - attn) * tokens * cfg["gdn_heads"] * 6 * DK * DK
    return nbytes, flops, attn * cfg["n_kv_heads"] * HD * 4, (cfg["layers"] - attn) * cfg["gdn_heads"] * DK * DK * 8


def work(case):
    op = case["op"]
    if op in ("gemv", "gemm"):
        m, rows, k = case.get("m", 1), case["rows"], case["k"]
        out = rows // 2 if case["epi"] == SWIGLU else rows
        return dict(bytes=_matrix_bytes(case["kind"], rows, k, case["group"]) + 4 * m * (k + out * (2 if case["epi"] == ACCUMULATE else 1)),
                    flops=2 * m * rows * k)
    if op in ("step", "chunk"):
        b, t, h = case["batch"], case.get("tokens", 1), case["heads"]
        return dict(bytes=b * h * (2 * 4 * DK * DK + t * (4 * 4 * DK + 8)), flops=b * h * t * 6 * DK * DK)
    if op == "attn":
        b, n = case["batch"], case["batch"] * ((case["low"] + case["high"]) // 2 + 1)
        return dict(bytes=n * case["nkv"] * HD * 4 + b * (2 * case["nq"] + 2 * case["nkv"]) * HD * 4, flops=4 * n * case["nq"] * HD)
    vocab = _config(case)["vocab"]
    if op == "prefill":
        t = case["tokens"]
        nbytes, flops, kv, state = _model_work(case, t, t * (t + 1) // 2, 1)
        return dict(bytes=nbytes + t * kv + state // 2 + vocab * 4, flops=flops)
    if op == "decode":
        t, n = case["tokens"], case["steps"] + 1
        nbytes, flops, kv, state = _model_work(case, 1, t, 1)
        return dict(bytes=n * (nbytes + t * kv + state) + vocab * 4, flops=n * flops)
    r, n, mean = case["rows"], case["steps"], (case["low"] + case["high"]) // 2
    nbytes, flops, kv, state = _model_work(case, r, r * mean, r)
    return dict(bytes=n * (nbytes + r * mean * kv + r * state) + r * vocab * 4, flops=n * flops)


def tolerance(case):
    """About four times the 2-norm errors against 64 bits that were measured: 4e-7 for one layer's
    products and attention, 1.9e-6 for the delta rule over a prompt, 5e-5 for a model's logits."""
    if case["op"] in ("gemv", "gemm", "step", "attn"):
        return dict(rel=2e-6)
    return dict(rel=8e-6) if case["op"] == "chunk" else dict(rel=2e-4)


# ---- the same in 64 bits ------------------------------------------------------------------------


def _rms(x, gain):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gain


def _silu(x):
    return x * torch.sigmoid(x)


def _delta_rule(q, k, v, beta, decay, state):
    """Token by token; q, k, v [T][...][dk], beta and decay [T][...], state [...][dk][dv]."""
    out = []
    for t in range(q.shape[0]):
        held = decay[t][..., None] * (state * k[t][..., None]).sum(-2)
        d = beta[t][..., None] * (v[t] - held)
        state = decay[t][..., None, None] * state + k[t][..., None] * d[..., None, :]
        out.append((state * q[t][..., None]).sum(-2))
    return torch.stack(out), state


def _attend(q, k, v, first):
    """q [T][nq][hd] at positions first.., k and v [L][nkv][hd]: causal softmax attention."""
    group, out = q.shape[1] // k.shape[1], []
    allowed = torch.arange(k.shape[0], device=DEV)[None, :] <= first + torch.arange(q.shape[0], device=DEV)[:, None]
    for h in range(q.shape[1]):
        scores = (q[:, h] @ k[:, h // group].T.contiguous()) / math.sqrt(HD)
        out.append(torch.softmax(scores.masked_fill(~allowed, -math.inf), -1) @ v[:, h // group])
    return torch.stack(out, 1)


class _Exact:
    """The hybrid decoder in 64 bits, with its cache in f16 as the format has it."""

    def __init__(self, case, seed):
        self.cfg, self.kind, self.seed = _config(case), MODELS[case["model"]], seed
        self.cache, self.length = {}, 0

    def _mul(self, x, name):
        return x @ _dense(_model_matrix(self.cfg, name, self.kind, self.seed)).T.contiguous()

    def _vec(self, name):
        return _model_vector(self.cfg, name, self.seed).double()

    def _rope(self, x):
        rot = self.cfg["rope_dim"]
        freq = torch.tensor([self.cfg["rope_theta"] ** (-2 * i / rot) for i in range(rot // 2)], dtype=torch.float32, device=DEV)
        at = torch.arange(self.length, self.length + x.shape[0], device=DEV).float()
        angle = (at[:, None] * freq).double()[:, None]
        a, b = x[..., :rot // 2], x[..., rot // 2:rot]
        return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin(), x[..., rot:]], -1)

    def _attention(self, i, p):
        c, t = self.cfg, p.shape[0]
        nq, nkv = c["n_q_heads"], c["n_kv_heads"]
        q, gate, k, v = p.split([nq * HD, nq * HD, nkv * HD, nkv * HD], 1)
        norms = self._vec(f"layer{i}.attn_norms")
        q = self._rope(_rms(q.reshape(t, nq, HD), norms[:HD]))
        k = self._rope(_rms(k.reshape(t, nkv, HD), norms[HD:])).half().double()
        v = v.reshape(t, nkv, HD).half().double()
        if i in self.cache:
            k, v = torch.cat([self.cache[i][0], k]), torch.cat([self.cache[i][1], v])
        self.cache[i] = (k, v)
        return _attend(q, k, v, self.length).reshape(t, -1) * torch.sigmoid(gate)

    def _delta(self, i, p):
        c, t, h = self.cfg, p.shape[0], self.cfg["gdn_heads"]
        w = h * DK
        mixed, z, a, b = p.split([3 * w, w, h, h], 1)
        past, state = self.cache.get(i, (mixed.new_zeros(3, 3 * w), mixed.new_zeros(h, DK, DK)))
        line = torch.cat([past, mixed])
        taps = self._vec(f"layer{i}.conv_w").view(3 * w, 4)
        mixed = _silu(sum(line[j:j + t] * taps[:, j] for j in range(4)))
        q, k, v = (x.reshape(t, h, DK) for x in mixed.split(w, 1))
        q, k = (x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        prm = self._vec(f"layer{i}.gdn_params")
        decay = torch.exp(prm[h:2 * h] * torch.nn.functional.softplus(a + prm[:h]))
        out, state = _delta_rule(q / math.sqrt(DK), k, v, torch.sigmoid(b), decay, state)
        self.cache[i] = (line[t:], state)
        return (_rms(out, prm[2 * h:]) * _silu(z.reshape(t, h, DK))).reshape(t, -1)

    def __call__(self, ids):
        """The last id's logits, after all that came before."""
        c = self.cfg
        x = _dense(_model_matrix(c, "embed", self.kind, self.seed), torch.as_tensor(ids, dtype=torch.long, device=DEV))
        for i in range(c["layers"]):
            p = self._mul(_rms(x, self._vec(f"layer{i}.input_norm")), f"layer{i}.mixer_in")
            o = self._attention(i, p) if weights.is_attn(c, i) else self._delta(i, p)
            x = x + self._mul(o, f"layer{i}.mixer_out")
            u = self._mul(_rms(x, self._vec(f"layer{i}.post_norm")), f"layer{i}.gate_up")
            half = u.shape[1] // 2
            x = x + self._mul(_silu(u[:, :half]) * u[:, half:], f"layer{i}.down")
        self.length += len(ids)
        return self._mul(_rms(x[-1:], self._vec("final_norm")), "lm_head")[0]


def exact(case, seed):
    op = case["op"]
    if op in ("gemv", "gemm"):
        x, gain, mat, y = _matmul_inputs(case, seed)
        x = x.double()
        p = (_rms(x, gain.double()) if gain is not None else x) @ _dense(mat).T.contiguous()
        if case["epi"] == SWIGLU:
            half = p.shape[1] // 2
            return _silu(p[:, :half]) * p[:, half:]
        return p + y.double() if case["epi"] == ACCUMULATE else p
    if op in ("step", "chunk"):
        q, k, v, beta, decay, state = (t.double() for t in _delta_inputs(case, seed))
        out, state = _delta_rule(*(t.transpose(0, 1) for t in (q, k, v, beta, decay)), state)
        return [out.transpose(0, 1), state]
    if op == "attn":
        q, k_new, v_new, kp, vp, table, ctx = _attn_inputs(case, seed)
        out = []
        for b, n in enumerate(ctx.tolist()):
            at = torch.arange(n, device=DEV)
            block, slot = table[b].long()[at // BLOCK], at % BLOCK
            k, v = (torch.cat([pool[block, :, slot], new[b:b + 1].half()]).double() for pool, new in ((kp, k_new), (vp, v_new)))
            out.append(_attend(q[b:b + 1].double(), k, v, n)[0])
        return torch.stack(out)
    if op == "prefill":
        return _Exact(case, seed)(_prompts(case, seed)[0])
    if op == "decode":
        model = _Exact(case, seed)
        logits = model(_prompts(case, seed)[0])
        for _ in range(case["steps"] + 1):
            logits = model([int(logits.argmax())])
        return [None, logits]
    return None  # dozens of whole prompts: minutes
