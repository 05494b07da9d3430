"""The work a user of this framework has it do, as measurable cases.

Two widths of the hybrid family appear throughout: "4b" (hidden 2560, MLP
9728, 16 DeltaNet heads, 16 query / 4 KV heads of 128) and "tiny" (hidden
1024, MLP 3584, 8 DeltaNet heads, 8 query / 2 KV heads of 128). Whole calls
go through `quicklm_amd.engine.Engine` on a few-layer checkpoint of that width
written from the seed; single layers go through the C ABI
(`quicklm_amd.hip.call`), a decode layer as a captured graph that is replayed
(as the engine does), a prefill layer as plain calls.

Kinds of case (`case["kind"]`):
  decode      Engine: `steps` decode steps of `batch` sequences over a known
              token stream (prompt positions forwarded one by one), logits of
              every sequence after the last
  verify      Engine: `rows` drafted tokens checked in one forward at position
              `context` (restore of the snapshot first), every row's logits
  prompt      Engine: a prompt of `rows` tokens prefilled, its first decode
              step, the logits
  mlp_decode / deltanet_decode / attention_decode
              `layers` layers' MLP / DeltaNet mixer / GQA attention for
              `batch` sequences, residual stream in and out
  head        final norm, lm_head and greedy pick of `batch` rows
  mlp_prefill / deltanet_prefill / attention_prefill
              one layer's part over `rows` prompt rows
  attention_cache
              the isolated decode attention over a [B, S, n_kv, hd] cache
"""

from __future__ import annotations

import contextlib
import json
import os
import random
import shutil
import struct
import tempfile

import numpy as np
import torch

from quicklm_amd import hip, synth
from quicklm_amd.engine import Engine

DEV = "cuda" if torch.cuda.is_available() else "cpu"
EPS = 1e-6
F64 = torch.float64
WIDTHS = {"4b": synth.HYBRID_4B, "tiny": synth.TINY}
ENGINE_LAYERS = {"4b": 4, "tiny": 8}  # three DeltaNet layers to each attention layer
ENGINE_VOCAB = 16384  # checkpoints are written anew for every state: the table is cut
ENGINE_KINDS = ("decode", "verify", "prompt")


# ---- the cases ---------------------------------------------------------------


def listed():
    return [
        # The smallest decode: a draft model at int4, one sequence. Its kernels
        # take a few us each, so launches and their gaps are what a user feels.
        dict(name="decode_tiny_int4_b1", kind="decode", width="tiny", precision="int4", batch=1,
             steps=48),
        # One chat: int8 (the reference's Q8_0), one sequence, the headline.
        dict(name="decode_4b_int8_b1", kind="decode", width="4b", precision="int8", batch=1,
             steps=32),
        # Speculative decoding's verify pass: four drafted tokens and the last
        # accepted one, in the middle of a chat.
        dict(name="verify_4b_int8_5", kind="verify", width="4b", precision="int8", rows=5,
             context=600),
        # Time to the first token of a long prompt.
        dict(name="prompt_4b_int8_2048", kind="prompt", width="4b", precision="int8", rows=2048),
        # A serving batch of 16, layer by layer: MLP,
        dict(name="mlp_4b_int8_b16", kind="mlp_decode", width="4b", precision="int8", batch=16,
             layers=2),
        # DeltaNet mixers (three in a row, as between two attention layers),
        dict(name="deltanet_4b_int8_b16", kind="deltanet_decode", width="4b", precision="int8",
             batch=16, layers=3),
        # attention with every sequence at a position of its own up to 2047,
        dict(name="attention_4b_int8_b16_2k", kind="attention_decode", width="4b",
             precision="int8", batch=16, layers=1, context=2048),
        # and the logits of the full vocabulary, here with one scale a row.
        dict(name="head_4b_int8row_b16", kind="head", width="4b", precision="int8_row", batch=16,
             vocab=151936),
        # A short, odd-sized prompt at the default precision (weights as stored).
        dict(name="mlp_4b_bf16_rows511", kind="mlp_prefill", width="4b", precision="bf16",
             rows=511),
        # A long prompt's layers: the DeltaNet mixer with its projections,
        dict(name="deltanet_4b_int8_rows2047", kind="deltanet_prefill", width="4b",
             precision="int8", rows=2047),
        # and the attention of a prompt's second pass (keys of the first before it).
        dict(name="attention_4b_int8_rows2048_at2048", kind="attention_prefill", width="4b",
             precision="int8", rows=2048, first=2048),
        # Long-context decode over a bf16 cache: a caller with a cache of its own.
        dict(name="attention_cache_bf16_b4_32k", kind="attention_cache", kv="bf16", n_q=16,
             n_kv=2, hd=256, batch=4, context=32768),
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["decode", "verify", "prompt", "mlp_decode", "deltanet_decode",
                       "attention_decode", "head", "mlp_prefill", "deltanet_prefill",
                       "attention_prefill", "attention_cache"])
    width = rng.choice(["4b", "tiny"])
    some = rng.choice(["int8", "int8", "int8_row", "int4", "bf16"])  # what the engine loads
    scales = rng.choice(["int8", "int8", "int8_row", "bf16"])
    c = dict(kind=kind, width=width, precision=some)
    if kind == "decode":
        c.update(batch=rng.choice([1, 1, rng.randint(2, 16)]), steps=rng.randint(16, 48))
    elif kind == "verify":
        c.update(rows=rng.randint(2, 9), context=_log(rng, 30, 1500))
    elif kind == "prompt":
        c.update(rows=_log(rng, 18, 2048))
    elif kind == "mlp_decode":
        c.update(precision="int8", batch=rng.randint(1, 16), layers=rng.randint(1, 2))
    elif kind == "deltanet_decode":
        c.update(precision="int8", batch=rng.randint(2, 16), layers=rng.randint(1, 3))
    elif kind == "attention_decode":
        c.update(precision="int8", batch=rng.randint(1, 16), layers=1,
                 context=_log(rng, 64, 2048))
    elif kind == "head":
        c.update(precision=rng.choice(["int8", "int8_row"]), batch=rng.randint(2, 64),
                 vocab=_log(rng, 8192, 151936))
    elif kind == "mlp_prefill":
        c.update(precision=scales, rows=_log(rng, 17, 2048))
    elif kind == "deltanet_prefill":
        c.update(precision=scales, rows=_log(rng, 65, 2047))
    elif kind == "attention_prefill":
        rows = _log(rng, 17, 2048)
        c.update(precision=scales, rows=rows, first=rng.choice([0, rng.randint(1, 4096 - rows)]))
    else:
        c = dict(kind=kind, kv=rng.choice(["bf16", "f32"]))
        c["n_q"], c["n_kv"], c["hd"] = rng.choice([(16, 2, 256), (16, 4, 128), (8, 2, 128)])
        c["batch"] = rng.choice([1, rng.randint(2, 16)])
        c["context"] = _log(rng, 200, 131072 // max(4, c["batch"]))
    return c


# ---- weights -------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, mean=0.0, std=1.0):
    t = torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)
    return t.mul_(std).add_(mean)


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float32)


def _init(g, shape, dtype, init):
    """A tensor of the synthetic checkpoints (quicklm_amd/synth.py's distributions)."""
    if init[0] == "normal":
        t = _normal(g, *shape, mean=init[1], std=init[2])
    elif init[0] == "A_log":
        t = torch.log(1.0 + 15.0 * _uniform(g, *shape))
    else:  # dt_bias: softplus^-1 of a log-uniform step size
        dt = torch.exp(float(np.log(1e-3)) + float(np.log(100.0)) * _uniform(g, *shape))
        t = dt + torch.log(-torch.expm1(-dt))
    return t.to(torch.bfloat16) if dtype == "BF16" else t


def _group(precision: str, K: int) -> int:
    return K if precision == "int8_row" else 32


def _dequantised(w: torch.Tensor, precision: str) -> torch.Tensor:
    """The values a stored weight stands for, in 64 bits: itself (bf16), or
    its Q8_0 / Q4_0 / per-row quantisation."""
    if precision == "bf16":
        return w.to(F64)
    w = w.float()
    N, K = w.shape
    g = w.reshape(N, -1, _group(precision, K))
    m = g.abs().amax(-1, keepdim=True)
    top = torch.full_like(m, 8.0 if precision == "int4" else 127.0)  # a true division
    s = torch.where(m > 0, m / top, torch.ones_like(m))
    q = torch.round(g * (1.0 / s))
    q = q.clamp(-8, 7) if precision == "int4" else q.clamp(-127, 127)
    return (q.to(F64) * s.to(F64)).reshape(N, K)


class Linear:
    """A weight [N, K] on the device as the kernels read it: int8 tiles with
    their scales, or the stored bf16 rows. `halves` 2: gate rows, then up rows."""

    def __init__(self, w: torch.Tensor, precision: str, halves: int = 1):
        self.N, self.K = w.shape
        self.halves, self.precision = halves, precision
        self.group = _group(precision, self.K)
        if precision == "bf16":
            self.q = w.contiguous()
            return
        N, K = self.N, self.K
        rows = torch.empty(N, K, dtype=torch.int8, device=DEV)
        scales = torch.empty(N, K // self.group, dtype=torch.float32, device=DEV)
        _call("qlm_quantize_q8_bf16", w.contiguous(), N, K, self.group, rows, scales)
        qb, sb = hip._sz(), hip._sz()
        _call("qlm_mx_layout_bytes", N // halves, K, self.group, halves, qb, sb, stream=False)
        self.q = torch.empty(qb.value, dtype=torch.int8, device=DEV)
        self.s = torch.empty(sb.value // 4, dtype=torch.float32, device=DEV)
        _call("qlm_mx_swizzle", rows, scales, self.group, N // halves, K, halves, self.q,
              self.s if sb.value else None)
        if not sb.value:
            self.s = scales
        torch.cuda.synchronize()

    def work_bytes(self, M: int, epilogue: int) -> int:
        L, N, K = hip.lib(), self.N // self.halves, self.K
        if self.precision == "bf16":
            return max(L.qlm_matmul_w_workspace_bytes(K), L.qlm_matmul_bf16_workspace_bytes(M, K))
        b = L.qlm_matmul_i8_workspace_bytes(M, N, K, epilogue)
        if 2 <= M <= 16:
            b = max(b, L.qlm_matmul_i8_t_workspace_bytes(M, N, K, epilogue))
        return max(b, 256)

    def __call__(self, x, ldx, M, y, ldy, norm=None, epilogue=0, work=None, stream=None):
        """y = x . W^T (0), y += (1) or SwiGLU (2), by the entry point for M rows."""
        N, K = self.N // self.halves, self.K
        wb = work.numel() if work is not None else 0
        if self.precision == "bf16":
            _call("qlm_matmul_w", x, ldx, norm, EPS, self.q, 1, y, ldy, M, N, K, epilogue, work,
                  wb, on=stream)
        elif M == 1:
            _call("qlm_gemv_i8_mx", x, norm, EPS, self.q, self.s, self.group, y, N, K, epilogue,
                  on=stream)
        else:
            few = M <= 16 and self.group == 32
            _call("qlm_matmul_i8_t" if few else "qlm_matmul_i8_tm", x, ldx, norm, EPS, self.q,
                  self.s, self.group, y, ldy, M, N, K, epilogue, work, wb, on=stream)


def _call(name, *args, on=None, stream=True):
    conv = []
    for a in args:
        if isinstance(a, torch.Tensor):
            conv.append(a.data_ptr())
        elif isinstance(a, hip._sz):
            conv.append(hip.C.byref(a))
        else:
            conv.append(a)
    hip.call(name, *conv, *([on] if stream else []))


class Replayed:
    """A captured sequence of calls, replayed on a stream of its own."""

    def __init__(self, enqueue):
        self.stream = hip.Stream()
        torch.cuda.synchronize()
        _call("qlm_graph_begin", self.stream.ptr, stream=False)
        enqueue(self.stream.ptr)
        g = hip._vp()
        hip.check(hip.lib().qlm_graph_end(self.stream.ptr, hip.C.byref(g)))
        self.graph = g.value

    def launch(self):
        hip.check(hip.lib().qlm_graph_launch(self.graph, self.stream.ptr))

    def __del__(self):
        with contextlib.suppress(Exception):
            self.stream.sync()
            hip.lib().qlm_graph_destroy(self.graph)


# ---- inputs --------------------------------------------------------------------


def _dims(case):
    c = WIDTHS[case["width"]]
    nh, nq, nkv, hd = (c["linear_num_heads"], c["num_attention_heads"],
                       c["num_key_value_heads"], c["head_dim"])
    return c["hidden_size"], c["intermediate_size"], nh, nq, nkv, hd


def _weight(g, N, K):
    return _normal(g, N, K, std=0.02).to(torch.bfloat16)


def _mlp_inputs(case, g, M):
    H, F, *_ = _dims(case)
    layers = [dict(ln=_normal(g, H, std=0.02), gate_up=_weight(g, 2 * F, H),
                   down=_weight(g, H, F)) for _ in range(case.get("layers", 1))]
    return layers, _normal(g, M, H)


def _deltanet_inputs(case, g, M, B):
    H, _, nh, *_ = _dims(case)
    HD = nh * 128
    layers = []
    for _ in range(case.get("layers", 1)):
        layers.append(dict(
            ln=_normal(g, H, std=0.02), w_in=_weight(g, 4 * HD + 2 * nh, H),
            w_out=_weight(g, H, HD), conv_w=_normal(g, 4, 3 * HD, std=0.3),
            A_log=_init(g, [nh], "F32", ("A_log",)), dt=_init(g, [nh], "F32", ("dt_bias",)),
            norm=_normal(g, 128, mean=1.0, std=0.02), conv=_normal(g, B, 3, 3 * HD, std=0.5),
            S=_normal(g, B, nh, 128, 128, std=0.05)))
    return layers, _normal(g, M, H)


def _rope(case, n):
    """The [n, rot / 2] tables of a quarter-rotated head, theta 1e6."""
    rot = _dims(case)[5] // 4
    inv = 1.0 / np.power(np.float32(1e6), np.arange(0, rot, 2, dtype=np.float32) / rot)
    a = torch.from_numpy(np.arange(n, dtype=np.float32)[:, None] * inv.astype(np.float32))
    return rot, torch.cos(a).to(DEV).contiguous(), torch.sin(a).to(DEV).contiguous()


def _attention_inputs(case, g, M, B, S):
    H, _, _, nq, nkv, hd = _dims(case)
    layers = [dict(ln=_normal(g, H, std=0.02), w_in=_weight(g, 2 * nq * hd + 2 * nkv * hd, H),
                   w_out=_weight(g, H, nq * hd), qn=_normal(g, hd, std=0.02),
                   kn=_normal(g, hd, std=0.02), kc=_normal(g, B, S, nkv, hd),
                   vc=_normal(g, B, S, nkv, hd))]
    return layers, _normal(g, M, H)


def _positions(case, seed):
    """Each sequence at a position of its own in the second half of the context."""
    n, r = case["context"], random.Random(seed)
    return [n - 1 - r.randrange(n // 2) if b else n - 1 for b in range(case["batch"])]


def _model_config(case, seed):
    return dict(WIDTHS[case["width"]], num_hidden_layers=ENGINE_LAYERS[case["width"]],
                vocab_size=ENGINE_VOCAB, index=seed % (1 << 20), linear_dtype="BF16")


def _model_tensors(cfg, g):
    for name, shape, dtype, init in synth.tensor_specs(cfg):
        yield name, shape, dtype, _init(g, shape, dtype, init)


def _tokens(case, seed):
    B = case.get("batch", 1)
    n = {"decode": case.get("steps", 0) + 1, "prompt": case.get("rows", 0),
         "verify": case.get("context", 0) + case.get("rows", 0)}[case["kind"]]
    return np.random.default_rng(seed).integers(0, ENGINE_VOCAB, (B, n), dtype=np.int32)


def _write_checkpoint(out_dir, cfg, g):
    header, off = {}, 0
    for name, shape, dtype, _ in synth.tensor_specs(cfg):
        nbytes = int(np.prod(shape)) * (4 if dtype == "F32" else 2)
        header[name] = {"dtype": dtype, "shape": shape, "data_offsets": [off, off + nbytes]}
        off += nbytes
    hj = json.dumps(header).encode()
    hj += b" " * (-len(hj) % 8)
    with open(os.path.join(out_dir, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(hj)) + hj)
        for _, _, dtype, t in _model_tensors(cfg, g):
            t = t.view(torch.int16) if dtype == "BF16" else t
            t.cpu().numpy().tofile(f)
    with open(os.path.join(out_dir, "config.json"), "w") as f:
        json.dump(synth.config_json(cfg), f)


def _engine(case, seed, max_seq):
    d = tempfile.mkdtemp(dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
    try:
        _write_checkpoint(d, _model_config(case, seed), _gen(seed))
        return Engine(d, max_seq_len=max_seq, max_batch=case.get("batch", 1),
                      precision=case["precision"])
    finally:
        shutil.rmtree(d, ignore_errors=True)


def _empty(*shape):
    return torch.zeros(*shape, dtype=torch.float32, device=DEV)


def _work(n):
    return torch.empty(max(int(n), 256), dtype=torch.uint8, device=DEV)


def prepare(case: dict, seed: int) -> dict:
    hip.check(hip.lib().qlm_set_device(0))
    kind = case["kind"]
    st = dict(case=case)
    if kind in ENGINE_KINDS:
        toks = _tokens(case, seed)
        eng = st["engine"] = _engine(case, seed, toks.shape[1] + 8)
        st["tokens"] = toks
        if kind == "verify":
            # the chat so far: positions 0..context-1 consumed, state snapshot kept
            n = case["context"]
            eng.start(toks[:, :n + 1], batched_prefill=True)
            eng.snapshot()
        return st
    g = _gen(seed)
    pr = case.get("precision")
    if kind == "attention_cache":
        B, S = case["batch"], case["context"]
        dt = torch.bfloat16 if case["kv"] == "bf16" else torch.float32
        st["q"] = _normal(g, B, case["n_q"], case["hd"])
        st["k"] = _normal(g, B, S, case["n_kv"], case["hd"]).to(dt)
        st["v"] = _normal(g, B, S, case["n_kv"], case["hd"]).to(dt)
        st["out"] = torch.empty_like(st["q"])
        st["work"] = _work(hip.lib().qlm_gqa_workspace_bytes(B, case["n_q"], case["hd"], S))
        return st
    H, F, nh, nq, nkv, hd = _dims(case)
    if kind == "head":
        M, V = case["batch"], case["vocab"]
        st["lm"] = Linear(_weight(g, V, H), pr)
        st["ln"], st["x"] = _normal(g, H, std=0.02), _normal(g, M, H)
        st["logits"] = _empty(M, V)
        st["pick"] = torch.zeros(M, dtype=torch.int32, device=DEV)
        st["work"] = _work(st["lm"].work_bytes(M, 0))
        st["work2"] = _work(hip.lib().qlm_argmax_workspace_bytes(M, V))
        return st
    decode = kind.endswith("_decode")
    M = case["batch"] if decode else case["rows"]
    if kind.startswith("mlp"):
        layers, h = _mlp_inputs(case, g, M)
        for w in layers:
            w["gate_up"] = Linear(w["gate_up"], pr, 2)
            w["down"] = Linear(w["down"], pr)
        st["act"] = _empty(M, F)
        need = max(layers[0]["gate_up"].work_bytes(M, 2), layers[0]["down"].work_bytes(M, 1))
    else:
        if kind.startswith("deltanet"):
            layers, h = _deltanet_inputs(case, g, M, M if decode else 1)
            st["core"] = _empty(M, nh * 128)
            pos = [0] * M
            st["mixer_work"] = _work(hip.lib().qlm_deltanet_chunk_workspace_bytes(M, nh, 128))
        else:
            S = case["context"] if decode else case["first"] + M
            layers, h = _attention_inputs(case, g, M, M if decode else 1, S)
            st["S"] = S
            st["core"] = _empty(M, nq * hd)
            st["rot"], st["cos"], st["sin"] = _rope(case, S)
            pos = _positions(case, seed) if decode else []
            L = hip.lib()
            st["mixer_work"] = _work(L.qlm_gqa_workspace_bytes(M, nq, hd, S) if decode
                                     else L.qlm_gqa_prefill_workspace_bytes(nq, hd, S))
        for w in layers:
            w["w_in"], w["w_out"] = Linear(w["w_in"], pr), Linear(w["w_out"], pr)
        st["proj"] = _empty(M, layers[0]["w_in"].N)
        st["pos"] = torch.tensor(pos or [0], dtype=torch.int32, device=DEV)
        need = max(layers[0]["w_in"].work_bytes(M, 0), layers[0]["w_out"].work_bytes(M, 1))
    st.update(layers=layers, h=h, M=M, work=_work(need))
    if decode:
        st["step"] = Replayed(lambda s: _layers(st, s))
    return st


# ---- one pass ------------------------------------------------------------------


def _mixer(st, w, stream):
    """The part of a layer between its two projections."""
    case, M, proj, core = st["case"], st["M"], st["proj"], st["core"]
    H, F, nh, nq, nkv, hd = _dims(case)
    P, C = proj.shape[1], core.shape[1]
    if case["kind"] == "deltanet_decode":
        _call("qlm_deltanet_decode", proj, P, w["conv"], w["conv_w"], w["A_log"], w["dt"],
              w["norm"], w["S"], st["pos"], core, C, M, nh, 128, on=stream)
    elif case["kind"] == "deltanet_prefill":
        _call("qlm_deltanet_prefill_chunked", proj, P, M, w["conv"], w["conv_w"], w["A_log"],
              w["dt"], w["norm"], w["S"], 0, core, C, nh, 128, st["mixer_work"],
              st["mixer_work"].numel(), on=stream)
    elif case["kind"] == "attention_decode":
        _call("qlm_gqa_decode", proj, P, w["qn"], w["kn"], st["cos"], st["sin"], st["rot"],
              w["kc"], w["vc"], st["S"], st["pos"], core, C, M, nq, nkv, hd, 1,
              st["mixer_work"], on=stream)
    else:
        _call("qlm_gqa_prefill", proj, P, w["qn"], w["kn"], st["cos"], st["sin"], st["rot"],
              w["kc"], w["vc"], st["S"], case["first"], M, core, C, nq, nkv, hd, 1,
              st["mixer_work"], on=stream)


def _layers(st, stream):
    h, M, work = st["h"], st["M"], st["work"]
    H = h.shape[1]
    for w in st["layers"]:
        if "gate_up" in w:
            act = st["act"]
            w["gate_up"](h, H, M, act, act.shape[1], w["ln"], 2, work, stream)
            w["down"](act, act.shape[1], M, h, H, None, 1, work, stream)
        else:
            proj, core = st["proj"], st["core"]
            w["w_in"](h, H, M, proj, proj.shape[1], w["ln"], 0, work, stream)
            _mixer(st, w, stream)
            w["w_out"](core, core.shape[1], M, h, H, None, 1, work, stream)


def _layer_outputs(h, layers):
    return dict(h=h, state=[[w[k] for k in ("conv", "S", "kc", "vc") if k in w] for w in layers])


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        eng, B = state["engine"], case["batch"]
        eng.start(state["tokens"])
        eng.steps(case["steps"])
        return [eng.last_logits(b) for b in range(B)]
    if kind == "verify":
        eng, n = state["engine"], case["context"]
        eng.restore()
        return eng.forward_batch(state["tokens"][0, n:], n, argmax=True, logits=True)[1]
    if kind == "prompt":
        eng = state["engine"]
        eng.start(state["tokens"], batched_prefill=True)
        eng.steps(1)
        return eng.last_logits(0)
    if kind == "attention_cache":
        _call("qlm_attention_decode", state["q"], state["k"], state["v"],
              1 if case["kv"] == "bf16" else 0, case["context"], case["context"], state["out"],
              case["batch"], case["n_q"], case["n_kv"], case["hd"], state["work"])
        return state["out"]
    if kind == "head":
        lg, M = state["logits"], case["batch"]
        V = lg.shape[1]
        state["lm"](state["x"], state["x"].shape[1], M, lg, V, state["ln"], 0, state["work"])
        _call("qlm_argmax", lg, V, V, M, state["pick"], state["work2"])
        return lg, state["pick"]
    if "step" in state:
        state["step"].launch()
    else:
        _layers(state, None)
    return _layer_outputs(state["h"], state["layers"])


# ---- what a pass cannot do without -----------------------------------------------


def _linear_work(M, N, K, precision):
    per = {"int8": 1.125, "int8_row": 1.0, "int4": 0.625, "bf16": 2.0}[precision]
    return N * K * per + 4 * M * (N + K), 2.0 * M * N * K


def _sum(*parts):
    return tuple(sum(p[i] for p in parts) for i in (0, 1))


def _mlp_work(case, M):
    H, F, *_ = _dims(case)
    p = case["precision"]
    return _sum(_linear_work(M, 2 * F, H, p), _linear_work(M, H, F, p))


def _deltanet_work(case, M, B):
    H, _, nh, *_ = _dims(case)
    HD, p = nh * 128, case["precision"]
    state = 2 * 4 * B * (nh * 128 * 128 + 9 * HD)
    return _sum(_linear_work(M, 4 * HD + 2 * nh, H, p), _linear_work(M, H, HD, p),
                (state, 6.0 * M * nh * 128 * 128))


def _attention_work(case, M, keys, pairs):
    """keys: cache rows read; pairs: (row, key) pairs attended."""
    H, _, _, nq, nkv, hd = _dims(case)
    p = case["precision"]
    return _sum(_linear_work(M, 2 * (nq + nkv) * hd, H, p), _linear_work(M, H, nq * hd, p),
                (8 * nkv * hd * (keys + M), 4.0 * nq * hd * pairs))


def _model_work(case, M, B, first):
    """M rows in all of B sequences that start at `first`."""
    n = ENGINE_LAYERS[case["width"]]
    T = M // B
    pairs = B * (T * first + T * (T + 1) // 2)
    a = _attention_work(case, M, B * (first + T), pairs)
    d = _deltanet_work(case, M, B)
    m = _mlp_work(case, M)
    return tuple(n * m[i] + (n - n // 4) * d[i] + (n // 4) * a[i] for i in (0, 1))


def work(case: dict) -> dict:
    kind, B = case["kind"], case.get("batch", 1)
    if kind == "attention_cache":
        pairs = B * case["context"]
        w = (2 * pairs * case["n_kv"] * case["hd"] * (2 if case["kv"] == "bf16" else 4) +
             8 * B * case["n_q"] * case["hd"], 4.0 * pairs * case["n_q"] * case["hd"])
    elif kind == "head":
        w = _linear_work(B, case["vocab"], _dims(case)[0], case["precision"])
    elif kind == "decode":
        head = _linear_work(B, ENGINE_VOCAB, _dims(case)[0], case["precision"])
        w = _sum(*[_sum(_model_work(case, B, B, t), head) for t in range(case["steps"])])
    elif kind == "verify":
        w = _sum(_model_work(case, case["rows"], 1, case["context"]),
                 _linear_work(case["rows"], ENGINE_VOCAB, _dims(case)[0], case["precision"]))
    elif kind == "prompt":
        w = _sum(_model_work(case, case["rows"], 1, 0),
                 _linear_work(1, ENGINE_VOCAB, _dims(case)[0], case["precision"]))
    else:
        n = case.get("layers", 1)
        M = case.get("rows", B)
        if kind.startswith("mlp"):
            w = _mlp_work(case, M)
        elif kind.startswith("deltanet"):
            w = _deltanet_work(case, M, B)
        elif kind == "attention_decode":
            keys = sum(p + 1 for p in _positions(case, 0))
            w = _attention_work(case, M, keys, keys)
        else:
            w = _attention_work(case, M, case["first"] + M,
                                M * case["first"] + M * (M + 1) // 2)
        w = (n * w[0], n * w[1])
    return {"bytes": float(w[0]), "flops": float(w[1])}


def tolerance(case: dict):
    """32-bit sums throughout; the largest errors against 64 bits are those of
    activations split into two bf16 terms (2^-17 of a value) in the
    matrix-core products, which a few layers' residual streams add up."""
    if case["kind"] in ENGINE_KINDS:
        return {"rel": 1.2e-4, "max": 4e-3}
    t = {"rel": 2e-5, "max": 1e-3}
    if case["kind"] == "head":
        t["differ"] = 0.005  # ties of the greedy pick
    return t


# ---- the same in 64 bits -----------------------------------------------------------


def _mm(x, w, step=32768):
    return torch.cat([x @ p.T for p in w.split(step)], -1)


def _rms(x, gain=None, eps=EPS):
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)
    return y if gain is None else y * (1.0 + gain.to(F64))


def _exact_linear(w, precision):
    return _dequantised(w, precision)


def _exact_mlp(h, w, precision):
    gu = _mm(_rms(h, w["ln"]), _exact_linear(w["gate_up"], precision))
    gate, up = gu.chunk(2, -1)
    act = gate * torch.sigmoid(gate) * up
    return h + _mm(act, _exact_linear(w["down"], precision))


def _exact_deltanet(h, w, precision, nh, conv, S):
    """h [B, T, H]; conv [B, 3, C] the three rows before (oldest first), S
    [B, nh, d, d]. Returns (h, conv, S) after the T rows."""
    B, T, _ = h.shape
    HD = nh * 128
    proj = _mm(_rms(h, w["ln"]), _exact_linear(w["w_in"], precision))
    x = torch.cat([conv, proj[..., :3 * HD]], 1)
    wt = w["conv_w"].to(F64)
    y = sum(x[:, j:j + T] * wt[j] for j in range(4))
    y = y * torch.sigmoid(y)
    q, k, v = (t.reshape(B, T, nh, 128) for t in y.chunk(3, -1))
    q = q / torch.sqrt(q.square().sum(-1, keepdim=True) + 1e-6)
    k = k / torch.sqrt(k.square().sum(-1, keepdim=True) + 1e-6)
    z, braw, araw = proj[..., 3 * HD:4 * HD], proj[..., 4 * HD:4 * HD + nh], proj[..., -nh:]
    decay = torch.exp(-torch.exp(w["A_log"].to(F64)) *
                      torch.nn.functional.softplus(araw + w["dt"].to(F64), threshold=50.0))
    beta = torch.sigmoid(braw)
    out = torch.empty(B, T, nh, 128, dtype=F64, device=h.device)
    S = S.to(F64)
    for t in range(T):
        S = S * decay[:, t, :, None, None]
        kt = k[:, t, :, :, None]
        delta = (v[:, t] - (kt * S).sum(2)) * beta[:, t, :, None]
        S = S + kt * delta[:, :, None, :]
        out[:, t] = (q[:, t, :, :, None] * S).sum(2) / 128.0 ** 0.5
    o = _rms(out) * w["norm"].to(F64)
    o = o.reshape(B, T, HD) * (z * torch.sigmoid(z))
    return h + _mm(o, _exact_linear(w["w_out"], precision)), x[:, -3:], S


def _exact_rope(t, cos, sin):
    """t [..., heads, hd]; cos/sin [..., rot / 2] of the same rows."""
    half = cos.shape[-1]
    c, s = cos.to(F64).unsqueeze(-2), sin.to(F64).unsqueeze(-2)
    a, b = t[..., :half], t[..., half:2 * half]
    return torch.cat([a * c - b * s, b * c + a * s, t[..., 2 * half:]], -1)


def _exact_attend(q, k, v, seen):
    """q [T, nq, hd] over k, v [S, nkv, hd]; row t sees its first seen[t] keys."""
    T, nq, hd = q.shape
    nkv = k.shape[1]
    out = torch.empty_like(q)
    hide = torch.arange(k.shape[0], device=q.device)[None, :] >= seen[:, None]
    for j in range(nq):
        kk, vv = k[:, j * nkv // nq], v[:, j * nkv // nq]
        s = (q[:, j] @ kk.T / hd ** 0.5).masked_fill(hide, float("-inf"))
        out[:, j] = torch.softmax(s, -1) @ vv
    return out


def _exact_attention(h, w, precision, dims, rope, pos, kc, vc):
    """h [B, T, H], rows of sequence b at positions pos[b]..pos[b] + T - 1;
    caches [B, S, nkv, hd], written in place."""
    nq, nkv, hd = dims
    B, T, _ = h.shape
    proj = _mm(_rms(h, w["ln"]), _exact_linear(w["w_in"], precision))
    qg, k, v = proj.split([2 * nq * hd, nkv * hd, nkv * hd], -1)
    q, gate = qg.reshape(B, T, nq, 2 * hd).split(hd, -1)
    k, v = k.reshape(B, T, nkv, hd), v.reshape(B, T, nkv, hd)
    q, k = _rms(q, w["qn"]), _rms(k, w["kn"])
    core = torch.empty(B, T, nq, hd, dtype=F64, device=h.device)
    for b in range(B):
        at = torch.arange(pos[b], pos[b] + T, device=h.device)
        cos, sin = rope[0][at], rope[1][at]
        kc[b, at], vc[b, at] = _exact_rope(k[b], cos, sin), v[b]
        n = pos[b] + T
        core[b] = _exact_attend(_exact_rope(q[b], cos, sin), kc[b, :n], vc[b, :n], at + 1)
    core = (core * torch.sigmoid(gate)).reshape(B, T, nq * hd)
    return h + _mm(core, _exact_linear(w["w_out"], precision))


def _exact_logits(case, seed, rows):
    """Logits [B, rows, V] of the last `rows` positions forwarded."""
    pr = case["precision"]
    H, F, nh, nq, nkv, hd = _dims(case)
    toks = torch.from_numpy(_tokens(case, seed)).long().to(DEV)
    if case["kind"] == "decode":
        toks = toks[:, :-1]
    B, T = toks.shape
    cfg = _model_config(case, seed)
    t = {name: v for name, _, _, v in _model_tensors(cfg, _gen(seed))}
    rope = _rope(case, T)[1:]
    embed = t["model.embed_tokens.weight"]
    h = embed.to(F64)[toks]
    for i, kind in enumerate(synth.layer_types(cfg["num_hidden_layers"])):
        def w(name, i=i):
            return t[f"model.layers.{i}.{name}"]
        if kind == "full_attention":
            lw = dict(ln=w("input_layernorm.weight"), w_out=w("self_attn.o_proj.weight"),
                      w_in=torch.cat([w(f"self_attn.{x}_proj.weight") for x in "qkv"]),
                      qn=w("self_attn.q_norm.weight"), kn=w("self_attn.k_norm.weight"))
            kc = torch.zeros(B, T, nkv, hd, dtype=F64, device=DEV)
            h = _exact_attention(h, lw, pr, (nq, nkv, hd), rope, [0] * B, kc, kc.clone())
        else:
            conv_w = w("linear_attn.conv1d.weight")
            lw = dict(ln=w("input_layernorm.weight"), w_out=w("linear_attn.out_proj.weight"),
                      w_in=torch.cat([w(f"linear_attn.in_proj_{x}.weight")
                                      for x in ("qkv", "z", "b", "a")]),
                      conv_w=conv_w.reshape(conv_w.shape[0], 4).T, A_log=w("linear_attn.A_log"),
                      dt=w("linear_attn.dt_bias"), norm=w("linear_attn.norm.weight"))
            conv = torch.zeros(B, 3, 3 * nh * 128, dtype=F64, device=DEV)
            S = torch.zeros(B, nh, 128, 128, dtype=F64, device=DEV)
            h = _exact_deltanet(h, lw, pr, nh, conv, S)[0]
        lw = dict(ln=w("post_attention_layernorm.weight"), down=w("mlp.down_proj.weight"),
                  gate_up=torch.cat([w("mlp.gate_proj.weight"), w("mlp.up_proj.weight")]))
        h = _exact_mlp(h, lw, pr)
    return _mm(_rms(h[:, -rows:], t["model.norm.weight"]), _exact_linear(embed, pr))


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "decode":
        return list(_exact_logits(case, seed, 1)[:, 0])
    if kind == "verify":
        return _exact_logits(case, seed, case["rows"])[0]
    if kind == "prompt":
        return _exact_logits(case, seed, 1)[0, 0]
    g = _gen(seed)
    if kind == "attention_cache":
        B, S = case["batch"], case["context"]
        dt = torch.bfloat16 if case["kv"] == "bf16" else torch.float32
        q = _normal(g, B, case["n_q"], case["hd"])
        k = _normal(g, B, S, case["n_kv"], case["hd"]).to(dt)
        v = _normal(g, B, S, case["n_kv"], case["hd"]).to(dt)
        seen = torch.tensor([S], device=DEV)
        return torch.stack([_exact_attend(q[b:b + 1].to(F64), k[b].to(F64), v[b].to(F64), seen)[0]
                            for b in range(B)])
    H, F, nh, nq, nkv, hd = _dims(case)
    pr = case["precision"]
    if kind == "head":
        w = _weight(g, case["vocab"], H)
        ln, x = _normal(g, H, std=0.02), _normal(g, case["batch"], H)
        lg = _mm(_rms(x.to(F64), ln), _exact_linear(w, pr))
        return lg, lg.argmax(-1).to(torch.int32)
    decode = kind.endswith("_decode")
    M = case["batch"] if decode else case["rows"]
    B = M if decode else 1
    if kind.startswith("mlp"):
        layers, h = _mlp_inputs(case, g, M)
        h = h.to(F64)
        for w in layers:
            h = _exact_mlp(h, w, pr)
        return _layer_outputs(h, [{} for _ in layers])
    outs = []
    if kind.startswith("deltanet"):
        layers, h = _deltanet_inputs(case, g, M, B)
        h = h.to(F64).reshape(B, M // B, H)
        for w in layers:
            h, conv, S = _exact_deltanet(h, w, pr, nh, w["conv"].to(F64), w["S"])
            # position 0 is the oldest tap's row: the ring holds position p at p % 3
            n = M // B
            ring = torch.stack([conv[:, (r - n) % 3] for r in range(3)], 1)
            outs.append(dict(conv=ring, S=S))
    else:
        S = case["context"] if decode else case["first"] + M
        layers, h = _attention_inputs(case, g, M, B, S)
        h = h.to(F64).reshape(B, M // B, H)
        pos = _positions(case, seed) if decode else [case["first"]]
        for w in layers:
            kc, vc = w["kc"].to(F64), w["vc"].to(F64)
            h = _exact_attention(h, w, pr, (nq, nkv, hd), _rope(case, S)[1:], pos, kc, vc)
            outs.append(dict(kc=kc, vc=vc))
    return _layer_outputs(h.reshape(M, H), outs)
