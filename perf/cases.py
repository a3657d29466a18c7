"""Performance cases of the decode backend: what its users run, through the C ABI and the engine.

listed() are the cases, draw() gives more of the same ranges. A case is the decode step of one model
(`kind` "decode"), the batched decode step ("batch"), the chunked prefill ("prefill") or the attention
stack of DeepSeek-V3 ("mla"). Apart from three whole models they are stacks of a few layers with a
small vocabulary, so that a case's time is its layers' time; a stack keeps more weights than the
memory-side cache holds, as a whole model does.

Weights, contexts and tokens come from the seed (torch's generator) and enter through the loaders and
the documented KV layouts; the caller owns every buffer (velox_hip_arena_bind). exact() recomputes a
case's outputs in float64 from the same values.
"""
from __future__ import annotations

import ctypes as C
import math

import torch

from velox_amd import _lib as L
from velox_amd.engine import HipDecodeEngine

# the builtin configurations: hidden, FFN, q heads, KV heads, head size, eps, theta, QKV bias, tied head
MODELS = {
    "smollm_135m": (576, 1536, 9, 3, 64, 1e-5, 1e4, False, True),
    "llama3_8b": (4096, 14336, 32, 8, 128, 1e-5, 5e5, False, False),
    "qwen2_5_7b": (3584, 18944, 28, 4, 128, 1e-6, 1e6, True, True),
    "qwen2_72b": (8192, 29568, 64, 8, 128, 1e-6, 1e6, True, False),
}
# DeepSeek-V3's attention: hidden, heads, q LoRA, KV LoRA, nope, rope, v
MLA = (7168, 128, 1536, 512, 128, 64, 128)
QUANT = {"q4_0": L.QUANT_GGML_Q4_0, "f32": L.QUANT_F32, "f16": L.QUANT_F16, "g64": L.QUANT_G64}
BYTES_PER_WEIGHT = {"q4_0": 18 / 32, "g64": 18 / 32, "f32": 4.0, "f16": 2.0}
WINDOW = 64   # positions a batched decode advances over before its states go back to the start
CHUNK = 128   # prefill chunk, the backend's largest


# ---- the cases ------------------------------------------------------------------------------------

def listed():
    return [
        # the smallest model in the reference's own fp32 format, one forward_step() of the Python
        # engine after another: launch latency and the logits' way to the host count
        {"name": "smollm_f32_forward_step", "kind": "decode", "model": "smollm_135m", "layers": 30, "vocab": 49152,
         "quant": "f32", "pos": 100, "cap": 512, "call": "engine"},
        # the same model in the reference's 4-bit format, the runner's graph-replayed step
        {"name": "smollm_g64_decode", "kind": "decode", "model": "smollm_135m", "layers": 30, "vocab": 49152,
         "quant": "g64", "pos": 37, "cap": 512, "call": "graph"},
        # the headline: a whole Llama-3-8B in Q4_0, one token at a short context
        {"name": "llama8b_q4_decode", "kind": "decode", "model": "llama3_8b", "layers": 32, "vocab": 128256,
         "quant": "q4_0", "pos": 256, "cap": 512, "call": "graph"},
        # fp16 rows (--quantize f16) at Llama-3-8B's layer sizes
        {"name": "llama8b_f16_decode", "kind": "decode", "model": "llama3_8b", "layers": 2, "vocab": 2048,
         "quant": "f16", "pos": 700, "cap": 1024, "call": "graph"},
        # one user with a 2048-token context on Qwen2.5-7B's layers
        {"name": "qwen7b_q4_decode_ctx2048", "kind": "decode", "model": "qwen2_5_7b", "layers": 4, "vocab": 2048,
         "quant": "q4_0", "pos": 2048, "cap": 2112, "call": "graph"},
        # the largest dense layers and the longest context
        {"name": "qwen72b_q4_decode_ctx8192", "kind": "decode", "model": "qwen2_72b", "layers": 2, "vocab": 2048,
         "quant": "q4_0", "pos": 8192, "cap": 8256, "call": "graph"},
        # serving: 8 and 32 sequences of unequal length per step
        {"name": "qwen7b_q4_batch8_ctx2048", "kind": "batch", "model": "qwen2_5_7b", "layers": 4, "vocab": 2048,
         "rows": 8, "pos": 2048},
        {"name": "qwen7b_q4_batch32_ctx2048", "kind": "batch", "model": "qwen2_5_7b", "layers": 4, "vocab": 2048,
         "rows": 32, "pos": 2048},
        # time to first token: a 128-token prompt in one chunk, and a 1000-token one whose last chunk is ragged
        {"name": "llama8b_q4_prefill128", "kind": "prefill", "model": "llama3_8b", "layers": 4, "vocab": 2048,
         "pos": 0, "rows": 128},
        {"name": "qwen7b_q4_prefill1000", "kind": "prefill", "model": "qwen2_5_7b", "layers": 2, "vocab": 2048,
         "pos": 0, "rows": 1000},
        # DeepSeek-V3's attention layers at 4096 latent positions, one user and sixteen
        {"name": "mla_b1_ctx4096", "kind": "mla", "layers": 2, "rows": 1, "pos": 4096},
        {"name": "mla_b16_ctx4096", "kind": "mla", "layers": 2, "rows": 16, "pos": 4096},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "batch", "batch", "prefill", "mla"))
    if kind == "mla":
        return {"kind": kind, "layers": rng.randint(1, 2), "rows": _log(rng, 1, 32), "pos": _log(rng, 16, 4200)}
    vocab = rng.randint(500, 4000)
    if kind == "prefill":
        return {"kind": kind, "model": rng.choice(("smollm_135m", "llama3_8b", "qwen2_5_7b")), "layers": rng.randint(1, 2),
                "vocab": vocab, "pos": rng.choice((0, 0, _log(rng, 16, 2000))), "rows": _log(rng, 2, 1000)}
    model = rng.choice(tuple(MODELS))
    if kind == "batch":
        return {"kind": kind, "model": model, "layers": rng.randint(1, 2), "vocab": vocab, "rows": _log(rng, 2, 32),
                "pos": _log(rng, 64, 4096)}
    small = model == "smollm_135m"
    quant = rng.choice(("q4_0", "q4_0", "q4_0", "g64", "f32", "f16") if small else ("q4_0", "q4_0", "q4_0", "g64", "f16"))
    pos = _log(rng, 1, 2000 if small else 8200)
    return {"kind": kind, "model": model, "layers": rng.randint(4, 30) if small else rng.randint(1, 3), "vocab": vocab,
            "quant": quant, "pos": pos, "cap": pos + rng.randint(1, 300), "call": rng.choice(("graph", "graph", "engine"))}


# ---- inputs ---------------------------------------------------------------------------------------

def _gen(seed, *tag):
    g = torch.Generator(device="cuda")
    x = (int(seed) + 1) * 1000003
    for t in tag:
        x = (x * 131 + int(t) + 7) % (1 << 61)
    return g.manual_seed(x)


def _randn(shape, g, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


class _Weights:
    """A dense model's tensors by (kind, layer): `raw` what the loaders take, `dense` their float64 values."""

    def __init__(self, case, seed):
        self.h, self.f, self.hq, self.hkv, self.d, self.eps, self.theta, self.bias, self.tied = MODELS[case["model"]]
        self.vocab, self.quant, self.seed, self.layers = case["vocab"], case.get("quant", "q4_0"), seed, case["layers"]

    def shape(self, kind):
        qd, kvd = self.hq * self.d, self.hkv * self.d
        return {L.T_EMBED: (self.vocab, self.h), L.T_HEAD: (self.vocab, self.h), L.T_Q: (qd, self.h), L.T_K: (kvd, self.h),
                L.T_V: (kvd, self.h), L.T_O: (self.h, qd), L.T_GATE: (self.f, self.h), L.T_UP: (self.f, self.h),
                L.T_DOWN: (self.h, self.f), L.T_ATTN_NORM: (self.h,), L.T_MLP_NORM: (self.h,), L.T_FINAL_NORM: (self.h,),
                L.T_BQ: (qd,), L.T_BK: (kvd,), L.T_BV: (kvd,)}[kind]

    def vector(self, kind, layer):
        v = _randn(self.shape(kind), _gen(self.seed, kind, layer))
        return v * 0.02 if kind in (L.T_BQ, L.T_BK, L.T_BV) else 1.0 + 0.1 * v

    def _codes(self, kind, layer):
        """4-bit codes [rows][blocks][32 or 64] and their fp16 scales: what quantizing N(0, 0.02) weights gives."""
        n, k = self.shape(kind)
        g = _gen(self.seed, kind, layer)
        if self.quant == "q4_0":
            q = _randn((n * k // 32, 32), g).mul_(2.8).round_().add_(8).clamp_(0, 15).to(torch.uint8)
            d = (0.0072 * (1.0 + 0.15 * _randn((n * k // 32, 1), g).clamp_(-3, 3))).half()
            return q, d
        q = _randn((n * k // 64, 64), g).mul_(3.0).add_(7.5).round_().clamp_(0, 15)
        at = torch.randint(0, 64, (n * k // 64, 1), generator=g, device="cuda")
        q.scatter_(1, at, 0.0).scatter_(1, (at + 17) % 64, 15.0)  # every group uses its whole range
        s = (0.0066 * (1.0 + 0.15 * _randn((n * k // 64, 1), g).clamp_(-3, 3))).half()
        m = (-7.5 * s.float() * (1.0 + 0.1 * _randn((n * k // 64, 1), g).clamp_(-3, 3))).half()
        return q, s, m

    def raw(self, kind, layer):
        """q4_0: GGML blocks (uint8), g64: fp32 rows on the format's grid, f32 / f16: rows."""
        if self.quant == "q4_0":
            q, d = self._codes(kind, layer)
            out = torch.empty((q.shape[0], 18), dtype=torch.uint8, device=q.device)
            out[:, :2] = d.view(torch.uint8)
            out[:, 2:] = q[:, :16] | (q[:, 16:] << 4)
            return out
        if self.quant == "g64":
            q, s, m = self._codes(kind, layer)
            return q * s.float() + m.float()
        w = _randn(self.shape(kind), _gen(self.seed, kind, layer)) * 0.02
        return w.half() if self.quant == "f16" else w

    def dense(self, kind, layer):
        if self.quant == "q4_0":
            q, d = self._codes(kind, layer)
            return ((q.double() - 8.0) * d.double()).view(self.shape(kind))
        if self.quant == "g64":
            q, s, m = self._codes(kind, layer)
            return (q.double() * s.double() + m.double()).view(self.shape(kind))
        return self.raw(kind, layer).double()

    def matrices(self):
        for layer in range(self.layers):
            for kind in (L.T_Q, L.T_K, L.T_V, L.T_O, L.T_GATE, L.T_UP, L.T_DOWN):
                yield kind, layer
        yield L.T_EMBED, 0
        if not self.tied:
            yield L.T_HEAD, 0

    def vectors(self):
        for layer in range(self.layers):
            for kind in (L.T_ATTN_NORM, L.T_MLP_NORM) + ((L.T_BQ, L.T_BK, L.T_BV) if self.bias else ()):
                yield kind, layer
        yield L.T_FINAL_NORM, 0


def _context(case, seed, layer, seq, n, shape):
    """bf16 context rows of one layer and sequence: N(0, 1), as K/V rows and normalized latents are."""
    return _randn((n,) + shape, _gen(seed, 77, layer, seq)).bfloat16()


def _tokens(case, seed, n, seq=0):
    return torch.randint(0, case["vocab"], (n,), generator=_gen(seed, 99, seq), device="cuda").tolist()


def _positions(case):
    """A batch's positions: evenly spaced from `pos` down to about half of it."""
    b, pos = case["rows"], case["pos"]
    step = pos // 2 // max(1, b - 1)
    if case["kind"] == "batch":
        step -= step % 32  # every sequence at the same slot of its V block: the new rows are one strided view
    return [pos - step * s for s in range(b)]


# position r of a V block of 32 lies in slot 8 ((r % 16) / 4) + 4 (r / 16) + r % 4
_SLOT = [8 * ((r % 16) // 4) + 4 * (r // 16) + r % 4 for r in range(32)]


def _v_blocks(v):
    """V rows [positions][hkv][d] -> [hkv][blocks][d][32], the last block padded with zeros."""
    n, hkv, d = v.shape
    nb = (n + 31) // 32
    full = torch.zeros((nb * 32, hkv, d), dtype=v.dtype, device=v.device)
    full[:n] = v
    out = torch.empty((hkv, nb, d, 32), dtype=v.dtype, device=v.device)
    out[..., torch.tensor(_SLOT, device=v.device)] = full.view(nb, 32, hkv, d).permute(2, 0, 3, 1)
    return out


_pinned = {}


def _host(t):
    """A device tensor's bytes in pinned host memory, as a program that reads its weights into a
    staging buffer has them: the loaders take host data."""
    flat = t.contiguous().view(torch.uint8).view(-1)
    if "buf" not in _pinned or _pinned["buf"].numel() < flat.numel():
        _pinned["buf"] = torch.empty(max(flat.numel(), 320 << 20), dtype=torch.uint8, pin_memory=True)
    out = _pinned["buf"][: flat.numel()]
    out.copy_(flat)
    torch.cuda.synchronize()
    return out


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _bytes(n):
    return torch.empty(max(256, int(n)), dtype=torch.uint8, device="cuda")


class _Dense:
    """A dense model with caller-owned buffers (or, for call "engine", inside a HipDecodeEngine)."""

    def __init__(self, case, seed):
        self.case, self.lib, self.w = case, L.load(), _Weights(case, seed)
        w, kind = self.w, case["kind"]
        cap = {"decode": case.get("cap"), "batch": case["pos"] + WINDOW, "prefill": case["pos"] + case.get("rows", 0)}[kind]
        dims = dict(vocab_size=w.vocab, hidden_dim=w.h, intermediate_dim=w.f, num_layers=w.layers, num_heads=w.hq,
                    num_kv_heads=w.hkv, head_dim=w.d, max_seq_len=cap, rms_norm_eps=w.eps, rope_theta=w.theta,
                    qkv_bias=int(w.bias), tied_lm_head=int(w.tied), quant_mode=QUANT[w.quant])
        if kind == "batch":
            dims["max_batch"] = case["rows"]
        if kind == "prefill":
            dims["prefill_chunk"] = CHUNK
        self.cap, self.s_cap = cap, (cap + 31) // 32 * 32
        self.seqs = case["rows"] if kind == "batch" else 1
        self.graph, self.engine, self.i = None, None, 0
        self.model = C.c_void_p()
        self.arena = L.Arena()
        if case.get("call") == "engine":
            self.engine = HipDecodeEngine(dims, synthesize=False)
            self.arena = self.engine.arena
            kv_bytes = self.engine.arena_bytes()["kv"]
            self.kv = torch.zeros(kv_bytes, dtype=torch.uint8, device="cuda")
        else:
            cfg = L.ModelConfig()
            cfg.name = b"stack"
            for k, v in dims.items():
                setattr(cfg, k, v)
            L.check(self.lib.velox_hip_model_create(C.byref(cfg), C.byref(self.model)), "model_create")
            size = [C.c_uint64() for _ in range(5)]
            L.check(self.lib.velox_hip_model_arena_bytes(self.model, *[C.byref(x) for x in size]), "arena_bytes")
            self.buf = [_bytes(x.value) for x in size]  # weights, scales, norms, KV pool, activations
            self.ring = torch.zeros(L.RING_SIZE * self.seqs, dtype=torch.int32, pin_memory=True)
            a = self.arena
            a.weight_arena, a.weight_scales, a.norm_weight_arena, a.kv_cache_pool, a.activation_arena = (
                b.data_ptr() for b in self.buf)
            a.host_pinned_ring = C.cast(self.ring.data_ptr(), C.POINTER(C.c_uint32))
            a.quant_mode, a.tied_lm_head = QUANT[w.quant], int(w.tied)
            torch.cuda.synchronize()
            L.check(self.lib.velox_hip_arena_bind(self.model, C.byref(a)), "arena_bind")
            self.kv, kv_bytes = self.buf[3], size[3].value
        load = self.lib.velox_hip_load_q4_0 if w.quant == "q4_0" else self.lib.velox_hip_load_rows
        for k, layer in w.matrices():
            x = _host(w.raw(k, layer))
            L.check(load(C.byref(self.arena), k, layer, x.data_ptr(), x.numel(), None), "load matrix")
        for k, layer in w.vectors():
            x = _host(w.vector(k, layer))
            L.check(self.lib.velox_hip_load_f32(C.byref(self.arena), k, layer, x.data_ptr(), x.numel() // 4, None), "load_f32")
        # [layer][sequence]: the K plane [hkv][s_cap][d], then the V plane [hkv][s_cap / 32][d][32]
        plane = w.hkv * self.s_cap * w.d
        self.pool = self.kv[:kv_bytes].view(torch.bfloat16).view(w.layers, self.seqs, -1)
        self.k = self.pool[..., :plane].view(w.layers, self.seqs, w.hkv, self.s_cap, w.d)
        self.v = self.pool[..., plane: 2 * plane].view(w.layers, self.seqs, w.hkv, self.s_cap // 32, w.d, 32)
        for layer in range(w.layers):
            for s, n in enumerate(_positions(case) if kind == "batch" else [case["pos"]]):
                if n:
                    ctx = _context(case, seed, layer, s, n, (2, w.hkv, w.d))
                    self.k[layer, s, :, :n] = ctx[:, 0].permute(1, 0, 2)
                    vb = _v_blocks(ctx[:, 1])
                    self.v[layer, s, :, : vb.shape[1]] = vb
        if self.engine:
            torch.cuda.synchronize()
            rc = L.hip().hipMemcpy(self.arena.kv_cache_pool, self.kv.data_ptr(), kv_bytes, 3)
            if rc:
                raise RuntimeError("hipMemcpy of the context failed: %d" % rc)
        else:
            act = self.buf[4]
            lo, ho = C.c_uint64(), C.c_uint64()
            rows = 1
            if kind == "decode":
                lo.value = self.lib.velox_hip_model_logits_offset(self.model)
                ho.value = self.lib.velox_hip_model_hidden_offset(self.model)
                self.hidden = act[ho.value: ho.value + 4 * w.h].view(torch.float32)
            else:
                L.check(self.lib.velox_hip_model_batch_layout(self.model, None, C.byref(lo), C.byref(ho)), "batch_layout")
                rows = case["rows"] if kind == "batch" else (case["rows"] - 1) % CHUNK + 1
            self.logits = act[lo.value: lo.value + 4 * rows * w.vocab].view(torch.float32).view(rows, w.vocab)
        if kind == "decode":
            self.token = _tokens(case, seed, 1)[0]
        elif kind == "prefill":
            t = (C.c_uint32 * cap)(*_tokens(case, seed, cap))
            L.check(self.lib.velox_hip_set_prompt(C.byref(self.arena), t, cap, None), "set_prompt")
        else:
            self.pos = _positions(case)
            self.tokens = [_tokens(case, seed, cap, s) for s in range(self.seqs)]
            for s, t in enumerate(self.tokens):  # the next tokens are given, as in scoring: a pass depends on its inputs alone
                L.check(self.lib.velox_hip_batch_set_prompt(C.byref(self.arena), s, (C.c_uint32 * cap)(*t), cap, None), "prompt")
        if case.get("call") == "graph" or kind == "batch":
            if kind == "batch":
                self.rewind()
            self.step()  # once eagerly: modules load outside the capture
            torch.cuda.synchronize()
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph):
                self.step()
            L.check(self.lib.velox_hip_last_error(), "decode step")
            if kind == "batch":
                self.rewind()
            torch.cuda.synchronize()

    def rewind(self):
        for s, p in enumerate(self.pos):
            L.check(self.lib.velox_hip_batch_set_state(C.byref(self.arena), s, p, self.tokens[s][p], _stream()), "set_state")
        self.i = 0

    def step(self):
        if self.case["kind"] == "decode":
            self.lib.velox_hip_decode(C.byref(self.arena), self.token, self.case["pos"], 1, _stream())
        else:
            self.lib.velox_hip_decode_batch_graph_step(C.byref(self.arena), self.seqs, 1, _stream())

    def new_rows(self, p0, step):
        """Views of the K and V rows written at positions p0 - step * s of sequence s, [layers][sequences][hkv][d]."""
        k, v = self.k, self.v
        shape = (k.shape[0], self.seqs, k.shape[2], k.shape[4])
        ks = torch.as_strided(k, shape, (k.stride(0), k.stride(1) - step * k.stride(3), k.stride(2), 1),
                              k.storage_offset() + p0 * k.stride(3))
        vs = torch.as_strided(v, shape, (v.stride(0), v.stride(1) - step // 32 * v.stride(3), v.stride(2), 32),
                              v.storage_offset() + p0 // 32 * v.stride(3) + _SLOT[p0 % 32])
        return ks, vs

    def run(self):
        c = self.case
        if self.engine:
            self.engine.forward_step(self.token, c["pos"])
            return {"logits": self.engine.logits}
        if c["kind"] == "decode":
            self.graph.replay()
            k, v = self.new_rows(c["pos"], 0)
            return {"logits": self.logits, "hidden": self.hidden, "k": k, "v": v}
        if c["kind"] == "batch":
            if self.i == WINDOW:
                self.rewind()
            self.graph.replay()
            p0 = self.pos[0] + self.i
            self.i += 1
            k, v = self.new_rows(p0, self.pos[0] - self.pos[1])
            return {"logits": self.logits, "k": k, "v": v}
        L.check(self.lib.velox_hip_prefill_batch(C.byref(self.arena), c["pos"], c["rows"], 1, _stream()), "prefill_batch")
        return {"logits": self.logits, "k": self.k, "v": self.v}

    def __del__(self):
        try:
            torch.cuda.synchronize()
            if self.engine:
                self.engine.close()
            elif self.model.value:
                self.lib.velox_hip_arena_destroy(C.byref(self.arena))
                self.lib.velox_hip_model_destroy(self.model)
        except Exception:
            pass


def _mla_shapes():
    h, nh, ql, lr, dn, dr, dv = MLA
    return {L.MLA_Q_A: (ql, h), L.MLA_Q_B: (nh * (dn + dr), ql), L.MLA_KV_A: (lr + dr, h), L.MLA_KV_B: (nh * (dn + dv), lr),
            L.MLA_O: (h, nh * dv), L.MLA_NORM: (h,), L.MLA_Q_A_NORM: (ql,), L.MLA_KV_A_NORM: (lr,)}


def _mla_matrix(seed, kind, layer):
    """fp8 e4m3fn codes [rows][cols] and fp32 scales per 128 x 128 block, as a checkpoint holds them."""
    n, k = _mla_shapes()[kind]
    g = _gen(seed, 40 + kind, layer)
    codes = _randn((n, k), g).mul_(100.0).clamp_(-448, 448).to(torch.float8_e4m3fn)
    scales = 0.0002 * (1.0 + 0.2 * _randn(((n + 127) // 128, (k + 127) // 128), g).clamp_(-3, 3))
    return codes, scales


def _mla_vector(seed, kind, layer):
    return 1.0 + 0.1 * _randn(_mla_shapes()[kind], _gen(seed, 40 + kind, layer))


def _mla_hidden(case, seed):
    return _randn((case["rows"], MLA[0]), _gen(seed, 98)) * 0.05  # of a layer's own update's size


class _Mla:
    """DeepSeek-V3 attention layers with caller-owned buffers; a pass starts from the given hidden rows."""

    def __init__(self, case, seed):
        self.case, self.lib = case, L.load()
        lib, rows, layers = self.lib, case["rows"], case["layers"]
        cap = case["pos"] + 1
        cfg = L.MlaConfig()
        L.check(lib.velox_hip_mla_builtin_config(b"deepseek_v3_mla", cap, rows, C.byref(cfg)), "mla config")
        cfg.num_layers = layers
        self.m = C.c_void_p()
        L.check(lib.velox_hip_mla_plan(C.byref(cfg), C.byref(self.m)), "mla_plan")
        size = [C.c_uint64() for _ in range(5)]
        L.check(lib.velox_hip_mla_arena_bytes(self.m, *[C.byref(x) for x in size]), "mla_arena_bytes")
        self.buf = [_bytes(x.value) for x in size]
        a = self.arena = L.Arena()
        a.weight_arena, a.weight_scales, a.norm_weight_arena, a.kv_cache_pool, a.activation_arena = (
            b.data_ptr() for b in self.buf)
        a.quant_mode = 3
        torch.cuda.synchronize()
        L.check(lib.velox_hip_mla_arena_bind(self.m, C.byref(a)), "mla_arena_bind")
        info = L.MlaBuffers()
        L.check(lib.velox_hip_mla_buffers(self.m, C.byref(info)), "mla_buffers")
        for layer in range(layers):
            for kind in (L.MLA_Q_A, L.MLA_Q_B, L.MLA_KV_A, L.MLA_KV_B, L.MLA_O):
                codes, scales = _mla_matrix(seed, kind, layer)
                scales = scales.cpu()
                x = _host(codes)
                L.check(lib.velox_hip_mla_load_fp8(self.m, kind, layer, x.data_ptr(), scales.data_ptr(), None), "load_fp8")
            for kind in (L.MLA_NORM, L.MLA_Q_A_NORM, L.MLA_KV_A_NORM):
                x = _mla_vector(seed, kind, layer).cpu()
                L.check(lib.velox_hip_mla_load_f32(self.m, kind, layer, x.data_ptr(), x.numel(), None), "load_f32")
        h, _, _, lr, _, dr, _ = MLA
        s_cap = info.s_cap
        self.cache = self.buf[3][: layers * rows * s_cap * (lr + dr) * 2].view(torch.bfloat16).view(layers, rows, s_cap, lr + dr)
        self.pos = _positions(case)
        for layer in range(layers):
            for s, n in enumerate(self.pos):
                self.cache[layer, s, :n] = _context(case, seed, layer, s, n, (lr + dr,))
        for s, n in enumerate(self.pos):
            L.check(lib.velox_hip_mla_set_position(self.m, s, n, None), "set_position")
        off = info.hidden - a.activation_arena
        self.hidden = self.buf[4][off: off + 4 * rows * h].view(torch.float32).view(rows, h)
        self.x = _mla_hidden(case, seed)
        self.hidden.copy_(self.x)
        self.step()  # once eagerly: modules load outside the capture
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.step()
        L.check(lib.velox_hip_last_error(), "mla_decode_step")
        torch.cuda.synchronize()

    def step(self):
        self.lib.velox_hip_mla_decode_step(self.m, self.case["rows"], 1, _stream())

    def run(self):
        self.hidden.copy_(self.x)
        self.graph.replay()
        step = self.pos[0] - self.pos[1] if len(self.pos) > 1 else 0
        c = self.cache
        rows = torch.as_strided(c, (c.shape[0], c.shape[1], c.shape[3]), (c.stride(0), c.stride(1) - step * c.stride(2), 1),
                                c.storage_offset() + self.pos[0] * c.stride(2))
        return {"hidden": self.hidden, "latent": rows}

    def __del__(self):
        try:
            torch.cuda.synchronize()
            if self.m.value:
                self.lib.velox_hip_mla_destroy(self.m)
        except Exception:
            pass


def prepare(case, seed):
    return _Mla(case, seed) if case["kind"] == "mla" else _Dense(case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without ------------------------------------------------------------------

def work(case):
    if case["kind"] == "mla":
        h, nh, ql, lr, dn, dr, dv = MLA
        b = case["rows"]
        shapes = _mla_shapes()
        weights = sum(s[0] * s[1] for s in shapes.values() if len(s) == 2)
        ctx = sum(p + 1 for p in _positions(case))
        # each row: every weight once (W_kvb as its two absorbed halves), scores over lr + dr, P V over lr
        flops = case["layers"] * (2 * weights * b + 2 * nh * (2 * lr + dr) * ctx)
        return {"bytes": case["layers"] * (weights + 2 * (lr + dr) * (ctx + b)) + 8 * b * h, "flops": flops}
    w = _Weights(case, 0)
    qd, kvd = w.hq * w.d, w.hkv * w.d
    layer = w.h * (qd + 2 * kvd) + qd * w.h + 3 * w.h * w.f
    head = w.vocab * w.h
    if case["kind"] == "prefill":
        n, p0 = case["rows"], case["pos"]
        last = (n - 1) % CHUNK + 1
        pairs = n * p0 + n * (n + 1) // 2
        kv = 2 * 2 * kvd * (p0 + 2 * n)
        return {"bytes": BYTES_PER_WEIGHT[w.quant] * (w.layers * layer + head) + w.layers * kv + 4 * last * w.vocab,
                "flops": 2 * n * w.layers * layer + 2 * last * head + 4 * w.layers * qd * pairs}
    pos = _positions(case) if case["kind"] == "batch" else [case["pos"]]
    kv = sum(2 * 2 * kvd * (p + 2) for p in pos)
    return {"bytes": BYTES_PER_WEIGHT[w.quant] * (w.layers * layer + head) + w.layers * kv + 4 * len(pos) * w.vocab,
            "flops": len(pos) * 2 * (w.layers * layer + head) + 4 * w.layers * qd * sum(p + 1 for p in pos)}


def tolerance(case):
    """About four times the measured distance to exact(): 1.7e-3 for the bf16 rounding of new K/V and latent
    rows, 4.1e-3 for logits behind 32 layers or 72B-wide ones, 7.1e-3 for a prefill whose rows attend to each
    other's bf16 rows behind fp16 activations."""
    return {"rel": {"mla": 1e-2, "decode": 1.5e-2, "batch": 1.5e-2, "prefill": 2.8e-2}[case["kind"]]}


# ---- float64 ----------------------------------------------------------------------------------------

def _norm(x, gain, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * gain.double()


def _rope(x, pos, theta):
    """Rotate-half RoPE of x [rows][heads][d] at positions pos [rows]."""
    half = x.shape[-1] // 2
    freq = theta ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / x.shape[-1])
    ang = pos.double()[:, None, None] * freq
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()), -1)


def _attend(q, k, v, mask=None):
    """q [rows][hkv][g][d] over k, v [positions][hkv][d]; mask [rows][positions] False where unseen."""
    s = torch.einsum("rhgd,phd->hgrp", q, k) / math.sqrt(q.shape[-1])
    if mask is not None:
        s = s.masked_fill(~mask, float("-inf"))
    return torch.einsum("hgrp,phd->rhgd", s.softmax(-1), v).reshape(q.shape[0], -1)


def _dense_exact(case, seed):
    w = _Weights(case, seed)
    kind = case["kind"]
    g = w.hq // w.hkv
    if kind == "prefill":
        n, p0 = case["rows"], case["pos"]
        tok = _tokens(case, seed, p0 + n)[p0:]
        pos = list(range(p0, p0 + n))
    elif kind == "batch":
        pos = _positions(case)
        tok = [_tokens(case, seed, case["pos"] + WINDOW, s)[p] for s, p in enumerate(pos)]
    else:
        pos, tok = [case["pos"]], _tokens(case, seed, 1)
    posn = torch.tensor(pos, device="cuda")
    x = w.dense(L.T_EMBED, 0)[torch.tensor(tok, device="cuda")]
    rows = x.shape[0]
    ks, vs = [], []
    for layer in range(w.layers):
        def lin(t, kinds):
            out = []
            for kd, b in kinds:
                y = t @ w.dense(kd, layer).T
                out.append(y + w.vector(b, layer).double() if w.bias and b else y)
            return out
        a = _norm(x, w.vector(L.T_ATTN_NORM, layer), w.eps)
        q, k, v = lin(a, ((L.T_Q, L.T_BQ), (L.T_K, L.T_BK), (L.T_V, L.T_BV)))
        q = _rope(q.view(rows, w.hq, w.d), posn, w.theta).view(rows, w.hkv, g, w.d)
        k = _rope(k.view(rows, w.hkv, w.d), posn, w.theta)
        v = v.view(rows, w.hkv, w.d)
        if kind == "prefill":
            if p0:
                ctx = _context(case, seed, layer, 0, p0, (2, w.hkv, w.d)).double()
                kk, vv = torch.cat((ctx[:, 0], k)), torch.cat((ctx[:, 1], v))
            else:
                kk, vv = k, v
            seen = torch.arange(p0 + n, device="cuda")[None, :] <= posn[:, None]
            att = torch.cat([_attend(q[i: i + 128], kk, vv, seen[i: i + 128]) for i in range(0, n, 128)])
            ks.append(kk)
            vs.append(vv)
        else:
            out = []
            for s, p in enumerate(pos):
                kk, vv = k[s: s + 1], v[s: s + 1]
                if p:
                    ctx = _context(case, seed, layer, s, p, (2, w.hkv, w.d)).double()
                    kk, vv = torch.cat((ctx[:, 0], kk)), torch.cat((ctx[:, 1], vv))
                out.append(_attend(q[s: s + 1], kk, vv))
            att = torch.cat(out)
            ks.append(k)
            vs.append(v)
        x = x + lin(att, ((L.T_O, 0),))[0]
        a = _norm(x, w.vector(L.T_MLP_NORM, layer), w.eps)
        gate, up = lin(a, ((L.T_GATE, 0), (L.T_UP, 0)))
        x = x + lin(gate * torch.sigmoid(gate) * up, ((L.T_DOWN, 0),))[0]
    head = w.dense(L.T_EMBED if w.tied else L.T_HEAD, 0)
    if kind == "prefill":
        last = (n - 1) % CHUNK + 1
        cap = (p0 + n + 31) // 32 * 32
        k = torch.zeros((w.layers, 1, w.hkv, cap, w.d), dtype=torch.float64, device="cuda")
        for layer in range(w.layers):
            k[layer, 0, :, : p0 + n] = ks[layer].permute(1, 0, 2)
        v = torch.stack([_v_blocks(t)[None] for t in vs])
        return {"logits": _norm(x[n - last:], w.vector(L.T_FINAL_NORM, 0), w.eps) @ head.T, "k": k, "v": v}
    logits = _norm(x, w.vector(L.T_FINAL_NORM, 0), w.eps) @ head.T
    if case.get("call") == "engine":
        return {"logits": logits.view(-1)}
    # [layers][sequences][hkv][d]
    out = {"logits": logits, "k": torch.stack(ks), "v": torch.stack(vs)}
    if kind == "decode":
        out["hidden"] = x.view(-1)
    return out


def _mla_exact(case, seed):
    h, nh, ql, lr, dn, dr, dv = MLA
    eps, theta = 1e-6, 1e4
    pos = _positions(case)
    posn = torch.tensor(pos, device="cuda")
    x = _mla_hidden(case, seed).double()
    b = x.shape[0]

    def mat(kind, layer):
        codes, scales = _mla_matrix(seed, kind, layer)
        s = scales.double().repeat_interleave(128, 0)[: codes.shape[0]].repeat_interleave(128, 1)[:, : codes.shape[1]]
        return codes.double() * s

    latent = []
    for layer in range(case["layers"]):
        a = _norm(x, _mla_vector(seed, L.MLA_NORM, layer), eps)
        qa = _norm(a @ mat(L.MLA_Q_A, layer).T, _mla_vector(seed, L.MLA_Q_A_NORM, layer), eps)
        q = (qa @ mat(L.MLA_Q_B, layer).T).view(b, nh, dn + dr)
        ckr = a @ mat(L.MLA_KV_A, layer).T
        new = torch.cat((_norm(ckr[:, :lr], _mla_vector(seed, L.MLA_KV_A_NORM, layer), eps),
                         _rope(ckr[:, None, lr:], posn, theta)[:, 0]), -1)
        latent.append(new)
        kvb = mat(L.MLA_KV_B, layer).view(nh, dn + dv, lr)
        qabs = torch.einsum("bhd,hdc->bhc", q[..., :dn], kvb[:, :dn])
        qr = _rope(q[..., dn:], posn, theta)
        out = []
        for s, p in enumerate(pos):
            rows = torch.cat((_context(case, seed, layer, s, p, (lr + dr,)).double(), new[s: s + 1]))
            sc = (torch.cat((qabs[s], qr[s]), -1) @ rows.T) / math.sqrt(dn + dr)
            out.append(sc.softmax(-1) @ rows[:, :lr])
        o = torch.einsum("bhc,hvc->bhv", torch.stack(out), kvb[:, dn:]).reshape(b, nh * dv)
        x = x + o @ mat(L.MLA_O, layer).T
    return {"hidden": x, "latent": torch.stack(latent)}


def exact(case, seed):
    return _mla_exact(case, seed) if case["kind"] == "mla" else _dense_exact(case, seed)
