"""What this framework is used for, as cases that can be timed and compared.

Every case goes through the public entry points (the C ABI of libllama2_hip.so through
managedllama2_amd.capi, or managedllama2_amd.transformer.Transformer) at the shapes of the
repository's own configurations (synth.LLAMA2_7B, synth.LLAMA2_13B, the small models of the tests).

kind "loop"    llama2_decode_run / llama2_decode_run_sampled: the device-resident token loop.  Positions
               below `prompt` take their token from the prompt, later ones generate.
kind "host"    llama2_decode_forward + llama2_decode_sample_top_p per token, the token read back each
               time: a host that drives the loop itself (Transformer.Generate, a server that streams).
kind "small"   Transformer.Generate of a small model: launches and host work, no bandwidth.
kind "set"     the int4 mat-vec modules of a stack of decoder layers, replayed as a captured graph.
kind "sample"  llama2_sample on a vector of logits: softmax, sort, prefix sums, pick.
kind "repack"  the converter's tensor repack of one AWQ tensor (weights, zero points, scales).

Weights are random but have a trained model's orders of magnitude: weight std about 0.02 (4-bit steps
of 0.002 .. 0.008 around zero points of 6 .. 9), and a classifier whose rows lean towards the embedding
of one preceding token, so that the greedy choice has a margin of a few logits, as it has in a trained
model, instead of being a tie-break among 32000 independent normal numbers.
"""
import ctypes as C
import math

import numpy as np
import torch

from managedllama2_amd import capi, synth
from managedllama2_amd.device import init
from managedllama2_amd.transformer import Transformer

MODELS = {"7b": synth.LLAMA2_7B, "13b": synth.LLAMA2_13B}
EMBEDDING_STD = 4.0  # next to layers that each add a few units to the residual stream
MODES = {"modules": capi.DECODE_MODULES, "fused_graph": capi.DECODE_FUSED | capi.DECODE_GRAPH}


def listed():
    return [
        # the repository's own decode benchmark: a 128-token prompt, 256 greedy tokens
        dict(name="generate_128_256", kind="loop", model="7b", position=0, prompt=128, steps=383, seq_len=512,
             temperature=0.0, top_p=0.9),
        # a document to be read before the first token of the answer appears
        dict(name="prompt_512", kind="loop", model="7b", position=0, prompt=512, steps=512, seq_len=1024,
             temperature=0.0, top_p=0.9),
        # a long question with a short answer; lengths as they come
        dict(name="prompt_1003_answer_24", kind="loop", model="7b", position=0, prompt=1003, steps=1026, seq_len=2048,
             temperature=0.0, top_p=0.9),
        # the next turn of a conversation: 75 new prompt tokens behind 600 rows of history, 16 tokens of answer
        dict(name="next_turn_75_13b", kind="loop", model="13b", position=600, prompt=675, steps=90, seq_len=1024,
             temperature=0.0, top_p=0.9),
        # generation deep inside a 4096-row context: the cache weighs as much as the weights
        dict(name="late_context", kind="loop", model="7b", position=3971, prompt=0, steps=12, seq_len=4096,
             temperature=0.0, top_p=0.9),
        # the larger model, ordinary context, greedy
        dict(name="decode_13b", kind="loop", model="13b", position=701, prompt=0, steps=12, seq_len=1024,
             temperature=0.0, top_p=0.9),
        # sampling with the reference's default parameters on the device
        dict(name="sampled_loop", kind="loop", model="7b", position=255, prompt=0, steps=16, seq_len=512,
             temperature=0.5, top_p=0.9),
        # the first tokens of an answer, streamed to a client one by one
        dict(name="host_loop", kind="host", model="7b", mode="fused_graph", position=37, steps=6, seq_len=256,
             temperature=0.0, top_p=0.9),
        # a host that keeps the reference's Forward: every module a launch of its own
        dict(name="module_loop", kind="host", model="7b", mode="modules", position=300, steps=2, seq_len=512,
             temperature=0.0, top_p=0.9),
        # a small model end to end through the Python host
        dict(name="small_model", kind="small", dim=512, hidden_dim=1408, n_layers=3, n_heads=4, vocab_size=1000,
             prompt=7, steps=24),
        # the mat-vec modules alone, weights cold (the repository's headline figure)
        dict(name="mat_vec_set", kind="set", model="7b", layers=8),
        # the sampler modules on a whole vocabulary
        dict(name="sample_32000", kind="sample", size=32000, temperature=0.5, top_p=0.9),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["loop", "loop", "loop", "turn", "sampled", "host", "small", "set", "sample", "repack"])
    if kind == "loop":  # prompt and answer from the start of a context
        prompt, answer = _log_int(rng, 2, 900), _log_int(rng, 1, 120)
        return dict(kind="loop", model="7b", position=0, prompt=prompt, steps=prompt + answer - 1,
                    seq_len=rng.choice([1024, 2048]), temperature=0.0, top_p=0.9)
    if kind == "turn":  # somewhere in a context: new prompt tokens (perhaps none), then generation
        position = _log_int(rng, 8, 3600)
        fresh = rng.choice([0, 0, _log_int(rng, 2, 400)])
        return dict(kind="loop", model=rng.choice(["7b", "13b"]), position=position,
                    prompt=position + fresh if fresh else 0, steps=fresh + rng.randint(3, 16), seq_len=4096,
                    temperature=0.0, top_p=0.9)
    if kind == "sampled":
        position = _log_int(rng, 8, 3000)
        return dict(kind="loop", model="7b", position=position, prompt=0, steps=rng.randint(4, 16), seq_len=4096,
                    temperature=round(rng.uniform(0.3, 0.9), 2), top_p=round(rng.uniform(0.5, 0.95), 2))
    if kind == "host":
        mode = rng.choice(["fused_graph", "fused_graph", "modules"])
        return dict(kind="host", model=rng.choice(["7b", "13b"]), mode=mode, position=_log_int(rng, 1, 2000),
                    steps=rng.randint(1, 6), seq_len=2048, temperature=0.0, top_p=0.9)
    if kind == "small":
        heads = rng.randint(2, 8)
        return dict(kind="small", dim=128 * heads, hidden_dim=8 * rng.randint(40, 350), n_layers=rng.randint(1, 6),
                    n_heads=heads, vocab_size=rng.randint(300, 8000), prompt=_log_int(rng, 2, 60),
                    steps=rng.randint(61, 100))
    if kind == "set":
        return dict(kind="set", model=rng.choice(["7b", "13b"]), layers=rng.randint(4, 8))
    if kind == "sample":
        return dict(kind="sample", size=_log_int(rng, 500, 65536), temperature=round(rng.uniform(0.3, 1.2), 2),
                    top_p=rng.choice([0.5, 0.9, 0.95, 1.0]))
    return dict(kind="repack", height=128 * rng.randint(16, 108), width=8 * rng.randint(64, 1728))


# ---------------------------------------------------------------- a model on the GPU

class _Arena:
    """One allocation that hands out 256-byte aligned windows, in the order TransformerWeights fills its own."""

    def __init__(self, nbytes):
        self.buffer = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        self.used = 0

    def take(self, nbytes):
        view = self.buffer[self.used:self.used + nbytes]
        self.used += (nbytes + 255) // 256 * 256
        return view


def _qweight_nbytes(K, N):
    ws, ss, zs = synth.qweight_sizes(K)
    return sum((n + 255) // 256 * 256 for n in (N * ws * 4, N * zs * 4, N * ss * 2))


def _qweight(arena, gen, K, N):
    ws, ss, zs = synth.qweight_sizes(K)
    w = arena.take(N * ws * 4).random_(0, 256, generator=gen)
    z = arena.take(N * zs * 4).random_(6, 10, generator=gen)
    z += 16 * torch.randint(6, 10, z.shape, dtype=torch.uint8, device="cuda", generator=gen)
    s = arena.take(N * ss * 2).view(torch.float16).uniform_(0.002, 0.008, generator=gen)
    return capi.QWeight(w.data_ptr(), z.data_ptr(), s.data_ptr())


def _qkvo_up_gate_down(cfg):
    dim, hidden = cfg["dim"], cfg["hidden_dim"]
    return ((dim, dim),) * 4 + ((dim, hidden),) * 2 + ((hidden, dim),)


def _generator(seed, salt):
    return torch.Generator("cuda").manual_seed((int(seed) * 1000003 + salt) % (1 << 62))


class _Model:
    """Weights, run state and decoder of a model, made on the GPU from the seed."""

    def __init__(self, cfg, seq_len, mode, seed):
        init(0)
        gen = _generator(seed, 1)
        cfg = dict(cfg, seq_len=seq_len)
        dim, hidden, L, vocab = cfg["dim"], cfg["hidden_dim"], cfg["n_layers"], cfg["vocab_size"]
        self.cfg = cfg
        per_layer = sum(_qweight_nbytes(K, N) for K, N in _qkvo_up_gate_down(cfg)) + 2 * (2 * dim + 256)
        self.arena = _Arena(2 * (vocab * dim * 2 + 256) + 2 * dim + 256 + L * per_layer)
        take = self.arena.take
        embedding = take(vocab * dim * 2).view(torch.float16).normal_(0.0, EMBEDDING_STD, generator=gen)
        classifier = take(vocab * dim * 2).view(torch.float16).normal_(0.0, 0.004, generator=gen)
        follows = torch.randperm(vocab, device="cuda", generator=gen)
        classifier.view(vocab, dim)[follows] += embedding.view(vocab, dim) * (0.02 / EMBEDDING_STD)
        rms_final = take(dim * 2).view(torch.float16).fill_(1.0)
        self.layers = (capi.LayerWeights * L)()
        for i in range(L):
            q, k, v, o, up, gate, down = (_qweight(self.arena, gen, K, N) for K, N in _qkvo_up_gate_down(cfg))
            rms = [take(dim * 2).view(torch.float16).fill_(1.0) for _ in range(2)]
            self.layers[i] = capi.LayerWeights(q, k, v, o, gate, up, down, rms[0].data_ptr(), rms[1].data_ptr())
        self.weights = capi.TransformerWeights(embedding.data_ptr(), classifier.data_ptr(), rms_final.data_ptr(),
                                               self.layers)
        half = dict(dtype=torch.float16, device="cuda")
        self.buffers = [torch.zeros(n, **half) for n in (dim, dim, hidden, dim, cfg["n_heads"] * max(dim, seq_len))]
        self.logits = torch.zeros(vocab, **half)
        self.key = torch.empty(L, seq_len, dim, **half).normal_(0.0, 1.5, generator=gen)
        self.value = torch.empty(L, seq_len, dim, **half).normal_(0.0, 1.5, generator=gen)
        self.tokens = torch.randint(3, vocab, (seq_len + 1,), dtype=torch.int32, device="cuda", generator=gen)
        self.indices = torch.zeros(vocab, dtype=torch.int32, device="cuda")
        state = capi.RunState(*[b.data_ptr() for b in self.buffers], self.logits.data_ptr(), self.key.data_ptr(),
                              self.value.data_ptr(), self.tokens.data_ptr(), self.indices.data_ptr())
        config = capi.Config(*[cfg[k] for k in ("dim", "hidden_dim", "n_layers", "n_heads", "n_kv_heads", "vocab_size",
                                                "seq_len", "rope_theta")])
        torch.cuda.synchronize()
        self.decoder = C.c_void_p()
        capi.call("llama2_decode_create", C.byref(self.decoder), C.byref(config), C.byref(self.weights),
                  C.byref(state), MODES[mode])

    def __del__(self):
        if getattr(self, "decoder", None):
            capi.raw("llama2_decode_destroy", self.decoder)
            self.decoder = None

    def outputs(self):
        return dict(tokens=self.tokens, logits=self.logits, key=self.key, value=self.value)


# ---------------------------------------------------------------- prepare and run, kind by kind

def _prepare_loop(case, seed):
    return _Model(MODELS[case["model"]], case["seq_len"], "fused_graph", seed)


def _run_loop(case, m):
    if case["temperature"] == 0.0:
        capi.call("llama2_decode_run", m.decoder, case["position"], case["steps"], case["prompt"])
    else:
        capi.call("llama2_decode_run_sampled", m.decoder, case["position"], case["steps"], case["prompt"],
                  case["temperature"], case["top_p"], 20240607)
    return m.outputs()


def _prepare_host(case, seed):
    return _Model(MODELS[case["model"]], case["seq_len"], case["mode"], seed)


def _run_host(case, m):
    tok, got = C.c_int(), []
    for pos in range(case["position"], case["position"] + case["steps"]):
        capi.call("llama2_decode_forward", m.decoder, pos, pos + 1)
        capi.call("llama2_decode_sample_top_p", m.decoder, pos + 1, 1, case["temperature"], case["top_p"], 0.5,
                  C.byref(tok))
        got.append(tok.value)
    return dict(m.outputs(), streamed=np.array(got, np.int32))


def _prepare_small(case, seed):
    cfg = dict(dim=case["dim"], hidden_dim=case["hidden_dim"], n_layers=case["n_layers"], n_heads=case["n_heads"],
               n_kv_heads=case["n_heads"], vocab_size=case["vocab_size"], seq_len=128, rope_theta=10000.0)
    model = synth.random_model(cfg, seed=seed)
    dim, vocab = case["dim"], case["vocab_size"]
    rng = synth.rng_for(seed, 2)
    embedding = synth.normal_f16(rng, vocab * dim, EMBEDDING_STD)
    classifier = synth.normal_f16(rng, vocab * dim, 0.004).reshape(vocab, dim)
    classifier[rng.permutation(vocab)] += embedding.reshape(vocab, dim) * np.float16(0.02 / EMBEDDING_STD)
    model["embedding"], model["classifier"] = embedding, classifier.ravel()
    for layer in model["layers"]:
        for name in ("q", "k", "v", "o", "gate", "up", "down"):
            W, Z, S = layer[name]
            Z = (Z & np.uint32(0x11111111)) + np.uint32(0x77777777)
            layer[name] = (W, Z, (S.astype(np.float32) * 0.4).astype(np.float16))
    t = Transformer(cfg, model, mode=MODES["fused_graph"])
    return t, [int(v) for v in rng.integers(3, vocab, case["prompt"])]


def _run_small(case, state):
    t, prompt = state
    tokens = list(t.Generate(prompt, case["steps"], stop_on_special=False))
    rs = t.runstate
    return dict(tokens=np.array(tokens, np.int32), logits=rs.logits.to_host())


def _prepare_set(case, seed):
    init(0)
    cfg, gen = MODELS[case["model"]], _generator(seed, 3)
    dim, hidden, L = cfg["dim"], cfg["hidden_dim"], case["layers"]
    arena = _Arena(L * sum(_qweight_nbytes(K, N) for K, N in _qkvo_up_gate_down(cfg)))
    layers = [[_qweight(arena, gen, K, N) for K, N in _qkvo_up_gate_down(cfg)] for _ in range(L)]
    half = dict(dtype=torch.float16, device="cuda")
    xb = torch.empty(dim, **half).normal_(generator=gen)
    x0 = torch.empty(dim, **half).normal_(generator=gen)
    x = torch.zeros(dim, **half)
    q, k, v = (torch.zeros(L, dim, **half) for _ in range(3))
    h = torch.zeros(L, hidden, **half)
    (ws, ss, zs), (hws, hss, hzs) = synth.qweight_sizes(dim), synth.qweight_sizes(hidden)
    torch.cuda.synchronize()

    def calls():
        capi.call("llama2_memcpy_d2d", x.data_ptr(), x0.data_ptr(), 2 * dim)
        for i, (wq, wk, wv, wo, wu, wg, wd) in enumerate(layers):
            capi.call("llama2_qkv_mat_vec", q[i].data_ptr(), k[i].data_ptr(), v[i].data_ptr(), xb.data_ptr(),
                      *_parts(wq), *_parts(wk), *_parts(wv), dim, dim, zs, ss, ws)
            capi.call("llama2_mat_vec_residual_int4", x.data_ptr(), xb.data_ptr(), *_parts(wo), dim, dim, zs, ss, ws)
            capi.call("llama2_mat_vec_swiglu", h[i].data_ptr(), xb.data_ptr(), *_parts(wg), *_parts(wu), dim, hidden,
                      zs, ss, ws)
            capi.call("llama2_mat_vec_residual_int4", x.data_ptr(), h[i].data_ptr(), *_parts(wd), hidden, dim, hzs, hss,
                      hws)

    return _Graph(calls, arena, xb, x0, (x, q, k, v, h))


def _parts(qw):
    return qw.weight, qw.zeros, qw.scales


class _Graph:
    def __init__(self, calls, *keep):
        self.keep, self.out = keep, keep[-1]
        self.graph = C.c_void_p()
        capi.call("llama2_graph_begin_capture")
        calls()
        capi.call("llama2_graph_end_capture", C.byref(self.graph))

    def __del__(self):
        if self.graph:
            capi.raw("llama2_graph_destroy", self.graph)
            self.graph = None


def _run_set(case, g):
    capi.call("llama2_graph_launch", g.graph)
    return g.out


def _prepare_sample(case, seed):
    init(0)
    gen, n = _generator(seed, 4), case["size"]
    padded = (n + 7) // 8 * 8  # whole 16-byte pieces for the copy
    source = torch.empty(padded, dtype=torch.float16, device="cuda").normal_(0.0, 2.0, generator=gen)
    logits = torch.zeros(padded, dtype=torch.float16, device="cuda")
    indices = torch.zeros(padded, dtype=torch.int32, device="cuda")
    token = torch.zeros(4, dtype=torch.int32, device="cuda")
    coin = float(np.float32(np.random.default_rng(seed).random()))
    torch.cuda.synchronize()
    return source, logits, indices, token, coin


def _run_sample(case, state):
    source, logits, indices, token, coin = state
    capi.call("llama2_memcpy_d2d", logits.data_ptr(), source.data_ptr(), logits.numel() * 2)  # the logits of this step
    capi.call("llama2_sample", logits.data_ptr(), indices.data_ptr(), case["size"], case["temperature"], case["top_p"],
              coin, token.data_ptr(), 1)
    return token, logits, indices


def _prepare_repack(case, seed):
    init(0)
    gen, K, N = _generator(seed, 5), case["height"], case["width"]
    ws, ss, zs = synth.qweight_sizes(K)
    # AWQ "GEMM" format: [K][N / 8] words, [K / 128][N / 8] words, [K / 128][N] scales
    ins = [torch.empty(n, dtype=torch.uint8, device="cuda").random_(0, 256, generator=gen) for n in (K * N // 2, ss * N // 2)]
    scales = torch.empty(ss * N, dtype=torch.float16, device="cuda").uniform_(0.002, 0.02, generator=gen)
    outs = [torch.zeros(n, dtype=torch.int32, device="cuda") for n in ((K // 8) * N, zs * N)]
    out_scales = torch.zeros(ss * N, dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    return ins, scales, outs, out_scales


def _run_repack(case, state):
    ins, scales, outs, out_scales = state
    K, N = case["height"], case["width"]
    ss = (K + 127) // 128
    capi.call("llama2_repack_qdata", outs[0].data_ptr(), ins[0].data_ptr(), K, N)
    capi.call("llama2_repack_qdata", outs[1].data_ptr(), ins[1].data_ptr(), ss, N)
    capi.call("llama2_repack_scales", out_scales.data_ptr(), scales.data_ptr(), ss, N)
    return outs[0], outs[1], out_scales


_KINDS = {"loop": (_prepare_loop, _run_loop), "host": (_prepare_host, _run_host), "small": (_prepare_small, _run_small),
          "set": (_prepare_set, _run_set), "sample": (_prepare_sample, _run_sample),
          "repack": (_prepare_repack, _run_repack)}


def prepare(case, seed):
    return case, _KINDS[case["kind"]][0](case, seed)


def run(state):
    case, held = state
    return _KINDS[case["kind"]][1](case, held)


# ---------------------------------------------------------------- what a pass cannot do without

def _decode_work(cfg, position, prompt, steps):
    """Tokens known beforehand share one reading of the weights; every generated token needs one of its own."""
    dim, hidden, L, vocab = cfg["dim"], cfg["hidden_dim"], cfg["n_layers"], cfg["vocab_size"]
    tensors = _qkvo_up_gate_down(cfg)
    weights = L * (sum(synth.qweight_bytes(K, N) for K, N in tensors) + 4 * dim) + 2 * dim
    classifier = 2 * vocab * dim
    row = L * 2 * dim * 2  # one position of both caches
    layer_macs = L * sum(K * N for K, N in tensors)
    known = min(steps, max(0, prompt - position))
    nbytes = flops = 0
    if known:
        nbytes += weights + classifier + row * (position + known)
        flops += 2 * layer_macs * known + 4 * L * dim * known * (position + (known + 1) // 2) + 2 * vocab * dim
    for pos in range(position + known, position + steps):
        nbytes += weights + classifier + row * (pos + 1)
        flops += 2 * layer_macs + 4 * L * dim * (pos + 1) + 2 * vocab * dim
    return nbytes, flops


def work(case):
    kind = case["kind"]
    if kind == "loop":
        nbytes, flops = _decode_work(MODELS[case["model"]], case["position"], case["prompt"], case["steps"])
    elif kind == "host":
        nbytes, flops = _decode_work(MODELS[case["model"]], case["position"], 0, case["steps"])
    elif kind == "small":
        cfg = {k: case[k] for k in ("dim", "hidden_dim", "n_layers", "vocab_size")}
        nbytes, flops = _decode_work(cfg, 0, case["prompt"], case["steps"])
    elif kind == "set":
        cfg = MODELS[case["model"]]
        nbytes = case["layers"] * synth.layer_matvec_set_bytes(cfg["dim"], cfg["hidden_dim"])["total"]
        flops = case["layers"] * 2 * sum(K * N for K, N in _qkvo_up_gate_down(cfg))
    elif kind == "sample":
        nbytes, flops = case["size"] * (2 + 2 + 4), case["size"] * 8
    else:
        K, N = case["height"], case["width"]
        nbytes, flops = 2 * (K * N // 2 + (K // 128) * N // 2 + (K // 128) * N * 2), 0
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("sample", "repack"):
        return "exact"  # integers, and sums and divisions whose order and rounding the modules fix
    if kind == "set":
        return {"rel": 4e-4, "max": 1e-2}  # fp16 results of fp32 sums
    # A decode step stores fp16 between the modules, and a rounding that falls the other way travels through all
    # later layers: the module sequence and the fused step (which differ in the attention arithmetic alone) are
    # 6e-3 apart in the logits and 3e-3 in the caches of 32 layers, 3.5e-2 in the single value furthest off.
    return {"rel": 2.5e-2, "max": 0.15, "differ": 0.0}
