"""The batched prompt of the device-resident loop (prefill.hip) against the fp64 oracle, token by token.

llama2_decode_run sends all but the last of the known tokens through the layers in batches when those are
at least 8; their only results are rows of the key and value caches, which every later step
attends, so the caches and the first logits are compared.  Both paths round the same quantities to fp16 and
sum in fp32, in other orders, so over a whole cache (thousands of values) their 2-norm distances from the
oracle are two samples of the same error: the batch may be 1.5 times as far off as single steps, plus a tenth
of an fp16 rounding (1e-4) where both are nearly exact.  Where single steps are the reference, the bound is
the end-to-end bound of the small models in test_gpu_transformer.py."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import assert_close_normwise
from managedllama2_amd import capi, synth
from managedllama2_amd.transformer import Transformer

pytestmark = pytest.mark.gpu
FUSED_GRAPH = capi.DECODE_FUSED | capi.DECODE_GRAPH
TOL = 1e-2


def config(dim, hidden, layers, seq_len):
    return dict(dim=dim, hidden_dim=hidden, n_layers=layers, n_heads=dim // 128, n_kv_heads=dim // 128, vocab_size=512,
                seq_len=seq_len, rope_theta=10000.0)


def caches(t, cfg, n):
    shape = (cfg["n_layers"], cfg["seq_len"], cfg["dim"])
    return [b.to_host().reshape(shape)[:, :n] for b in (t.runstate.keyCache, t.runstate.valueCache)]


def clear_caches(t):
    """Every row NaN: what a run does not write cannot pass for what it should have written."""
    for b in (t.runstate.keyCache, t.runstate.valueCache):
        b.copy_to_device(np.full(b.size, np.nan, np.float16))


def step_by_step(cfg, model, prompt, first, history=None):
    """The same positions through single steps (what the loop did for fewer known tokens)."""
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    if history:
        t.runstate.keyCache.copy_to_device(history[0])
        t.runstate.valueCache.copy_to_device(history[1])
    t.runstate.tokens.copy_to_device(prompt, first)
    for pos in range(first, first + len(prompt)):
        t.Forward(pos, pos + 1)
    return t


# batch = known - 1: around the tile of 32 tokens and the block of 128; hidden sizes that are no multiple of a tile
# or of a group; the largest goes through in two batches
@pytest.mark.parametrize("dim,hidden,known", [(256, 640, 16), (256, 640, 17), (256, 328, 33), (384, 1000, 34),
                                              (256, 640, 65), (512, 1408, 97), (128, 136, 129), (256, 640, 130),
                                              (384, 1000, 258), (256, 328, 1060)])
def test_prompt_fills_the_caches(oracle, dim, hidden, known):
    cfg = config(dim, hidden, 2, known + 3)
    model = synth.random_model(cfg, seed=61, rms_random=True)
    prompt = synth.rng_for(801, known).integers(3, 512, known).astype(np.int32)
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    t.runstate.tokens.copy_to_device(prompt)
    capi.call("llama2_decode_run", t._decoder, 0, known, known)
    ref = step_by_step(cfg, model, prompt, 0)
    hm = oracle.HostModel(cfg, model)
    hm.tokens[:known] = prompt
    for pos in range(known):
        hm.forward(pos, pos + 1)
    shape = (cfg["n_layers"], cfg["seq_len"], dim)
    for name, g, s, w in zip("kv", caches(t, cfg, known), caches(ref, cfg, known), (hm.key_cache, hm.value_cache)):
        want = w.reshape(shape)[:, :known].astype(np.float64)
        for layer in range(cfg["n_layers"]):
            batch, steps = (float(np.linalg.norm(v[layer] - want[layer]) / np.linalg.norm(want[layer])) for v in (g, s))
            print(name, layer, "batch %.2e steps %.2e" % (batch, steps))
            assert batch <= 1.5 * steps + 1e-4, (name, layer, batch, steps)
    token = int(t.runstate.tokens.to_host(1, known)[0])
    assert token == int(np.argmax(t.runstate.logits.to_host()))
    assert np.array_equal(t.runstate.tokens.to_host(known), prompt)
    for tr in (t, ref):
        tr.close()


# The smallest batches: most of the one token tile is padding.  One known token fewer goes step by step, bit for bit.
@pytest.mark.parametrize("dim,hidden", [(128, 136), (384, 1000), (2176, 648)])
def test_shortest_batches(dim, hidden):
    cfg = config(dim, hidden, 2, 20)
    model = synth.random_model(cfg, seed=66, rms_random=True)
    prompt = synth.rng_for(806, dim).integers(3, 512, 16).astype(np.int32)
    ref = step_by_step(cfg, model, prompt, 0)
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    for known in (8, 9, 12, 15, 16):
        t.runstate.tokens.copy_to_device(prompt)
        clear_caches(t)
        capi.call("llama2_decode_run", t._decoder, 0, known, known)
        for g, w in zip(caches(t, cfg, known), caches(ref, cfg, known)):
            if known == 8:
                assert np.array_equal(g.view(np.uint16), w.view(np.uint16))
            for layer in range(cfg["n_layers"]):
                want = w[layer].astype(np.float64)
                # as in test_wide_prompt_blocks
                assert np.linalg.norm(g[layer] - want) <= 4e-3 * np.linalg.norm(want), (known, layer)
    assert_close_normwise(t.runstate.logits.to_host(), ref.runstate.logits.to_host().astype(np.float64), "logits", TOL)
    for tr in (t, ref):
        tr.close()


@pytest.mark.parametrize("first,known", [(1, 17), (63, 40), (200, 131)])
def test_prompt_behind_a_history(first, known):
    cfg = config(256, 640, 2, first + known + 2)
    model = synth.random_model(cfg, seed=62)
    rng = synth.rng_for(802, first)
    n = cfg["n_layers"] * cfg["seq_len"] * cfg["dim"]
    history = synth.normal_f16(rng, n), synth.normal_f16(rng, n)
    prompt = rng.integers(3, 512, known).astype(np.int32)
    ref = step_by_step(cfg, model, prompt, first, history)
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    t.runstate.keyCache.copy_to_device(history[0])
    t.runstate.valueCache.copy_to_device(history[1])
    t.runstate.tokens.copy_to_device(prompt, first)
    # a prompt that reaches beyond the steps asked for: every step of the call is known, nothing is generated
    capi.call("llama2_decode_run", t._decoder, first, known, first + known + 5)
    for g, w in zip(caches(t, cfg, first + known), caches(ref, cfg, first + known)):
        assert np.array_equal(g[:, :first].view(np.uint16), w[:, :first].view(np.uint16))
        assert_close_normwise(g.ravel(), w.ravel().astype(np.float64), "cache", TOL)
    assert_close_normwise(t.runstate.logits.to_host(), ref.runstate.logits.to_host().astype(np.float64), "logits", TOL)
    for tr in (t, ref):
        tr.close()


# Attention's passes shared by several workgroups per tile: as many pieces as passes (1 head), more passes than the
# 32 pieces, pieces of unequal length, a last piece that the first queries of a tile do not attend at all (128 + 33:
# timesteps 128 .. 161 in passes 2 and 3 with a tile's edge inside), two tiles per workgroup (16 heads, 1003 rows)
@pytest.mark.parametrize("dim,hidden,first,known", [(128, 136, 700, 9), (128, 136, 3000, 40), (384, 1000, 175, 33),
                                                    (384, 1000, 128, 34), (640, 648, 1111, 130), (2048, 328, 0, 1004)])
def test_attention_in_pieces(dim, hidden, first, known):
    cfg = config(dim, hidden, 2, first + known + 1)
    model = synth.random_model(cfg, seed=67)
    rng = synth.rng_for(807, dim, first)
    n = cfg["n_layers"] * cfg["seq_len"] * dim
    history = synth.normal_f16(rng, n), synth.normal_f16(rng, n)
    prompt = rng.integers(3, 512, known).astype(np.int32)
    ref = step_by_step(cfg, model, prompt, first, history)
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    t.runstate.keyCache.copy_to_device(history[0])
    t.runstate.valueCache.copy_to_device(history[1])
    t.runstate.tokens.copy_to_device(prompt, first)
    capi.call("llama2_decode_run", t._decoder, first, known, first + known)
    for g, w in zip(caches(t, cfg, first + known), caches(ref, cfg, first + known)):
        assert np.array_equal(g[:, :first].view(np.uint16), w[:, :first].view(np.uint16))
        for layer in range(cfg["n_layers"]):
            want = w[layer, first:].astype(np.float64)
            # as in test_wide_prompt_blocks
            assert np.linalg.norm(g[layer, first:] - want) <= 4e-3 * np.linalg.norm(want), layer
    assert_close_normwise(t.runstate.logits.to_host(), ref.runstate.logits.to_host().astype(np.float64), "logits", TOL)
    for tr in (t, ref):
        tr.close()


# Scores below fp16's range round to -infinity and get no weight, also where a whole pass of 64 timesteps has no
# other: 17 heads x 1003 rows go unsplit, 3 heads x 40 rows in one piece per pass.
@pytest.mark.parametrize("dim,known", [(2176, 1004), (384, 41)])
def test_scores_below_the_range_of_fp16(oracle, dim, known):
    first, heads = 64, dim // 128
    cfg = config(dim, 328, 2, first + known + 1)
    model = synth.random_model(cfg, seed=69)
    W, Z, S = model["layers"][0]["q"]
    model["layers"][0]["q"] = W, Z, S * np.float16(4)
    token = 9
    x = model["embedding"].reshape(512, dim)[token].astype(np.float64)
    x = (x / np.sqrt(np.mean(x * x) + 1e-5)).astype(np.float16)
    q = oracle.f64_matvec_int4(x, *model["layers"][0]["q"], dim, dim).reshape(heads, 2, 64)
    # keys opposite to the query in the 14 slowest pairs of RoPE, which turn by less than half a radian either way
    angle = (first + known / 2) * 10000.0 ** (-np.arange(64) / 64)
    q = np.stack([q[:, 0] * np.cos(angle) - q[:, 1] * np.sin(angle), q[:, 0] * np.sin(angle) + q[:, 1] * np.cos(angle)], 1)
    q[:, :, :50] = 0
    key = np.zeros((2, cfg["seq_len"], dim), np.float16)
    key[0, :first] = (-60000.0 * q / np.abs(q).max()).reshape(dim)
    lowest = np.sum(q * q, (1, 2)) * np.cos(0.5) * 60000.0 / np.abs(q).max() / np.sqrt(128)
    assert np.all(lowest > 70000), lowest.min()
    value = synth.normal_f16(synth.rng_for(809), key.size)
    prompt = np.full(known, token, np.int32)
    ref = step_by_step(cfg, model, prompt, first, (key.ravel(), value))
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    t.runstate.keyCache.copy_to_device(key.ravel())
    t.runstate.valueCache.copy_to_device(value)
    t.runstate.tokens.copy_to_device(prompt, first)
    capi.call("llama2_decode_run", t._decoder, first, known, first + known)
    for g, w in zip(caches(t, cfg, first + known), caches(ref, cfg, first + known)):
        assert np.all(np.isfinite(w)) and np.all(np.isfinite(g))
        want = w[1, first:].astype(np.float64)
        assert np.linalg.norm(g[1, first:] - want) <= 4e-3 * np.linalg.norm(want)  # as in test_wide_prompt_blocks
    for tr in (t, ref):
        tr.close()


# Probabilities keep fp32's precision however small they are: the first timestep has all the weight and no value, all
# others are 27.2 lower (p = 2^-39.2) and have values whose sum the residual stream, small itself, feels.  In one piece
# of the history (128) and in an unsplit launch (2176).
@pytest.mark.parametrize("dim,first,known", [(128, 64, 9), (2176, 200, 1004)])
def test_small_probabilities(oracle, dim, first, known):
    heads = dim // 128
    cfg = config(dim, 136, 2, first + known + 1)
    model = synth.random_model(cfg, seed=70)
    layer, token = model["layers"][0], 9
    layer["v"] = layer["v"][0], layer["v"][1], np.zeros_like(layer["v"][2])  # the new rows have neither keys
    layer["k"] = layer["k"][0], layer["k"][1], np.zeros_like(layer["k"][2])  # nor values: scores of 0
    layer["o"] = layer["o"][0], layer["o"][1], layer["o"][2] * np.float16(8)
    embedding = model["embedding"].reshape(512, dim)
    embedding[token] = synth.normal_f16(synth.rng_for(810), dim, 2.0 ** -14)
    x = embedding[token].astype(np.float64)
    x = (x / np.sqrt(np.mean(x * x) + 1e-5)).astype(np.float16)
    q = oracle.f64_matvec_int4(x, *layer["q"], dim, dim).reshape(heads, 2, 64)
    angle = (first + known / 2) * 10000.0 ** (-np.arange(64) / 64)  # RoPE's slowest pairs turn by 0.12 at most from here
    q = np.stack([q[:, 0] * np.cos(angle) - q[:, 1] * np.sin(angle), q[:, 0] * np.sin(angle) + q[:, 1] * np.cos(angle)], 1)
    q[:, :, :58] = 0
    unit = (q * np.sqrt(128) / np.sum(q * q, (1, 2), keepdims=True)).reshape(dim)  # a score of 1
    key = np.zeros((2, cfg["seq_len"], dim), np.float16)
    key[0, 0], key[0, 1:first] = 12 * unit, (12 - 27.2) * unit
    assert np.all(np.isfinite(key))
    value = np.zeros_like(key)
    value[0, 1:first] = 60000.0 * synth.rng_for(811).choice([-1.0, 1.0], dim)
    prompt = np.full(known, token, np.int32)
    ref = step_by_step(cfg, model, prompt, first, (key.ravel(), value.ravel()))
    none = step_by_step(cfg, model, prompt, first, (key.ravel(), np.zeros(key.size, np.float16)))
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    t.runstate.keyCache.copy_to_device(key.ravel())
    t.runstate.valueCache.copy_to_device(value.ravel())
    t.runstate.tokens.copy_to_device(prompt, first)
    capi.call("llama2_decode_run", t._decoder, first, known, first + known)
    for g, w, z in zip(*(caches(tr, cfg, first + known) for tr in (t, ref, none))):
        g, w, z = (v[1, first:].astype(np.float64) for v in (g, w, z))
        assert np.linalg.norm(z - w) >= 0.1 * np.linalg.norm(w)
        # as in test_wide_prompt_blocks
        assert np.linalg.norm(g - w) <= 4e-3 * np.linalg.norm(w), np.linalg.norm(g - w) / np.linalg.norm(w)
    for tr in (t, ref, none):
        tr.close()


# No known token whatever a negative n_prompt's distance from the position, all of them with the largest.
@pytest.mark.parametrize("run", ["llama2_decode_run", "llama2_decode_run_sampled"])
@pytest.mark.parametrize("first", [0, 1, 20])
def test_extreme_prompt_lengths(run, first):
    cfg = config(256, 640, 2, first + 21)
    model = synth.random_model(cfg, seed=68)
    prompt = synth.rng_for(808).integers(3, 512, cfg["seq_len"]).astype(np.int32)
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    sampling = (0.5, 0.9, 7) if run.endswith("sampled") else ()
    got = {}
    for n_prompt in (0, -1, -2**31, -2**31 + first, -2**31 + 30, 2**31 - 1):
        t.runstate.tokens.copy_to_device(prompt)
        capi.call(run, t._decoder, first, 20, n_prompt, *sampling)
        got[n_prompt] = t.runstate.tokens.to_host(first + 21)
    assert np.array_equal(got[2**31 - 1], prompt)
    assert not np.array_equal(got[0], prompt) and np.array_equal(got[0][:first + 1], prompt[:first + 1])
    for n_prompt in (-1, -2**31, -2**31 + first, -2**31 + 30):
        assert np.array_equal(got[n_prompt], got[0]), n_prompt
    t.close()


def test_overflowing_token_reaches_only_later_positions():
    """One token whose embedding overflows to infinities: the rows of the positions before it stay finite."""
    cfg = config(256, 640, 3, 96)
    model = synth.random_model(cfg, seed=63)
    embedding = model["embedding"].reshape(512, 256)
    embedding[7] = np.float16(np.inf)
    prompt = synth.rng_for(803).integers(8, 512, 90).astype(np.int32)
    bad = 45
    prompt[bad] = 7
    ref = step_by_step(cfg, model, prompt, 0)
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    t.runstate.tokens.copy_to_device(prompt)
    capi.call("llama2_decode_run", t._decoder, 0, 90, 90)
    for g, w in zip(caches(t, cfg, 90), caches(ref, cfg, 90)):
        assert np.array_equal(np.isfinite(g), np.isfinite(w))
        assert np.all(np.isfinite(g[:, :bad])) and not np.any(np.isfinite(g[1:, bad:]))
        assert_close_normwise(g[:, :bad].ravel(), w[:, :bad].ravel().astype(np.float64), "cache", TOL)
    for tr in (t, ref):
        tr.close()


def test_infinite_values_in_the_history():
    """Attended infinite values: the same rows of the caches end up infinite or NaN as in single steps."""
    first, known = 70, 33
    cfg = config(256, 640, 3, first + known + 1)
    model = synth.random_model(cfg, seed=71)
    rng = synth.rng_for(812)
    shape = 3, cfg["seq_len"], 256
    key, value = (synth.normal_f16(rng, int(np.prod(shape))).reshape(shape) for _ in range(2))
    value[1, 3, 5], value[1, 40, 130] = np.inf, -np.inf  # in layer 1, one per head
    prompt = rng.integers(3, 512, known).astype(np.int32)
    ref = step_by_step(cfg, model, prompt, first, (key.ravel(), value.ravel()))
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    t.runstate.keyCache.copy_to_device(key.ravel())
    t.runstate.valueCache.copy_to_device(value.ravel())
    t.runstate.tokens.copy_to_device(prompt, first)
    capi.call("llama2_decode_run", t._decoder, first, known, first + known)
    for g, w in zip(caches(t, cfg, first + known), caches(ref, cfg, first + known)):
        for same in (np.isnan, np.isposinf, np.isneginf):
            assert np.array_equal(same(g), same(w)), same
        assert np.all(np.isnan(g[2, first:])) and np.all(np.isfinite(g[:2, first:]))
        assert_close_normwise(g[:2, first:].ravel(), w[:2, first:].ravel().astype(np.float64), "cache", TOL)
    for tr in (t, ref):
        tr.close()


# Where memory is short the workspace shrinks (here to 128 and 64 rows), and without one the loop goes step by
# step as it does for short prompts, bit for bit; the decoder is never refused.
@pytest.mark.parametrize("mib", [None, "2", "1", "0"])
def test_short_of_memory(mib, monkeypatch):
    cfg = config(256, 640, 2, 420)
    model = synth.random_model(cfg, seed=72)
    prompt = synth.rng_for(813).integers(3, 512, 401).astype(np.int32)
    ref = step_by_step(cfg, model, prompt, 0)
    if mib is not None:
        monkeypatch.setenv("LLAMA2_PREFILL_MIB", mib)
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    t.runstate.tokens.copy_to_device(prompt)
    capi.call("llama2_decode_run", t._decoder, 0, 401, 401)
    for g, w in zip(caches(t, cfg, 401), caches(ref, cfg, 401)):
        assert np.array_equal(g.view(np.uint16), w.view(np.uint16)) == (mib == "0")
        for layer in range(2):
            want = w[layer].astype(np.float64)
            assert np.linalg.norm(g[layer] - want) <= 4e-3 * np.linalg.norm(want), layer  # as in test_wide_prompt_blocks
    for tr in (t, ref):
        tr.close()


def test_captured_prompt_replays():
    """The whole prompt as a graph of the caller's: every replay gives the caches of the eager call."""
    cfg = config(256, 640, 2, 64)
    model = synth.random_model(cfg, seed=64)
    prompt = synth.rng_for(804).integers(3, 512, 50).astype(np.int32)
    t = Transformer(dict(cfg), model, mode=capi.DECODE_FUSED)
    t.runstate.tokens.copy_to_device(prompt)
    capi.call("llama2_decode_run", t._decoder, 0, 52, 50)
    want = caches(t, cfg, 52), t.runstate.tokens.to_host(53)
    g = C.c_void_p()
    capi.call("llama2_graph_begin_capture")
    capi.call("llama2_decode_run", t._decoder, 0, 52, 50)
    capi.call("llama2_graph_end_capture", C.byref(g))
    for rep in range(3):
        capi.call("llama2_memset", t.runstate.keyCache.ptr, 0, 2 * 64 * 256 * 2)
        capi.call("llama2_memset", t.runstate.valueCache.ptr, 0, 2 * 64 * 256 * 2)
        t.runstate.tokens.copy_to_device(np.concatenate([prompt, np.zeros(3, np.int32)]))
        capi.call("llama2_graph_launch", g)
        assert np.array_equal(t.runstate.tokens.to_host(53), want[1]), rep
        for a, b in zip(caches(t, cfg, 52), want[0]):
            assert np.array_equal(a.view(np.uint16), b.view(np.uint16)), rep
        t.Forward(51, 52)  # the decoder's own path between the replays
    capi.call("llama2_graph_destroy", g)
    t.close()


# Widths at which some of the products take the larger blocks, K in up to 4 pieces; the pairs of a width that is an odd
# multiple of 128 do not fill the last block
@pytest.mark.parametrize("dim,hidden,known", [(1408, 328, 131), (2176, 648, 301), (2176, 648, 601), (1408, 328, 1004),
                                              (2176, 648, 1004)])
def test_wide_prompt_blocks(dim, hidden, known):
    cfg = config(dim, hidden, 2, known + 1)
    model = synth.random_model(cfg, seed=65, rms_random=True)
    prompt = synth.rng_for(805, known).integers(3, 512, known).astype(np.int32)
    ref = step_by_step(cfg, model, prompt, 0)
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    t.runstate.tokens.copy_to_device(prompt)
    capi.call("llama2_decode_run", t._decoder, 0, known, known)
    for g, w in zip(caches(t, cfg, known), caches(ref, cfg, known)):
        for layer in range(cfg["n_layers"]):
            want = w[layer].astype(np.float64)
            # two orders of the same fp32 sums, each rounded to fp16 (2^-11) between the modules
            assert np.linalg.norm(g[layer] - want) <= 4e-3 * np.linalg.norm(want), layer
            assert_close_normwise(g[layer].ravel(), want.ravel(), "cache", TOL)
    assert_close_normwise(t.runstate.logits.to_host(), ref.runstate.logits.to_host().astype(np.float64), "logits", TOL)
    for tr in (t, ref):
        tr.close()


# The widths of 7B and 13B, two layers deep (the last one leaves its attention and MLP out).  On 256 compute units the
# prompt lengths reach, in token tiles x pairs of weight tiles per workgroup:
#   QKV         11 12 14 22 24 34 44 (7B: 11, 51, 151, 76, 251, 385, 512 tokens)
#   SwiGLU      12 22 24 34 44 (11, 51, 76, 151, 251)
#   two heights SwiGLU 34 and 24 (385; 13B 321), 44 and 24 (512; 13B 1004), QKV 44 and 24 (1004)
#   o-, down-proj  11 14 22 24 34 44, K in 1 to 8 pieces (1x4: 13B, 75)
#   attention   1, 2 and 4 tiles per workgroup (11, 512, 1004), 1 to 4 pieces (11, 76, 151, 251)
@pytest.mark.parametrize("widths,lengths", [(synth.LLAMA2_7B, (11, 51, 76, 151, 251, 385, 512, 1004)),
                                            (synth.LLAMA2_13B, (75, 321, 1004))])
def test_model_widths(widths, lengths):
    cfg = dict(widths, n_layers=2, vocab_size=512, seq_len=max(lengths))
    model = synth.random_model(cfg, seed=73, rms_random=True)
    for layer in model["layers"]:
        # scores of ordinary size: with the scales as drawn they reach hundreds, where ONE fp16 rounding of a score
        # moves its probability by a quarter and single rows say nothing
        for name in ("q", "k"):
            layer[name] = layer[name][:2] + (layer[name][2] * np.float16(0.25),)
    prompt = synth.rng_for(814).integers(3, 512, max(lengths)).astype(np.int32)
    ref = step_by_step(cfg, model, prompt, 0)
    want = [v.astype(np.float64) for v in caches(ref, cfg, max(lengths))]
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    for known in lengths:
        t.runstate.tokens.copy_to_device(prompt)
        clear_caches(t)
        capi.call("llama2_decode_run", t._decoder, 0, known, known)
        for name, g, w in zip("kv", caches(t, cfg, known), want):
            for layer in range(2):
                d = g[layer].astype(np.float64) - w[layer, :known]
                # the whole as in test_wide_prompt_blocks; a row by itself (a misplaced tile) by the 7 roundings to fp16
                # between a layer's rows and the next one's, each off by 2^-11 at most, doubled on the way by the MLP
                rows = np.linalg.norm(d, axis=1) / np.linalg.norm(w[layer, :known], axis=1)
                print(known, name, layer, "%.2e, worst row %.2e" % (np.sqrt(np.mean(rows * rows)), rows.max()))
                assert np.linalg.norm(d) <= 4e-3 * np.linalg.norm(w[layer, :known]), (known, name, layer)
                assert rows.max() <= 14 * 2.0 ** -11, (known, name, layer, int(rows.argmax()), rows.max())
    assert_close_normwise(t.runstate.logits.to_host(), ref.runstate.logits.to_host().astype(np.float64), "logits", TOL)
    for tr in (t, ref):
        tr.close()


# Products around the sizes at which workgroups come in two heights, on 256 compute units: 3 and 2 token tiles, 4 and 3, of SwiGLU and of
# QKV (dim 4352: QKV 4 and 3; 4352 hidden and dim 2816 keep one height); row by row as above.
@pytest.mark.parametrize("dim,hidden,known", [(1024, 4352, 950), (1024, 5376, 740), (1024, 6400, 950), (2816, 256, 950),
                                              (3456, 256, 740), (4352, 256, 950)])
def test_workgroups_of_two_heights(dim, hidden, known):
    test_model_widths(config(dim, hidden, 2, known), (known,))


# A row's sums do not depend on how many rows are with it, as long as a step takes one group of K and K comes in the same pieces: the
# same rows in a batch whose QKV or SwiGLU has workgroups of two heights and in one that has one height, bit for
# bit.  (product, dim, hidden, rows with two heights, rows with one); tests/test_prompt_product_shapes.py holds them to that.
TWO_HEIGHTS = [("qkv", 2816, 256, 991, 960), ("qkv", 3456, 256, 750, 800), ("qkv", 4352, 256, 930, 890),
               ("swiglu", 2304, 4224, 992, 920), ("swiglu", 2304, 6272, 915, 990), ("swiglu", 3200, 5248, 700, 670)]


@pytest.mark.parametrize("product,dim,hidden,two,one", TWO_HEIGHTS)
def test_two_heights_equal_one_bit_for_bit(product, dim, hidden, two, one):
    layers = 1 if product == "qkv" else 2  # the last layer ends with its cache rows
    cfg = config(dim, hidden, layers, max(two, one) + 1)
    model = synth.random_model(cfg, seed=77, rms_random=True)
    prompt = synth.rng_for(817, dim).integers(3, 512, max(two, one) + 1).astype(np.int32)
    t, got = Transformer(dict(cfg), model, mode=FUSED_GRAPH), []
    for rows in (two, one):
        t.runstate.tokens.copy_to_device(prompt)
        clear_caches(t)
        capi.call("llama2_decode_run", t._decoder, 0, rows + 1, rows + 1)
        got.append(caches(t, cfg, min(two, one)))
    for name, a, b in zip("kv", *got):
        assert np.all(np.isfinite(a)) and np.array_equal(a.view(np.uint16), b.view(np.uint16)), name
    t.close()


# The other loops that batch their prompt: sampling, and the persistent step (same bits as the launch sequence behind
# the same batch).
def test_sampled_run_behind_a_batch():
    cfg, known, steps, seed = config(256, 640, 2, 64), 41, 60, 99
    model = synth.random_model(cfg, seed=74)
    prompt = synth.rng_for(815).integers(3, 512, known).astype(np.int32)
    ref = step_by_step(cfg, model, prompt, 0)
    t = Transformer(dict(cfg), model, mode=FUSED_GRAPH)
    clear_caches(t)
    t.runstate.tokens.copy_to_device(prompt)
    capi.call("llama2_decode_run_sampled", t._decoder, 0, steps, known, 0.7, 0.9, seed)
    for g, w in zip(caches(t, cfg, known), caches(ref, cfg, known)):
        for layer in range(cfg["n_layers"]):
            want = w[layer].astype(np.float64)
            assert np.linalg.norm(g[layer] - want) <= 4e-3 * np.linalg.norm(want), layer  # as in test_wide_prompt_blocks
    tokens = t.runstate.tokens.to_host(steps + 1)
    assert np.array_equal(tokens[:known], prompt) and len(set(tokens[known:].tolist())) > 4
    token = C.c_int()
    for pos in range(known - 1, steps):  # the steps behind the batch again, one by one, with the same coins
        t.Forward(pos, pos + 1)
        coin = float(capi.load().llama2_sampler_coin(seed, pos + 1))
        capi.call("llama2_decode_sample_top_p", t._decoder, pos + 1, 1, 0.7, 0.9, coin, C.byref(token))
        assert token.value == tokens[pos + 1], pos
    for tr in (t, ref):
        tr.close()


def test_persistent_run_behind_a_batch():
    cfg, known, steps = config(256, 640, 2, 64), 41, 60
    model = synth.random_model(cfg, seed=75)
    prompt = synth.rng_for(816).integers(3, 512, known).astype(np.int32)
    ref = step_by_step(cfg, model, prompt, 0)
    got = []
    for mode in (capi.DECODE_FUSED | capi.DECODE_PERSISTENT, FUSED_GRAPH | capi.DECODE_PERSISTENT, FUSED_GRAPH):
        t = Transformer(dict(cfg), model, mode=mode)
        clear_caches(t)
        t.runstate.tokens.copy_to_device(prompt)
        capi.call("llama2_decode_run", t._decoder, 0, steps, known)
        capi.call("llama2_decode_check", t._decoder)
        got.append([v.view(np.uint16) for v in caches(t, cfg, steps)] + [t.runstate.tokens.to_host(steps + 1)])
        t.close()
    for g, w in zip(got[2], caches(ref, cfg, known)):
        for layer in range(cfg["n_layers"]):
            want = w[layer].astype(np.float64)
            d = g.view(np.float16)[layer, :known] - want
            assert np.linalg.norm(d) <= 4e-3 * np.linalg.norm(want), layer  # as in test_wide_prompt_blocks
    for other in got[:2]:
        for a, b in zip(other, got[2]):
            assert np.array_equal(a, b)
    ref.close()
