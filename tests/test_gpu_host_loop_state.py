"""A host's sampling call leaves the state of the next position's step on the device, so that the forward call for
that position need not set it.  Every other call in between -- another position, the device-resident loop, a graph the caller
captured -- has to set it again, and a recorded step sets its own: each step's logits and cache rows are compared with those of a decoder that never sampled."""
import ctypes as C

import numpy as np
import pytest

from managedllama2_amd import capi, synth
from managedllama2_amd.transformer import Transformer

pytestmark = pytest.mark.gpu
CFG = dict(dim=256, hidden_dim=640, n_layers=2, n_heads=2, n_kv_heads=2, vocab_size=1000, seq_len=48, rope_theta=10000.0)


@pytest.mark.parametrize("temperature", [0.0, 0.7])
@pytest.mark.parametrize("mode", [capi.DECODE_MODULES, capi.DECODE_FUSED, capi.DECODE_FUSED | capi.DECODE_GRAPH])
def test_steps_in_any_order(mode, temperature):
    model = synth.random_model(CFG, seed=91)
    t, ref = (Transformer(dict(CFG), model, mode=mode, temperature=temperature, random=lambda: 0.37) for _ in range(2))
    other = Transformer(dict(CFG), model, mode=mode, temperature=temperature, random=lambda: 0.61)
    tokens = synth.rng_for(971).integers(3, 1000, CFG["seq_len"]).astype(np.int32)
    for x in (t, ref, other):
        x.runstate.tokens.copy_to_device(tokens)

    def check(pos):
        t.Forward(pos, pos + 1)
        ref.runstate.tokens.copy_to_device(t.runstate.tokens.to_host(CFG["seq_len"]))
        ref.runstate.keyCache.copy_to_device(t.runstate.keyCache.to_host())
        ref.runstate.valueCache.copy_to_device(t.runstate.valueCache.to_host())
        ref.Forward(pos, pos + 1)
        for a, b in ((t.runstate.logits, ref.runstate.logits), (t.runstate.keyCache, ref.runstate.keyCache),
                     (t.runstate.valueCache, ref.runstate.valueCache)):
            assert np.array_equal(a.to_host().view(np.uint16), b.to_host().view(np.uint16)), pos

    def sample(nxt, generate=True):
        got = t.Sample(nxt, generate)
        if nxt < CFG["seq_len"]:
            assert got == int(t.runstate.tokens.to_host(1, nxt)[0])
        if temperature == 0.0 and generate:
            assert got == int(np.argmax(t.runstate.logits.to_host()))
        elif not generate:
            assert got == int(tokens[nxt])
        return got

    check(0), sample(1, False), check(1), sample(2), check(2)  # the next position
    sample(3), check(7), check(3)                              # another one
    sample(4), sample(4), check(4), check(4)                   # twice
    sample(5), other.Forward(9, 10), other.Sample(10, True), check(5)  # another decoder
    sample(6), capi.call("llama2_decode_run", t._decoder, 20, 3, 0), check(6)  # the device-resident loop
    sample(7), capi.call("llama2_decode_run_sampled", t._decoder, 24, 3, 0, 0.7, 0.9, 5), check(7), sample(8), check(8)
    check(46), sample(47), check(47), sample(48), check(0)     # the last row of the context
    graph = C.c_void_p()
    capi.call("llama2_graph_begin_capture")
    capi.call("llama2_decode_forward", t._decoder, 30, 31)
    assert capi.raw("llama2_decode_sample", t._decoder, 31, 1, C.byref(C.c_int())) == capi.ERR_INVALID_ARGUMENT
    capi.call("llama2_graph_end_capture", C.byref(graph))
    for pos in (9, 10, 11):
        sample(pos)
        capi.call("llama2_graph_launch", graph)
        check(pos)
    capi.call("llama2_graph_destroy", graph)
    for x in (t, ref, other):
        x.close()


@pytest.mark.parametrize("loop", [False, True])
def test_a_caller_that_captures_the_stream_itself(loop):
    """llama2_stream() may be captured with the runtime's own calls: what is recorded sets its own state, and the
    replays count like those of a graph of the library."""
    model = synth.random_model(CFG, seed=92)
    t, ref = (Transformer(dict(CFG), model, mode=capi.DECODE_FUSED) for _ in range(2))
    tokens = synth.rng_for(972).integers(3, 1000, CFG["seq_len"]).astype(np.int32)
    for x in (t, ref):
        x.runstate.tokens.copy_to_device(tokens)
        for pos in range(12):
            x.Forward(pos, pos + 1)
    want = {}
    for pos in (9, 10):
        ref.Forward(pos, pos + 1)
        want[pos] = ref.runstate.logits.to_host().view(np.uint16)
    def logits_are_those_of(pos):
        return np.array_equal(t.runstate.logits.to_host().view(np.uint16), want[pos])

    lib = capi.load()
    stream = C.c_void_p(lib.llama2_stream())
    graph, replay = C.c_void_p(), C.c_void_p()

    t.Forward(9, 10), t.Sample(10, False)  # leaves the state of position 10
    assert lib.hipStreamBeginCapture(stream, 1) == 0  # of this thread
    if loop:
        capi.call("llama2_decode_run", t._decoder, 9, 1, 11)
    else:
        capi.call("llama2_decode_forward", t._decoder, 10, 11)
    assert lib.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert lib.hipGraphInstantiate(C.byref(replay), graph, None, None, 0) == 0
    for _ in range(3):
        t.Forward(3, 4), t.Sample(4, False)
        assert lib.hipGraphLaunch(replay, stream) == 0
        assert logits_are_those_of(9 if loop else 10)
        t.Forward(8, 9), t.Sample(9, False)  # leaves the state of position 9 ...
        assert lib.hipGraphLaunch(replay, stream) == 0  # ... which is gone then
        t.Forward(9, 10)
        assert logits_are_those_of(9)
    assert lib.hipGraphExecDestroy(replay) == 0 and lib.hipGraphDestroy(graph) == 0
    for x in (t, ref):
        x.close()
