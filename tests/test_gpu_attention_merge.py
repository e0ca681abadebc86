"""Two blocks of timesteps are merged by the o-projection, more by the attention launch itself: the same
arithmetic, so the same bits.  A step that the caller captures gets the launch shape of the whole context, whatever the
position: with a context of up to 256 rows that is the merging o-projection also for a single block, with a longer one the
attention launch's own merge also for two; a direct call picks by position."""
import ctypes as C

import numpy as np
import pytest

from managedllama2_amd import capi, synth
from managedllama2_amd.transformer import Transformer

pytestmark = pytest.mark.gpu


# one and two chunk columns per lane (dim up to 2048, up to 4096), a number of heads that does not fill a wavefront's 4
# rows of lanes, more threads than pieces of the input
@pytest.mark.parametrize("dim", [128, 384, 2048, 2176, 4096])
@pytest.mark.parametrize("seq_len", [256, 512])
def test_merged_in_the_o_projection_or_in_the_attention_launch(dim, seq_len):
    cfg = dict(dim=dim, hidden_dim=256, n_layers=2, n_heads=dim // 128, n_kv_heads=dim // 128, vocab_size=512,
               seq_len=seq_len, rope_theta=10000.0)
    model = synth.random_model(cfg, seed=31)
    rng = synth.rng_for(961, dim)
    history = [synth.normal_f16(rng, 2 * seq_len * dim) for _ in range(2)]
    t = Transformer(dict(cfg), model, mode=capi.DECODE_FUSED | capi.DECODE_GRAPH)
    t.runstate.tokens.copy_to_device(rng.integers(3, 512, seq_len).astype(np.int32))

    def step(run):
        t.runstate.keyCache.copy_to_device(history[0])
        t.runstate.valueCache.copy_to_device(history[1])
        run()
        return [b.to_host().view(np.uint16) for b in (t.runstate.logits, t.runstate.keyCache, t.runstate.valueCache)]

    for pos in (0, 1, 63, 126, 127, 128, 129, 191, 254, 255):
        graph = C.c_void_p()
        capi.call("llama2_graph_begin_capture")
        capi.call("llama2_decode_forward", t._decoder, pos, pos + 1)
        capi.call("llama2_graph_end_capture", C.byref(graph))
        direct = step(lambda: t.Forward(pos, pos + 1))
        for _ in range(2):
            captured = step(lambda: capi.call("llama2_graph_launch", graph))
            assert all(np.array_equal(a, b) for a, b in zip(direct, captured)), pos
        capi.call("llama2_graph_destroy", graph)
    t.close()
