"""Two blocks of timesteps are merged by the o-projection, more by the attention launch itself, and the persistent step has
a merge of its own: the same arithmetic, so the same bits.  A step that the caller captures gets the launch shape of the
whole context, whatever the position: with a context of up to 256 rows that is the merging o-projection also for a
single block, with a longer one the attention launch's own merge also for two; a direct call picks by position.

The model shows every bit of the attention output: its o-projection is the identity, its feed-forward part adds nothing, the
embedding is small and the classifier is the identity too.  A denominator that is rounded once more
moves only one output in 100000 or fewer, and only where the second block holds the larger maximum: hence flat scores,
larger keys in that block, and all positions from 128 to 255 several times (1.6 million outputs of dim 4096)."""
import ctypes as C

import numpy as np
import pytest

from managedllama2_amd import capi, synth
from managedllama2_amd.transformer import Transformer

pytestmark = pytest.mark.gpu


def identity_qweight(n):
    ws, ss, zs = synth.qweight_sizes(n)
    W = np.zeros((n, ws), np.uint32)
    k = np.arange(n)
    W[k, k // 8] = np.uint32(1) << (4 * (k % 8)).astype(np.uint32)
    return W.ravel(), np.zeros(n * zs, np.uint32), np.ones(n * ss, np.float16)


def transparent_model(dim, hidden):
    rng = synth.rng_for(962, dim)

    def small(K, N, scale):
        W, Z, S = synth.random_qweight(rng, K, N)
        return W, Z, (S.astype(np.float32) * scale).astype(np.float16)

    def nothing(K, N):
        ws, ss, zs = synth.qweight_sizes(K)
        return np.zeros(N * ws, np.uint32), np.zeros(N * zs, np.uint32), np.zeros(N * ss, np.float16)

    scale = 0.5 * (4096 / dim) ** 0.5  # queries and keys of about the history's size
    layer = dict(q=small(dim, dim, scale), k=small(dim, dim, scale), v=small(dim, dim, scale), o=identity_qweight(dim),
                 gate=nothing(dim, hidden), up=nothing(dim, hidden), down=nothing(hidden, dim),
                 rms_att=np.ones(dim, np.float16), rms_ffn=np.ones(dim, np.float16))
    return dict(embedding=synth.normal_f16(rng, dim * dim, 0.001), classifier=np.eye(dim, dtype=np.float16).ravel(),
                rms_final=np.ones(dim, np.float16), layers=[layer])


# Merged in the o-projection: an even number of 128-input groups.  256 .. 2048 and 2304 .. 4096 are its two instantiations; 768
# and 1280 have heads that do not fill a wavefront's 4 rows of lanes, 2304 and 3840 a zero tail; 384 has 3 groups and never
# gets there.
@pytest.mark.parametrize("dim", [256, 384, 512, 768, 1280, 2048, 2304, 3840, 4096])
@pytest.mark.parametrize("seq_len", [256, 512])
def test_merged_in_the_o_projection_or_elsewhere(dim, seq_len):
    merges = dim // 128 % 2 == 0
    hidden = 11008 if dim == 4096 else 256  # that of the persistent step's 7B kernel
    cfg = dict(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=dim // 128, n_kv_heads=dim // 128, vocab_size=dim,
               seq_len=seq_len, rope_theta=10000.0)
    model = transparent_model(dim, hidden)
    rng = synth.rng_for(961, dim)
    key = synth.normal_f16(rng, seq_len * dim).reshape(seq_len, dim)
    key[128:] *= np.float16(1.1)
    value = synth.normal_f16(rng, seq_len * dim)
    mode = capi.DECODE_FUSED | capi.DECODE_GRAPH
    t, other = Transformer(dict(cfg), model, mode=mode), None
    if dim in (256, 4096):
        other = Transformer(dict(cfg), model, mode=capi.DECODE_FUSED | capi.DECODE_PERSISTENT)
    for x in (t, other):
        if x:
            x.runstate.keyCache.copy_to_device(key)
            x.runstate.valueCache.copy_to_device(value)
    untouched = np.full(dim, 77.0, np.float16)  # xb: what the attention launch writes unless it leaves the merge to others

    def step(run, x, merged):
        t.runstate.xb.copy_to_device(untouched)
        run()
        if x is t:
            assert np.array_equal(t.runstate.xb.to_host(), untouched) == merged
        return x.runstate.logits.to_host().view(np.uint16)

    all_positions = seq_len == 512
    differ, outputs = 0, 0
    for pos in range(126, 256) if all_positions else (0, 1, 63, 126, 127, 128, 129, 191, 254, 255):
        graph = C.c_void_p()
        capi.call("llama2_graph_begin_capture")
        capi.call("llama2_decode_forward", t._decoder, pos, pos + 1)
        capi.call("llama2_graph_end_capture", C.byref(graph))
        for token in synth.rng_for(963, pos).integers(0, dim, 3).astype(np.int32):
            for x in (t, other):
                if x:
                    x.runstate.tokens.copy_to_device(np.array([token], np.int32), pos)
            direct = step(lambda: t.Forward(pos, pos + 1), t, merges and pos >= 128)
            captured = step(lambda: capi.call("llama2_graph_launch", graph), t, merges and seq_len == 256)
            results = [captured]
            if other:
                results.append(step(lambda: other.Forward(pos, pos + 1), other, False))
            for r in results:
                differ += int(np.count_nonzero(direct != r))
                outputs += dim
        capi.call("llama2_graph_destroy", graph)
    assert len(np.unique(direct)) > min(dim, 1000) // 2  # the outputs are no constants
    for x in (t, other):
        if x:
            capi.call("llama2_decode_check", x._decoder)
            x.close()
    assert differ == 0, "%d of %d outputs differ" % (differ, outputs)
