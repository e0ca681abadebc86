"""Which rows a wavefront of the int4 mat-vecs takes, at the edges of the rules that decide it.

Rows of 4097 .. 6144 inputs: one workgroup per compute unit takes its whole share of the rows, QKV in 12 wavefronts of two rows
(with RoPE the two rows of a pair), SwiGLU in 8 of seven.  Workgroups full and partly empty, the last size that one
workgroup per compute unit holds and the next.

The order in which a row is added up is the same in every int4 kernel, and so are the RMSNorm and the rotation of the fused
step and of the modules: cache rows, query and single mat-vecs are compared bit for bit, SwiGLU with fp64.
"""
import numpy as np
import pytest

from managedllama2_amd import capi, synth
from managedllama2_amd.transformer import Transformer
from gpu_util import assert_close, sizes, up, upq

pytestmark = pytest.mark.gpu


def bits(a):
    return np.asarray(a).view(np.uint16)


@pytest.mark.parametrize("heads", [33, 34, 40, 48])
def test_qkv_rope_pairs_equal_the_modules(heads):
    dim, seq = 128 * heads, 24
    cfg = dict(dim=dim, hidden_dim=256, n_layers=1, n_heads=heads, n_kv_heads=heads, vocab_size=64, seq_len=seq,
               rope_theta=10000.0)
    model = synth.random_model(cfg, seed=31, rms_random=True)
    prompt = synth.rng_for(612, heads).integers(3, 64, seq).astype(np.int32)
    outs = []
    for mode in (capi.DECODE_MODULES, capi.DECODE_FUSED):
        t = Transformer(dict(cfg), model, mode=mode)
        t.runstate.tokens.copy_to_device(prompt)
        q = []
        for pos in (0, 1, 7, 8, 23):
            t.Forward(pos, pos + 1)
            q.append(t.runstate.q.to_host())
        outs.append((np.stack(q), t.runstate.keyCache.to_host(), t.runstate.valueCache.to_host()))
        t.close()
    for a, b, what in zip(outs[0], outs[1], ("query", "key cache", "value cache")):
        assert np.array_equal(bits(a), bits(b)), what


# An infinite scale spoils its own row and no other, also where a wavefront takes several rows and the one in front has lanes
# without inputs: rows of up to 2048 inputs, three tensors of longer ones, and SwiGLU of longer ones with one row per wavefront.
# Odd and even numbers of groups; one, two, three and four rows of SwiGLU, one and two of the others.
@pytest.mark.parametrize("K,N", [(136, 96), (384, 77), (384, 4100), (640, 8200), (1408, 6100), (1920, 8204), (512, 13000),
                                 (2304, 2048), (4224, 1500), (4224, 4300), (5120, 5120), (5120, 6144)])
def test_infinite_scale_stays_in_its_row(K, N):
    rng = synth.rng_for(617, K, N)
    zs, ss, ws = sizes(K)
    x, res = up(synth.normal_f16(rng, K)), synth.normal_f16(rng, N)
    qs = [synth.random_qweight(rng, K, N) for _ in range(3)]
    rows = np.arange(1, N, 11)  # comes to every place among a wavefront's rows
    spoilt = []
    for i, (W, Z, S) in enumerate(qs):
        S = S.copy().reshape(N, ss)
        S[rows, rng.integers(0, ss, rows.size) if i else 0] = np.inf
        spoilt.append((W, Z, S.ravel()))

    def run(tensors):
        dev = [upq(q) for q in tensors]
        ptrs = [p for q in dev for p in (q.Weight.ptr, q.Zeros.ptr, q.Scales.ptr)]
        outs = dict((name, up(np.zeros(N, np.float16))) for name in "qkv")
        capi.call("llama2_qkv_mat_vec", *[o.ptr for o in outs.values()], x.ptr, *ptrs, K, N, zs, ss, ws)
        if K <= 2048 or N <= 2048:
            outs["swiglu"] = up(np.zeros(N, np.float16))
            capi.call("llama2_mat_vec_swiglu", outs["swiglu"].ptr, x.ptr, *ptrs[:6], K, N, zs, ss, ws)
        if K <= 2048:
            outs["plain"], outs["residual"] = up(np.zeros(N, np.float16)), up(res)
            capi.call("llama2_mat_vec_int4", outs["plain"].ptr, x.ptr, *ptrs[:3], K, N, zs, ss, ws)
            capi.call("llama2_mat_vec_residual_int4", outs["residual"].ptr, x.ptr, *ptrs[:3], K, N, zs, ss, ws)
        return dict((name, o.to_host()) for name, o in outs.items())

    others = np.setdiff1d(np.arange(N), rows)
    clean, got = run(qs), run(spoilt)
    for what in clean:
        assert np.array_equal(bits(got[what][others]), bits(clean[what][others])), what
        if what != "swiglu":  # a gate of -infinity gives 0 times the up row
            assert not np.any(np.isfinite(got[what][rows])), what


# An infinite scale of one row spoils that row and the one it is rotated with, and nothing else.
@pytest.mark.parametrize("heads", [3, 34, 40])
def test_qkv_rope_infinite_scale_stays_in_its_pair(heads):
    dim = 128 * heads
    cfg = dict(dim=dim, hidden_dim=256, n_layers=1, n_heads=heads, n_kv_heads=heads, vocab_size=64, seq_len=16,
               rope_theta=10000.0)
    model = synth.random_model(cfg, seed=32, rms_random=True)
    ss, outs = synth.qweight_sizes(dim)[1], []
    rows = np.arange(0, dim, 41)
    for spoil in (False, True):
        if spoil:
            for i, name in enumerate(("q", "k", "v")):
                W, Z, S = model["layers"][0][name]
                S = S.copy().reshape(dim, ss)
                S[rows, i] = np.inf
                model["layers"][0][name] = W, Z, S.ravel()
        t = Transformer(dict(cfg), model, mode=capi.DECODE_FUSED)
        t.runstate.tokens.copy_to_device(np.array([5] * 16, np.int32))
        t.Forward(9, 10)
        outs.append([t.runstate.q.to_host(), t.runstate.keyCache.to_host(dim, 9 * dim), t.runstate.valueCache.to_host(dim, 9 * dim)])
        t.close()
    for what, clean, got in zip(("query", "key", "value"), *outs):
        touched = rows if what == "value" else np.union1d(rows, rows ^ 64)
        others = np.setdiff1d(np.arange(dim), touched)
        assert np.array_equal(bits(got[others]), bits(clean[others])), what
        assert not np.any(np.isfinite(got[rows])), what


# (the last three: an odd number of groups below, at and above four rows per compute unit)
@pytest.mark.parametrize("K,N", [(5120, 5120), (5120, 6144), (5120, 6152), (4224, 4096), (6144, 4097), (4352, 24), (384, 1023),
                                 (1920, 1024), (640, 1025)])
def test_three_tensors_equal_one_at_a_time(K, N):
    rng = synth.rng_for(613, K, N)
    zs, ss, ws = sizes(K)
    x = up(synth.normal_f16(rng, K))
    qs = [upq(synth.random_qweight(rng, K, N)) for _ in range(3)]
    three = [up(np.zeros(N, np.float16)) for _ in range(3)]
    capi.call("llama2_qkv_mat_vec", *[o.ptr for o in three], x.ptr,
              *[p for q in qs for p in (q.Weight.ptr, q.Zeros.ptr, q.Scales.ptr)], K, N, zs, ss, ws)
    for q, got in zip(qs, three):
        one = up(np.zeros(N, np.float16))
        capi.call("llama2_mat_vec_int4", one.ptr, x.ptr, q.Weight.ptr, q.Zeros.ptr, q.Scales.ptr, K, N, zs, ss, ws)
        assert np.array_equal(bits(got.to_host()), bits(one.to_host()))


# A single tensor of 3841 .. 4096 rows and 2049 .. 4096 inputs goes in workgroups of 16 wavefronts, the rows around that in fours:
# a row's result does not depend on how many there are.
@pytest.mark.parametrize("K", [2056, 4096])
def test_rows_that_fill_one_workgroup_per_compute_unit(K):
    rng = synth.rng_for(616, K)
    zs, ss, ws = sizes(K)
    x, q = up(synth.normal_f16(rng, K)), upq(synth.random_qweight(rng, K, 4104))
    res = synth.normal_f16(rng, 4104)
    outs = {}
    for N in (3840, 3841, 4095, 4096, 4104):
        plain, residual = up(np.zeros(N, np.float16)), up(res[:N].copy())
        capi.call("llama2_mat_vec_int4", plain.ptr, x.ptr, q.Weight.ptr, q.Zeros.ptr, q.Scales.ptr, K, N, zs, ss, ws)
        capi.call("llama2_mat_vec_residual_int4", residual.ptr, x.ptr, q.Weight.ptr, q.Zeros.ptr, q.Scales.ptr, K, N, zs, ss, ws)
        outs[N] = bits(plain.to_host()), bits(residual.to_host())
    for N, (plain, residual) in outs.items():
        assert np.array_equal(plain, outs[4104][0][:N]) and np.array_equal(residual, outs[4104][1][:N]), N


# Rows of up to 2048 inputs may have an odd number of scales and begin at any of them: scales that lie 2 bytes off a word, odd
# and even numbers of groups, ragged last groups and rows that do not fill the last wavefront.
@pytest.mark.parametrize("K,N", [(8, 5), (136, 9), (384, 77), (640, 640), (1408, 512), (1928, 33), (2048, 35)])
def test_scales_at_any_two_bytes(oracle, K, N):
    rng = synth.rng_for(615, K, N)
    zs, ss, ws = sizes(K)
    qs = [synth.random_qweight(rng, K, N) for _ in range(3)]
    x, res = synth.normal_f16(rng, K), synth.normal_f16(rng, N)
    want = [oracle.f64_matvec_int4(x, *q, K, N) for q in qs]
    dx, results = up(x), []
    for shift in (0, 1):
        parts = []
        for W, Z, S in qs:
            dev = up(W), up(Z), up(np.concatenate([np.full(shift, np.inf, np.float16), S]))
            parts.append((dev, (dev[0].ptr, dev[1].ptr, dev[2].ptr + 2 * shift)))
        ptrs = [p for _, q in parts for p in q]
        outs = [up(np.zeros(N, np.float16)) for _ in range(4)] + [up(res)]
        capi.call("llama2_qkv_mat_vec", *[o.ptr for o in outs[:3]], dx.ptr, *ptrs, K, N, zs, ss, ws)
        capi.call("llama2_mat_vec_swiglu", outs[3].ptr, dx.ptr, *ptrs[:6], K, N, zs, ss, ws)
        capi.call("llama2_mat_vec_residual_int4", outs[4].ptr, dx.ptr, *ptrs[:3], K, N, zs, ss, ws)
        results.append([o.to_host() for o in outs])
        for got, w in zip(results[-1], want + [want[0] / (1 + np.exp(-want[0])) * want[1], want[0] + res.astype(np.float64)]):
            assert_close(got, w, "any two bytes %dx%d" % (K, N))  # 2e-3: fp16 results of fp32 sums
    for a, b in zip(*results):
        assert np.array_equal(bits(a), bits(b))


# SwiGLU takes one, two or three rows per wavefront as the compute units allow: the edges on 256 of them, then the wide rows.
@pytest.mark.parametrize("K,N", [(128, 1), (256, 2048), (512, 2049), (256, 4096), (256, 4097), (256, 6144), (384, 6145),
                                 (256, 8192), (256, 8193), (2304, 1409), (4096, 8187),
                                 (5120, 12288), (5120, 12296), (4224, 14336), (6144, 14344)])
def test_swiglu_rows_per_wavefront(oracle, K, N):
    rng = synth.rng_for(614, K, N)
    zs, ss, ws = sizes(K)
    g, u = synth.random_qweight(rng, K, N), synth.random_qweight(rng, K, N)
    x = synth.normal_f16(rng, K)
    dg, du, dx, out = upq(g), upq(u), up(x), up(np.zeros(N, np.float16))
    capi.call("llama2_mat_vec_swiglu", out.ptr, dx.ptr, dg.Weight.ptr, dg.Zeros.ptr, dg.Scales.ptr, du.Weight.ptr,
              du.Zeros.ptr, du.Scales.ptr, K, N, zs, ss, ws)
    gv, uv = oracle.f64_matvec_int4(x, *g, K, N), oracle.f64_matvec_int4(x, *u, K, N)
    assert_close(out.to_host(), gv / (1 + np.exp(-gv)) * uv, "swiglu %dx%d" % (K, N))  # 2e-3: two fp16 roundings
