"""Which shape the prompt's matrix products get (csrc/gemm_shape.hpp, plain host code, compiled here): workgroups of two
heights where they are worth it, on 256 compute units."""
import ctypes
import os
import shutil
import subprocess

import pytest

from managedllama2_amd import synth
from test_gpu_prefill import TWO_HEIGHTS

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "managedllama2_amd", "csrc")
SOURCE = """
namespace l2 { inline int ceil_div(int a, int b) { return (a + b - 1) / b; } }
#include "gemm_shape.hpp"
extern "C" void shape(int tiles, int pairs, int groups, int may_split, int cus, int* out)
{
    const l2::GemmShape s = l2::gemm_shape(tiles, pairs, groups, may_split, cus);
    out[0] = s.mt, out[1] = s.wn, out[2] = s.splits, out[3] = s.mt2, out[4] = s.first;
}
"""

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    out = tmp_path_factory.mktemp("shape")
    (out / "shape.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-I", CSRC,
                           str(out / "shape.cpp"), "-o", str(out / "shape.so")])
    lib = ctypes.CDLL(str(out / "shape.so"))

    def call(rows, pairs, K, may_split=False):
        result = (ctypes.c_int * 5)()
        lib.shape(-(-rows // 32), pairs, -(-K // 128), may_split, 256, result)
        return tuple(result)

    return call


def qkv(shape, dim, rows):
    return shape(rows, 3 * dim // 64, dim)


def swiglu(shape, dim, hidden, rows):
    return shape(rows, -(-hidden // 32), dim)


def heights(s):
    return s[0], s[3]


def test_two_heights_of_the_model_widths(shape):
    """At the edges of the rows that take them; 385 .. 448 rows of 7B are predicted 0.3 % and lose 1 %."""
    dim, hidden = (synth.LLAMA2_7B[k] for k in ("dim", "hidden_dim"))
    two = dict((rows, heights(swiglu(shape, dim, hidden, rows))) for rows in range(1, 1025)
               if len(set(heights(swiglu(shape, dim, hidden, rows)))) > 1)
    assert two == dict([(r, (3, 2)) for r in range(321, 385)] + [(r, (4, 2)) for r in range(481, 513)] +
                       [(r, (4, 3)) for r in range(897, 961)])
    two = dict((rows, heights(qkv(shape, dim, rows))) for rows in range(1, 1025)
               if len(set(heights(qkv(shape, dim, rows)))) > 1)
    assert two == dict([(r, (3, 2)) for r in range(673, 769)] + [(r, (4, 2)) for r in range(961, 1025)])
    dim, hidden = (synth.LLAMA2_13B[k] for k in ("dim", "hidden_dim"))
    two = [rows for rows in range(32, 1025, 32) if len(set(heights(swiglu(shape, dim, hidden, rows)))) > 1]
    assert two == [320, 416, 448, 480, 928, 960, 992, 1024]
    assert all(len(set(heights(qkv(shape, dim, rows)))) == 1 for rows in range(32, 1025, 32))


@pytest.mark.parametrize("product,dim,hidden,two,one", TWO_HEIGHTS)
def test_compared_batches_differ_in_the_heights_alone(shape, product, dim, hidden, two, one):
    a, b = ((qkv(shape, dim, r) if product == "qkv" else swiglu(shape, dim, hidden, r)) for r in (two, one))
    assert a[0] != a[3] and b[0] == b[3] and a[1] == b[1] == 4  # one group of K per step on both sides
    if product == "swiglu":
        for K in (dim, hidden):  # o- and down-projection: groups per step and pieces of K
            assert shape(two, dim // 64, K, True)[1:3] == shape(one, dim // 64, K, True)[1:3]
        for rows in (two, one):  # attention in one piece: at most 4 workgroups per compute unit
            assert 4 * 256 // (-(-rows // 32) * (dim // 128)) <= 1
            # and the other product of the layer has the same groups per step
            assert qkv(shape, dim, rows)[1] == 4


def test_all_pairs_of_heights_are_compared(shape):
    assert {(p, heights(qkv(shape, d, r) if p == "qkv" else swiglu(shape, d, h, r))) for p, d, h, r, _ in TWO_HEIGHTS} == {
        (p, pair) for p in ("qkv", "swiglu") for pair in ((4, 3), (4, 2), (3, 2))}
