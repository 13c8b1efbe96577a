"""The posts of the pivoted QR (csrc/pte_post.h, compiled for the host): every
bit of the two values and the column survive the packing into tagged words, a
word of another step is told, and the tags tell a step
from the one that used the same place before, past their wrap too."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

import oqupy_amd

CSRC = os.path.join(os.path.dirname(oqupy_amd.__file__), "csrc")

SOURCE = """
#include "pte_post.h"
typedef unsigned long long u64;
extern "C" {
u64 tag(int j) { return qrcp_tag(j); }
void pack(u64 norm, u64 sum, unsigned local, int j, u64* w) {
  const QrcpPost p{norm, sum, local};
  for (int k = 0; k < kQrPostWords; ++k) w[k] = qrcp_word(p, k, qrcp_tag(j));
}
int unpack(const u64* w, int j, u64* norm, u64* sum, unsigned* local) {
  for (int k = 0; k < kQrPostWords; ++k)
    if (!qrcp_tagged(w[k], qrcp_tag(j))) return 0;
  const QrcpPost p = qrcp_unpack(w[0], w[1]);
  *norm = p.norm | qrcp_norm_low(w[2]); *sum = p.sum; *local = p.local;
  return 1;
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    path = tmp_path_factory.mktemp("post")
    (path / "post.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC,
                    str(path / "post.cpp"), "-o", str(path / "post.so")], check=True)
    out = ctypes.CDLL(str(path / "post.so"))
    out.tag.restype = ctypes.c_ulonglong
    return out


def _bits(x):
    return int(np.float64(x).view(np.uint64))


def test_round_trip(lib):
    rng = np.random.default_rng(3)
    values = [0.0, 5e-324, 2.2e-308, 1.0, 1.0 + 2.0 ** -52, 1.25 * (1 + 2.0 ** -25),
              1.7976931348623157e308, np.inf]
    values += list(rng.random(200) * 10.0 ** rng.integers(-300, 300, 200))
    cols = [0, 1, 39, 254, 255]
    words = (ctypes.c_ulonglong * 4)()
    norm, total, col = ctypes.c_ulonglong(), ctypes.c_ulonglong(), ctypes.c_uint()
    for i, v in enumerate(values):
        s, c, j = values[-1 - i], cols[i % len(cols)], int(rng.integers(0, 20000))
        lib.pack(ctypes.c_ulonglong(_bits(v)), ctypes.c_ulonglong(_bits(s)), c, j, words)
        assert lib.unpack(words, j, ctypes.byref(norm), ctypes.byref(total),
                          ctypes.byref(col)) == 1
        assert (norm.value, total.value, col.value) == (_bits(v), _bits(s), c)
        # one word of another step: not complete
        for k in range(3):
            old = words[k]
            lib.pack(ctypes.c_ulonglong(_bits(v)), ctypes.c_ulonglong(_bits(s)), c, j + 2,
                     words)
            new = words[k]
            lib.pack(ctypes.c_ulonglong(_bits(v)), ctypes.c_ulonglong(_bits(s)), c, j, words)
            words[k] = new
            assert lib.unpack(words, j, ctypes.byref(norm), ctypes.byref(total),
                              ctypes.byref(col)) == 0
            words[k] = old


def test_tags(lib):
    tags = [lib.tag(j) for j in range(20000)]
    assert min(tags) >= 1 and max(tags) <= 0xfff
    # posts are double-buffered by the parity of the step
    assert all(tags[j] != tags[j - 2] for j in range(2, len(tags)))
