"""Plans of the three CRT routes (several words, one word, integers) share one map
of a context.  A modulus of several words may hold any bytes, those of another
plan's key included: the keys must differ all the same, and a product modulo
such a P must not be given the other plan's constants."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "cpp", "plan_key_harness.cpp")
OUT = os.path.join(HERE, "cpp", "_build", "libplankey.so")


def words_of(text):
    assert len(text) % 4 == 0
    return [int.from_bytes(text[i:i + 4].encode(), "little") for i in range(0, len(text), 4)]


@pytest.fixture(scope="module")
def key():
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-o", OUT, SRC], check=True)
    lib = ctypes.CDLL(OUT)
    size, buf = ctypes.c_size_t, ctypes.create_string_buffer(512)

    def mp(P, k, minsz, lpts):
        n = lib.lbx_test_mp_key((ctypes.c_uint32 * len(P))(*P), len(P), size(k), size(minsz), lpts, buf, 512)
        return buf.raw[:n]

    def few(p, k, minsz, lpts):
        n = lib.lbx_test_few_key(ctypes.c_uint32(p), size(k), size(minsz), lpts, buf, 512)
        return buf.raw[:n]

    def zz(lab, k, minsz, lpts, nl, cl):
        n = lib.lbx_test_zz_key(lab, size(k), size(minsz), lpts, nl, cl, buf, 512)
        return buf.raw[:n]

    return mp, few, zz


def test_modulus_that_spells_another_key(key):
    mp, few, zz = key
    assert mp(words_of("fp|12345"), 3, 8, 4) != few(12345, 3, 8, 4)
    assert mp(words_of("zz|130|7|200"), 9, 2, 5) != zz(130, 7, 200, 9, 2, 5)
    assert not mp(words_of("zz|9"), 3, 8, 4).startswith(b"zz|")  # integer plans are counted by their tag
    # a modulus that spells the beginning of another one's fields, and other word counts
    assert mp(words_of("abcd"), 3, 8, 4) != mp(words_of("abcd|3|8"), 8, 4, 4)
    keys = [mp([5] * n, k, s, lg) for n in (1, 2, 3) for k in (1, 11) for s in (1, 11) for lg in (1, 11)]
    assert len(set(keys)) == len(keys)


@pytest.mark.gpu
def test_product_modulo_such_a_modulus():
    """A product modulo 12345 keeps a one-word plan; the product of the same shape
    modulo the two words whose bytes spell "fp|12345" needs its own."""
    import linbox_amd as lbx
    from linbox_amd import PolynomialMatrix
    m, k, n, sa, sb = 3, 4, 2, 9, 8
    rng = np.random.default_rng(3)
    ctx = lbx.Context(0)
    try:
        for P, nl in ((12345, 1), (int.from_bytes(b"fp|12345", "little"), 2)):
            a = [[int(x) * int(y) % P for x, y in zip(*rng.integers(1, 1 << 62, (2, sa)))] for _ in range(m * k)]
            b = [[int(x) * int(y) % P for x, y in zip(*rng.integers(1, 1 << 62, (2, sb)))] for _ in range(k * n)]

            def stored(x, rows, cols, size):
                w = [(v >> (32 * j)) & 0xffffffff for row in x for v in row for j in range(nl)]
                return PolynomialMatrix(rows, cols, size, nlimbs=nl, data=np.array(w, np.uint32))

            C = PolynomialMatrix(m, n, sa + sb - 1, nlimbs=nl)
            print("[case] plan key", hex(P), flush=True)
            lbx.mul_mp(P, C, stored(a, m, k, sa), stored(b, k, n, sb), ctx=ctx)
            got = np.asarray(C.data, np.uint64).reshape(m * n, sa + sb - 1, nl)
            for i in range(m):
                for j in range(n):
                    want = [0] * (sa + sb - 1)
                    for q in range(k):
                        for u, x in enumerate(a[i * k + q]):
                            for v, y in enumerate(b[q * n + j]):
                                want[u + v] += x * y
                    have = [sum(int(w) << (32 * l) for l, w in enumerate(c)) for c in got[i * n + j]]
                    assert have == [w % P for w in want]
    finally:
        ctx.close()
