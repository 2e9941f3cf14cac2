"""The AMG set-up's Galerkin products, 16 and 64 lanes a pair of aggregates, block
by block against the FP64 triple product on the host: pairs of no block, of fewer
blocks than lanes, of as many, one more and one less, and of thousands; fewer
pairs than a block of the launch takes and a remainder.

The kernel and the reference sum the same products of FP32 numbers in FP64 in
another order: they differ by the count of terms (9 n of a pair's n blocks) times
2^-53 of the terms' absolute sum, and by the rounding to FP32 (2^-24)."""
import ctypes as C
import os

import numpy as np
import pytest

from lowlevelfem import _lib

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(_lib.LIB_PATH), "libllfem_check.so")


def _run(lanes, counts, seed):
    rng = np.random.default_rng(seed)
    npairs, nfine, nadjf = len(counts), 500, 4000
    adjf = rng.integers(0, nfine, nadjf).astype(np.int32)
    Q = rng.uniform(-1.0, 1.0, (nfine, 3, 6)).astype(np.float32)
    blocks = rng.uniform(-1.0, 1.0, (nadjf, 3, 3)).astype(np.float32)
    flat = blocks.reshape(nadjf, 9)
    valf = np.concatenate([flat[:, :4].ravel(), flat[:, 4:8].ravel(), flat[:, 8]])
    gptr = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    n = int(gptr[-1])
    gblk = rng.integers(0, nadjf, n).astype(np.int32)
    gcol = rng.integers(0, nfine, n).astype(np.int32)
    # each pair's two rows of two coarse blocks, anywhere
    nadjc = 4 * npairs
    pair_o = (2 * rng.permutation(2 * npairs)).astype(np.int32).reshape(npairs, 2)
    out = np.full(9 * nadjc, np.nan, np.float32)
    args = [np.ascontiguousarray(a) for a in (gptr, gblk, gcol, adjf, Q, valf, pair_o)]
    lib = C.CDLL(LIB)
    assert lib.galerkin_check(C.c_int(lanes), *(C.c_int64(k) for k in (npairs, nfine, nadjf, nadjc, n)),
                              *(a.ctypes.data_as(C.c_void_p) for a in args), out.ctypes.data_as(C.c_void_p)) == 0
    got = np.concatenate([out[:4 * nadjc].reshape(nadjc, 4), out[4 * nadjc:8 * nadjc].reshape(nadjc, 4),
                          out[8 * nadjc:, None]], axis=1).reshape(nadjc, 3, 3)
    for p in range(npairs):
        c = slice(gptr[p], gptr[p + 1])
        Qj, B, Qi = (a.astype(np.float64) for a in (Q[gcol[c]], blocks[gblk[c]], Q[adjf[gblk[c]]]))
        ref = (Qj.transpose(0, 2, 1) @ B @ Qi).sum(0)
        mag = (abs(Qj).transpose(0, 2, 1) @ abs(B) @ abs(Qi)).sum(0)
        res = np.block([[got[pair_o[p, s] + v] for v in range(2)] for s in range(2)])
        assert (abs(res - ref) <= 2.0 ** -24 * abs(ref) + 18 * counts[p] * 2.0 ** -53 * mag).all(), (p, counts[p])


@pytest.mark.parametrize("lanes", [16, 64])
def test_blocks(lanes):
    counts = [0, 1, 2, lanes // 2, lanes - 1, lanes, lanes + 1, 2 * lanes, 2 * lanes + 3, 5000, 0, 37, 9 * lanes - 1]
    _run(lanes, counts, 1)
    _run(lanes, [3], 2)
    _run(lanes, np.random.default_rng(3).integers(0, 4 * lanes, 257).tolist(), 4)
