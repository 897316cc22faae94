"""GPU block-index builder vs the oracle: bit-exact kv_idx / kv_num / kv_partial /
wave codes, elements and live (gpu/blockindex.py:32-51 semantics)."""
import numpy as np
import pytest

from oracle import blockindex as obi
from oracle import masks as om
from oracle import permute as op
from polyhedral_amd import index as pindex
from polyhedral_amd.polyattn import masks as pm
from polyhedral_amd.registry import SPECS, numpy_mask

pytestmark = pytest.mark.gpu

TILES = [(128, 128), (128, 32), (64, 64), (32, 32), (16, 16), (128, 16), (16, 128), (32, 64)]


def _compare(bi, ref):
    assert np.array_equal(bi.kv_num, ref["kv_num"])
    assert bi.kv_idx.shape == ref["kv_idx"].shape
    assert np.array_equal(bi.kv_idx, ref["kv_idx"])
    assert np.array_equal(bi.kv_partial, ref["kv_partial"])
    assert np.array_equal(bi.kv_wave_bits, ref["wave"])
    assert bi.elements == ref["elements"] and bi.live == ref["live"]


@pytest.mark.parametrize("name", [n for n in SPECS])
@pytest.mark.parametrize("N", [256, 1024])
def test_named_masks_all_tiles(gpu, name, N):
    spec = om.NAMED[name]
    m = numpy_mask(name)
    for BQ, A in TILES:
        _compare(pindex.build(m, N, BQ, A), obi.build(spec, N, BQ, A))


@pytest.mark.parametrize("name,s,N", [("dilated-4", 4, 1024), ("dilated-8", 8, 1024),
                                      ("local256+str8", 2, 2048), ("local256+str8", 4, 2048),
                                      ("local256+str8", 8, 2048), ("band256+lat16", 16, 2048),
                                      ("lat16-band256", 16, 4096), ("sinks4+win256", 8, 1024)])
def test_class_a_permuted(gpu, name, s, N):
    perm = op.residue_perm(N, s)
    m = pm.Permuted(numpy_mask(name), perm)
    for BQ, A in [(128, 32), (16, 16), (128, 128), (64, 64)]:
        _compare(pindex.build(m, N, BQ, A), obi.build(om.NAMED[name], N, BQ, A, perm_q=perm, perm_kv=perm))


@pytest.mark.parametrize("basis", ["identity", "rp8", "random"])
@pytest.mark.parametrize("N", [1168, 1296])
def test_block_verdicts_at_their_edges(gpu, basis, N):
    """Masks whose bounds fall just inside, on and just outside blocks of 16, 32 and 64
    positions, unions and differences of them, N no multiple of 64 (a wave's last columns
    missing), in bases where blocks have one residue and where they have not."""
    perm = {"identity": None, "rp8": op.residue_perm(N, 8),
            "random": np.random.default_rng(N).permutation(N).astype(np.int32)}[basis]
    ms = [pm.Causal(), pm.SlidingWindow(63), pm.SlidingWindow(64), pm.SlidingWindow(65), pm.SlidingWindow(1),
          pm.Dilated(8), pm.Dilated(4), pm.Dilated(1), pm.Dilated(3), pm.LocalStrided(64, 8), pm.LocalStrided(33, 4),
          pm.TwoBand(64, 256, 64), pm.TwoBand(31, 100, 65), pm.SinksWindow(64, 128), pm.SinksWindow(17, 33),
          pm.PrefixLM(64), pm.PrefixLM(513), pm.Full(), pm.Union(pm.SlidingWindow(64), pm.Dilated(8)),
          pm.Difference(pm.Dilated(8), pm.SlidingWindow(64)), pm.Difference(pm.Full(), pm.Causal()),
          pm.Difference(pm.Causal(), pm.Union(pm.Dilated(4), pm.PrefixLM(128)))]
    p = np.arange(N) if perm is None else perm.astype(np.int64)
    for m in ms:
        M = m.live(p[:, None], p[None, :])
        for BQ, A in [(16, 16)]:
            bi = pindex.build(m if perm is None else pm.Permuted(m, perm), N, BQ, A)
            ref = obi.build_dense(M, BQ, A)
            for key in ("kv_idx", "kv_num", "kv_partial"):
                assert np.array_equal(getattr(bi, key), ref[key]), f"{m.name} {basis} {BQ}x{A} {key}"
            assert bi.elements == ref["elements"] and bi.live == ref["live"], f"{m.name} {basis}"
    # the larger tiles, N a multiple of 128, and the bitmaps against the dense mask
    N2 = 1152
    p2 = np.arange(N2) if perm is None else (op.residue_perm(N2, 8) if basis == "rp8" else
                                             np.random.default_rng(N2).permutation(N2)).astype(np.int64)
    for m in ms:
        M = m.live(p2[:, None], p2[None, :])
        mm = m if perm is None else pm.Permuted(m, p2.astype(np.int32))
        for BQ, A in [(128, 32), (128, 128), (64, 64)]:
            kv_idx, kv_num, kv_partial, _, tiles, live, (off, pool) = pindex.build_device(mm, N2, BQ, A, device=gpu,
                                                                                          bits=True)
            ref = obi.build_dense(M, BQ, A)
            kv_idx, kv_num, kv_partial = (t.cpu().numpy() for t in (kv_idx, kv_num, kv_partial))
            assert np.array_equal(kv_idx, ref["kv_idx"]) and np.array_equal(kv_num, ref["kv_num"])
            assert np.array_equal(kv_partial, ref["kv_partial"]) and live == ref["live"], f"{m.name} {basis}"
            off, pool = off.cpu().numpy(), pool.cpu().numpy().view(np.uint32)
            for i in range(N2 // BQ):
                for j in range(kv_idx.shape[1]):
                    if j >= kv_num[i] or not kv_partial[i, j]:
                        assert off[i, j] == -1
                        continue
                    w = pool[off[i, j]:off[i, j] + BQ * (A // 32)].reshape(BQ, A // 32)
                    got = ((w[:, :, None] >> np.arange(32, dtype=np.uint32)) & 1).reshape(BQ, A).astype(bool)
                    k0 = kv_idx[i, j] * A
                    assert np.array_equal(got, M[i * BQ:(i + 1) * BQ, k0:k0 + A]), f"{m.name} {basis} bits {i},{j}"


class _Dense:
    """The reference's explicit-matrix wrapper (gpu/test_correctness.py:90-95)."""
    def __init__(self, M):
        self.M, self.name = M, "permuted"

    def row_cols(self, q, N):
        return self.M[q]


def test_explicit_matrix_input(gpu):
    N, s = 1024, 8
    perm = op.residue_perm(N, s)
    M = om.dense(om.NAMED["dilated-8"], N)[perm][:, perm]
    bi = pindex.build(_Dense(M), N, 16, 16)
    ref = obi.build_dense(M, 16, 16)
    for key in ("kv_idx", "kv_num", "kv_partial"):
        assert np.array_equal(getattr(bi, key), ref[key])
    assert bi.elements == ref["elements"] and bi.live == ref["live"]


def test_empty_mask_gives_zero_pitch(gpu):
    # a lattice restricted to pairs a prefix-LM does not cover
    N = 4096
    bi = pindex.build(numpy_mask("lat32-prefixlm2048"), N, 128, 32)
    assert bi.kv_idx.shape == (N // 128, 0) and bi.live == 0 and bi.elements == 0
    assert not bi.kv_num.any()
