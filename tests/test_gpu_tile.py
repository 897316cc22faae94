"""The f16 / bf16 kernels on plain block lists (pa_attn_fwd_tile) against the general kernel on
the same arguments, over tile shapes, bases, bitmaps, strides and both sides of the rules that
give a list groups of waves and cut a block into pieces, and every instantiation against the
float64 oracle.  The two kernels agree up to the rounding of P to 16 bits, which happens at the
running maximum and differs between them: with u the unit roundoff of the type, an element
moves by at most u sum p |v| in each kernel and by u |o| in each one's own rounding.  (A row's
largest P is at least 1, so in f16 a P below 2^-14 is off by at most 2^-25 beside it.)"""
import numpy as np
import pytest
import torch

from oracle import attention as oatt
from oracle import masks as om
from oracle import permute as op
from polyhedral_amd import attention as pattn
from polyhedral_amd import index as pindex
from polyhedral_amd.polyattn import masks as pm
from polyhedral_amd.registry import numpy_mask, triton_params
from tests.util import as64, make_qkv

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _bound(oa, o, kernels, dtype, N, v):
    """Largest difference of an element from its value, `kernels` times (one against the oracle,
    two against each other); oa: sum p |v|, o: the value.  Its own rounding may be an ulp of the
    next binade: 2^-10 more of it; 2^-18 for the sums and exponentials in float32."""
    eps = EPS[dtype]
    small = N * 2.0 ** -25 * float(v.float().abs().max()) if dtype == torch.float16 else 0.0
    return kernels * ((eps + 2.0 ** -18) * oa * (1 + 4 * eps) + eps * o.abs() * (1 + 2.0 ** -10) + small) + 2.0 ** -25


def _both(q, k, v, lists, kind, BQ, A, **kw):
    BH, N, _ = q.shape
    out = []
    # the third run: sum p |v| of every element, by the general kernel (merged with |prev|)
    abs_kw = dict(kw, prev=(kw["prev"][0].abs(), kw["prev"][1])) if kw.get("prev") else kw
    for entry, vx, kws in (("pa_attn_fwd_tile", v, kw), ("pa_attn_fwd", v, kw), ("pa_attn_fwd", v.abs(), abs_kw)):
        lse = torch.full((BH, N), 7.0, device=q.device)
        launch = pattn.prepare(q, k, vx, *lists, *kind, BQ, A, kernel="general", lse=lse, **kws)
        assert launch.entry == "pa_attn_fwd"
        launch.entry = entry
        with torch.cuda.device(q.device):
            o = launch()
        out.append((o.float(), lse))
    (o1, l1), (o2, l2), (oa, _) = out
    bound = _bound(oa, o2, 2, q.dtype, N, v)
    over = (o1 - o2).abs() / bound
    assert bool((over <= 1).all()), f"output differs by {float(over.max()):.2f} of its bound"
    assert torch.equal(torch.isneginf(l1), torch.isneginf(l2))
    fin = ~torch.isneginf(l2)
    assert float((l1[fin] - l2[fin]).abs().max()) < 2e-5 if bool(fin.any()) else True


def _built(mask, N, BQ, A, gpu):
    """(lists, wave codes, bitmaps) of a mask."""
    kv_idx, kv_num, kv_partial, wave, _, _, bits = pindex.build_device(mask, N, BQ, A, device=gpu, bits=True)
    return (kv_idx, kv_num, kv_partial), wave, bits


@pytest.mark.parametrize("bitmaps", [True, False])
@pytest.mark.parametrize("BQ,A", [(128, 16), (128, 32), (128, 128), (64, 16), (64, 64), (64, 128),
                                  (32, 16), (32, 32), (32, 128), (16, 16), (16, 32), (16, 64)])
@pytest.mark.parametrize("name,D,dtype,BH,N", [
    ("causal", 64, torch.float16, 3, 1152),            # odd list lengths, two groups of waves
    ("local256+str8", 64, torch.bfloat16, 2, 640),
    ("sinks4+win256", 128, torch.bfloat16, 2, 1152),
    ("twoband-1000", 128, torch.float16, 2, 2176),     # 34 segments apart: lists past 16 steps with gaps
    ("causal", 64, torch.bfloat16, 130, 1024),         # 1040 / 2080 work-groups: one group
    ("window-128", 128, torch.float16, 40, 1152),      # 360 / 720
    ("causal", 64, torch.float16, 9, 2048),            # 144 with long lists: blocks of 128 rows in two pieces
    ("window-128", 64, torch.bfloat16, 20, 1152),      # 180 / 360 with short ones: whole blocks, two groups
    ("window-128", 128, torch.bfloat16, 20, 1152),
])
def test_equals_general_kernel(gpu, name, D, dtype, BH, N, BQ, A, bitmaps):
    q, k, v = (x.to(gpu) for x in make_qkv(BH, N, D, dtype, seed=N + A))
    lists, wave, bits = _built(numpy_mask(name), N, BQ, A, gpu)
    _both(q, k, v, lists, triton_params(name), BQ, A, kv_wave_bits=wave, kv_bits=bits if bitmaps else None,
          heads_desc=bitmaps)


@pytest.mark.parametrize("name,D,BH,N", [
    # work-groups of 128 / 64 rows, whether the lists are uneven (a covering mask in order, 2048 and longer)
    ("causal", 128, 9, 2048),        # 144 / 288 uneven: two groups
    ("window-128", 128, 9, 2048),    # 144 / 288: one group for 64 rows
    ("causal", 64, 20, 2048),        # 320 / 640 uneven: pieces by two groups / two groups
    ("causal", 64, 26, 2048),        # 416 / 832 uneven: two groups
    ("window-128", 64, 20, 2048),    # 320 / 640: one group
    ("causal", 64, 40, 1024),        # 320 / 640, covering but shorter than 2048: one group
])
@pytest.mark.parametrize("BQ,A", [(128, 32), (64, 64)])
def test_groups_by_the_lists_evenness(gpu, name, D, BH, N, BQ, A):
    q, k, v = (x.to(gpu) for x in make_qkv(BH, N, D, torch.float16, seed=BH + N))
    lists, wave, bits = _built(numpy_mask(name), N, BQ, A, gpu)
    _both(q, k, v, lists, triton_params(name), BQ, A, kv_wave_bits=wave, kv_bits=bits)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("BQ,A", [(128, 32), (64, 64), (32, 32), (16, 16)])
def test_bases_strides_order_and_merge(gpu, BQ, A, D):
    """A table permutation of the mask alone, the closed-form residue basis gathered and
    scattered, rows that are not adjacent in memory, an issue order, and a merge input."""
    BH, N, s, name = 3, 2048, 8, "dilated-8"
    g = torch.Generator().manual_seed(D)
    # [N, BH, D] storage: row stride BH * D
    q, k, v = (torch.randn(N, BH, D, generator=g).to(torch.float16).to(gpu).transpose(0, 1) for _ in range(3))
    p = op.residue_perm(N, s)
    perm = torch.from_numpy(p).to(gpu)
    lists, wave, bits = _built(pm.Permuted(numpy_mask(name), p), N, BQ, A, gpu)
    order = torch.from_numpy(np.random.default_rng(1).permutation(N // BQ).astype(np.int32)).to(gpu)
    kind = triton_params(name)
    for kb in (bits, None):
        _both(q, k, v, lists, kind, BQ, A, kv_wave_bits=wave, kv_bits=kb, perm_q=perm, qblock_order=order)
        prev = (torch.randn(BH, N, D, generator=torch.Generator().manual_seed(3)).to(torch.float16).to(gpu),
                torch.randn(BH, N, generator=torch.Generator().manual_seed(4)).to(gpu))
        _both(q, k, v, lists, kind, BQ, A, kv_wave_bits=wave, kv_bits=kb, perm_q=perm, gather_q=True, gather_kv=True,
              scatter_o=True, residue=s, prev=prev)
    # no wave codes: the partial flags alone
    _both(q, k, v, lists, kind, BQ, A, kv_bits=bits, perm_q=perm)


@pytest.mark.parametrize("BQ", [16, 32, 64, 128])
def test_dead_rows_and_empty_lists(gpu, BQ):
    from polyhedral_amd.spec import device_mask
    N, D = 1024, 64
    M = numpy_mask("window-128").dense(N).copy()
    M[5] = False
    M[256:384] = False
    q, k, v = (x.to(gpu) for x in make_qkv(2, N, D, torch.float16, seed=1))
    dm = device_mask(pm.DenseMask(M), N, gpu)
    lists, wave, bits = _built(pm.DenseMask(M), N, BQ, 64, gpu)
    for kb in (bits, None):
        lse = torch.empty(2, N, device=gpu)
        launch = pattn.prepare(q, k, v, *lists, dm, 0, 0, 0, BQ, 64, kv_wave_bits=wave, kv_bits=kb, lse=lse)
        assert launch.entry == "pa_attn_fwd_tile"
        with torch.cuda.device(gpu):
            o = launch()
        dead = torch.zeros(N, dtype=torch.bool, device=gpu)
        dead[5] = dead[256:384] = True
        assert torch.count_nonzero(o[:, dead]) == 0 and torch.isneginf(lse[:, dead]).all()
        assert torch.isfinite(o).all() and torch.isfinite(lse[:, ~dead]).all()


@pytest.mark.parametrize("N", [16, 48, 80])
def test_narrow_blocks_of_a_short_sequence(gpu, N):
    """Heads whose 16-row units do not fill a work-group of four."""
    for D in (64, 128):
        q, k, v = (x.to(gpu) for x in make_qkv(3, N, D, torch.bfloat16, seed=N))
        lists, wave, bits = _built(numpy_mask("causal"), N, 16, 16, gpu)
        for kb in (bits, None):
            _both(q, k, v, lists, triton_params("causal"), 16, 16, kv_wave_bits=wave, kv_bits=kb)


@pytest.mark.parametrize("dtype,D,BQ,A,ext,want", [
    (torch.float16, 64, 128, 32, {}, "attn_tile_kernel"),
    (torch.bfloat16, 128, 64, 64, {}, "attn_tile_kernel"),
    (torch.bfloat16, 128, 128, 128, {}, "attn_tile_kernel"),
    (torch.float16, 128, 32, 16, {}, "attn_narrow_kernel"),
    (torch.bfloat16, 64, 16, 16, {}, "attn_narrow_kernel"),
    (torch.bfloat16, 128, 128, 32, {}, "attn_stream_kernel"),
    (torch.bfloat16, 128, 128, 32, dict(kernel="general"), "attn_fwd_kernel"),
    (torch.float16, 64, 64, 64, dict(kernel="general"), "attn_fwd_kernel"),
    (torch.float32, 64, 64, 64, {}, "attn_wsplit_kernel"),
    (torch.float32, 64, 16, 16, {}, "attn_fwd_kernel"),
    (torch.float16, 64, 64, 64, dict(perm=True), "attn_tile_kernel"),                   # the mask alone relabelled
    (torch.float16, 64, 64, 64, dict(perm=True, gather_kv=True), "attn_fwd_kernel"),    # through a table
    (torch.float16, 64, 64, 64, dict(perm=True, gather_kv=True, residue=8), "attn_tile_kernel"),
    (torch.float16, 64, 16, 16, dict(gather_mult=2), "attn_fwd_kernel"),
])
def test_the_kernel_a_call_takes(gpu, dtype, D, BQ, A, ext, want):
    N = 512
    q = torch.zeros(1, N, D, dtype=dtype, device=gpu)
    bi = pindex.build(numpy_mask("window-128"), N, BQ, A)
    ext = dict(ext)
    if ext.pop("perm", False):
        ext["perm_q"] = torch.from_numpy(op.residue_perm(N, 8)).to(gpu)
    launch = pattn.prepare(q, q, q, *pindex.to_cuda(bi), *triton_params("window-128"), BQ, A, **ext)
    assert launch.device_kernel == want


@pytest.mark.parametrize("name,D,BH,N,BQ,A", [
    # work-groups of BQ rows -> rows of waves, key groups, pieces of a block
    ("causal", 64, 3, 1152, 64, 64),        # 54: 2, 4, 1
    ("causal", 64, 20, 1024, 64, 32),       # 320: 2, 2, 1
    ("window-128", 64, 40, 1152, 64, 64),   # 720: 2, 1, 1
    ("causal", 64, 3, 1152, 128, 32),       # 27: 2, 4, 2
    ("causal", 64, 9, 2048, 128, 128),      # 144 uneven: 2, 2, 2
    ("window-128", 64, 20, 1152, 128, 16),  # 180: 4, 2, 1
    ("window-128", 64, 40, 1152, 128, 64),  # 360: 4, 1, 1
    ("causal", 128, 2, 1152, 64, 64),       # 36: 2, 2, 1
    ("window-128", 128, 40, 1152, 64, 32),  # 720: 2, 1, 1
    ("causal", 128, 2, 1152, 128, 128),     # 18: 2, 2, 2
    ("causal", 128, 20, 1152, 128, 32),     # 180: 4, 2, 1
    ("causal", 128, 40, 1152, 128, 128),    # 360: 4, 1, 1
    ("causal", 64, 3, 1152, 32, 32), ("causal", 128, 3, 1152, 32, 16),
    ("causal", 64, 3, 1152, 16, 16), ("causal", 128, 3, 1152, 16, 64),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_every_instantiation_equals_the_oracle(gpu, name, D, BH, N, BQ, A, dtype):
    q, k, v = make_qkv(BH, N, D, dtype, seed=BH + N + A)
    lists, wave, bits = _built(numpy_mask(name), N, BQ, A, gpu)
    rows = oatt.spec_rows(om.NAMED[name], N)
    heads = slice(BH - 1, BH)
    args = [as64(x[heads]) for x in (q, k, v)]
    want, want_lse = (torch.from_numpy(x) for x in oatt.dense_attention(*args, rows))
    oa = torch.from_numpy(oatt.dense_attention(args[0], args[1], abs(args[2]), rows)[0])
    bound = _bound(oa, want, 1, dtype, N, v)
    for kb in (bits, None):
        lse = torch.empty(BH, N, device=gpu)
        launch = pattn.prepare(*(x.to(gpu) for x in (q, k, v)), *lists, *triton_params(name), BQ, A, kernel="general",
                               kv_wave_bits=wave, kv_bits=kb, lse=lse)
        launch.entry = "pa_attn_fwd_tile"
        with torch.cuda.device(gpu):
            o = launch()
        over = (o[heads].double().cpu() - want).abs() / bound
        assert float(over.max()) <= 1, f"output off by {float(over.max()):.2f} of its bound"
        assert float((lse[heads].double().cpu() - want_lse).abs().max()) < 2e-5


@pytest.mark.parametrize("D", [64, 128])
def test_heads_of_up_to_4_gib(gpu, D):
    """Row offsets of K and V inside a head reach past 2 GiB (they are unsigned 32-bit numbers
    in the kernels) and, at 4 GiB, leave the call to the general kernel."""
    BH, N = 2, 512
    q, k, v = (x.to(gpu) for x in make_qkv(BH, N, D, torch.float16, seed=D))
    storage = torch.empty(2 ** 31, dtype=torch.float16, device=gpu)  # 4 GiB
    for row_bytes, entry in ((2 ** 23 - 16, "pa_attn_fwd_tile"), (2 ** 23, "pa_attn_fwd")):
        far = []
        for i, x in enumerate((k, v)):
            t = storage.as_strided((BH, N, D), (D, row_bytes // 2, 1), i * BH * D)
            t.copy_(x)
            far.append(t)
        for BQ, A in ((128, 128), (64, 64), (32, 32), (16, 16)):
            for name in ("causal", "window-128"):
                lists, wave, bits = _built(numpy_mask(name), N, BQ, A, gpu)
                kw = dict(kv_wave_bits=wave, kv_bits=bits)
                near = pattn.prepare(q, k, v, *lists, *triton_params(name), BQ, A, **kw)
                launch = pattn.prepare(q, *far, *lists, *triton_params(name), BQ, A, **kw)
                assert near.entry == "pa_attn_fwd_tile" and launch.entry == entry
                if entry == "pa_attn_fwd":
                    near = pattn.prepare(q, k, v, *lists, *triton_params(name), BQ, A, kernel="general", **kw)
                with torch.cuda.device(gpu):
                    assert torch.equal(launch(), near())
