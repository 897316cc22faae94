"""What infinities and NaN in the inputs do: the f16 / bf16 kernels on plain block lists
(pa_attn_fwd_tile) give them in the same places as the general kernel on the same arguments,
and rows that the forward found no weight for stay out of the backward."""
import pytest
import torch

from polyhedral_amd import attention as pattn
from polyhedral_amd import backward
from polyhedral_amd import index as pindex
from polyhedral_amd.polyattn import masks as pm
from tests.util import make_qkv

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
INF, NAN = float("inf"), float("nan")


def _v_inf(q, k, v):
    # one key of every 16-column segment, each in a column of its own (N / 16 <= D)
    for t in range(v.shape[1] // 16):
        v[:, 16 * t + (5 * t) % 16, t % v.shape[2]] = INF if t % 2 else -INF


def _v_nan(q, k, v):
    v[:, 37, 3] = NAN


def _q_nan(q, k, v):
    q[:, [0, 77, 300], 5] = NAN


def _q_inf(q, k, v):
    q[:, 130, 1] = INF
    q[:, 131, 2] = -INF


def _k_nan(q, k, v):
    k[:, 200, 0] = NAN


def _k_inf(q, k, v):
    # scores of +inf for some rows (their result is NaN), -inf for the others (no weight)
    k[:, 260] = 0
    k[:, 260, 0] = INF


INPUTS = {f.__name__[1:]: f for f in (_v_inf, _v_nan, _q_nan, _q_inf, _k_nan, _k_inf)}


@pytest.mark.parametrize("inputs", list(INPUTS))
@pytest.mark.parametrize("BQ,A", [(128, 16), (128, 32), (64, 16), (64, 64), (32, 16), (32, 32), (16, 16), (16, 64)])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
def test_same_places_as_the_general_kernel(gpu, D, dtype, BQ, A, inputs):
    # (a window of 100: lists of an odd number of 16-column segments)
    BH, N, w = 2, 512, 100
    q, k, v = make_qkv(BH, N, D, dtype, seed=BQ + A)
    big = float(v.float().abs().max())
    INPUTS[inputs](q, k, v)
    q, k, v = (x.to(gpu) for x in (q, k, v))
    kv_idx, kv_num, kv_partial, wave, _, _, bits = pindex.build_device(pm.SlidingWindow(w), N, BQ, A, device=gpu,
                                                                       bits=True)
    g = torch.Generator().manual_seed(7)
    prev = (torch.randn(BH, N, D, generator=g).to(dtype).to(gpu), torch.randn(BH, N, generator=g).to(gpu))
    for kb in (bits, None):
        for merge in (None, prev):
            out = []
            for entry in ("pa_attn_fwd", "pa_attn_fwd_tile"):
                lse = torch.full((BH, N), 7.0, device=gpu)
                launch = pattn.prepare(q, k, v, kv_idx, kv_num, kv_partial, pattn.WINDOW, w, 0, 0, BQ, A,
                                       kernel="general", kv_wave_bits=wave, kv_bits=kb, lse=lse, prev=merge)
                launch.entry = entry
                with torch.cuda.device(gpu):
                    out.append((launch().float(), lse))
            for name, a, b in zip(("o", "lse"), *out):
                for what, f in (("NaN", torch.isnan), ("+inf", torch.isposinf), ("-inf", torch.isneginf)):
                    d = f(a) != f(b)
                    assert not bool(d.any()), f"{name}: {int(d.sum())} values differ in being {what}"
            (o1, l1), (o2, l2) = ((torch.nan_to_num(o, 0, 0, 0), torch.nan_to_num(x, 0, 0, 0)) for o, x in out)
            eps = EPS[dtype]
            # (P is rounded at another running maximum: at most 2 eps sum p |v|, and an ulp of the result's rounding)
            assert bool(((o1 - o2).abs() <= 2 * eps * big + 2 * eps * o1.abs()).all())
            assert float((l1 - l2).abs().max()) < 2e-5


@pytest.mark.parametrize("bitmaps", [True, False])
@pytest.mark.parametrize("BH", [2, 40])  # 16 work-groups of two groups of waves, 320 of one
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
def test_backward_rows_without_weight(gpu, D, dtype, BH, bitmaps):
    """A row whose lse is -inf (no live key, or scores that are not finite: the forward gives
    both) has P = 0 whatever its scores: dV of every key and dQ of every row are those of the
    same row with finite values."""
    N = 512
    q, k, v = (x.to(gpu) for x in make_qkv(BH, N, D, dtype, seed=D))
    o, do, _ = (x.to(gpu) for x in make_qkv(BH, N, D, dtype, seed=D + 1))
    lse = torch.full((BH, N), 6.0, device=gpu)
    rows = [0, 77, 200, 511]  # in partial tiles and in full ones
    lse[:, rows] = -INF
    o[:, rows] = 0
    plan = backward.BackwardPlan(pm.Causal(), N, gpu, bitmaps=bitmaps)
    dq, _, dv = plan.backward(q, k, v, o, lse, do)
    assert bool(torch.isfinite(dq).all()) and bool(torch.isfinite(dv).all())
    assert torch.count_nonzero(dq[:, rows]) == 0
    for value in (NAN, INF):
        bad = q.clone()
        bad[:, rows, 3] = value
        dq2, _, dv2 = plan.backward(bad, k, v, o, lse, do)
        assert torch.equal(dv, dv2) and torch.equal(dq, dq2)
    # the last key, which only the last row (without weight) sees
    bad = k.clone()
    bad[:, 511, 3] = INF
    assert torch.equal(plan.backward(q, bad, v, o, lse, do)[2], dv)
