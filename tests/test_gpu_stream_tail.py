"""The weight-streaming kernel (csrc/int4_stream.hip) where K ends inside a 256-k
line: MXFP4 rows of an even scale count that is no multiple of four (2-byte scale
loads) over one to twelve lines and two blocks of scales, several 16-row passes,
dropped slots under an expert map and align-fed batches, against the oracle; and
columns whose neighbour holds infinite weights where their own row has ended."""
from __future__ import annotations

import pytest
import torch

from oracle.torch_ref import moe_mxfp4_ref
from tests._helpers import softmax_weights, uniform_topk, zipf_topk
from tests.test_gpu_int4_exact import REL, REL_F32, _bounded_check, _device_inputs, _gemm_rows
from xkernels_amd import Backend, _lib, fused_moe_mxfp4, make_mxfp4_moe_weights

pytestmark = pytest.mark.gpu
KEYS = ("w13", "w13_scale", "w2", "w2_scale")


def _mxfp4(A, wts, ids, w, dev, **kw):
    d = lambda t: None if t is None else t.to(dev)  # noqa: E731
    return fused_moe_mxfp4(d(A), *(d(wts[k]) for k in KEYS), d(ids), d(w), b13=d(wts["b13"]), b2=d(wts["b2"]),
                           backend=Backend.HIP, **kw).float().cpu()


def _ref(A, wts, ids, w, **kw):
    return moe_mxfp4_ref(A, *(wts[k] for k in KEYS), ids, w, b13=wts["b13"], b2=wts["b2"], **kw).float()


@pytest.mark.parametrize("hidden,ispp", [(192, 320), (320, 192), (2112, 192), (192, 2112), (2880, 2880)])
@pytest.mark.parametrize("M,E,k,routing", [(1, 4, 2, "uniform"), (7, 4, 3, "uniform"), (64, 8, 2, "zipf"),
                                           (530, 256, 8, "uniform")])
@pytest.mark.parametrize("ep", [False, True])
def test_mxfp4_partial_line(hidden, ispp, M, E, k, routing, ep, dev):
    """530 x 8 slots are more than the kernel routes by itself: align-fed."""
    if hidden * ispp > 1 << 20 and E > 8:
        E, M = 32, 75  # 2880 x 2880: 600 slots, 19 rows per expert
    print(f"mxfp4 tail M={M} E={E} k={k} hidden={hidden} ispp={ispp} {routing} ep={ep}", flush=True)
    ids = uniform_topk(M, k, E, 3) if routing == "uniform" else zipf_topk(M, k, E, 1.2, 3)
    w = softmax_weights(M, k, 4)
    kw = {}
    local = E
    if ep:  # every second expert is local
        local = E // 2
        emap = torch.full((E,), -1, dtype=torch.int32)
        emap[::2] = torch.arange(local, dtype=torch.int32)
        kw["expert_map"] = emap
    wts = make_mxfp4_moe_weights(local, hidden, ispp, with_bias=True, device="cpu", seed=hidden, scale_lo=115,
                                 scale_hi=122)
    wts["w13_scale"][:, 3, -1] = 255  # the reserved scale code in the last, partial line reads as 0
    wts["w2_scale"][:, 5, -1] = 255
    A = torch.randn(M, hidden, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    got = _mxfp4(A, wts, ids, w, dev, **kw)
    want = _ref(A, wts, ids, w, **kw)
    assert torch.isfinite(got).all()
    # bf16 roundings of the gate/up sums, the activation and the down sums that
    # fall on other sides of a tie: 2^-9 relative each on a small share of terms
    assert float((got - want).norm()) <= 2e-3 * float(want.norm()) + 1e-6


@pytest.mark.parametrize("ispp", [64, 192, 320, 384, 640])
def test_mxfp4_infinite_neighbour(ispp, dev):
    """Scale byte 254 and weights of 4 or more make the first groups of every
    third down-projection row infinite; the rows before them stay finite."""
    M, E, hidden, k = 5, 4, 256, 2
    wts = make_mxfp4_moe_weights(E, hidden, ispp, with_bias=True, device="cpu", seed=ispp, scale_lo=115, scale_hi=122)
    wts["w2_scale"][:, 2::3, :6] = 254
    wts["w2"][:, 2::3, :96] |= 0x66
    A = torch.randn(M, hidden, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    ids, w = uniform_topk(M, k, E, 3), softmax_weights(M, k, 4)
    got, want = _mxfp4(A, wts, ids, w, dev), _ref(A, wts, ids, w)
    keep = torch.arange(hidden) % 3 != 2
    assert torch.isfinite(want[:, keep]).all() and not torch.isfinite(want[:, ~keep]).all()
    assert torch.isfinite(got[:, keep]).all()
    assert float((got - want)[:, keep].norm() / want[:, keep].norm()) < 4e-3


@pytest.mark.parametrize("N,K,gs", [(64, 96, 32), (48, 320, 32), (64, 384, 64), (80, 2080, 32), (64, 640, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_int4_infinite_neighbour(N, K, gs, dtype, dev):
    ids = uniform_topk(5, 2, 4, 3)
    A, packed, scale, ids = _device_inputs(5, 4, N, K, ids, seed=K, gs=gs)
    A = A.to(dtype)
    scale[:, 2::3, :3] = float("inf")
    rows = _gemm_rows(A, packed, scale, ids, flags=_lib._XK_INT4_TEST_FORCE_STREAM, gs=gs)
    keep = torch.arange(N, device=rows.device) % 3 != 2
    assert torch.isfinite(rows[:, keep]).all()
    _bounded_check(A, packed[:, keep].contiguous(), scale[:, keep].contiguous(), ids, rows[:, keep], gs=gs,
                   rel=REL_F32 if dtype == torch.float32 else REL, w_dtype=dtype)
