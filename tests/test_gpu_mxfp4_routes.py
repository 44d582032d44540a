"""fused_moe_mxfp4 off its stream path: 32-row passes, 128-row tiles, and one for
each projection, as the rows per expert, the contraction and the number of tiles choose. fp32
activations, sizes that are odd multiples of 32, more than 512 experts, scales
at odd addresses and expert maps, each at few and at many rows, against the
oracle; every scratch byte starts as a NaN pattern, so a row that nothing wrote
and something read would show."""
from __future__ import annotations

import pytest
import torch

from oracle.torch_ref import moe_mxfp4_ref
from tests._helpers import softmax_weights, uniform_topk, zipf_topk
from tests.test_capi import _mxfp4_tiles
from xkernels_amd import Backend, MoeMxfp4Workspace, fused_moe_mxfp4, make_mxfp4_moe_weights

pytestmark = pytest.mark.gpu
KEYS = ("w13", "w13_scale", "w2", "w2_scale")


def _check(M, E, hidden, ispp, k, dev, dtype=torch.bfloat16, experts=0, routing="uniform", shift=0):
    print(f"mxfp4 M={M} E={E} hidden={hidden} ispp={ispp} k={k} {dtype} of {experts} {routing}", flush=True)
    n = experts or E
    ids = uniform_topk(M, k, n, 3) if routing == "uniform" else zipf_topk(M, k, n, 1.2, 3)
    kw = {}
    if experts:  # the first E are local
        kw["expert_map"] = torch.cat([torch.arange(E), torch.full((experts - E,), -1)]).to(torch.int32)
    w = softmax_weights(M, k, 4)
    wts = make_mxfp4_moe_weights(E, hidden, ispp, with_bias=True, device="cpu", seed=hidden, scale_lo=115,
                                 scale_hi=122)
    wts["w13_scale"][0, 3, 0] = 255  # the reserved scale code reads as 0
    wts["w2_scale"][E - 1, 5, -1] = 255
    A = torch.randn(M, hidden, generator=torch.Generator().manual_seed(1)).to(dtype)
    ws = MoeMxfp4Workspace.allocate(M, k, E, 16, ispp, hidden, dtype=dtype, device=dev)
    ws.scratch.fill_(255)
    ws.out.fill_(float("nan"))
    d = {name: t.to(dev) for name, t in wts.items()}
    for name in ("w13_scale", "w2_scale"):  # the same bytes `shift` past an aligned address
        if shift:
            raw = torch.zeros(d[name].numel() + shift, dtype=torch.uint8, device=dev)
            raw[shift:] = d[name].reshape(-1)
            d[name] = raw[shift:].view(d[name].shape)
    dkw = {name: t.to(dev) for name, t in kw.items()}
    got = fused_moe_mxfp4(A.to(dev), *(d[n] for n in KEYS), ids.to(dev), w.to(dev), b13=d["b13"], b2=d["b2"],
                          backend=Backend.HIP, workspace=ws, **dkw)
    assert got.data_ptr() == ws.out.data_ptr() and got.dtype == dtype
    got = got.float().cpu()
    want = moe_mxfp4_ref(A, *(wts[n] for n in KEYS), ids, w, b13=wts["b13"], b2=wts["b2"], **kw).float()
    assert torch.isfinite(got).all()
    # bf16 roundings of the gate/up sums, the activation and the down sums that
    # fall on other sides of a tie: 2^-9 relative each on a small share of terms
    assert float((got - want).norm()) <= 2e-3 * float(want.norm()) + 1e-6


@pytest.mark.parametrize("M,E,hidden,ispp,k,routing,tiles", [  # tiles: of gate/up, of down; else passes
    (1, 8, 512, 512, 2, "uniform", (False, False)),
    (33, 2, 256, 160, 2, "uniform", (False, False)),  # 33 rows an expert: two passes
    (40, 4, 544, 96, 1, "zipf", (False, False)),
    (300, 8, 2048, 256, 4, "zipf", (True, True)),
    (300, 8, 2048, 64, 4, "zipf", (True, False)),
    (600, 8, 32, 1536, 4, "zipf", (False, True)),
    (600, 8, 2048, 1408, 4, "zipf", (True, True)),
])
def test_fp32_activations(M, E, hidden, ispp, k, routing, tiles, dev):
    assert _mxfp4_tiles(M, E, hidden, ispp, k, True) == tiles
    _check(M, E, hidden, ispp, k, dev, dtype=torch.float32, routing=routing)


@pytest.mark.parametrize("hidden,ispp", [(32, 32), (160, 96), (96, 544), (2080, 160)])
@pytest.mark.parametrize("M,E,k,routing", [(3, 4, 2, "uniform"), (65, 4, 1, "zipf"), (150, 5, 2, "uniform")])
def test_odd_multiples_of_32(hidden, ispp, M, E, k, routing, dev):
    _check(M, E, hidden, ispp, k, dev, routing=routing)


@pytest.mark.parametrize("M,tiles", [(7, False), (300, False), (6000, True)])
def test_more_than_512_experts(M, tiles, dev):
    assert _mxfp4_tiles(M, 600, 256, 128, 8) == (tiles, tiles)
    _check(M, 600, 256, 128, 8, dev)


@pytest.mark.parametrize("hidden,ispp,shift", [(192, 64, 1), (192, 320, 3), (160, 96, 1)])
@pytest.mark.parametrize("M", [5, 120])
def test_scales_at_odd_addresses(hidden, ispp, shift, M, dev):
    _check(M, 4, hidden, ispp, 2, dev, shift=shift)


@pytest.mark.parametrize("M,E,experts,hidden,ispp,k", [
    (60, 8, 64, 256, 192, 6),      # few local rows of many slots: passes
    (300, 4, 16, 256, 96, 4),      # 75 local rows an expert, three passes
    (300, 4, 16, 1024, 96, 4),     # tiles for gate/up, passes for down
    (400, 4, 16, 96, 1024, 4),     # the other way round
    (400, 4, 16, 2048, 1024, 4),   # tiles for both
    (64, 2, 64, 544, 160, 8),
    (200, 4, 8, 512, 512, 3),      # top_k with no fixed-size combine
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_expert_map(M, E, experts, hidden, ispp, k, dtype, dev):
    """Slots of other ranks' experts: no row of theirs is written or read."""
    _check(M, E, hidden, ispp, k, dev, dtype=dtype, experts=experts)


def test_batch_past_buffer_reach_runs_in_token_chunks(dev):
    """262,145 tokens of 4096: activations past the 2^31 bytes that the tile kernel
    addresses run as token chunks; a token's output depends only on its own slots,
    so it equals two calls over another split of the batch bit for bit."""
    M, E, hidden, ispp, cut = 262_145, 4, 4096, 64, 100_001
    wts = make_mxfp4_moe_weights(E, hidden, ispp, device=dev, seed=3, scale_lo=115, scale_hi=122)
    g = torch.Generator(device=dev).manual_seed(5)
    A = torch.randn(M, hidden, generator=g, device=dev, dtype=torch.bfloat16)
    ids = torch.randint(0, E, (M, 1), generator=g, device=dev, dtype=torch.int32)
    w = torch.rand(M, 1, generator=g, device=dev) + 0.5
    call = lambda a, b: fused_moe_mxfp4(A[a:b], *(wts[n] for n in KEYS), ids[a:b], w[a:b],  # noqa: E731
                                        backend=Backend.HIP)
    whole = call(0, M)
    parts = torch.cat([call(0, cut), call(cut, M)])
    assert torch.isfinite(whole.float()).all()
    assert torch.equal(whole, parts)
