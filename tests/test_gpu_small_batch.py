"""The one-launch kernels of the smallest decode batches (csrc/small_batch.hip):
one to six tokens, up to 64 routed slots, duplicated experts within a token,
dropped slots under an expert map, no routed slot at all, unweighted sums, more
column blocks than compute units, one 512-k unit and many, and the first sizes
past their limits (7 tokens, 65 slots, more experts than the INT4 kernel takes at
few columns), against the oracle."""
from __future__ import annotations

import pytest
import torch

from oracle.torch_ref import moe_mxfp4_ref, moe_w4a16_ref
from tests._helpers import assert_close, softmax_weights
from xkernels_amd import (Backend, fused_moe_int4_w4a16, fused_moe_mxfp4, make_mxfp4_moe_weights,
                          make_w4a16_weights)

pytestmark = pytest.mark.gpu

CASES = [(1, 8, 1), (1, 8, 8), (2, 4, 4), (3, 48, 8), (6, 16, 8), (6, 3, 10), (1, 64, 64), (7, 8, 8), (5, 16, 13),
         (1, 3, 64), (2, 12, 32)]


def _route(M, E, k, seed):
    """Random experts (duplicates within a token included)."""
    return torch.randint(0, E, (M, k), generator=torch.Generator().manual_seed(seed), dtype=torch.int32)


def _emap(E, seed):
    """Every second of 2 E global experts is local, in shuffled order."""
    m = torch.full((2 * E,), -1, dtype=torch.int32)
    m[::2] = torch.randperm(E, generator=torch.Generator().manual_seed(seed)).to(torch.int32)
    return m


@pytest.mark.parametrize("M,E,k", CASES)
@pytest.mark.parametrize("N,K", [(16, 512), (4112, 1024), (256, 3584)])
@pytest.mark.parametrize("mode", ["plain", "map", "unweighted"])
def test_int4(M, E, k, N, K, mode, dev):
    packed, scale, _ = make_w4a16_weights(E, N, K, 32, device="cpu", seed=M + E, scale_hi=0.02)
    A = torch.randn(M, K, generator=torch.Generator().manual_seed(K)).to(torch.bfloat16)
    emap = _emap(E, 5) if mode == "map" else None
    ids, w = _route(M, 2 * E if mode == "map" else E, k, M * k), softmax_weights(M, k, 3)
    kw = dict(mul_routed_weight=mode != "unweighted", expert_map=emap)
    want = moe_w4a16_ref(A, packed, scale, ids, w, **kw)
    if emap is not None:
        kw["expert_map"] = emap.to(dev)
    got = fused_moe_int4_w4a16(A.to(dev), packed.to(dev), scale.to(dev), ids.to(dev), w.to(dev),
                               backend=Backend.HIP, **kw)
    # the op spec's bf16 tolerance at the output's own scale (sums cancel)
    assert_close(got, want, 2e-2, 2e-2 * float(want.float().abs().mean()) + 1e-6, f"int4 {mode}")


@pytest.mark.parametrize("M,E,k", CASES)
@pytest.mark.parametrize("hidden,ispp", [(512, 512), (1536, 512), (512, 1024)])
@pytest.mark.parametrize("mode", ["plain", "map", "unweighted"])
def test_mxfp4(M, E, k, hidden, ispp, mode, dev):
    wts = make_mxfp4_moe_weights(E, hidden, ispp, with_bias=mode != "plain", device="cpu", seed=M + k, scale_lo=115,
                                 scale_hi=122)
    wts["w13_scale"][0, 7, 1] = 255  # the reserved scale code reads as 0
    wts["w2_scale"][E - 1, 3, 2] = 255
    A = torch.randn(M, hidden, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16)
    emap = _emap(E, 6) if mode == "map" else None
    ids, w = _route(M, 2 * E if mode == "map" else E, k, M + k), softmax_weights(M, k, 4)
    kw = dict(mul_routed_weight=mode != "unweighted", expert_map=emap)
    keys = ("w13", "w13_scale", "w2", "w2_scale")
    want = moe_mxfp4_ref(A, *(wts[n] for n in keys), ids, w, b13=wts["b13"], b2=wts["b2"], **kw)
    d = lambda t: None if t is None else t.to(dev)  # noqa: E731
    if emap is not None:
        kw["expert_map"] = emap.to(dev)
    got = fused_moe_mxfp4(d(A), *(d(wts[n]) for n in keys), d(ids), d(w), b13=d(wts["b13"]), b2=d(wts["b2"]),
                          backend=Backend.HIP, **kw).float().cpu()
    want = want.float()
    # relative L2 of test_gpu_mxfp4's full-scale test: bf16 roundings of the
    # gate/up, activation and down values that fall on other sides of a tie
    assert float((got - want).norm()) <= 2e-3 * float(want.norm()) + 1e-6


def test_no_routed_slot(dev):
    """Every slot dropped: the output is zero."""
    packed, scale, _ = make_w4a16_weights(4, 256, 512, 32, device=dev, seed=1)
    A = torch.randn(2, 512, device=dev).to(torch.bfloat16)
    ids, w = torch.full((2, 3), 9, dtype=torch.int32, device=dev), torch.ones(2, 3, device=dev)
    assert not fused_moe_int4_w4a16(A, packed, scale, ids, w, backend=Backend.HIP).any()
