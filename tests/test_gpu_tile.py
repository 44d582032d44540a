"""The 128-row MFMA tile kernel (csrc/tile_gemm.hip) at the edges of its tiles:
expert row counts around every tile height (multiples of 32 rows), one to nine
128-k chunks (its chunk buffers are four deep up to 64 rows, two above), K and N
that leave partial chunks and column tiles, groups of 64 and 128, and more
tiles than workgroups.

INT4 rows meet the fp32-summation bound of test_gpu_int4_exact; the MXFP4 MLP is
held to the relative-L2 bound of test_gpu_mxfp4.
"""
from __future__ import annotations

import pytest
import torch

from oracle.torch_ref import moe_mxfp4_ref
from tests._helpers import softmax_weights
from tests.test_capi import _mxfp4_tiles
from tests.test_gpu_int4_exact import _bounded_check, _device_inputs, _gemm_rows
from xkernels_amd import Backend, _lib, fused_moe_mxfp4, make_mxfp4_moe_weights

pytestmark = pytest.mark.gpu

ROWS = [1, 16, 31, 32, 33, 64, 65, 0, 96, 97, 127, 128, 129, 257]


def _row_ids(rows, seed):
    """top_k = 1 routing with exactly rows[e] tokens on expert e, shuffled."""
    ids = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(rows)])
    return ids[torch.randperm(ids.numel(), generator=torch.Generator().manual_seed(seed))].reshape(-1, 1)


@pytest.mark.parametrize("N,K,gs", [(256, 512, 32), (272, 1024, 32), (512, 2048, 32), (256, 1536, 32)]
                         + [(48, 128 * c, 32) for c in (1, 2, 3, 5, 7, 9)]
                         + [(304, 32, 32), (256, 96, 32), (256, 160, 32), (256, 640, 64), (528, 1152, 128)])
def test_int4_tile_edges(N, K, gs, dev):
    ids = _row_ids(ROWS, K)
    print(f"int4 tile N={N} K={K} gs={gs}", flush=True)
    A, packed, scale, ids = _device_inputs(ids.shape[0], len(ROWS), N, K, ids, seed=K + N, gs=gs)
    # 77 rows per expert on average: the 128-row kernel
    rows = _gemm_rows(A, packed, scale, ids, flags=_lib._XK_INT4_TEST_FORCE_TILE, gs=gs)
    assert not torch.isnan(rows).any(), "a routed slot's row was not written"
    _bounded_check(A, packed, scale, ids, rows, gs=gs)


@pytest.mark.parametrize("N", [16, 48, 272])
@pytest.mark.parametrize("K,gs", [(32, 32), (160, 32), (2080, 32), (192, 64), (2048, 32)])
@pytest.mark.parametrize("M", [1, 2])
def test_int4_tile_of_one_row(N, K, gs, M, dev):
    """Activations, weights and scales that are shorter than the last chunk's
    offset into them: the loads past K, past N and of pad rows return zeros
    whatever part of their offset the range check counts."""
    print(f"int4 tile M={M} N={N} K={K} gs={gs}", flush=True)
    ids = torch.tensor([[1], [0]][:M], dtype=torch.int32)
    A, packed, scale, ids = _device_inputs(M, 2, N, K, ids, seed=K + N + M, gs=gs)
    rows = _gemm_rows(A, packed, scale, ids, flags=_lib._XK_INT4_TEST_FORCE_TILE, gs=gs)
    assert not torch.isnan(rows).any(), "a routed slot's row was not written"
    _bounded_check(A, packed, scale, ids, rows, gs=gs)


@pytest.mark.parametrize("hidden,ispp", [(32, 32), (32, 160), (160, 32), (2080, 160), (160, 2080)])
def test_mxfp4_one_token(hidden, ispp, dev):
    """The same for one token's activation row in both MXFP4 projections."""
    print(f"mxfp4 one token hidden={hidden} ispp={ispp}", flush=True)
    wts = make_mxfp4_moe_weights(2, hidden, ispp, with_bias=True, device="cpu", seed=ispp, scale_lo=115, scale_hi=122)
    A = torch.randn(1, hidden, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    ids, w = torch.tensor([[1]], dtype=torch.int32), torch.full((1, 1), 0.7)
    keys = ("w13", "w13_scale", "w2", "w2_scale")
    got = fused_moe_mxfp4(A.to(dev), *(wts[k].to(dev) for k in keys), ids.to(dev), w.to(dev),
                          b13=wts["b13"].to(dev), b2=wts["b2"].to(dev), backend=Backend.HIP).float().cpu()
    want = moe_mxfp4_ref(A, *(wts[k] for k in keys), ids, w, b13=wts["b13"], b2=wts["b2"]).float()
    # one slot of few columns: a bf16 rounding of a sum that falls on the other
    # side of a tie moves that column by 2^-8 of its size
    assert float((got - want).norm() / want.norm()) < 4e-3


@pytest.mark.parametrize("queue_bytes", [32, 256, 1024, 4096])
@pytest.mark.parametrize("E,N", [(63, 2048), (64, 2048), (64, 2064), (65, 2048), (200, 2048)])
def test_queue_of_any_spacing_takes_every_tile_once(E, N, queue_bytes, dev):
    """Tile counts around the 512 places (up to them the tiles are dealt without
    the queue) and far above, with the XCDs' counters 4 to 128 bytes apart: the
    rows equal the static deal's bit for bit, from a buffer of NaNs, twice with
    one queue of old counts."""
    from tests.test_gpu_int4_prefill import _inputs, _slot_rows
    K, M = 256, E * 20
    print(f"tile queue E={E} N={N} bytes={queue_bytes}", flush=True)
    ids = torch.arange(E, dtype=torch.int32).repeat_interleave(20).reshape(M, 1)
    A, packed, scale, ids, _ = _inputs(M, E, N, K, ids, seed=E)
    force = _lib._XK_INT4_TEST_FORCE_TILE
    static = _slot_rows(A, packed, scale, ids, force)
    queue = torch.randint(0, 256, (queue_bytes,), dtype=torch.uint8, device=dev)
    for _ in range(2):
        queued = _slot_rows(A, packed, scale, ids, force, queue)
        torch.cuda.synchronize()
        assert not torch.isnan(queued).any(), "a routed slot row was not written"
        assert torch.equal(queued, static)


@pytest.mark.parametrize("hidden,ispp", [(512, 512), (1024, 160), (96, 512), (32, 32), (2080, 96), (544, 1536)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_mxfp4_tile_edges(hidden, ispp, dtype, dev):
    E, M = len(ROWS), sum(ROWS)
    print(f"mxfp4 tile hidden={hidden} ispp={ispp} {dtype}", flush=True)
    wts = make_mxfp4_moe_weights(E, hidden, ispp, with_bias=True, device="cpu", seed=hidden, scale_lo=115,
                                 scale_hi=122)
    wts["w13_scale"][0, 3, 0] = 255  # the reserved scale code reads as 0
    wts["w2_scale"][1, 5, 0] = 255
    A = torch.randn(M, hidden, generator=torch.Generator().manual_seed(1)).to(dtype)
    ids, w = _row_ids(ROWS, ispp), softmax_weights(M, 1, 3) * 0.7
    keys = ("w13", "w13_scale", "w2", "w2_scale")
    got = fused_moe_mxfp4(A.to(dev), *(wts[k].to(dev) for k in keys), ids.to(dev), w.to(dev),
                          b13=wts["b13"].to(dev), b2=wts["b2"].to(dev), backend=Backend.HIP)
    want = moe_mxfp4_ref(A, *(wts[k] for k in keys), ids, w, b13=wts["b13"], b2=wts["b2"])
    assert got.dtype == dtype
    got, want = got.float().cpu(), want.float()
    assert torch.isfinite(got).all()
    # bf16 roundings of the gate/up sums, the activation and the down sums that
    # fall on other sides of a tie: 2^-9 relative each on a small share of terms
    assert float((got - want).norm() / want.norm()) < 2e-3


# 128-row blocks and tails of every height, at rows enough for tiles of any K
LONG_ROWS = [770, 801, 897, 577]


@pytest.mark.parametrize("hidden,ispp", [(32, 32), (96, 32), (160, 96), (2080, 160), (544, 1376)])
def test_mxfp4_tiles_of_short_contractions(hidden, ispp, dev):
    """K below, between and past the multiples of a chunk (128) and of a scale
    block (512), in both projections."""
    E, M = len(LONG_ROWS), sum(LONG_ROWS)
    print(f"mxfp4 tiles hidden={hidden} ispp={ispp}", flush=True)
    assert _mxfp4_tiles(M, E, hidden, ispp, 1) == (True, True)
    wts = make_mxfp4_moe_weights(E, hidden, ispp, with_bias=True, device="cpu", seed=hidden, scale_lo=115,
                                 scale_hi=122)
    A = torch.randn(M, hidden, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    ids, w = _row_ids(LONG_ROWS, ispp), softmax_weights(M, 1, 3) * 0.7
    keys = ("w13", "w13_scale", "w2", "w2_scale")
    got = fused_moe_mxfp4(A.to(dev), *(wts[k].to(dev) for k in keys), ids.to(dev), w.to(dev),
                          b13=wts["b13"].to(dev), b2=wts["b2"].to(dev), backend=Backend.HIP).float().cpu()
    want = moe_mxfp4_ref(A, *(wts[k] for k in keys), ids, w, b13=wts["b13"], b2=wts["b2"]).float()
    assert torch.isfinite(got).all()
    # the bound of test_mxfp4_tile_edges
    assert float((got - want).norm() / want.norm()) < 2e-3


@pytest.mark.parametrize("hidden,ispp,tiles", [(60064, 32, (True, False)), (32, 60064, (False, True))])
def test_mxfp4_tile_of_one_token(hidden, ispp, tiles, dev):
    """One activation row and a partial last chunk, at a contraction long enough
    that one token takes the tile kernel: loads past K and of pad rows land zeros
    though their scalar offset passes the end of A."""
    assert _mxfp4_tiles(1, 1, hidden, ispp, 1, False) == tiles
    print(f"mxfp4 one token in tiles hidden={hidden} ispp={ispp}", flush=True)
    wts = make_mxfp4_moe_weights(1, hidden, ispp, with_bias=True, device="cpu", seed=3, scale_lo=112, scale_hi=118)
    A = torch.randn(1, hidden, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    ids, w = torch.zeros(1, 1, dtype=torch.int32), torch.full((1, 1), 0.7)
    keys = ("w13", "w13_scale", "w2", "w2_scale")
    # fp32 activations: no stream kernel
    got = fused_moe_mxfp4(A.float().to(dev), *(wts[k].to(dev) for k in keys), ids.to(dev), w.to(dev),
                          b13=wts["b13"].to(dev), b2=wts["b2"].to(dev), backend=Backend.HIP).cpu()
    want = moe_mxfp4_ref(A.float(), *(wts[k] for k in keys), ids, w, b13=wts["b13"], b2=wts["b2"])
    # the bound of test_mxfp4_one_token
    assert float((got - want).norm() / want.norm()) < 4e-3
