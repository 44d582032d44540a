"""xk_moe_topk_combine under an expert map: dropped slots' rows hold NaNs and are
never used, at row widths around a wavefront and a workgroup (a workgroup per row
part) and below (rows share a workgroup), 1-, 4- and 8-wide rows, one and several
partial planes; and a batch of more rows than one launch has workgroups."""
from __future__ import annotations

import pytest
import torch

from xkernels_amd import _lib

pytestmark = pytest.mark.gpu


def _combine(y, w, ids, emap, local, out_dtype):
    parts, M, k, N = y.shape
    out = torch.empty(M, N, dtype=out_dtype, device=y.device)
    _lib.call("xk_moe_topk_combine", y.data_ptr(), M, k, N, None if w is None else w.data_ptr(), int(w is not None),
              ids.data_ptr(), local, None if emap is None else emap.data_ptr(), 0 if emap is None else emap.numel(),
              out.data_ptr(), _lib.XK_DT_BF16 if out_dtype == torch.bfloat16 else _lib.XK_DT_FP32, parts,
              torch.cuda.current_stream().cuda_stream)
    return out


@pytest.mark.parametrize("N", [3, 8, 128, 252, 256, 260, 1020, 1024, 1028, 2880])
@pytest.mark.parametrize("M,k,parts", [(5, 8, 1), (33, 3, 2), (70, 2, 3), (7, 1, 1), (2100, 6, 1)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_dropped_slots(N, M, k, parts, out_dtype, dev):
    print(f"combine N={N} M={M} k={k} parts={parts} {out_dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(N + M)
    experts, local = 12, 4
    emap = torch.full((experts,), -1, dtype=torch.int32, device=dev)
    emap[::3] = torch.arange(local, dtype=torch.int32, device=dev)
    ids = torch.randint(0, experts + 1, (M, k), generator=g, device=dev, dtype=torch.int32)  # 12: outside the map
    keep = (ids < experts) & (ids % 3 == 0)
    y = torch.randn(parts, M, k, N, generator=g, device=dev)
    y[:, ~keep] = float("nan")
    for w in (torch.rand(M, k, generator=g, device=dev), None):
        got = _combine(y, w, ids, emap, local, out_dtype)
        rows = y.double().sum(0) * (1.0 if w is None else w.double().unsqueeze(-1))
        want = torch.where(keep.unsqueeze(-1), rows, torch.zeros_like(rows)).sum(1)
        # fp32 sums of at most 18 terms of size one; bf16 adds its own rounding
        tol = 1e-5 + (2.0 ** -8 if out_dtype == torch.bfloat16 else 2e-6) * want.abs()
        assert ((got.double() - want).abs() <= tol).all()


def test_more_rows_than_workgroups(dev):
    """2^24 rows and more: a workgroup for each would pass the 2^32 threads a launch takes."""
    M, N = (1 << 24) + 5, 8
    ids = torch.arange(M, device=dev, dtype=torch.int32).remainder_(3).view(M, 1)
    emap = torch.tensor([0, -1, 1], dtype=torch.int32, device=dev)
    y = torch.arange(M, device=dev, dtype=torch.float32).remainder_(1021).view(1, M, 1, 1).expand(1, M, 1, N).contiguous()
    got = _combine(y, None, ids, emap, 2, torch.float32)
    want = torch.where(ids == 1, torch.zeros_like(y.view(M, N)), y.view(M, N))
    assert torch.equal(got, want)
