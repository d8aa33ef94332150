"""The forward state scan at the sizes where its unit mapping and pipeline can go
wrong: one to four chunks (fewer than it loads ahead, odd and even), a short last
chunk, unit counts that are not a multiple of the 8 XCDs, and both column-slice
widths (16 while every slice has a CU of its own, 32 beyond that), with and
without an entry state, against the float64 token recurrence."""
import numpy as np
import pytest
import torch

from oracle import gdn2_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,D,BT", [
    (torch.bfloat16, 64, 64), (torch.bfloat16, 64, 128), (torch.bfloat16, 128, 64),
    (torch.bfloat16, 128, 128), (torch.bfloat16, 256, 64), (torch.float32, 64, 64),
    (torch.float32, 128, 64), (torch.float32, 256, 64)])
@pytest.mark.parametrize("chunks,short", [(1, 0), (1, 63), (2, 5), (3, 0), (4, 17)])
@pytest.mark.parametrize("wide", [False, True])
def test_scan_edges(dtype, D, BT, chunks, short, wide):
    import gdn2_package as gp
    # 16-column slices fit 256 CUs up to 256 / (D / 16) units
    B, H = (1, 3) if not wide else (3, 256 // (D // 16) // 3 + 1)
    T = chunks * BT - short
    xs = O.make_inputs(B, T, H, D, seed=chunks * 100 + short + D)
    h0 = np.random.default_rng(7).standard_normal((B, H, D, D)).astype(np.float32) * 0.3 \
        if chunks % 2 else None
    dev = torch.device("cuda")
    xt = [torch.tensor(x, device=dev).to(dtype) for x in xs[:5]] + [torch.tensor(xs[5], device=dev)]
    ht = None if h0 is None else torch.tensor(h0, device=dev)
    out, hf = gp.gdn2_pallas_forward(*xt, D ** -0.5, ht, chunk_size=BT)
    host = [x.double().cpu().numpy() for x in xt]
    ro, rh = O.recurrent_fwd(*host, D ** -0.5, h0=h0)
    # the bounds of the other forward tests: bfloat16 operands 2e-2, float32 1e-4
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-4
    assert np.allclose(out.cpu().numpy(), ro, rtol=tol, atol=tol)
    assert np.allclose(hf.cpu().numpy(), rh, rtol=tol, atol=tol)
