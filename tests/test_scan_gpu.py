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


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("chunks,short", [(1, 0), (2, 9), (3, 0), (4, 0)])
@pytest.mark.parametrize("full", [False, True])
def test_training_scan_edges(D, chunks, short, full):
    """Forward and reverse scan of the training path on both sides of the rule that
    lays its float32 tiles out (more units than one 16-column slice per CU holds:
    rows, else fragments): all gradients, dh0 and a cotangent on h_final included,
    against the float64 recurrence's."""
    import gdn2_package as gp
    B, H = 1, 256 // (D // 16) + 1 if full else 3
    T = chunks * 64 - short
    xs = O.make_inputs(B, T, H, D, seed=chunks * 10 + D)
    rng = np.random.default_rng(5)
    h0 = (0.3 * rng.standard_normal((B, H, D, D))).astype(np.float32)
    do = rng.standard_normal((B, T, H, D)).astype(np.float32)
    dhf = (0.1 * rng.standard_normal((B, H, D, D))).astype(np.float32)
    dev = torch.device("cuda")
    xt = [torch.tensor(x, device=dev, requires_grad=True) for x in (*xs, h0)]
    out, hf = gp.gdn2_pallas_forward_trainable(*xt[:6], D ** -0.5, xt[6])
    got = torch.autograd.grad([out, hf], xt, [torch.tensor(do, device=dev),
                                              torch.tensor(dhf, device=dev)])
    # the same in float64 by autograd of the token recurrence
    x64 = [x.detach().double().requires_grad_(True) for x in xt]
    q, k, v, w, b, g, s = x64
    o = []
    for t in range(T):
        s = torch.exp(g[:, t]).unsqueeze(-1) * s
        d = w[:, t] * v[:, t] - ((b[:, t] * k[:, t]).unsqueeze(-1) * s).sum(-2)
        s = s + k[:, t].unsqueeze(-1) * d.unsqueeze(-2)
        o.append(D ** -0.5 * (q[:, t].unsqueeze(-1) * s).sum(-2))
    ref = torch.autograd.grad([torch.stack(o, 1), s], x64, [torch.tensor(do, device=dev).double(),
                                                           torch.tensor(dhf, device=dev).double()])
    for name, a, r in zip("q k v w b g h0".split(), got, ref):
        # 1e-4 as the other float32 gradient tests
        assert torch.all((a.double() - r).abs() <= 1e-4 + 1e-4 * r.abs()), name


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("chunks,H", [(2, 3), (3, 3), (3, None)])
def test_kept_tiles_of_both_layouts(D, chunks, H):
    """The float32 tiles that a residual-keeping forward leaves, on both sides of each
    line of the layout rule (rows for up to two chunks and for a full device, else
    fragments), against the oracle's restatement of the reference's kernels."""
    import gdn2_package as gp
    H = H or 256 // (D // 16) + 1
    xs = O.make_inputs(1, chunks * 64, H, D, seed=chunks + D)
    h0 = (0.1 * np.random.default_rng(2).standard_normal((1, H, D, D))).astype(np.float32)
    dev = torch.device("cuda")
    _, _, res = gp.gdn2_pallas_forward_with_residuals(
        *[torch.tensor(x, device=dev) for x in xs], D ** -0.5, h0=torch.tensor(h0, device=dev),
        chunk_size=64)
    _, _, ref = O.chunked_fwd(*xs, D ** -0.5, h0=h0, BT=64, clip=False, return_residuals=True)
    for key in ["w_pseudo", "u", "kg", "qg", "gc_last", "h_pre_all", "v_new_all"]:
        # 1e-4 as test_fwd_gpu.py's intermediates
        assert np.allclose(res[key].cpu().numpy(), ref[key], rtol=1e-4, atol=1e-4), key


@pytest.mark.parametrize("dtype,D,BT,H,S,save", [
    # more than 256 16-column slices in the final pass, with and without kept residuals
    (torch.float32, 64, 64, 9, 8, False), (torch.float32, 64, 64, 9, 8, True),
    (torch.float32, 128, 64, 5, 7, False), (torch.float32, 256, 64, 2, 9, False),
    (torch.float32, 256, 64, 2, 9, True),
    (torch.bfloat16, 64, 64, 9, 8, False), (torch.bfloat16, 64, 128, 9, 8, True),
    (torch.bfloat16, 128, 64, 5, 7, True), (torch.bfloat16, 128, 128, 5, 7, False),
    (torch.bfloat16, 256, 64, 2, 9, False), (torch.bfloat16, 256, 64, 2, 9, True),
    # in the summary pass only (twice the slices)
    (torch.float32, 128, 64, 3, 7, False), (torch.bfloat16, 256, 64, 1, 9, False),
    (torch.bfloat16, 128, 128, 3, 7, False),
    # forced segments where the (b,h) pairs alone fill the device (float32: rows)
    (torch.float32, 64, 64, 65, 2, True), (torch.float32, 128, 64, 33, 2, False),
    (torch.float32, 256, 64, 17, 2, False), (torch.bfloat16, 128, 64, 33, 2, False)])
def test_segments_of_a_full_device(dtype, D, BT, H, S, save):
    """The segmented scan's three passes in the forms that a full device takes, from a
    state and with a short last chunk, against the serial scan and the recurrence."""
    from gdn2_package import _lib
    from gdn2_package.gdn2_fwd import _Prepared, _run_forward
    T = (2 * S - 1) * BT - 9          # segments of two chunks, the last of one
    xs = O.make_inputs(1, T, H, D, seed=D + H)
    h0 = (0.3 * np.random.default_rng(8).standard_normal((1, H, D, D))).astype(np.float32)
    dev = torch.device("cuda")
    xt = [torch.tensor(x, device=dev).to(dtype) for x in xs[:5]] + [torch.tensor(xs[5], device=dev)]
    p = _Prepared(*xt, D ** -0.5, torch.tensor(h0, device=dev), BT)
    keep = _lib.FWD_SAVE_A if save else 0
    out, hf, _, _ = _run_forward(p, flags=_lib.FWD_SEGMENTS(S) | keep)
    out_1, hf_1, _, _ = _run_forward(p, flags=_lib.FWD_SEGMENTS(1) | keep)
    # as test_fwd_gpu.py's segments: the order of the boundary-state products
    near = 1e-5 if dtype == torch.float32 else 2e-3
    assert torch.allclose(out, out_1, rtol=near, atol=near)
    assert torch.allclose(hf, hf_1, rtol=near, atol=near)
    ro, rh = O.recurrent_fwd(*[x.double().cpu().numpy() for x in xt], D ** -0.5, h0=h0)
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-4
    assert np.allclose(out.cpu().numpy(), ro, rtol=tol, atol=tol)
    assert np.allclose(hf.cpu().numpy(), rh, rtol=tol, atol=tol)


@pytest.mark.parametrize("D,H,seqs", [(64, 5, 12), (64, 5, 13), (128, 3, 10), (128, 3, 11),
                                      (256, 1, 16), (256, 1, 17),
                                      # one, two and four chunks in all
                                      (128, 3, 2), (64, 5, 3), (128, 3, 3), (256, 1, 3),
                                      (128, 3, 4)])
def test_packed_training_layouts(D, H, seqs):
    """Packed training with (head, sequence) counts on both sides of the rule that lays
    the float32 tiles out, which the forward and the backward apply separately: every
    gradient, dh0 included, against the float64 recurrence's; empty, short and exact
    sequences among them."""
    import gdn2_package as gp
    lens = [(0, 17, 64, 65, 1, 100, 33)[i % 7] for i in range(seqs)]
    T, cu = sum(lens), np.concatenate([[0], np.cumsum(lens)]).tolist()
    xs = O.make_inputs(1, T, H, D, seed=D + seqs)
    rng = np.random.default_rng(4)
    h0 = (0.3 * rng.standard_normal((seqs, H, D, D))).astype(np.float32)
    do = rng.standard_normal((1, T, H, D)).astype(np.float32)
    dhf = (0.1 * rng.standard_normal((seqs, H, D, D))).astype(np.float32)
    dev = torch.device("cuda")
    xt = [torch.tensor(x, device=dev, requires_grad=True) for x in (*xs, h0)]
    dt, dht = torch.tensor(do, device=dev), torch.tensor(dhf, device=dev)
    out, hf = gp.gdn2_pallas_forward_varlen_trainable(*xt[:6], D ** -0.5, cu, xt[6])
    got = torch.autograd.grad([out, hf], xt, [dt, dht])
    x64 = [x.detach().double().requires_grad_(True) for x in xt]
    q, k, v, w, b, g, s0 = x64
    o, ends = [], []
    for i, (a, e) in enumerate(zip(cu, cu[1:])):
        s = s0[i]
        for t in range(a, e):
            s = torch.exp(g[0, t]).unsqueeze(-1) * s
            d = w[0, t] * v[0, t] - ((b[0, t] * k[0, t]).unsqueeze(-1) * s).sum(-2)
            s = s + k[0, t].unsqueeze(-1) * d.unsqueeze(-2)
            o.append(D ** -0.5 * (q[0, t].unsqueeze(-1) * s).sum(-2))
        ends.append(s)
    ref = torch.autograd.grad([torch.stack(o)[None], torch.stack(ends)], x64,
                              [dt.double(), dht.double()])
    for name, x, r in zip("q k v w b g h0".split(), got, ref):
        # 1e-4 as the other float32 gradient tests
        assert torch.all((x.double() - r).abs() <= 1e-4 + 1e-4 * r.abs()), name


@pytest.mark.parametrize("D,H,T,S", [(128, 8, 16384, 8), (256, 12, 4096, 1)])
def test_segments_of_a_residual_keeping_call(D, H, T, S):
    """A bfloat16 forward that keeps its residuals runs the segments that its 32-column
    passes ask for, whatever its workspace is sized for: bit for bit the forced count."""
    from gdn2_package import _lib
    from gdn2_package.gdn2_fwd import _Prepared, _run_forward
    gen = torch.Generator(device="cuda").manual_seed(D)
    q, k, v, w, b, g = (torch.randn((1, T, H, D), generator=gen, device="cuda") for _ in range(6))
    f = torch.nn.functional
    xs = [x.bfloat16() for x in (f.normalize(q, dim=-1), f.normalize(k, dim=-1), v,
                                 torch.sigmoid(w), torch.sigmoid(b))] + [-f.softplus(g)]
    p = _Prepared(*xs, D ** -0.5, None, 64)
    out, hf, _, _ = _run_forward(p, flags=_lib.FWD_SAVE_A)
    out_s, hf_s, _, _ = _run_forward(p, flags=_lib.FWD_SAVE_A | _lib.FWD_SEGMENTS(S))
    assert torch.equal(out, out_s) and torch.equal(hf, hf_s)
