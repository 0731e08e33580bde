"""The fp32 VJP's direct products (few tokens) where their 32 x 32 tiles, K
chunks of 16 and adapter addressing can go wrong, and on both sides of the size
rule, against the float64 oracle."""
import numpy as np
import pytest

from oracle import moe_backward as MB

pytestmark = pytest.mark.gpu

# fp32 sums of at most 4000 terms in chains of up to 1000
TOL = 1e-5


@pytest.mark.parametrize("N,C,E,k,r", [(1, 64, 1, 1, 1), (2, 64, 2, 1, 3), (31, 64, 3, 2, 5), (33, 128, 5, 3, 7),
                                       (65, 192, 17, 2, 8), (70, 64, 64, 8, 32), (257, 256, 8, 2, 24),
                                       (1000, 768, 8, 2, 32), (1025, 64, 4, 4, 16), (4000, 64, 2, 1, 32),
                                       (2100, 768, 16, 2, 32), (2110, 768, 16, 4, 32)])
def test_backward_matches_oracle(device, N, C, E, k, r):
    import torch
    from rwkv_mlx_amd import _lib
    rng = np.random.default_rng(N + 7 * C + E + r)
    f = lambda *s, sc=1.0: (rng.standard_normal(s) * sc).astype(np.float32)
    x, dO, A, B, Wg = f(N, C), f(N, C), f(E, C, r, sc=C ** -0.5), f(E, r, C, sc=0.1), f(E, C, sc=C ** -0.5)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)
    desc = _lib.make_desc(1, N, C, 64, E, k, r, "f32")
    s = _lib.current_stream(device)
    nb = _lib.workspace_bytes(desc)
    ws = torch.empty(nb, dtype=torch.uint8, device=device)
    logits = torch.empty(N, E, device=device)
    inds = torch.empty(N, k, dtype=torch.int32, device=device)
    xd, wgd = up(x), up(Wg)
    _lib.call("rwkvmoe_router_topk", desc, _lib.make_tensors(x=xd, w_gate=wgd, logits=logits, inds=inds), ws, nb, s)
    bn = _lib.backward_workspace_bytes(desc)
    bws = torch.full((bn,), 0xFF, dtype=torch.uint8, device=device)  # NaN wherever nothing was written
    outs = {n: torch.full(sh, float("nan"), device=device) for n, sh in
            (("d_x", (N, C)), ("d_lora_A", (E, C, r)), ("d_lora_B", (E, r, C)), ("d_w_gate", (E, C)))}
    Ad, Bd, dOd, dl = up(A), up(B), up(dO), torch.tensor([0.3, -0.7], device=device)
    _lib.backward(desc, bws, bn, s, x=xd, w_gate=wgd, lora_A=Ad, lora_B=Bd, logits=logits, inds=inds, d_out=dOd,
                  d_losses=dl, **outs)
    torch.cuda.synchronize()
    ref = MB.moe_backward(x, Wg, A, B, k, "f32", dO, 0.3, -0.7)
    assert np.array_equal(inds.cpu().numpy(), ref["inds"])
    for name, key in (("d_x", "dx"), ("d_lora_A", "dA"), ("d_lora_B", "dB"), ("d_w_gate", "dWg")):
        got, want = outs[name].cpu().numpy(), ref[key].reshape(outs[name].shape)
        err = np.max(np.abs(got - want)) / np.max(np.abs(want))
        assert err <= TOL, f"{name}: {err:.2e}"
