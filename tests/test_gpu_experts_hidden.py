"""The full-expert backward where its 64x64 tiles and packed token ranges end:
one and several tiles of hidden columns, experts with no row, with one, and with
counts just around 64 and 128, each weight gradient alone, and more experts than
the routing kernel's group has lanes."""
import numpy as np
import pytest

import test_gpu_experts_backward as B

pytestmark = pytest.mark.gpu

# name: (dtype, B, T, C, F, E, k, x_prev, bias); the zipf bias leaves experts empty
EDGES = {
    "hid-f64-e1-n63-bf16": ("bf16", 1, 63, 64, 64, 1, 1, False, False),
    "hid-f64-e1-n129-f32": ("f32", 1, 129, 64, 64, 1, 1, False, False),
    "hid-e2-k2-n64-f16": ("f16", 1, 64, 64, 192, 2, 2, False, False),
    "hid-e2-k2-n65-bf16": ("bf16", 1, 65, 128, 64, 2, 2, False, False),
    "hid-e17-k1-n9-f32-bias": ("f32", 1, 9, 64, 128, 17, 1, False, True),
    "hid-e33-k8-n40-f16": ("f16", 2, 20, 64, 320, 33, 8, True, False),
    "hid-f1088-e16-k2-f32-bias": ("f32", 2, 70, 64, 1088, 16, 2, False, True),
}


@pytest.fixture(params=list(EDGES))
def layer(request, device):
    B.CASES.update(EDGES)
    try:
        L = B.ExpertsLayer(request.param, device)
    finally:
        for n in EDGES:
            del B.CASES[n]
    L.forward()
    return L


def test_gradients_and_each_weight_alone(layer):
    ref = layer.oracle()
    got = layer.backward()
    for name, t in got.items():
        mx, nrm = B._errs(t.float().cpu().numpy(), ref[B.ORACLE_NAME[name]].reshape(t.shape))
        assert max(mx, nrm) <= B.BWD_TOL[layer.dtype], (name, mx, nrm)
    for name in ("d_w_key", "d_w_value", "d_w_gate"):
        alone = layer.backward((name,))[name]
        assert np.array_equal(B._bits(alone), B._bits(got[name])), name


def test_more_token_tiles_than_a_second_grid_dimension(device):
    """Frozen expert weights and more than 65535 tiles of 64 routed rows: dx of
    the last sequences is that of these sequences alone."""
    import torch
    from rwkv_mlx_amd import _lib
    Bn, T, C, F, E, k = 65600, 32, 64, 64, 2, 2
    g = torch.Generator(device=device).manual_seed(7)
    rand = lambda *s, sc=1.0: (torch.randn(*s, generator=g, device=device) * sc).half()
    x, dO, xk = rand(Bn, T, C), rand(Bn, T, C), torch.rand(E, C, generator=g, device=device).half()
    wk, wv, wg = rand(E, F, C, sc=C ** -0.5), rand(E, C, F, sc=F ** -0.5), rand(E, C)
    logits = torch.randn(Bn * T, E, generator=g, device=device)
    inds = logits.topk(k, -1)[1].int()

    def dx(at):
        n = Bn - at
        desc = _lib.make_desc(n, T, C, F, E, k, 1, "f16")
        nb = _lib.experts_backward_workspace_bytes(desc)
        ws = torch.full((nb,), 0xFF, dtype=torch.uint8, device=device)
        out = torch.full((n, T, C), float("nan"), dtype=torch.float16, device=device)
        _lib.experts_backward(desc, ws, nb, _lib.current_stream(device), x=x[at:], x_k=xk, w_key=wk, w_value=wv,
                              w_gate=wg, logits=logits[at * T:], inds=inds[at * T:], d_out=dO[at:], d_x=out)
        torch.cuda.synchronize()
        return out
    whole, last = dx(0), dx(Bn - 40)
    assert torch.isfinite(whole).all()
    assert (whole[-40:].double() - last.double()).norm() <= 4 * 2.0 ** -11 * last.double().norm()
