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
