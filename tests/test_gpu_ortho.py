"""The orthogonality loss (rwkvmoe_ortho_loss) against the oracle where its
16 x 16 tiles of the adapters' Gram matrix can go wrong: one expert, ranks
that put several experts or a part of one into a tile, a ragged last tile, the
smallest and largest layers."""
import math

import numpy as np
import pytest

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu

# The sums over C run in fp32 in another order than the oracle's.  fp32: 64
# terms a chain, error below 64 · 2^-24.  16-bit: a cross product may round to
# the neighbouring value (one unit), its square then moves by two and one more.
TOL = {"f32": 1e-5, "f16": 3 * 2.0 ** -11, "bf16": 3 * 2.0 ** -8}


@pytest.mark.parametrize("E,C,r", [(1, 64, 32), (2, 64, 1), (3, 64, 5), (5, 192, 3), (2, 128, 16), (4, 512, 8),
                                   (3, 128, 24), (8, 768, 32), (17, 64, 7), (64, 256, 32), (4, 8192, 32)])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
def test_ortho_loss_matches_oracle(device, dtype, E, C, r):
    import torch
    from helpers import to_dev
    from rwkv_mlx_amd import _lib
    rng = np.random.default_rng(E * 10000 + C + r)
    A = O.round_to(rng.standard_normal((E, C, r)) / np.sqrt(C), dtype)
    ref = O.ortho_loss(A, dtype)
    desc = _lib.make_desc(1, 1, C, 64, E, 1, r, dtype)
    nbytes = _lib.workspace_bytes(desc)
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=device)
    got = []
    for _ in range(2):
        out = torch.full((1,), math.nan, dtype=torch.float32, device=device)
        t = _lib.make_tensors(lora_A=to_dev(A, dtype, device), ortho_loss=out)
        _lib.call("rwkvmoe_ortho_loss", desc, t, ws, nbytes, _lib.current_stream(device))
        got.append(float(out.item()))
    assert got[0] == got[1]
    assert abs(got[0] - ref) <= TOL[dtype] * ref, f"{got[0]} vs {ref}"


@pytest.mark.parametrize("E,C,r", [(1, 64, 32), (2, 64, 1), (3, 64, 5), (5, 192, 3), (2, 128, 16), (3, 128, 24),
                                   (8, 768, 32), (17, 64, 7), (64, 64, 32), (4, 8192, 8)])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
def test_ortho_gradient_matches_oracle(device, dtype, E, C, r):
    """Its gradient, on both sides of the size rule (E=64, r=32 in 16 bits is
    past it).  fp32 sums of at most 8192 terms; 16-bit results round once, or
    on the GEMM tiles with the Gram matrix rounded too."""
    import torch
    from helpers import to_dev, to_np
    from oracle import moe_backward as MB
    from rwkv_mlx_amd import _lib
    rng = np.random.default_rng(E * 10000 + C + r + 1)
    A = O.round_to(rng.standard_normal((E, C, r)) / np.sqrt(C), dtype)
    ref = 0.25 * MB.ortho_grad(A)
    desc = _lib.make_desc(1, 1, C, 64, E, 1, r, dtype)
    nbytes = _lib.backward_workspace_bytes(desc)
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=device)
    Ad = to_dev(A, dtype, device)
    dA = torch.full_like(Ad, math.nan)
    _lib.backward(desc, ws, nbytes, _lib.current_stream(device), entry="rwkvmoe_ortho_backward", lora_A=Ad,
                  d_lora_A=dA, d_ortho=torch.tensor([0.25], device=device))
    torch.cuda.synchronize()
    scale = max(np.max(np.abs(ref)), 1e-30)
    err = np.max(np.abs(to_np(dA).reshape(ref.shape) - ref)) / scale
    assert err <= {"f32": 1e-5, "f16": 4 * 2.0 ** -11, "bf16": 4 * 2.0 ** -8}[dtype], err
