"""The bf16 router with its chunk products on MFMA blocks beside the shift mix
(and ln2): the chunk sums lie over the two LDS rows that only the mix reads, the
row before the tile and x_k.  Sequences that start inside a tile, a carried
x_prev, ragged last tiles, W_gate in LDS and in registers, one and two rows of
blocks: logits bit for bit, and every token's output by itself (a row mixed
from overwritten LDS is off by its own size)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

UNIT = 2.0 ** -8
# (B, T, C, F, E, r): more than 256 tiles of 16 (8 where E·C >= 32768) tokens,
# E·r > 128 or such a tile of 8: the adapter columns are the key product's
SHAPES = [(5, 901, 256, 256, 8, 32), (3, 1377, 768, 768, 8, 32), (9, 239, 2048, 512, 16, 32), (66, 63, 64, 256, 5, 32),
          (4, 1031, 1024, 512, 13, 16), (5, 601, 512, 256, 64, 8)]


@pytest.mark.parametrize("B,T,C,F,E,r", SHAPES)
@pytest.mark.parametrize("prev,ln", [(False, False), (True, False), (True, True)])
def test_mixed_rows(device, B, T, C, F, E, r, prev, ln):
    import torch
    from oracle import moe_oracle as O
    from rwkv_mlx_amd import LoRAMoE_CMix, RWKV_CMix_x070, RWKVConfig
    g = torch.Generator(device=device).manual_seed(B * T + C)
    rand = lambda *s, sc=1.0: (torch.randn(*s, generator=g, device=device) * sc).bfloat16()
    m = LoRAMoE_CMix(RWKV_CMix_x070(RWKVConfig(n_embd=C, dim_ffn=F), 0), E, r, 2).to(device, torch.bfloat16)
    m.requires_grad_(False)
    m.base.x_k.copy_(torch.rand(m.base.x_k.shape, generator=g, device=device))
    for p, fan in ((m.base.key.weight, C), (m.base.value.weight, F), (m.router.gate.weight, C), (m.lora_A, C)):
        p.copy_(rand(*p.shape, sc=fan ** -0.5))
    m.lora_B.copy_(rand(*m.lora_B.shape, sc=0.02))
    x, xp = rand(B, T, C), rand(B, C) if prev else None
    lnp = ((1 + 0.1 * rand(C).float()).bfloat16(), rand(C, sc=0.1)) if ln else None
    ex = {}
    with torch.no_grad():
        out, _, _ = m(x, x_prev=xp, extras=ex, ln=lnp)
    xl = ex["x_ln"] if ln else x
    logits = O.router_logits(xl.float().cpu().numpy().reshape(B * T, C), m.router.gate.weight.float().cpu().numpy(),
                             acc="f32")
    assert np.array_equal(ex["logits"].cpu().numpy(), logits)

    d = lambda t: t.double()
    first = (d(xp) if prev else torch.zeros(B, C, dtype=torch.float64, device=device))[:, None]
    xd = d(xl).reshape(B, T, C)
    xk = xd + (torch.cat([first, xd[:, :-1]], 1) - xd) * d(m.base.x_k).reshape(C)
    ref = (torch.relu(xk @ d(m.base.key.weight).T) ** 2 @ d(m.base.value.weight).T).reshape(-1, C)
    flat = xd.reshape(-1, C)
    top, inds = torch.from_numpy(logits).to(device).double().topk(2, -1)
    w = torch.zeros(B * T, E, dtype=torch.float64, device=device).scatter(1, inds, top.softmax(-1))
    for e in range(E):
        ref += w[:, e:e + 1] * (flat @ d(m.lora_A[e]) @ d(m.lora_B[e]))
    got = d(out).reshape(-1, C)
    # shift, product and sum of the mix, p, h (twice p's share), u and the output each round to bf16
    err = ((got - ref).norm(dim=1) / ref.norm(dim=1)).max().item()
    assert np.isfinite(err) and err <= 8 * UNIT, err
