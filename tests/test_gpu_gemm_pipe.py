"""The pipelined 16-bit products (key with relu², value) at the sizes where
their tiles, rings and tile choice can go wrong: one K slice per tile (fewer
than the ring holds) with many tiles per workgroup, ragged last rows, the
smallest widths, the K-extension with the residual, and row groups that are
empty, ragged or hold almost every token.  INSTANCES, ROW_GROUPS and K_GROUPS
reach every tile that the planner can choose, split and unsplit, in every form
(test_gemm_plan.py holds them to it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# out and h are rounded once (h twice: the product and its square), after an
# fp32 sum whose own error is far below that
UNIT = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}

SHAPES = [(65, 64, 64), (66, 128, 64), (129, 64, 192), (200, 2048, 1024), (200, 512, 8192), (257, 192, 384),
          (300, 320, 576), (1000, 64, 960), (2031, 1024, 3584), (4096, 768, 3072), (4100, 768, 256),
          (8192, 1024, 4096), (9001, 256, 512), (33000, 64, 128), (70000, 64, 64)]
# (N, C, F): the value product is N x C over K = F, the key product N x F over K = C
INSTANCES = [(4100, 2048, 64), (4100, 64, 2048), (3000, 3072, 256), (3000, 256, 3072), (513, 8192, 192),
             (513, 192, 8192), (1474, 3072, 256), (1474, 256, 3072), (700, 3072, 768), (700, 768, 3072),
             (513, 4096, 64), (513, 64, 4096), (9340, 896, 64), (65, 64, 2048), (65, 2048, 64), (131, 3072, 4096),
             (131, 4096, 3072), (65, 2048, 4096), (65, 4096, 2048), (200, 2048, 8192)]
# (N, C, F, E, k, one popular expert)
ROW_GROUPS = [(3, 64, 64, 2, 1, False), (130, 128, 192, 64, 1, False), (600, 64, 320, 8, 2, True),
              (3000, 256, 512, 16, 2, True), (20000, 64, 64, 4, 1, True), (2500, 768, 768, 5, 3, False),
              (3, 320, 64, 1, 1, False), (17, 64, 512, 64, 2, False), (17, 1024, 64, 32, 1, False),
              (4000, 64, 512, 8, 4, False), (1000, 2048, 128, 4, 4, False), (10000, 128, 192, 64, 4, False),
              (10000, 192, 128, 64, 4, False), (300, 192, 3072, 4, 4, False), (300, 3072, 192, 4, 4, False),
              (1000, 192, 576, 64, 4, False), (1000, 576, 192, 64, 4, False), (130, 768, 3072, 8, 4, False),
              (130, 3072, 768, 8, 4, False), (4000, 64, 768, 8, 4, False), (10000, 64, 576, 8, 2, False),
              (4000, 768, 64, 8, 4, False), (10000, 576, 64, 8, 2, False)]
# (N, C, F, E, k): the weight gradients, F x C and C x F for each expert
K_GROUPS = [(3, 64, 64, 1, 1), (3, 64, 64, 4, 1), (3, 64, 512, 64, 1), (3, 384, 768, 32, 1), (3, 576, 192, 64, 1),
            (3, 768, 3072, 2, 1), (600, 192, 576, 32, 4), (1500, 768, 384, 8, 4), (2048, 1024, 4096, 8, 2)]


@pytest.mark.parametrize("N,C,F", SHAPES + INSTANCES)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_key_and_value_products(device, dtype, N, C, F):
    import torch
    from rwkv_mlx_amd import _lib
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device=device).manual_seed(N + C + F)
    rand = lambda *s, sc=1.0: (torch.randn(*s, generator=g, device=device) * sc).to(dt)
    x, xk = rand(1, N, C), torch.zeros(C, device=device, dtype=dt)  # x_k = 0: no token shift
    wk, wv = rand(F, C, sc=C ** -0.5), rand(C, F, sc=F ** -0.5)
    desc = _lib.make_desc(1, N, C, F, 1, 1, 1, dtype)
    nb = _lib.workspace_bytes(desc)
    ws = torch.full((nb,), 0xFF, dtype=torch.uint8, device=device)
    h = torch.full((N + 1, F), float("nan"), dtype=dt, device=device)  # (the last row: past the end)
    out = torch.full((N + 1, C), float("nan"), dtype=dt, device=device)
    s = _lib.current_stream(device)
    _lib.call("rwkvmoe_cmix_key", desc, _lib.make_tensors(x=x, x_k=xk, w_key=wk, hidden=h), ws, nb, s)
    _lib.call("rwkvmoe_cmix_value", desc, _lib.make_tensors(hidden=h, w_value=wv, base_out=out), ws, nb, s)
    torch.cuda.synchronize()
    ref_h = torch.relu(x[0].double() @ wk.double().T) ** 2
    ref_o = h[:N].double() @ wv.double().T
    for got, ref, units in ((h, ref_h, 3), (out, ref_o, 1)):
        assert torch.isnan(got[N]).all(), "a row past the end was written"
        err = (got[:N].double() - ref).abs().max().item() / ref.abs().max().item()
        assert err <= units * UNIT[dtype], err


@pytest.mark.parametrize("N,C,F,E,k,r", [(100, 64, 64, 4, 2, 8), (700, 192, 320, 32, 4, 16), (2031, 1024, 1792, 8, 2, 32),
                                         (5000, 128, 256, 16, 2, 8), (300, 2048, 1024, 16, 2, 32)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_layer_with_adapter_columns_and_residual(device, dtype, N, C, F, E, k, r):
    """The whole FUSED layer (adapter columns, K-extension, residual) against
    float64 with the dtype's rounding of each stage bounded."""
    import torch
    from rwkv_mlx_amd.moe import build_layer
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    torch.manual_seed(N + E)
    m = build_layer(C, F, E, k, r).to(device=device, dtype=dt).requires_grad_(False)
    m.base.x_k.uniform_(0, 1)
    m.lora_A.normal_(0, C ** -0.5)
    m.lora_B.normal_(0, 0.3)
    x = torch.randn(1, N, C, device=device).to(dt)
    res = torch.randn(1, N, C, device=device).to(dt)
    ex = {}
    with torch.no_grad():
        out = m(x, residual=res, extras=ex)[0]
        out2 = m(x, residual=res)[0]
    assert torch.equal(out, out2)
    xd = x.double()
    sh = torch.cat([torch.zeros_like(xd[:, :1]), xd[:, :-1]], 1)
    base = torch.relu((xd + (sh - xd) * m.base.x_k.double()) @ m.base.key.weight.double().T) ** 2 \
        @ m.base.value.weight.double().T
    w = torch.zeros(N, E, dtype=torch.float64, device=device).scatter(1, ex["inds"].long(), ex["gates"].double())
    delta = sum(w[:, e:e + 1] * (xd[0] @ m.lora_A[e].double() @ m.lora_B[e].double()) for e in range(E))
    ref = res.double() + base + delta
    err = (out.double() - ref).norm().item() / ref.norm().item()
    # the mix, h, U, the output and the residual sum each round to dtype
    assert err <= 5 * UNIT[dtype], err


@pytest.mark.parametrize("N,C,F,E,k", [(3584, 768, 256, 16, 2), (3585, 768, 256, 16, 2), (4096, 768, 384, 16, 1),
                                       (4097, 768, 256, 16, 2), (2048, 1536, 256, 16, 4), (2049, 1536, 192, 16, 2)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_sparse_combine_at_one_tile_a_cu(device, dtype, N, C, F, E, k):
    """The SPARSE layer on both sides of the range in which the combine runs in
    the value product's epilogue (231 to 256 tiles of 128x96, F % 128 == 0), token
    by token against float64."""
    import torch
    from rwkv_mlx_amd.moe import build_layer
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    torch.manual_seed(N + F)
    m = build_layer(C, F, E, k, 16).to(device=device, dtype=dt).requires_grad_(False)
    m.base.x_k.uniform_(0, 1)
    m.lora_A.normal_(0, C ** -0.5)
    m.lora_B.normal_(0, 0.3)
    x = torch.randn(1, N, C, device=device).to(dt)
    res = torch.randn(1, N, C, device=device).to(dt)
    ex = {}
    with torch.no_grad():
        out = m(x, residual=res, mode="sparse", extras=ex)[0]
    xd = x[0].double()
    sh = torch.cat([torch.zeros_like(xd[:1]), xd[:-1]])
    ref = res[0].double() + torch.relu((xd + (sh - xd) * m.base.x_k.double().reshape(-1)) @ m.base.key.weight.double().T) \
        ** 2 @ m.base.value.weight.double().T
    w = torch.zeros(N, E, dtype=torch.float64, device=device).scatter(1, ex["inds"].long(), ex["gates"].double())
    for e in range(E):
        ref += w[:, e:e + 1] * (xd @ m.lora_A[e].double() @ m.lora_B[e].double())
    err = ((out[0].double() - ref).norm(dim=1) / ref.norm(dim=1)).max().item()
    # the mix, h, the adapter rows, the base, their sum and the residual's each round to dtype
    assert err <= 6 * UNIT[dtype], err


@pytest.mark.parametrize("N,C,F,E,k,hot", ROW_GROUPS)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_row_groups(device, dtype, N, C, F, E, k, hot):
    """MoE_CMix's grouped products: groups that are empty, ragged, or hold
    nearly every token, against the routed rows in float64."""
    import torch
    from rwkv_mlx_amd import MoE_CMix, RWKVConfig
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    torch.manual_seed(N + E)
    m = MoE_CMix(RWKVConfig(n_embd=C, dim_ffn=F), 0, E, k).to(device=device, dtype=dt).requires_grad_(False)
    m.x_k.uniform_(0, 1)
    m.expert_key.normal_(0, C ** -0.5)
    m.expert_val.normal_(0, F ** -0.5)
    if hot:
        m.router.logit_bias = torch.tensor([20.0] + [0.0] * (E - 1), device=device)
    x = torch.randn(1, N, C, device=device).to(dt)
    ex = {}
    with torch.no_grad():
        out = m(x, extras=ex)[0][0].double()
    xd = x[0].double()
    mix = torch.cat([torch.zeros_like(xd[:1]), xd[:-1]]) - xd
    ref = torch.zeros_like(xd)
    w = torch.zeros(N, E, dtype=torch.float64, device=device).scatter(1, ex["inds"].long(), ex["gates"].double())
    for e in range(E):
        at = (ex["inds"] == e).any(1).nonzero()[:, 0]
        y = torch.relu((xd[at] + mix[at] * m.x_k[e, 0, 0].double()) @ m.expert_key[e].double().T) ** 2 \
            @ m.expert_val[e].double().T
        ref = ref.index_add(0, at, w[at, e:e + 1] * y)
    err = (out - ref).norm().item() / ref.norm().item()
    assert np.isfinite(err) and err <= 5 * UNIT[dtype], err


@pytest.mark.parametrize("N,C,F,E,k", [(1, 64, 64, 2, 1), (1, 512, 2048, 4, 1), (9, 64, 64, 64, 8), (64, 512, 2048, 4, 1),
                                       (200, 768, 3072, 8, 2), (513, 64, 320, 5, 3), (3000, 256, 512, 16, 2),
                                       (20000, 64, 64, 4, 1)])
def test_row_groups_reduce_the_losses(device, N, C, F, E, k):
    """The aux and z losses that the grouped key product reduces, in a workgroup
    without a tile or in the first to end, against float64 of the same logits;
    the same bits in every pass."""
    import torch
    from rwkv_mlx_amd import MoE_CMix, RWKVConfig
    torch.manual_seed(N + F)
    m = MoE_CMix(RWKVConfig(n_embd=C, dim_ffn=F), 0, E, k).to(device=device, dtype=torch.float16).requires_grad_(False)
    m.expert_key.normal_(0, C ** -0.5)
    m.expert_val.normal_(0, F ** -0.5)
    x = torch.randn(1, N, C, device=device).half()
    ex = {}
    with torch.no_grad():
        _, aux, z = m(x, extras=ex)
        for _ in range(3):
            _, aux2, z2 = m(x)
            assert torch.equal(aux, aux2) and torch.equal(z, z2)
    lg = ex["logits"].double().reshape(N, E)
    share = torch.zeros(N, E, dtype=torch.float64, device=device).scatter(1, ex["inds"].reshape(N, k).long(), 1.0)
    ref_aux = E * (share.mean(0) / k * lg.softmax(-1).mean(0)).sum()
    ref_z = torch.logsumexp(lg, -1).square().mean()
    assert abs(aux.item() - ref_aux.item()) <= 1e-6 * ref_aux.item()
    assert abs(z.item() - ref_z.item()) <= 1e-6 * ref_z.item()


@pytest.mark.parametrize("N,C,F,E,k", K_GROUPS)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_k_groups(device, dtype, N, C, F, E, k):
    """The weight gradients of the full-expert layer, each expert's over its own
    routed rows, against float64; an expert without rows gets zeros."""
    import torch
    from rwkv_mlx_amd import _lib
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device=device).manual_seed(N + C + F + E)
    rand = lambda *s, sc=1.0: (torch.randn(*s, generator=g, device=device) * sc).to(dt)
    x, dO, xk = rand(1, N, C), rand(1, N, C), torch.rand(E, C, generator=g, device=device).to(dt)
    wk, wv, wg = rand(E, F, C, sc=C ** -0.5), rand(E, C, F, sc=F ** -0.5), rand(E, C)
    logits = torch.randn(N, E, generator=g, device=device)
    sel, inds = logits.topk(k, -1)
    inds = inds.int()
    desc = _lib.make_desc(1, N, C, F, E, k, 1, dtype)
    nb = _lib.experts_backward_workspace_bytes(desc)
    ws = torch.full((nb,), 0xFF, dtype=torch.uint8, device=device)
    dwk, dwv = torch.full_like(wk, float("nan")), torch.full_like(wv, float("nan"))
    _lib.experts_backward(desc, ws, nb, _lib.current_stream(device), x=x, x_k=xk, w_key=wk, w_value=wv, w_gate=wg,
                          logits=logits, inds=inds, d_out=dO, d_w_key=dwk, d_w_value=dwv)
    torch.cuda.synchronize()
    gates = sel.double().softmax(-1)
    xd, dOd = x[0].double(), dO[0].double()
    mix = torch.cat([torch.zeros_like(xd[:1]), xd[:-1]]) - xd
    for e in range(E):
        at, slot = (inds == e).nonzero(as_tuple=True)
        rows = xd[at] + mix[at] * xk[e].double()
        p = torch.relu(rows @ wk[e].double().T)
        gdo = gates[at, slot][:, None] * dOd[at]
        for got, ref in ((dwk[e], (2 * p * (gdo @ wv[e].double())).T @ rows), (dwv[e], gdo.T @ (p * p))):
            # the mixed rows, p, h, u, dp, g dO and the gradient each round to dtype
            err = (got.double() - ref).norm().item()
            assert err <= 7 * UNIT[dtype] * ref.norm().item(), (e, err)
