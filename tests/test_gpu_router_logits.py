"""Router logits bit for bit where the chunk products' blocks (4 tokens x 4
experts x 16 chunks) end: ragged tokens, experts that are no multiple of 4, one
chunk, W_gate in LDS and in registers, one and two rows of blocks, few and many
tiles, and terms that underflow to subnormal fp32 or overflow it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (tokens, C, E): more than 256 tiles of 16 (8 where E·C >= 32768) tokens run the blocks
SHAPES = [(7, 64, 3), (1030, 768, 8), (300, 2048, 16), (20001, 64, 1), (5003, 128, 5), (4500, 192, 6), (4110, 768, 8),
          (4201, 1024, 13), (2050, 2048, 16), (2063, 2048, 8), (4099, 1024, 32), (3001, 704, 33), (3000, 512, 64)]


def _run(device, dtype, x, wg, k):
    import torch
    from rwkv_mlx_amd import _lib
    N, C = x.shape
    E = wg.shape[0]
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    X, W = (torch.from_numpy(a).to(device=device, dtype=dt) for a in (x, wg))
    desc = _lib.make_desc(1, N, C, 64, E, k, 1, dtype)
    nb = _lib.workspace_bytes(desc)
    ws = torch.full((nb,), 0xFF, dtype=torch.uint8, device=device)
    inds = torch.full((N, k), -1, dtype=torch.int32, device=device)
    gates = torch.empty(N, k, dtype=dt, device=device)
    losses = torch.empty(2, dtype=torch.float32, device=device)
    logits = torch.full((N + 1, E), -7.0, dtype=torch.float32, device=device)  # (the last row: past the end)
    _lib.call("rwkvmoe_router_topk", desc, _lib.make_tensors(x=X, w_gate=W, inds=inds, gates=gates, losses=losses,
                                                             logits=logits), ws, nb, _lib.current_stream(device))
    torch.cuda.synchronize()
    assert (logits[N] == -7.0).all()
    return X.float().cpu().numpy(), W.float().cpu().numpy(), logits[:N].cpu().numpy(), inds.cpu().numpy()


@pytest.mark.parametrize("N,C,E", SHAPES)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_logits_bit_exact(device, dtype, N, C, E):
    from oracle import moe_oracle as O
    rng = np.random.default_rng(N + C + E)
    k = min(2, E)
    x = O.round_to(rng.standard_normal((N, C)).astype(np.float32), dtype)
    w = O.round_to((rng.standard_normal((E, C)) / np.sqrt(C)).astype(np.float32), dtype)
    xg, wg, logits, inds = _run(device, dtype, x, w, k)
    assert np.array_equal(xg, x) and np.array_equal(wg, w)
    ref = O.router(x, w, k, dtype)
    assert np.array_equal(logits, ref["logits"])
    assert np.array_equal(inds, ref["inds"])


@pytest.mark.parametrize("sx,sw", [(2.0 ** -70, 2.0 ** -68), (2.0 ** -100, 2.0 ** -40), (2.0 ** 63, 2.0 ** 64)])
def test_subnormal_and_overflowing_terms(device, sx, sw):
    """bf16 has fp32's exponents: chains of subnormal sums, and infinities (and
    NaN where two of them cancel) at the other end."""
    from oracle import moe_oracle as O
    rng = np.random.default_rng(3)
    x = O.round_to((rng.standard_normal((4230, 256)) * sx).astype(np.float32), "bf16")
    w = O.round_to((rng.standard_normal((8, 256)) * sw).astype(np.float32), "bf16")
    _, _, logits, _ = _run(device, "bf16", x, w, 2)
    with np.errstate(all="ignore"):
        ref = O.router_logits(x, w, acc="f32")
    assert np.array_equal(np.isnan(logits), np.isnan(ref))
    at = ~np.isnan(ref)
    assert np.array_equal(logits[at], ref[at])
    assert sx > 1 or np.count_nonzero(ref) > ref.size // 2
