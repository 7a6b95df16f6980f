"""The element-wise decoder kernels (residual + RMSNorm, rotary embedding, SiLU * up) against the torch op
chains they replace, on the same tensors.  Both round at the same points; an fp32 intermediate that differs
in its last bits may round to the neighbouring value of the dtype: one unit in the last place per rounding."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -20}


def model(dim, dtype, gpu, d=128):
    from minference_amd.llama import LlamaConfig, LlamaPrefill
    return LlamaPrefill(LlamaConfig(vocab_size=8, hidden_size=dim, intermediate_size=8, num_layers=0, num_heads=1,
                                    num_kv_heads=1, head_dim=d), device=gpu, dtype=dtype)


def close(a, b, dtype, units=2):
    return ((a.float() - b.float()).abs() <= units * ULP[dtype] * b.float().abs() + 1e-6).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,dim", [(1, 8), (3, 100), (7, 2048), (5, 4096), (2, 4104), (2, 20000), (3, 2051)])
def test_add_rms_norm(gpu, dtype, rows, dim):
    m = model(dim, dtype, gpu)
    g = torch.Generator(device=gpu).manual_seed(dim)
    x, delta = (torch.randn(rows, dim, device=gpu, generator=g).to(dtype) for _ in range(2))
    w = (1 + 0.1 * torch.randn(dim, device=gpu, generator=g)).to(dtype)
    for d in (None, delta):
        h = x.clone()
        out = m._rms(h, w, delta=d)
        want_h = x if d is None else x + d
        xf = want_h.float()
        want = (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + m.cfg.rms_eps)).to(dtype) * w
        assert torch.equal(h, want_h) and close(out, want, dtype)


@pytest.mark.parametrize("dim", [1000, 3072, 4096, 16384])
def test_rms_norm_of_fp32_rows_rounds_three_times(gpu, dim):
    """Against fp64: the root, its product with the row and that with the weight are rounded once each, the sum is
    not: a relative error of 2^-24 sqrt(3 / 3 * E[m^-2]) = 0.736 * 2^-24 over log-uniform significands m
    (0.76 for the sample; a sum in fp32 gives 0.85 and more)."""
    m = model(dim, torch.float32, gpu)
    g = torch.Generator(device=gpu).manual_seed(dim)
    x, w = torch.randn(4096, dim, device=gpu, generator=g), torch.randn(dim, device=gpu, generator=g)
    want = x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + m.cfg.rms_eps) * w.double()
    assert (m._rms(x, w).double() - want).norm() <= 0.76 * 2.0 ** -24 * want.norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,hq,hk,d", [(1, 1, 1, 128), (33, 5, 2, 128), (70, 2, 1, 96), (9, 3, 3, 20), (5, 1, 1, 6)])
def test_rope_in_place(gpu, dtype, n, hq, hk, d):
    m = model(16, dtype, gpu, d)
    g = torch.Generator(device=gpu).manual_seed(n)
    q, k = torch.randn(n, hq, d, device=gpu, generator=g).to(dtype), torch.randn(n, hk, d, device=gpu, generator=g).to(dtype)
    cos, sin = m._rope_tables(n)
    c2, s2 = (torch.cat([t, t], -1)[:, None] for t in (cos, sin))
    want = [(t.float() * c2 + torch.cat([-t[..., d // 2:], t[..., :d // 2]], -1).float() * s2) for t in (q, k)]
    largest = max(q.float().abs().max().item(), k.float().abs().max().item())
    m._rotate(q, k, cos, sin)
    for got, w in zip((q, k), want):
        # one rounding to the dtype, and the fp32 roundings of two products (fused or not) of numbers up to
        # `largest`, which a result near zero does not shrink: 2 * 2^-24 * largest
        assert ((got.float() - w).abs() <= ULP[dtype] * w.abs() + 2.0 ** -23 * largest).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n", [1, 7, 8, 4097, 70000])
def test_silu_mul(gpu, dtype, n):
    m = model(16, dtype, gpu)
    g = torch.Generator(device=gpu).manual_seed(n)
    gate, up = (4 * torch.randn(n, device=gpu, generator=g).to(dtype) for _ in range(2))
    want = torch.nn.functional.silu(gate) * up
    assert close(m._silu_mul(gate.clone(), up), want, dtype, 3)


def test_silu_mul_fp32_far_from_zero(gpu):
    """fp32 tensors, x in [-80, 80], against fp64: a few roundings (exponential, sum, quotient, product: 2^-21),
    not the 2^-19 that rounding x log2(e) to fp32 would leave at the ends."""
    m = model(16, torch.float32, gpu)
    gate = torch.linspace(-80, 80, 4097, device=gpu)
    up = torch.full_like(gate, 1.5)
    got = m._silu_mul(gate.clone(), up).double()
    want = torch.nn.functional.silu(gate.double()) * up.double()
    assert ((got - want).abs() <= 2.0 ** -21 * want.abs()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_mul_of_every_gate(gpu, dtype):
    """Every finite 16-bit gate: the bits of the torch chain, whose fp32 exponential, sum and quotient are the
    same operations."""
    m = model(16, dtype, gpu)
    gate = torch.arange(-32768, 32768, device=gpu).to(torch.int16).view(dtype)
    gate = gate[torch.isfinite(gate)].contiguous()
    up = torch.ones_like(gate)
    assert torch.equal(m._silu_mul(gate.clone(), up), torch.nn.functional.silu(gate) * up)
