"""GPU: the W8 product's plans for more than one row tile (and the short-K residual plan of one) at the
edges of their rules: slabs of four, two and one tile, K splits with a shorter last one, short K, wide
and narrow gated projections. Against float64: at most K float32 terms per sum (K * 2^-24 of the sum of
magnitudes), and the stores' roundings."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _weight(N, K, paired, dev):
    from mlx_dspark.ops import W8Weight
    g = torch.Generator(device=dev).manual_seed(N + K)
    q, s, b = W8Weight.quantize_mlx(torch.randn(N, K, generator=g, device=dev) * 0.02)
    qs = q.double().view(N, K // 64, 64) * s.double()[..., None]
    bb = b.double()[..., None].expand(N, K // 64, 64)
    return W8Weight.from_mlx(q, s, b, paired), (qs + bb).reshape(N, K), (qs + bb.abs()).reshape(N, K)


@pytest.mark.parametrize("M", [9, 17, 32, 36, 48, 64])
@pytest.mark.parametrize("N,K", [(1024, 2048), (3840, 2304), (96, 2048), (48, 512), (512, 1024), (16384, 256)])
def test_row_tile_plans(dev, M, N, K):
    from mlx_dspark.ops import (DSK_EPI_PARTIAL, DSK_EPI_SWIGLU, gemm_plan, pack, pack_rn, w8_gemm, w8_residual)
    print(f"row tiles M={M} N={N} K={K} partial plan {gemm_plan(M, N, K, DSK_EPI_PARTIAL)}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + K)
    h = (torch.randn(M, K, generator=g, device=dev) * 3).to(torch.bfloat16)
    norm = (1 + 0.2 * torch.randn(K, generator=g, device=dev)).to(torch.bfloat16)
    W, w64, mag = _weight(N, K, False, dev)
    x64 = (h.float() * norm.float()).to(torch.bfloat16).double()
    r = torch.rsqrt(h.double().square().mean(1, keepdim=True) + 1e-6)
    xn = pack_rn(M=M, K=K, h=h.clone(), norm_w=norm, eps=1e-6)
    ref, bound = x64 @ w64.T, K * 2.0 ** -24 * (x64.abs() @ mag.T)
    part = w8_gemm(xn.plain(), W, epi=DSK_EPI_PARTIAL)
    assert bool(((part.double().sum(0) - ref).abs() <= bound).all())
    y = w8_gemm(xn, W, out_dtype=torch.float32)
    assert bool(((y.double() - ref * r).abs() <= (bound + ref.abs() * 2.0 ** -18) * r).all())
    if N % 64 == 0:
        res = torch.randn(M, N, generator=g, device=dev).to(torch.bfloat16)
        hh = res.clone()
        w8_residual(pack(h), W, hh, next_norm=None, eps=1e-6, out=False)
        want, mags = res.double() + h.double() @ w64.T, K * 2.0 ** -24 * (h.double().abs() @ mag.T)
        assert bool(((hh.double() - want).abs() <= mags + want.abs() * 2.0 ** -8).all())
    if N % 256 == 0:
        Wp, w64, mag = _weight(N, K, True, dev)
        act = w8_gemm(xn, Wp, epi=DSK_EPI_SWIGLU).unpack().double()
        ref = (x64 @ w64.T) * r
        gate, up = ref[:, :N // 2], ref[:, N // 2:]
        s = torch.nn.functional.silu(gate)
        # bf16 roundings of gate, up, their activation and the product
        assert bool(((act - s * up).abs() <= 2.0 ** -6 * (gate.abs() + s.abs() + 2.0 ** -8) * (up.abs() + 2.0 ** -8)).all())
