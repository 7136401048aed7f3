"""Convolutions without a stored im2col matrix (nn_conv, nn_conv_dx, nn_conv_dw)
against im2col + GEMM of the same library: forward and input gradient bit for
bit, weight gradients on operands whose FP32 sums are exact, at image sizes
around the 32-pixel tiles and for every layer shape and input mode."""
import numpy as np
import pytest
import torch

from thesis_amd import nn
from thesis_amd import surrogate as S
from test_gpu_nn import DEV, bf16_words, dev, rng

pytestmark = pytest.mark.gpu
SHAPES = sorted({(cin, cout, k) for _, cin, cout, k, _ in S.ARCH})


def exact(r, n, q=4.0):
    """Multiples of 1/q in [-1, 1]: exact in bf16, their products' sums in FP32."""
    return r.integers(-int(q), int(q) + 1, n) / q


def f32(n):
    return torch.empty(n, dtype=torch.float32, device=DEV)


def i16(n):
    return torch.empty(n, dtype=torch.int16, device=DEV)


def inputs(r, B, H, W, cin, mode, draw):
    """x and skip as given to nn_conv, and the convolution's plain input."""
    small = B * (H // 2) * (W // 2) * cin
    x = dev(draw(small if mode == nn.IN_UP else B * H * W * cin))
    skip = dev(draw(B * H * W * cin)) if mode == nn.IN_ADD else None
    if mode == nn.IN_X:
        return x, skip, x
    full = f32(B * H * W * cin)
    if mode == nn.IN_UP:
        nn.up2(x, B, H // 2, W // 2, cin, full)
    else:
        nn.add(x, skip, full)
    return x, skip, full


# one pixel, a tile's edge and one over, several images; even where upsampled
@pytest.mark.parametrize("B,H,W", [(1, 1, 1), (2, 3, 31), (1, 8, 32), (2, 9, 33), (3, 6, 70), (1, 16, 128)])
@pytest.mark.parametrize("cin,cout,k", SHAPES)
def test_forward_and_input_gradient_same_bits(B, H, W, cin, cout, k):
    r = rng(cin + cout + W)
    M, kp = B * H * W, S.kpad(cin, k)
    w = r.standard_normal((cout, kp)).astype(np.float32)
    w[:, cin * k * k:] = 0
    wb = i16(cout * kp)
    nn.to_bf16(dev(w), wb)
    bias = dev(r.standard_normal(cout))
    modes = [nn.IN_X] if k == 1 or cin == 4 else [nn.IN_X, nn.IN_ADD] + [nn.IN_UP] * (H % 2 == 0 and W % 2 == 0)
    for mode in modes:
        x, skip, full = inputs(r, B, H, W, cin, mode, r.standard_normal)
        col = i16(M * kp)
        nn.im2col(full, B, H, W, cin, kp, col) if k == 3 else nn.to_bf16(full, col)
        for relu in (0, 1):
            want, got = f32(M * cout), f32(M * cout)
            nn.gemm(M, cout, kp, col, kp, 0, wb, kp, 0, want, cout, bias, nn.RELU if relu else 0, 1)
            nn.conv(x, skip, mode, B, H, W, cin, cout, k, wb, kp, bias, relu, got)
            assert torch.equal(got, want), (mode, relu)
    if k == 1 or cin == 4:
        return
    dz = i16(M * cout)
    nn.to_bf16(dev(r.standard_normal(M * cout)), dz)
    dcol, want, got, wt = f32(M * kp), f32(M * cin), f32(M * cin), i16(9 * cin * cout)
    nn.gemm(M, kp, cout, dz, cout, 0, wb, kp, 1, dcol, kp, None, 0, 1)
    nn.col2im(dcol, B, H, W, cin, kp, want)
    nn.weight_t(wb, [(0, 0, cin, cout, kp)], wt)
    nn.conv_dx(dz, B, H, W, cin, cout, wt, got)
    assert torch.equal(got, want)


@pytest.mark.parametrize("B,H,W", [(1, 1, 1), (2, 9, 33), (3, 6, 70), (2, 64, 128)])
@pytest.mark.parametrize("cin,cout,k", SHAPES)
def test_weight_gradient_exact(B, H, W, cin, cout, k):
    r = rng(cin + cout + H)
    M, kp = B * H * W, S.kpad(cin, k)
    dz = bf16_words(exact(r, M * cout))
    modes = [nn.IN_X] if k == 1 or cin == 4 else [nn.IN_X, nn.IN_ADD] + [nn.IN_UP] * (H % 2 == 0 and W % 2 == 0)
    for mode in modes:
        # sums of two multiples of 1/4 stay exact in bf16
        x, skip, full = inputs(r, B, H, W, cin, mode, lambda n: exact(r, n))
        col = i16(M * kp)
        nn.im2col(full, B, H, W, cin, kp, col) if k == 3 else nn.to_bf16(full, col)
        want = torch.full((cout * kp,), 0.5, dtype=torch.float32, device=DEV)
        got = want.clone()
        nn.gemm(kp, cout, M, col, kp, 1, dz, cout, 1, want, kp, None, nn.ATOMIC | nn.TRANSC, 1)
        nn.conv_dw(x, skip, mode, dz, B, H, W, cin, cout, k, kp, got)
        assert torch.equal(got, want), mode


@pytest.mark.parametrize("N", [32, 64, 128])
@pytest.mark.parametrize("M", [1, 7, 40000])
def test_grad_sum(N, M):
    r = rng(N + M)
    dy, y = dev(exact(r, M * N)), dev(r.standard_normal(M * N))
    for relu in (0, 1):
        want, got, wb, gb = i16(M * N), i16(M * N), torch.ones(N, device=DEV), torch.ones(N, device=DEV)
        nn.grad_bf16(dy, y, relu, want)
        nn.colsum(dy, y, relu, M, N, wb)
        nn.grad_sum(dy, y, relu, N, got, gb)
        assert torch.equal(got, want) and torch.equal(gb, wb)


@pytest.mark.parametrize("N", [32, 64, 128])
@pytest.mark.parametrize("B,H,W", [(1, 2, 2), (3, 6, 10), (2, 64, 34)])
def test_grad_sum_through_upsampling_and_pooling(N, B, H, W):
    """The same bits as the adjoint's own pass, then the plain gradient."""
    r, n = rng(N + H), B * H * W * N
    y, skip = dev(r.standard_normal(n)), dev(exact(r, n))
    for mode, m in ((nn.GRAD_UP, 4 * n), (nn.GRAD_POOL, n // 4)):
        dy, g = dev(exact(r, m)), f32(n)
        if mode == nn.GRAD_UP:
            nn.up2_bwd(dy, B, H, W, N, g)
        else:
            nn.avgpool2_bwd(dy, B, H, W, N, g)
            nn.axpy(1.0, skip, g)
        want, got, wb, gb = i16(n), i16(n), torch.ones(N, device=DEV), torch.ones(N, device=DEV)
        nn.grad_sum(g, y, 1, N, want, wb)
        nn.grad_sum(dy, y, 1, N, got, gb, mode, skip, (B, H, W))
        assert torch.equal(got, want) and torch.equal(gb, wb)


def test_rounding_of_special_values():
    """Ties, values next to them, the smallest, the largest and infinities round as
    the integer rounding of grad_bf16 does; NaN stays NaN."""
    hi = np.arange(0, 1 << 16, 7, dtype=np.uint32)
    words = (hi[:, None] << 16 | np.array([0, 1, 0x7FFF, 0x8000, 0x8001, 0x8003, 0xFFFF], np.uint32)).ravel()
    words = np.concatenate([words, np.array([0x7F800000, 0xFF800000, 0x7F7FFFFF, 1, 0x7F800001, 0x7FFFFFFF], np.uint32)])
    words = np.resize(words, (words.size + 31) // 32 * 32)
    dy, n = dev(words.view(np.float32)), words.size
    want, got, db = i16(n), i16(n), torch.zeros(32, device=DEV)
    nn.grad_bf16(dy, dy, 0, want)
    nn.grad_sum(dy, dy, 0, 32, got, db)
    nan = np.isnan(words.view(np.float32))
    w, g = want.cpu().numpy(), got.cpu().numpy()
    assert np.array_equal(w[~nan], g[~nan]) and ((g[nan] & 0x7FFF) > 0x7F80).all()


def test_refused_shapes():
    z, w = f32(64), i16(64)
    for cin, cout, k, mode in ((5, 32, 3, 0), (32, 48, 3, 0), (32, 33, 1, 0), (32, 32, 3, 1), (32, 32, 3, 2)):
        with pytest.raises(Exception):   # the last two: odd image upsampled, no skip
            nn.conv(z, None, mode, 1, 1, 1, cin, cout, k, w, S.kpad(cin, k), z, 0, z)
