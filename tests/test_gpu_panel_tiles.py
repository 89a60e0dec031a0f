"""The tilings of 1025 rows and more that are chosen by price (8-bit 256x256, the 128x128 of one round, 192x128, 192x256, 160x256),
at the edges of their rows, columns and K, three of them in one launch, and rows too far apart for 32-bit panel offsets.
Bit for bit against an exact fp64 product on the device."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _s8(gen, shape, std):
    return torch.randn(shape, device=DEV, generator=gen).mul_(std).round_().clamp_(-127, 127).to(torch.int8)


def _run(M, N, K, out_dtype, seed):
    """-> (result, exact int64 accumulator, bias) of a linear whose epilogue is exact: scale 1, int32 or int8 output."""
    import torch_int._CUDA as C
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x, w = _s8(gen, (M, K), 3.0), _s8(gen, (N, K), 3.0)
    acc = x.double() @ w.double().t()
    if out_dtype == torch.int32:
        bias = torch.randint(-65535, 65536, (N,), dtype=torch.int32, device=DEV, generator=gen)
        out, want = C.linear_a8_w8_b32_o32(x, w, bias), (acc.long() + bias.long()).int()
    else:   # a power of two: products and sums of the epilogue are exact in fp32
        bias = _s8(gen, (N,), 20.0)
        scale = 2.0 ** -round(0.5 * torch.log2(torch.tensor(float(K))).item() - 1)
        out = C.linear_a8_w8_b8_o8(x, w, bias, scale, 0.5)
        want = torch.clamp(torch.round(acc * scale + 0.5 * bias.double()), -128, 127).to(torch.int8)
    return out, want


@pytest.mark.parametrize("out_dtype", [torch.int8, torch.int32])
@pytest.mark.parametrize("M,N,K,family", [
    (1025, 2048, 512, "pipe_128x128"), (2048, 2048, 640, "pipe_128x128"), (2047, 2033, 2048, "pipe_128x128"),
    (1921, 2041, 4224, "pipe_128x128"), (2048, 7168, 2048, "pipe_256x256"), (2047, 7151, 2176, "pipe_256x256"),
    (1793, 7424, 4096, "pipe_256x256"),
    (3000, 2048, 2048, "pipe16_192x128"), (2881, 2048, 768, "pipe16_192x128"), (2945, 2001, 1024, "pipe16_192x128"),
    (2112, 5120, 5120, "pipe16_192x256"), (2113, 5120, 2048, "pipe16_192x256"), (2111, 5104, 1152, "pipe16_192x256"),
    (2400, 4096, 4096, "pipe16_160x256"), (2241, 4096, 1280, "pipe16_160x256")])
def test_panel_tiles(M, N, K, family, out_dtype):
    import torch_int._CUDA as C
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    print(f"panel tiles {M}x{N}x{K} {out_dtype}", flush=True)
    out, want = _run(M, N, K, out_dtype, M + N + K)
    assert C._lib.ti_last_kernel().decode() == family
    assert torch.equal(out, want)


def test_rows_too_far_apart_for_panel_offsets():
    out, want = _run(20, 24, (1 << 23) + 128, torch.int32, 5)
    assert torch.equal(out, want)


@pytest.mark.parametrize("B,T,H,d,K", [(8, 256, 32, 64, 2048), (1, 1905, 16, 128, 2048), (3, 683, 32, 64, 2176)])
def test_three_projections_on_256x256_tiles(B, T, H, d, K):
    import torch_int._CUDA as C
    import torch_int._hip_ext as X
    C._lib.ti_last_kernel.restype = ctypes.c_char_p
    gen = torch.Generator(device=DEV).manual_seed(T)
    M, N = B * T, H * d
    x, ws, bs = _s8(gen, (M, K), 3.0), [_s8(gen, (N, K), 3.0) for _ in range(3)], [_s8(gen, (N,), 20.0) for _ in range(3)]
    al, be = [2.0 ** -8, 2.0 ** -7, 2.0 ** -9], [0.5, 1.0, 0.25]
    print(f"group {M}x{N}x{K}", flush=True)
    out = X.linear_a8_w8_b8_o8_group_heads(x, ws, bs, al, be, B, T, H, d)
    assert C._lib.ti_last_kernel().decode() == "pipe16_256x256_group"
    for o, w, b, a, c in zip(out, ws, bs, al, be):
        want = torch.clamp(torch.round((x.double() @ w.double().t()) * a + c * b.double()), -128, 127).to(torch.int8)
        assert torch.equal(o, want.view(B, T, H, d).transpose(1, 2))
