"""Where the waves that share K leave wide outputs of a long K to the kernels that had them (csrc/gemm_kwaves.h, kwaves_behind), and where they
do not: the kernel by its name, and exact results."""
import pytest
import torch

from oracle import oracle as orc
from test_gpu_kwaves import _name
from test_gpu_rows import _s8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,N,K,waves", [
    (160, 7168, 7680, False), (80, 8192, 8192, False), (100, 7680, 7168, False), (100, 10240, 5120, False), (150, 10240, 5120, False),
    (170, 10240, 5120, False), (240, 5120, 7680, False), (70, 17920, 2560, False), (120, 13312, 5120, False), (700, 2560, 2048, False),
    (100, 5120, 7168, True), (100, 4096, 8192, True), (100, 10240, 4096, True), (150, 10240, 2560, True), (90, 20480, 5120, True),
    (120, 12800, 5120, True), (700, 2560, 2560, True)])
def test_wide_outputs_of_a_long_k(M, N, K, waves):
    import torch_int._CUDA as C
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = (torch.randint(-127, 128, s, dtype=torch.int8, device=DEV, generator=g) for s in ((M, K), (N, K)))
    b8 = _s8(torch.Generator().manual_seed(N), N)
    print("wide outputs", M, N, K, flush=True)
    acc = torch.mm(x.double(), w.double().t().contiguous()).to(torch.int32).cpu()   # sums below 2^53
    out = C.linear_a8_w8_b8_o8(x, w, b8.to(DEV), 3e-4, 0.02)
    assert _name().startswith("mid_waves_") == waves, _name()
    assert torch.equal(out.cpu(), orc.epi_b8_o8(acc, b8, 3e-4, 0.02))
