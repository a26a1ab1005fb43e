"""Row-grouped TQUANT around the size at which a thread takes two pieces instead of one: a matrix quantised whole equals, bit for bit,
its rows quantised in small matrices (which the oracle's tests cover)."""
import pytest
import torch

from test_gpu_parity import pa  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alg", range(4))
@pytest.mark.parametrize("dtype,rows,cols", [(torch.bfloat16, 2048, 4096), (torch.bfloat16, 2049, 4096), (torch.float16, 2040, 4128), (torch.float32, 2040, 2080)])
def test_whole_matrix_equals_its_rows(pa, alg, dtype, rows, cols):  # noqa: F811
    gen = torch.Generator(device="cuda").manual_seed(rows + alg)
    src = torch.randn((rows, cols), generator=gen, device="cuda") * torch.exp2(torch.randint(-20, 20, (rows, 1), generator=gen, device="cuda").float())
    src[::7, ::13] = 0
    src[5, 40], src[9, 70], src[11, 100] = float("nan"), float("inf"), -float("inf")
    src = src.to(dtype)
    whole = pa.tquant_mx(src, alg)
    parts = [pa.tquant_mx(src[r:r + 300].contiguous(), alg) for r in range(0, rows, 300)]
    for w, *p in zip(whole, *parts):
        assert torch.equal(w.view(torch.uint8), torch.cat(p).view(torch.uint8))
