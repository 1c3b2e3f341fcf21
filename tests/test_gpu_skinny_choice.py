"""The built-in choice at the edges of its rules for few rows: 32 / 64 rows per tile, 64 or 128 columns (by layout, by the
columns one round holds and by the size of B), K cuts, and the fourth ring slot of a k-contiguous B.

Bound per element against the float64 product: the rounding of the 16-bit result and k fp32 additions on the sum of
magnitudes; int8 is exact."""
import importlib

import pytest
import torch

import tritonix_amd

mm = importlib.import_module("tritonix_amd.ops.matmul")
sg = importlib.import_module("tritonix_amd.ops.swiglu")
pytestmark = pytest.mark.gpu


def _operands(m, n, k, layout, dtype, device):
    g = torch.Generator().manual_seed(m + n + k)
    if dtype == torch.int8:
        a, b = (torch.randint(-127, 128, s, generator=g, dtype=dtype) for s in ((m, k), (k, n)))
    else:
        a, b = torch.randn(m, k, generator=g).to(dtype), (torch.randn(k, n, generator=g) / k ** 0.5).to(dtype)
    ad = a.t().contiguous().to(device).t() if layout[0] == "t" else a.to(device)
    bd = b.t().contiguous().to(device).t() if layout[1] == "t" else b.to(device)
    return ad, bd, ad.double() @ bd.double(), ad.double().abs() @ bd.double().abs()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.int8], ids=["bf16", "f16", "i8"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
def test_few_rows(layout, dtype, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    for m, n, k in ((1, 64, 64), (32, 65, 100), (33, 1000, 1030), (64, 127, 4096), (65, 256, 512), (16, 16384, 448), (16, 16385, 200),
                    (17, 4096, 9728), (31, 4104, 9800), (2, 2048, 14336)):
        a, b, ref, mag = _operands(m, n, k, layout, dtype, device)
        outs = [tritonix_amd.triton_matmul(a, b), mm.matmul_splitk(a, b)]
        for out in outs:
            if dtype == torch.int8:
                assert torch.equal(out.double(), ref), (m, n, k, layout)
            else:
                eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
                assert bool(((out.double() - ref).abs() <= eps * ref.abs() + k * 2.0 ** -23 * mag + 1e-7).all()), (m, n, k, layout)


@pytest.mark.parametrize("m,n,k", [(65, 512, 4096), (512, 4096, 320), (500, 4090, 333), (512, 4224, 256)])
def test_fourth_slot_of_a_k_contiguous_b(m, n, k, device, monkeypatch):
    """Around the sizes where 64x128 tiles fill one round, K loops shorter and longer than the ring, whole and ragged."""
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    a, b, ref, mag = _operands(m, n, k, "nt", torch.bfloat16, device)
    cfg = dict(block_m=64, block_n=128, block_k=64, group_m=8, num_stages=4, num_warps=8)
    for out in (tritonix_amd.triton_matmul(a, b), mm._launch_matmul(a, b, cfg)):
        assert bool(((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + k * 2.0 ** -23 * mag + 1e-7).all())


@pytest.mark.parametrize("m,d,h", [(16, 512, 1024), (32, 520, 8192), (33, 512, 8200), (64, 4096, 1000)])
def test_gated_product_of_few_rows(m, d, h, device, monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")
    g = torch.Generator().manual_seed(m + d + h)
    x, w = torch.randn(m, d, generator=g).bfloat16().to(device), (torch.randn(d, 2 * h, generator=g) * d ** -0.5).bfloat16().to(device)
    z = sg.glu(x, w, activation="silu").double()
    y = x.double() @ w.double()
    ref = torch.nn.functional.silu(y[:, 0::2]) * y[:, 1::2]
    # fp32 inside, one rounding of the result: 2^-8, and the sums' k * 2^-23 of values of order one on either factor
    assert bool(((z - ref).abs() <= 2.0 ** -8 * ref.abs() + 2 * d * 2.0 ** -23 * (1 + y[:, 0::2].abs()) * (1 + y[:, 1::2].abs())).all())
