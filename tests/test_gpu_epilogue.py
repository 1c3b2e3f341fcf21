"""The tile kernels' epilogue: the gate over its whole range of arguments, and outputs whose rows and columns end anywhere
inside a wave tile, on uncut and cut launches (GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _built_in_choice(monkeypatch):
    monkeypatch.setenv("TRITONIX_AUTOTUNE", "0")


def _gated(values, act, dtype):
    """act(v) of every v through the gated kernel: column 0 of x is the gate's argument, column 1 the constant one."""
    from tritonix_amd.ops.swiglu import glu

    m, h = values.numel(), 64
    x = torch.zeros(m, 64, dtype=dtype, device="cuda")
    x[:, 0], x[:, 1] = values.to("cuda"), 1.0
    w = torch.zeros(64, 2 * h, dtype=dtype, device="cuda")
    w[0, 0::2], w[1, 1::2] = 1.0, 1.0
    return glu(x, w, activation=act)


@pytest.mark.parametrize("act", ["silu", "sigmoid"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_over_its_range(dtype, act):
    """One rounding to 16 bits (2^-9, 2^-12) and a few units of binary32; 2^-8 and 2^-10 asked for.  Below -88 exp(-g) leaves
    binary32 and the gate is zero; float16 results below 2^-14 are subnormal, with steps of 2^-24."""
    v = torch.cat([torch.linspace(-87, 87, 701), torch.tensor([-66.5, -67.0, 0.0, -0.0, 1e-6, -1e-6, 66.5, 200.0, 6e4])]).to(dtype)
    z = _gated(v, act, dtype).double().cpu()
    g = v.double()
    want = (g if act == "silu" else torch.ones_like(g)) / (1.0 + torch.exp(-g))
    rel, step = (2.0 ** -8, 2.0 ** -126) if dtype == torch.bfloat16 else (2.0 ** -10, 2.0 ** -24)
    err = (z - want[:, None]).abs()
    assert bool((err <= rel * want.abs()[:, None] + step).all()), (err / (want.abs()[:, None] + step)).max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_of_infinities_and_nans(dtype):
    # x holds no infinity next to another column's finite value here: an infinite gate argument meets weights of 1 and 0,
    # and inf * 0 is NaN in every column but its own, so the argument is made infinite by the sum instead
    from tritonix_amd.ops.swiglu import glu

    big = torch.finfo(dtype).max
    x = torch.zeros(3, 64, dtype=dtype, device="cuda")
    x[:, 1] = 1.0
    x[0, 2:] = big
    x[1, 2:] = -big
    x[2, 0] = float("nan")
    w = torch.zeros(64, 128, dtype=dtype, device="cuda")
    w[2:, 0::2], w[1, 1::2] = big, 1.0
    w[0, 0::2] = 1.0
    for act, want in (("silu", (float("inf"), None)), ("sigmoid", (1.0, 0.0))):
        z = glu(x, w, activation=act).float().cpu()
        if dtype == torch.bfloat16:                       # the sums overflow binary32
            assert bool((z[0] == want[0]).all())
            assert bool((z[1].isnan() if want[1] is None else z[1] == want[1]).all())   # -inf * 0, as silu(-inf) is written
        assert bool(z[2].isnan().all())


@pytest.mark.parametrize("cut", [1, 2, 3, 5])
@pytest.mark.parametrize("tile", [(32, 64, 4, 4), (64, 64, 4, 4), (64, 128, 8, 3), (128, 128, 8, 3), (128, 256, 8, 3), (192, 192, 8, 3),
                                  (256, 192, 8, 2), (256, 256, 8, 2), (256, 256, 4, 2)])
def test_edges_of_a_wave_tile(tile, cut):
    """Rows and columns that end one before, at and one after a row-block and a chunk, cut and uncut, bit for bit against the
    float32 product of small integers (exact in bfloat16 and in every partial sum)."""
    from tritonix_amd.ops.matmul import matmul_kernel

    bm, bn, nw, st = tile
    gen = torch.Generator("cpu").manual_seed(17 * bm + bn + cut)
    k = 64 * 5 * cut // max(cut - 1, 1)
    for m, n in ((1, 8), (15, 9), (bm - 1, bn), (bm, bn + 8), (bm + 17, bn - 7), (2 * bm - 15, 2 * bn - 1)):
        a = torch.randint(-2, 3, (m, k), generator=gen).bfloat16()
        b = torch.randint(-1, 2, (k, n), generator=gen).bfloat16()
        c = torch.full((m + 2, n + 3), 7.0, dtype=torch.bfloat16, device="cuda")
        view = c[1:m + 1, 1:n + 1]
        matmul_kernel[(1, 1)](a.cuda(), b.cuda(), view, m, n, k, k, 1, n, 1, c.stride(0), 1, block_m=bm, block_n=bn, block_k=64,
                              group_m=8, num_stages=st, num_warps=nw, split_k=cut)
        want = (a.float() @ b.float()).bfloat16()
        got = c.cpu()
        assert torch.equal(got[1:m + 1, 1:n + 1], want), (m, n)
        got[1:m + 1, 1:n + 1] = 7.0
        assert bool((got == 7.0).all()), f"written outside C at {(m, n)}"


@pytest.mark.parametrize("cut", [2, 4, 7, 9])
@pytest.mark.parametrize("tile", [(32, 64, 4, 2), (32, 128, 4, 2), (64, 64, 4, 2), (64, 128, 8, 2), (128, 64, 4, 2), (128, 128, 8, 2)])
def test_slices_of_tiles_that_share_a_compute_unit(tile, cut):
    """Tiles of few registers add the slices of a cut in small batches: slice counts around a batch, bit for bit (small
    integers, exact in every partial sum), with rows that end inside the first and the last row-block."""
    from tritonix_amd.ops.matmul import matmul_kernel

    bm, bn, nw, st = tile
    gen = torch.Generator("cpu").manual_seed(bm + bn + cut)
    k, n = 64 * 2 * cut, 2 * bn - 8
    for m in (3, bm, bm + 17):
        a = torch.randint(-2, 3, (m, k), generator=gen).bfloat16()
        b = torch.randint(-1, 2, (k, n), generator=gen).bfloat16()
        c = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        matmul_kernel[(1, 1)](a.cuda(), b.cuda(), c, m, n, k, k, 1, n, 1, n, 1, block_m=bm, block_n=bn, block_k=64, group_m=8,
                              num_stages=st, num_warps=nw, split_k=cut)
        assert torch.equal(c.cpu(), (a.float() @ b.float()).bfloat16()), m
