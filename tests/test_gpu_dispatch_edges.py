"""Edges of the kernel selection on the GPU: layouts without a packed side or with 64-bit offsets,
half-precision input of prime lengths, ragged batches of prime lengths and of many work-groups,
against torch's FFT in 64 bits."""
import math

import pytest

import bbfft_amd as bb
import oracle
from gpu_util import have_gpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not have_gpu(), reason="needs a HIP GPU")]


def _err(y, ref):
    return ((y - ref).abs().square().sum() / ref.abs().square().sum()).sqrt().item()


def _dft(x, d):
    import torch
    x = x.to(torch.complex128)
    return torch.fft.fft(x, dim=1) if d < 0 else torch.fft.ifft(x, dim=1, norm="forward")


@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("M,N,K,row,col", [
    (8, 32, 700, 8, 8 * 32 + 8), (8, 128, 500, 10, 1280), (6, 363, 300, 6, 6 * 363 + 1),
    (39, 315, 40, 40, 40 * 315), (16, 128, 300, 18, 18 * 128), (17, 512, 64, 17, 17 * 512 + 3),
    (2, 67, 3, 2, 1 << 27), (3, 35, 3, 3, 1 << 27), (8, 64, 2, 8, 1 << 27)])
def test_output_layouts(M, N, K, row, col, fp):
    """Output rows `row` and K-columns `col` elements apart, input packed or laid out alike."""
    import torch
    ct = torch.complex64 if fp == 4 else torch.complex128
    g = torch.Generator(device="cuda")
    g.manual_seed(M * N)
    x = torch.rand((K, N, M, 2), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    x = torch.view_as_complex(x).to(ct).contiguous()
    size = (K - 1) * col + (N - 1) * row + M
    for d in (-1, 1):
        cfg = bb.configuration(1, [M, N, K], bb.precision(fp), bb.direction(d),
                               bb.transform_type(0))
        cfg.set_strides_default(False)
        cfg.ostride = [1, row, col]
        out = torch.full((size,), 7.0, dtype=ct, device="cuda")
        bb.make_plan(cfg).execute(x, out)
        torch.cuda.synchronize()
        y = out.as_strided((K, N, M), (col, row, 1))
        assert _err(y, _dft(x, d)) <= oracle.tolerance(fp, N)
        gap = out.clone()
        gap.as_strided((K, N, M), (col, row, 1)).fill_(7.0)
        assert (gap == 7.0).all()
        if col < 1 << 20:  # the same layout on both sides
            cfg.istride = [1, row, col]
            src = torch.zeros(size, dtype=ct, device="cuda")
            src.as_strided((K, N, M), (col, row, 1)).copy_(x)
            plan = bb.make_plan(cfg)
            plan.execute(src, out)
            torch.cuda.synchronize()
            assert _err(y, _dft(x, d)) <= oracle.tolerance(fp, N), plan.launches()[0]["kernel"]


@pytest.mark.parametrize("storage", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(4, 37, 3000), (3, 61, 40000), (16, 122, 500), (8, 509, 100),
                                   (4, 512, 60000), (4, 74, 1)])
def test_half_input(M, N, K, storage):
    import torch
    x = (torch.rand((K, N, M, 2), device="cuda") * 2 - 1).to(
        torch.float16 if storage == "f16" else torch.bfloat16)
    y = torch.empty((K, N, M), dtype=torch.complex64, device="cuda")
    bb.make_half_input_plan(f"scfo{M}.{N}*{K}", storage, False).execute(x, y)
    torch.cuda.synchronize()
    rows = slice(0, 2000)
    ref = _dft(torch.view_as_complex(x[rows].to(torch.float64)), -1)
    assert _err(y[rows], ref) <= oracle.tolerance(4, N)


@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("jobs", [40, 3])
def test_ragged_batches(jobs, fp):
    """Prime lengths of one wide stage beside others; with 40 jobs the work split comes from the
    device."""
    import random
    import torch
    from bbfft_amd import ragged
    rng = random.Random(fp)
    lengths = (17, 31, 41, 61, 60, 128, 315) if jobs > 3 else (61, 12, 512)
    js = ragged.pack([ragged.Job(rng.choice((1, 2, 3, 8)), lengths[i % len(lengths)],
                                 rng.randint(1, 9000 if jobs > 3 else 40),
                                 rng.choice((-1, 1))) for i in range(jobs)])
    ct = torch.complex64 if fp == 4 else torch.complex128
    n = ragged.total_elements(js)
    x = torch.view_as_complex(torch.rand((n, 2), device="cuda", dtype=torch.float64) * 2 - 1).to(ct)
    y = torch.empty_like(x)
    plan = ragged.make_ragged_plan(js, precision=fp)
    assert (plan.launches()[0]["grid"] >= 4096) == (jobs > 3)
    for _ in range(2):
        y.zero_()
        plan.execute(x, y)
        torch.cuda.synchronize()
        for j in js:
            s = slice(j.in_offset, j.in_offset + j.elements)
            ref = _dft(x[s].reshape(j.K, j.N, j.M), j.direction)
            assert _err(y[s].reshape(j.K, j.N, j.M), ref) <= oracle.tolerance(fp, j.N), j


@pytest.mark.parametrize("fp", [4, 8])
def test_infinite_input_of_a_prime_length(fp):
    """Output 0 on the matrix cores: infinite where the input is, not NaN."""
    import torch
    M, N, K = 8, 37, 4000
    ct = torch.complex64 if fp == 4 else torch.complex128
    x = torch.ones((K, N, M), dtype=ct, device="cuda")
    x[5, 3, 2] = complex(math.inf, 0.0)
    y = torch.empty_like(x)
    plan = bb.make_plan(f"{'s' if fp == 4 else 'd'}cfo{M}.{N}*{K}")
    assert int(plan.launches()[0]["kernel"].split("_g")[1]) & 2048
    plan.execute(x, y)
    torch.cuda.synchronize()
    assert y[5, 0, 2].real == math.inf and y[5, 0, 2].imag == 0.0
    y[5, :, 2] = 0
    assert torch.isfinite(torch.view_as_real(y)).all()
