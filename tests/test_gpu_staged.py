"""Plain kernels of shapes without a table entry on the GPU (staged tiles, M tiles, XCD runs),
compiled by the hiprtc of the running process, against torch's FFT in 64 bits."""
import math

import pytest

import bbfft_amd as bb
import oracle
from gpu_util import have_gpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not have_gpu(), reason="needs a HIP GPU")]

# M tiles and seams (17, 39, 64 columns), one column, odd and even lengths, the largest lengths
SHAPES = [(1, 2), (1, 16), (1, 27), (1, 64), (1, 315), (1, 512), (2, 128), (3, 60), (5, 35),
          (5, 315), (6, 77), (17, 105), (17, 512), (32, 96), (39, 300), (64, 64), (64, 512),
          (70, 20)]
# lengths whose largest prime factor runs on the matrix cores: one to sixteen tiles of output
# pairs, more stages, M tiles, idle columns
MATRIX = [(1, 37), (8, 94), (4, 74), (17, 82), (8, 212), (1, 61), (1, 67), (3, 67), (8, 134),
          (5, 201), (17, 127), (8, 199), (40, 254), (2, 331), (8, 509), (1, 509)]


def _run(M, N, K, fp, t, d, inplace=False, off_in=0, off_out=0):
    import torch
    rt, ct = (torch.float32, torch.complex64) if fp == 4 else (torch.float64, torch.complex128)
    cfg = bb.configuration(1, [M, N, K], bb.precision(fp), bb.direction(d),
                           bb.transform_type(t))
    cfg.set_strides_default(inplace)
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 * M + N)
    H = N // 2 + 1
    field = torch.rand((K, N, M), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    if t == 0:
        im = torch.rand((K, N, M), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
        x = torch.complex(field, im).to(ct)
        ref = torch.fft.fft(x.to(torch.complex128), dim=1)
        if d > 0:
            ref = torch.fft.ifft(x.to(torch.complex128), dim=1, norm="forward")
        out_shape = (K, N, M)
    elif t == 1:
        x = field.to(rt)
        ref = torch.fft.fft(x.double().to(torch.complex128), dim=1)[:, :H].contiguous()
        out_shape = (K, H, M)
    else:
        x = torch.fft.fft(field.to(torch.complex128), dim=1)[:, :H].contiguous().to(ct)
        ref = field * N
        out_shape = (K, N, M)
    plan = bb.make_plan(cfg)
    if inplace:
        buf = torch.empty((K, 2 * H if t else 2 * N, M), dtype=rt, device="cuda")
        if t == 1:
            buf[:, :N] = x
        else:
            buf.reshape(-1).view(ct).copy_(x.reshape(-1))
        plan.execute(buf)
        y = buf[:, :N] if t == 2 else buf.reshape(-1).view(ct).reshape(out_shape)
    else:
        src = torch.zeros(x.numel() + 32, dtype=x.dtype, device="cuda")
        y_t = rt if t == 2 else ct
        dst = torch.full((math.prod(out_shape) + 32,), 7.0, dtype=y_t, device="cuda")
        src[off_in:off_in + x.numel()] = x.reshape(-1)
        y = dst[off_out:off_out + math.prod(out_shape)]
        plan.execute(src[off_in:], y)
        torch.cuda.synchronize()
        assert (dst[:off_out] == 7.0).all() and (dst[off_out + y.numel():] == 7.0).all()
        y = y.reshape(out_shape)
    torch.cuda.synchronize()
    err = ((y - ref).abs().square().sum() / ref.abs().square().sum()).sqrt().item()
    assert err <= oracle.tolerance(fp, N), (plan.launches()[0]["kernel"], err)
    return plan.launches()[0]["kernel"]


@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("t,d", [(0, -1), (0, 1), (1, -1), (2, 1)])
@pytest.mark.parametrize("M,N", SHAPES)
def test_untabled_shapes(M, N, t, d, fp):
    """Enough K-columns to fill the chip (odd counts), and one."""
    _run(M, N, (1 << 20) // (M * N) | 1, fp, t, d)
    _run(M, N, 1, fp, t, d)


@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("t,d", [(0, -1), (0, 1), (1, -1), (2, 1)])
@pytest.mark.parametrize("M,N", MATRIX)
def test_matrix_sums(M, N, t, d, fp):
    _run(M, N, (1 << 20) // (M * N) | 1, fp, t, d)
    _run(M, N, 1, fp, t, d)


@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("t,d", [(0, -1), (1, -1), (2, 1)])
def test_buffers_off_the_16_byte_boundary(t, d, fp):
    for M, N in [(3, 35), (1, 315), (5, 64)]:
        for off_in, off_out in [(1, 0), (0, 1), (1, 3), (3, 2)]:
            _run(M, N, 9001, fp, t, d, off_in=off_in, off_out=off_out)


@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("t,d", [(0, -1), (1, -1), (2, 1)])
@pytest.mark.parametrize("M,N", [(1, 64), (3, 20), (3, 35), (16, 60), (3, 67), (4, 134)])
def test_in_place(M, N, t, d, fp):
    _run(M, N, (1 << 20) // (M * N) | 1, fp, t, d, inplace=True)


@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("t,d", [(0, -1), (1, -1), (2, 1)])
@pytest.mark.parametrize("M,N", [(8, 16), (8, 32), (8, 60), (8, 64), (8, 105), (8, 243), (8, 256),
                                 (8, 384), (8, 512), (1, 64), (1, 128), (4, 512)])
def test_data_in_and_beyond_the_l2(M, N, t, d, fp):
    """Tiles of the tuning table and of the estimate, direct (data that fits the L2) and staged."""
    for elems in (1 << 14, 1 << 20, 5 << 20):
        _run(M, N, elems // (M * N) | 1, fp, t, d)
