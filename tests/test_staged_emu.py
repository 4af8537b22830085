"""Staged tiles, per-tile work-item ids and XCD runs of the plain kernels, on the CPU emulator:
the same bits as the kernels without them, over packed layouts of odd and even sizes, K
remainders, tiles of less than 16 bytes and buffers that do not start on 16-byte boundaries."""
import numpy as np
import pytest

import bbfft_amd as bb
import oracle
from emu import runner

STAGE_IN, STAGE_OUT, PER_TILE_IDS, XCD_RUNS = 128, 256, 512, 1024
SHAPES = [(1, 64, 37), (3, 60, 11), (5, 35, 7), (1, 16, 9), (7, 9, 5), (2, 512, 3), (1, 27, 130),
          (1, 3, 2), (1, 2, 1), (17, 33, 3)]
KINDS = [(0, -1), (0, 1), (1, -1), (2, 1)]  # (type, direction)


def _cfg(M, N, K, fp, d, t, inplace=False):
    cfg = bb.configuration(1, [M, N, K], bb.precision(fp), bb.direction(d),
                           bb.transform_type(t))
    cfg.set_strides_default(inplace)
    return cfg


def _tuning(cfg, M, flags):
    kc = bb.kernel_configuration(cfg)
    return dict(factorization=kc["factorization"], Nt=kc["Nt"], Mb=M, Kb=min(kc["Kb"], 3),
                lds_pad=kc["lds_pad"], no_pad=kc["lds_pad"] == 0, flags=flags)


def _sizes(M, N, K, t):
    h = N // 2 + 1
    return M * (h if t == 2 else N) * K, M * (h if t == 1 else N) * K


def _input(N, n, t):
    x = oracle.uniform_complex(N, n)
    return x.real.copy() if t == 1 else x


@pytest.mark.parametrize("flags", [PER_TILE_IDS, STAGE_IN, STAGE_OUT,
                                   STAGE_IN | STAGE_OUT | PER_TILE_IDS | XCD_RUNS | 3])
@pytest.mark.parametrize("t,d", KINDS)
@pytest.mark.parametrize("fp", [4, 8])
def test_same_bits_as_direct_access(fp, t, d, flags):
    for M, N, K in SHAPES:
        cfg = _cfg(M, N, K, fp, d, t)
        n_in, n_out = _sizes(M, N, K, t)
        x = _input(N, n_in, t)
        plain = runner.run(bb, cfg, x, n_out, tuning=_tuning(cfg, M, 0), grid_cap=2)
        other = runner.run(bb, cfg, x, n_out, tuning=_tuning(cfg, M, flags), grid_cap=2)
        assert np.array_equal(plain, other), (M, N, K)


@pytest.mark.parametrize("t,d", KINDS)
@pytest.mark.parametrize("fp", [4, 8])
def test_buffers_off_the_16_byte_boundary(fp, t, d):
    """Element-aligned buffers at every offset from a 16-byte boundary: the words before the
    first and after the last boundary move singly, and nothing outside the tensors changes."""
    npr, npc = (np.float32, np.complex64) if fp == 4 else (np.float64, np.complex128)
    real_t, cplx_t = ("float", "float2") if fp == 4 else ("double", "double2")
    for M, N, K in [(3, 35, 4), (1, 27, 9), (5, 9, 2), (1, 64, 3)]:
        cfg = _cfg(M, N, K, fp, d, t)
        tun = _tuning(cfg, M, STAGE_IN | STAGE_OUT | PER_TILE_IDS | 3)
        kc = bb.kernel_configuration(cfg, tuning=tun)
        in_t, out_t = (real_t if t == 1 else cplx_t), (real_t if t == 2 else cplx_t)
        fn = runner.compile_kernel(bb.generate_source(cfg, tuning=tun), kc["name"], in_t, out_t)
        n_in, n_out = _sizes(M, N, K, t)
        x = _input(N, n_in, t).astype(npr if t == 1 else npc)
        ref = runner.run(bb, cfg, x, n_out, tuning=_tuning(cfg, M, 0))
        kcols = (K + 1) // 2 if t and N % 2 else K
        grid = -(-kcols // kc["Kb"])
        # offsets that keep the kernel's element alignment (pairs of reals for even N, M = 1)
        pair = M == 1 and N % 2 == 0
        step_in = fp if t == 1 and not pair else 2 * fp
        step_out = fp if t == 2 and not pair else 2 * fp
        for oi in range(0, 16, step_in):
            for oo in range(0, 16, step_out):
                src = np.zeros(x.nbytes + 32, np.uint8)
                dst = np.full(ref.nbytes + 48, 0xA5, np.uint8)
                bi = -src.ctypes.data % 16 + oi
                bo = -dst.ctypes.data % 16 + oo
                src[bi:bi + x.nbytes] = x.view(np.uint8).ravel()
                assert fn(src.ctypes.data + bi, dst.ctypes.data + bo, K, grid,
                          kc["work_group_size"]) == 0
                out = dst[bo:bo + ref.nbytes]
                assert np.array_equal(out, ref.view(np.uint8).ravel()), (M, N, K, oi, oo)
                assert (dst[:bo] == 0xA5).all() and (dst[bo + ref.nbytes:] == 0xA5).all()


@pytest.mark.parametrize("M,N,K,mb", [(17, 20, 5, 9), (40, 16, 3, 16), (9, 64, 40, 4)])
def test_xcd_runs_cover_every_m_tile(M, N, K, mb):
    cfg = _cfg(M, N, K, 4, -1, 0)
    tun = dict(_tuning(cfg, M, PER_TILE_IDS), Mb=mb, Kb=1)
    x = _input(N, M * N * K, 0)
    plain = runner.run(bb, cfg, x, M * N * K, tuning=dict(tun, flags=0))
    for cap in (None, 7):
        runs = runner.run(bb, cfg, x, M * N * K, tuning=dict(tun, flags=PER_TILE_IDS | XCD_RUNS),
                          grid_cap=cap)
        assert np.array_equal(plain, runs)


@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("t,d", [(1, -1), (2, 1)])
def test_in_place_real_transforms_stage_the_packed_side(fp, t, d):
    """In place, the real side is padded (not packed): only the spectrum's side is staged."""
    M, N, K = 3, 20, 40000
    kc = bb.kernel_configuration(_cfg(M, N, K, fp, d, t, True))
    flags = int(kc["name"].split("_g")[1].split("_")[0])
    assert bool(flags & STAGE_OUT) == (t == 1) and bool(flags & STAGE_IN) == (t == 2)
    K = 5
    cfg = _cfg(M, N, K, fp, d, t, True)
    tun = dict(_tuning(cfg, M, flags))
    H = N // 2 + 1
    npr, npc = (np.float32, np.complex64) if fp == 4 else (np.float64, np.complex128)
    buf = np.zeros(M * H * K, npc)
    rng = np.random.default_rng(3)
    field = rng.uniform(-1, 1, (K, N, M))
    spec = np.fft.rfft(field, axis=1)
    if t == 1:
        r = buf.view(npr).reshape(K, 2 * H, M)
        r[:, :N, :] = field
    else:
        buf[:] = spec.reshape(-1)
    runner.run(bb, cfg, None, 0, in_place_buffer=buf, tuning=tun)
    tol = oracle.tolerance(fp, N)
    if t == 1:
        assert oracle.rel_l2(buf, spec.reshape(-1)) <= tol
    else:
        assert oracle.rel_l2(buf.view(npr).reshape(K, 2 * H, M)[:, :N, :].ravel() / N,
                             field.ravel()) <= tol


def test_staged_sides_need_packed_columns():
    def bad(cfg, flags, **kw):
        with pytest.raises(bb.BadConfiguration):
            bb.kernel_configuration(cfg, tuning=dict(flags=flags, **kw))
    cfg = bb.configuration(1, [2, 16, 3], istride=[1, 3, 48], ostride=[1, 3, 48])
    bad(cfg, STAGE_IN)
    bad(cfg, STAGE_OUT)
    cfg = _cfg(4, 16, 3, 4, -1, 0)
    bad(cfg, STAGE_IN, Mb=2)
    bad(cfg, STAGE_IN | bb.PREFETCH)
    bad(cfg, PER_TILE_IDS | bb.PREFETCH)
    cfg.callbacks = bb.user_module("__device__ float2 ld(float2* p, size_t o) { return p[o]; }",
                                   "ld")
    bad(cfg, STAGE_IN)
    assert "_g" in bb.kernel_configuration(cfg, tuning=dict(flags=STAGE_OUT))["name"]


@pytest.mark.skipif(not runner.have_tsan(), reason="no ThreadSanitizer runtime")
@pytest.mark.parametrize("M,N,K,fp,t,d,inplace", [
    (3, 60, 7, 4, 0, -1, False), (2, 16, 9, 4, 0, 1, True), (1, 27, 8, 4, 1, -1, False),
    (3, 20, 5, 4, 1, -1, False), (5, 9, 4, 8, 2, 1, False), (1, 64, 6, 4, 2, 1, False)])
def test_staged_kernels_are_race_free(M, N, K, fp, t, d, inplace):
    """Copies in and out share the LDS buffer with the stages' exchange (several tiles per
    work-group, in place included)."""
    cfg = _cfg(M, N, K, fp, d, t, inplace)
    tun = dict(_tuning(cfg, M, STAGE_IN | STAGE_OUT | PER_TILE_IDS | XCD_RUNS), Kb=2)
    kc = bb.kernel_configuration(cfg, tuning=tun)
    rt, ct = ("float", "float2") if fp == 4 else ("double", "double2")
    call = (f'{kc["name"]}((const {rt if t == 1 else ct}*)in, ({rt if t == 2 else ct}*)out, '
            f'{K}ul)')
    n_in, n_out = _sizes(M, N, K, t)
    in_b, out_b = n_in * fp * (1 if t == 1 else 2), n_out * fp * (1 if t == 2 else 2)
    ok, report = runner.race_check(bb.generate_source(cfg, tuning=tun), call, in_b, out_b, 2,
                                   kc["work_group_size"], in_place=inplace)
    assert ok, report[-3000:]


MATRIX = 2048
MATRIX_CASES = [  # M, N, K, factorisation, work-items per transform, M tile, K tile
    (1, 67, 5, [67], 64, 1, 2), (2, 134, 3, [67, 2], 32, 2, 1), (2, 134, 3, [2, 67], 32, 2, 1),
    (4, 212, 3, [53, 4], 16, 4, 1), (3, 67, 9, [67], 64, 3, 2), (2, 37, 7, [37], 32, 2, 2),
    (4, 127, 3, [127], 16, 4, 2), (5, 17, 3, [17], 32, 2, 1), (2, 469, 3, [7, 67], 224, 2, 1),
    (2, 509, 2, [509], 32, 2, 1), (3, 67, 7, [67], 8, 3, 3), (5, 74, 3, [37, 2], 12, 5, 2)]


@pytest.mark.parametrize("flags", [PER_TILE_IDS, PER_TILE_IDS | STAGE_IN | STAGE_OUT | 3])
@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("M,N,K,fac,Nt,Mb,Kb", MATRIX_CASES)
def test_matrix_sums(M, N, K, fac, Nt, Mb, Kb, fp, flags):
    """The direct stage on the matrix cores against the FP64 oracle: c2c of the length and the
    real transforms of twice the length (even) and of the length (odd)."""
    if flags & STAGE_IN and Mb != M:
        pytest.skip("staged tiles hold all M columns")
    tun = dict(factorization=fac, Nt=Nt, Mb=Mb, Kb=Kb, no_pad=True, flags=flags | MATRIX)
    for t, d, n in [(0, -1, N), (0, 1, N), (1, -1, 2 * N), (2, 1, 2 * N), (1, -1, N), (2, 1, N)]:
        if n == N and t and N % 2 == 0:
            continue
        cfg = _cfg(M, n, K, fp, d, t)
        n_in, n_out = _sizes(M, n, K, t)
        x = _input(n, n_in, t)
        y = runner.run(bb, cfg, x, n_out, tuning=tun, grid_cap=2)
        ref = oracle.fft(1, cfg.shape, cfg.istride, cfg.ostride, t, d, x)
        assert oracle.rel_l2(y, ref) <= oracle.tolerance(fp, n), (t, d, n)


def test_matrix_sums_are_planned_for_large_primes():
    for desc, on in [("scfo8.509*8192", True), ("dcfo8.62*1000", True), ("scfo8.62*1000", False),
                     ("scfo1.74*5000", True), ("scfo8.64*1000", False), ("srfo8.134*900", True)]:
        kc = bb.kernel_configuration(bb.parse_fft_descriptor(desc + ""))
        flags = int(kc["name"].split("_g")[1].split("_")[0]) if "_g" in kc["name"] else 0
        assert bool(flags & MATRIX) == on, desc
        assert not on or kc["work_group_size"] % 64 == 0
    cfg = _cfg(2, 64, 3, 4, -1, 0)
    with pytest.raises(bb.BadConfiguration):
        bb.kernel_configuration(cfg, tuning=dict(flags=MATRIX))
    kc = bb.kernel_configuration(_cfg(3, 67, 3, 4, -1, 0), tuning=dict(
        factorization=[67], Nt=8, Mb=3, Kb=3, no_pad=True, flags=MATRIX))
    assert kc["work_group_size"] == 128  # 72 work-items, whole waves


def test_tiles_are_staged_beyond_the_l2():
    """Data up to 34 MB (real transforms 26 MB) is accessed directly with streamed stores; real
    transforms of short rows and larger data are staged; layouts that are not packed are not."""
    def flags(desc, strides=None):
        cfg = bb.parse_fft_descriptor(desc)
        if strides:
            cfg.istride, cfg.ostride = strides
        kc = bb.kernel_configuration(cfg)
        return int(kc["name"].split("_g")[1].split("_")[0]) if "_g" in kc["name"] else 0
    staged = STAGE_IN | STAGE_OUT
    for desc, want in [("scfo8.256*1000", 0), ("scfo8.256*1100", staged), ("dcfo3.100*3500", 0),
                       ("dcfo3.100*3800", staged), ("srfo8.64*6000", 0),
                       ("srfo8.64*6800", staged), ("srfo1.64*1000", staged),
                       ("srfo1.512*1000", 0), ("dcfo8.512*500", staged),
                       ("dcfo8.512*8192", 0)]:
        f = flags(desc)
        assert f & staged == want and f & PER_TILE_IDS, desc
    assert flags("scfo8.256*1000") & 3 == 2 and flags("scfo8.256*1100") & 3 == 3
    padded = [1, 9, 9 * 256]
    assert flags("scfo8.256*1100", (padded, padded)) & staged == 0


@pytest.mark.parametrize("fp", [4, 8])
def test_ragged_variants_stage_whole_tiles(fp):
    """A ragged kernel of staged variants (all M columns in a tile) and an M-tiled one, jobs at
    odd offsets."""
    from bbfft_amd import ragged
    jobs, off = [], 1
    for M, N, K, d in [(3, 20, 5, -1), (200, 12, 2, 1), (1, 27, 9, -1), (2, 16, 1, 1), (1, 5, 3, -1)]:
        jobs.append(ragged.Job(M, N, K, d, off, off + 2))
        off += M * N * K + 1
    tiles = [ragged.variant_configuration(jobs, v, fp)["Mb"] for v in ragged.job_variants(jobs, fp)]
    assert tiles[0] == 3 and tiles[1] < 200
    x = oracle.uniform_complex(9, off + 4)
    y = runner.run_ragged(ragged, jobs, x, off + 4, precision=fp, grid=3)
    for j in jobs:
        st = [1, j.M, j.M * j.N]
        ref = oracle.fft(1, [j.M, j.N, j.K], st, st, 0, j.direction,
                         x[j.in_offset:j.in_offset + j.elements])
        assert oracle.rel_l2(y[j.out_offset:j.out_offset + j.elements],
                             ref) <= oracle.tolerance(fp, j.N), j


@pytest.mark.parametrize("mfma", [False, True])
def test_half_input_stages_its_output_only(mfma):
    for K, staged in [(1000, False), (40000, not mfma), (100000, True)]:
        kc = bb.half_input_kernel_configuration(f"scfo4.512*{K}", "f16", mfma)
        flags = int(kc["name"].split("_g")[1].split("_")[0])
        assert bool(flags & STAGE_OUT) == staged and not flags & STAGE_IN
        assert flags & PER_TILE_IDS and flags & 3 == 2
