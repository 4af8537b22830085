"""Edges of the kernel selection on the CPU (configurations, generated sources, emulator): what
a general path accepts and computes, a faster path accepts and computes as well."""
import numpy as np
import pytest

import bbfft_amd as bb
from emu import runner

STAGE_IN, STAGE_OUT, PER_TILE_IDS, MATRIX = 128, 256, 512, 2048


def _cfg(M, N, K, fp, d, t, istride=None, ostride=None):
    cfg = bb.configuration(1, [M, N, K], bb.precision(fp), bb.direction(d),
                           bb.transform_type(t))
    cfg.set_strides_default(False)
    if istride:
        cfg.istride = istride
    if ostride:
        cfg.ostride = ostride
    return cfg


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("M,N,fac,Nt,Kb", [(1, 37, [37], 16, 4), (2, 61, [61], 32, 1),
                                           (1, 74, [37, 2], 32, 2)])
def test_matrix_sums_of_values_that_are_not_finite(M, N, fac, Nt, Kb, fp, bad):
    """One infinite or NaN input: the matrix products leave the same outputs infinite and NaN,
    component by component, as the butterfly in registers does."""
    K = 3
    for d in (-1, 1):
        for at in (0, 1, N - 2):
            x = np.ones((K, N, M), np.complex64 if fp == 4 else np.complex128)
            x[1, at, M - 1] = bad
            cfg = _cfg(M, N, K, fp, d, 0)
            y = [runner.run(bb, cfg, x.ravel(), x.size, tuning=dict(
                factorization=fac, Nt=Nt, Mb=M, Kb=Kb, no_pad=True, flags=f))
                for f in (PER_TILE_IDS, PER_TILE_IDS | MATRIX)]
            for part in (np.real, np.imag):
                assert np.array_equal(np.isnan(part(y[0])), np.isnan(part(y[1]))), (d, at)
                assert np.array_equal(np.isinf(part(y[0])), np.isinf(part(y[1]))), (d, at)


def _flags(kc):
    return int(kc["name"].split("_g")[1].split("_")[0]) if "_g" in kc["name"] else 0


@pytest.mark.parametrize("desc,p", [
    ("scfo1.509x509x509", 2), ("dcfo1.331x331x331", 2), ("scfo1024x1024x67", 2),
    ("dcfo512x512x131", 2), ("scfo640x640x166", 2), ("dcfo2048x2048x47", 2),
    ("scfo1048576.67", 0), ("srfo3.243x315x131*6", 2)])
def test_large_prime_factors_far_apart_are_planned(desc, p):
    """Rows so far apart that a tile may need 64-bit offsets: the sums of a large prime then stay
    in vector code or registers, which have such offsets, instead of on the matrix cores."""
    cfg = bb.parse_fft_descriptor(desc)
    kc = bb.kernel_configuration(cfg, p)
    rows, cols = (int(v) for v in kc["name"].split("_os1_")[1].split("_")[:2])
    span = kc["Mb"] + (kc["N"] + 2) * rows + (kc["Kb"] + 1) * cols
    assert not _flags(kc) & MATRIX or span * 2 * int(cfg.fp) < 1 << 31
    assert (_flags(kc) & MATRIX != 0) == (desc not in ("scfo1.509x509x509", "dcfo2048x2048x47"))


def test_matrix_sums_with_64_bit_offsets_stay_refused():
    cfg = bb.parse_fft_descriptor("scfo2097152.67")
    tun = dict(factorization=[67], Nt=16, Mb=16, Kb=1, no_pad=True)
    assert bb.kernel_configuration(cfg, tuning=dict(tun, flags=PER_TILE_IDS))["Mb"] == 16
    with pytest.raises(bb.BadConfiguration):
        bb.kernel_configuration(cfg, tuning=dict(tun, flags=PER_TILE_IDS | MATRIX))


@pytest.mark.parametrize("t,d", [(0, -1), (1, -1), (2, 1)])
@pytest.mark.parametrize("N", [41, 67, 134])
def test_large_prime_factors_with_64_bit_offsets(N, t, d):
    """K-columns 2^27 elements apart (the buffers' pages in between are never touched)."""
    M, K, far, H = 2, 2, 1 << 27, N // 2 + 1
    n_in, n_out = (H if t == 2 else N), (H if t == 1 else N)
    packed = [1, M, M * n_in] if t == 1 else [1, M, M * n_out]
    cfg = _cfg(M, N, K, 4, d, t, *((packed, [1, M, far]) if t < 2 else ([1, M, far], packed)))
    kc = bb.kernel_configuration(cfg)
    assert not _flags(kc) & MATRIX
    rng = np.random.default_rng(N)
    field = rng.uniform(-1, 1, (K, N, M))
    if t == 2:
        x = np.zeros(far + M * H, np.complex64)
        for k in range(K):
            x[k * far:k * far + M * H] = np.fft.rfft(field[k], axis=0).ravel()
        y = runner.run(bb, cfg, x, M * N * K).reshape(K, N, M) / N
        ref = field
    else:
        y = runner.run(bb, cfg, field.astype(np.float32).ravel(), far + M * n_out)
        y = np.stack([y[k * far:k * far + M * n_out].reshape(n_out, M) for k in range(K)])
        ref = (np.fft.fft if t == 0 else np.fft.rfft)(field, axis=1)
    assert np.linalg.norm(y - ref) <= 8 * 1.2e-7 * np.log2(N) * np.linalg.norm(ref)


@pytest.mark.parametrize("fp", [4, 8])
@pytest.mark.parametrize("t,d", [(0, -1), (0, 1), (1, -1), (2, 1)])
@pytest.mark.parametrize("M,N,K,far", [(1, 16, 32, 1 << 24), (3, 35, 4, 1 << 26),
                                       (8, 64, 2, 1 << 27)])
def test_packed_side_beside_64_bit_offsets(M, N, K, far, t, d, fp):
    """One side packed, the K-columns of the other so far apart that a tile needs 64-bit
    offsets (shapes of the estimate and of the tuning table): no side is staged, and the kernel
    computes what the packed layout's does."""
    H = N // 2 + 1
    n_in, n_out = M * (H if t == 2 else N), M * (H if t == 1 else N)
    rng = np.random.default_rng(M)
    x = rng.uniform(-1, 1, (K, n_in, 1 if t == 1 else 2))
    x = (x[..., 0] if t == 1 else x[..., 0] + 1j * x[..., 1])
    npr, npc = (np.float32, np.complex64) if fp == 4 else (np.float64, np.complex128)
    x = x.astype(npr if t == 1 else npc)
    packed = _cfg(M, N, K, fp, d, t)
    tun = bb.kernel_configuration(packed)
    tun = dict(factorization=tun["factorization"], Nt=tun["Nt"], Mb=M, Kb=1, flags=0)
    ref = runner.run(bb, packed, x.ravel(), K * n_out, tuning=tun)
    cfg = _cfg(M, N, K, fp, d, t, ostride=[1, M, far])
    assert not _flags(bb.kernel_configuration(cfg)) & (STAGE_IN | STAGE_OUT)
    y = runner.run(bb, cfg, x.ravel(), (K - 1) * far + n_out)
    y = np.concatenate([y[k * far:k * far + n_out] for k in range(K)])
    assert np.linalg.norm(y - ref) <= 4 * np.finfo(npr).eps * np.log2(N) * np.linalg.norm(ref)
    cfg = _cfg(M, N, K, fp, d, t, istride=[1, M, far])
    assert not _flags(bb.kernel_configuration(cfg)) & (STAGE_IN | STAGE_OUT)
    assert bb.compile_kernel(cfg) > 1000
    for flag, st in ((STAGE_OUT, dict(istride=[1, M, far])), (STAGE_IN, dict(ostride=[1, M, far]))):
        with pytest.raises(bb.BadConfiguration):  # asked for, it is refused
            bb.kernel_configuration(_cfg(M, N, K, fp, d, t, **st),
                                    tuning=dict(tun, flags=flag, Kb=(1 << 28) // far))


def test_half_input_output_beside_64_bit_offsets():
    cfg = _cfg(4, 512, 40000, 4, -1, 0, istride=[1, 4, 1 << 28])
    assert not _flags(bb.half_input_kernel_configuration(cfg, "f16", False)) & STAGE_OUT


@pytest.mark.parametrize("fp", [4, 8])
def test_ragged_batches_take_every_register_length(fp):
    """One stage of a large prime has a wide K tile and no LDS of its own: its staged tile is
    made narrower or the variant is not staged, never refused."""
    from bbfft_amd import ragged
    for N in (13, 17, 31, 37, 41, 43, 47, 53, 59, 61, 122):
        for M in (1, 3, 8, 33):
            jobs = [ragged.Job(M, N, 300, -1, 0, 0)]
            kc = ragged.kernel_configuration(jobs, fp)
            vc = ragged.variant_configuration(jobs, 0, fp)
            assert kc["lds_bytes"] <= 32 * 1024 or vc["Kb"] == 1, (N, M)
            assert vc["Kb"] * M * vc["Nt"] * 3 > 256 - M * vc["Nt"] or len(vc["factorization"]) > 1


@pytest.mark.parametrize("fp", [4, 8])
def test_ragged_jobs_of_one_prime_stage(fp):
    """Staged and unstaged single stages in one launch, in place and not."""
    import oracle
    from bbfft_amd import ragged
    jobs = ragged.pack([ragged.Job(1, 17, 70, -1), ragged.Job(4, 31, 9, 1),
                        ragged.Job(1, 41, 5, -1), ragged.Job(3, 12, 30, 1)])
    n = ragged.total_elements(jobs)
    x = oracle.uniform_complex(17, n)
    for in_place in (False, True):
        y = runner.run_ragged(ragged, jobs, x.copy(), n, precision=fp, grid=3, in_place=in_place)
        for j in jobs:
            st = [1, j.M, j.M * j.N]
            s = slice(j.in_offset, j.in_offset + j.elements)
            ref = oracle.fft(1, [j.M, j.N, j.K], st, st, 0, j.direction, x[s])
            assert oracle.rel_l2(y[s], ref) <= oracle.tolerance(fp, j.N), j


def test_ragged_batches_take_every_table_row():
    """A row may carry the load-first loop, which a staged variant has not: 8 columns of 60 points
    fp64 are planned and right."""
    import os
    import oracle
    from bbfft_amd import autotune, ragged
    inc = os.path.join(os.path.dirname(os.path.dirname(bb.__file__)), "tuning", "gfx950.inc")
    rows = [autotune._key(ln) for ln in open(inc) if autotune._key(ln)]
    for prec, typ, N, M in rows:
        if typ in ("c2c", "c2c-ragged") and int(M) < 64:
            ragged.kernel_configuration([ragged.Job(int(M), int(N), 300, -1, 0, 0)],
                                        int(prec[1:]) // 8)
    jobs = ragged.pack([ragged.Job(8, 60, 7, -1), ragged.Job(8, 60, 2, 1)])
    n = ragged.total_elements(jobs)
    x = oracle.uniform_complex(60, n)
    y = runner.run_ragged(ragged, jobs, x.copy(), n, precision=8, grid=3)
    for j in jobs:
        st = [1, j.M, j.M * j.N]
        s = slice(j.in_offset, j.in_offset + j.elements)
        ref = oracle.fft(1, [j.M, j.N, j.K], st, st, 0, j.direction, x[s])
        assert oracle.rel_l2(y[s], ref) <= oracle.tolerance(8, j.N), j


@pytest.mark.parametrize("grid", [1, 2, 7, 255, 256, 257, 3000])
def test_ragged_split_kernel_writes_the_job_table(grid):
    """The kernel that divides a batch's tiles on the device writes the work split of the host's
    job table, with fewer, as many and more work-groups than tiles, and nothing beside it."""
    import ctypes
    from bbfft_amd import ragged
    rng = np.random.default_rng(grid)
    jobs = ragged.pack([ragged.Job(int(rng.integers(1, 4)), int(n), int(k), -1) for n, k in zip(
        rng.choice([16, 60, 105, 128], 9), np.exp(rng.uniform(0, 8, 9)))])
    nj = len(jobs)
    name = ragged.kernel_configuration(jobs)["name"] + "_split"
    tu = ('#include "hip_emu.hpp"\n' + ragged.generate_source(jobs) + "\n"
          'extern "C" int emu_split(unsigned long* table, unsigned long n, unsigned long g) {\n'
          f"  return emu::launch(g / 256 + 1, 256, [&] {{ {name}(table, n, g); }});\n}}\n")
    fn = runner._build_so(tu).emu_split
    fn.argtypes = [ctypes.c_void_p, ctypes.c_ulong, ctypes.c_ulong]
    want = ragged.job_table(jobs, grid=grid)
    recs = want[nj + 1:5 * nj + 1].reshape(nj, 4)
    weight = np.empty(nj)
    for p in range(nj):
        vc = ragged.variant_configuration(jobs, int(recs[p][3]))
        weight[p] = vc["Mb"] * vc["Kb"] * vc["N"]
    cum = np.concatenate([[0.0], np.cumsum(weight * np.diff(want[:nj + 1]))])
    buf = np.full(2 * nj + 1 + len(want) + 4, 77, np.uint64)
    buf[:nj + 1], buf[nj + 1:2 * nj + 1] = cum.view(np.uint64), weight.view(np.uint64)
    buf[2 * nj + 1:7 * nj + 2] = want[:5 * nj + 1]
    assert fn(buf.ctypes.data + 8 * (2 * nj + 1), nj, grid) == 0
    assert np.array_equal(buf[2 * nj + 1:-4], want) and (buf[-4:] == 77).all()


@pytest.mark.parametrize("desc,Nt,radix", [
    ("scfo4.37*100000", 1, 37), ("scfo3.61*50000", 1, 61), ("scfo4.74*40000", 2, 37),
    ("scfo16.122*10000", 2, 61), ("scfo8.509*3000", 32, 509)])
def test_half_input_of_large_primes_keeps_the_tiling_of_its_kernel(desc, Nt, radix):
    """Half-precision input has no matrix sums: its work-items per transform are those of the
    butterflies in registers (one of them per work-item) and of the vector sums."""
    kc = bb.half_input_kernel_configuration(desc, "f16", False)
    assert kc["factorization"][0] == radix and not _flags(kc) & MATRIX
    assert kc["Nt"] == Nt and kc["work_group_size"] <= 512


_NAMES = """
import sys
sys.path.insert(0, sys.argv[1])
import bbfft_amd as bb
for d in sys.argv[2:]:
    desc, _, storage = d.partition("@")
    print(bb.half_input_kernel_configuration(desc, storage.split("-")[0], "mfma" in storage)["name"]
          if storage else bb.kernel_configuration(bb.parse_fft_descriptor(desc))["name"])
"""


def _names(descs, env):
    import os
    import subprocess
    import sys
    pkg = os.path.dirname(os.path.dirname(bb.__file__))
    r = subprocess.run([sys.executable, "-c", _NAMES, pkg, *descs], capture_output=True, text=True,
                       env=dict(os.environ, **env), check=True)
    return r.stdout.split()


def test_table_entries_mean_the_same_compiled_in_and_from_a_file(tmp_path):
    """The compiled-in table read from BBFFT_TUNING_FILE gives the same kernels; a file's own flags
    apply as given, half-precision input included, and `rule` leaves them to the library."""
    import os
    from bbfft_amd import autotune
    inc = os.path.join(os.path.dirname(os.path.dirname(bb.__file__)), "tuning", "gfx950.inc")
    rows = [autotune._key(ln) for ln in open(inc) if autotune._key(ln)]
    descs = []
    for prec, typ, N, M in rows:
        base, *storage = typ.split("-")
        if storage != ["ragged"]:
            d = f"{'s' if prec == 'f32' else 'd'}{'c' if base == 'c2c' else 'r'}" \
                f"{'b' if base == 'c2r' else 'f'}o{M}.{N}"
            descs += [f"{d}*{K}" + ("@" + "-".join(storage) if storage else "")
                      for K in (3, 3000, 300000)]
    table = tmp_path / "copy.inc"
    table.write_text(open(inc).read().split('R"TABLE(', 1)[1].split(')TABLE"', 1)[0])
    assert _names(descs, {}) == _names(descs, {"BBFFT_TUNING_FILE": str(table)})
    table.write_text("f32 c2c-f16 512 4 : 32x16 16 4 1 16 67\n"
                     "f32 c2c 60 8 : 10x6 6 8 4 16 0\n"
                     "f32 c2c 105 8 : 15x7 7 8 2 16 1 4 2\n"
                     "f64 c2c 60 8 : 6x5x2 12 8 2 16 0 rule 2\n")
    half, plain, hints, rule = _names(["scfo4.512*60000@f16", "scfo8.60*30000", "scfo8.105*30000",
                                       "dcfo8.60*30000"], {"BBFFT_TUNING_FILE": str(table)})
    assert half.endswith("_g75") and "_Kb1_" in half
    assert "_g" not in plain and "_f10x6_" in plain
    assert hints.endswith("_g1_w4")
    assert int(rule.split("_g")[1]) & (STAGE_IN | STAGE_OUT) == STAGE_IN | STAGE_OUT


@pytest.mark.parametrize("desc,below,above", [
    ("dcfo3.100", 27900, 28000), ("scfo8.384", 5461, 5462), ("srfo1.512", 65300, 65500),
    ("dcfo8.105", 9980, 10000), ("srbo5.315", 21200, 21350)])
def test_loads_stream_where_input_and_output_outgrow_the_last_level_cache(desc, below, above):
    """256 MB of input and output: the largest data that staged kernels load plainly."""
    def flags(K):
        return _flags(bb.kernel_configuration(bb.parse_fft_descriptor(f"{desc}*{K}")))
    assert flags(below) & (STAGE_IN | 3) == STAGE_IN | 2
    assert flags(above) & (STAGE_IN | 3) == STAGE_IN | 3
    assert flags(below) | 1 == flags(above)


def test_streamed_rows_stream_their_loads_beyond_the_l2(tmp_path):
    table = tmp_path / "rows.inc"
    table.write_text("f32 c2c 60 8 : 10x6 6 8 4 16 0 streamed\nf64 c2c 60 8 : 6x5x2 12 8 2 16 0 rule\n")
    names = _names(["scfo8.60*12000", "scfo8.60*3000", "scfo8.60*60000", "dcfo8.60*6000"],
                   {"BBFFT_TUNING_FILE": str(table)})
    assert [int(n.split("_g")[1]) & 3 for n in names] == [3, 2, 3, 2]
    assert all("_f10x6_" in n for n in names[:3])
    assert _flags(bb.kernel_configuration(bb.parse_fft_descriptor("scfo8.256*1100"))) & 3 == 3


def test_access_by_rule_is_the_default_access_of_a_tiling():
    for desc in ["scfo8.256*32768", "scfo8.256*100", "dcfo3.100*40000", "srfo1.512*65536",
                 "scfo8.509*8192", "srbo5.315*9000"]:
        cfg = bb.parse_fft_descriptor(desc)
        kc = bb.kernel_configuration(cfg)
        tun = dict(factorization=kc["factorization"], Nt=kc["Nt"], Mb=kc["Mb"], Kb=kc["Kb"],
                   lds_pad=kc["lds_pad"], no_pad=kc["lds_pad"] == 0,
                   flags=bb.ACCESS_BY_RULE | (_flags(kc) & MATRIX))
        assert bb.kernel_configuration(cfg, tuning=tun)["name"] == kc["name"], desc
    # an incomplete tiling or one of M tiles has no rule: the hints of a shape without staging
    cfg = bb.parse_fft_descriptor("scfo8.256*32768")
    assert _flags(bb.kernel_configuration(cfg, tuning=dict(flags=bb.ACCESS_BY_RULE))) == 3


def _strided_rows():
    import os
    from bbfft_amd import autotune
    inc = os.path.join(os.path.dirname(os.path.dirname(bb.__file__)), "tuning",
                       "gfx950_strided.inc")
    return [ln for ln in open(inc) if autotune._key(ln)]


@pytest.mark.parametrize("row", _strided_rows())
def test_layouts_without_a_packed_side_have_their_own_entries(row):
    """Padded K-columns, padded rows: the tiling and flags of the row. One packed side: not."""
    (prec, typ, N, M), rhs = row.split(":")[0].split(), row.split("#")[0].split(":")[1].split()
    N, M, t = int(N), int(M), {"c2c": 0, "r2c": 1, "c2r": 2}[typ]
    fac, (Nt, Mb, Kb, pad, flags) = [int(v) for v in rhs[0].split("x")], map(int, rhs[1:6])
    H = N // 2 + 1
    ni, no = (H if t == 2 else N), (H if t == 1 else N)
    for st in ([1, M, M * ni + 1], [1, M, M * no + M]), ([1, M + 2, (M + 2) * ni],
                                                       [1, M + 1, (M + 1) * no]):
        kc = bb.kernel_configuration(_cfg(M, N, 5000, 4 if prec == "f32" else 8,
                                          1 if t == 2 else -1, t, *st))
        assert (kc["factorization"], kc["Nt"], kc["Mb"], kc["Kb"], kc["lds_pad"], _flags(kc)) == \
            (fac, Nt, Mb, Kb, pad, flags)
    kc = bb.kernel_configuration(_cfg(M, N, 5000, 4 if prec == "f32" else 8, 1 if t == 2 else -1, t,
                                      istride=[1, M, M * ni + M]))
    assert _flags(kc) & (STAGE_OUT | PER_TILE_IDS)


@pytest.mark.parametrize("M,N,K,fp,t,pad,Mb", [
    (6, 363, 6000, 8, 0, 1, 6), (16, 128, 1200, 4, 0, 1, 16), (8, 300, 138, 4, 0, 8, 8),
    (5, 500, 209, 8, 0, 0, 5), (10, 384, 142, 4, 0, 0, 10), (57, 64, 26, 8, 0, 0, 57),
    (36, 243, 4, 4, 1, 0, 18), (31, 512, 31, 4, 2, 0, 16)])
def test_m_tiles_only_where_a_tile_does_not_hold_all_columns(M, N, K, fp, t, pad, Mb):
    """Layouts without a packed side and few K-columns keep the default tiling and its streamed
    accesses where that tile holds all M columns; so do real transforms of few K-columns."""
    H = N // 2 + 1
    cfg = _cfg(M, N, K, fp, 1 if t == 2 else -1, t, *(
        ([1, M, M * N + pad], [1, M, M * (H if t == 1 else N) + pad]) if pad else ()))
    kc = bb.kernel_configuration(cfg)
    assert kc["Mb"] == Mb and _flags(kc) == 3
    general = bb.kernel_configuration(cfg, tuning=dict(factorization=kc["factorization"]))
    assert kc["name"] == general["name"]


def test_half_input_stages_long_rows_of_large_data_only():
    """Output rows of 32 bytes and more are staged from 0.9 GB on (radices to 32), with two
    K-columns a tile where one is a single wave; shorter rows beyond the L2."""
    def conf(desc):
        kc = bb.half_input_kernel_configuration(desc, "f16", False)
        return bool(_flags(kc) & STAGE_OUT), kc["Kb"]
    assert conf("scfo4.512*16384") == (False, 1) and conf("scfo4.512*65536") == (True, 2)
    assert conf("scfo16.122*60000")[0] is False and conf("scfo3.61*50000")[0] is True
    assert conf("scfo3.61*2000")[0] is False


@pytest.mark.parametrize("desc,stages", [("dcfo3.96*70000", 2), ("dcfo3.100*3000", 2),
                                         ("dcfo1.384*40000", 3), ("dcfo5.500*3000", 3),
                                         ("drfo3.500*3000", 3)])
def test_fp64_transforms_take_no_stage_for_a_rounding(desc, stages):
    """c2c of two stages and any length of three keep the fewest stages in double precision."""
    assert len(bb.kernel_configuration(bb.parse_fft_descriptor(desc))["factorization"]) == stages


@pytest.mark.parametrize("M,N,fp,staged", [(9, 256, 8, False), (14, 243, 8, False),
                                           (48, 128, 4, False), (8, 256, 8, True),
                                           (12, 384, 8, True), (20, 315, 4, True)])
def test_large_c2c_tiles_keep_streamed_accesses(M, N, fp, staged):
    """Tiles of 36 KB and more are staged only where the default tile splits the columns."""
    kc = bb.kernel_configuration(_cfg(M, N, (1 << 28) // (M * N * 16), fp, -1, 0))
    assert bool(_flags(kc) & STAGE_IN) == staged
    if not staged:
        assert kc["Mb"] == M and _flags(kc) == 3


def test_m_tiles_split_for_few_k_columns_and_aligned_real_rows():
    kc = bb.kernel_configuration(_cfg(39, 315, 20, 8, -1, 0, [1, 40, 40 * 315], [1, 40, 40 * 315]))
    assert kc["Mb"] == 6  # 7 x 20 work-groups
    kc = bb.kernel_configuration(_cfg(32, 256, 20, 8, -1, 0, [1, 40, 40 * 256], [1, 40, 40 * 256]))
    assert kc["Mb"] == 4  # 64-byte segments
    for M, flags in ((32960, 3), (32961, 1536)):
        kc = bb.kernel_configuration(_cfg(M, 8, 127, 4, 1, 2))
        assert kc["Mb"] == 64 and _flags(kc) == flags


@pytest.mark.parametrize("desc,storage", [("scfo8.256*32768", ""), ("scfo8.509*8192", ""),
                                          ("dcfo3.100*40000", ""), ("srbo5.315*9000", ""),
                                          ("scfo4.512*65536", "f16"), ("scfo4.512*65536", "bf16-mfma"),
                                          ("scfo3.61*50000", "f16")])
def test_autotuner_starts_from_the_default_plan(desc, storage):
    """The tuner's first candidate, written as a row, is the kernel of the plan without a tuning;
    a hint row writes its flags and occupancy as they are."""
    from bbfft_amd import autotune
    t = autotune.Tuner.__new__(autotune.Tuner)
    t.cfg = bb.parse_fft_descriptor(desc)
    t.variant = bb.half_input_flags(storage.split("-")[0], "mfma" in storage) if storage else 0
    first = t.default_tuning()
    want = bb.half_input_kernel_configuration(t.cfg, *t.storage())["name"] if storage else \
        bb.kernel_configuration(t.cfg)["name"]
    assert bb.kernel_configuration(t.cfg, tuning=first)["name"].split("_w")[0] == want
    line = autotune.table_line(t.cfg, first, 1.0, 1.0, 1e9, desc)
    rhs = line.split("#")[0].split(":")[1].split()
    assert rhs[6] == "rule" and int(rhs[5]) == (MATRIX if "509" in desc else 0)
    line = autotune.table_line(t.cfg, dict(first, flags=2 | t.variant, waves_per_eu=5), 1.0, 0.5,
                               1e9, desc)
    assert line.split("#")[0].split(":")[1].split()[5:] == ["2", "5"]


@pytest.mark.parametrize("desc", ["scfo8.256", "srfo8.128", "dcfo3.100", "scfo5.315", "srfo1.512",
                                  "scfo17.363", "scfo8.509", "drbo8.256", "dcfo32x32",
                                  "srfo96x96x80"])
def test_archives_serve_any_batch_count(desc):
    """The descriptors an archive is made from hold the kernels of every batch count from 64 on,
    whichever count was named; tested at counts between those that were looked at."""
    import random
    from bbfft_amd import aot
    rng = random.Random(desc)
    d = aot.batch_descriptors(f"{desc}*{rng.randint(64, 10000)}")
    held = {n for b in d for n in aot.kernel_names(b)}
    assert len(d) <= 12 and d == list(dict.fromkeys(d))
    cfg = bb.parse_fft_descriptor(desc)
    most = (200 << 30) // (4 * int(cfg.fp) * int(np.prod(cfg.shape[:cfg.dim + 1])))
    for _ in range(200):
        K = int(round(np.exp(rng.uniform(np.log(64), np.log(max(65, most))))))
        assert set(aot.kernel_names(f"{desc}*{K}")) <= held, K
    assert aot.batch_descriptors(desc + "*5")[0] == desc + "*5"


def _race(cfg, tun, K, fp, t, drop=None, grid=2):
    kc = bb.kernel_configuration(cfg, tuning=tun)
    src = bb.generate_source(cfg, tuning=tun)
    if drop is not None:  # a planted mistake: barrier number `drop` of the kernel's tile taken out
        at = [i for i in range(len(src)) if src.startswith("__syncthreads();", i)][drop]
        src = src[:at] + src[at + len("__syncthreads();"):]
    rt, ct = ("float", "float2") if fp == 4 else ("double", "double2")
    call = (f'{kc["name"]}((const {rt if t == 1 else ct}*)in, ({rt if t == 2 else ct}*)out, '
            f'{K}ul)')
    M, N = cfg.shape[:2]
    H = N // 2 + 1
    n_in, n_out = M * (H if t == 2 else N) * K, M * (H if t == 1 else N) * K
    return runner.race_check(src, call, n_in * fp * (1 if t == 1 else 2),
                             n_out * fp * (1 if t == 2 else 2), grid, kc["work_group_size"])


@pytest.mark.skipif(not runner.have_tsan(), reason="no ThreadSanitizer runtime")
@pytest.mark.parametrize("flags", [PER_TILE_IDS | MATRIX,
                                   PER_TILE_IDS | MATRIX | STAGE_IN | STAGE_OUT,
                                   PER_TILE_IDS])  # and the vector sums
@pytest.mark.parametrize("M,N,K,fp,t,d,fac,Nt,Kb", [
    (2, 67, 7, 4, 0, -1, [67], 32, 2), (2, 134, 3, 8, 0, 1, [67, 2], 64, 1),
    (2, 134, 3, 8, 0, 1, [2, 67], 64, 1), (1, 134, 5, 4, 1, -1, [67], 64, 2),
    (2, 67, 5, 4, 2, 1, [67], 32, 1)])
def test_direct_stages_are_race_free(M, N, K, fp, t, d, fac, Nt, Kb, flags):
    """Several waves and tiles per work-group; matrix instructions order nothing but a wave's
    operands."""
    tun = dict(factorization=fac, Nt=Nt, Mb=M, Kb=Kb, no_pad=True, flags=flags)
    ok, report = _race(_cfg(M, N, K, fp, d, t), tun, K, fp, t)
    assert ok, report[-3000:]


@pytest.mark.skipif(not runner.have_tsan(), reason="no ThreadSanitizer runtime")
@pytest.mark.parametrize("drop", range(4))
def test_race_check_sees_barriers_around_matrix_sums(drop):
    """[2, 67]: stage 2's exchange, phase 1's slots, the sums' reads, the tile's end."""
    cfg = _cfg(2, 134, 5, 4, -1, 0)
    tun = dict(factorization=[2, 67], Nt=64, Mb=2, Kb=1, no_pad=True,
               flags=PER_TILE_IDS | MATRIX | STAGE_OUT)
    assert _race(cfg, tun, 5, 4, 0)[0]
    ok, report = _race(cfg, tun, 5, 4, 0, drop=drop)
    assert not ok and "ThreadSanitizer" in report


@pytest.mark.parametrize("M,N,fp,t", [(22, 205, 8, 0), (23, 82, 8, 0), (21, 410, 8, 2),
                                      (8, 287, 4, 0), (14, 188, 4, 0), (4, 58, 4, 0),
                                      (1, 87, 8, 1), (6, 473, 4, 0)])
def test_wide_prime_radices_keep_one_butterfly_per_work_item(M, N, fp, t):
    """Prime radices above 23 in registers: as many work-items as the stage has butterflies, in
    groups whose waves leave each the registers it needs."""
    for K in (20, 300, 5000):
        kc = bb.kernel_configuration(_cfg(M, N, K, fp, 1 if t == 2 else -1, t))
        if _flags(kc) & MATRIX:
            continue
        n = N // 2 if t and N % 2 == 0 else N
        assert kc["Nt"] == n // max(kc["factorization"])
        waves = -(-kc["work_group_size"] // 64)
        assert (36 + fp // 2 * max(kc["factorization"])) * -(-waves // 4) <= 512
