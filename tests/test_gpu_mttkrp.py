"""GPU MTTKRP parity against the oracle's brute-force COO MTTKRP (long
double accumulation, the reference's own known-answer procedure,
tests/mttkrp_test.c:36-88).

Tolerances (normwise relative, ||got - ref||_F / ||ref||_F):
  FP64 path 1e-12, FP32 path 1e-5  -- as stated for this path.
Covered: every mode of every allocation scheme (root, internal and leaf
kernels; internal and leaf outputs both over row-sorted copies and by the
CSF walk with atomics), 3- to 8-mode tensors, tiled tensors, ranks that exercise every
lane layout (1, 3, 8, 16, 32, 64, 100), Zipf-skewed tensors whose heavy
slices span many work items, the device-pointer entry point, and at a
larger size the mode-independence of <X, [[A_1..A_N]]> = sum(M_m * A_m).
"""
import ctypes

import numpy as np
import pytest

from conftest import DATASETS, tensor_path
import oracle_py as orc
import pysplatt as ps

pytestmark = pytest.mark.gpu

TOL64 = 1e-12
TOL32 = 1e-5
DEFAULT = (1 << 64) - 1          # the dispatch limits' setters: back to the default


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - np.asarray(b, np.float64))
                 / max(np.linalg.norm(np.asarray(b, np.float64)), 1e-300))


def _set_precision(p):
    assert ps.lib().splatt_amd_set_mttkrp_precision(p) == ps.SUCCESS


def _set_layout(x):
    assert ps.lib().splatt_amd_set_mttkrp_layout(x) == ps.SUCCESS


@pytest.fixture(autouse=True)
def _reset_precision():
    yield
    ps.lib().splatt_amd_set_mttkrp_precision(ps.F64)
    ps.lib().splatt_amd_set_mttkrp_layout(ps.LAYOUT_AUTO)


@pytest.mark.parametrize("name", DATASETS)
@pytest.mark.parametrize("kind", [ps.CSF_ONEMODE, ps.CSF_TWOMODE, ps.CSF_ALLMODE])
@pytest.mark.parametrize("layout", [ps.LAYOUT_AUTO, ps.LAYOUT_CSF])
def test_fixtures_fp64(gpu_available, name, kind, layout):
    print("case", name, kind, layout, flush=True)
    _set_layout(layout)
    coo = orc.Coo.read(tensor_path(name))
    s = ps.CsfSet.convert(coo.inds(), coo.vals(), ps.Opts(csf_alloc=kind))
    mats = [ps.synth_matrix(d, 16, 100 + m) for m, d in enumerate(coo.dims)]
    for mode in range(coo.nmodes):
        assert rel(s.mttkrp(mode, mats), orc.mttkrp_coo(coo, mats, mode)) <= TOL64


@pytest.mark.parametrize("name", ["med.tns", "med4.tns", "med5.tns"])
@pytest.mark.parametrize("layout", [ps.LAYOUT_AUTO, ps.LAYOUT_CSF])
def test_fixtures_fp32(gpu_available, name, layout):
    print("case fp32", name, layout, flush=True)
    _set_layout(layout)
    coo = orc.Coo.read(tensor_path(name))
    s = ps.CsfSet.convert(coo.inds(), coo.vals(), ps.Opts(csf_alloc=ps.CSF_ONEMODE))
    mats = [ps.synth_matrix(d, 32, 200 + m).astype(np.float32) for m, d in enumerate(coo.dims)]
    _set_precision(ps.F32)
    for mode in range(coo.nmodes):
        got = s.mttkrp(mode, [m.astype(np.float64) for m in mats])
        assert rel(got, orc.mttkrp_coo(coo, mats, mode, f32=True)) <= TOL32


@pytest.mark.parametrize("R", [1, 3, 8, 16, 32, 64, 100])
@pytest.mark.parametrize("prec", [ps.F64, ps.F32])
@pytest.mark.parametrize("layout", [ps.LAYOUT_AUTO, ps.LAYOUT_CSF])
def test_ranks_and_layouts(gpu_available, R, prec, layout):
    print("case rank", R, prec, layout, flush=True)
    _set_layout(layout)
    inds, vals, dims = ps.synth_coord([300, 200, 100], 30000, zipf=[1.2, 1.1, 0.0],
                                      vals="lognormal", seed=R)
    coo = orc.Coo.from_arrays(inds, vals, dims)
    s = ps.CsfSet.convert(inds, vals, ps.Opts(csf_alloc=ps.CSF_ONEMODE))
    mats = [ps.synth_matrix(d, R, 7 + m) for m, d in enumerate(dims)]
    _set_precision(prec)
    for mode in range(3):
        got = s.mttkrp(mode, mats)
        if prec == ps.F64:
            assert rel(got, orc.mttkrp_coo(coo, mats, mode)) <= TOL64
        else:
            m32 = [m.astype(np.float32) for m in mats]
            assert rel(got, orc.mttkrp_coo(coo, m32, mode, f32=True)) <= TOL32


@pytest.mark.parametrize("nmodes", [4, 5, 6, 8])
@pytest.mark.parametrize("layout", [ps.LAYOUT_AUTO, ps.LAYOUT_CSF])
def test_higher_order(gpu_available, nmodes, layout):
    print("case nmodes", nmodes, layout, flush=True)
    _set_layout(layout)
    dims = [40, 30, 20, 12, 9, 7, 5, 4][:nmodes]
    inds, vals, d2 = ps.synth_coord(dims, 40000, zipf=[1.1] * nmodes, seed=nmodes)
    coo = orc.Coo.from_arrays(inds, vals, d2)
    mats = [ps.synth_matrix(d, 8, 30 + m) for m, d in enumerate(d2)]
    for kind in (ps.CSF_ONEMODE, ps.CSF_TWOMODE, ps.CSF_ALLMODE):
        s = ps.CsfSet.convert(inds, vals, ps.Opts(csf_alloc=kind))
        for mode in range(nmodes):
            assert rel(s.mttkrp(mode, mats), orc.mttkrp_coo(coo, mats, mode)) <= TOL64


@pytest.mark.parametrize("tilelevel", [1, 2])
def test_tiled(gpu_available, tilelevel):
    coo = orc.Coo.read(tensor_path("med4.tns"))
    opts = ps.Opts(csf_alloc=ps.CSF_TWOMODE, tile=ps.DENSETILE, tilelevel=tilelevel,
                   nthreads=5)
    s = ps.CsfSet.convert(coo.inds(), coo.vals(), opts)
    mats = [ps.synth_matrix(d, 16, 40 + m) for m, d in enumerate(coo.dims)]
    for mode in range(4):
        assert rel(s.mttkrp(mode, mats), orc.mttkrp_coo(coo, mats, mode)) <= TOL64


@pytest.mark.parametrize("layout", [ps.LAYOUT_AUTO, ps.LAYOUT_CSF])
def test_heavy_zipf_slices(gpu_available, layout):
    _set_layout(layout)
    # a few slices hold most nonzeros, so they span many work items and are
    # completed through the partial (atomic) flushes
    inds, vals, dims = ps.synth_coord([2000, 1500, 1000], 1000000, zipf=[1.6, 1.6, 1.6],
                                      vals="lognormal", seed=3)
    coo = orc.Coo.from_arrays(inds, vals, dims)
    mats = [ps.synth_matrix(d, 32, 50 + m) for m, d in enumerate(dims)]
    for kind in (ps.CSF_ONEMODE, ps.CSF_ALLMODE):
        s = ps.CsfSet.convert(inds, vals, ps.Opts(csf_alloc=kind))
        for mode in range(3):
            assert rel(s.mttkrp(mode, mats), orc.mttkrp_coo(coo, mats, mode)) <= TOL64


def _edge_tensor(seed):
    """A 3-mode tensor whose mode-0 slices have lengths around the kernels'
    work-item (32 nonzeros), wave (256) and block (1024) edges, long slices
    spanning many waves next to runs of one-nonzero slices, and fibers of
    1 to 40 nonzeros: every path of the partial-slice combines (one slice per
    wave or block, several slices, empty items) and of the carry fix-up."""
    rng = np.random.default_rng(seed)
    pattern = [1, 31, 32, 33, 1, 1, 255, 256, 257, 2, 511, 512, 513, 1023, 1024, 1025,
               7, 1, 20000, 3, 1, 1, 1, 64, 96, 300, 1, 45000, 5, 129]
    flen = [1, 2, 7, 31, 33, 40, 3, 1, 1]
    D1, D2 = 4999, 3001
    i0, i1, i2 = [], [], []
    s = 0
    for rep in range(3):
        for L in pattern:
            f = 0
            left = L
            while left > 0:
                n = min(left, flen[(s + f) % len(flen)])
                j = (f * 37 + s) % D1
                ks = (np.arange(n) * 17 + f + s) % D2
                i0.append(np.full(n, s, np.uint64))
                i1.append(np.full(n, j, np.uint64))
                i2.append(ks.astype(np.uint64))
                left -= n
                f += 1
            s += 1
    inds = [np.concatenate(i0), np.concatenate(i1), np.concatenate(i2)]
    # no empty index in any mode (an untiled CSF's root rows are then its
    # slice positions, as in the reference)
    dims = [s]
    for m in (1, 2):
        used, inds[m] = np.unique(inds[m], return_inverse=True)
        inds[m] = inds[m].astype(np.uint64)
        dims.append(len(used))
    vals = rng.lognormal(0.0, 1.0, len(inds[0]))
    perm = rng.permutation(len(vals))
    return [a[perm] for a in inds], vals[perm], dims


@pytest.mark.parametrize("prec", [ps.F64, ps.F32])
@pytest.mark.parametrize("layout", [ps.LAYOUT_AUTO, ps.LAYOUT_CSF])
def test_slice_edges(gpu_available, prec, layout):
    print("case slice edges", prec, layout, flush=True)
    inds, vals, dims = _edge_tensor(11)
    coo = orc.Coo.from_arrays(inds, vals, dims)
    mats = [ps.synth_matrix(d, 32, 70 + m) for m, d in enumerate(dims)]
    m32 = [m.astype(np.float32) for m in mats]
    _set_precision(prec)
    _set_layout(layout)
    for kind in (ps.CSF_ONEMODE, ps.CSF_TWOMODE, ps.CSF_ALLMODE):
        s = ps.CsfSet.convert(inds, vals, ps.Opts(csf_alloc=kind))
        try:
            for mode in range(3):
                got = s.mttkrp(mode, mats)
                if prec == ps.F64:
                    assert rel(got, orc.mttkrp_coo(coo, mats, mode)) <= TOL64, (kind, mode)
                else:
                    assert rel(got, orc.mttkrp_coo(coo, m32, mode, f32=True)) <= TOL32, (kind, mode)
        finally:
            s.free()


def test_slice_edges_two_level_fixup(gpu_available):
    # the carry fix-up's two-pass form (taken by long carry buffers, from
    # 65536 entries) forced on every size
    L = ps.lib()
    L.spd_mttkrp_set_fix_two_level.argtypes = [ctypes.c_uint64]
    assert L.spd_mttkrp_set_fix_two_level(0) == 0
    try:
        for prec in (ps.F64, ps.F32):
            test_slice_edges(gpu_available, prec, ps.LAYOUT_AUTO)
        _set_precision(ps.F64)
        test_heavy_zipf_slices(gpu_available, ps.LAYOUT_AUTO)
    finally:
        L.spd_mttkrp_set_fix_two_level(DEFAULT)
        _set_precision(ps.F64)
        _set_layout(ps.LAYOUT_AUTO)


def test_device_entry_point(gpu_available):
    inds, vals, dims = ps.synth_coord([500, 400, 300], 50000, zipf=[1.2] * 3, seed=9)
    coo = orc.Coo.from_arrays(inds, vals, dims)
    opts = ps.Opts(csf_alloc=ps.CSF_ALLMODE)
    s = ps.CsfSet.convert(inds, vals, opts)
    R = 32
    mats = [ps.synth_matrix(d, R, 60 + m) for m, d in enumerate(dims)]
    L = ps.lib()
    for prec, dt in ((ps.F64, np.float64), (ps.F32, np.float32)):
        dm = [ps.DevBuf.from_host(m.astype(dt)) for m in mats]
        arr = (ctypes.c_void_p * 3)(*[b.ptr for b in dm])
        for mode in range(3):
            out = ps.DevBuf(dims[mode] * R * np.dtype(dt).itemsize)
            assert L.splatt_amd_mttkrp_dev(mode, R, s.ptr, arr, out.ptr, prec, opts.ptr,
                                           None) == ps.SUCCESS
            assert L.splatt_amd_sync() == ps.SUCCESS
            got = out.to_host((dims[mode], R), dt)
            if prec == ps.F64:
                assert rel(got, orc.mttkrp_coo(coo, mats, mode)) <= TOL64
            else:
                m32 = [m.astype(np.float32) for m in mats]
                assert rel(got, orc.mttkrp_coo(coo, m32, mode, f32=True)) <= TOL32


def test_inner_product_is_mode_independent(gpu_available):
    # <X, [[A_1,...,A_N]]> = sum_i sum_r M_m[i,r] A_m[i,r] for every mode m
    inds, vals, dims = ps.synth_coord([20000, 15000, 5000], 5000000, zipf=[1.2] * 3,
                                      vals="lognormal", seed=12)
    s = ps.CsfSet.convert(inds, vals, ps.Opts(csf_alloc=ps.CSF_ONEMODE))
    mats = [ps.synth_matrix(d, 16, 70 + m) for m, d in enumerate(dims)]
    inner = [float(np.sum(s.mttkrp(m, mats) * mats[m])) for m in range(3)]
    scale = float(np.sum(np.abs(vals))) * 1.0
    assert max(inner) - min(inner) <= 1e-10 * scale
    # linearity in the values
    s2 = ps.CsfSet.convert(inds, 2.0 * vals, ps.Opts(csf_alloc=ps.CSF_ONEMODE))
    assert rel(s2.mttkrp(0, mats), 2.0 * s.mttkrp(0, mats)) <= 1e-14


def _hip():
    h = ctypes.CDLL("libamdhip64.so")
    h.hipStreamCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
    h.hipStreamDestroy.argtypes = [ctypes.c_void_p]
    h.hipStreamSynchronize.argtypes = [ctypes.c_void_p]
    return h


def test_device_entry_point_two_caller_streams(gpu_available):
    # splatt_amd_mttkrp_dev returns without synchronising and accepts any
    # stream: back-to-back calls on two caller streams (no wait between
    # them) must not share partial-row buffers. Both results against the
    # oracle, for every mode of an all-mode CSF (each a root output with
    # carried partial rows), FP32 and FP64.
    inds, vals, dims = ps.synth_coord([3000, 2500, 2000], 400000, zipf=[1.2] * 3, seed=91)
    coo = orc.Coo.from_arrays(inds, vals, dims)
    opts = ps.Opts(csf_alloc=ps.CSF_ALLMODE)
    s = ps.CsfSet.convert(inds, vals, opts)
    R = 32
    sets = [[ps.synth_matrix(d, R, 300 + 10 * k + m) for m, d in enumerate(dims)]
            for k in range(2)]
    L = ps.lib()
    h = _hip()
    streams = [ctypes.c_void_p(), ctypes.c_void_p()]
    for st in streams:
        assert h.hipStreamCreate(ctypes.byref(st)) == 0
    try:
        for prec, dt in ((ps.F64, np.float64), (ps.F32, np.float32)):
            dms = [[ps.DevBuf.from_host(m.astype(dt)) for m in mats] for mats in sets]
            arrs = [(ctypes.c_void_p * 3)(*[b.ptr for b in dm]) for dm in dms]
            for mode in range(3):
                outs = [ps.DevBuf(dims[mode] * R * np.dtype(dt).itemsize) for _ in range(2)]
                for k in range(2):
                    assert L.splatt_amd_mttkrp_dev(mode, R, s.ptr, arrs[k], outs[k].ptr, prec,
                                                   opts.ptr, streams[k]) == ps.SUCCESS
                for st in streams:
                    assert h.hipStreamSynchronize(st) == 0
                for k in range(2):
                    got = outs[k].to_host((dims[mode], R), dt)
                    if prec == ps.F64:
                        assert rel(got, orc.mttkrp_coo(coo, sets[k], mode)) <= TOL64
                    else:
                        m32 = [m.astype(np.float32) for m in sets[k]]
                        assert rel(got, orc.mttkrp_coo(coo, m32, mode, f32=True)) <= TOL32
    finally:
        for st in streams:
            h.hipStreamDestroy(st)


@pytest.mark.parametrize("R", [16, 32, 48, 64, 100])
@pytest.mark.parametrize("prec", [ps.F64, ps.F32])
def test_root_kernel_variants(gpu_available, R, prec):
    # every 3-mode root kernel variant against the oracle and against the
    # default (per-nonzero k_root3): 1 the persistent kernel with hot leaf
    # rows in LDS (one A gather per fiber, runs carried across a wave's
    # chunks), 2 the same with every row from HBM, 3 k_root3 with one A
    # gather per fiber. Untiled all-mode CSF (root rows are slice positions)
    # and a tiled one (root ids stored). Zipf(1.5) roots give slices that
    # span many waves; at R=64 FP64 only 64 hot rows fit in LDS, so
    # hotter-ranked rows beyond them are read from HBM through the rank table.
    print("case root variants", R, prec, flush=True)
    inds, vals, dims = ps.synth_coord([4000, 3000, 2000], 600000, zipf=[1.5, 1.3, 1.2],
                                      vals="lognormal", seed=17 + R)
    coo = orc.Coo.from_arrays(inds, vals, dims)
    mats = [ps.synth_matrix(d, R, 900 + m) for m, d in enumerate(dims)]
    m32 = [m.astype(np.float32) for m in mats]
    L = ps.lib()
    _set_precision(prec)
    for opts in (ps.Opts(csf_alloc=ps.CSF_ALLMODE),
                 ps.Opts(csf_alloc=ps.CSF_ALLMODE, tile=ps.DENSETILE, tilelevel=1, nthreads=4)):
        s = ps.CsfSet.convert(inds, vals, opts)
        try:
            for mode in range(3):
                assert L.spd_mttkrp_set_root_variant(0) == 0
                base = s.mttkrp(mode, mats)
                for v in (1, 2, 3):
                    assert L.spd_mttkrp_set_root_variant(v) == 0
                    got = s.mttkrp(mode, mats)
                    if prec == ps.F64:
                        assert rel(got, orc.mttkrp_coo(coo, mats, mode)) <= TOL64, (mode, v)
                        assert rel(got, base) <= TOL64, (mode, v)
                    else:
                        assert rel(got, orc.mttkrp_coo(coo, m32, mode, f32=True)) <= TOL32, (mode, v)
                        assert rel(got, base) <= TOL32, (mode, v)
        finally:
            L.spd_mttkrp_set_root_variant(0)
            s.free()


@pytest.mark.parametrize("R", [2, 4, 5, 6, 7, 9, 10, 13, 31, 33, 35, 63, 65, 67, 70])
@pytest.mark.parametrize("prec", [ps.F64, ps.F32])
@pytest.mark.parametrize("layout", [ps.LAYOUT_AUTO, ps.LAYOUT_CSF])
def test_ranks_off_the_vector_width(gpu_available, R, prec, layout):
    # ranks that are no multiple of a lane's columns: the last lane's columns
    # overlap the lane's before it (stores and additions, one and two column
    # tiles, root, internal and leaf outputs), and nothing is written past
    # the last row
    print("case odd rank", R, prec, layout, flush=True)
    _set_layout(layout)
    L = ps.lib()
    dt = np.float32 if prec == ps.F32 else np.float64
    for dims, zipf in (([90, 70, 50], [1.2, 1.1, 0.0]), ([40, 30, 20, 12], [1.2, 0.0, 1.1, 0.0])):
        inds, vals, dims = ps.synth_coord(dims, 6000, zipf=zipf, vals="lognormal", seed=R)
        opts = ps.Opts(csf_alloc=ps.CSF_ONEMODE)
        s = ps.CsfSet.convert(inds, vals, opts)
        coo = orc.Coo.from_arrays(inds, vals, dims)
        mats = [ps.synth_matrix(d, R, 60 + m).astype(dt) for m, d in enumerate(dims)]
        bufs = [ps.DevBuf.from_host(m) for m in mats]
        arr = (ctypes.c_void_p * len(bufs))(*[b.ptr for b in bufs])
        for mode, d in enumerate(dims):
            out = ps.DevBuf.from_host(np.full((d + 2, R), 3.5, dtype=dt))
            assert L.splatt_amd_mttkrp_dev(mode, R, s.ptr, arr, out.ptr, prec, opts.ptr,
                                           None) == ps.SUCCESS
            got = out.to_host((d + 2, R), dt)
            assert np.all(got[d:] == 3.5)
            want = orc.mttkrp_coo(coo, mats, mode, f32=(prec == ps.F32))
            assert rel(got[:d], want) <= (TOL32 if prec == ps.F32 else TOL64)


@pytest.mark.parametrize("small", [0, 1 << 40])
@pytest.mark.parametrize("prec", [ps.F64, ps.F32])
def test_slice_edges_by_wave_size(gpu_available, small, prec):
    # both sizes of the 3-mode root kernel's waves (256 nonzeros, and the 64
    # of small tensors) forced on the slice-edge tensor and on ranks of every
    # lane count, with nonzeros that end inside a wave
    L = ps.lib()
    L.spd_mttkrp_set_root_small.argtypes = [ctypes.c_uint64]
    assert L.spd_mttkrp_set_root_small(small) == 0
    try:
        test_slice_edges(gpu_available, prec, ps.LAYOUT_AUTO)
        for R in (2, 5, 10, 16, 35, 64, 100):
            inds, vals, dims = ps.synth_coord([70, 60, 50], 1000 + 37 * R, zipf=[1.1, 1.2, 0.0],
                                              vals="lognormal", seed=R)
            coo = orc.Coo.from_arrays(inds, vals, dims)
            mats = [ps.synth_matrix(d, R, 90 + m) for m, d in enumerate(dims)]
            m32 = [m.astype(np.float32) for m in mats]
            s = ps.CsfSet.convert(inds, vals, ps.Opts(csf_alloc=ps.CSF_ALLMODE))
            for mode in range(3):
                got = s.mttkrp(mode, mats)
                if prec == ps.F64:
                    assert rel(got, orc.mttkrp_coo(coo, mats, mode)) <= TOL64, (R, mode)
                else:
                    assert rel(got, orc.mttkrp_coo(coo, m32, mode, f32=True)) <= TOL32, (R, mode)
        # the tree walks: roots and row-sorted copies of 4 and 5 modes
        for dims, R in (([60, 40, 30, 20], 16), ([60, 40, 30, 20], 35), ([50, 20, 30, 9, 12], 8)):
            inds, vals, dims = ps.synth_coord(dims, 7001, zipf=[1.1] + [0.0] * (len(dims) - 1),
                                              vals="lognormal", seed=R)
            coo = orc.Coo.from_arrays(inds, vals, dims)
            mats = [ps.synth_matrix(d, R, 20 + m) for m, d in enumerate(dims)]
            m32 = [m.astype(np.float32) for m in mats]
            for kind in (ps.CSF_ONEMODE, ps.CSF_ALLMODE):
                s = ps.CsfSet.convert(inds, vals, ps.Opts(csf_alloc=kind))
                for mode in range(len(dims)):
                    got = s.mttkrp(mode, mats)
                    if prec == ps.F64:
                        assert rel(got, orc.mttkrp_coo(coo, mats, mode)) <= TOL64, (dims, mode)
                    else:
                        assert rel(got, orc.mttkrp_coo(coo, m32, mode, f32=True)) <= TOL32, (dims, mode)
    finally:
        L.spd_mttkrp_set_root_small(DEFAULT)


@pytest.mark.parametrize("R", [4, 7, 8, 16, 40])
@pytest.mark.parametrize("prec", [ps.F64, ps.F32])
def test_short_slices_and_empty_rows(gpu_available, R, prec):
    # slices of one to a few nonzeros, so that every wave ends many runs in
    # every group, and outputs written without a fill: all rows in use, and
    # tensors with unused rows at the end of a mode (cleared). The output
    # starts as NaN.
    print("case short slices", R, prec, flush=True)
    L = ps.lib()
    dt = np.float32 if prec == ps.F32 else np.float64
    rng = np.random.default_rng(R)
    n = 3001
    i = np.sort(rng.integers(0, 1500, n))
    i = np.unique(i, return_inverse=True)[1]
    j = (np.arange(n) * 7) % 611
    for extra in (0, 5):
        inds = [i.astype(np.uint64), j.astype(np.uint64), (np.arange(n) % 1000).astype(np.uint64)]
        vals = rng.lognormal(0.0, 1.0, n)
        if extra:
            inds[1] = inds[1] + 0
            inds[1][-1] = 611 + extra          # rows 611 .. of mode 1 stay empty
        dims = [int(x.max()) + 1 for x in inds]
        coo = orc.Coo.from_arrays(inds, vals, dims)
        mats = [ps.synth_matrix(d, R, 30 + m).astype(dt) for m, d in enumerate(dims)]
        bufs = [ps.DevBuf.from_host(m) for m in mats]
        arr = (ctypes.c_void_p * 3)(*[b.ptr for b in bufs])
        for kind in (ps.CSF_ONEMODE, ps.CSF_ALLMODE):
            opts = ps.Opts(csf_alloc=kind)
            s = ps.CsfSet.convert(inds, vals, opts)
            dims_in = [int(s.ptr[0].dims[m]) for m in range(3)]
            assert dims_in == dims
            for mode in range(3):
                # an untiled root with empty rows writes slice positions
                depth0 = int(s.ptr[mode if kind == ps.CSF_ALLMODE else 0].dim_perm[0])
                if extra and depth0 == 1:
                    continue
                out = ps.DevBuf.from_host(np.full((dims[mode], R), np.nan, dtype=dt))
                assert L.splatt_amd_mttkrp_dev(mode, R, s.ptr, arr, out.ptr, prec, opts.ptr,
                                               None) == ps.SUCCESS
                got = out.to_host((dims[mode], R), dt)
                want = orc.mttkrp_coo(coo, mats, mode, f32=(prec == ps.F32))
                assert np.all(np.isfinite(got)), (kind, mode)
                assert rel(got, want) <= (TOL32 if prec == ps.F32 else TOL64), (kind, mode)


@pytest.mark.parametrize("hole", [None, 0, 150, 298])
@pytest.mark.parametrize("wave", [64, 256])
def test_copy_outputs_with_and_without_empty_rows(gpu_available, hole, wave):
    # internal and leaf outputs over row-sorted copies: written without a fill
    # when every row occurs; a first, middle or last but one row that does not
    # occur is zero. The output starts as NaN.
    print("case copy rows", hole, wave, flush=True)
    L = ps.lib()
    L.spd_mttkrp_set_root_small.argtypes = [ctypes.c_uint64]
    rng = np.random.default_rng(5)
    n, R = 4001, 12
    dims = [20, 300, 500]
    inds = [(np.arange(n) % 20), rng.permutation(np.arange(n) % 300), (np.arange(n) * 7) % 500]
    if hole is not None:
        for m in (1, 2):
            inds[m] = np.where(inds[m] == hole, hole + 1, inds[m])
    inds = [x.astype(np.uint64) for x in inds]
    vals = rng.lognormal(0.0, 1.0, n)
    coo = orc.Coo.from_arrays(inds, vals, dims)
    mats = [ps.synth_matrix(d, R, 30 + m) for m, d in enumerate(dims)]
    bufs = [ps.DevBuf.from_host(m) for m in mats]
    arr = (ctypes.c_void_p * 3)(*[b.ptr for b in bufs])
    opts = ps.Opts(csf_alloc=ps.CSF_ONEMODE)
    assert L.spd_mttkrp_set_root_small(0 if wave == 256 else 1 << 40) == 0
    try:
        s = ps.CsfSet.convert(inds, vals, opts)
        assert [int(s.ptr[0].dims[m]) for m in range(3)] == dims
        for mode in range(3):
            out = ps.DevBuf.from_host(np.full((dims[mode], R), np.nan))
            assert L.splatt_amd_mttkrp_dev(mode, R, s.ptr, arr, out.ptr, ps.F64, opts.ptr,
                                           None) == ps.SUCCESS
            got = out.to_host((dims[mode], R), np.float64)
            assert np.all(np.isfinite(got)), mode
            assert rel(got, orc.mttkrp_coo(coo, mats, mode)) <= TOL64, mode
        s.free()
    finally:
        L.spd_mttkrp_set_root_small(DEFAULT)


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("wave", [64, 256])
@pytest.mark.parametrize("prec", [ps.F64, ps.F32])
def test_every_output_row_is_written(gpu_available, prec, wave, two_level):
    # outputs start as NaN: root and copy outputs with and without a fill
    # before them, at both wave sizes and both forms of the fix-up. One row of
    # every mode holds a third of the nonzeros (it spans many blocks and is
    # carried), the others a few; untiled with every row in use, and tiled
    # with row ids and rows that do not occur, the root's among them.
    print("case written", prec, wave, two_level, flush=True)
    L = ps.lib()
    L.spd_mttkrp_set_root_small.argtypes = [ctypes.c_uint64]
    L.spd_mttkrp_set_fix_two_level.argtypes = [ctypes.c_uint64]
    dt = np.float32 if prec == ps.F32 else np.float64
    rng = np.random.default_rng(21)
    n, R = 9001, 9
    assert L.spd_mttkrp_set_root_small(0 if wave == 256 else 1 << 40) == 0
    assert L.spd_mttkrp_set_fix_two_level(0 if two_level else DEFAULT) == 0
    try:
        for full in ([701, 499, 302], [401, 299, 102, 53]):
            for tiled in (False, True):
                inds = []
                for m, d in enumerate(full):
                    x = rng.permutation(np.arange(n) % d)
                    x[rng.permutation(n)[:n // 3]] = 7 + m
                    x[:d] = np.arange(d)
                    if tiled:
                        x[x % 10 == 3] = d - 1
                    inds.append(x.astype(np.uint64))
                vals = rng.lognormal(0.0, 1.0, n)
                coo = orc.Coo.from_arrays(inds, vals, full)
                mats = [ps.synth_matrix(d, R, 80 + m).astype(dt) for m, d in enumerate(full)]
                bufs = [ps.DevBuf.from_host(m) for m in mats]
                arr = (ctypes.c_void_p * len(full))(*[b.ptr for b in bufs])
                for kind in (ps.CSF_ONEMODE, ps.CSF_ALLMODE):
                    opts = ps.Opts(csf_alloc=kind, tile=ps.DENSETILE, tilelevel=1, nthreads=5) \
                        if tiled else ps.Opts(csf_alloc=kind)
                    s = ps.CsfSet.convert(inds, vals, opts)
                    assert [int(s.ptr[0].dims[m]) for m in range(len(full))] == full
                    for mode, d in enumerate(full):
                        out = ps.DevBuf.from_host(np.full((d + 1, R), np.nan, dtype=dt))
                        assert L.splatt_amd_mttkrp_dev(mode, R, s.ptr, arr, out.ptr, prec,
                                                       opts.ptr, None) == ps.SUCCESS
                        got = out.to_host((d + 1, R), dt)
                        want = orc.mttkrp_coo(coo, mats, mode, f32=(prec == ps.F32))
                        what = (full, tiled, kind, mode)
                        assert np.all(np.isnan(got[d])), what
                        assert np.all(np.isfinite(got[:d])), what
                        assert rel(got[:d], want) <= (TOL32 if prec == ps.F32 else TOL64), what
                    s.free()
                for b in bufs:
                    b.free()
    finally:
        L.spd_mttkrp_set_root_small(DEFAULT)
        L.spd_mttkrp_set_fix_two_level(DEFAULT)
