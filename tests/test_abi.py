"""CPU tests of the shipped library's C ABI and host logic (no GPU needed):
every symbol include/oxhip.h declares is exported, the eligibility helpers
agree with the oracle's restatement of the reference's rules, declines happen
before any device work, and without a device the library fails loudly instead
of computing anything."""
import ctypes
import os
import re

import numpy as np
import pytest

import oxlibs
from oxidize_amd import _lib, synth
from oxidize_amd import matvec as mv

ROOT = oxlibs.ROOT


def declared_functions():
    names = set()
    for header in ("oxhip.h", "oxhip_lab.h"):
        text = open(os.path.join(ROOT, "include", header)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names.update(re.findall(r"\b((?:oxh|oc)_[a-z0-9_]+)\s*\(", text))
    return sorted(names)


def test_library_exports_every_declared_symbol():
    lib = _lib.lib()
    names = declared_functions()
    assert len(names) >= 40
    for n in names:
        assert hasattr(lib, n), "missing export: " + n
    assert set(_lib.SIGNATURES) == set(names)


def test_no_oracle_or_reference_symbols_in_the_product():
    out = os.popen("nm -D --defined-only %s" % _lib.LIB_PATH).read()
    assert "oxo_" not in out
    needed = os.popen("readelf -d %s" % _lib.LIB_PATH).read()
    assert "oxoracle" not in needed and "oxref" not in needed


def test_shape_helpers_match_the_reference_rules():
    lib = _lib.lib()
    o = oxlibs.oracle()
    handled = (3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 19, 20, 25, 36)
    for qt in tuple(range(0, 40)):
        for cols in (0, 32, 96, 256, 896, 900, 2816, 4096, 14336):
            want = o.oxo_act_kind(qt, cols) if qt in handled else 0      # every other id: declined
            assert lib.oxh_act_kind(qt, cols) == want
            assert (lib.oxh_act_kind(qt, cols) != 0) == (qt in handled and want != 0)
    assert lib.oxh_row_bytes(13, 4096) == 2304
    assert lib.oxh_row_bytes(16, 14336) == 11760
    assert lib.oxh_row_bytes(7, 896) == 952
    assert lib.oxh_row_bytes(13, 896) == 0
    assert lib.oxh_row_bytes(15, 4096) == 2816 and lib.oxh_row_bytes(14, 256) == 176
    assert [lib.oxh_row_bytes(q, 896) for q in (3, 4, 5, 6)] == [28 * 18, 28 * 20, 28 * 22, 28 * 24]
    assert [lib.oxh_row_bytes(q, 896) for q in (17, 18, 19, 20)] == [28 * 18, 28 * 14, 28 * 22, 28 * 34]
    assert [lib.oxh_row_bytes(q, 4096) for q in (8, 9, 10, 11)] == [16 * 84] + [16 * 110] * 3
    assert lib.oxh_act_bytes(13, 4096) == 4672
    assert lib.oxh_act_bytes(7, 896) == 952
    for cols in (0, 31, 256, 896, 4096, 14336, 1 << 20, 3 << 20):
        assert lib.oc_matvec_batch_scratch_bytes(cols) == o.oxo_matvec_batch_scratch_bytes(cols)


def test_fused_switch_and_counters():
    lib = _lib.lib()
    assert lib.oc_matvec_fused_enabled() is True
    lib.oc_matvec_set_fused(False)
    assert lib.oc_matvec_fused_enabled() is False
    lib.oc_matvec_set_fused(True)
    lib.oc_matvec_fused_test_reset()
    st = lib.oc_matvec_fused_test_stats()
    assert (st.activation_quantizations, st.parallel_dispatches, st.fallback_calls) == (0, 0, 0)


def test_declines_need_no_device():
    x = synth.normal(4096, seed=1)
    w = synth.weights(13, 2, 4096, seed=1)
    out = np.full(2, 9.0, np.float32)
    temp = np.zeros(4096, np.float32)
    assert mv.matvec_quantized(13, w, 2, 896, 504, x, out, temp) == mv.DECLINED
    assert mv.matvec_quantized(13, w, 2, 4096, 2320, x, out, temp) == mv.DECLINED
    assert mv.matvec_quantized(2, w, 2, 4096, 8192, x, out, temp) == mv.DECLINED
    assert b"declined" in _lib.lib().oxh_last_error()
    assert np.all(out == 9.0)


def test_without_a_device_the_library_reports_it():
    """In a GPU-less container the compute entry points must return an error
    (never a result): there is no CPU path behind them."""
    lib = _lib.lib()
    rc = lib.oxh_init(0)
    if rc == 0:
        return                                   # a GPU is present: covered by the gpu tests
    assert rc == _lib.ERR_NO_DEVICE
    assert b"no HIP device" in lib.oxh_last_error()
    x = synth.normal(256, seed=1)
    w = synth.weights(13, 4, 256, seed=1)
    out = np.full(4, 9.0, np.float32)
    temp = np.zeros(256, np.float32)
    try:
        mv.matvec_quantized(13, w, 4, 256, 144, x, out, temp)
    except mv.OxhError as e:
        assert e.status == _lib.ERR_NO_DEVICE
    else:
        raise AssertionError("expected an error without a device")
    assert np.all(out == 9.0)


def test_synthetic_generator_is_deterministic():
    a = synth.weights(13, 64, 1024, seed=5, stream=2)
    b = synth.weights(13, 64, 1024, seed=5, stream=2)
    c = synth.weights(13, 64, 1024, seed=6, stream=2)
    assert np.array_equal(a, b) and not np.array_equal(a, c)
    blk = a.reshape(-1, 144)
    d = blk[:, :2].copy().view(np.float16).astype(np.float32)
    assert np.all(np.isfinite(d)) and np.all(d >= 0) and 0.012 < d.mean() < 0.020
    x = synth.normal(1 << 16, seed=0)
    assert abs(float(x.mean())) < 0.02 and abs(float(x.std()) - 1.0) < 0.02
    q = synth.weights(7, 16, 896, seed=1).reshape(-1, 34)[:, 2:].copy().view(np.int8)
    assert q.min() >= -127 and q.max() <= 127
    s6 = synth.weights(16, 4, 512, seed=1).reshape(-1, 210)[:, 192:208].copy().view(np.int8)
    assert s6.min() >= -32 and s6.max() <= 31


def test_void_symbols_hand_declined_calls_to_the_cpu_fallback():
    """A link-time replacement must not kill the process on a shape the reference's own code handles
    (matvec.c:833-907 falls back to its dequantise path): with a CPU fallback installed the void
    oc_matvec_quantized* symbols forward the call with its original arguments."""
    lib = _lib.lib()
    o = oxlibs.oracle()
    seen = []

    ONE = ctypes.CFUNCTYPE(None, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t, ctypes.c_size_t,
                           ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p)
    BATCH = ctypes.CFUNCTYPE(None, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t,
                             ctypes.c_size_t, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p, ctypes.c_size_t,
                             ctypes.c_size_t, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t)

    def cpu_one(qt, data, rows, cols, rb, x, out, temp):
        seen.append(("one", qt, rows, cols, rb))
        # the caller's CPU path: here the oracle's integer path over the same arguments
        o.oxo_matvec_quantized(qt, data, rows, cols, rb, x, out, temp)

    def cpu_batch(qt, data, rows, cols, rb, xs, in_stride, outs, out_stride, n_vec, temp, scratch, nscratch):
        seen.append(("batch", qt, rows, cols, n_vec))

    class Table(ctypes.Structure):
        _fields_ = [("one", ONE), ("fused", ctypes.c_void_p), ("multi", ctypes.c_void_p), ("batch", BATCH)]

    table = Table(ONE(cpu_one), None, None, BATCH(cpu_batch))
    lib.oxh_set_cpu_fallback(ctypes.byref(table))
    try:
        before = lib.oxh_cpu_fallback_calls()
        rows, cols = 4, 512
        w = synth.weights(13, rows, cols, seed=3)
        x = synth.normal(cols, seed=3)
        out = np.full(rows, 9.0, np.float32)
        temp = np.zeros(cols, np.float32)
        lib.oc_matvec_set_fused(False)             # OC_NO_FUSED: every call is declined
        lib.oc_matvec_quantized(13, w.ctypes.data, rows, cols, 288, x.ctypes.data, out.ctypes.data,
                                temp.ctypes.data)
        lib.oc_matvec_set_fused(True)
        assert seen == [("one", 13, rows, cols, 288)]
        want = np.zeros(rows, np.float32)
        wtmp = np.zeros(cols, np.float32)
        o.oxo_matvec_quantized(13, w.ctypes.data, rows, cols, 288, x.ctypes.data, want.ctypes.data,
                               wtmp.ctypes.data)
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
        # a padded row stride is declined too (matvec.c:961-985) and goes to the batch fallback
        scratch = np.zeros(1 << 16, np.uint8)
        lib.oc_matvec_quantized_batch(13, w.ctypes.data, rows, cols, 304, x.ctypes.data, cols, out.ctypes.data,
                                      rows, 1, temp.ctypes.data, scratch.ctypes.data, scratch.size)
        assert seen[-1] == ("batch", 13, rows, cols, 1)
        assert lib.oxh_cpu_fallback_calls() == before + 2
    finally:
        lib.oxh_set_cpu_fallback(None)


def test_weight_stats_and_unregister_need_no_device():
    lib = _lib.lib()
    n = [ctypes.c_size_t(7) for _ in range(4)]
    assert lib.oxh_weight_stats(*[ctypes.byref(v) for v in n]) == 0
    assert lib.oxh_init(0) != 0 or True
    buf = np.zeros(64, np.uint8)
    assert lib.oxh_weight_unregister(buf.ctypes.data) == 0      # nothing there: not an error


def test_plan_deals_rows_within_the_grid():
    """How a plan spreads an operation's rows over the device is host arithmetic: never more workgroups
    than the grid, every segment served, no wave beyond 32 table rows."""
    lib = _lib.lib()

    def deal(rows, paired, grid):
        n = len(rows)
        r = (ctypes.c_size_t * n)(*rows)
        p = (ctypes.c_int * n)(*paired)
        wg = (ctypes.c_uint32 * n)()
        cap = ctypes.c_uint32()
        rc = lib.oxh_plan_deal(r, p, n, grid, wg, ctypes.byref(cap))
        return rc, list(wg), cap.value

    rc, wg, cap = deal([4096, 1024, 1024], [0, 0, 0], 256)       # q/k/v: plain rounding would take 257
    assert rc == 0 and sum(wg) <= 256 and wg[1] == wg[2] == 43 and wg[0] in (170, 171) and cap == 2
    rc, wg, cap = deal([14336], [1], 256)                        # gate/up pair: 3.5 rows per wave, both matrices
    assert rc == 0 and wg == [256] and cap == 8
    rc, wg, cap = deal([4096], [0], 256)
    assert rc == 0 and wg == [256] and cap == 1
    rc, wg, cap = deal([100], [0], 256)                          # fewer rows than waves: 7 workgroups are enough
    assert rc == 0 and wg == [7] and cap == 1
    rc, wg, cap = deal([7, 9000, 3], [0, 0, 0], 304)
    assert rc == 0 and sum(wg) <= 304 and min(wg) >= 1
    assert deal([1 << 20], [0], 256)[0] == _lib.ERR_TOO_WIDE     # 256 rows per wave: beyond the table
    assert deal([0], [0], 256)[0] == _lib.ERR_ARG


def test_mmq_tile_choice_is_host_arithmetic():
    """Which tile a matrix-core launch runs on depends on the launch and the number of compute units
    only: the benchmark's two prefill shapes take the big tiles on a 256-CU device, a device with fewer
    units takes them sooner, small batches take the small tiles (the smallest when that leaves no unit more
    than one), Q6_K has the 64 x 128 tile for matrices with few rows."""
    lib = _lib.lib()
    Q4K, Q5K, Q6K, Q80, WIDE2 = 13, 15, 16, 7, 0x1008

    def tile(qtype, rows, n_vec, n_cu=256):
        r, t = ctypes.c_uint32(), ctypes.c_uint32()
        rc = lib.oxh_mmq_tile(qtype, rows, n_vec, n_cu, ctypes.byref(r), ctypes.byref(t))
        return rc, r.value, t.value

    assert tile(Q4K, 14336, 512) == (0, 256, 128)        # 56 x 4 = 224 workgroups = 256 - 32
    assert tile(Q4K, 4096, 512) == (0, 128, 64)          # 16 x 4 = 64 big tiles would idle three quarters
    assert tile(Q4K, 4096, 512, n_cu=64) == (0, 256, 128)
    assert tile(Q4K, 14336, 16) == (0, 64, 16)
    assert tile(Q4K, 14336, 32) == (0, 64, 32)
    assert tile(Q4K, 1000, 100) == (0, 64, 16)           # neither larger tile fills the device; 16 x 7 small ones
    assert tile(Q4K, 7000, 40) == (0, 64, 32)            # 110 x 3 of the smallest would be more than one to a unit
    assert tile(Q4K, 4096, 64) == (0, 64, 16)            # 64 x 4 = one per unit
    assert tile(Q4K, 4096, 128) == (0, 64, 32)
    assert tile(Q5K, 28672, 512) == (0, 128, 128)        # one row chunk per wave: 128-row tiles
    assert tile(Q5K, 3600, 500) == (0, 128, 64)
    assert tile(Q6K, 4096, 512) == (0, 64, 128)          # 32 x 4 tiles of 128 x 128 are too few
    assert tile(Q6K, 14336, 512) == (0, 128, 128)
    assert tile(WIDE2, 14336, 512) == (0, 128, 128)
    # the rule itself, stated independently: the first of the candidates with at least 7/8 of the units busy
    def rule(qtype, rows, n_vec, n_cu):
        need = n_cu - n_cu // 8
        small = (64, 16) if -(-rows // 64) * -(-n_vec // 16) <= n_cu else (64, 32)
        if n_vec <= 16:
            return 64, 16
        if n_vec <= 32:
            return small
        cands = [(256, 128), (128, 64)] if qtype == Q4K else \
                [(128, 128), (128, 64)] if qtype == Q5K else [(128, 128), (64, 128), (128, 64)]
        for tr, tt in cands:
            if -(-rows // tr) * -(-n_vec // tt) >= need:
                return tr, tt
        return small
    for qtype in (Q4K, Q5K, Q6K):
        for rows in (1, 63, 64, 1000, 4096, 7165, 14336, 28672, 151936):
            for n_vec in (1, 16, 17, 32, 33, 64, 100, 128, 129, 512, 2048):
                for n_cu in (64, 256, 304):
                    assert tile(qtype, rows, n_vec, n_cu) == (0,) + rule(qtype, rows, n_vec, n_cu)
    # the 32-value formats have two, and run on the one named; the codebook formats have no matrix-core kernel
    for qtype in (Q80, 3, 4, 5, 6, 17, 18, 19, 20):
        assert tile(qtype, 4096, 512) == (0, 128, 64)
        for rows, n_vec in ((64, 17), (4096, 64), (4096, 512), (4224, 448), (14336, 512), (151936, 2048)):
            for n_cu in (64, 256, 304):
                assert tile(qtype, rows, n_vec, n_cu)[1:] == mv.mmq_kernel(qtype, rows, 4096, n_vec, n_cu)[1:3]
        assert tile(qtype, 14336, 512) == (0, 64, 64)
    assert tile(25, 4096, 512)[0] == _lib.DECLINED
    assert tile(Q4K, 0, 512)[0] == _lib.DECLINED
    assert lib.oxh_mmq_tile(Q4K, 4096, 512, 256, None, None) == 0


def test_which_kernel_a_matrix_core_launch_runs_on_is_host_arithmetic():
    """oxh_lab()->mmq_kernel and ->experts_tile answer with what the launches themselves ask, also where oxh_mmq_tile
    names another tile: Q6_K prompts, small batches with and without a workspace, expert layers."""
    Q4K, Q5K, Q6K, Q80, WIDE2, T16 = 13, 15, 16, 7, 0x1008, 0x100A
    k = mv.mmq_kernel
    assert k(Q4K, 14336, 4096, 512)[:3] == (mv.MMQ_TILES, 256, 128)
    assert k(Q5K, 28672, 4096, 512)[:3] == (mv.MMQ_TILES, 128, 128)
    assert k(Q5K, 3600, 512, 500)[:3] == (mv.MMQ_TILES, 128, 64)
    assert k(Q6K, 4096, 14336, 333) == (mv.MMQ_SHARED, 64, 128, 4)          # 21 chunks of 16 tokens in 4 tiles, not 3
    assert k(Q6K, 4096, 14336, 128) == (mv.MMQ_SHARED, 64, 128, 4)          # two chunks a tile
    assert k(WIDE2, 4096, 14336, 512) == (mv.MMQ_SHARED, 64, 128, 4)
    assert k(Q6K, 14336, 14336, 144) == (mv.MMQ_SHARED, 64, 128, 2)         # 224 row tiles: what the tokens need
    assert k(Q80, 4096, 4096, 512)[:3] == (mv.MMQ_TILES, 128, 64)
    kernel, rows, tokens, waves = k(Q6K, 4096, 14336, 16)           # one 16-row group per CU, columns shared in LDS
    assert (kernel, rows, tokens) == (mv.MMQ_BATCH, 16, 16) and 4 <= waves <= 16
    assert k(Q4K, 4096, 4096, 24)[:3] == (mv.MMQ_BATCH, 16, 32)
    assert k(Q4K, 32, 14336, 16, ws_bytes=1 << 30)[0] == mv.MMQ_SPLIT      # few rows, many columns, room for the terms
    assert k(Q4K, 32, 14336, 16, ws_bytes=0)[:3] == (mv.MMQ_BATCH, 16, 16)
    assert k(Q4K, 28672, 4096, 16) == (mv.MMQ_TILES, 64, 16, 0)
    for qtype, cols in ((25, 4096), (Q4K, 300)):
        out = (ctypes.c_uint32 * 4)()
        assert _lib.lab().mmq_kernel(qtype, 4096, cols, 16, 256, 0, ctypes.byref(out)) == _lib.DECLINED
    t = mv.experts_tile
    assert t(Q4K, 2, 8, 14336, 32) == t(T16, 2, 8, 14336, 32) == (64, 16)
    assert t(Q4K, 2, 8, 14336, 8 * 50) == (128, 64)
    assert t(Q4K, 2, 8, 14336, 8 * 128) == (256, 144)
    assert t(Q6K, 2, 8, 14336, 8 * 128) == (128, 144)
    out = (ctypes.c_uint32 * 2)()
    assert _lib.lab().experts_tile(Q80, 2, 8, 14336, 32, 256, ctypes.byref(out)) == _lib.DECLINED


def test_small_batches_go_where_they_measured_fastest():
    """Sizes at which the workgroups of 16 rows measured slower than the tiles, or than tiles that share their columns
    through a workspace (one super-block; grids a little past the CUs; few rows under many super-blocks; few
    super-blocks under more than 16 activations), and sizes at which they measured faster, on 256 compute units."""
    Q4K, Q5K, Q6K, WIDE2, ROOM = 13, 15, 16, 0x1008, 1 << 40
    slower = [(Q4K, 4096, 256, 24, 0), (Q6K, 64, 256, 64, 0), (Q4K, 16384, 1024, 16, 0), (Q4K, 16384, 1024, 1, 0),
              (Q5K, 14336, 9216, 16, 0), (Q4K, 14336, 24320, 16, 0), (WIDE2, 14336, 8192, 16, 0), (Q6K, 5120, 1024, 17, 0),
              (Q4K, 5120, 1024, 32, 0), (WIDE2, 5120, 2048, 24, 0), (Q4K, 5120, 24320, 1, ROOM), (Q4K, 1024, 24320, 1, ROOM),
              (Q5K, 5120, 14336, 16, ROOM), (Q6K, 1024, 24320, 5, ROOM), (Q4K, 500, 8192, 24, ROOM),
              (Q6K, 500, 8192, 33, ROOM), (Q4K, 5120, 8704, 24, ROOM), (Q6K, 500, 8192, 16, ROOM), (Q5K, 16, 9216, 16, ROOM)]
    for case in slower:
        qtype, rows, cols, n_vec, ws = case
        assert mv.mmq_kernel(qtype, rows, cols, n_vec, 256, ws)[0] != mv.MMQ_BATCH, case
    for case in [(Q6K, 4096, 14336, 16, ROOM), (Q6K, 4096, 14336, 16, 0), (Q4K, 4096, 4096, 24, ROOM), (Q4K, 8192, 4096, 16, 0),
                 (Q4K, 5120, 24320, 16, 0), (Q4K, 14336, 4096, 16, 0), (Q6K, 14336, 4096, 16, 0), (Q5K, 4096, 4096, 9, ROOM),
                 (Q6K, 5120, 2048, 32, 0), (Q4K, 1500, 4096, 64, ROOM), (WIDE2, 4096, 14336, 16, ROOM), (Q4K, 16, 2560, 1, 0)]:
        qtype, rows, cols, n_vec, ws = case
        assert mv.mmq_kernel(qtype, rows, cols, n_vec, 256, ws)[0] == mv.MMQ_BATCH, case


def test_q6_k_prompts_go_to_the_tile_that_measured_fastest():
    """Q6_K and widened Q2_K above the small batches, on 256 compute units: sizes at which the 64 x 128 tiles measured
    slower than the 64 x 32, the 64 x 16 or the 128 x 128 ones (one super-block, two rounds against one), and sizes at which
    they measured faster, among them launches of one round, which are cut into more tiles than the tokens need."""
    Q6K, WIDE2 = 16, 0x1008
    for qtype, rows, cols, n_vec, tile in (
            (Q6K, 8300, 512, 256, (128, 128)), (Q6K, 4096, 4096, 2048, (128, 128)), (Q6K, 12544, 4096, 4096, (128, 128)),
            (Q6K, 6144, 256, 40, (64, 32)), (Q6K, 14336, 256, 129, (128, 128)), (WIDE2, 8192, 256, 48, (64, 32)),
            (WIDE2, 4099, 512, 130, (64, 32)), (Q6K, 414, 1024, 135, (64, 16)), (Q6K, 14336, 4096, 512, (128, 128)),
            (Q6K, 4096, 14336, 333, (64, 128)), (Q6K, 4096, 14336, 512, (64, 128)), (Q6K, 4096, 14336, 80, (64, 128)),
            (Q6K, 4096, 14336, 128, (64, 128)), (Q6K, 14336, 14336, 144, (64, 128)), (Q6K, 16384, 8192, 160, (64, 128)),
            (Q6K, 8192, 4096, 129, (64, 128)), (Q6K, 7736, 17664, 42, (64, 128)), (Q6K, 10240, 14336, 64, (64, 128)),
            (Q6K, 164, 16640, 448, (64, 128)), (WIDE2, 4096, 14336, 512, (64, 128)), (WIDE2, 4096, 14336, 80, (64, 128)),
            (WIDE2, 10240, 5120, 64, (64, 128)), (WIDE2, 8180, 5120, 75, (64, 128)), (WIDE2, 7168, 14336, 48, (64, 128)),
            (WIDE2, 6144, 5120, 33, (64, 128)), (WIDE2, 8192, 14336, 96, (64, 128)), (WIDE2, 2049, 1280, 390, (64, 128))):
        assert mv.mmq_kernel(qtype, rows, cols, n_vec)[1:3] == tile, (qtype, rows, cols, n_vec)


def test_prompts_of_the_32_value_formats_take_the_wide_tile_where_one_round_of_it_holds_on_every_xcd():
    """The row tiles are dealt to eight XCDs of 32 compute units: what counts is the tiles of the one that gets the most, not
    those of the device.  Sizes at which both tiles measured, between 231 and 256 tiles of 128 rows in all."""
    for rows, n_vec, tile in ((4224, 448, (64, 64)), (2100, 960, (64, 64)), (2199, 703, (64, 64)), (4250, 410, (64, 64)),
                              (2776, 666, (64, 64)), (3551, 542, (64, 64)), (4096, 512, (128, 64)), (3072, 512, (128, 64)),
                              (1717, 519, (128, 64)), (5354, 165, (128, 64)), (2048, 512, (64, 64)), (14336, 512, (64, 64)),
                              (8192, 512, (64, 64)), (64, 1024, (64, 64))):
        assert mv.mmq_kernel(7, rows, 4096, n_vec) == (mv.MMQ_TILES,) + tile + (0,), (rows, n_vec)


def test_the_prompt_tiles_of_the_32_value_formats_keep_everything_in_registers(tmp_path):
    """No k_mmq_32 has scratch memory: what the compiler notes beside each kernel of the built library."""
    import shutil
    import subprocess
    tools = "/opt/rocm/llvm/bin"
    shutil.copy(_lib.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([tools + "/llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    scratch = {}
    for obj in tmp_path.glob("*gfx950"):
        name = None
        for line in subprocess.run([tools + "/llvm-readelf", "--notes", str(obj)], check=True, capture_output=True,
                                   text=True).stdout.splitlines():
            if ".name:" in line and "_Z" in line:
                name = line.split()[-1]
            elif ".private_segment_fixed_size:" in line and name:
                scratch[name] = int(line.split()[-1])
    tiles = {n: v for n, v in scratch.items() if "k_mmq_32" in n}
    assert len(tiles) == 12 and not any(tiles.values()), tiles


@pytest.mark.parametrize("block_bytes", [14, 18, 20, 22, 24, 34])
def test_prompts_of_the_32_value_formats_find_every_block_of_the_longest_rows(block_bytes):
    """A lane's place in its wave's eight rows is a 32-bit offset: eight rows of 34-byte blocks pass 2^32 bytes from
    15 790 321 blocks on, and oxh_mmq takes 0xFFFFFF.  Also the shortest rows and those that end within a step."""
    at = _lib.lab().mmq32_fetched
    for blocks in (1, 7, 8, 9, 63, 64, 15790320, 15790321, 0xFFFFF7, 0xFFFFFF):
        last = (blocks - 1) // 8
        for step in sorted({0, min(1, last), last // 2, max(last - 1, 0), last}):
            for row in range(8):
                for blk in range(8):
                    b = 8 * step + blk
                    if b >= blocks:
                        b = b - 8 if step else blocks - 1
                    assert at(block_bytes, blocks, row, blk, step) == (row * blocks + b) * block_bytes, (blocks, row, blk, step)


def test_expert_launches_go_to_the_tile_that_measured_fastest():
    """Expert launches on 256 compute units: Q5_K and Q6_K keep the 64 x 16 tiles up to more tokens per expert than Q4_K
    while those are many, and leave them earlier where there are two or three to a unit."""
    Q4K, Q5K, Q6K, T5 = 13, 15, 16, 0x100B
    for qtype, n_mat, n_expert, rows, tokens, small in (
            (Q5K, 2, 8, 14336, 12, True), (T5, 2, 8, 14336, 16, True), (Q6K, 2, 8, 14336, 12, True), (Q5K, 2, 16, 5632, 12, True),
            (Q4K, 2, 8, 14336, 10, True), (Q5K, 2, 4, 14336, 20, True), (Q5K, 1, 4, 4096, 48, False), (Q6K, 1, 4, 4096, 48, False),
            (Q6K, 2, 4, 2048, 48, False), (Q5K, 2, 8, 14336, 20, False), (Q6K, 2, 8, 14336, 16, False),
            (Q4K, 2, 8, 14336, 16, False), (Q4K, 1, 4, 4096, 48, True), (Q4K, 2, 4, 2048, 50, True), (Q6K, 1, 4, 1024, 48, True),
            (Q6K, 2, 60, 2048, 13, False), (Q5K, 2, 32, 2048, 16, False), (Q5K, 2, 16, 2048, 16, True)):
        assert (mv.experts_tile(qtype, n_mat, n_expert, rows, n_expert * tokens) == (64, 16)) == small, (qtype, rows, tokens)


def test_expert_launches_of_few_workgroups_go_to_those_of_16_rows():
    """On 256 compute units: up to four (Q6_K six) workgroups of 16 rows to a unit where LDS holds two, three quarters of that
    where it holds one; never over one super-block, nor against the switch that fixes the tiles."""
    Q4K, Q5K, Q6K, T16, Q80 = 13, 15, 16, 0x100A, 7
    b = mv.experts_batch
    for qtype, n_mat, n_expert, rows, cols, k, n_tok, takes in (
            (Q4K, 2, 8, 14336, 4096, 2, 16, False), (Q4K, 1, 8, 4096, 14336, 2, 16, False), (Q6K, 1, 16, 2560, 6144, 1, 3, True),
            (T16, 1, 4, 1536, 5120, 1, 36, True), (T16, 2, 16, 3072, 4096, 1, 2, True), (Q4K, 2, 16, 3072, 4096, 1, 8, False),
            (Q4K, 1, 4, 4096, 7168, 1, 4, True), (Q5K, 1, 4, 4096, 14336, 3, 4, False), (Q6K, 1, 4, 4096, 14336, 3, 4, True),
            (Q4K, 1, 4, 4096, 256, 1, 4, False), (Q4K, 1, 8, 1024, 2048, 2, 1024, False), (Q80, 1, 4, 512, 512, 1, 1, False),
            (Q4K, 1, 4, 512, 129 * 256, 1, 1, False)):
        assert b(qtype, n_mat, n_expert, rows, cols, k, n_tok) == takes, (qtype, n_mat, n_expert, rows, cols, k, n_tok)
    import subprocess
    import sys
    code = "from oxidize_amd import matvec as mv; print(mv.experts_batch(16, 1, 16, 2560, 6144, 1, 3))"
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=dict(os.environ, OXH_MOE_BIG_TILE_FROM="24"), check=True,
                         capture_output=True, text=True).stdout
    assert out.strip() == "False"


@pytest.mark.parametrize("value,from_tokens", [("8", 8), ("24", 24), ("100", 100), ("0", None)])
def test_the_tokens_per_expert_to_start_the_long_tiles_from_can_be_set(value, from_tokens):
    """OXH_MOE_BIG_TILE_FROM, read once per process: that average and nothing else decides, also for launches of few
    tiles, to which the rule on sizes gives the 64 x 16 ones."""
    import subprocess
    import sys
    code = ("from oxidize_amd import matvec as mv\n"
            "for rows in (256, 14336):\n"
            "    print(' '.join(str(mv.experts_tile(13, 2, 4, rows, 4 * t)[1]) for t in (1, 7, 8, 23, 24, 99, 100, 300)))\n")
    env = dict(os.environ, OXH_MOE_BIG_TILE_FROM=value)
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=env, check=True, capture_output=True, text=True).stdout
    for line in out.splitlines():
        for tokens, tile in zip((1, 7, 8, 23, 24, 99, 100, 300), line.split()):
            assert (int(tile) > 16) == (from_tokens is not None and tokens >= from_tokens), (value, tokens, tile)


def test_bindings_lay_the_structs_out_as_the_header_does(tmp_path):
    """The ctypes structures of the bindings against the C compiler's view of include/oxhip.h: size and
    the offset of every field (a field added to the header and not to the bindings would shift what
    follows it)."""
    import subprocess
    structs = {"OxhSegment": _lib.OxhSegment, "OxhPrologue": _lib.OxhPrologue, "OxhPlanOp": _lib.OxhPlanOp,
               "OxhMoe": _lib.OxhMoe, "OxhTensor": _lib.OxhTensor}
    lines = ['#include <stdio.h>', '#include <stddef.h>', '#include "oxhip.h"', 'int main(void) {']
    for name, cls in structs.items():
        lines.append('printf("%s size %%zu\\n", sizeof(%s));' % (name, name))
        for field, _ in cls._fields_:
            lines.append('printf("%s %s %%zu\\n", offsetof(%s, %s));' % (name, field, name, field))
    lines += ['return 0; }']
    src = tmp_path / "layout.c"
    src.write_text("\n".join(lines))
    exe = tmp_path / "layout"
    subprocess.run(["gcc", "-std=c11", "-I", os.path.join(ROOT, "include"), "-o", str(exe), str(src)], check=True)
    seen = {}
    for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines():
        name, field, value = line.split()
        seen[(name, field)] = int(value)
    for name, cls in structs.items():
        assert seen[(name, "size")] == ctypes.sizeof(cls), name
        for field, _ in cls._fields_:
            assert seen[(name, field)] == getattr(cls, field).offset, (name, field)


def test_shared_operand_tiles_wait_for_their_lds_bound_loads_before_each_barrier(tmp_path):
    """Loads that go straight to LDS are counted by nobody but the kernel's own waits.  In the compiled 64 x 128 tiles
    (oxh_mmq6.hip), before every barrier that such loads stand in front of: in the prologue, ahead of all results, a wait for
    everything on its way, stated in the source, whatever the compiler asks for next; inside the walk a wait (the source's, or
    the compiler's for a younger load) that leaves out no more loads than were asked for after them."""
    import subprocess
    from oxidize_amd import build
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path / "mmq6.s")
    subprocess.run([build.HIPCC] + build.HIP_FLAGS + ["-I", build.INCLUDE, "-I", build.CSRC, "-S", "--cuda-device-only",
                   os.path.join(build.CSRC, "oxh_mmq6.hip"), "-o", out], check=True, capture_output=True)
    prologues = steps = 0
    lds = own = product = False
    loads = 0           # vector loads since the last LDS-bound one
    for line in open(out):
        word = line.split()
        if not word or word[0].startswith((".", "_Z")):
            continue
        if word[0].startswith("global_load_lds"):
            lds, waited, loads = True, False, 0
        elif word[0].startswith("global_load"):
            loads += 1
        elif "mfma" in word[0]:
            product = True
        elif word[0] == ";;#ASMSTART":
            own = True
        elif word[0] == ";;#ASMEND":
            own = False
        elif word[0] == "s_waitcnt" and lds and "vmcnt" in line:
            left = int(re.search(r"vmcnt\((\d+)\)", line).group(1))
            waited = waited or (left <= loads if product else own and left == 0)
        elif word[0] == "s_barrier" and lds:
            assert waited, line
            prologues, steps = prologues + (not product), steps + product
            lds = product = False
        elif word[0] == "s_endpgm":
            lds = product = False
    assert prologues == 8 and steps >= 16           # halves of one to four chunks, two formats
