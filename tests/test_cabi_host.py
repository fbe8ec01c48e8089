"""CPU-only checks of the C ABI: the shared library loads, exports every symbol the header
declares, and its pure-host entry points (plan encoding, size queries, status strings)
behave as documented. No kernel is launched here.
"""
import ctypes as C
import os
import re

import numpy as np
import pytest

from jabas_amd import _lib as L

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "jabas_sync.h")


def _declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(jabas_[a-z_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = _declared_functions()
    assert len(names) >= 15
    lib = L.lib()
    for n in names:
        assert hasattr(lib, n), f"{n} declared in jabas_sync.h but not exported"
    assert set(names) == set(L.SIGNATURES), "ctypes signature table and header disagree"


def test_struct_layouts_match_the_header():
    # sizes a C compiler gives the header's structs on x86-64 / amdgcn host ABI
    K = L.MAX_K
    assert K == 16 and L.STATS_STRIDE == 40 >= max(4 + K, 4 + 8 + 28)     # full rows of 16 VSWs, pair products of 8
    assert C.sizeof(L.JabasSpan) == K * 8 + 5 * 8 + (K - 1) * 8 + 8 + 6 * 4
    assert C.sizeof(L.JabasBound) == 16
    assert C.sizeof(L.JabasGroup) == 24
    assert C.sizeof(L.JabasStepArgs) == 4 + 4 + 4 * K + 4 + K + 4 * K + 4 * 4 + 4 + 5 * 8 + 16 * 24 + 8 + 8
    assert L.JabasStepArgs.scalars_dev.offset == C.sizeof(L.JabasStepArgs) - 8
    assert L.JabasStepArgs.groups.offset % 8 == 0 and L.JabasStepArgs.momentum.offset % 8 == 0


def test_version_and_status_strings():
    lib = L.lib()
    assert b"jabas_sync" in lib.jabas_sync_version()
    assert lib.jabas_status_string(0) == b"ok"
    seen = {lib.jabas_status_string(s) for s in range(-11, 0)}
    assert len(seen) == 11 and b"unknown status" not in seen
    assert lib.jabas_status_string(-99) == b"unknown status"


def _span(numel, base=0x7f0000000000, K=2, gs=4, skew=0, opt=False, stride=1 << 32):
    s = L.JabasSpan()
    for k in range(K):
        s.grads[k] = base + k * stride + skew * gs
    s.agg_out = base + 16 * stride + skew * 4
    if opt:
        s.param = base + 17 * stride + skew * 4
        s.state1 = base + 18 * stride + skew * 4
        s.state2 = base + 19 * stride + skew * 4
    s.numel = numel
    return s


def _encode(spans, bounds=(), K=2, dtype=L.F32, opt=L.OPT_NONE):
    lib = L.lib()
    arr = (L.JabasSpan * len(spans))(*spans)
    barr = (L.JabasBound * max(1, len(bounds)))()
    for i, (st, g) in enumerate(bounds):
        barr[i].start, barr[i].group = st, g
    nbytes = lib.jabas_plan_bytes(arr, len(spans), len(bounds), dtype)
    blob = np.zeros(nbytes // 8 + 1, dtype=np.uint64)
    rc = lib.jabas_plan_encode(arr, len(spans), barr if bounds else None, len(bounds), K, dtype, opt,
                               blob.ctypes.data, nbytes)
    return rc, blob, nbytes


def test_plan_encode_counts_chunks():
    """A tile is 1024 elements; a workgroup takes 2 tiles for K <= 4 and 4 tiles above."""
    lib = L.lib()
    sizes = [4096, 4097, 1, 0, 10 * 4096 + 5]
    rc, blob, _ = _encode([_span(n) for n in sizes])
    assert rc == L.OK
    assert lib.jabas_plan_chunks(blob.ctypes.data, 0) == 2 + 3 + 1 + 0 + 21
    assert lib.jabas_plan_chunks(blob.ctypes.data, 1) == 2 + 3 + 1 + 0 + 21      # K <= 4 without optimizer: one shape
    assert lib.jabas_plan_workspace_bytes(blob.ctypes.data) >= (27 + 5) * L.STATS_STRIDE * 8     # a row per chunk and per span, at least
    for K in (8, 16):                  # K > 4 without optimizer: 4 tiles of 1024 for both kinds of launch
        rc, blob, _ = _encode([_span(n, K=K) for n in sizes], K=K)
        assert rc == L.OK
        assert lib.jabas_plan_chunks(blob.ctypes.data, 1) == 1 + 2 + 1 + 0 + 11
        assert lib.jabas_plan_chunks(blob.ctypes.data, 0) == 1 + 2 + 1 + 0 + 11
    # a span that starts 3 elements into a 16-byte line needs one more tile when it is exactly full
    rc, blob, _ = _encode([_span(4096, skew=3)])
    assert rc == L.OK and lib.jabas_plan_chunks(blob.ctypes.data, 0) == 3


@pytest.mark.parametrize("K,sizes,rows", [
    # rows of the level with the most workgroups: chunks of four tiles for full rows and K > 4, else two (similarity sums)
    (8, [700] * 200, 200), (8, [5] * 211, 211), (16, [700] * 5000, 5000), (2, [1000] * 210, 210),      # one tile in every chunk
    (8, [1500] * 210, 420), (16, [3000] * 3000, 6000),                   # two and three tiles
    (8, [4096] * 200, 400), (8, [1 << 20], 512), (16, [1 << 24], 8192), (4, [1 << 18], 256), (8, [4096] * 145, 580),       # whole chunks
    (8, [700] * 12, 48), (8, [5000], 5 + 3), (8, [700] * 64, 256),       # empty workgroups on compute units that are left
    (8, [300] * 50 + [60000] * 13, 490)])                                # 50 + 13 * 15 chunks, 440 of 490 workgroups with a tile
def test_plan_splits_chunks_that_hold_tiles_for_it(K, sizes, rows):
    """A launch with statistics shares its chunks between workgroups until there are enough of them (full rows of more than eight
    workers: always two), but not where more than a quarter of them would find no tile: scratch holds one row per workgroup. A
    blob that does not record this (encoded before it was) is launched by the number of chunks alone."""
    lib = L.lib()
    rc, blob, _ = _encode([_span(n, K=K) for n in sizes], K=K)
    assert rc == L.OK
    stripes = 32 * len(sizes) + 1
    assert lib.jabas_plan_workspace_bytes(blob.ctypes.data) == (rows + stripes) * L.STATS_STRIDE * 8
    old = blob.copy()
    old.view(np.uint32)[9] = 0
    unlimited = []
    for level, split in ((L.STATS_FULL, int(K > 8)), (L.STATS_SIMILARITY, 0)):
        n = lib.jabas_plan_chunks(blob.ctypes.data, level)
        tiles = 4 if K > 4 and level == L.STATS_FULL else 2
        while 2 << split <= tiles and n << split < 384:
            split += 1
        unlimited.append(n << split)
    assert lib.jabas_plan_workspace_bytes(old.ctypes.data) == (max(unlimited) + stripes) * L.STATS_STRIDE * 8
    for junk in (0x04040404, 0x20202020, 0x21212121, 0xffffffff):                # more workgroups than a chunk has tiles: not taken
        old.view(np.uint32)[9] = junk
        assert lib.jabas_plan_workspace_bytes(old.ctypes.data) == (max(unlimited) + stripes) * L.STATS_STRIDE * 8


@pytest.mark.parametrize("groups,rows", [((0,), 450), ((0, 1), 900)])
def test_plan_splits_further_where_parameter_groups_change(groups, rows):
    """With statistics, 450 chunks are shared where the parameter group changes inside a span (up to 512 workgroups), not where it
    does not (up to 384)."""
    lib = L.lib()
    span = _span(900 * 1024, K=4, opt=True)
    span.bound_count = len(groups)
    bounds = [(i * 70_001, g) for i, g in enumerate(groups)]
    rc, blob, _ = _encode([span], bounds, K=4, opt=L.OPT_SGD)
    assert rc == L.OK and lib.jabas_plan_chunks(blob.ctypes.data, L.STATS_FULL) == 450
    assert lib.jabas_plan_workspace_bytes(blob.ctypes.data) == (rows + 33) * L.STATS_STRIDE * 8


def test_plan_encode_starts_the_element_grid_at_a_256_byte_line_when_all_buffers_allow_it():
    """2048 elements per workgroup here (K = 2, no optimizer). With every buffer 61 elements into a
    256-byte line the grid starts at that line: 61 + 4036 elements still fit two workgroups, one
    more element does not. With one buffer elsewhere in its 256-byte line (but at the same place of
    its 16-byte line) the grid starts at the first element's 16-byte line, 1 element in."""
    lib = L.lib()
    for numel, want in ((4096 - 61, 2), (4096 - 60, 3)):
        rc, blob, _ = _encode([_span(numel, skew=61)])
        assert rc == L.OK and lib.jabas_plan_chunks(blob.ctypes.data, 0) == want
    for numel, want in ((4096 - 60, 2), (4095, 2), (4096, 3)):
        s = _span(numel, skew=61)
        s.agg_out -= 16 * 4                  # 45 elements in: congruent mod 4, not mod 64
        rc, blob, _ = _encode([s])
        assert rc == L.OK and lib.jabas_plan_chunks(blob.ctypes.data, 0) == want
    # the bound jabas_plan_bytes and jabas_sync_workspace_bytes are sized by holds in either case
    rc, blob, nbytes = _encode([_span(1, skew=63), _span(2048 - 63, skew=63), _span(2048 - 62, skew=63)])
    assert rc == L.OK and lib.jabas_plan_chunks(blob.ctypes.data, 0) == 1 + 1 + 2
    assert lib.jabas_sync_workspace_bytes(2048 - 62, L.F32) >= 3 * L.STATS_STRIDE * 8


def test_plan_encode_bf16_positions_are_counted_in_elements():
    # bf16 gradients 2 elements into an 8-byte line, fp32 buffers 2 elements into a 16-byte line: congruent
    rc, _, _ = _encode([_span(5000, gs=2, skew=2)], dtype=L.BF16)
    assert rc == L.OK
    s = _span(5000, gs=2, skew=2)
    s.agg_out += 4                      # now 3 elements in: not congruent with the gradients
    rc, _, _ = _encode([s], dtype=L.BF16)
    assert rc == L.ERR_ALIGN


def test_plan_encode_rejects_bad_spans():
    s = _span(4096)
    s.grads[1] += 4
    assert _encode([s])[0] == L.ERR_ALIGN                       # gradients not mutually congruent
    s = _span(4096)
    s.grads[1] = 0
    assert _encode([s])[0] == L.ERR_NULL
    assert _encode([_span(4096)], K=17)[0] == L.ERR_K
    assert _encode([_span(4096)], dtype=7)[0] == L.ERR_DTYPE
    assert _encode([_span(4096)], opt=9)[0] == L.ERR_OPT
    assert _encode([_span(4096)], opt=L.OPT_SGD)[0] == L.ERR_NULL    # optimizer without weights
    s = _span(4096, opt=True)
    s.state2 = 0
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_NULL
    assert _encode([s], opt=L.OPT_SGD)[0] == L.OK
    s = _span(4096)
    s.agg_out = s.grads[0] + 16                                 # overlaps VSW 0's buffer, not in place
    assert _encode([s])[0] == L.ERR_ALIAS
    s = _span(4096)
    s.agg_out = s.grads[0]                                      # exactly in place: allowed for fp32
    assert _encode([s])[0] == L.OK
    s = _span(4096, gs=2)
    s.agg_out = s.grads[0]
    assert _encode([s], dtype=L.BF16)[0] == L.ERR_ALIAS          # fp32 output over bf16 input
    s = _span(4096, opt=True)
    s.n_fanout = 16
    assert _encode([s], opt=L.OPT_SGD)[0] == L.ERR_SIZE


@pytest.mark.parametrize("word,loose", [(0, False), (1, True), (2, False), (3, False), (0x80000001, False), (0xCDCDCDCD, False), (0xFFFFFFFF, False)])
def test_loose_gradients_are_asked_for_by_one_value_of_the_word(word, loose):
    """The span's last word was not read before it came to say that fp32 gradients may sit at any element: whatever else a caller
    left in it changes nothing, neither for a span that is accepted nor for one that is refused."""
    for dtype, gs in ((L.F32, 4), (L.BF16, 2)):
        aligned, off = _span(4096, gs=gs, opt=True), _span(4096, gs=gs, opt=True)
        off.grads[1] += gs
        aligned.reserved = off.reserved = word
        if dtype == L.BF16:
            aligned.agg_out = off.agg_out = None
        plain = _span(4096, gs=gs, opt=True)
        plain.agg_out = aligned.agg_out
        rc, blob, _ = _encode([aligned], dtype=dtype, opt=L.OPT_ADAMW)
        rc0, blob0, _ = _encode([plain], dtype=dtype, opt=L.OPT_ADAMW)
        assert rc == rc0 == L.OK and np.array_equal(blob, blob0)
        rc, _, _ = _encode([off], dtype=dtype, opt=L.OPT_ADAMW)
        assert rc == (L.OK if loose and dtype == L.F32 else L.ERR_ALIGN)


_CASES_OF_SPLITS = [
    # K, dtype, optimizer, level, elements of a chunk, {(chunks, group change): log2 of the workgroups that share one}
    (4, L.F32, L.OPT_ADAMW, 0, 4096, {(1023, True): 2, (1024, True): 1, (2047, True): 1, (2048, True): 0, (447, False): 1, (448, False): 0}),
    (1, L.F32, L.OPT_ADAM_AMSGRAD, 0, 4096, {(1023, True): 2, (2047, True): 1, (2048, True): 0}),
    (2, L.F32, L.OPT_SGD, 0, 1024, {(639, True): 1, (640, True): 0, (447, False): 1, (448, False): 0}),
    (2, L.BF16, L.OPT_SGD, 0, 2048, {(2047, True): 1, (2048, True): 0}),
    (9, L.F32, L.OPT_ADAM, 0, 2048, {(447, False): 1, (448, False): 0, (2047, False): 0, (2048, False): 1, (2047, True): 1, (2048, True): 1}),
    (16, L.BF16, L.OPT_SGD, 0, 2048, {(2047, False): 0, (2048, False): 1, (2047, True): 1}),
    (9, L.BF16, L.OPT_ADAMW, 2, 2048, {(511, True): 1, (512, True): 0, (4095, False): 0, (4096, False): 1, (4095, True): 0, (4096, True): 1}),
    (16, L.F32, L.OPT_SGD, 2, 2048, {(4095, False): 0, (4096, False): 1}),
]


@pytest.mark.parametrize("K,dtype,opt,level,chunk,splits", _CASES_OF_SPLITS)
def test_recorded_splits_on_both_sides_of_every_limit(K, dtype, opt, level, chunk, splits):
    """How many workgroups share a chunk, as the plan records it (byte `level` of the header's word 9: 1 + its log2), on both sides of the
    lengths at which that changes, for spans of one parameter group and with a change inside."""
    for (chunks, change), want in splits.items():
        n = chunks * chunk
        s = _span(n, K=K, gs=4 if dtype == L.F32 else 2, opt=True)
        s.state3 = s.state2 + (1 << 32) if opt == L.OPT_ADAM_AMSGRAD else None
        bounds = [(0, 0), (n // 2 + 77, 1)] if change else [(0, 0)]
        s.bound_count = len(bounds)
        rc, blob, _ = _encode([s], bounds, K=K, dtype=dtype, opt=opt)
        assert rc == L.OK
        assert L.lib().jabas_plan_chunks(blob.ctypes.data, level) == chunks
        assert int(blob.view(np.uint8)[36 + level]) == 1 + want, (chunks, change)


def test_plan_encode_checks_bounds():
    def with_bounds(bounds, count=None, begin=0):
        s = _span(10000, opt=True)
        s.bound_begin, s.bound_count = begin, len(bounds) if count is None else count
        return _encode([s], bounds=bounds, opt=L.OPT_SGD)[0]
    assert with_bounds([(0, 0), (100, 1), (9999, 0)]) == L.OK
    assert with_bounds([(1, 0)]) == L.ERR_GROUP                 # first bound must start at 0
    assert with_bounds([(0, 0), (100, 1), (100, 0)]) == L.ERR_GROUP   # not strictly increasing
    assert with_bounds([(0, 0), (10000, 1)]) == L.ERR_GROUP     # starts past the end
    assert with_bounds([(0, 16)]) == L.ERR_GROUP                # group index out of range
    assert with_bounds([(0, 0)], count=2) == L.ERR_GROUP        # table shorter than claimed


def test_plan_blob_too_small_and_garbage_header():
    lib = L.lib()
    spans = (L.JabasSpan * 1)(_span(4096))
    nbytes = lib.jabas_plan_bytes(spans, 1, 0, L.F32)
    blob = np.zeros(nbytes // 8 + 1, dtype=np.uint64)
    # jabas_plan_bytes is an upper bound over the launch shapes; the header and one span do not fit 128 bytes
    assert lib.jabas_plan_encode(spans, 1, None, 0, 2, L.F32, L.OPT_NONE, blob.ctypes.data, 128) == L.ERR_PLAN
    assert lib.jabas_plan_encode(spans, 1, None, 0, 2, L.F32, L.OPT_NONE, blob.ctypes.data, nbytes) == L.OK
    junk = np.zeros(64, dtype=np.uint64)
    assert lib.jabas_plan_chunks(junk.ctypes.data, 0) == L.ERR_PLAN
    assert lib.jabas_plan_workspace_bytes(junk.ctypes.data) == 0
    args = L.JabasStepArgs()
    args.K = 2
    assert lib.jabas_sync_fused(junk.ctypes.data, 0x1000, C.byref(args), None, None, 0, None) == L.ERR_PLAN
    assert lib.jabas_sync_fused(None, None, C.byref(args), None, None, 0, None) == L.ERR_NULL


def test_workspace_bytes_cover_any_line_position():
    lib = L.lib()
    row = L.STATS_STRIDE * 8
    assert lib.jabas_sync_workspace_bytes(0, L.F32) >= row
    assert lib.jabas_sync_workspace_bytes(4096, L.F32) >= 3 * row      # a shifted start adds a chunk
    assert lib.jabas_sync_workspace_bytes(1 << 30, L.BF16) >= ((1 << 30) // 2048) * row


def test_entry_points_validate_before_launching():
    """Argument errors are reported on a machine without a GPU because nothing is launched."""
    lib = L.lib()
    w = (C.c_float * 2)(0.5, 0.5)
    g = (C.c_void_p * 2)(0x7f0000000000, 0x7f0100000000)
    assert lib.jabas_aggregate(g, 0, L.F32, w, 0x7f0200000000, 100, None) == L.ERR_K
    assert lib.jabas_aggregate(g, 2, L.F32, w, None, 100, None) == L.ERR_NULL
    assert lib.jabas_aggregate(g, 2, 5, w, 0x7f0200000000, 100, None) == L.ERR_DTYPE
    g[1] = 0x7f0100000004
    assert lib.jabas_aggregate(g, 2, L.F32, w, 0x7f0200000000, 100, None) == L.ERR_ALIGN
    assert lib.jabas_sgd(None, 0x7f0000000000, None, 10, 0.1, 0.0, 0.0, 0.0, 0, 0, None) == L.ERR_NULL
    # momentum without a buffer
    assert lib.jabas_sgd(0x7f0000000000, 0x7f0100000000, None, 10, 0.1, 0.0, 0.9, 0.0, 0, 0, None) == L.ERR_NULL
    # nesterov needs momentum and zero dampening
    assert lib.jabas_sgd(0x7f0000000000, 0x7f0100000000, 0x7f0200000000, 10, 0.1, 0.0, 0.9, 0.1, 1, 0, None) == L.ERR_OPT
    # Adam's step count is 1-based
    assert lib.jabas_adam(0x7f0000000000, 0x7f0100000000, 0x7f0200000000, 0x7f0300000000, None, 10, 1e-3, 0.0, 0.9,
                          0.999, 1e-8, 0, 0, None) == L.ERR_OPT
    # amsgrad: the maximum is one more written buffer (it must not overlap the second moment), and its launches
    # take their scalars by value only
    assert lib.jabas_adam(0x7f0000000000, 0x7f0100000000, 0x7f0200000000, 0x7f0300000000, 0x7f0300000010, 10, 1e-3, 0.0,
                          0.9, 0.999, 1e-8, 1, 0, None) == L.ERR_ALIAS
    ams = L.JabasStepArgs()
    ams.K, ams.grad_dtype, ams.opt_kind, ams.n_groups = 1, L.F32, L.OPT_ADAMW_AMSGRAD, 1
    ams.weight[0], ams.beta1, ams.beta2, ams.eps = 1.0, 0.9, 0.999, 1e-8
    ams.groups[0].lr, ams.groups[0].step = 1e-3, 1
    sp = _span(1000, K=1, opt=True)
    assert lib.jabas_sync_bucket(C.byref(sp), None, C.byref(ams), None, None, 0, None) == L.ERR_NULL     # no state3
    block = np.zeros(L.STEP_SCALARS_BYTES, dtype=np.uint8)
    assert lib.jabas_step_scalars_encode(C.byref(ams), block.ctypes.data, block.nbytes) == L.ERR_OPT
    sp.state3 = 0x7f0000000000 + 21 * (1 << 32)
    ams.scalars_dev = 0x7f0000000000 + 22 * (1 << 32)
    assert lib.jabas_sync_bucket(C.byref(sp), None, C.byref(ams), None, None, 0, None) == L.ERR_OPT
    # statistics level 'gram' (pair products in the fused launch): up to STATS_GRAM_MAX_K workers; no level beyond it;
    # the static entry point's array holds rows of up to 4 + 16 sums and refuses the wider ones (six workers and more)
    many = L.JabasStepArgs()
    for dt, gs in ((L.F32, 4), (L.BF16, 2)):
        many.K, many.grad_dtype, many.stats = L.STATS_GRAM_MAX_K + 1, dt, L.STATS_GRAM
        spk = _span(1000, K=L.STATS_GRAM_MAX_K + 1, gs=gs)
        assert lib.jabas_sync_bucket(C.byref(spk), None, C.byref(many), 0x7f0400000000, 0x7f0500000000, 1 << 20, None) == L.ERR_K
        many.K = L.STATS_GRAM_MAX_K
        spk = _span(1000, K=L.STATS_GRAM_MAX_K, gs=gs)
        assert lib.jabas_sync_bucket(C.byref(spk), None, C.byref(many), 0x7f0400000000, 0x7f0500000000, 8, None) == L.ERR_WORKSPACE
        assert lib.jabas_sync_bucket_static(C.byref(spk), None, C.byref(many), 0x7f0400000000, None) == L.ERR_SIZE
        many.K = 6
        assert lib.jabas_sync_bucket_static(C.byref(_span(1000, K=6, gs=gs)), None, C.byref(many), 0x7f0400000000, None) == L.ERR_SIZE
    assert L.STAT_NORM_VSW0 + 8 + 28 == L.STATS_STRIDE == L.stat_pair(8, 6, 7) + 1
    many.K, many.stats = 2, L.STATS_GRAM + 1
    assert lib.jabas_sync_bucket(C.byref(spk), None, C.byref(many), 0x7f0400000000, 0x7f0500000000, 1 << 20, None) == L.ERR_OPT
    hid = (C.c_uint8 * 2)(0, 1)
    assert lib.jabas_stats(g, 2, L.F32, w, hid, w, 100, 0x7f0400000000, None, 0, None) == L.ERR_ALIGN
    g[1] = 0x7f0100000000
    assert lib.jabas_stats(g, 2, L.F32, w, hid, w, 100, 0x7f0400000000, None, 0, None) == L.ERR_WORKSPACE
    assert lib.jabas_gram(g, 2, L.F32, 100, 0x7f0400000000, None, 0, None) == L.ERR_WORKSPACE


def test_plain_c_client_sees_the_same_layout_and_drives_the_host_entry_points(tmp_path):
    """gcc -std=c99 compiles the header and a C client; the client links the library, reports the struct
    layout its compiler sees (compared field by field with the ctypes mirror) and encodes a plan."""
    import shutil
    import subprocess
    if shutil.which("gcc") is None:
        pytest.skip("no gcc")
    libdir = os.path.dirname(os.path.abspath(L.LIB_PATH))
    exe = str(tmp_path / "cabi_client")
    cmd = ["gcc", "-std=c99", "-Wall", "-Wextra", "-pedantic", "-Werror", "-I", os.path.join(ROOT, "include"),
           os.path.join(ROOT, "tests", "cabi_client.c"), "-o", exe, "-L", libdir, "-ljabas_sync",
           "-Wl,-rpath," + libdir, "-Wl,--allow-shlib-undefined"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    seen = {}
    for line in out.stdout.splitlines():
        kind, name, *rest = line.split(" ", 2)
        seen[(kind, name)] = rest[0] if rest else ""
    structs = {"JabasSpan": L.JabasSpan, "JabasBound": L.JabasBound, "JabasGroup": L.JabasGroup,
               "JabasStepArgs": L.JabasStepArgs}
    checked = 0
    for (kind, name), val in seen.items():
        if kind == "sizeof":
            assert C.sizeof(structs[name]) == int(val), name
            checked += 1
        elif kind == "offsetof":
            s, f = name.split(".")
            assert getattr(structs[s], f).offset == int(val), name
            checked += 1
    assert checked == 40
    # every field of the ctypes mirror was reported by the C side (reserved words aside)
    for sname, st in structs.items():
        for f, _ in st._fields_:
            if not f.startswith("reserved") and not f.startswith("_"):
                assert ("offsetof", f"{sname}.{f}") in seen, f"{sname}.{f}"
    assert seen[("version", "jabas_sync")].startswith("0.")
    assert seen[("status0", "ok")] == ""
    assert seen[("encode", "0")] == ""
    assert seen[("chunks", "14")] == ""                      # SGD, K = 2, fp32, plain: 1024 elements per chunk -> 5 + 9
    assert seen[("chunks_stats", "8")] == ""                 # with statistics: 2048 per chunk -> 3 + 5
    assert int(next(n for (k, n) in seen if k == "workspace")) >= (8 + 2) * L.STATS_STRIDE * 8
    assert ("encode_misaligned", str(L.ERR_ALIGN)) in seen
    # the ctypes mirror places the pair products of a 'gram' row where the header's macro does: behind the K norms,
    # in the order (0,1), (0,2), ..., (K-2,K-1), and within the row's JABAS_STATS_STRIDE slots
    for K, key in ((4, "pairs4"), (3, "pairs3")):
        want = [L.stat_pair(K, a, b) for a in range(K) for b in range(a + 1, K)]
        assert ("pairs%d" % K, ",".join(map(str, want))) in seen
        assert want == list(range(4 + K, 4 + K + K * (K - 1) // 2)) and want[-1] < L.STATS_STRIDE


def test_plan_encode_checks_interleaved_moments():
    """A span whose Adam moments sit interleaved in one arena (state_block_log2): the layout rules, and the
    moments from the first element's exp_avg to the last element's last moment as ONE written range."""
    T, n = 1 << 10, 5000
    arena = 0x7f0000000000 + 40 * (1 << 32)

    def span(pos=0, first_block=0, ways=2):
        s = _span(n, opt=True)
        s.state1 = arena + 4 * (first_block * ways * T + pos)
        s.state2 = s.state1 + 4 * T
        s.state3 = s.state1 + 8 * T if ways == 3 else None
        s.state_block_log2, s.state_block_pos = 10, pos
        return s
    assert _encode([span()], opt=L.OPT_ADAM)[0] == L.OK
    assert _encode([span()], opt=L.OPT_ADAMW)[0] == L.OK
    assert _encode([span(ways=3)], opt=L.OPT_ADAM_AMSGRAD)[0] == L.OK
    assert _encode([span()], opt=L.OPT_ADAM_AMSGRAD)[0] == L.ERR_NULL          # the maximum has no place in a two-way arena
    assert _encode([span()], opt=L.OPT_SGD)[0] == L.ERR_OPT
    s = span()
    s.state_block_log2 = 7
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_SIZE
    s = span()
    s.state_block_log2 = 25
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_SIZE
    s = span()
    s.state_block_pos = T
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_SIZE
    s = span()
    s.state2 += 16
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_ALIGN
    s = span(ways=3)
    s.state3 -= 4 * T
    assert _encode([s], opt=L.OPT_ADAM_AMSGRAD)[0] == L.ERR_ALIGN
    s = span()
    s.state_block_pos = 2                                         # the block group would start 8 bytes off a 16-byte line
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_ALIGN
    # a span in the middle of a block, at the other buffers' element of a 16-byte line
    s = _span(n, opt=True, skew=3)
    s.state1 = arena + 4 * (2 * T + 64 * 3 + 3)
    s.state2, s.state_block_log2, s.state_block_pos = s.state1 + 4 * T, 10, 64 * 3 + 3
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.OK
    s.state_block_pos -= 1                                        # another element of the line than the weights'
    s.state1 -= 4
    s.state2 -= 4
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_ALIGN
    # 5000 elements from position 0: blocks 0..4 of exp_avg and of exp_avg_sq, the last ends 4 * (9 * T + 904) bytes in
    end = arena + 4 * (9 * T + n - 4 * T)
    s = span()
    s.param = end                                                 # right behind the last second moment: fine
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.OK
    s.param = end - 16
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_ALIAS
    s = span()
    s.agg_out = arena + 4 * T + 256                               # inside the first block of second moments
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_ALIAS
    s = span()
    s.grads[1] = arena + 4 * (3 * T)                              # a gradient buffer inside a block the span does not own
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_ALIAS         # ... but which lies inside the one written range


def test_plan_encode_rejects_overlapping_written_buffers():
    def span():
        return _span(4096, opt=True)
    s = span()
    s.state1 = s.param + 4096 * 4 - 16                          # last four weights = first four momentum entries
    assert _encode([s], opt=L.OPT_SGD)[0] == L.ERR_ALIAS
    s = span()
    s.state1 = s.param + 4096 * 4                               # back to back: fine
    assert _encode([s], opt=L.OPT_SGD)[0] == L.OK
    s = span()
    s.state2 = s.state1
    assert _encode([s], opt=L.OPT_ADAM)[0] == L.ERR_ALIAS
    assert _encode([s], opt=L.OPT_SGD)[0] == L.OK               # SGD never touches state2
    s = span()
    s.param = s.grads[1]                                        # weights over a worker's gradients
    assert _encode([s], opt=L.OPT_SGD)[0] == L.ERR_ALIAS
    s = span()
    s.param = s.agg_out
    assert _encode([s], opt=L.OPT_SGD)[0] == L.ERR_ALIAS
    s = span()
    s.n_fanout = 2
    s.fanout[0] = s.param + (1 << 30)
    s.fanout[1] = s.fanout[0] + 16
    assert _encode([s], opt=L.OPT_SGD)[0] == L.ERR_ALIAS
    s.fanout[1] = s.fanout[0] + 4096 * 4
    assert _encode([s], opt=L.OPT_SGD)[0] == L.OK
    s.fanout[1] = s.param
    assert _encode([s], opt=L.OPT_SGD)[0] == L.ERR_ALIAS
    s = span()
    s.param = s.grads[0]                                        # ignored without an optimizer
    assert _encode([s], opt=L.OPT_NONE)[0] == L.OK


def test_launch_shape_follows_what_the_plan_is_encoded_for():
    """Launches with full statistics rows run 256-thread workgroups of 2 tiles (K <= 4) or 4 tiles, with
    similarity sums only 2 tiles for every K; plain launches with an optimizer 256 threads x 2 tiles for K > 4,
    128 threads x 2 tiles for SGD with fp32 gradients and K <= 4, 256 x 4 for the Adam kinds and K <= 4, else 256 x 2;
    aggregate-only launches 256 x 2 (K <= 4) or 256 x 4. A plan holds a chunk table per shape and serves launches of its own optimizer class only."""
    lib = L.lib()
    n = 10 * 4096
    def chunks(K, dtype, opt, gs=4):
        rc, blob, _ = _encode([_span(n, K=K, gs=gs, opt=True)], K=K, dtype=dtype, opt=opt)
        assert rc == L.OK
        return (lib.jabas_plan_chunks(blob.ctypes.data, 0), lib.jabas_plan_chunks(blob.ctypes.data, 1)), blob
    assert chunks(2, L.F32, L.OPT_SGD)[0] == (n // 1024, n // 2048)
    assert chunks(4, L.F32, L.OPT_SGD)[0] == (n // 1024, n // 2048)
    assert chunks(5, L.F32, L.OPT_SGD)[0] == (n // 2048, n // 4096)
    assert chunks(2, L.BF16, L.OPT_SGD, gs=2)[0] == (n // 2048, n // 2048)
    assert chunks(2, L.F32, L.OPT_ADAM)[0] == (n // 4096, n // 2048)
    assert chunks(8, L.BF16, L.OPT_ADAMW, gs=2)[0] == (n // 2048, n // 4096)
    assert chunks(2, L.F32, L.OPT_NONE)[0] == (n // 2048, n // 2048)
    assert chunks(8, L.F32, L.OPT_NONE)[0] == (n // 4096, n // 4096)
    _, blob8 = chunks(8, L.BF16, L.OPT_ADAMW, gs=2)
    assert lib.jabas_plan_chunks(blob8.ctypes.data, L.STATS_SIMILARITY) == n // 2048
    _, blob2 = chunks(2, L.F32, L.OPT_SGD)
    assert lib.jabas_plan_chunks(blob2.ctypes.data, L.STATS_SIMILARITY) == n // 2048
    # the level with pair products launches in the shape of the full rows and uses their chunk table
    assert lib.jabas_plan_chunks(blob2.ctypes.data, L.STATS_GRAM) == lib.jabas_plan_chunks(blob2.ctypes.data, L.STATS_FULL)
    assert lib.jabas_plan_chunks(blob2.ctypes.data, L.STATS_GRAM + 1) == L.ERR_OPT
    _, blob = chunks(2, L.F32, L.OPT_SGD)
    assert lib.jabas_plan_workspace_bytes(blob.ctypes.data) >= (n // 2048 + 1) * L.STATS_STRIDE * 8
    args = L.JabasStepArgs()
    args.K, args.grad_dtype, args.opt_kind = 2, L.F32, L.OPT_NONE
    assert lib.jabas_sync_fused(blob.ctypes.data, 0x1000, C.byref(args), None, None, 0, None) == L.ERR_PLAN
    args.opt_kind, args.n_groups = L.OPT_ADAM, 1
    args.groups[0].step = 1
    assert lib.jabas_sync_fused(blob.ctypes.data, 0x1000, C.byref(args), None, None, 0, None) == L.ERR_PLAN


def test_product_paths_fail_when_the_library_is_missing(tmp_path):
    """No CPU fallback: with no shared library the loader raises, and product entries given host
    tensors refuse them or raise the loader's error; none computes anything (checked in a child
    process so that this process keeps its loaded library)."""
    import subprocess
    import sys
    code = """
import torch
from jabas_amd import _lib, sync
from jabas_amd.local_sync import LocalBucketSync
g = [torch.ones(8), torch.ones(8)]
for name, call in (("lib", lambda: _lib.lib()),
                   ("aggregate", lambda: sync.aggregate(g, (1, 1))),
                   ("gradient_stats", lambda: sync.gradient_stats(g, (1, 1))),
                   ("plan", lambda: sync.SyncPlan([sync.SpanSpec(g, agg_out=torch.zeros(8))], _lib.OPT_NONE))):
    try:
        call()
    except (RuntimeError, ValueError) as exc:
        assert "no CPU fallback" in str(exc) or (name != "lib" and "must live on the GPU" in str(exc)), (name, exc)
    else:
        raise SystemExit(name + " did not raise")
print("all raised")
"""
    env = dict(os.environ, JABAS_SYNC_LIB=str(tmp_path / "absent.so"))
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, "-c", code], cwd=root, env=env, capture_output=True, text=True, timeout=300)
    assert res.returncode == 0 and "all raised" in res.stdout, res.stdout + res.stderr


def test_statistics_over_too_many_spans_are_refused_before_any_launch():
    """The finalize launch indexes spans by a grid dimension of 16 bits; a plan beyond that must be
    turned down with a status, not fail after the weights have moved."""
    lib = L.lib()
    n_span = 65536
    arr = (L.JabasSpan * n_span)()
    base = 0x7f0000000000
    for i in range(n_span):
        arr[i].grads[0] = base + 4096 * i
        arr[i].grads[1] = base + (1 << 36) + 4096 * i
        arr[i].agg_out = base + (2 << 36) + 4096 * i
        arr[i].numel = 8
    nbytes = lib.jabas_plan_bytes(arr, n_span, 0, L.F32)
    blob = np.zeros(nbytes // 8 + 1, dtype=np.uint64)
    assert lib.jabas_plan_encode(arr, n_span, None, 0, 2, L.F32, L.OPT_NONE, blob.ctypes.data, nbytes) == L.OK
    args = L.JabasStepArgs()
    args.K, args.grad_dtype, args.opt_kind, args.stats = 2, L.F32, L.OPT_NONE, 1
    args.weight[0] = args.weight[1] = 0.5
    args.half_id[1] = 1
    args.half_weight[0] = args.half_weight[1] = 1.0
    fake_dev = 0x7e0000000000
    ws_bytes = lib.jabas_plan_workspace_bytes(blob.ctypes.data)
    rc = lib.jabas_sync_fused(blob.ctypes.data, fake_dev, C.byref(args), fake_dev + (1 << 30), fake_dev + (2 << 30),
                              ws_bytes, None)
    assert rc == L.ERR_SIZE


def _shape_model(K, dtype, opt_class, stats):
    """(threads per workgroup, tiles per workgroup) as documented for the launch shapes."""
    if stats or opt_class == 0 or K > 4:
        block = 256
    else:
        block = 128 if (opt_class == 1 and dtype == L.F32) else 256
    if K > 4:
        tiles = 2 if stats == 2 else (4 if (stats or opt_class == 0) else 2)
    else:
        tiles = 4 if (not stats and opt_class >= 2) else 2
    return block, tiles


@pytest.mark.parametrize("seed", range(40))
def test_plan_encode_against_a_python_statement_of_the_chunking_rule(seed):
    """Random spans at random addresses: the encoder's verdict (OK / JABAS_ERR_ALIGN) and its chunk
    counts for both launch shapes must equal an independent statement of the rule: buffers must agree
    within 4 elements; the element grid starts at the 256-byte line when they agree within 64 elements,
    else at the 16-byte line; a span takes ceil(ceil((skew + numel) / tile) / tiles_per_workgroup) chunks."""
    rng = np.random.RandomState(seed)
    lib = L.lib()
    K = int(rng.randint(1, 17))
    dtype = L.BF16 if rng.rand() < 0.4 else L.F32
    opt = [L.OPT_NONE, L.OPT_SGD, L.OPT_ADAM, L.OPT_ADAMW][int(rng.randint(0, 4))]
    opt_class = {L.OPT_NONE: 0, L.OPT_SGD: 1, L.OPT_ADAM: 2, L.OPT_ADAMW: 2}[opt]
    gs = 2 if dtype == L.BF16 else 4
    n_span = int(rng.randint(1, 12))
    spans, want_chunks, want_rc = [], [0, 0, 0], L.OK
    stride = 1 << 36
    for i in range(n_span):
        numel = int(rng.choice([0, 1, 3, 500, 1023, 1024, 1025, 4096, 4097, 70000, 1 << 20])) + int(rng.randint(0, 3))
        mode = rng.rand()
        base_off = int(rng.randint(0, 64))
        n_buf = K + 4
        if mode < 0.6:
            offs = [base_off] * n_buf                                   # one place within the 256-byte line
        elif mode < 0.9:
            offs = [base_off % 4 + 4 * int(rng.randint(0, 16)) for _ in range(n_buf)]   # agree within 16 bytes only
        else:
            offs = [int(rng.randint(0, 64)) for _ in range(n_buf)]      # arbitrary
        s = L.JabasSpan()
        region = (2 * i + 1) * (1 << 28)                                # spans far apart: no overlap between buffers
        for k in range(K):
            s.grads[k] = 0x700000000000 + k * stride + region + offs[k] * gs
        s.agg_out = 0x700000000000 + 16 * stride + region + offs[K] * 4
        used = offs[:K + 1]
        if opt_class:
            s.param = 0x700000000000 + 17 * stride + region + offs[K + 1] * 4
            s.state1 = 0x700000000000 + 18 * stride + region + offs[K + 2] * 4
            used = offs[:K + 3]
            if opt_class == 2:
                s.state2 = 0x700000000000 + 19 * stride + region + offs[K + 3] * 4
                used = offs[:K + 4]
        s.numel = numel
        spans.append(s)
        if numel == 0:
            continue
        if len({o % 4 for o in used}) != 1:
            want_rc = L.ERR_ALIGN
            continue
        skew = used[0] if len(set(used)) == 1 else used[0] % 4
        for v, stats in enumerate((0, 1, 2)):                           # statistics level of the launch
            block, tiles = _shape_model(K, dtype, opt_class, stats)
            te = block * 4
            want_chunks[v] += -(-(-(-(skew + numel) // te)) // tiles)
    arr = (L.JabasSpan * n_span)(*spans)
    nbytes = lib.jabas_plan_bytes(arr, n_span, 0, dtype)
    blob = np.zeros(nbytes // 8 + 1, dtype=np.uint64)
    rc = lib.jabas_plan_encode(arr, n_span, None, 0, K, dtype, opt, blob.ctypes.data, nbytes)
    if want_rc != L.OK:
        assert rc == L.ERR_ALIGN
        return
    assert rc == L.OK, rc
    assert lib.jabas_plan_chunks(blob.ctypes.data, 0) == want_chunks[0]
    assert lib.jabas_plan_chunks(blob.ctypes.data, 1) == want_chunks[1]
    assert lib.jabas_plan_chunks(blob.ctypes.data, 2) == want_chunks[2]
    assert lib.jabas_plan_chunks(blob.ctypes.data, 3) == want_chunks[1]        # pair products: the shape of the full rows
    assert lib.jabas_plan_chunks(blob.ctypes.data, 4) == L.ERR_OPT


def test_rendezvous_calls_validate_their_arguments():
    """The meeting point's argument checks (no GPU: creating the object itself needs a device and is covered by
    the GPU tests)."""
    lib = L.lib()
    h = C.c_void_p()
    assert lib.jabas_rdv_create(0, C.byref(h)) == L.ERR_K and not h.value
    assert lib.jabas_rdv_create(L.MAX_K + 1, C.byref(h)) == L.ERR_K
    assert lib.jabas_rdv_create(2, None) == L.ERR_NULL
    args, span = L.JabasStepArgs(), L.JabasSpan()
    assert lib.jabas_rdv_publish(None, 0, 0, 0, None, None, C.byref(args), L.STATS_SIMILARITY) == L.ERR_NULL
    assert lib.jabas_rdv_set_bucket(None, 0, C.byref(span), None, None, None, 0, 0) == L.ERR_NULL
    assert lib.jabas_rdv_drop_bucket(None, 0) == L.ERR_NULL
    assert lib.jabas_rdv_reset(None) == L.ERR_NULL
    lib.jabas_rdv_destroy(None)
    assert b"rendezvous" in lib.jabas_status_string(L.ERR_STATE)


_HIP_RECORDER = r"""
#include "rendezvous.hip"
#include <string>
static std::string g_log;
static long g_events = 0;
extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = reinterpret_cast<hipEvent_t>(++g_events); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    g_log += "record " + std::to_string(reinterpret_cast<long>(e)) + " " + std::to_string(reinterpret_cast<long>(s)) + "\n"; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    g_log += "wait " + std::to_string(reinterpret_cast<long>(e)) + " " + std::to_string(reinterpret_cast<long>(s)) + "\n"; return hipSuccess; }
int jabas_sync_bucket(const JabasSpan*, const JabasBound*, const JabasStepArgs*, double*, void*, size_t, jabas_stream_t s) {
    g_log += "launch 0 " + std::to_string(reinterpret_cast<long>(s)) + "\n"; return 0; }
const char* take_log() { static std::string out; out = g_log; g_log.clear(); return out.c_str(); }
}
"""


def test_rendezvous_waits_for_every_hand_over_whatever_the_streams_are_called(tmp_path):
    """The host code of the meeting point over a recorder in place of the HIP runtime: the launch is preceded by a wait for the event
    of every hand-over, also where hand-overs, or one of them and the launch, name the same stream handle. The handle of a stream that
    was destroyed after its hand-over may name a new stream by then, and hipStreamPerThread (2) names one per thread. Only the null
    stream (0) is always the same one: the last event on it stands for the earlier ones."""
    import itertools
    import shutil
    import subprocess
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    src, so = tmp_path / "recorder.cpp", str(tmp_path / "recorder.so")
    src.write_text(_HIP_RECORDER)
    r = subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-Wno-attributes", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                        "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "jabas_amd", "csrc"), str(src), "-o", so,
                        "-Wl,-Bsymbolic"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    rec = C.CDLL(so)
    for name, (res, argtypes) in L.SIGNATURES.items():
        if name.startswith("jabas_rdv_"):
            getattr(rec, name).restype, getattr(rec, name).argtypes = res, argtypes
    rec.take_log.restype = C.c_char_p
    K, rdv, span, args = 3, C.c_void_p(), L.JabasSpan(), L.JabasStepArgs()
    args.K = K
    assert rec.jabas_rdv_create(K, C.byref(rdv)) == 0
    assert rec.jabas_rdv_set_bucket(rdv, 0, C.byref(span), None, None, None, 0, 0) == 0
    for streams in itertools.product((16, 32, 2, 0), repeat=K):
        for launch in (16, 64, 2, 0):
            for order in itertools.permutations(range(K)):
                codes = [rec.jabas_rdv_publish(rdv, k, 0, 0, streams[k], launch, C.byref(args), L.STATS_SIMILARITY) for k in order]
                assert codes == [L.RDV_WAITING] * (K - 1) + [L.RDV_LAUNCHED]
                log = [line.split() for line in rec.take_log().decode().splitlines()]
                assert log[-1] == ["launch", "0", str(launch)]
                recorded = {int(e): int(s) for what, e, s in log if what == "record"}
                # the completing hand-over on the launch's own stream, the same one in the same call, needs none
                needed = [k for k in order if not (k == order[-1] and streams[k] == launch)]
                assert recorded == {k + 1: streams[k] for k in needed}
                on_null = [k for k in needed if streams[k] == 0]
                waits = [k + 1 for k in needed if k not in on_null[:-1]]
                assert sorted(int(e) for what, e, s in log if what == "wait" and int(s) == launch) == sorted(waits)
                assert [what for what, _, _ in log] == ["record"] * len(needed) + ["wait"] * len(waits) + ["launch"]
    rec.jabas_rdv_destroy(rdv)


@pytest.mark.parametrize("K", (1, 2, 5, 16))
@pytest.mark.parametrize("half", (None, "blocks"))
def test_step_args_hold_every_field_in_its_place(K, half):
    """The arguments are written as packed bytes: every field of the struct read back, the weights against numpy's
    rounding, the first and the last parameter group, a step beyond 32 bits."""
    import torch
    from jabas_amd import sync
    batches = tuple(3 + 7 * k % 31 for k in range(K))
    half_id = None if half is None else [int(k >= K // 2) for k in range(K)]
    groups = [dict(lr=0.1 * (i + 1), weight_decay=1e-4 * i, step=2 ** 40 + i) for i in range(L.MAX_GROUPS)]
    opt = dict(kind="sgd", momentum=0.9, dampening=0.1, nesterov=True, betas=(0.8, 0.98), eps=1e-6, groups=groups)
    a = sync.make_step_args(batches, torch.bfloat16, stats="full", opt=opt, first_step=True, half_id=half_id, lr_scale=0.5,
                            accumulations=3)
    hid = [k % 2 for k in range(K)] if half_id is None else half_id
    tot = [3.0 * sum(b for b, h in zip(batches, hid) if h == x) for x in (0, 1)]
    w = np.array([b / (3.0 * sum(batches)) for b in batches]).astype(np.float32)
    hw = np.array([b / tot[h] for b, h in zip(batches, hid)]).astype(np.float32)
    zeros = [0] * (L.MAX_K - K)
    assert (a.K, a.grad_dtype, a.stats, a.opt_kind, a.n_groups) == (K, L.BF16, L.STATS_FULL, L.OPT_SGD, L.MAX_GROUPS)
    assert list(a.weight) == w.tolist() + zeros and list(a.half_weight) == hw.tolist() + zeros and list(a.half_id) == hid + zeros
    assert (a.first_step, a.nesterov, a.momentum, a.dampening) == (1, 1, 0.9, 0.1)
    assert (a.beta1, a.beta2, a.eps, a.grad_scale, a.scalars_dev) == (0.8, 0.98, 1e-6, None, None)
    assert [(g.lr, g.weight_decay, g.step) for g in a.groups] == [(g["lr"] * 0.5, g["weight_decay"], g["step"]) for g in groups]
    got = sync.batch_weights(batches, half_id, 3)
    assert [x.dtype for x in got] == [np.float32, np.uint8, np.float32]
    assert np.array_equal(got[0], w) and got[1].tolist() == hid and np.array_equal(got[2], hw)


def test_step_scalar_block_holds_the_constants_a_plain_call_derives():
    """jabas_step_scalars_encode is host code: its block is compared, slot by slot, with the constants derived
    here in Python doubles and rounded once to fp32 (what a Python float becomes as an fp32 kernel scalar)."""
    import torch
    from jabas_amd import sync
    lib = L.lib()
    f32 = lambda x: np.float32(x)
    opt = dict(kind="adamw", betas=(0.9, 0.999), eps=1e-8,
               groups=[dict(lr=5e-4, weight_decay=0.05, step=7), dict(lr=1e-3, weight_decay=0.0, step=3)])
    batches = (48, 32, 32, 16, 8)
    m = 2.5 ** 0.5
    args = sync.make_step_args(batches, torch.bfloat16, stats="similarity", opt=opt, lr_scale=m,
                               half_id=[0, 1, 1, 0, 1])
    block = np.zeros(L.STEP_SCALARS_BYTES, dtype=np.uint8)
    assert lib.jabas_step_scalars_encode(C.byref(args), block.ctypes.data, block.nbytes) == L.OK
    fl, u32 = block.view(np.float32), block.view(np.uint32)
    w, hid, hw = sync.batch_weights(batches, [0, 1, 1, 0, 1])
    assert np.array_equal(fl[0:5], w) and not fl[5:16].any()
    assert np.array_equal(fl[16:21], hw) and not fl[21:32].any()
    o = 32                                                       # OptDev: 7 floats, 4 flags
    assert fl[o + 2] == f32(0.9) and fl[o + 3] == f32(1.0 - 0.9)
    assert fl[o + 4] == f32(0.999) and fl[o + 5] == f32(1.0 - 0.999) and fl[o + 6] == f32(1e-8)
    assert list(u32[o + 7:o + 11]) == [0, 0, 0, 1]               # has_momentum, first_step, nesterov, adamw
    assert u32[o + 11] == 0b10110                                # half B: workers 1, 2, 4
    for i, g in enumerate(opt["groups"]):
        base = 44 + 8 * i
        lr = g["lr"] * m
        assert fl[base + 0] == f32(g["weight_decay"])
        assert fl[base + 1] == f32(-lr)
        assert fl[base + 2] == f32(1.0 - lr * g["weight_decay"])
        assert fl[base + 3] == f32(-(lr / (1.0 - 0.9 ** g["step"])))
        assert fl[base + 4] == f32((1.0 - 0.999 ** g["step"]) ** 0.5)
    assert not fl[44 + 16:].any()
    # SGD: momentum, dampening, the first-step flag
    sgd = dict(kind="sgd", momentum=0.9, dampening=0.1, nesterov=False, groups=[dict(lr=0.1, weight_decay=1e-4)])
    args = sync.make_step_args((2, 2), torch.float32, opt=sgd, first_step=True)
    assert lib.jabas_step_scalars_encode(C.byref(args), block.ctypes.data, block.nbytes) == L.OK
    assert fl[o] == f32(0.9) and fl[o + 1] == f32(1.0 - 0.1) and list(u32[o + 7:o + 11]) == [1, 1, 0, 0]
    assert fl[44 + 1] == f32(-0.1) and fl[44 + 3] == 0.0 and fl[44 + 4] == 1.0
    # argument checks
    assert lib.jabas_step_scalars_encode(None, block.ctypes.data, block.nbytes) == L.ERR_NULL
    assert lib.jabas_step_scalars_encode(C.byref(args), None, block.nbytes) == L.ERR_NULL
    assert lib.jabas_step_scalars_encode(C.byref(args), block.ctypes.data, L.STEP_SCALARS_BYTES - 1) == L.ERR_SIZE
    none = sync.make_step_args((2, 2), torch.float32)
    assert lib.jabas_step_scalars_encode(C.byref(none), block.ctypes.data, block.nbytes) == L.ERR_OPT
    adam0 = sync.make_step_args((2, 2), torch.float32, opt=dict(opt, groups=[dict(lr=1e-3, step=0)]))
    assert lib.jabas_step_scalars_encode(C.byref(adam0), block.ctypes.data, block.nbytes) == L.ERR_OPT
    assert lib.jabas_step_scalars_upload(None, 0x7f0000001000, None) == L.ERR_NULL
    assert lib.jabas_step_scalars_upload(C.byref(args), None, None) == L.ERR_NULL
    assert lib.jabas_step_scalars_upload(C.byref(args), 0x7f0000001004, None) == L.ERR_ALIGN
    assert lib.jabas_step_scalars_upload(C.byref(none), 0x7f0000001000, None) == L.ERR_OPT
    # a launch without optimizer has nothing that moves between steps: a block is refused, as is a misaligned one
    span = _span(5000)
    none.scalars_dev = 0x7f0000001000
    assert lib.jabas_sync_bucket(C.byref(span), None, C.byref(none), None, None, 0, None) == L.ERR_OPT
    span = _span(5000, opt=True)
    args.scalars_dev = 0x7f0000001008
    assert lib.jabas_sync_bucket(C.byref(span), None, C.byref(args), None, None, 0, None) == L.ERR_ALIGN


def test_rows_are_not_read_behind_a_recorder():
    """A launch through the C ABI is not in a recorded graph: under every recorder gram_from_stats has to stay torch
    operations, so that the recording answers for other rows too."""
    import torch
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from jabas_amd import sync

    seen = []

    def total(rows):
        seen.append(sync._watched())
        return sync.gram_from_stats(rows, 2)

    class Pass(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class PassBelow(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    rows, other = (torch.randn(3, L.STATS_STRIDE, dtype=torch.float64, generator=torch.Generator().manual_seed(i)) for i in (1, 2))
    want = total(other)
    assert seen == [False]
    recorded = [torch.jit.trace(total, rows, check_trace=False)]
    recorded += [make_fx(total, tracing_mode=mode)(rows) for mode in ("real", "fake", "symbolic")]
    assert seen[1:] == [True] * 4
    for graph in recorded:
        assert torch.equal(graph(other), want)
    del seen[:]
    for mode in (Pass(), PassBelow()):
        with mode:
            assert torch.equal(total(other), want)
    with torch.device("cpu"):                     # the mode of torch.set_default_device replaces no operation on rows
        assert torch.equal(total(other), want)
    assert seen == [True, True, False]


@pytest.mark.filterwarnings("ignore::UserWarning")
def test_rows_without_values_of_their_own_are_not_plain():
    """Tensors that are strided, contiguous and of the right type and size, but whose memory is not their values."""
    import torch
    from jabas_amd import sync

    rows = torch.randn(3, L.STATS_STRIDE, dtype=torch.float64, generator=torch.Generator().manual_seed(3))
    assert sync._plain(rows) and sync._plain(rows[1]) and sync._plain(rows.detach().requires_grad_())
    zeros = torch._efficientzerotensor(3, L.STATS_STRIDE, dtype=torch.float64)
    negated = torch._neg_view(rows)
    nested = torch.nested.nested_tensor([rows, rows])
    functional = torch._to_functional_tensor(rows)
    assert not any(sync._plain(t) for t in (zeros, negated, nested, functional, torch.nn.Parameter(rows)))
    torch.func.vmap(lambda r: torch.tensor(0.0) if not sync._plain(r) else 1 / 0)(rows)
    assert torch.equal(sync.gram_from_stats(zeros, 2), torch.zeros(2, 2, dtype=torch.float64))
    assert torch.equal(sync.gram_from_stats(negated, 2), -sync.gram_from_stats(rows, 2))
    with pytest.raises(RuntimeError):
        sync.gram_from_stats(nested, 2)


def test_library_without_an_entry_point_is_refused_by_name(monkeypatch):
    """A library of an older build lacks an entry point that the package calls."""
    monkeypatch.setattr(L, "_lib", None)
    monkeypatch.setitem(L.SIGNATURES, "jabas_of_a_later_build", (C.c_int, []))
    with pytest.raises(RuntimeError, match="jabas_of_a_later_build.*build it again"):
        L.lib()
    assert L._lib is None


def test_library_of_an_older_version_is_refused_by_its_version(monkeypatch):
    """An older library may have every entry point and still not know a flag that the package passes."""
    monkeypatch.setattr(L, "_lib", None)
    monkeypatch.setattr(L, "MIN_VERSION", (99, 0))
    with pytest.raises(RuntimeError, match="older than 99.0.*build it again"):
        L.lib()
    assert L._lib is None
