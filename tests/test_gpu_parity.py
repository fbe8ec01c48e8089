"""GPU parity: the HIP path, called through the C ABI (ctypes), against the CPU oracle on
the same seeded inputs. Bars (from the path's specification):
  aggregate            bit-exact (fp32 and bf16 inputs)
  statistics           1e-6 relative (fp32 inputs), 1e-2 relative (bf16 inputs)
  updated weights/state 1e-6 relative (plus an absolute floor of a few ulp of the operands,
                       because m and buf are sums that may cancel)
The optimizer checks additionally report how many elements are bit-identical.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

BATCHES = {1: (32,), 2: (32, 32), 3: (4, 2, 2), 4: (48, 32, 32, 16), 5: (5, 4, 3, 2, 1),
           6: (7, 7, 5, 3, 2, 1), 7: (64, 56, 48, 40, 32, 24, 16), 8: tuple(range(64, 0, -8)),
           9: (9, 8, 7, 6, 5, 4, 3, 2, 1), 10: (16,) * 10, 11: tuple(range(11, 0, -1)), 12: (32, 16, 8) * 4,
           13: tuple(range(1, 14)), 14: (3, 5) * 7, 15: tuple(range(30, 0, -2)), 16: tuple(range(64, 0, -4))}

SGD = dict(kind="sgd", momentum=0.9, dampening=0.0, nesterov=False,
           groups=[dict(lr=0.1, weight_decay=0.0), dict(lr=0.1, weight_decay=1e-4)])
ADAMW = dict(kind="adamw", betas=(0.9, 0.999), eps=1e-8,
             groups=[dict(lr=5e-4, weight_decay=0.0), dict(lr=5e-4, weight_decay=0.05)])
ADAM = dict(kind="adam", betas=(0.9, 0.999), eps=1e-8, groups=[dict(lr=2e-3, weight_decay=0.0),
                                                                dict(lr=2e-3, weight_decay=1e-2)])


def _bits(t):
    return t.detach().cpu().contiguous().view(torch.int32)


def _host_grads(K, n, seed, std=1e-3, dtype=torch.float32):
    out = []
    for k in range(K):
        g = torch.Generator().manual_seed(1234 + 17 * seed + k)
        out.append((torch.randn(n, generator=g) * std).to(dtype))
    return out


def _host_state(n, seed, scale=0.05):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(n, generator=g) * scale


def _dev(t, gpu, skew=0):
    """Device copy of t placed `skew` elements into a 256-byte aligned allocation."""
    buf = torch.zeros(t.numel() + 128, dtype=t.dtype, device=gpu)
    view = buf[skew:skew + t.numel()]
    view.copy_(t)
    return view


def _close(got, want, rtol, atol):
    got, want = got.detach().cpu().double(), want.detach().cpu().double()
    err = (got - want).abs()
    ok = err <= rtol * want.abs() + atol
    return bool(ok.all()), float(err.max()) if err.numel() else 0.0


def _same_bits(a, b):
    a, b = _bits(a), _bits(b)
    return int((a == b).sum()), a.numel()


# ---------------------------------------------------------------------------- aggregate
@pytest.mark.parametrize("K", range(1, 17))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_aggregate_bit_exact(gpu, K, dtype):
    from jabas_amd import sync
    for n, skew in ((1, 0), (3, 1), (1023, 0), (1024, 2), (1025, 3), (4099, 0), (262144 + 77, 0), (1 << 20, 3),
                    (4099, 37), (70001, 63), (5, 61)):
        print(f"aggregate K={K} {dtype} n={n} skew={skew}", flush=True)
        hg = _host_grads(K, n, K + n % 7, dtype=dtype)
        dg = [_dev(t, gpu, skew) for t in hg]
        out = _dev(torch.zeros(n), gpu, skew)
        sync.aggregate(dg, BATCHES[K], out=out)
        torch.cuda.synchronize()
        want = O.aggregate(hg, BATCHES[K])
        assert torch.equal(_bits(out), _bits(want)), f"K={K} n={n} skew={skew}"


def test_aggregate_in_place_into_vsw0_bucket(gpu):
    from jabas_amd import sync
    K, n = 4, 50001
    hg = _host_grads(K, n, 3)
    dg = [_dev(t, gpu) for t in hg]
    sync.aggregate(dg, BATCHES[K], out=dg[0])
    torch.cuda.synchronize()
    assert torch.equal(_bits(dg[0]), _bits(O.aggregate(hg, BATCHES[K])))
    for k in range(1, K):
        assert torch.equal(_bits(dg[k]), _bits(hg[k]))        # other workers' buckets untouched


def test_aggregate_keeps_zero_rows_exactly_zero(gpu):
    from jabas_amd import sync
    K, rows, cols = 4, 512, 1024
    mask = torch.rand(rows, generator=torch.Generator().manual_seed(0)) < 0.1
    hg = [torch.where(mask[:, None], t.view(rows, cols), torch.zeros(())).reshape(-1)
          for t in _host_grads(K, rows * cols, 5)]
    out = sync.aggregate([_dev(t, gpu) for t in hg], BATCHES[K])
    torch.cuda.synchronize()
    got = out.cpu().view(rows, cols)
    assert torch.all(got[~mask].view(torch.int32) == 0)
    assert torch.equal(_bits(out), _bits(O.aggregate(hg, BATCHES[K])))


# --------------------------------------------------------------------------- statistics
@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 8, 9, 12, 13, 16])
@pytest.mark.parametrize("dtype,rtol", [(torch.float32, 1e-6), (torch.bfloat16, 1e-2)])
def test_stats_row(gpu, K, dtype, rtol):
    from jabas_amd import sync
    for n, skew in ((5, 0), (4099, 1), (300007, 0), (1 << 21, 2), (4099, 45), (3, 63)):
        print(f"stats K={K} {dtype} n={n} skew={skew}", flush=True)
        hg = _host_grads(K, n, 20 + K, std=5e-4, dtype=dtype)
        row = sync.gradient_stats([_dev(t, gpu, skew) for t in hg], BATCHES[K])
        torch.cuda.synchronize()
        want = O.stats(hg, BATCHES[K])
        got = row.cpu()
        ok, err = _close(got[:4 + K], want[:4 + K], rtol, 1e-30)
        assert ok, f"K={K} n={n}: {got} vs {want}"
        assert torch.count_nonzero(got[4 + K:]) == 0
        # fp64 accumulation (fp32 gradients): in fact far inside the bar; bf16 gradients keep fp32 partial
        # sums over a thread's chunk (products of bf16 values are exact in fp32) and fp64 from there on
        tight = 1e-11 if dtype == torch.float32 else 1e-5
        assert _close(got[1:4 + K], want[1:4 + K], tight, 1e-30)[0], f"K={K} n={n}: {got} vs {want}"
        # the dot product of the halves cancels: its error is measured against |g_A| |g_B| (the cosine's scale)
        assert abs(float(got[0] - want[0])) <= tight * float(torch.sqrt(want[1] * want[2])) + 1e-30


@pytest.mark.parametrize("K", [1, 2, 4, 5, 8, 11, 16])
@pytest.mark.parametrize("dtype,rtol", [(torch.float32, 1e-11), (torch.bfloat16, 1e-5)])
def test_similarity_level_rows(gpu, K, dtype, rtol):
    """Statistics level 2: the four sums of the halves and of the aggregate, per-VSW slots zero; the
    aggregate and an optimizer step in the same launch stay bit-exact."""
    from jabas_amd import sync, _lib as L
    for n, skew in ((5, 0), (4099, 1), (300007, 0), (1 << 21, 2), (4099, 45)):
        print(f"similarity stats K={K} {dtype} n={n} skew={skew}", flush=True)
        hg = _host_grads(K, n, 60 + K, std=5e-4, dtype=dtype)
        dg = [_dev(t, gpu, skew) for t in hg]
        p_h = torch.randn(n, generator=torch.Generator().manual_seed(3)) * 0.05
        m_h, v_h = torch.zeros(n), torch.zeros(n)
        p_d, m_d, v_d, out = _dev(p_h, gpu, skew), _dev(m_h, gpu, skew), _dev(v_h, gpu, skew), _dev(torch.zeros(n), gpu, skew)
        span = sync.SpanSpec(dg, agg_out=out, param=p_d, state1=m_d, state2=v_d)
        args = sync.make_step_args(BATCHES[K], dtype, stats="similarity", opt=ADAMW, step=1)
        assert args.stats == L.STATS_SIMILARITY
        row = sync.sync_bucket(span, args).cpu()
        torch.cuda.synchronize()
        agg_h, rows_h = O.sync_step(hg, BATCHES[K], [(0, n, ())], ADAMW, p_h, m_h, v_h, step=1, want_stats=True)
        assert _close(row[1:4], rows_h[0][1:4], rtol, 1e-30)[0], f"K={K} n={n}: {row[:4]} vs {rows_h[0][:4]}"
        assert abs(float(row[0] - rows_h[0][0])) <= rtol * float(torch.sqrt(rows_h[0][1] * rows_h[0][2])) + 1e-30
        assert torch.count_nonzero(row[4:]) == 0
        assert torch.equal(_bits(out), _bits(agg_h)) and torch.equal(_bits(p_d), _bits(p_h))
        assert torch.equal(_bits(m_d), _bits(m_h)) and torch.equal(_bits(v_d), _bits(v_h))


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("dtype,rtol", [(torch.float32, 1e-11), (torch.bfloat16, 1e-5)])
@pytest.mark.parametrize("opt", [None, SGD, ADAMW], ids=["aggregate", "sgd", "adamw"])
def test_gram_level_rows(gpu, K, dtype, rtol, opt):
    """Statistics level 3: the full row plus the product of every pair of workers, out of the launch that
    aggregates and steps (up to eight workers). Row against the float64
    oracle (the four sums and the norms as at the full level, the pair slots against the Gram matrix), pair order
    as the header's JABAS_STAT_PAIR, slots beyond the row zero, and the aggregate and the optimizer step of the
    same launch bit-exact."""
    from jabas_amd import sync, _lib as L
    for n, skew in ((5, 0), (4099, 1), (300007, 0), (1 << 21, 2), (4099, 45)):
        print(f"gram level K={K} {dtype} n={n} skew={skew}", flush=True)
        hg = _host_grads(K, n, 90 + K, std=5e-4, dtype=dtype)
        dg = [_dev(t, gpu, skew) for t in hg]
        out = _dev(torch.zeros(n), gpu, skew)
        p_h = torch.randn(n, generator=torch.Generator().manual_seed(3)) * 0.05
        m_h, v_h = torch.zeros(n), torch.zeros(n)
        if opt is None:
            span = sync.SpanSpec(dg, agg_out=out)
        else:
            p_d, m_d, v_d = _dev(p_h, gpu, skew), _dev(m_h, gpu, skew), _dev(v_h, gpu, skew)
            span = sync.SpanSpec(dg, agg_out=out, param=p_d, state1=m_d, state2=v_d if opt is ADAMW else None)
        args = sync.make_step_args(BATCHES[K], dtype, stats="gram", opt=opt, step=1, first_step=True)
        assert args.stats == L.STATS_GRAM
        row = sync.sync_bucket(span, args).cpu()
        torch.cuda.synchronize()
        want = O.stats(hg, BATCHES[K])
        G = O.gram(hg)
        width = 4 + K + K * (K - 1) // 2
        assert _close(row[1:4 + K], want[1:4 + K], rtol, 1e-30)[0], f"K={K} n={n}: {row} vs {want}"
        assert abs(float(row[0] - want[0])) <= rtol * float(torch.sqrt(want[1] * want[2])) + 1e-30
        slot = 4 + K
        for a in range(K):
            for b in range(a + 1, K):
                assert L.stat_pair(K, a, b) == slot
                # a pair product cancels: its error is measured against |g_a| |g_b|
                assert abs(float(row[slot] - G[a, b])) <= rtol * float(torch.sqrt(G[a, a] * G[b, b])) + 1e-30, (K, n, a, b)
                slot += 1
        assert slot == width and torch.count_nonzero(row[width:]) == 0
        got = sync.gram_from_stats(row, K)
        assert torch.equal(got, got.t()) and torch.equal(torch.diagonal(got), row[4:4 + K])
        if opt is None:
            assert torch.equal(_bits(out), _bits(O.aggregate(hg, BATCHES[K])))
        else:
            agg_h, _ = O.sync_step(hg, BATCHES[K], [(0, n, ())], opt, p_h, m_h, v_h if opt is ADAMW else None,
                                   step=1, first_step=True, want_stats=False)
            assert torch.equal(_bits(out), _bits(agg_h)) and torch.equal(_bits(p_d), _bits(p_h))
            assert torch.equal(_bits(m_d), _bits(m_h))
            if opt is ADAMW:
                assert torch.equal(_bits(v_d), _bits(v_h))


def test_gram_level_limits_and_the_separate_pass(gpu):
    """More than STATS_GRAM_MAX_K workers are refused before anything is launched; the fused sums agree with
    jabas_gram's own pass over the same buffers (fp32 gradients: both exact products and fp64 sums)."""
    from jabas_amd import sync, _lib as L
    n = 1_000_003
    hg = _host_grads(9, n, 97)
    dg = [_dev(t, gpu, 3) for t in hg]
    out = _dev(torch.zeros(n), gpu, 3)
    before = out.clone()
    with pytest.raises(L.JabasSyncError) as e:
        sync.sync_bucket(sync.SpanSpec(dg, agg_out=out), sync.make_step_args(BATCHES[9], torch.float32, stats="gram"))
    assert e.value.status == L.ERR_K
    assert torch.equal(out, before)
    with pytest.raises(ValueError):
        sync.gram_from_stats(torch.zeros(L.STATS_STRIDE, dtype=torch.float64), 9)
    # the entry point that allocates nothing stops at five workers (its array holds rows of 4 + 16 sums)
    row8 = sync.sync_bucket(sync.SpanSpec(dg[:8], agg_out=out), sync.make_step_args(BATCHES[8], torch.float32, stats="gram"))
    fused8, apart8 = sync.gram_from_stats(row8, 8).cpu(), sync.gram(dg[:8]).cpu()
    scale8 = torch.sqrt(torch.outer(torch.diagonal(apart8), torch.diagonal(apart8)))
    assert bool(((fused8 - apart8).abs() <= 1e-12 * scale8).all())
    hb = _host_grads(9, 70001, 98, std=5e-4, dtype=torch.bfloat16)
    db = [_dev(t, gpu, 3) for t in hb]
    outb = _dev(torch.zeros(70001), gpu, 3)
    with pytest.raises(L.JabasSyncError) as e:
        sync.sync_bucket(sync.SpanSpec(db, agg_out=outb), sync.make_step_args(BATCHES[9], torch.bfloat16, stats="gram"))
    assert e.value.status == L.ERR_K and torch.count_nonzero(outb) == 0
    with pytest.raises(L.JabasSyncError) as e:
        sync.sync_bucket_static(sync.SpanSpec(db[:8], agg_out=outb), sync.make_step_args(BATCHES[8], torch.bfloat16, stats="gram"),
                                stats_out=torch.zeros(L.STATS_STRIDE, dtype=torch.float64, device=gpu))
    assert e.value.status == L.ERR_SIZE and torch.count_nonzero(outb) == 0
    args5 = sync.make_step_args(BATCHES[5], torch.float32, stats="gram")
    row5 = sync.sync_bucket(sync.SpanSpec(dg[:5], agg_out=out), args5).clone()
    row5s = sync.sync_bucket_static(sync.SpanSpec(dg[:5], agg_out=out), args5,
                                    stats_out=torch.zeros(L.STATS_STRIDE, dtype=torch.float64, device=gpu))
    assert torch.equal(row5.cpu().view(torch.int64), row5s.cpu().view(torch.int64)) and float(row5[4 + 5 + 9]) != 0.0
    rowb = sync.sync_bucket(sync.SpanSpec(db[:8], agg_out=outb), sync.make_step_args(BATCHES[8], torch.bfloat16, stats="gram"))
    fusedb, apartb = sync.gram_from_stats(rowb, 8).cpu(), sync.gram(db[:8]).cpu()
    scaleb = torch.sqrt(torch.outer(torch.diagonal(apartb), torch.diagonal(apartb)))
    assert bool(((fusedb - apartb).abs() <= 2e-5 * scaleb).all())
    row = sync.sync_bucket(sync.SpanSpec(dg[:4], agg_out=out), sync.make_step_args(BATCHES[4], torch.float32, stats="gram"))
    fused = sync.gram_from_stats(row, 4).cpu()
    apart = sync.gram(dg[:4]).cpu()
    scale = torch.sqrt(torch.outer(torch.diagonal(apart), torch.diagonal(apart)))
    assert bool(((fused - apart).abs() <= 1e-12 * scale).all())
    again = sync.sync_bucket(sync.SpanSpec(dg[:4], agg_out=out), sync.make_step_args(BATCHES[4], torch.float32, stats="gram"))
    assert torch.equal(again.cpu().view(torch.int64), row.cpu().view(torch.int64))


def test_stats_run_to_run_deterministic(gpu):
    from jabas_amd import sync
    hg = _host_grads(4, 3_000_001, 41)
    dg = [_dev(t, gpu) for t in hg]
    a = sync.gradient_stats(dg, BATCHES[4]).cpu().clone()
    for _ in range(3):
        b = sync.gradient_stats(dg, BATCHES[4]).cpu()
        assert torch.equal(a.view(torch.int64), b.view(torch.int64))


def test_stats_cosine_identities(gpu):
    from jabas_amd import sync
    g0 = _dev(_host_grads(1, 100003, 43)[0], gpu)
    assert sync.cosine_from_stats(sync.gradient_stats([g0, g0.clone()], (8, 8))) == pytest.approx(1.0, abs=1e-12)
    assert sync.cosine_from_stats(sync.gradient_stats([g0, -g0], (8, 8))) == pytest.approx(-1.0, abs=1e-12)
    z = torch.zeros(1000, device=gpu)
    assert sync.cosine_from_stats(sync.gradient_stats([z, z], (1, 1))) == 0.0


@pytest.mark.parametrize("K", list(range(1, 17)))
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gram(gpu, K, dtype):
    """fp32 gradients and up to seven bf16 workers: exact fp64 products and fp64 sums on the vector ALU or the fp64 matrix
    cores, 1e-11 against the float64 oracle. More bf16 workers run on the bf16 matrix cores: exact products, fp32 running
    sums moved into fp64 every few thousand elements, 5e-6 of |g_a| |g_b| against a bar of 1e-2."""
    from jabas_amd import sync
    for n, skew in ((7, 0), (100003, 2), (1 << 20, 0), (100003, 61), (3_000_001, 5)):
        hg = _host_grads(K, n, 30 + K, dtype=dtype)
        G = sync.gram([_dev(t, gpu, skew) for t in hg]).cpu()
        want = O.gram(hg)
        # off-diagonal entries cancel: their error is measured against |g_a| |g_b|
        scale = torch.sqrt(torch.outer(torch.diagonal(want), torch.diagonal(want)))
        off, diag = (1e-12, 1e-11) if dtype == torch.float32 or K <= 7 else (5e-6, 5e-6)
        assert bool(((G - want).abs() <= off * scale + 1e-30).all()), f"K={K} n={n}"
        assert _close(torch.diagonal(G), torch.diagonal(want), diag, 1e-30)[0], f"K={K} n={n}"
        assert torch.equal(G, G.t())


@pytest.mark.parametrize("dtype,K", [(torch.float32, 1), (torch.float32, 3), (torch.float32, 4), (torch.float32, 5),
                                     (torch.float32, 6), (torch.float32, 8), (torch.float32, 12), (torch.float32, 13),
                                     (torch.float32, 16), (torch.bfloat16, 2), (torch.bfloat16, 5), (torch.bfloat16, 7)])
def test_gram_at_the_edges_of_runs_and_routes(gpu, dtype, K):
    """One element, one less and one more than a run of a wave (128 elements), starts inside a vector; then a full grid: one run per
    wave of 512 workgroups (2048 waves; fp32 matrix cores below 2**21 elements, with two sums, whose runs alternate) and of 1024,
    one vector more than a grid of 2**18 threads holds at a time, a third and a fourth run of the first wave, with and without an
    end; both sides of the line at 2**21 elements and a fifth round of runs beyond it; and a worker with infinities and NaN reaches no product but its own (the first worker's
    values stand in for the missing ones of a group of four). fp64 sums of n exact products in any order: n * 2**-53 *
    |g_a| |g_b| apart at most."""
    from jabas_amd import sync
    grid, far = 1024 * 1024, 1 << 21
    sizes = [(1, 0), (1, 3), (127, 0), (128, 0), (129, 1), (253, 3), (257, 0), (2048 * 128 + 1, 0), (2049 * 128 + 3, 3),
             (4096 * 128 + 1, 0), (4097 * 128 + 3, 3), (grid + 1, 0), (grid + 128, 0), (grid + 129, 3), (grid + 4097 * 128 + 3, 1)]
    if dtype == torch.float32 and K > 5:
        sizes += [(far - 1, 0), (far - 1, 1), (far, 0), (far + 1, 3), (far + 4096 * 128 + 1, 0), (far + 4097 * 128 + 3, 3)]
    for n, skew in sizes:
        hg = _host_grads(K, n, 70 + K, dtype=dtype)
        G = sync.gram([_dev(t, gpu, skew) for t in hg]).cpu()
        wide = torch.stack([t.double() for t in hg])
        norm = wide.norm(dim=1)
        bound = 2.0 * (n + 2) * 2.0 ** -53 * torch.outer(norm, norm)
        assert bool(((G - wide @ wide.t()).abs() <= bound).all()), f"K={K} n={n} skew={skew}"
    hg = _host_grads(K, 5003, 90 + K, dtype=dtype)
    clean = sync.gram([_dev(t, gpu, 0) for t in hg])
    for w in sorted({0, 1, K - 1} if K > 1 else ()):
        bad = [t.clone() for t in hg]
        bad[w][17], bad[w][4000] = float("inf"), float("nan")
        G = sync.gram([_dev(t, gpu, 0) for t in bad])
        keep = [k for k in range(K) if k != w]
        assert torch.equal(G[keep][:, keep], clean[keep][:, keep])
        assert bool(G[w].isnan().all()) and bool(G[:, w].isnan().all())


@pytest.mark.parametrize("dtype,K", [(torch.float32, 1), (torch.float32, 2), (torch.float32, 5), (torch.float32, 6), (torch.float32, 9),
                                     (torch.float32, 16), (torch.bfloat16, 7), (torch.bfloat16, 8), (torch.bfloat16, 11), (torch.bfloat16, 13)])
def test_gram_sum_of_the_workgroup_rows(gpu, dtype, K):
    """A workgroup of the finalize holds four entries and takes the rows in classes of 256: one row, one class short, full and
    one over, two rows per class, and three and four where the launch has more than 512 workgroups (fp32 of six workers and more
    only from 2**21 elements on); scratch that starts as NaN tells how many rows there were. Every entry of the 16 x 16 result is written: the product, mirrored, or zero
    beyond the workers. Integers of at most 3 in size: every product and sum is exact, in fp32 as in fp64."""
    from jabas_amd import sync, _lib as L
    ws = torch.empty(1024 * L.GRAM_STRIDE, dtype=torch.float64, device=gpu)
    sizes = [(rows, rows * 1024 - 5) for rows in (1, 2, 255, 256, 257, 511, 512)]
    if dtype == torch.float32 and K > 5:
        sizes.append((1024, (1 << 21) + 5))
    elif K < (3 if dtype == torch.float32 else 13):
        sizes += [(rows, rows * 1024 - 5) for rows in (767, 769, 1023, 1024)]
    for rows, n in sizes:
        gen = torch.Generator().manual_seed(rows + K)
        hg = [torch.randint(-3, 4, (n,), generator=gen).to(dtype) for _ in range(K)]
        dg = [t.to(gpu) for t in hg]
        out = torch.full((L.GRAM_STRIDE,), float("nan"), dtype=torch.float64, device=gpu)
        ws.fill_(float("nan"))
        L.check(L.lib().jabas_gram(sync._ptr_array(dg), K, sync.grad_dtype_code(dtype), n, out.data_ptr(), ws.data_ptr(),
                                   ws.numel() * 8, sync._stream_ptr()), "jabas_gram")
        wide = torch.stack([t.double() for t in hg])
        want = torch.zeros(L.GRAM_MAX_K, L.GRAM_MAX_K, dtype=torch.float64)
        want[:K, :K] = wide @ wide.t()
        assert torch.equal(out.cpu().view(L.GRAM_MAX_K, L.GRAM_MAX_K), want), f"K={K} rows={rows}"
        assert int((~ws.view(1024, L.GRAM_STRIDE)[:, 0].isnan()).sum()) == rows


@pytest.mark.parametrize("K", [8, 9, 12, 13, 16])
def test_gram_bf16_runs_and_ends(gpu, K):
    """The bf16 matrix-core kernels take whole runs of a wave (256 elements, 512 from 2**21 elements on) in their loop and the
    span's ends after it: one element, one off a vector, a block and a run, starts inside a vector, a block and a line; one
    run per wave of 512 and of 1024 workgroups, one more, a second round with and without an end; and both sides of the
    line between the two shapes, by elements and by where the span starts. Integers of at most 3 in size: every product and
    sum is exact."""
    from jabas_amd import sync
    run, far = 256, 1 << 21
    for n, skew in ((1, 0), (1, 3), (7, 1), (9, 61), (127, 0), (129, 2), (run - 1, 0), (run, 0), (run, 1), (run + 1, 3), (2 * run, 61),
                    (3 * run - 3, 3), (2048 * run, 0), (2048 * run, 1), (2049 * run + 5, 2), (4096 * run - 1, 0), (4097 * run + 9, 61),
                    (far - 1, 0), (far - 1, 1), (far, 0), (far + 1, 3), (far + 512, 0), (far + 513, 2), (3 * far + 517, 61)):
        gen = torch.Generator().manual_seed(n + K)
        hg = [torch.randint(-3, 4, (n,), generator=gen, dtype=torch.int8).to(torch.bfloat16) for _ in range(K)]
        G = sync.gram([_dev(t, gpu, skew) for t in hg]).cpu()
        wide = torch.stack([t.double() for t in hg])
        assert torch.equal(G, wide @ wide.t()), f"K={K} n={n} skew={skew}"


@pytest.mark.parametrize("n", [(1 << 26) - 70, 1 << 26, (1 << 26) + 77, 3 * (1 << 27) + 77])
def test_gram_bf16_four_groups_of_very_long_spans(gpu, n):
    """Both sides of the line at 2**26 elements beyond which the kernel of thirteen and more bf16 workers takes the span's ends in
    its loop; and a span whose waves have 192 runs, so that their sums move to fp64 once on the way (after 128) and once at the
    end. Integers: exact."""
    from jabas_amd import sync
    gen = torch.Generator(device=gpu).manual_seed(n)
    flat = [torch.randint(-3, 4, (n,), generator=gen, device=gpu, dtype=torch.int8).to(torch.bfloat16) for _ in range(3)]
    grads = [flat[k % 3][:n] for k in range(13)]                     # thirteen workers over three buffers
    want = torch.zeros(3, 3, dtype=torch.float64, device=gpu)
    for i in range(3):
        for j in range(3):
            want[i, j] = (flat[i][:n].float() * flat[j][:n].float()).double().sum()      # |product| <= 9: exact
    index = [k % 3 for k in range(13)]
    assert torch.equal(sync.gram(grads).cpu(), want.cpu()[index][:, index])


def test_gram_limits_and_determinism(gpu):
    from jabas_amd import sync, _lib as L
    g = [torch.zeros(4096, device=gpu) for _ in range(17)]
    with pytest.raises(L.JabasSyncError) as e:
        sync.gram(g)
    assert e.value.status == L.ERR_K
    hg = _host_grads(11, 2_000_003, 77)
    dg = [_dev(t, gpu, 3) for t in hg]
    a = sync.gram(dg).cpu().clone()
    for _ in range(3):
        assert torch.equal(sync.gram(dg).cpu().view(torch.int64), a.view(torch.int64))
    # the diagonal is the per-worker norm row of the statistics kernel's full level
    row = sync.gradient_stats(dg, BATCHES[11]).cpu()
    assert torch.allclose(torch.diagonal(a), row[4:4 + 11], rtol=1e-12, atol=0.0)
    # a workspace of exactly the rows the call needs: the same values
    small = torch.empty(1024 * L.GRAM_STRIDE, dtype=torch.float64, device=gpu)
    b = sync.gram(dg, workspace=small).cpu()
    assert torch.allclose(a, b, rtol=1e-13, atol=1e-24)
    with pytest.raises(L.JabasSyncError) as e:
        sync.gram(dg, workspace=small[:1000 * L.GRAM_STRIDE])
    assert e.value.status == L.ERR_WORKSPACE
    hb = _host_grads(13, 1_000_003, 78, dtype=torch.bfloat16)
    db = [_dev(t, gpu, 1) for t in hb]
    a = sync.gram(db).cpu().clone()
    for _ in range(3):
        assert torch.equal(sync.gram(db).cpu().view(torch.int64), a.view(torch.int64))


# ---------------------------------------------------------------------------- optimizer
@pytest.mark.parametrize("hp", [
    dict(lr=0.1, weight_decay=1e-4, momentum=0.9, dampening=0.0, nesterov=False),
    dict(lr=0.05, weight_decay=5e-4, momentum=0.8, dampening=0.0, nesterov=True),
    dict(lr=0.05, weight_decay=1e-3, momentum=0.7, dampening=0.3, nesterov=False),
    dict(lr=0.3, weight_decay=1e-2, momentum=0.0, dampening=0.0, nesterov=False),
])
def test_sgd_steps(gpu, hp):
    from jabas_amd import sync
    n, steps = 70001, 4
    p_h, buf_h = _host_state(n, 1), torch.zeros(n)
    p_d, buf_d = _dev(p_h, gpu), _dev(buf_h, gpu)
    for s in range(steps):
        g = _host_grads(1, n, 50 + s)[0]
        O.sgd_step(p_h, g, buf_h, first_step=(s == 0), **hp)
        sync.sgd_step(_dev(g, gpu), p_d, buf_d if hp["momentum"] else None, first_step=(s == 0), **hp)
        torch.cuda.synchronize()
        ok, err = _close(p_d, p_h, 1e-6, 1e-9)
        assert ok, f"step {s}: max err {err}"
        if hp["momentum"]:
            assert _close(buf_d, buf_h, 1e-6, 2e-9)[0]
    same, tot = _same_bits(p_d, p_h)
    print(f"sgd {hp}: {same}/{tot} weights bit-identical after {steps} steps")
    assert same == tot


@pytest.mark.parametrize("hp", [
    dict(lr=5e-4, weight_decay=0.05, betas=(0.9, 0.999), eps=1e-8, adamw=True),
    dict(lr=2e-3, weight_decay=0.0, betas=(0.9, 0.999), eps=1e-8, adamw=False),
    dict(lr=1e-3, weight_decay=1e-2, betas=(0.8, 0.99), eps=1e-6, adamw=False),
])
def test_adam_steps(gpu, hp):
    from jabas_amd import sync
    n, steps = 70001, 5
    p_h, m_h, v_h = _host_state(n, 3), torch.zeros(n), torch.zeros(n)
    p_d, m_d, v_d = _dev(p_h, gpu), _dev(m_h, gpu), _dev(v_h, gpu)
    for s in range(1, steps + 1):
        g = _host_grads(1, n, 70 + s, std=5e-4)[0]
        O.adam_step(p_h, g, m_h, v_h, step=s, **hp)
        sync.adam_step(_dev(g, gpu), p_d, m_d, v_d, step=s, **hp)
        torch.cuda.synchronize()
        assert _close(p_d, p_h, 1e-6, 1e-9)[0], f"step {s}"
        assert _close(m_d, m_h, 1e-6, 2e-10)[0], f"step {s}"
        assert _close(v_d, v_h, 1e-6, 1e-16)[0], f"step {s}"
    for name, a, b in (("p", p_d, p_h), ("m", m_d, m_h), ("v", v_d, v_h)):
        same, tot = _same_bits(a, b)
        print(f"adam {hp} {name}: {same}/{tot} bit-identical after {steps} steps")
        assert same == tot


@pytest.mark.parametrize("hp", [
    dict(lr=5e-4, weight_decay=0.05, betas=(0.9, 0.999), eps=1e-8, adamw=True),
    dict(lr=2e-3, weight_decay=0.0, betas=(0.9, 0.999), eps=1e-8, adamw=False),
    dict(lr=1e-3, weight_decay=1e-2, betas=(0.8, 0.99), eps=1e-6, adamw=False),
])
def test_amsgrad_steps(gpu, hp):
    """Adam / AdamW with amsgrad (examples/gnmt/seq2seq/train/shard_optimizer.py:58-66,79-90): weights, both
    moments and the running maximum bit-identical to the oracle over six steps whose gradients shrink after
    the second, so that the maximum and the moment part ways; a NaN gradient element poisons its maximum."""
    from jabas_amd import sync
    n, steps = 70001, 6
    p_h, m_h, v_h, x_h = _host_state(n, 3), torch.zeros(n), torch.zeros(n), torch.zeros(n)
    p_d, m_d, v_d, x_d = _dev(p_h, gpu), _dev(m_h, gpu), _dev(v_h, gpu), _dev(x_h, gpu)
    for s in range(1, steps + 1):
        g = _host_grads(1, n, 170 + s, std=5e-3 if s <= 2 else 2e-4)[0]
        if s == steps:
            g[12345] = float("nan")
        O.adam_step(p_h, g, m_h, v_h, step=s, vmax=x_h, **hp)
        sync.adam_step(_dev(g, gpu), p_d, m_d, v_d, step=s, max_exp_avg_sq=x_d, **hp)
        torch.cuda.synchronize()
        for name, a, b in (("p", p_d, p_h), ("m", m_d, m_h), ("v", v_d, v_h), ("max", x_d, x_h)):
            a = a.detach().cpu()
            nan = torch.isnan(b)                            # (a NaN's payload is not part of the contract)
            assert torch.equal(torch.isnan(a), nan) and int(nan.sum()) == (1 if s == steps else 0), (s, name)
            same, tot = _same_bits(a[~nan], b[~nan])
            assert same == tot, (s, name, same, tot)
    assert float((x_h > v_h).float().mean()) > 0.5 and bool(torch.isnan(x_d[12345])) and bool(torch.isnan(p_d[12345]))


@pytest.mark.parametrize("K,dtype,kind,stats", [(3, torch.float32, "adam", "full"), (8, torch.bfloat16, "adamw", "similarity"),
                                                (4, torch.float32, "adamw", False), (16, torch.bfloat16, "adam", "full"),
                                                (9, torch.float32, "adamw", "similarity")])
def test_sync_bucket_fused_amsgrad(gpu, K, dtype, kind, stats):
    """The fused launch with the amsgrad kinds: aggregate, statistics, weights, moments, maximum and the
    replica all from one pass, bit-identical to the oracle (statistics within their bar)."""
    from jabas_amd import sync
    n = 200003
    skew = 3 if dtype == torch.bfloat16 else 1
    bounds = ((0, 1), (5, 0), (1029, 1), (70000, 0), (70001, 1), (150000, 0))
    opt = dict(ADAMW if kind == "adamw" else ADAM, amsgrad=True)
    p_h, s1_h, s2_h, s3_h = _host_state(n, 5), torch.zeros(n), torch.zeros(n), torch.zeros(n)
    agg_d = _dev(torch.zeros(n), gpu, skew)
    p_d, s1_d, s2_d, s3_d = (_dev(t, gpu, skew) for t in (p_h, s1_h, s2_h, s3_h))
    fan = [_dev(torch.zeros(n), gpu, skew)]
    dg = [_dev(torch.zeros(n, dtype=dtype), gpu, skew) for _ in range(K)]
    span = sync.SpanSpec(dg, agg_out=agg_d, param=p_d, state1=s1_d, state2=s2_d, state3=s3_d, fanout=fan, bounds=bounds)
    ws = sync.Workspace.for_span(n, dtype, gpu)
    for step in (1, 2, 3, 4):
        hg = _host_grads(K, n, 460 + K + step, std=5e-3 if step <= 2 else 2e-4, dtype=dtype)
        for d, h in zip(dg, hg):
            d.copy_(h)
        args = sync.make_step_args(BATCHES[K], dtype, stats=stats, opt=opt, step=step)
        row = sync.sync_bucket(span, args, workspace=ws)
        torch.cuda.synchronize()
        agg_h, rows_h = O.sync_step(hg, BATCHES[K], [(0, n, bounds)], opt, p_h, s1_h, s2_h, step=step,
                                    want_stats=bool(stats), state3=s3_h)
        assert torch.equal(_bits(agg_d), _bits(agg_h)), f"step {step}"
        for name, a, b in (("p", p_d, p_h), ("m", s1_d, s1_h), ("v", s2_d, s2_h), ("max", s3_d, s3_h), ("replica", fan[0], p_h)):
            same, tot = _same_bits(a, b)
            assert same == tot, (step, name, same, tot)
        if stats:
            rtol = 1e-2 if dtype == torch.bfloat16 else 1e-6
            width = 4 + K if stats == "full" else 4
            assert _close(row.cpu()[1:width], rows_h[0][1:width], rtol, 1e-30)[0]
            assert abs(float(row[0].cpu() - rows_h[0][0])) <= rtol * float(torch.sqrt(rows_h[0][1] * rows_h[0][2]))
    assert float((s3_h > s2_h).float().mean()) > 0.1          # the maximum did part from the moment


@pytest.mark.parametrize("K,dtype,kind,stats,amsgrad", [
    (4, torch.float32, "adamw", "similarity", False), (8, torch.bfloat16, "adamw", "similarity", False),
    (8, torch.bfloat16, "adamw", False, False), (2, torch.float32, "adam", "full", True),
    (8, torch.bfloat16, "adam", "full", True), (3, torch.float32, "adamw", "gram", False),
    (12, torch.float32, "adam", False, False), (1, torch.float32, "adamw", False, True)])
@pytest.mark.parametrize("block_log2", [8, 11, 13])
def test_interleaved_moments(gpu, K, dtype, kind, stats, amsgrad, block_log2):
    """Adam's moments in one arena of alternating blocks (JabasSpan.state_block_log2): spans that start at
    arbitrary elements of the arena, in the middle of a block, shorter than a block and across many blocks, with
    parameter-group bounds and element skews; aggregate, weights and every moment bit-identical to the oracle's
    flat arrays, nothing of the arena outside the span's own elements touched."""
    from jabas_amd import sync
    opt = dict(ADAMW if kind == "adamw" else ADAM, amsgrad=amsgrad)
    ways, T = (3 if amsgrad else 2), 1 << block_log2
    total = 5 * T + 70001
    arena = sync.MomentArena(total, ways, gpu, block_log2)
    marker = 7.25
    arena.buf.fill_(marker)
    cases = [(0, 4099, 0), (T - 64, 3 * T + 200, 0), (T + 320, 37, 0), (2 * T + 64 * 5 + 3, 70001, 3), (4 * T - 4 + 1, 2 * T, 1)]
    for ci, (first, n, skew) in enumerate(cases):
        skew = first % 64                          # every buffer of a span sits at the same element of a 256-byte line
        print(f"interleaved K={K} {dtype} T={T} first={first} n={n}", flush=True)
        bounds = ((0, 1), (5, 0), (min(1029, n - 1), 1)) if n > 1100 else ((0, 0),)
        p_h = _host_state(n, 5 + ci)
        m_h, v_h, x_h = torch.zeros(n), torch.zeros(n), torch.zeros(n)
        for j in range(ways):
            arena.write(j, torch.zeros(n, device=gpu), first)
        agg_d = _dev(torch.zeros(n), gpu, skew)
        p_d = _dev(p_h, gpu, skew)
        dg = [_dev(torch.zeros(n, dtype=dtype), gpu, skew) for _ in range(K)]
        span = sync.SpanSpec(dg, agg_out=agg_d, param=p_d, bounds=bounds, moments=(arena, first))
        ws = sync.Workspace.for_span(n, dtype, gpu)
        for step in (1, 2, 3):
            hg = _host_grads(K, n, 700 + K + step + ci, std=5e-3 if step <= 2 else 2e-4, dtype=dtype)
            for d, h in zip(dg, hg):
                d.copy_(h)
            row = sync.sync_bucket(span, sync.make_step_args(BATCHES[K], dtype, stats=stats, opt=opt, step=step), workspace=ws)
            torch.cuda.synchronize()
            agg_h, rows_h = O.sync_step(hg, BATCHES[K], [(0, n, bounds)], opt, p_h, m_h, v_h, step=step,
                                        want_stats=bool(stats), state3=x_h if amsgrad else None)
            assert torch.equal(_bits(agg_d), _bits(agg_h)), (first, step)
            got = [arena.read(j, first, n) for j in range(ways)]
            for name, a, b in (("p", p_d, p_h), ("m", got[0], m_h), ("v", got[1], v_h)) + ((("max", got[2], x_h),) if amsgrad else ()):
                same, tot = _same_bits(a, b)
                assert same == tot, (first, n, step, name, same, tot)
            if stats:
                rtol = 1e-2 if dtype == torch.bfloat16 else 1e-6
                assert _close(row.cpu()[1:4], rows_h[0][1:4], rtol, 1e-30)[0]
    # what the spans did not own still holds the marker
    owned = torch.zeros(arena.blocks * T, dtype=torch.bool, device=gpu)
    for first, n, _ in cases:
        owned[first:first + n] = True
    for j in range(ways):
        rest = arena.way(j).reshape(-1)[~owned]
        assert bool((rest == marker).all()), j


def test_interleaved_moments_are_checked(gpu):
    """Layout rules of interleaved moments: Adam kinds only, state2 / state3 whole blocks behind state1, the
    block position inside the block, the block group on a 16-byte line; the moments count as one written range."""
    import ctypes as C
    from jabas_amd import sync, _lib as L
    lib = L.lib()
    n, b = 5000, 10
    T = 1 << b
    arena = sync.MomentArena(8 * T, 2, gpu, b)
    g = [torch.zeros(n, device=gpu)]
    p = torch.zeros(n, device=gpu)
    adam = sync.make_step_args((1,), torch.float32, opt=ADAM, step=1)
    sgd = sync.make_step_args((1,), torch.float32, opt=SGD, first_step=True)

    def call(span, args=adam):
        return lib.jabas_sync_bucket(C.byref(span), None, C.byref(args), None, None, 0, None)
    good = sync.SpanSpec(g, param=p, moments=(arena, 0)).to_c()
    assert call(good) == L.OK
    assert call(good, sgd) == L.ERR_OPT
    bad = sync.SpanSpec(g, param=p, moments=(arena, 0)).to_c()
    bad.state2 = bad.state1 + 4 * T + 16
    assert call(bad) == L.ERR_ALIGN
    bad = sync.SpanSpec(g, param=p, moments=(arena, 0)).to_c()
    bad.state_block_pos = T
    assert call(bad) == L.ERR_SIZE
    bad = sync.SpanSpec(g, param=p, moments=(arena, 0)).to_c()
    bad.state_block_log2 = 7
    assert call(bad) == L.ERR_SIZE
    bad = sync.SpanSpec(g, param=p, moments=(arena, 0)).to_c()
    bad.state_block_pos = 2                                   # the block group would start 8 bytes off a 16-byte line
    assert call(bad) == L.ERR_ALIGN
    # the weights inside the moments' range (the gap between two of the span's blocks is part of that range)
    inside = arena.buf[2 * T:2 * T + n]
    assert call(sync.SpanSpec(g, param=inside, moments=(arena, 0)).to_c()) == L.ERR_ALIAS
    ams = sync.make_step_args((1,), torch.float32, opt=dict(ADAM, amsgrad=True), step=1)
    assert call(good, ams) == L.ERR_NULL                      # two moments interleaved where the optimizer keeps three
    torch.cuda.synchronize()


def test_amsgrad_needs_its_maximum_and_is_not_replayed_from_a_block(gpu):
    from jabas_amd import sync, _lib as L
    n = 4096
    g = [torch.zeros(n, device=gpu)]
    p, m, v = (torch.zeros(n, device=gpu) for _ in range(3))
    opt = dict(ADAM, amsgrad=True)
    args = sync.make_step_args((1,), torch.float32, opt=opt, step=1)
    assert args.opt_kind == L.OPT_ADAM_AMSGRAD
    with pytest.raises(L.JabasSyncError) as e:
        sync.sync_bucket(sync.SpanSpec(g, param=p, state1=m, state2=v), args)
    assert e.value.status == L.ERR_NULL
    with pytest.raises(L.JabasSyncError) as e:
        sync.SyncPlan([sync.SpanSpec(g, param=p, state1=m, state2=v)], L.OPT_ADAMW_AMSGRAD)
    assert e.value.status == L.ERR_NULL
    with pytest.raises(ValueError):
        sync.opt_kind(dict(SGD, amsgrad=True))


# ------------------------------------------------------------------ fused, single bucket
@pytest.mark.parametrize("K,dtype,opt", [(2, torch.float32, SGD), (4, torch.float32, ADAMW),
                                         (3, torch.float32, ADAM), (8, torch.bfloat16, ADAMW),
                                         (5, torch.bfloat16, SGD), (1, torch.float32, ADAM),
                                         (9, torch.float32, ADAM), (12, torch.float32, SGD),
                                         (13, torch.bfloat16, ADAM), (16, torch.bfloat16, ADAMW),
                                         (16, torch.float32, ADAMW)])
def test_sync_bucket_fused(gpu, K, dtype, opt):
    from jabas_amd import sync
    n = 200003
    skew = 3 if dtype == torch.bfloat16 else 1
    bounds = ((0, 1), (5, 0), (1029, 1), (70000, 0), (70001, 1), (150000, 0))
    hg = _host_grads(K, n, 60 + K, std=5e-4, dtype=dtype)
    p_h, s1_h, s2_h = _host_state(n, 5), torch.zeros(n), torch.zeros(n)
    dg = [_dev(t, gpu, skew) for t in hg]
    agg_d = _dev(torch.zeros(n), gpu, skew)
    p_d, s1_d, s2_d = _dev(p_h, gpu, skew), _dev(s1_h, gpu, skew), _dev(s2_h, gpu, skew)
    fan = [_dev(torch.zeros(n), gpu, skew) for _ in range(2)]
    adam = opt["kind"] != "sgd"
    span = sync.SpanSpec(dg, agg_out=agg_d, param=p_d, state1=s1_d, state2=s2_d if adam else None, fanout=fan,
                         bounds=bounds)
    ws = sync.Workspace.for_span(n, dtype, gpu)
    for step in (1, 2, 3):
        args = sync.make_step_args(BATCHES[K], dtype, stats=True, opt=opt, step=step, first_step=(step == 1))
        row = sync.sync_bucket(span, args, workspace=ws)
        torch.cuda.synchronize()
        agg_h, rows_h = O.sync_step(hg, BATCHES[K], [(0, n, bounds)], opt, p_h, s1_h, s2_h if adam else None,
                                    step=step, first_step=(step == 1), want_stats=True)
        assert torch.equal(_bits(agg_d), _bits(agg_h)), f"step {step}"
        rtol = 1e-2 if dtype == torch.bfloat16 else 1e-6
        assert _close(row.cpu()[:4 + K], rows_h[0][:4 + K], rtol, 1e-30)[0]
        assert _close(p_d, p_h, 1e-6, 1e-9)[0], f"step {step}"
        assert _close(s1_d, s1_h, 1e-6, 2e-9)[0], f"step {step}"
        if adam:
            assert _close(s2_d, s2_h, 1e-6, 1e-16)[0], f"step {step}"
        for f in fan:
            assert torch.equal(_bits(f), _bits(p_d))
    same, tot = _same_bits(p_d, p_h)
    print(f"fused bucket K={K} {dtype} {opt['kind']}: {same}/{tot} weights bit-identical")
    assert same == tot


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("skews", [
    "37 for every buffer",                # one offset within 256 bytes: the launch's element grid starts at that line
    "differs within 256 bytes",           # equal only within 16 bytes: the grid starts at the first element's 16-byte line
    "63 for every buffer", "60 for every buffer"])
def test_sync_bucket_buffer_offsets_within_a_256_byte_line(gpu, dtype, skews):
    """Where the launch's element grid starts depends on how the buffers sit relative to 256-byte
    lines; the results must not."""
    from jabas_amd import sync
    K, n = 3, 150001
    bounds = ((0, 1), (3, 0), (61, 1), (1024, 0), (99999, 1))
    if skews.endswith("for every buffer"):
        sk = [int(skews.split()[0])] * 8
    else:
        sk = [5, 9, 61, 33, 1, 17, 49, 13]             # all 1 mod 4
    hg = _host_grads(K, n, 300, std=5e-4, dtype=dtype)
    p_h, s1_h, s2_h = _host_state(n, 6), torch.zeros(n), torch.zeros(n)
    dg = [_dev(t, gpu, sk[k]) for k, t in enumerate(hg)]
    agg_d = _dev(torch.zeros(n), gpu, sk[3])
    p_d, s1_d, s2_d = _dev(p_h, gpu, sk[4]), _dev(s1_h, gpu, sk[5]), _dev(s2_h, gpu, sk[6])
    fan = [_dev(torch.zeros(n), gpu, sk[7])]
    guard = [t._base if t._base is not None else t for t in dg + [agg_d, p_d, s1_d, s2_d] + fan]
    before = [(b[:sk_i].clone(), b[sk_i + n:].clone()) for b, sk_i in zip(guard, sk)]
    span = sync.SpanSpec(dg, agg_out=agg_d, param=p_d, state1=s1_d, state2=s2_d, fanout=fan, bounds=bounds)
    ws = sync.Workspace.for_span(n, dtype, gpu)
    for step in (1, 2):
        args = sync.make_step_args(BATCHES[K], dtype, stats=True, opt=ADAMW, step=step, first_step=(step == 1))
        row = sync.sync_bucket(span, args, workspace=ws)
        torch.cuda.synchronize()
        agg_h, rows_h = O.sync_step(hg, BATCHES[K], [(0, n, bounds)], ADAMW, p_h, s1_h, s2_h, step=step,
                                    first_step=(step == 1), want_stats=True)
        assert torch.equal(_bits(agg_d), _bits(agg_h)), step
        rtol = 1e-2 if dtype == torch.bfloat16 else 1e-6
        assert _close(row.cpu()[:4 + K], rows_h[0][:4 + K], rtol, 1e-30)[0]
        for got, want in ((p_d, p_h), (s1_d, s1_h), (s2_d, s2_h), (fan[0], p_h)):
            assert torch.equal(_bits(got), _bits(want)), step
    # nothing outside the live range was written
    for b, sk_i, (head, tail) in zip(guard, sk, before):
        assert torch.equal(b[:sk_i], head) and torch.equal(b[sk_i + n:], tail)


# ---------------------------------------------------------------- fused, multi-span plan
@pytest.mark.parametrize("K,dtype,opt,in_place", [
    (2, torch.float32, SGD, True), (4, torch.float32, ADAMW, True), (3, torch.float32, SGD, False),
    (4, torch.float32, ADAM, False), (8, torch.bfloat16, ADAMW, False), (6, torch.float32, None, True),
    (7, torch.bfloat16, None, False), (10, torch.float32, ADAMW, True), (16, torch.bfloat16, SGD, False),
    (15, torch.float32, None, False)])
def test_sync_fused_plan_ragged_spans(gpu, K, dtype, opt, in_place):
    from jabas_amd import sync, _lib as L
    # span sizes: tiny, exactly one tile, ragged, empty, large; offsets chosen so that some
    # spans start off a 16-byte line (all buffers share the offset, as views of one layout do)
    sizes = [1, 1024, 2048, 0, 4097, 333, 8192 * 3 + 5, 7, 500000, 64, 2048 * 40]
    gaps = [0, 3, 0, 1, 0, 2, 0, 0, 5, 0, 0]
    offs, off = [], 0
    for s, gp in zip(sizes, gaps):
        off += gp
        offs.append(off)
        off += s
    total = off
    hg = _host_grads(K, total, 80 + K, std=5e-4, dtype=dtype)
    p_h, s1_h, s2_h = _host_state(total, 7), torch.zeros(total), torch.zeros(total)
    dg = [_dev(t, gpu) for t in hg]
    agg_d = dg[0] if in_place else _dev(torch.zeros(total), gpu)
    p_d, s1_d, s2_d = _dev(p_h, gpu), _dev(s1_h, gpu), _dev(s2_h, gpu)
    kind = sync.opt_kind(opt)
    adam = kind in (L.OPT_ADAM, L.OPT_ADAMW)
    spans_h, spans_d = [], []
    for i, (o, s) in enumerate(zip(offs, sizes)):
        if s > 3000:
            bounds = ((0, i % 2), (s // 3, 1 - i % 2), (s // 3 + 1, i % 2), (s - 1, 1))
        elif s > 0:
            bounds = ((0, i % 2),)
        else:
            bounds = ()
        sl = slice(o, o + s)
        spans_h.append((o, s, bounds))
        spans_d.append(sync.SpanSpec([g[sl] for g in dg], agg_out=agg_d[sl],
                                     param=p_d[sl] if opt else None, state1=s1_d[sl] if opt else None,
                                     state2=s2_d[sl] if adam else None, bounds=bounds if opt else ()))
    plan = sync.SyncPlan(spans_d, kind)
    hg_work = [t.clone() for t in hg]
    for step in (1, 2):
        args = sync.make_step_args(BATCHES[K], dtype, stats=True, opt=opt, step=step, first_step=(step == 1))
        rows = plan.run(args)
        torch.cuda.synchronize()
        agg_h, rows_h = O.sync_step(hg_work, BATCHES[K], spans_h, opt, p_h, s1_h, s2_h if adam else None,
                                    step=step, first_step=(step == 1), want_stats=True)
        for (o, s, _), i in zip(spans_h, range(len(spans_h))):
            assert torch.equal(_bits(agg_d[o:o + s]), _bits(agg_h[o:o + s])), f"span {i} step {step}"
        rtol = 1e-2 if dtype == torch.bfloat16 else 1e-6
        ok, err = _close(rows.cpu()[:, :4 + K], rows_h[:, :4 + K], rtol, 1e-30)
        assert ok, f"stats step {step}: {rows.cpu()} vs {rows_h}"
        if opt:
            assert _close(p_d, p_h, 1e-6, 1e-9)[0], f"step {step}"
            assert _close(s1_d, s1_h, 1e-6, 2e-9)[0]
            if adam:
                assert _close(s2_d, s2_h, 1e-6, 1e-16)[0]
        if in_place:
            # the next step aggregates what is now in VSW 0's buckets, on both sides
            for (o, s, _) in spans_h:
                hg_work[0][o:o + s] = agg_h[o:o + s]
    # elements in the gaps between spans are never written
    covered = torch.zeros(total, dtype=torch.bool)
    for o, s, _ in spans_h:
        covered[o:o + s] = True
    if opt:
        assert torch.equal(_bits(p_d)[~covered], _bits(_host_state(total, 7))[~covered])


def test_fused_rejects_bad_arguments(gpu):
    from jabas_amd import sync, _lib as L
    n = 4096
    g = [torch.zeros(n + 8, device=gpu) for _ in range(2)]
    out = torch.zeros(n + 8, device=gpu)
    with pytest.raises(L.JabasSyncError) as e:
        sync.aggregate([g[0][1:n + 1], g[1][:n]], (1, 1), out=out[:n])       # mutually misaligned
    assert e.value.status == L.ERR_ALIGN
    with pytest.raises(L.JabasSyncError) as e:
        sync.aggregate([g[0][:n], g[1][:n]], (1, 1), out=g[0][4:n + 4])      # partial overlap
    assert e.value.status == L.ERR_ALIAS
    with pytest.raises(ValueError):
        sync.aggregate([g[0][:n]] * 17, (1,) * 17)
    span = sync.SpanSpec([g[0][:n], g[1][:n]], param=None)
    args = sync.make_step_args((1, 1), torch.float32, opt=SGD)
    with pytest.raises(L.JabasSyncError) as e:
        sync.sync_bucket(span, args)                                          # optimizer without weights
    assert e.value.status == L.ERR_NULL


def test_span_beyond_two_to_the_31_elements(gpu):
    """64-bit element indexing: one span of 2^31 + 4099 elements (8.6 GB per buffer)."""
    from jabas_amd import sync
    n = (1 << 31) + 4099
    g0 = torch.empty(n, dtype=torch.float32, device=gpu)
    g1 = torch.empty(n, dtype=torch.float32, device=gpu)
    step = 1 << 27
    for lo in range(0, n, step):                       # value depends on the position, cheap to regenerate
        hi = min(n, lo + step)
        idx = torch.arange(lo, hi, device=gpu, dtype=torch.int64)
        g0[lo:hi] = ((idx % 1021).float() - 510.0) * 2.0 ** -10
        g1[lo:hi] = ((idx % 4093).float() - 2046.0) * 2.0 ** -12
        del idx
    out = torch.empty(n, dtype=torch.float32, device=gpu)
    sync.aggregate([g0, g1], (1, 1), out=out)          # weights 0.5, 0.5: every product and the sum are exact
    row = sync.gradient_stats([g0, g1], (1, 1)).cpu()
    torch.cuda.synchronize()
    norm0 = 0.0
    for lo in range(0, n, step):
        hi = min(n, lo + step)
        want = g0[lo:hi] * 0.5 + g1[lo:hi] * 0.5
        assert torch.equal(out[lo:hi].view(torch.int32), want.view(torch.int32)), lo
        norm0 += float((g0[lo:hi].double() ** 2).sum())
        del want
    assert float(row[4]) == pytest.approx(norm0, rel=1e-10)


def test_special_values_denormals_infinities_nans(gpu):
    """Denormal inputs and results are kept (no flush to zero), infinities and NaNs stay in
    the element they entered, signed zeros follow IEEE addition."""
    from jabas_amd import sync
    K, n = 3, 5000
    hg = _host_grads(K, n, 99)
    hg[0][:64] = torch.logspace(-45, -38, 64)                 # denormal inputs
    hg[1][:64] = -torch.logspace(-44.5, -38.2, 64)
    hg[2][:64] = 0.0
    hg[0][100], hg[1][101], hg[2][102] = float("inf"), float("-inf"), float("nan")
    hg[0][103], hg[1][103] = float("inf"), float("-inf")       # inf - inf -> nan
    hg[0][200:210], hg[1][200:210], hg[2][200:210] = -0.0, -0.0, -0.0
    hg[0][210:220], hg[1][210:220], hg[2][210:220] = -0.0, 0.0, -0.0
    out = sync.aggregate([_dev(t, gpu) for t in hg], BATCHES[K]).cpu()
    want = O.aggregate(hg, BATCHES[K])
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(out), nan) and int(nan.sum()) == 2
    assert torch.equal(out[~nan].view(torch.int32), want[~nan].view(torch.int32))
    assert torch.count_nonzero(out[:64]) > 32                  # denormal results survived
    assert torch.all(out[200:210].view(torch.int32) == torch.tensor(-0.0).view(torch.int32))
    assert torch.all(out[210:220].view(torch.int32) == 0)
    # Adam on a gradient whose square is denormal: v stays denormal, the step is still the sign step
    g = torch.full((2048,), 1e-21)
    p_h, m_h, v_h = torch.ones(2048), torch.zeros(2048), torch.zeros(2048)
    p_d, m_d, v_d = _dev(p_h, gpu), _dev(m_h, gpu), _dev(v_h, gpu)
    hp = dict(lr=1e-3, weight_decay=0.0, betas=(0.9, 0.999), eps=1e-30, adamw=False)
    O.adam_step(p_h, g, m_h, v_h, step=1, **hp)
    sync.adam_step(_dev(g, gpu), p_d, m_d, v_d, step=1, **hp)
    torch.cuda.synchronize()
    assert 0 < float(v_h[0]) < 1.2e-38                         # denormal second moment
    for a, b in ((p_d, p_h), (m_d, m_h), (v_d, v_h)):
        assert torch.equal(_bits(a), _bits(b))


# ------------------------------------------------------------- randomized plans vs the oracle
def _random_case(seed):
    rng = np.random.RandomState(seed)
    K = int(rng.randint(1, 9)) if seed < 16 else int(rng.randint(9, 17))
    dtype = torch.bfloat16 if rng.rand() < 0.4 else torch.float32
    opt = [None, SGD, ADAM, ADAMW][int(rng.randint(0, 4))]
    if opt is SGD and rng.rand() < 0.3:
        opt = dict(SGD, nesterov=True, momentum=0.8)
    n_span = int(rng.randint(1, 25))
    sizes = []
    for _ in range(n_span):
        kind = rng.rand()
        if kind < 0.1:
            sizes.append(0)
        elif kind < 0.5:
            sizes.append(int(rng.randint(1, 3000)))
        elif kind < 0.8:
            sizes.append(int(1024 * rng.randint(1, 9) + rng.choice([-1, 0, 1, 2])))
        else:
            sizes.append(int(rng.randint(20000, 120000)))
    gaps = [int(rng.randint(0, 9)) for _ in sizes]
    half_id = None
    if K >= 2 and rng.rand() < 0.5:                      # arbitrary halves, both non-empty
        while True:
            half_id = [int(v) for v in rng.randint(0, 2, size=K)]
            if 0 < sum(half_id) < K:
                break
    batches = tuple(int(v) for v in rng.randint(1, 65, size=K))
    in_place = dtype == torch.float32 and rng.rand() < 0.5
    n_fan = int(rng.randint(0, 3)) if opt else 0
    bounds = []
    for s in sizes:
        if opt is None or s == 0:
            bounds.append(())
            continue
        nb = int(rng.randint(0, 5))
        starts = sorted(set([0] + [int(v) for v in rng.randint(1, max(2, s), size=nb) if v < s]))
        bounds.append(tuple((st, int(rng.randint(0, 2))) for st in starts))
    return K, dtype, opt, sizes, gaps, half_id, batches, in_place, n_fan, bounds


@pytest.mark.parametrize("seed", range(24))
def test_random_plans_match_the_oracle(gpu, seed):
    """Random K, dtype, optimizer, span sizes (empty, sub-tile, tile-edge, large), line offsets, group
    bounds, halves, fan-out and in-place aggregation: the planned launch against the oracle over 3 steps."""
    from jabas_amd import sync, _lib as L
    K, dtype, opt, sizes, gaps, half_id, batches, in_place, n_fan, bounds = _random_case(seed)
    print(f"seed {seed}: K={K} {dtype} opt={opt and opt['kind']} spans={sizes} gaps={gaps} halves={half_id} "
          f"in_place={in_place} fan={n_fan}", flush=True)
    offs, off = [], 0
    for s, gp in zip(sizes, gaps):
        off += gp
        offs.append(off)
        off += s
    total = max(off, 1)
    hg = _host_grads(K, total, 300 + seed, std=5e-4, dtype=dtype)
    p_h, s1_h, s2_h = _host_state(total, 40 + seed), torch.zeros(total), torch.zeros(total)
    base_skew = seed % 4
    srng = np.random.RandomState(7000 + seed)

    def skew():
        """Every third seed puts each buffer at its own place of a 256-byte line (equal within 16
        bytes only: the launch falls back to the 16-byte element grid); the others share one place."""
        return base_skew + (4 * int(srng.randint(0, 16)) if seed % 3 == 2 else 4 * (seed % 16))
    dg = [_dev(t, gpu, skew()) for t in hg]
    agg_d = dg[0] if in_place else _dev(torch.zeros(total), gpu, skew())
    p_d, s1_d, s2_d = _dev(p_h, gpu, skew()), _dev(s1_h, gpu, skew()), _dev(s2_h, gpu, skew())
    fans = [_dev(torch.zeros(total), gpu, skew()) for _ in range(n_fan)]
    kind = sync.opt_kind(opt)
    adam = kind in (L.OPT_ADAM, L.OPT_ADAMW)
    # every other Adam case keeps the moments interleaved in one arena (blocks of 256, 1024 or 8192 elements), the
    # arena's element 0 at the weights' place of a 16-byte line (of a 256-byte line when all buffers share one)
    arena = None
    if adam and seed % 4 >= 2:
        arena_first = skew()
        arena = sync.MomentArena(arena_first + total, 2, gpu, (8, 10, 13)[seed % 3])
    spans_h, spans_d = [], []
    for o, s, b in zip(offs, sizes, bounds):
        sl = slice(o, o + s)
        spans_h.append((o, s, b))
        state = dict(moments=(arena, arena_first + o)) if arena is not None else \
            dict(state1=s1_d[sl] if opt else None, state2=s2_d[sl] if adam else None)
        spans_d.append(sync.SpanSpec([g[sl] for g in dg], agg_out=agg_d[sl], param=p_d[sl] if opt else None,
                                     fanout=[f[sl] for f in fans], bounds=b, **state))
    plan = sync.SyncPlan(spans_d, kind)
    hg_work = [t.clone() for t in hg]
    block = sync.StepScalars(gpu) if opt and seed % 2 else None
    for step in (1, 2, 3):
        # full rows on the first step, none on the second; on the third the similarity sums or, up to eight
        # workers, the full rows with the pair products
        stats = (True, False, "gram" if K <= L.STATS_GRAM_MAX_K and seed % 3 else "similarity")[step - 1]
        args = sync.make_step_args(batches, dtype, stats=stats, opt=opt, step=step, first_step=(step == 1),
                                   half_id=half_id)
        if block is not None:
            # odd seeds: the step's scalars travel in the device block; the by-value arguments of the call are
            # those of another step at another learning rate, as in a launch recorded once and replayed
            block.update(args)
            args = block.attach(sync.make_step_args(batches, dtype, stats=stats, opt=opt, step=5, first_step=(step != 1),
                                                    half_id=half_id, lr_scale=3.0))
        rows = plan.run(args)
        torch.cuda.synchronize()
        hg_in = [t.clone() for t in hg_work]            # what this step's launch read (the in-place aggregate moves worker 0's)
        agg_h, rows_h = O.sync_step(hg_work, batches, spans_h, opt, p_h, s1_h, s2_h if adam else None, step=step,
                                    first_step=(step == 1), want_stats=bool(stats), half_id=half_id)
        for i, (o, s, _) in enumerate(spans_h):
            assert torch.equal(_bits(agg_d[o:o + s]), _bits(agg_h[o:o + s])), f"span {i} step {step}"
        if stats:
            rtol = 1e-2 if dtype == torch.bfloat16 else 1e-6
            width = 4 if stats == "similarity" else 4 + K
            got, want = rows.cpu()[:, :width], rows_h[:, :width]
            scale = want[:, 1:3].abs().max(dim=1, keepdim=True).values.clamp_min(1e-300)   # dot may cancel: bound it by the norms
            assert bool(((got - want).abs() <= rtol * want.abs() + 1e-9 * scale).all()), f"stats step {step}"
            pairs = K * (K - 1) // 2 if stats == "gram" else 0
            assert torch.count_nonzero(rows[:, width + pairs:]) == 0
            if pairs:
                for i, (o, sz, _) in enumerate(spans_h):
                    G = O.gram([t[o:o + sz] for t in hg_in])
                    for a in range(K):
                        for b in range(a + 1, K):
                            err = abs(float(rows[i, L.stat_pair(K, a, b)]) - float(G[a, b]))
                            assert err <= (1e-5 if dtype == torch.bfloat16 else 1e-11) * float(torch.sqrt(G[a, a] * G[b, b])) + 1e-300, \
                                f"pair ({a}, {b}) span {i}"
        if opt:
            if arena is not None:
                s1_d, s2_d = arena.read(0, arena_first, total), arena.read(1, arena_first, total)
            for i, (o, s, _) in enumerate(spans_h):
                assert torch.equal(_bits(p_d[o:o + s]), _bits(p_h[o:o + s])), f"weights span {i} step {step}"
                assert torch.equal(_bits(s1_d[o:o + s]), _bits(s1_h[o:o + s])), f"state1 span {i} step {step}"
                if adam:
                    assert torch.equal(_bits(s2_d[o:o + s]), _bits(s2_h[o:o + s])), f"state2 span {i} step {step}"
                for f in fans:
                    assert torch.equal(_bits(f[o:o + s]), _bits(p_d[o:o + s]))
        if in_place:
            for (o, s, _) in spans_h:
                hg_work[0][o:o + s] = agg_h[o:o + s]
    # nothing outside the spans was written
    covered = torch.zeros(total, dtype=torch.bool)
    for o, s, _ in spans_h:
        covered[o:o + s] = True
    if opt and (~covered).any():
        assert torch.equal(_bits(p_d)[~covered], _bits(_host_state(total, 40 + seed))[~covered])
        if arena is not None:                                # the moments of elements no span owns stayed zero
            assert torch.count_nonzero(arena.read(0, arena_first, total)[~covered.to(gpu)]) == 0
            assert torch.count_nonzero(arena.read(1, arena_first, total)[~covered.to(gpu)]) == 0
        for f in fans:
            assert torch.count_nonzero(f.cpu()[~covered]) == 0
    if not in_place and (~covered).any():
        assert torch.count_nonzero(agg_d.cpu()[~covered]) == 0


@pytest.mark.parametrize("seed", list(range(100, 112)) + [116, 117, 119, 121])
def test_random_buckets_through_the_inline_path(gpu, seed):
    """The same random cases, one jabas_sync_bucket call per span (span by value, bound table on the
    device, first bound of each workgroup found by binary search)."""
    from jabas_amd import sync, _lib as L
    K, dtype, opt, sizes, gaps, half_id, batches, in_place, n_fan, bounds = _random_case(seed - 100 if seed % 2 else seed)
    rng = np.random.RandomState(seed)
    sizes = [s for s in sizes if s > 0][:8] or [777]
    bounds = [b for s, b in zip(sizes, [b for b in bounds if b] + [()] * len(sizes))]
    print(f"seed {seed}: K={K} {dtype} opt={opt and opt['kind']} sizes={sizes} halves={half_id}", flush=True)
    kind = sync.opt_kind(opt)
    adam = kind in (L.OPT_ADAM, L.OPT_ADAMW)
    for si, n in enumerate(sizes):
        skew = int(rng.randint(0, 4))
        b = tuple((st, g) for st, g in bounds[si] if st < n) if opt else ()
        if opt and (not b or b[0][0] != 0):
            b = ((0, 1),) + tuple(x for x in b if x[0] > 0)
        hg = _host_grads(K, n, 500 + 13 * seed + si, std=5e-4, dtype=dtype)
        p_h, s1_h, s2_h = _host_state(n, 60 + seed + si), torch.zeros(n), torch.zeros(n)
        dg = [_dev(t, gpu, skew) for t in hg]
        agg_d = _dev(torch.zeros(n), gpu, skew)
        p_d, s1_d, s2_d = _dev(p_h, gpu, skew), _dev(s1_h, gpu, skew), _dev(s2_h, gpu, skew)
        span = sync.SpanSpec(dg, agg_out=agg_d, param=p_d if opt else None, state1=s1_d if opt else None,
                             state2=s2_d if adam else None, bounds=b)
        call = sync.BucketCall(span)
        block = sync.StepScalars(gpu) if opt and (seed + si) % 2 else None
        for step in (1, 2, 3):
            stats = step != 2                  # the plain launch may run another workgroup shape
            args = sync.make_step_args(batches, dtype, stats=stats, opt=opt, step=step, first_step=(step == 1),
                                       half_id=half_id)
            if block is not None:              # every other bucket: scalars from the device block, stale ones by value
                block.update(args)
                args = block.attach(sync.make_step_args(batches, dtype, stats=stats, opt=opt, step=9,
                                                        first_step=(step != 1), half_id=half_id, lr_scale=0.25))
            row = call.run(args)
            torch.cuda.synchronize()
            agg_h, rows_h = O.sync_step(hg, batches, [(0, n, b)], opt, p_h, s1_h, s2_h if adam else None, step=step,
                                        first_step=(step == 1), want_stats=stats, half_id=half_id)
            assert torch.equal(_bits(agg_d), _bits(agg_h)), (si, step)
            if stats:
                rtol = 1e-2 if dtype == torch.bfloat16 else 1e-6
                got, want = row.cpu()[:4 + K], rows_h[0][:4 + K]
                scale = want[1:3].abs().max().clamp_min(1e-300)
                assert bool(((got - want).abs() <= rtol * want.abs() + 1e-9 * scale).all()), (si, step)
            else:
                assert row is None
            if opt:
                assert torch.equal(_bits(p_d), _bits(p_h)), (si, step)
                assert torch.equal(_bits(s1_d), _bits(s1_h)), (si, step)
                if adam:
                    assert torch.equal(_bits(s2_d), _bits(s2_h)), (si, step)


def test_plan_with_nothing_but_empty_spans(gpu):
    """No workgroup to launch: the statistics rows still come back, all zero, and nothing is touched."""
    from jabas_amd import sync, _lib as L
    g = [torch.zeros(16, device=gpu) for _ in range(2)]
    p, m = torch.ones(16, device=gpu), torch.zeros(16, device=gpu)
    spans = [sync.SpanSpec([t[4:4] for t in g], agg_out=g[0][4:4], param=p[4:4], state1=m[4:4]) for _ in range(3)]
    plan = sync.SyncPlan(spans, L.OPT_SGD)
    assert plan.n_chunks == 0 and plan.n_chunks_stats == 0
    rows = plan.run(sync.make_step_args((1, 1), torch.float32, stats=True, opt=SGD, step=1, first_step=True))
    torch.cuda.synchronize()
    assert rows.shape == (3, L.STATS_STRIDE) and torch.count_nonzero(rows) == 0
    assert plan.run(sync.make_step_args((1, 1), torch.float32, stats=False, opt=SGD, step=2)) is None
    torch.cuda.synchronize()
    assert torch.equal(p, torch.ones(16, device=gpu)) and torch.count_nonzero(m) == 0


@pytest.mark.parametrize("K", [1, 2, 5, 8])
@pytest.mark.parametrize("n_rows", [1, 2, 16, 17, 63, 1025])
def test_gram_from_rows_on_the_device(gpu, K, n_rows):
    """The launch that sums rows of level 'gram' and unfolds them against the torch path the host takes: fewer rows
    than waves, one more, many. Both add n_rows doubles of at most m in some order: n_rows * 2**-53 * n_rows * m apart
    at most."""
    from jabas_amd import sync, _lib as L
    rows = torch.randn(n_rows, L.STATS_STRIDE, dtype=torch.float64, generator=torch.Generator().manual_seed(K + n_rows))
    want = sync.gram_from_stats(rows, K)
    dev = rows.to(gpu)
    got = sync.gram_from_stats(dev, K)
    assert got.shape == (K, K) and got.is_contiguous() and torch.equal(got, got.t())
    bound = n_rows * n_rows * 2.0 ** -53 * float(rows.abs().max())
    assert float((got.cpu() - want).abs().max()) <= bound
    assert torch.equal(sync.gram_from_stats(dev, K), got)                              # the same call, the same bits
    strided = torch.cat([dev, dev], dim=1)[:, :L.STATS_STRIDE]                         # not whole rows in memory
    assert float((sync.gram_from_stats(strided, K).cpu() - want).abs().max()) <= bound
    assert torch.equal(sync.gram_from_stats(dev[:0], K), torch.zeros(K, K, dtype=torch.float64, device=gpu))
    with pytest.raises(ValueError):
        sync.gram_from_stats(dev, 9)
    assert L.lib().jabas_gram_from_rows(None, 1, K, dev.data_ptr(), None) == L.ERR_NULL
    assert L.lib().jabas_gram_from_rows(dev.data_ptr(), 1, 9, dev.data_ptr(), None) == L.ERR_K
    assert L.lib().jabas_gram_from_rows(dev.data_ptr() + 4, 1, K, dev.data_ptr(), None) == L.ERR_ALIGN


def test_gram_from_rows_recorded(gpu):
    """Recordings of gram_from_stats answer for rows they were not made with. Four rows of small whole numbers: every sum is exact."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from jabas_amd import sync, _lib as L
    rows, other = (torch.randint(-99, 99, (4, L.STATS_STRIDE), generator=torch.Generator().manual_seed(i)).double().to(gpu) for i in (1, 2))
    want = sync.gram_from_stats(other, 3)
    for graph in (torch.jit.trace(lambda r: sync.gram_from_stats(r, 3), rows, check_trace=False),
                  make_fx(lambda r: sync.gram_from_stats(r, 3))(rows)):
        stale = torch.full((3, 3), float("nan"), dtype=torch.float64, device=gpu)       # left in the block an unwritten output would get
        del stale
        assert torch.equal(graph(other), want)


@pytest.mark.filterwarnings("ignore::UserWarning")
def test_gram_from_rows_that_hold_no_memory(gpu):
    """Zeros without memory are summed like any others; a list of row tensors is refused."""
    from jabas_amd import sync, _lib as L
    zeros = torch._efficientzerotensor(3, L.STATS_STRIDE, dtype=torch.float64, device=gpu)
    assert torch.equal(sync.gram_from_stats(zeros, 2), torch.zeros(2, 2, dtype=torch.float64, device=gpu))
    rows = torch.ones(3, L.STATS_STRIDE, dtype=torch.float64, device=gpu)
    assert torch.equal(sync.gram_from_stats(torch._neg_view(rows), 2), torch.full((2, 2), -3.0, dtype=torch.float64, device=gpu))
    with pytest.raises(RuntimeError):
        sync.gram_from_stats(torch.nested.nested_tensor([rows, rows]), 2)


@pytest.mark.parametrize("K", [3, 4, 5])
def test_gram_of_few_workers_rounds_in_short_chains(gpu, K):
    """2**25 elements of 1 + d and 1 - d, d = 2**-22: products 1 +- 2**-21 + 2**-44 and 1 - 2**-44. A running sum of a thread
    holds 128 of them (two sums of 64 vectors each, 2**17 threads), exactly (seven bits and 45). What follows rounds at most
    36 times (two sums 1, wave 8, workgroup 16, rows of a class 2, classes 9): 50 are allowed. In chains of 2048
    products, as long as a wave's sums on the matrix cores are, the 2**-44 is lost from a sum of 512 on: 4e-14 off."""
    from jabas_amd import sync
    n, d = 1 << 25, 2.0 ** -22
    G = sync.gram([torch.full((n,), 1 - d if k % 2 else 1 + d, dtype=torch.float32, device=gpu) for k in range(K)]).cpu()
    for a in range(K):
        for b in range(K):
            exact = n * (1 - d * d if (a + b) % 2 else 1 - 2 * d + d * d if a % 2 else 1 + 2 * d + d * d)
            assert abs(float(G[a, b]) - exact) <= 50 * 2.0 ** -53 * exact, (a, b)


def _chain(c, m):
    """m products c * c (exact in fp64) added one after the other."""
    s, c2 = 0.0, float(c) * float(c)
    for _ in range(m):
        s += c2
    return s


@pytest.mark.parametrize("K,vectors", [(3, 24), (4, 24), (5, 24), (6, 24), (9, 24), (13, 24), (16, 24)])
def test_gram_fp32_sums_are_as_short_with_half_the_workgroups(gpu, K, vectors):
    """Equal elements: every running sum of the kernel is the same chain of additions, and their number is a power of two, so
    what follows adds equal numbers, exactly, and the result tells how long the chains were. fp32 on the vector ALU (K <= 5): 2**18
    sums of 24 vectors of four; on the matrix cores 2**14 sums of 96 products, in spans under 2**21 elements, where half as
    many waves keep two sums each. Chains of 192 products, one sum per thread or wave, give another number."""
    from jabas_amd import sync
    sums = 1 << (18 if K <= 5 else 14)
    m = 4 * vectors
    rng = np.random.default_rng(K)
    c = next(x for x in rng.uniform(1.0, 2.0, 200).astype(np.float32) if abs(_chain(x, 2 * m) - 2 * _chain(x, m)) > 10 * 2.0 ** -53 * m)
    G = sync.gram([torch.full((sums * m,), float(c), dtype=torch.float32, device=gpu)] * K).cpu()
    assert torch.equal(G, torch.full((K, K), sums * _chain(c, m), dtype=torch.float64))


def _exact_row(grads, level):
    """Statistics row of whole numbers under weights of a quarter: every sum is exact in fp64 (and fp32) in any order."""
    from jabas_amd import _lib as L
    K = len(grads)
    want = torch.zeros(L.STATS_STRIDE, dtype=torch.float64, device=grads[0].device)
    quarter = [sum(g.float() for g in grads[h::2]) * 0.25 if K > h else torch.zeros_like(grads[0], dtype=torch.float32) for h in (0, 1)]
    agg = sum(g.float() for g in grads) * 0.25
    want[0] = (quarter[0] * quarter[1]).sum(dtype=torch.float64)
    for slot, x in ((1, quarter[0]), (2, quarter[1]), (3, agg)):
        want[slot] = (x * x).sum(dtype=torch.float64)
    if level != "similarity":
        for k, g in enumerate(grads):
            want[4 + k] = g.float().square().sum(dtype=torch.float64)
    if level == "gram":
        for i in range(K):
            for j in range(i + 1, K):
                want[L.stat_pair(K, i, j)] = (grads[i].float() * grads[j].float()).sum(dtype=torch.float64)
    return want


def _quarter_args(K, dtype, level):
    from jabas_amd import sync
    args = sync.make_step_args((1,) * K, dtype, stats=level)
    for k in range(K):                                         # powers of two instead of the batch quotients
        args.weight[k] = args.half_weight[k] = 0.25
    return args


def _whole_numbers(gpu, n, K, dtype, seed):
    gen = torch.Generator(device=gpu).manual_seed(seed)
    return [torch.randint(-3, 4, (n,), generator=gen, device=gpu, dtype=torch.int8).to(dtype) for _ in range(K)]


@pytest.mark.parametrize("rows", [1, 64, 65, 255, 256, 257, 512, 1024, 1025, 2049, 4096, 4097, 5000, 16900])
@pytest.mark.parametrize("K,level", [(4, "similarity"), (5, "full"), (8, "gram"), (16, "full")])
def test_statistics_over_many_chunks_are_exact(gpu, K, level, rows):
    """The row has to be the integer result whatever the number of partial rows (edges of the second level's waves per span, of
    its batches, of its classes and of its split into stripes, stripes of 512 rows and 32 longer ones) and the width of the row.
    Scratch and output start as NaN, which tells how many rows the launch wrote; the number of tiles per workgroup is the
    launch's own, so the size that gives the wanted rows is looked for among one, two and four, then among whole chunks."""
    from jabas_amd import sync
    width = {"similarity": 4, "full": 4 + K, "gram": 4 + K + K * (K - 1) // 2}[level]
    stripes = 0 if rows <= 4096 else min(32, -(-rows // 512))
    args = _quarter_args(K, torch.bfloat16, level)
    for tight in (False, True):                                # scratch of whole chunks: the launch is not split
        for tiles in (1, 2, 4):
            n = 1024 * tiles * (rows - 1) + 5
            grads = _whole_numbers(gpu, n, min(K, 4), torch.bfloat16, rows + K)
            grads = [grads[k % len(grads)] for k in range(K)]  # the kernel only reads
            ws = sync.Workspace.for_span(n, torch.bfloat16, gpu)
            ws.buf.fill_(float("nan"))
            ws.stats.fill_(float("nan"))
            if tight:
                ws.nbytes = min(ws.nbytes, (-(-n // (2048 if K <= 4 else 4096)) + 33) * width * 8)
            row = sync.sync_bucket(sync.SpanSpec(grads), args, workspace=ws)
            assert torch.equal(row, _exact_row(grads, level))
            if int((~ws.buf.isnan()).sum()) == (rows + stripes) * width:
                return
    pytest.fail(f"no launch wrote {rows} rows")


@pytest.mark.parametrize("K,level,sizes", [
    (9, "full", [700, 13_000_123, 3000]),                      # two workgroups per chunk and stripes, short spans beside them
    (4, "similarity", [5, 9_000_001, 1 << 20, 1]), (4, "gram", [300_001, 1025, 1024, 70_000]), (1, "similarity", [1 << 20] * 2),
    (3, "full", [1000] * 301), (8, "gram", [1 + 37 * i for i in range(130)]), (8, "full", [4097] * 67 + [400_000]), (2, "similarity", [9])])
def test_statistics_of_plans_are_exact(gpu, K, level, sizes):
    """Every span's row of a plan is the integer result: rows of split chunks behind the spans' table of whole ones, the second
    level in one launch and in stripes, one, four and sixteen waves per span, full and ragged groups of four spans."""
    from jabas_amd import sync
    sets = [_whole_numbers(gpu, n, K, torch.float32, 7 * i + K) for i, n in enumerate(sizes)]
    plan = sync.SyncPlan([sync.SpanSpec(g) for g in sets])
    plan.ws.buf.fill_(float("nan"))
    plan.ws.stats.fill_(float("nan"))
    rows = plan.run(_quarter_args(K, torch.float32, level))
    for g, row in zip(sets, rows):
        assert torch.equal(row, _exact_row(g, level))


@pytest.mark.parametrize("K,dtype,level", [(1, torch.float32, None), (4, torch.float32, None), (4, torch.float32, "full"),
                                           (8, torch.bfloat16, "gram"), (9, torch.float32, "full"), (16, torch.bfloat16, "full")])
@pytest.mark.parametrize("numel", [1, 1023, 1025, 5 * 1024 + 3, 512 * 1024, 1024 * 1024 + 1, 2100 * 1024])
def test_short_launches_give_the_result_of_whole_chunks(gpu, K, dtype, level, numel):
    """How many workgroups share a chunk moves no element and no weight by a bit, whether the span comes by value or from a
    plan, in spans that end inside a tile: against K one-span launches, each with the elements of one chunk at most, where
    nothing is left to share. With scratch for a row per chunk only the launch takes whole chunks: same sums but for their order."""
    from jabas_amd import sync, _lib as L
    gen = torch.Generator(device=gpu).manual_seed(numel + K)
    grads = [torch.randn(numel, generator=gen, device=gpu).to(dtype) for _ in range(K)]
    p0, m0, v0 = (torch.randn(numel, generator=gen, device=gpu), torch.randn(numel, generator=gen, device=gpu) * 0.1,
                  torch.rand(numel, generator=gen, device=gpu))
    opt = dict(kind="adamw", betas=(0.9, 0.999), eps=1e-8, groups=[dict(lr=1e-2, weight_decay=0.0), dict(lr=2e-2, weight_decay=0.05)])
    args = sync.make_step_args((1,) * K, dtype, stats=level or False, opt=opt, step=3)
    cut = numel // 3
    bounds = [(0, 1)] if cut == 0 else [(0, 1), (cut, 0)]

    def launch(kind):
        p, m, v, agg = p0.clone(), m0.clone(), v0.clone(), torch.zeros(numel, device=gpu)
        span = sync.SpanSpec(grads, agg_out=agg, param=p, state1=m, state2=v, bounds=bounds)
        row = None
        if kind == "plan":
            row = sync.SyncPlan([span], sync.opt_kind(opt)).run(args)
        elif kind == "tight":
            ws = sync.Workspace.for_span(numel, dtype, gpu)
            tiles = -(-(numel + 63) // 1024)
            chunks = -(-tiles // (2 if K <= 4 and level else 4))
            width = {None: 1, "full": 4 + K, "gram": 4 + K + K * (K - 1) // 2}[level]
            ws.nbytes = (chunks + 33) * width * 8
            row = sync.sync_bucket(span, args, workspace=ws)
        elif kind == "span":
            row = sync.sync_bucket(span, args, workspace=sync.Workspace.for_span(numel, dtype, gpu))
        else:                                                   # one tile a launch
            for a in range(0, numel, 256):
                b = min(numel, a + 256)
                sl = slice(a, b)
                inner = [(0, 1 if a < cut or cut == 0 else 0)] + ([(cut - a, 0)] if a < cut < b else [])
                part = sync.make_step_args((1,) * K, dtype, opt=opt, step=3)
                sync.sync_bucket(sync.SpanSpec([g[sl] for g in grads], agg_out=agg[sl], param=p[sl], state1=m[sl], state2=v[sl],
                                               bounds=inner), part)
        return agg, p, m, v, None if row is None else row.reshape(-1).clone()

    ways = [launch("span"), launch("plan"), launch("tight")]
    if numel <= 8192:
        ways.append(launch("tiles"))
    for other in ways[1:]:
        for x, y in zip(ways[0][:4], other[:4]):
            assert torch.equal(x.view(torch.int32), y.view(torch.int32))
        if level and other[4] is not None:
            # fp64 sums of fp32 gradients: 2^-53 per addition of a chain of at most 700; bf16 gradients: fp32 chains of at
            # most 16 products per thread and 4 more over a row of lanes, 20 * 2^-24 of the sum of magnitudes
            tol = 700 * 2.0 ** -53 if dtype == torch.float32 else 20 * 2.0 ** -24
            norm = float(ways[0][4].abs().max())
            assert float((ways[0][4] - other[4]).abs().max()) <= tol * norm
    if level:
        norms = torch.stack([(g.double() ** 2).sum() for g in grads])
        tol = 1e-12 if dtype == torch.float32 else 20 * 2.0 ** -24
        torch.testing.assert_close(ways[0][4][4:4 + K], norms, rtol=tol, atol=0.0)


@pytest.mark.parametrize("K,dtype,kind,level", [
    (2, torch.float32, "sgd", None), (4, torch.float32, "sgd", "similarity"), (4, torch.bfloat16, "sgd", None), (8, torch.float32, "sgd", "similarity"),
    (1, torch.float32, "adam", "full"), (4, torch.bfloat16, "adamw_amsgrad", None), (8, torch.bfloat16, "adamw_amsgrad", "gram"),
    (12, torch.bfloat16, "adamw", "full"), (16, torch.float32, "adam", "similarity"), (16, torch.bfloat16, None, "full"), (6, torch.float32, None, None)])
@pytest.mark.parametrize("numel", [517, 2049, 90_001, 400_003])
def test_split_launches_of_every_kind(gpu, K, dtype, kind, level, numel):
    """Every optimizer, block size and level under a split: aggregate, weights and state against the first elements of a span that is
    not split (too long for it, too short for the rule of long steps), bit for bit; by value, as a plan of spans of unequal length (one of a single element, most shorter than a
    chunk) and with the step's scalars in device memory."""
    from jabas_amd import sync, _lib as L
    far = numel + (2_000_000 if K > 8 else 4_000_000)
    gen = torch.Generator(device=gpu).manual_seed(numel + K)
    grads = [torch.randn(far, generator=gen, device=gpu).to(dtype) for _ in range(K)]
    start = [torch.randn(far, generator=gen, device=gpu) * 0.1 for _ in range(2)] + [torch.rand(far, generator=gen, device=gpu) * 0.1 for _ in range(2)]
    n_state = {None: 0, "sgd": 2, "adam": 3, "adamw": 3, "adamw_amsgrad": 4}[kind]
    opt = None if kind is None else dict(kind=kind.replace("_amsgrad", ""), amsgrad="amsgrad" in kind, momentum=0.9, betas=(0.9, 0.999),
                                         eps=1e-8, groups=[dict(lr=1e-2, weight_decay=0.05)])

    def launch(cuts, stats, dyn=False):
        n = cuts[-1]
        state, agg = [t[:n].clone() for t in start[:n_state]], torch.zeros(n, device=gpu)
        args = sync.make_step_args((1,) * K, dtype, stats=stats or False, opt=opt, step=3)
        if dyn:
            scalars = sync.StepScalars(gpu)
            scalars.update(args)
            scalars.attach(args)
        spans = [sync.SpanSpec([g[a:b] for g in grads], agg_out=agg[a:b], **dict(zip(("param", "state1", "state2", "state3"), (t[a:b] for t in state))))
                 for a, b in zip(cuts, cuts[1:])]
        if len(spans) > 1:
            rows = sync.SyncPlan(spans, sync.opt_kind(opt)).run(args)
        else:
            rows = sync.sync_bucket(spans[0], args, workspace=sync.Workspace.for_span(n, dtype, gpu))
        return [agg, *state], None if not stats else rows.reshape(-1, L.STATS_STRIDE).sum(0)

    whole = sync.SyncPlan([sync.SpanSpec(grads, agg_out=torch.zeros(far, device=gpu), **dict(zip(("param", "state1", "state2", "state3"), start[:n_state])))],
                          sync.opt_kind(opt))
    assert int(whole._host.view(torch.uint8)[36]) == 1          # one workgroup per chunk
    want, _ = launch((0, far), None)
    ways = [launch((0, numel), level), launch((0, 256, 257, 300, 2 * numel // 3, numel), level)]
    if kind in ("sgd", "adam", "adamw"):
        ways.append(launch((0, numel), level, dyn=True))
    for got, row in ways:
        for x, y in zip(got, want):
            assert torch.equal(x.view(torch.int32), y[:numel].view(torch.int32))
        if level:
            # fp32 gradients: fp64 sums; bf16 gradients: fp32 chains of at most 16 products per thread and 4 more over a row of lanes
            tol = 1e-12 if dtype == torch.float32 else 20 * 2.0 ** -24
            torch.testing.assert_close(row[3], (got[0].double() ** 2).sum(), rtol=tol, atol=0.0)
            if level != "similarity":
                norms = torch.stack([(g[:numel].double() ** 2).sum() for g in grads])
                torch.testing.assert_close(row[4:4 + K], norms, rtol=tol, atol=0.0)


@pytest.mark.parametrize("K,dtype,kind,level", [(9, torch.float32, "adam", None), (16, torch.bfloat16, "sgd", None), (12, torch.bfloat16, "adamw_amsgrad", None),
                                                (9, torch.bfloat16, "adamw", "similarity"), (16, torch.float32, "sgd", "similarity")])
@pytest.mark.parametrize("change", [False, True])
@pytest.mark.parametrize("off_by", [-1, 1, 2049])
def test_long_steps_of_many_workers(gpu, K, dtype, kind, level, off_by, change):
    """On both sides of the length from which two workgroups share a chunk (2048 elements; from 2048 chunks on, with similarity sums
    4096; plain spans in which the group changes share theirs on both sides): weights, state and aggregate bit for bit those of
    three shorter launches, by value and as a plan, on the scratch that the sizing function names and on the least, which holds
    whole chunks only. The plan records which of them the launch is."""
    from jabas_amd import sync, _lib as L
    chunks = 4096 if level else 2048
    n = (chunks - 1) * 2048 + off_by
    gen = torch.Generator(device=gpu).manual_seed(K + off_by)
    grads = [torch.randn(n, generator=gen, device=gpu).to(dtype) for _ in range(K)]
    start = [torch.randn(n, generator=gen, device=gpu) * 0.1 for _ in range(2)] + [torch.rand(n, generator=gen, device=gpu) * 0.1 for _ in range(2)]
    start = start[:{"sgd": 2, "adamw_amsgrad": 4}.get(kind, 3)]
    opt = dict(kind=kind.replace("_amsgrad", ""), amsgrad="amsgrad" in kind, momentum=0.9, betas=(0.9, 0.999), eps=1e-8,
               groups=[dict(lr=1e-2, weight_decay=0.05), dict(lr=3e-3, weight_decay=0.0)])
    at = n // 2 + 77 if change else n

    def launch(cuts, plan, scratch=None):
        state, agg, rows = [t.clone() for t in start], torch.zeros(n, device=gpu), []
        args = sync.make_step_args((1,) * K, dtype, stats=level or False, opt=opt, step=3)
        for a, b in zip(cuts, cuts[1:]):
            bounds = ((0, 0), (at - a, 1)) if a < at < b else ((0, int(a >= at)),)
            span = sync.SpanSpec([g[a:b] for g in grads], agg_out=agg[a:b], bounds=bounds,
                                 **dict(zip(("param", "state1", "state2", "state3"), (t[a:b] for t in state))))
            if plan:
                p = sync.SyncPlan([span], sync.opt_kind(opt))
                assert int(p._host.view(torch.uint8)[36 + (2 if level else 0)]) == 1 + int(off_by > 0 or (change and not level))
                row = p.run(args)
            else:
                ws = sync.Workspace.for_span(b - a, dtype, gpu)
                ws.nbytes = scratch or ws.nbytes
                row = sync.sync_bucket(span, args, workspace=ws)
            if level:
                rows.append(row.reshape(-1)[:4].clone())
        return [agg, *state], sum(rows) if level else None

    want, sums = launch((0, n // 3 + 1, 2 * n // 3 + 2, n), False)
    ways = [launch((0, n), False), launch((0, n), True)]
    if level:
        ways.append(launch((0, n), False, scratch=(-(-n // 2048) + 33) * 4 * 8))    # a row per chunk, 33 for the finalize
    for got, row in ways:
        assert all(torch.equal(_bits(x), _bits(y)) for x, y in zip(got, want))
        if level:
            # as in the test of split launches above; the product of the halves against the size of its terms
            tol = 1e-12 if dtype == torch.float32 else 20 * 2.0 ** -24
            torch.testing.assert_close(row[1:], sums[1:], rtol=tol, atol=0.0)
            assert abs(float(row[0] - sums[0])) <= tol * float((sums[1] * sums[2]).sqrt())


@pytest.mark.parametrize("K,dtype,numel,levels", [(8, torch.bfloat16, 1_200_011, ("full", "gram")),
                                                  (4, torch.float32, 700_001, ("similarity", "full", "gram"))])
def test_levels_share_their_bits_on_any_scratch(gpu, K, dtype, numel, levels):
    """The sums that two statistics levels share are the same bits whatever scratch a call brings: what the sizing function
    returns, the least that every level takes, and sizes in between, which hold the rows of one level's split launch and only
    the whole chunks of a wider one."""
    from jabas_amd import sync, _lib as L
    gen = torch.Generator(device=gpu).manual_seed(numel)
    grads = [(torch.randn(numel, generator=gen, device=gpu) * 0.3 + 0.1).to(dtype) for _ in range(K)]
    span = sync.SpanSpec(grads)
    full_size = sync.Workspace.for_span(numel, dtype, gpu).nbytes
    chunks = -(-(-(-numel // 1024)) // (2 if K <= 4 else 4))
    widths = [{"similarity": 4, "full": 4 + K, "gram": 4 + K + K * (K - 1) // 2}[x] for x in levels]
    least = (chunks + 33) * widths[-1] * 8
    between = [(2 * chunks + 33) * w * 8 for w in widths[:-1]]
    for nbytes in (full_size, least, *(b for b in between if b > least), least + 4096):
        rows = []
        for level in levels:
            ws = sync.Workspace.for_span(numel, dtype, gpu)
            ws.nbytes = nbytes
            rows.append(sync.sync_bucket(span, sync.make_step_args((1,) * K, dtype, stats=level), workspace=ws).clone())
        for row, width in zip(rows[:-1], widths):
            assert torch.equal(row[:width].view(torch.int64), rows[-1][:width].view(torch.int64)), nbytes
    ws.nbytes = least - 8
    with pytest.raises(L.JabasSyncError):
        sync.sync_bucket(span, sync.make_step_args((1,) * K, dtype, stats=levels[-1]), workspace=ws)


@pytest.mark.parametrize("numel", [3, 1024, 1025, 70001])
@pytest.mark.parametrize("kind", ["sgd", "adamw", None])
@pytest.mark.parametrize("weight,scale,out", [(1.0, None, "own"), (1.0, 1.0, "own"), (1.0, 2.5, "own"), (1.0, float("nan"), "own"),
                                              (1.0, 0.37, "own"), (0.5, None, "own"), (0.5, 0.37, "own"), (1.0, None, "other"),
                                              (1.0, 2.5, "other")])
def test_aggregate_of_one_worker_over_its_own_buffer(gpu, numel, kind, weight, scale, out):
    """One fp32 worker of weight 1 that nothing scales is its own aggregate, and the launch writes none; any other weight, a
    coefficient under 1 and an output elsewhere are written. Every buffer against the oracle, bit for bit; infinities,
    negative zeros and denormals among the gradients."""
    from jabas_amd import sync
    gen = torch.Generator().manual_seed(numel)
    g = torch.randn(numel, generator=gen)
    g[:3] = torch.tensor([-0.0, float("-inf"), 1e-40])
    p0, m0, v0 = torch.randn(numel, generator=gen), torch.randn(numel, generator=gen), torch.rand(numel, generator=gen)
    opt = None if kind is None else dict(kind=kind, momentum=0.9, betas=(0.9, 0.999), eps=1e-8, groups=[dict(lr=1e-2, weight_decay=0.1)])
    want = g * weight
    if scale is not None and scale < 1.0:
        want = want * torch.tensor(scale)
    g_dev, res = g.to(gpu), []
    for own in (out == "own", False):                          # the second time out of place: the update is the same
        grad = g_dev.clone()
        agg = grad if own else torch.full((numel,), 7.0, device=gpu)
        state = [t.to(gpu).clone() for t in (p0, m0, v0)]
        coef = None if scale is None else torch.tensor([scale], device=gpu)
        args = sync.make_step_args((1,), torch.float32, opt=opt, step=2, grad_scale=coef)
        args.weight[0] = weight
        kw = {} if kind is None else dict(param=state[0], state1=state[1], state2=state[2] if kind == "adamw" else None)
        sync.sync_bucket(sync.SpanSpec([grad], agg_out=agg, **kw), args)
        res.append([agg, *state])
        if not own:
            assert torch.equal(grad.view(torch.int32), g_dev.view(torch.int32))
    for a, b in zip(*res):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    assert torch.equal(res[0][0].cpu().view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("K,dtype,kind,level", [(1, torch.float32, "adam", None), (3, torch.float32, "sgd", None), (4, torch.float32, "adamw", "similarity"),
                                                (8, torch.bfloat16, "adamw", "gram"), (8, torch.float32, "sgd", "gram"),
                                                (8, torch.float32, "adamw_amsgrad", "gram"), (13, torch.float32, "adam", "full"), (16, torch.bfloat16, "adamw_amsgrad", "full")])
@pytest.mark.parametrize("skew", [0, 1, 63])
def test_group_changes_and_ends_anywhere_in_a_wave(gpu, K, dtype, kind, level, skew):
    """Parameter groups that change at every place a wave's 256 elements can have it (inside a thread's four elements, between
    threads, waves and tiles, several times in one wave, every element), and spans that begin and end inside a wave, inside a
    thread's four elements or within one of them: aggregate, weights and state bit for bit, as one span by value and as a plan,
    nothing written beyond the span."""
    from jabas_amd import sync
    groups = [dict(lr=1e-2, weight_decay=0.05), dict(lr=3e-3, weight_decay=0.0), dict(lr=5e-2, weight_decay=0.01)]
    opt = dict(kind=kind.replace("_amsgrad", ""), amsgrad="amsgrad" in kind, momentum=0.9, betas=(0.9, 0.999), eps=1e-8, groups=groups)
    n_state = 1 if kind == "sgd" else 3 if "amsgrad" in kind else 2
    every = tuple(range(700, 720))
    for n, starts in ((1, ()), (2, (1,)), (3, (1, 2)), (255, (254,)), (257, (3, 4, 256)), (1021, (253, 255, 256, 257, 258, 511, 1020)),
                      (5003, (1, 2, 5, 1023, 1024, 1025, 2047, 2050, 4095, 4097, 5002)), (9001, every + (3001, 8191, 8192, 8999, 9000))):
        bounds = tuple((s, i % 3) for i, s in enumerate((0,) + starts))
        hg = _host_grads(K, n, 400 + K, dtype=dtype)
        p_h, state_h = _host_state(n, 11), [_host_state(n, 12, 1e-3), _host_state(n, 13, 1e-3).abs(), _host_state(n, 14, 1e-3).abs()][:n_state]
        start = [p_h.clone()] + [t.clone() for t in state_h]
        agg_h, rows_h = O.sync_step(hg, BATCHES[K], [(0, n, bounds)], opt, p_h, *state_h[:2], step=3, want_stats=True,
                                    **({"state3": state_h[2]} if n_state == 3 else {}))
        for plan in (False, True):
            def place(t):
                buf = torch.full((n + 192,), 7.25, dtype=t.dtype, device=gpu)
                buf[skew:skew + n].copy_(t)
                return buf
            whole = [place(t) for t in hg] + [place(torch.zeros(n))] + [place(t) for t in start]
            views = [b[skew:skew + n] for b in whole]
            span = sync.SpanSpec(views[:K], agg_out=views[K], param=views[K + 1], bounds=bounds,
                                 **{f"state{j + 1}": t for j, t in enumerate(views[K + 2:])})
            args = sync.make_step_args(BATCHES[K], dtype, stats=level or False, opt=opt, step=3)
            row = sync.SyncPlan([span], sync.opt_kind(opt)).run(args) if plan else sync.sync_bucket(span, args)
            for got, want in zip(views[K:], [agg_h, p_h, *state_h]):
                assert torch.equal(_bits(got), _bits(want)), (n, plan)
            for b in whole:
                assert bool((b[:skew] == 7.25).all()) and bool((b[skew + n:] == 7.25).all())
            if level:
                tol = 1e-11 if dtype == torch.float32 else 20 * 2.0 ** -24      # bf16: as in the test of split launches above
                torch.testing.assert_close(row.reshape(-1)[1:4].cpu(), rows_h[0][1:4], rtol=tol, atol=0.0)


@pytest.mark.parametrize("K,kind,level", [(1, "adamw", None), (1, "sgd", None), (3, "adam", "full"), (4, "adamw", "gram"), (12, "sgd", "similarity"),
                                          (2, None, "similarity")])
@pytest.mark.parametrize("n", [1, 5, 255, 1027, 70_003, 3_000_001])
def test_loose_gradients_at_any_element(gpu, K, kind, level, n):
    """Gradients (and an aggregate in one of them) at other positions of a 16-byte line than the buffers they update: aggregate,
    weights and state bit for bit those of aligned ones, by value and as a plan; refused without the flag and for bf16."""
    from jabas_amd import sync, _lib as L
    opt = None if kind is None else dict(kind=kind, momentum=0.9, betas=(0.9, 0.999), eps=1e-8,
                                         groups=[dict(lr=1e-2, weight_decay=0.05), dict(lr=3e-3, weight_decay=0.0)])
    bounds = ((0, 0), (n // 3, 1)) if kind and n > 3 else ((0, 0),)
    hg = _host_grads(K, n, 7)
    start = [_host_state(n, 21 + j).abs() for j in range({None: 0, "sgd": 2}.get(kind, 3))]
    args = sync.make_step_args(BATCHES[K], torch.float32, stats=level or False, opt=opt, step=3)

    def step(at, out_at, plan, loose=True, dtype=torch.float32):
        grads = [_dev(t.to(dtype), gpu, (at + 3 * k) % 7 if at else 0) for k, t in enumerate(hg)]
        state = [_dev(t, gpu, 5 if at else 0) for t in start]
        agg = grads[out_at] if isinstance(out_at, int) else _dev(torch.zeros(n), gpu, 5 if at else 0) if out_at else None
        span = sync.SpanSpec(grads, agg_out=agg, bounds=bounds if kind else (), loose_grads=loose,
                             **dict(zip(("param", "state1", "state2"), state)))
        a = args if dtype == torch.float32 else sync.make_step_args(BATCHES[K], dtype, stats=level or False, opt=opt, step=3)
        rows = sync.SyncPlan([span], sync.opt_kind(opt)).run(a) if plan else sync.sync_bucket(span, a)
        torch.cuda.synchronize()
        return [t for t in (agg, *state) if t is not None], rows, grads

    for out_at in ("own", 0, K - 1, None) if kind else ("own", 0, K - 1):
        want, rows, _ = step(0, out_at, False)
        for at in (1, 2, 6):
            for plan in (False, True):
                got, loose_rows, grads = step(at, out_at, plan)
                assert all(torch.equal(_bits(x), _bits(y)) for x, y in zip(got, want)), (out_at, at, plan)
                if level:
                    torch.testing.assert_close(loose_rows.reshape(-1), rows.reshape(-1), rtol=1e-11, atol=1e-25)
                for k, t in enumerate(grads):
                    if k != out_at:
                        assert torch.equal(_bits(t), _bits(hg[k]))
    with pytest.raises(L.JabasSyncError) as e:
        step(2, "own", False, loose=False)
    assert e.value.status == L.ERR_ALIGN
    if K > 1:
        with pytest.raises(L.JabasSyncError) as e:
            step(2, "own", True, dtype=torch.bfloat16)
        assert e.value.status == L.ERR_ALIGN


def test_a_copy_of_a_plan_outlives_the_plan(gpu):
    """copy.deepcopy of a plan carries its own tables, on the host and on the device: it runs after the plan it was made of is gone
    and its memory holds something else."""
    import copy
    import gc
    from jabas_amd import sync
    K, n = 3, 70_001
    hg = _host_grads(K, n, 3)
    grads, out = [_dev(t, gpu) for t in hg], torch.zeros(n, device=gpu)
    plan = sync.SyncPlan([sync.SpanSpec([g[a:b] for g in grads], agg_out=out[a:b]) for a, b in ((0, 30_004), (30_004, n))])
    size = plan._dev.numel()
    twin = copy.deepcopy(plan)
    del plan
    gc.collect()
    torch.cuda.synchronize()
    overwritten = [torch.zeros(size, dtype=torch.int64, device=gpu) for _ in range(64)]
    for seed in (3, 4):
        for g, t in zip(grads, _host_grads(K, n, seed)):
            g.copy_(t)
        twin.run(sync.make_step_args(BATCHES[K], torch.float32))
        torch.cuda.synchronize()
        assert torch.equal(_bits(out), _bits(O.aggregate(_host_grads(K, n, seed), BATCHES[K])))
    assert all(not bool(t.any()) for t in overwritten)


@pytest.mark.parametrize("K,dtype,kind,level", [(1, torch.float32, "adam", None), (2, torch.bfloat16, "sgd", "similarity"),
                                                (8, torch.float32, "adamw_amsgrad", "gram"), (16, torch.bfloat16, "adamw", "full")])
@pytest.mark.parametrize("every", [1, 3, 16, 100])
def test_dense_group_changes(gpu, K, dtype, kind, level, every):
    """Up to sixteen groups that come again and again inside a wave, up to 256 changes in it, over full tiles and span ends: the
    weights and state of one single-group step per group, bit for bit, by value and as a plan."""
    from jabas_amd import sync
    n, skew = 9_001, 3
    groups = [dict(lr=1e-3 * (1 + i), weight_decay=0.01 * (i % 5)) for i in range(16)]
    opt = dict(kind=kind.replace("_amsgrad", ""), amsgrad="amsgrad" in kind, momentum=0.9, betas=(0.9, 0.999), eps=1e-8, groups=groups)
    n_state = 1 if kind == "sgd" else 3 if "amsgrad" in kind else 2
    order = torch.randint(16, (-(-n // every),), generator=torch.Generator().manual_seed(every + K))
    order[:40] %= 2                  # and two groups in turn
    bounds = tuple((i * every, int(g)) for i, g in enumerate(order))
    group_of = order.repeat_interleave(every)[:n].to(gpu)
    hg = _host_grads(K, n, 41, dtype=dtype)
    start = [_host_state(n, 11)] + [_host_state(n, 12 + j, 1e-3).abs() for j in range(n_state)]

    def step(bounds, plan):
        grads, agg, state = [_dev(t, gpu, skew) for t in hg], _dev(torch.zeros(n), gpu, skew), [_dev(t, gpu, skew) for t in start]
        span = sync.SpanSpec(grads, agg_out=agg, bounds=bounds, **dict(zip(("param", "state1", "state2", "state3"), state)))
        args = sync.make_step_args(BATCHES[K], dtype, stats=level or False, opt=opt, step=3)
        row = sync.SyncPlan([span], sync.opt_kind(opt)).run(args) if plan else sync.sync_bucket(span, args)
        return [agg, *state], row

    want = [torch.zeros(n, device=gpu) for _ in range(2 + n_state)]
    for g in range(16):
        got, row_1 = step(((0, g),), False)
        want = [torch.where(group_of == g, x, w) for x, w in zip(got, want)]
    for plan in (False, True):
        got, row = step(bounds, plan)
        assert all(torch.equal(_bits(x), _bits(w)) for x, w in zip(got, want))
        if level:
            assert torch.equal(row.reshape(-1), row_1.reshape(-1))


@pytest.mark.parametrize("kind", [None, "sgd", "adamw", "adamw_amsgrad"])
@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 4099, 70_003])
def test_pair_products_of_eight_fp32_workers(gpu, kind, n):
    """The kernels that take every tile by itself, on both sides of a tile and of a workgroup's four, default halves and others:
    aggregate, weights and state bit for bit, every sum of the row against fp64, by value and as a plan."""
    from jabas_amd import sync
    K = 8
    opt = None if kind is None else dict(kind=kind.replace("_amsgrad", ""), amsgrad="amsgrad" in kind, momentum=0.9, betas=(0.9, 0.999), eps=1e-8,
                                         groups=[dict(lr=1e-2, weight_decay=0.05), dict(lr=3e-3, weight_decay=0.0)])
    bounds = ((0, 0), (n // 2, 1)) if kind and n > 1 else ((0, 0),)
    hg, n_state = _host_grads(K, n, 5), {None: 0, "sgd": 1, "adamw": 2, "adamw_amsgrad": 3}[kind]
    start = [_host_state(n, 11)] + [_host_state(n, 12 + j, 1e-3).abs() for j in range(n_state)]
    want = [t.clone() for t in start]
    if kind:
        agg_h, _ = O.sync_step(hg, BATCHES[K], [(0, n, bounds)], opt, *want[:3], step=3, **({"state3": want[3]} if n_state == 3 else {}))
    else:
        agg_h = O.aggregate(hg, BATCHES[K])
    products = torch.stack([t.double() for t in hg]) @ torch.stack([t.double() for t in hg]).t()
    size = products.diagonal().sqrt()
    for half in (None, (0, 1, 1, 0, 1, 0, 0, 1)):
        args = sync.make_step_args(BATCHES[K], torch.float32, stats="gram", opt=opt, step=3, half_id=half)
        for plan in (False, True):
            grads, agg, state = [_dev(t, gpu, 5) for t in hg], _dev(torch.zeros(n), gpu, 5), [_dev(t, gpu, 5) for t in start]
            span = sync.SpanSpec(grads, agg_out=agg, bounds=bounds if kind else (),
                                 **(dict(zip(("param", "state1", "state2", "state3"), state)) if kind else {}))
            row = (sync.SyncPlan([span], sync.opt_kind(opt)).run(args) if plan else sync.sync_bucket(span, args)).reshape(-1).cpu()
            assert torch.equal(_bits(agg), _bits(agg_h))
            if kind:
                assert all(torch.equal(_bits(x), _bits(y)) for x, y in zip(state, want))
            # fp64 sums of exact products: 2^-53 per addition, a thread's 16 and 256 threads of 18 workgroups
            tol = 1e-12
            torch.testing.assert_close(row[4:4 + K], products.diagonal(), rtol=tol, atol=0.0)
            pairs = [(i, j) for i in range(K) for j in range(i + 1, K)]
            for at, (i, j) in enumerate(pairs):
                assert abs(float(row[4 + K + at] - products[i, j])) <= tol * float(size[i] * size[j])
            torch.testing.assert_close(row[3], (agg_h.double() ** 2).sum(), rtol=tol, atol=0.0)


def test_dense_group_changes_cost_a_pass_per_group(gpu):
    """Two groups that change every 16 elements take two passes over the arithmetic, not one per change: 50 us against 30 for one
    group, of three million elements of four workers with similarity sums (107 with a pass per change, 3.6 times)."""
    from jabas_amd import sync
    K, n, n_set = 4, 3_000_000, 4
    opt = dict(kind="adamw", betas=(0.9, 0.999), eps=1e-8, groups=[dict(lr=1e-6, weight_decay=0.0), dict(lr=1e-6, weight_decay=0.01)])
    args = sync.make_step_args((1,) * K, torch.float32, stats="similarity", opt=opt, step=3)
    sets = [[torch.rand(n, device=gpu) * 1e-3 for _ in range(K + 3)] for _ in range(n_set)]

    def best(every):
        plans = [sync.SyncPlan([sync.SpanSpec(t[:K], agg_out=t[0], param=t[K], state1=t[K + 1], state2=t[K + 2],
                                              bounds=tuple((e, i & 1) for i, e in enumerate(range(0, n, every))))], sync.opt_kind(opt)) for t in sets]
        for p in plans:
            p.run(args)
        torch.cuda.synchronize()
        graph, begin, end, times = torch.cuda.CUDAGraph(), torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True), []
        with torch.cuda.graph(graph):
            for p in plans:
                p.run(args)
        for _ in range(20):
            begin.record()
            graph.replay()
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    one, dense = best(n), best(16)
    assert dense < 2.5 * one, (one, dense)
