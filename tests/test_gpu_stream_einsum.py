"""Tile einsums on extents the blocked MFMA kernels do not take (the streaming
GEMM): every number of 16-wide fragments and its edges, K tails, all operand
layouts, one and four waves per output block, short and long segments, against
float64; the same bits on every path that plans an einsum."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import reference_path as R

import einjax_amd as ej
from einjax_amd import _device, _lib
from einjax_amd.execution.engine import ContractionPlan, ContractionStep

pytestmark = pytest.mark.gpu

# m, k, n: fragment edges (16), block edges (5 fragments), K blocks of 16 (fp32)
# and 32 (bf16) with their tails, single rows and columns, several blocks.
SIZES = [(1, 8, 1), (90, 33, 1), (16, 16, 16), (17, 15, 33), (33, 31, 17), (48, 33, 49), (75, 75, 75),
         (80, 80, 81), (81, 47, 80), (5, 100, 64), (64, 9, 1), (100, 20, 125), (161, 24, 97)]
SPECS = {"ij,jk->ik": ("mk", "kn"), "ij,kj->ik": ("mk", "nk"), "ji,jk->ik": ("km", "kn"),
         "ji,kj->ik": ("km", "nk"), "ij,jk->ki": ("mk", "kn")}


def _tol(dtype, out, products):
    """rel-L2 bound: every product and partial sum rounds to 2^-24 of its
    value, which over a sum of n terms grows as sqrt(n); a bf16 result (8
    significand bits) rounds once more, by at most 2^-8 of itself."""
    return 2.0 ** -24 * np.sqrt(products) * 2 + (2.0 ** -8 if out == torch.bfloat16 else 0)


def _case(spec, m, k, n, dtype, seed, tiles=7, pairs=40, segs=9):
    rng = np.random.default_rng(seed)
    ext = dict(m=m, k=k, n=n)
    lt, rt = (tuple(ext[x] for x in t) for t in SPECS[spec])
    lv, rv = (rng.standard_normal((tiles, *t)).astype(np.float32) for t in (lt, rt))
    if dtype == torch.bfloat16:
        lv, rv = R.bf16_round(lv), R.bf16_round(rv)
    li, ri = rng.integers(0, tiles, pairs), rng.integers(0, tiles, pairs)
    off = np.sort(np.concatenate([[0, pairs], rng.integers(0, pairs, segs - 1)])).astype(np.int32)
    perm = rng.permutation(pairs).astype(np.int32)
    return lt, rt, lv, rv, li, ri, perm, off


def _run(spec, lt, rt, lv, rv, li, ri, perm, off, dtype, out=None):
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    return _device.segment_einsum(_device.describe(spec, lt, rt), dev(lv).to(dtype),
                                  dev(rv).to(dtype), dev(li), dev(ri), dev(perm), dev(off), out)


@pytest.mark.parametrize("spec", SPECS)
@pytest.mark.parametrize("m,k,n", SIZES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_segments(gpu, spec, m, k, n, dtype):
    """Segments of zero to many pairs: few blocks, four waves each."""
    print("[case] stream segments", spec, m, k, n, dtype, flush=True)
    c = _case(spec, m, k, n, dtype, m * 131 + k * 17 + n)
    lt, rt, lv, rv, li, ri, perm, off = c
    pv = R.kernel_einsum(lv, rv, li, ri, spec, precision="fp64")[perm]
    want = np.stack([pv[a:b].sum(0) for a, b in zip(off[:-1], off[1:])])
    longest = int(np.diff(off).max()) * k
    for out in {dtype, torch.float32}:
        got = _run(spec, *c, dtype, out)
        assert got.dtype == out
        err = R.rel_l2(got.float().cpu().numpy(), want)
        assert err <= _tol(dtype, out, longest), (out, err)
    empty = np.flatnonzero(np.diff(off) == 0)
    assert not got[torch.from_numpy(empty).cuda()].any()


@pytest.mark.parametrize("m,k,n,spec", [(20, 20, 20, "ij,jk->ik"), (75, 75, 75, "ij,jk->ik"),
                                        (36, 25, 50, "ij,kj->ik"), (50, 45, 33, "ji,jk->ik")])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_many_pairs_one_wave_each(gpu, m, k, n, spec, dtype):
    """Per-pair results of more pairs than split blocks, and of a few of them
    (four waves), both within rounding of float64."""
    print("[case] stream pairs", spec, m, k, n, dtype, flush=True)
    lt, rt, lv, rv, li, ri, _, _ = _case(spec, m, k, n, dtype, 3, pairs=2500)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    desc = _device.describe(spec, lt, rt)
    args = dev(lv).to(dtype), dev(rv).to(dtype)
    many = _device.pair_einsum(desc, *args, dev(li), dev(ri))
    few = _device.pair_einsum(desc, *args, dev(li[:300]), dev(ri[:300]))
    want = R.kernel_einsum(lv, rv, li, ri, spec, precision="fp64")
    for got, ref in ((many, want), (few, want[:300])):
        assert R.rel_l2(got.float().cpu().numpy(), ref) <= _tol(dtype, dtype, k)


def _segment_sums(lv, rv, li, ri, perm, off, spec):
    """float64 segment sums on the GPU; a pair with an index out of range adds nothing."""
    ok = (li >= 0) & (li < len(lv)) & (ri >= 0) & (ri < len(rv))
    pv = R.kernel_einsum(lv, rv, np.where(ok, li, 0), np.where(ok, ri, 0), spec, precision="fp64")
    pv[~ok] = 0
    pv = pv[perm]
    return np.stack([pv[a:b].sum(0) for a, b in zip(off[:-1], off[1:])])


@pytest.mark.parametrize("spec,m,k,n", [("ij,jk->ik", 20, 37, 33), ("ij,kj->ik", 75, 21, 18),
                                        ("ji,jk->ik", 33, 40, 50)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_long_segments(gpu, spec, m, k, n, dtype):
    """Segments of more pairs than a wave's lanes hold (64 at a time): 63 to
    129 and 300 pairs, invalid pairs on both sides of a reload."""
    print("[case] stream long segments", spec, m, k, n, dtype, flush=True)
    lens = [63, 64, 65, 0, 128, 129, 1, 300]
    off = np.cumsum([0] + lens).astype(np.int32)
    lt, rt, lv, rv, li, ri, perm, _ = _case(spec, m, k, n, dtype, 5, pairs=int(off[-1]))
    li[perm[off[2] + 63]], ri[perm[off[2] + 64]], li[perm[off[7] + 191]] = -1, len(rv), len(lv)
    want = _segment_sums(lv, rv, li, ri, perm, off, spec)
    got = _run(spec, lt, rt, lv, rv, li, ri, perm, off, dtype, torch.float32).cpu().numpy()
    assert R.rel_l2(got, want) <= _tol(dtype, torch.float32, 300 * k)
    for u, x in enumerate(lens):
        assert R.rel_l2(got[u], want[u]) <= _tol(dtype, torch.float32, max(x, 1) * k), u
    assert not got[3].any()


@pytest.mark.parametrize("live", [0, 1, 200, 2047, 2048, 2600])
@pytest.mark.parametrize("t,dtype", [(40, torch.float32), (20, torch.bfloat16)])
def test_segment_bound(gpu, t, dtype, live):
    """A launch sized for 2,600 segments of 0 to several pairs of which `live`
    are there: bitwise the launch of exactly those, float64 within rounding,
    nothing written past them."""
    print("[case] stream bound", t, dtype, live, flush=True)
    rng = np.random.default_rng(live)
    bound, pairs = 2600, 6000
    lt, rt, lv, rv, li, ri, perm, _ = _case("ij,jk->ik", t, t, t, dtype, 9, pairs=pairs)
    off = np.sort(rng.integers(0, pairs, bound + 1)).astype(np.int32)
    off[3] = off[2]
    li[5], ri[11] = len(lv), -1
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    a, b, dli, dri, dperm, doff = (dev(lv).to(dtype), dev(rv).to(dtype), dev(li), dev(ri),
                                   dev(perm), dev(off))
    desc = _device.describe("ij,jk->ik", lt, rt)
    out = torch.full((bound, t, t), 7.0, device="cuda")
    desc.out_dtype = _lib.EJ_F32
    nlive = torch.tensor([live], dtype=torch.int64, device="cuda")
    assert _lib.load().ej_segment_einsum_async(
        ctypes.byref(desc), _lib.EJ_BF16 if dtype == torch.bfloat16 else _lib.EJ_F32,
        _device.ptr(a), _device.ptr(b), a.shape[0], b.shape[0], _device.ptr(dli),
        _device.ptr(dri), _device.ptr(dperm), _device.ptr(doff), bound, _device.ptr(nlive), None,
        0, _device.ptr(out), _device.stream_ptr()) == _lib.EJ_OK
    assert bool((out[live:] == 7.0).all())
    if live == 0:
        return
    exact = _device.segment_einsum(desc, a, b, dli, dri, dperm, doff[:live + 1].contiguous(),
                                   torch.float32)
    assert torch.equal(out[:live], exact)
    want = _segment_sums(lv, rv, li, ri, perm, off[:live + 1], "ij,jk->ik")
    longest = max(int(np.diff(off[:live + 1]).max()), 1) * t
    assert R.rel_l2(exact.cpu().numpy(), want) <= _tol(dtype, torch.float32, longest)


def _relation(rng, keep, t, dtype):
    c = np.ascontiguousarray(np.argwhere(keep), dtype=np.int32)
    v = torch.from_numpy(rng.standard_normal((len(c), t, t)).astype(np.float32)).cuda().to(dtype)
    return ej.SparseTensorRelation(torch.from_numpy(c).cuda(), v,
                                   tuple(g * t for g in keep.shape), (t, t))


@pytest.mark.parametrize("rhs", ["sparse", "dense"])
@pytest.mark.parametrize("t,dtype", [(40, torch.float32), (75, torch.float32), (80, torch.bfloat16)])
def test_same_bits_on_every_path(gpu, t, dtype, rhs):
    """Fewer output tiles than the split's 2,048, bounds above it: the plan
    counted first, the row or dense plan, the prepared step, the queued plan,
    an engine step on new relations, all bitwise alike (fp32 results)."""
    print("[case] stream paths", t, dtype, rhs, flush=True)
    rng = np.random.default_rng(t)
    if rhs == "sparse":  # about 2,800 pairs, 1,700 output tiles, bound 2,500
        ka, kb = rng.random((50, 50)) < 0.15, rng.random((50, 50)) < 0.15
        ka[7], kb[9] = False, False
    else:  # 60 lhs tiles in 40 of 70 rows, 40 rhs columns: 1,600 output tiles, bound 2,400
        ka, kb = np.zeros((70, 12), bool), np.ones((12, 40), bool)
        rows = rng.permutation(70)[:40]
        ka[rows, rng.integers(0, 6, 40)] = True
        ka[rows[:20], rng.integers(6, 12, 20)] = True
    L, Rr = _relation(rng, ka, t, dtype), _relation(rng, kb, t, dtype)
    join, spec, agg = [(1, 0)], "ij,jk->ik", [(0, 0), (1, 1)]
    li, ri = ej.coordinate_join(L, Rr, join)
    coords, offsets, perm, _ = _device.segment_plan(L.coords, Rr.coords, li, ri, agg,
                                                    [ka.shape[0], kb.shape[1]])
    P, U = li.numel(), coords.shape[0]
    assert P > 2048 > U and int(torch.diff(offsets).max()) > 1
    desc = _device.describe(spec, (t, t), (t, t))
    want = _device.segment_einsum(desc, L.values, Rr.values, li, ri, perm, offsets, torch.float32)
    for call in range(3):  # counted first (or the dense plan), then queued, then prepared
        got = ej.execute_sparse(L, Rr, join, spec, agg, out_dtype=torch.float32)
        assert torch.equal(got.coords, coords) and torch.equal(got.values, want), call
    status, res = _device.queued_segment_einsum(
        L.coords, Rr.coords, join, [kb.shape[0]], agg, [ka.shape[0], kb.shape[1]],
        _device.describe(spec, (t, t), (t, t)), L.values, Rr.values, 4 * P, torch.float32)
    assert status == "ok" and torch.equal(res[4], want)
    anew = [ej.SparseTensorRelation(r.coords.clone(), r.values.clone(), r.shape, r.tile_shape)
            for r in (L, Rr)]
    engine = ej.ExecutionEngine(out_dtype=torch.float32)
    got = engine.execute_plan(ContractionPlan(spec, [ContractionStep(0, spec, (0, 1))]), anew)
    assert torch.equal(got.coords, coords) and torch.equal(got.values, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("spec", ["ij,jk->ik", "ij,kj->ik", "ji,jk->ik", "ji,kj->ik"])
def test_neighbour_tiles_and_invalid_pairs(gpu, spec, dtype):
    """A K tail or an edge never mixes in the neighbouring tiles (all NaN
    here), and a pair with an index out of range adds nothing."""
    print("[case] stream neighbours", spec, dtype, flush=True)
    m, k, n = 35, 21, 50
    lt, rt, lv, rv, _, _, _, _ = _case(spec, m, k, n, dtype, 11)
    lv[[0, 2]] = np.nan
    rv[[0, 2]] = np.nan
    li, ri = np.array([1, 1, 9, 1, -1]), np.array([1, 1, 1, 9, 1])
    off, perm = np.array([0, 1, 5], np.int32), np.arange(5, dtype=np.int32)
    got = _run(spec, lt, rt, lv, rv, li, ri, perm, off, dtype, torch.float32).cpu().numpy()
    want = R.kernel_einsum(lv, rv, li[:1], ri[:1], spec, precision="fp64")[0]
    assert R.rel_l2(got[0], want) <= _tol(dtype, torch.float32, k)
    np.testing.assert_array_equal(got[0], got[1])


THIN = [("ij,ij->i", (5, 8), (5, 8)), ("ij,ij->i", (33, 75), (33, 75)),
        ("ij,ij->i", (130, 256), (130, 256)), ("ij,ij->j", (19, 70), (19, 70)),
        ("ij,ij->j", (64, 3), (64, 3)), ("bij,bjk->bik", (3, 2, 21), (3, 21, 4)),
        ("bij,bjk->bik", (65, 6, 8), (65, 8, 6)), ("bij,bjk->bik", (7, 1, 32), (7, 32, 36)),
        ("bij,bjk->bik", (4, 1, 16), (4, 16, 128)), ("bij,bkj->bik", (9, 2, 45), (9, 4, 45)),
        ("bij,bkj->ikb", (6, 4, 8), (6, 2, 8)), ("bji,bkj->bik", (11, 17, 5), (11, 3, 17)),
        ("bij,bjk->kib", (32, 4, 16), (32, 16, 4)), ("ijb,jkb->ikb", (16, 9, 7), (9, 16, 7)),
        ("bji,bjk->bik", (3, 13, 6), (3, 13, 6))]


@pytest.mark.parametrize("spec,lt,rt", THIN)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_thin_batched_products(gpu, spec, lt, rt, dtype):
    """Few outputs per batch index: both operands, one or neither contiguous
    along the contraction, tails of the vectors and of the lanes that share an
    output, every order of the output; empty segments, invalid pairs, NaN in
    tiles that no pair names, an address off 16 bytes; a launch sized for more
    segments than are there."""
    print("[case] thin", spec, lt, rt, dtype, flush=True)
    rng = np.random.default_rng(sum(lt) + sum(rt))
    lv, rv = (R.bf16_round(rng.standard_normal((6, *t)).astype(np.float32)) for t in (lt, rt))
    li, ri = rng.integers(0, 5, 40), rng.integers(0, 5, 40)
    li[[0, 7]], ri[11] = (-1, 6), 6
    off = np.array([0, 1, 1, 9, 30, 30, 40], np.int32)
    perm = rng.permutation(40).astype(np.int32)
    want = _segment_sums(lv, rv, li, ri, perm, off, spec)
    lv[5], rv[5] = np.nan, np.nan

    def shifted(a):
        flat = torch.zeros(a.size + 1, dtype=dtype, device="cuda")
        flat[1:] = torch.from_numpy(a.reshape(-1)).cuda().to(dtype)
        return flat[1:].view(a.shape)

    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    a, b, idx = shifted(lv), shifted(rv), [dev(x) for x in (li, ri, perm, off)]
    desc = _device.describe(spec, lt, rt)
    f32 = _device.segment_einsum(desc, a, b, *idx, torch.float32)
    assert R.rel_l2(f32.cpu().numpy(), want) <= _tol(dtype, torch.float32, 21 * desc.k)
    assert not f32[1].any() and not f32[4].any()
    assert torch.equal(_device.segment_einsum(desc, a, b, *idx, dtype), f32.to(dtype))
    out = torch.full((6, *f32.shape[1:]), 7.0, device="cuda")
    desc.out_dtype = _lib.EJ_F32
    nlive = torch.tensor([4], dtype=torch.int64, device="cuda")
    assert _lib.load().ej_segment_einsum_async(
        ctypes.byref(desc), _lib.EJ_BF16 if dtype == torch.bfloat16 else _lib.EJ_F32,
        _device.ptr(a), _device.ptr(b), 6, 6, *(_device.ptr(x) for x in idx), 6,
        _device.ptr(nlive), None, 0, _device.ptr(out), _device.stream_ptr()) == _lib.EJ_OK
    assert torch.equal(out[:4], f32[:4]) and bool((out[4:] == 7.0).all())


@pytest.mark.parametrize("spec,lt,rt", [
    ("ij,ij->j", (64, 64), (64, 64)), ("ij,ij->i", (16, 16), (16, 16)),
    ("bij,bjk->bik", (64, 2, 8), (64, 8, 2)), ("bij,bjk->bik", (64, 1, 8), (64, 8, 16)),
    ("ijb,jkb->ikb", (8, 8, 32), (8, 8, 32))])
def test_thin_batched_products_are_no_slower(gpu, spec, lt, rt):
    """These shapes are no slower than one thread per output, which integer
    tiles take: measured at a tenth to a half of its time."""
    print("[case] thin time", spec, lt, rt, flush=True)
    rng = np.random.default_rng(1)
    idx = [torch.from_numpy(rng.integers(0, 256, 20000)).cuda() for _ in range(2)]
    desc = _device.describe(spec, lt, rt)
    times = {}
    for dt in (torch.float32, torch.int32):
        a, b = (torch.randint(-9, 9, (256, *t), device="cuda", dtype=torch.int32).to(dt)
                for t in (lt, rt))
        ts = []
        for _ in range(8):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(5):
                _device.pair_einsum(desc, a, b, *idx)
            t1.record()
            torch.cuda.synchronize()
            ts.append(t0.elapsed_time(t1))
        times[dt] = sorted(ts)[4]
    assert times[torch.float32] <= 1.3 * times[torch.int32], times


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_unaligned_base_and_batch(gpu, dtype):
    """Tiles at an address that is no multiple of 16, and a batch label."""
    print("[case] stream unaligned", dtype, flush=True)
    rng = np.random.default_rng(2)
    spec, lt, rt = "bij,bjk->bik", (3, 19, 37), (3, 37, 21)
    lv, rv = (R.bf16_round(rng.standard_normal((5, *t)).astype(np.float32)) for t in (lt, rt))
    li, ri = rng.integers(0, 5, 30), rng.integers(0, 5, 30)

    def shifted(a):
        flat = torch.zeros(a.size + 1, dtype=dtype, device="cuda")
        flat[1:] = torch.from_numpy(a.reshape(-1)).cuda().to(dtype)
        return flat[1:].view(a.shape)

    got = _device.pair_einsum(_device.describe(spec, lt, rt), shifted(lv), shifted(rv),
                              torch.from_numpy(li).cuda(), torch.from_numpy(ri).cuda())
    want = R.kernel_einsum(lv, rv, li, ri, spec, precision="fp64")
    assert R.rel_l2(got.float().cpu().numpy(), want) <= _tol(dtype, dtype, 37)


@pytest.mark.parametrize("m,k,n", [(64, 32, 64), (64, 96, 192), (128, 32, 128), (256, 64, 128),
                                   (128, 160, 256)])
@pytest.mark.parametrize("spec", ["ij,jk->ik", "ij,jk->ki"])
def test_pair_results_in_lines(gpu, m, k, n, spec):
    """Per-pair bf16 results of 64 and 128 blocks: rows stored in lines (bf16
    results), as they come (fp32 results, transposed results, an output that is
    not 16-byte aligned): all of them one fp32 result, rounded once."""
    print("[case] pair lines", spec, m, k, n, flush=True)
    lt, rt, lv, rv, li, ri, _, _ = _case("ij,jk->ik", m, k, n, torch.bfloat16, m + k + n)
    li[3] = len(lv)  # out of range: a tile of zeros
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    a, b, dli, dri = dev(lv).bfloat16(), dev(rv).bfloat16(), dev(li), dev(ri)
    desc = _device.describe(spec, lt, rt)
    f32 = _device.pair_einsum(desc, a, b, dli, dri, out_dtype=torch.float32)
    got = _device.pair_einsum(desc, a, b, dli, dri)
    want = R.kernel_einsum(lv, rv, np.where(li < len(lv), li, 0), ri, spec, precision="fp64")
    want[3] = 0
    assert R.rel_l2(f32.cpu().numpy(), want) <= _tol(torch.bfloat16, torch.float32, k)
    assert torch.equal(got, f32.bfloat16())
    flat = torch.zeros(got.numel() + 1, dtype=torch.bfloat16, device="cuda")
    assert _lib.load().ej_pair_einsum(
        ctypes.byref(desc), _lib.EJ_BF16, _device.ptr(a), _device.ptr(b), a.shape[0], b.shape[0],
        _device.ptr(dli), _device.ptr(dri), len(li), _device.ptr(flat[1:]),
        _device.stream_ptr()) == _lib.EJ_OK
    assert torch.equal(flat[1:].view(got.shape), got)


@pytest.mark.parametrize("m,n", [(64, 64), (128, 128), (128, 256)])
@pytest.mark.parametrize("k", [448, 512, 576])
def test_pair_results_of_few_long_products(gpu, m, n, k):
    """Per-pair bf16 products of a long contraction, few of them (deep stages)
    and many (the ring): the same bits, and float64 within rounding."""
    print("[case] few long pairs", m, n, k, flush=True)
    lt, rt, lv, rv, li, ri, _, _ = _case("ij,jk->ik", m, k, n, torch.bfloat16, k, pairs=600)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    a, b, li_, ri_ = dev(lv).bfloat16(), dev(rv).bfloat16(), dev(li), dev(ri)
    desc = _device.describe("ij,jk->ik", lt, rt)
    for out in (torch.float32, torch.bfloat16):
        many = _device.pair_einsum(desc, a, b, li_, ri_, out_dtype=out)
        few = _device.pair_einsum(desc, a, b, li_[:40], ri_[:40], out_dtype=out)
        assert torch.equal(many[:40], few)
        want = R.kernel_einsum(lv, rv, li[:40], ri[:40], "ij,jk->ik", precision="fp64")
        assert R.rel_l2(few.float().cpu().numpy(), want) <= _tol(torch.bfloat16, out, k)


@pytest.mark.parametrize("spec", ["ij,kj->ik", "ji,jk->ik"])
@pytest.mark.parametrize("m,k,n", [(32, 32, 32), (64, 64, 64), (128, 32, 128), (96, 160, 32),
                                   (32, 64, 192), (192, 96, 96)])
def test_fp32_ring_transposed_layouts(gpu, spec, m, k, n):
    """The backward's fp32 layouts on blocked extents: every block shape, one
    and several K stages, segments of zero to many pairs (one and several to a
    workgroup), an invalid pair, NaN tiles that no pair names."""
    print("[case] fp32 ring", spec, m, k, n, flush=True)
    for pairs, segs in ((40, 9), (150, 2100)):
        lt, rt, lv, rv, li, ri, perm, off = _case(spec, m, k, n, torch.float32, m + k + n,
                                                  pairs=pairs, segs=segs)
        li[li == 3], ri[ri == 5] = 2, 4
        pv = R.kernel_einsum(lv, rv, li, ri, spec, precision="fp64")
        lv[3], rv[5] = np.nan, np.nan
        li[7] = len(lv)
        pv[7] = 0
        pv = pv[perm]
        want = np.stack([pv[a:b].sum(0) for a, b in zip(off[:-1], off[1:])])
        got = _run(spec, lt, rt, lv, rv, li, ri, perm, off, torch.float32)
        longest = int(np.diff(off).max()) * k
        assert R.rel_l2(got.cpu().numpy(), want) <= _tol(torch.float32, torch.float32, longest)


@pytest.mark.parametrize("spec,lt,rt", [("ij,jk->ik", (64, 32), (32, 64)),
                                        ("ij,kj->ik", (32, 64), (64, 64)),
                                        ("ji,jk->ik", (32, 128), (32, 32)),
                                        ("ji,kj->ik", (32, 32), (32, 32)),
                                        ("ij,jk->ik", (20, 20), (20, 20)),
                                        ("ij,ij->ij", (8, 8), (8, 8))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_tile_counts_beyond_31_bits(gpu, spec, lt, rt, dtype):
    """Relations said to hold 2^31 tiles (the pairs name the first few) are
    taken, by the kernels whose tile indices are 64-bit."""
    print("[case] tile counts", spec, lt, rt, dtype, flush=True)
    rng = np.random.default_rng(4)
    lv, rv = (R.bf16_round(rng.standard_normal((5, *t)).astype(np.float32)) for t in (lt, rt))
    li, ri = rng.integers(0, 5, 12), rng.integers(0, 5, 12)
    dev = lambda a: torch.from_numpy(a).cuda()
    a, b, dli, dri = dev(lv).to(dtype), dev(rv).to(dtype), dev(li), dev(ri)
    desc = _device.describe(spec, lt, rt)
    desc.out_dtype = _lib.EJ_F32
    want = R.kernel_einsum(lv, rv, li, ri, spec, precision="fp64")
    out = torch.empty(want.shape, device="cuda")
    assert _lib.load().ej_pair_einsum(
        ctypes.byref(desc), _lib.EJ_BF16 if dtype == torch.bfloat16 else _lib.EJ_F32,
        _device.ptr(a), _device.ptr(b), 1 << 31, 1 << 31, _device.ptr(dli), _device.ptr(dri), 12,
        _device.ptr(out), _device.stream_ptr()) == _lib.EJ_OK
    assert R.rel_l2(out.cpu().numpy(), want) <= _tol(dtype, torch.float32, max(desc.k, 1))


@pytest.mark.parametrize("pairs", [(1 << 23) - 1, 1 << 23])
def test_launches_near_their_limit(gpu, pairs):
    """Row products of 33 outputs, eight lanes each: two workgroups a pair, of
    which 2^24 are one too many for a launch; the generic kernel takes those."""
    print("[case] launch limit", pairs, flush=True)
    torch.manual_seed(0)
    a, b = (torch.randint(-3, 4, (50, 33, 32), device="cuda").float() for _ in range(2))
    li, ri = (torch.randint(0, 50, (pairs,), device="cuda") for _ in range(2))
    got = _device.pair_einsum(_device.describe("ij,ij->i", (33, 32), (33, 32)), a, b, li, ri)
    table = (a[:, None] * b[None]).sum(-1)  # small whole numbers: exact in any order
    assert torch.equal(got, table[li, ri])


@pytest.mark.parametrize("spec", ["ij,ik->jk", "ik,jk->ij"])
def test_fp32_gradients_of_several_blocks_are_no_slower(gpu, spec):
    """Gradient layouts on 96 x 96 tiles (3 x 3 blocks) are no slower than both
    operands transposed, which the register-staged kernel takes: measured at
    0.8 of its time (a walk over several blocks took 1.5 times as long)."""
    print("[case] fp32 gradient time", spec, flush=True)
    rng = np.random.default_rng(1)
    pairs, tiles, t = 10496, 4096, 96
    a = torch.randn((128, t, t), device="cuda")
    g = torch.randn((pairs, t, t), device="cuda")
    ident = torch.arange(pairs, device="cuda")
    other = torch.from_numpy(rng.integers(0, 128, pairs)).cuda()
    seg = np.sort(rng.integers(0, tiles, pairs))
    off = torch.from_numpy(np.searchsorted(seg, np.arange(tiles + 1)).astype(np.int32)).cuda()
    perm = torch.from_numpy(rng.permutation(pairs).astype(np.int32)).cuda()
    times = []
    for s in (spec, "ji,kj->ik"):
        desc = _device.describe(s, (t, t), (t, t))
        args = (a, g, other, ident) if spec == "ij,ik->jk" else (g, a, ident, other)
        ts = []
        for _ in range(8):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(5):
                _device.segment_einsum(desc, *args, perm, off)
            t1.record()
            torch.cuda.synchronize()
            ts.append(t0.elapsed_time(t1))
        times.append(sorted(ts)[4])
    assert times[0] <= 1.15 * times[1], times
