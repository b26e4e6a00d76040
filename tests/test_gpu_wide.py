"""Rows wider than 1536 (needs an MI355X).

The reference accepts any width that is a multiple of 64: ``check_matrix``
tests only ``% 64`` (``csrc/kernels.cu:451-458``) and its score tile loops over
the whole width (``kernels.cu:150``).  Here rows wider than 1536 run scan
kernels whose query fragments ride through LDS beside the corpus rows instead
of staying in registers, a GEMV that takes the row 8 pieces at a time, and a
two-pass row preparation.  Everything is checked against the oracle at the
north star's bar (ids identical outside the 1e-3 near-tie band, scores within
1e-3; score matrices within 1e-3 fp32 / 3e-3 fp16), and ``Index.search``'s
"auto" must stay on the exact kernels at these widths.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from cuda_vector_search import Index, _ext
from cuda_vector_search import index as index_mod

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def make(n, d, b, seed=0):
    """Unit rows as tests/test_search.py:11-18."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, d, generator=g)
    q = torch.randn(b, d, generator=g)
    x = x / x.norm(dim=1, keepdim=True)
    q = q / q.norm(dim=1, keepdim=True)
    return x.half(), q.half()


@pytest.mark.parametrize("nq,n,d", [(37, 3001, 1600), (5, 1000, 2048), (32, 5000, 2048), (130, 2001, 3072),
                                    (3, 517, 4096), (257, 700, 1728), (64, 64, 4096)])
def test_wide_scores_match_oracle(eng, nq, n, d):
    say(f"wide scores nq={nq} n={n} d={d}")
    x, q = make(n, d, nq, seed=n + d)
    ref = oracle.scores(q, x)
    s = eng.scores(q.cuda(), x.cuda()).cpu().numpy()
    assert s.shape == (nq, n)
    np.testing.assert_allclose(s, ref, rtol=0, atol=1e-3)
    s16 = eng.scores(q.cuda(), x.cuda(), False)
    assert s16.dtype == torch.float16
    np.testing.assert_allclose(s16.float().cpu().numpy(), ref, rtol=0, atol=3e-3)


# The tiled-GEMM scan's tiles of 64 to 256 queries and 128 or 256 rows: batches a
# query past and short of them, odd row counts (stores off 16-byte alignment, a
# last tile of few rows), the narrowest width and ones past 1536; and sizes
# either side of where the query-stationary scan takes over.
TILED_SCORES = [(33, 60001, 64), (64, 50003, 512), (48, 16387, 1024), (64, 9001, 2048),  # 64 x 128
                (40, 270001, 256), (33, 263001, 1600),                                   # 64 x 256
                (65, 30005, 128), (255, 20002, 1088), (257, 30007, 192), (300, 8193, 384), (512, 40003, 640),
                (300, 8192, 1536), (129, 25007, 768), (513, 4101, 2048),                 # 128 x 128
                (100, 131077, 832), (300, 200003, 832),                                  # 128 x 256
                (256, 240001, 64), (512, 200003, 768),                                   # 256 x 256
                (128, 2049, 64), (200, 32770, 384), (300, 200003, 128), (128, 131077, 128)]


@pytest.mark.parametrize("nq,n,d", TILED_SCORES)
def test_tiled_scores_match_fp64(eng, nq, n, d):
    """The whole matrix, and nothing past its ends."""
    say(f"tiled scores nq={nq} n={n} d={d}")
    x, q = make(n, d, nq, seed=n + d)
    x, q = x.cuda(), q.cuda()
    ref = torch.cat([q.double() @ r.double().T for r in x.split(1 << 14)], 1)
    guard = 64
    for dtype in (torch.float32, torch.float16):
        buf = torch.full((nq * n + 2 * guard,), 7.0, dtype=dtype, device="cuda")
        out = buf[guard:guard + nq * n]
        rc = eng.lib.cvs_scores(q.data_ptr(), x.data_ptr(), nq, n, d, out.data_ptr(), int(dtype == torch.float32), 0, None)
        torch.cuda.synchronize()
        assert rc == 0, eng.lib.cvs_last_error()
        # unit rows: a sum of d products in fp32 is off by at most d 2^-24 (1 + rounding of the
        # norms); fp16 rounds scores below 1.01 by 2^-11 at most
        bound = 1.1 * d * 2.0**-24 + (2.0**-11 if dtype == torch.float16 else 0.0)
        assert float((out.view(nq, n).double() - ref).abs().max()) <= bound
        assert bool((buf[:guard] == 7).all()) and bool((buf[guard + nq * n:] == 7).all())


@pytest.mark.parametrize("n,d", [(1, 64), (5003, 384), (32768, 768), (32769, 768), (117022, 1024), (300007, 1024)])
def test_one_query_scores_match_fp64(eng, n, d):
    """The GEMV below 48 MB of corpus and from 512 MB on, the scan between them."""
    say(f"one-query scores n={n} d={d}")
    g = torch.Generator(device="cuda").manual_seed(n + d)
    x = torch.nn.functional.normalize(torch.randn(n, d, generator=g, device="cuda"), dim=1).half()
    q = torch.nn.functional.normalize(torch.randn(2, d, generator=g, device="cuda"), dim=1).half()
    ref = torch.cat([q[:1].double() @ r.double().T for r in x.split(1 << 16)], 1)
    for fp32 in (True, False):
        bound = 1.1 * d * 2.0**-24 + (0.0 if fp32 else 2.0**-11)
        assert float((eng.scores(q[:1], x, fp32).double() - ref).abs().max()) <= bound

    def best(rows):
        out = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            a.record()
            for _ in range(20):
                eng.scores(q[:rows], x)
            b.record()
            torch.cuda.synchronize()
            out.append(a.elapsed_time(b))
        return min(out)

    if n > 100000:  # (a second query costs the scan nothing; the GEMV took 1.25 times its time out of the MALL)
        assert best(1) < 1.15 * best(2)


WIDE_FUSED = [
    (20000, 1600, 1, 10),     # batch-1 GEMV
    (20000, 2048, 16, 10),    # 16-query block (16x16x32 MFMA)
    (30000, 2048, 32, 100),   # 32-query block, 4 row splits
    (20000, 3072, 64, 256),   # 64-query block, k = 256
    (40000, 4096, 128, 64),   # 128-query block
    (20000, 1728, 256, 10),   # two 128-query groups, odd stage count (27)
    (5000, 4096, 3, 1),       # k = 1 (arg-max)
    (300, 2048, 5, 150),      # tiny corpus, k > tile rows
]


@pytest.mark.parametrize("n,d,b,k", WIDE_FUSED)
def test_wide_fused_matches_oracle(eng, n, d, b, k):
    say(f"wide fused n={n} d={d} b={b} k={k}")
    x, q = make(n, d, b, seed=n + d + b + k)
    index = Index(x.cuda(), metric="ip")
    v, i = index.search(q.cuda(), k, method="fused")
    assert oracle.check_exact(q, x, k, v, i) >= 0.999


@pytest.mark.parametrize("flags", [_ext.FLAG_NO_PREPASS, _ext.FLAG_FORCE_PREPASS])
def test_wide_prepass_does_not_change_results(eng, flags):
    n, d, b, k = 30000, 2048, 100, 20
    say(f"wide prepass flags={flags}")
    x, q = make(n, d, b, seed=7)
    qd, xd = q.cuda(), x.cuda()
    v0, i0, _ = eng.fused_topk(qd, xd, k)
    v1, i1, _ = eng.fused_topk(qd, xd, k, flags=flags)
    torch.cuda.synchronize()
    assert torch.equal(v0, v1) and torch.equal(i0, i1)
    oracle.check_exact(q, x, k, v0.cpu().numpy(), i0.cpu().numpy().astype(np.int64))


@pytest.mark.parametrize("d", [1600, 2048, 4096])
@pytest.mark.parametrize("k", [1, 10, 100])
def test_wide_gemv_matches_oracle_and_scan(eng, d, k):
    say(f"wide gemv d={d} k={k}")
    x, q = make(30011, d, 1, seed=d + k)
    qd, xd = q.cuda(), x.cuda()
    v, i, plan = eng.fused_topk(qd, xd, k)
    v2, i2, plan2 = eng.fused_topk(qd, xd, k, flags=_ext.FLAG_NO_GEMV)
    torch.cuda.synchronize()
    assert plan.tolist()[0] == 1 and plan2.tolist()[0] == 16
    v, i = v.cpu().numpy(), i.cpu().numpy().astype(np.int64)
    oracle.check_exact(q, x, k, v, i)
    np.testing.assert_allclose(v, v2.cpu().numpy(), rtol=0, atol=1e-5)


def test_wide_forced_plans(eng):
    say("wide forced plans")
    x, q = make(20000, 2048, 50, seed=4)
    qd, xd = q.cuda(), x.cuda()
    base_v, base_i, _ = eng.fused_topk(qd, xd, 10)
    for bq, chunks in [(16, 1), (32, 7), (64, 1000), (128, 3)]:
        v, i, plan = eng.fused_topk(qd, xd, 10, bq, chunks)
        assert plan.tolist()[0] == bq
        assert torch.allclose(v, base_v, atol=1e-5) and torch.equal(i, base_i)
    with pytest.raises(RuntimeError, match="not supported at width"):
        eng.fused_topk(qd, xd, 10, 256)


def test_wide_index_auto_stays_exact_on_the_kernels(eng, monkeypatch):
    """"auto" never takes the fp16 torch path on gfx950 at these widths: k <= 256
    runs the fused kernels, 256 < k <= 1024 the exact large-k path."""
    n, d, b = 20000, 2000, 40  # d pads to 2048 (prep kernel, wide rows)
    say(f"wide index auto n={n} d={d} b={b}")
    x, q = make(n, d, b, seed=12)

    def no_torch(*a, **kw):
        raise AssertionError("auto took the torch path")

    monkeypatch.setattr(index_mod, "torch_topk", no_torch)
    index = Index(x.cuda(), metric="cosine")
    assert index._x.shape[1] == 2048 and index._xq is None
    qq = index._prep_queries(q.cuda())[:, :d].cpu()
    xs = index.embeddings.cpu()
    for k in (10, 256, 300, 1024):
        v, i = index.search(q.cuda(), k)
        assert v.dtype == torch.float32 and i.dtype == torch.int64
        oracle.check_exact(qq, xs, k, v, i)
    s = index.scores(q.cuda())
    np.testing.assert_allclose(s.cpu().numpy(), oracle.scores(qq, xs), rtol=0, atol=1e-3)
    with pytest.raises(ValueError, match="widths up to 1536"):
        index.search(q.cuda(), 10, method="int8")


def test_wide_twopass(eng):
    n, d, b, k = 10000, 3072, 8, 10
    say("wide twopass")
    x, q = make(n, d, b, seed=13)
    index = Index(x.cuda(), metric="ip")
    v, i = index.search(q.cuda(), k, method="twopass")
    oracle.check_exact(q, x, k, v, i, tol=2e-3)


@pytest.mark.parametrize("n,d,width", [(100, 2000, 2048), (33, 4096, 4096), (5, 1537, 1600), (64, 1600, 1600)])
def test_wide_prep_rows_matches_oracle(eng, n, d, width):
    say(f"wide prep_rows n={n} d={d} width={width}")
    g = torch.Generator().manual_seed(n + d)
    x = (torch.randn(n, d, generator=g) * torch.rand(n, 1, generator=g) * 10).half()
    x[0] = 0
    src = x.cuda()
    out = torch.full((n, width), float("nan"), dtype=torch.float16, device="cuda")
    eng.prep_rows(src, out, True)
    torch.cuda.synchronize()
    want = oracle.normalize_rows(x.numpy(), width=width)
    got = out.cpu().numpy()
    a, b = got.astype(np.float32), want.astype(np.float32)
    ulp = np.maximum(np.abs(np.spacing(got)), np.abs(np.spacing(want))).astype(np.float32)
    assert np.all(np.abs(a - b) <= ulp)
    assert not got[:, d:].any() and not got[0].any()
    if width == d:
        inplace = x.cuda()
        eng.prep_rows(inplace, inplace, True)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(inplace.cpu().numpy(), got)


def test_wide_int8_is_refused_by_the_engine(eng):
    x = torch.zeros(128, 2048, dtype=torch.float16, device="cuda")
    with pytest.raises(RuntimeError, match="widths up to 1536"):
        eng.q8_build(x)
    with pytest.raises(RuntimeError, match="widths up to 1536"):
        eng.q8_plan(4, 128, 2048, 10)


# The tiled-GEMM scan (auto plans past 32 queries at widths other than 384 and
# 768, once the corpus is too large for the score matrix): each tile shape,
# widths of one stage and up, partial tiles and query blocks, several
# groups, ties and lists that fill.
@pytest.mark.parametrize("nq,n,d,k,tile", [
    (33, 50001, 64, 1, (64, 128)), (64, 40001, 128, 100, (64, 128)), (60, 33001, 960, 10, (64, 128)),
    (40, 90001, 1024, 10, (64, 256)), (64, 70003, 1600, 64, (64, 256)),
    (257, 40003, 192, 17, (128, 128)), (600, 50000, 1088, 100, (128, 128)), (1000, 200001, 64, 10, (128, 128)),
    (65, 50001, 256, 10, (128, 256)), (128, 70000, 1024, 64, (128, 256)), (100, 33000, 1600, 256, (128, 256)),
    (300, 33001, 2048, 5, (128, 256)),
    (200, 33000, 640, 256, (256, 256)), (512, 60000, 1088, 100, (256, 256)), (256, 50000, 1088, 3, (256, 256)),
])
def test_tiled_scan_is_exact(eng, nq, n, d, k, tile):
    say(f"tiled scan nq={nq} n={n} d={d} k={k}")
    x, q = make(n, d, nq, seed=n + d + k)
    x[n // 2:n // 2 + 40] = x[3]  # exact ties
    q[1] = x[3]
    assert eng.search_path(nq, n, d, k) == ("tiled", *tile)
    xd, qd = x.cuda(), q.cuda()
    v, i, _ = eng.fused_topk(qd, xd, k)
    forced = 16 if d > 768 or k > 128 else 32
    assert eng.search_path(nq, n, d, k, bq=forced)[0] == "scan"  # the query-stationary scan
    v2, i2, p2 = eng.fused_topk(qd, xd, k, bq=forced)
    torch.cuda.synchronize()
    assert p2.tolist()[0] == forced
    oracle.check_exact(q, x, k, v.cpu().numpy(), i.cpu().numpy())
    # both sum the fp16 products in fp32 (in other orders): |S - S'| <= 2 d 2^-24 |q||x|
    torch.testing.assert_close(v, v2, rtol=0, atol=2 * d * 2.0**-24)
    assert (i != i2).float().mean().item() < 0.02


# Rows per list of 3 to 7 times its capacity (the last rows all pass), every tile
# and lists of 128, 256 and 512 entries.
@pytest.mark.parametrize("nq,n,d,k,tile", [(64, 400000, 64, 10, (64, 128)), (33, 260000, 1024, 10, (64, 256)),
                                           (1000, 100000, 128, 100, (128, 128)), (300, 340000, 576, 200, (128, 128)),
                                           (128, 200000, 1024, 10, (128, 256)), (256, 300000, 1024, 10, (256, 256))])
def test_tiled_scan_cuts_full_lists(eng, nq, n, d, k, tile):
    """Rows in ascending order of their scores fill every list several times over
    (no sampling), so that lists are cut to their k best as they go."""
    say(f"tiled scan, full lists nq={nq} n={n} d={d} k={k}")
    flags = _ext.FLAG_NO_PREPASS
    assert eng.search_path(nq, n, d, k) == eng.search_path(nq, n, d, k, flags=flags) == ("tiled", *tile)
    plan, _ = eng.plan(nq, n, d, k, flags=flags)
    cap = 128 if k <= 64 else 256 if k <= 192 else 512
    assert n / (2 * plan[1]) > 1.9 * cap
    g = torch.Generator(device="cuda").manual_seed(5)
    base = torch.nn.functional.normalize(torch.randn(1, d, generator=g, device="cuda"), dim=1)
    x = torch.empty(n, d, dtype=torch.float16, device="cuda")
    for lo in range(0, n, 1 << 16):
        r = torch.arange(lo, min(n, lo + (1 << 16)), device="cuda")
        x[r] = (base * (0.1 + 0.9 * r[:, None] / n) + 0.001 * torch.randn(len(r), d, generator=g, device="cuda")).half()
    q = (base + 0.01 * torch.randn(nq, d, generator=g, device="cuda")).half()
    v, i, _ = eng.fused_topk(q, x, k, flags=flags)
    v2, i2, _ = eng.fused_topk(q, x, k)
    torch.cuda.synchronize()
    assert torch.equal(v, v2) and torch.equal(i, i2)
    sel = torch.arange(0, nq, max(1, nq // 8))
    oracle.check_exact(q[sel].cpu(), x.cpu(), k, v[sel].cpu().numpy(), i[sel].cpu().numpy())


@pytest.mark.parametrize("nq,n,d,k,zeros,bq", [(64, 100000, 512, 10, 1, 64), (64, 100000, 512, 10, 8, 64),
                                               (48, 60001, 1024, 100, 2, 16), (300, 60001, 192, 200, 3, 16),
                                               (130, 40001, 640, 10, 40, 64)])
def test_tiled_scan_of_queries_of_zeros(eng, nq, n, d, k, zeros, bq):
    """Queries (padding) whose scores all tie: the smallest ids, the other queries'
    results as without them, and no longer than the query-stationary scan."""
    say(f"queries of zeros nq={nq} n={n} d={d} k={k} zeros={zeros}")
    x, q = make(n, d, nq, seed=n + d)
    q[:: nq // zeros][:zeros] = 0
    empty = (q == 0).all(1)
    assert eng.search_path(nq, n, d, k)[0] == "tiled" and eng.search_path(nq, n, d, k, bq=bq)[0] == "scan"
    xd, qd = x.cuda(), q.cuda()

    def best(**kw):
        out = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            a.record()
            for _ in range(3):
                r = eng.fused_topk(qd, xd, k, **kw)
            b.record()
            torch.cuda.synchronize()
            out.append(a.elapsed_time(b))
        return min(out), r[0].cpu(), r[1].cpu()

    tiled, v, i = best()
    qstat, v2, i2 = best(bq=bq)
    assert int(empty.sum()) == zeros
    assert torch.equal(i[empty], torch.arange(k, dtype=i.dtype).expand(zeros, k)) and not v[empty].any()
    oracle.check_exact(q[~empty], x, k, v[~empty].numpy(), i[~empty].numpy())
    torch.testing.assert_close(v, v2, rtol=0, atol=2 * d * 2.0**-24)
    assert tiled < 1.3 * qstat


@pytest.mark.parametrize("nq,n,d,k,bq,chunks", [
    (176, 29864, 448, 2, 128, 240), (256, 27757, 704, 1, 128, 224),  # 234, 217 tiles: one per workgroup, the last chunks
    (480, 21729, 448, 12, 256, 88), (2002, 7654, 512, 11, 256, 32),  # empty; 85, 30 tiles of 256 rows
    (192, 18339, 832, 2, 128, 144), (112, 16857, 832, 1, 128, 132)])  # several groups: no longer the 64-query scan
def test_tiles_are_chosen_by_the_plan_that_runs(eng, nq, n, d, k, bq, chunks):
    """The costs compared are those of the chunk counts that are then run."""
    say(f"tile choice nq={nq} n={n} d={d} k={k}")
    plan, _ = eng.plan(nq, n, d, k)
    assert plan == [bq, chunks] and eng.search_path(nq, n, d, k)[0] == "tiled"
    x, q = make(n, d, nq, seed=nq)
    v, i, _ = eng.fused_topk(q.cuda(), x.cuda(), k)
    torch.cuda.synchronize()
    oracle.check_exact(q, x, k, v.cpu().numpy(), i.cpu().numpy())


@pytest.mark.parametrize("nq,n,d,k,path", [
    (55, 135823, 1408, 1, "scan"), (36, 218849, 2048, 5, "scan"), (62, 799357, 896, 3, "scan"),
    (81, 485581, 576, 254, "scan"), (82, 197167, 128, 80, "scan"),  # 7 to 33% slower through the tiles
    (46, 120242, 1792, 5, "tiled"), (64, 300000, 256, 10, "tiled"), (100, 600000, 1024, 50, "tiled")])
def test_one_query_group_takes_the_tiles_where_they_are_faster(eng, nq, n, d, k, path):
    assert eng.search_path(nq, n, d, k)[0] == path


def test_noalloc_keeps_what_its_scratch_held(eng):
    """The allocation-free search of sizes whose tiled plan outgrows its scratch
    runs the query-stationary plan, as it did."""
    nq, n, d, k = 1000, 200000, 128, 10
    assert eng.search_path(nq, n, d, k)[0] == "tiled"
    _, ws = eng.plan(nq, n, d, k)
    assert ws > _ext.NOALLOC_SCRATCH_BYTES
    x, q = make(n, d, nq, seed=9)
    xd, qd = x.cuda(), q.cuda()
    v = torch.empty((nq, k), dtype=torch.float32, device="cuda")
    i = torch.empty((nq, k), dtype=torch.int32, device="cuda")
    rc = eng.lib.cvs_fused_topk_noalloc(qd.data_ptr(), xd.data_ptr(), nq, n, d, k, 0, v.data_ptr(), i.data_ptr(), None,
                                        0, eng._stream(qd.device))
    assert rc == 0, eng.lib.cvs_last_error()
    v2, i2, _ = eng.fused_topk(qd, xd, k)
    torch.cuda.synchronize()
    torch.testing.assert_close(v, v2, rtol=0, atol=2 * d * 2.0**-24)
    assert (i != i2).float().mean().item() < 0.001


@pytest.mark.parametrize("nq,n,d,k", [(513, 9000, 384, 10), (700, 4100, 768, 20), (300, 2100, 768, 5), (257, 600, 320, 3)])
def test_several_query_groups_are_exact(eng, nq, n, d, k):
    """3, 5 and 6 query groups: chunk counts that are multiples of 8 and not, some
    chunks empty, on every path that splits its corpus by groups."""
    say(f"groups nq={nq} n={n} d={d} k={k}")
    x, q = make(n, d, nq, seed=nq + n)
    index = Index(x.cuda(), metric="ip", int8_prefilter=True)
    for method in ("fused", "int8"):
        v, i = index.search(q.cuda(), k, method=method)
        oracle.check_exact(q, x, k, v.cpu().numpy(), i.cpu().numpy())
    np.testing.assert_allclose(index.scores(q.cuda()).cpu().numpy(), oracle.scores(q, x), rtol=0, atol=1e-3)
