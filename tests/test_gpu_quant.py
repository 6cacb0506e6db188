"""int8 scalar-quantized scan and PQ-ADC scan on the GPU against the oracle.
Both are bit-exact paths: int32 scores, fp32 tables/ADC sums formed in the
reference's order, L1 re-rank summed in index order."""
import numpy as np
import pytest

from oracle import oracle as O
from parity import assert_sorted_unique, recall
from vectorstorekit_amd import (ProductQuantizer, ScalarQuantizer, SQ8Database, VectorDatabase,
                                VSKError)
from vectorstorekit_amd._lib import METRIC_COSINE, METRIC_L1, METRIC_L2, METRIC_L2SQ

pytestmark = pytest.mark.gpu


# ------------------------------------------------------------------ SQ8 ---

@pytest.mark.parametrize("per_dim", [True, False])
def test_sq8_train_encode_bit_exact(ctx, per_dim):
    rng = np.random.default_rng(1)
    x = rng.standard_normal((5000, 45)).astype(np.float32) * 3
    sq = ScalarQuantizer(ctx, per_dim=per_dim)
    s, o = sq.train(x)
    es, eo = O.sq8_train(x, per_dim)
    np.testing.assert_array_equal(s, es)
    np.testing.assert_array_equal(o, eo)
    np.testing.assert_array_equal(sq.quantizeBatch(x), O.sq8_encode(x, es, eo))


@pytest.mark.parametrize("shape", [(20_000, 128, 37, 100), (3000, 45, 70, 10), (500, 7, 3, 1),
                                   (30_000, 200, 130, 50), (20_000, 300, 40, 20),
                                   (8000, 700, 20, 10), (3000, 1100, 9, 5),
                                   (40_000, 64, 1100, 10)])
def test_sq8_search_bit_exact(ctx, shape):
    """Every scan variant: code lengths of 1, 2, 4, 8 and 16 64-byte k-steps
    (register-resident kernel) and over 1024 bytes (LDS kernel); several
    query groups and filtered chunks; a duplicated row for the tie rule."""
    n, d, nq, k = shape
    print(f"sq8 n={n} d={d} nq={nq} k={k}", flush=True)
    rng = np.random.default_rng(n + d)
    codes = rng.integers(-128, 128, (n, d)).astype(np.int8)
    qc = rng.integers(-128, 128, (nq, d)).astype(np.int8)
    codes[7] = codes[3]
    qc[0] = codes[3]
    db = SQ8Database(ctx, codes)
    gs, gi = db.search(qc, k)
    os_, oi = O.sq8_search(qc, codes, k)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gs, os_)


def test_sq8_scores_past_float_precision(ctx):
    """Scores above 2^24 that differ by 1 (d = 2048, the LDS kernel): the
    higher score ranks first, ties by row id; int64 brute force."""
    d = 2048
    q = np.full((2, d), 127, np.int8)
    q[0, 5] = 1
    codes = np.full((300, d), 127, np.int8)
    codes[0, 5] = 126
    codes[2, 7] = 126
    codes[4:] = np.random.default_rng(3).integers(-128, 128, (296, d)).astype(np.int8)
    gs, gi = SQ8Database(ctx, codes).search(q, 6)
    os_, oi = O.sq8_search(q, codes, 6)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gs, os_)
    ref = codes.astype(np.int64) @ q[0].astype(np.int64)
    assert list(gi[0, :4]) == [1, 3, 0, 2] and ref[1] - ref[0] == 1


def test_sq8_chunked_and_overflow(ctx):
    """Scores fall with the row id, so every filtered chunk overflows."""
    n, d = 150_000, 32
    codes = np.zeros((n, d), np.int8)
    codes[:, 0] = (np.arange(n) * 255 // n - 128).astype(np.int8)
    codes[:, 1] = np.random.default_rng(2).integers(-128, 128, n).astype(np.int8)
    qc = np.zeros((3, d), np.int8)
    qc[0, 0] = 127
    qc[1, 0] = -128
    qc[2, 1] = 5
    gs, gi = SQ8Database(ctx, codes).search(qc, 50)
    os_, oi = O.sq8_search(qc, codes, 50)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gs, os_)


def test_config4_full_size(ctx):
    """10M x 128 N(0,1) quantised per dimension, 1,000
    queries quantised with the same parameters, k=100; scores and ids
    bit-exact on all 1,000 queries."""
    import torch

    n, d, nq, k = 10_000_000, 128, 1000, 100
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    x = torch.randn(n, d, generator=g, device="cuda")
    g.manual_seed(2)
    q = torch.randn(nq, d, generator=g, device="cuda")
    print("config4 sq8 10Mx128 q1000 k100", flush=True)
    sq = ScalarQuantizer(ctx, per_dim=True)
    s, o = sq.train(x)
    codes = sq.quantizeBatch(x)
    xs = x[:4096].cpu().numpy()
    del x
    qc = sq.quantizeBatch(q)
    db = SQ8Database(ctx, codes)
    gs, gi = db.search(qc, k)
    gs, gi = gs.cpu().numpy(), gi.cpu().numpy()
    assert (np.diff(gs, axis=1) <= 0).all()
    ch, qh = codes.cpu().numpy(), qc.cpu().numpy()
    os_, oi = O.sq8_search(qh, ch, k)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gs, os_)
    # scores are the integer dots of the returned rows
    for qi in (100, 999):
        np.testing.assert_array_equal(
            gs[qi], ch[gi[qi]].astype(np.int64) @ qh[qi].astype(np.int64))
    # encode parity on a row sample
    np.testing.assert_array_equal(ch[:4096], O.sq8_encode(xs, s, o))


# ------------------------------------------------------------------- PQ ---

def _pq_data(seed, n, d, M, ksub, nq, ncent=64):
    rng = np.random.default_rng(seed)
    cent = (2.0 * rng.standard_normal((ncent, d))).astype(np.float32)
    x = (cent[rng.integers(0, ncent, n)] + 0.5 * rng.standard_normal((n, d))).astype(np.float32)
    q = (cent[rng.integers(0, ncent, nq)] + 0.5 * rng.standard_normal((nq, d))).astype(np.float32)
    dsub = d // M
    cb = np.stack([O.kmeans(x[:4096, m * dsub:(m + 1) * dsub].copy(), ksub, iters=4, seed=m)
                   for m in range(M)])
    return x, q, cb


@pytest.mark.parametrize("shape", [(20_000, 128, 16, 256, 30), (5000, 24, 6, 100, 9),
                                   (6000, 64, 4, 256, 70)])
def test_pq_lut_encode_adc_bit_exact(ctx, shape):
    """Tables, codes and ADC search bit-exact; the shapes cover the table
    kernel's segment lengths 8, 4 and 16, fewer codewords than threads, and
    two query batches (70 queries)."""
    n, d, M, ksub, nq = shape
    print(f"pq n={n} d={d} M={M} ksub={ksub} nq={nq}", flush=True)
    x, q, cb = _pq_data(n, n, d, M, ksub, nq)
    pq = ProductQuantizer(ctx, cb)
    codes = pq.encode(x)
    np.testing.assert_array_equal(codes, O.pq_encode(x, cb))
    lut = pq.precomputeDistanceTables(q)
    for qi in range(nq):
        np.testing.assert_array_equal(lut[qi], O.pq_lut(q[qi], cb))
    pq.add(codes)
    for k_adc, k in [(100, 100), (300, 10)]:
        gd, gi = pq.search(q, k, k_adc=k_adc)
        od, oi = O.pq_search(q, cb, codes, k_adc, k)
        np.testing.assert_array_equal(gi, oi)
        np.testing.assert_array_equal(gd, od)


@pytest.mark.parametrize("shape", [(3000, 20, 4, 64), (3000, 64, 4, 256), (2000, 192, 2, 256)])
def test_pq_encode_codebook_layouts(ctx, shape):
    """Encode through each kernel variant: generic dsub in LDS (dsub 5),
    compile-time dsub (16), and codebooks too large for LDS (dsub 96, 96 KB)
    read from global memory.  Codes bit-exact against the oracle."""
    n, d, M, ksub = shape
    print(f"pq encode n={n} d={d} M={M} ksub={ksub}", flush=True)
    x, q, cb = _pq_data(n + 7, n, d, M, ksub, 4)
    pq = ProductQuantizer(ctx, cb)
    np.testing.assert_array_equal(pq.encode(x), O.pq_encode(x, cb))


@pytest.mark.parametrize("dsub", [4, 8, 16])
@pytest.mark.parametrize("M,ksub", [(1, 129), (3, 256), (5, 200), (16, 256)])
def test_pq_encode_matrix_cores_bit_exact(ctx, M, ksub, dsub):
    """The matrix-core encoder at the edges of its 64-row waves and of its
    16-codeword tiles, on data its screen cannot decide: codewords in exact
    and near ties (the lower index, the smaller fp32 sum), rows on codewords,
    a large common offset, magnitudes of 1e-25 and 1e25, zeros, infinities
    and NaN, and rows that start at 4 bytes past an aligned address."""
    import torch

    rng = np.random.default_rng(M + ksub + dsub)
    for n, offset, scale in [(1, 0, 1), (63, 0, 1), (65, 100, 1), (1000, 0, 1), (700, 0, 1e-25),
                             (500, 0, 1e25), (300, 1e4, 1)]:
        cb = rng.standard_normal((M, ksub, dsub)).astype(np.float32) + np.float32(offset)
        cb[:, 7] = cb[:, 3]  # exact ties
        cb[:, 100] = cb[:, 50] * np.float32(1 + 2e-7)
        x = rng.standard_normal((n, M * dsub)).astype(np.float32) + np.float32(offset)
        x[::5] = cb[:, rng.integers(0, ksub, len(x[::5]))].transpose(1, 0, 2).reshape(-1, M * dsub)
        x[1::9] = np.tile(cb[:, 50].reshape(-1), (len(x[1::9]), 1))
        cb, x = cb * np.float32(scale), x * np.float32(scale)
        x[2::50] = 0
        if n == 1000:
            x[10, ::3], x[20, 1], x[30] = np.inf, np.nan, -np.inf
        print(f"pq encode M={M} ksub={ksub} dsub={dsub} n={n} scale={scale}", flush=True)
        with np.errstate(all="ignore"):
            want = O.pq_encode(x, cb)
        pq = ProductQuantizer(ctx, cb)
        np.testing.assert_array_equal(pq.encode(x), want)
        flat = torch.zeros(1 + x.size, device="cuda")
        flat[1:] = torch.from_numpy(x).reshape(-1)
        torch.cuda.synchronize()
        got = pq.encode(flat[1:].view(n, M * dsub))
        np.testing.assert_array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("metric", [METRIC_L1, METRIC_L2, METRIC_L2SQ, METRIC_COSINE])
def test_pq_rerank_bit_exact(ctx, metric):
    x, q, cb = _pq_data(5, 30_000, 64, 8, 256, 20)
    pq = ProductQuantizer(ctx, cb)
    codes = O.pq_encode(x, cb)
    pq.add(codes[:10_000])
    pq.add(codes[10_000:])  # appended in two calls
    db = VectorDatabase(ctx, x)
    gd, gi = pq.search(q, 100, k_adc=1000, rerank_metric=metric, rerank_db=db)
    od, oi = O.pq_search(q, cb, codes, 1000, 100, x=x, rerank_metric=metric)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)


@pytest.mark.parametrize("shape", [(200_000, 32, 8, 256, 40, 300, 50),
                                   (60_000, 128, 16, 256, 20, 1000, 100),
                                   (60_000, 64, 32, 64, 25, 200, 20)])
def test_pq_screen_bit_exact(shape):
    """The ADC scan through the bf16 screen (forced at these sizes): decoded
    rows in a bf16 plane, the flat screen with each query's exact threshold
    plus the bound, the survivors' exact ADC keys.  Segment lengths 4, 8 and
    2; one or two filtered chunks after the dense first; with and without
    the L1 re-rank; rows added after the plane was made.  Bit-exact against
    the oracle."""
    import os

    from vectorstorekit_amd import Context

    n, d, M, ksub, nq, k_adc, k = shape
    print(f"pq screen n={n} d={d} M={M} nq={nq} kadc={k_adc} k={k}", flush=True)
    x, q, cb = _pq_data(n + d, n, d, M, ksub, nq)
    codes = O.pq_encode(x, cb)
    old = os.environ.get("VSK_FLAT_KERNEL")
    os.environ["VSK_FLAT_KERNEL"] = "screen"
    try:
        sctx = Context(0)
    finally:
        if old is None:
            del os.environ["VSK_FLAT_KERNEL"]
        else:
            os.environ["VSK_FLAT_KERNEL"] = old
    sctx.profile(True)
    pq = ProductQuantizer(sctx, cb)
    pq.add(codes)
    gd, gi = pq.search(q, k, k_adc=k_adc)
    assert "pq_screen_rescore" in sctx.profile_stats(), "the screen did not run"
    od, oi = O.pq_search(q, cb, codes, k_adc, k)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd.view(np.uint32), od.view(np.uint32))
    db = VectorDatabase(sctx, x)
    gd, gi = pq.search(q, k, k_adc=k_adc, rerank_metric=METRIC_L1, rerank_db=db)
    od, oi = O.pq_search(q, cb, codes, k_adc, k, x=x, rerank_metric=O.L1)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd.view(np.uint32), od.view(np.uint32))
    # rows added after the plane was made: it is made again
    pq.add(codes[:5000])
    gd, gi = pq.search(q[:5], k, k_adc=k_adc)
    od, oi = O.pq_search(q[:5], cb, np.concatenate([codes, codes[:5000]]), k_adc, k)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd.view(np.uint32), od.view(np.uint32))
    sctx.close()


def test_pq_upload_one_call_matches_create_add(ctx):
    x, q, cb = _pq_data(6, 12_000, 32, 4, 256, 15)
    codes = O.pq_encode(x, cb)
    up = ProductQuantizer.upload(ctx, cb, codes)
    ref = ProductQuantizer(ctx, cb)
    ref.add(codes)
    ud, ui = up.search(q, 50, k_adc=50)
    rd, ri = ref.search(q, 50, k_adc=50)
    np.testing.assert_array_equal(ui, ri)
    np.testing.assert_array_equal(ud, rd)
    od, oi = O.pq_search(q, cb, codes, 50, 50)
    np.testing.assert_array_equal(ui, oi)
    np.testing.assert_array_equal(ud, od)
    with pytest.raises(VSKError):
        ProductQuantizer.upload(ctx, cb[:, :100], codes)


def test_config5_full_size(ctx):
    """10M x 128 from a 1,024-Gaussian mixture, PQ M=16 x
    256 (codebooks trained on a 65,536-row sample), 1,000 queries, ADC top-1000
    then exact L1 re-rank -> k=100.  Bit-exact on all 1,000 queries; recall@100
    vs exact L1 search equal to the oracle's on the first 100."""
    import torch

    n, d, nq, M, ksub = 10_000_000, 128, 1000, 16, 256
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    cent = 2.0 * torch.randn(1024, d, generator=g, device="cuda")
    g.manual_seed(5)
    a = torch.randint(0, 1024, (n,), generator=g, device="cuda")
    qa = torch.randint(0, 1024, (nq,), generator=g, device="cuda")
    g.manual_seed(1)
    x = cent[a] + 0.5 * torch.randn(n, d, generator=g, device="cuda")
    g.manual_seed(2)
    q = cent[qa] + 0.5 * torch.randn(nq, d, generator=g, device="cuda")
    print("config5 pq 10Mx128 M16x256 q1000 kadc1000 k100 L1", flush=True)
    sample = x[:65536].cpu().numpy()
    dsub = d // M
    cb = np.stack([O.kmeans(sample[:, m * dsub:(m + 1) * dsub].copy(), ksub, iters=8, seed=m)
                   for m in range(M)])
    pq = ProductQuantizer(ctx, cb)
    codes = pq.encode(x)
    pq.add(codes)
    db = VectorDatabase(ctx, x)
    gd, gi = pq.search(q, 100, k_adc=1000, rerank_metric=METRIC_L1, rerank_db=db)
    gd, gi = gd.cpu().numpy(), gi.cpu().numpy()
    assert_sorted_unique(gd, gi)
    xh, qh, ch = x.cpu().numpy(), q.cpu().numpy(), codes.cpu().numpy()
    np.testing.assert_array_equal(ch[:20_000], O.pq_encode(xh[:20_000], cb))
    od, oi = O.pq_search(qh, cb, ch, 1000, 100, x=xh, rerank_metric=O.L1)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd.view(np.uint32), od.view(np.uint32))
    sub = 100
    td, ti = O.search_flat(qh[:sub], xh, 100, O.L1)
    assert recall(gi[:sub], ti) == recall(oi[:sub], ti)
    print(f"config5 recall@100 on {sub} queries: {recall(gi[:sub], ti):.4f}", flush=True)


@pytest.mark.parametrize("per_dim", [True, False])
def test_sq8_dequantize_bit_exact(ctx, per_dim):
    """dequantizeFromInt8 on the GPU: (code - offset) / scale, rounded per
    operation, bit-exact against the oracle; device tensors stay on device."""
    import torch

    rng = np.random.default_rng(7)
    x = rng.standard_normal((4000, 33)).astype(np.float32) * 2
    sq = ScalarQuantizer(ctx, per_dim=per_dim)
    s, o = sq.train(x)
    codes = sq.quantizeBatch(x)
    np.testing.assert_array_equal(sq.dequantize(codes), O.sq8_decode(codes, s, o))
    out = sq.dequantize(torch.from_numpy(codes).cuda())
    assert out.is_cuda
    np.testing.assert_array_equal(out.cpu().numpy(), O.sq8_decode(codes, s, o))


def test_pq_decode_bit_exact(ctx):
    x, q, cb = _pq_data(11, 5000, 48, 6, 256, 3)
    pq = ProductQuantizer(ctx, cb)
    codes = O.pq_encode(x, cb)
    np.testing.assert_array_equal(pq.decode(codes), O.pq_decode(codes, cb))
