"""Failure handling, forced from the host (VSK_FAULT=<kind>:<n>): the n-th
device allocation, launch check or end-of-call synchronisation of a context
reports an error although the GPU work itself ran normally.  Each injected
fault must surface as the status the reference's error vocabulary maps it
to (outOfMemory / executionFailed), and the same context must then answer
a search exactly as the oracle does (recovery: the fault fires once, the
call's partial state is dropped)."""
import os

import numpy as np
import pytest

from oracle import oracle as O
from vectorstorekit_amd import Context, IVFConfiguration, IVFIndex, VectorDatabase, VSKError

OUT_OF_MEMORY, EXECUTION_FAILED = -5, -6  # vsk_status (vsk_hip.h)

pytestmark = pytest.mark.gpu


def _armed(spec):
    old = os.environ.get("VSK_FAULT")
    os.environ["VSK_FAULT"] = spec
    try:
        return Context(0)
    finally:
        if old is None:
            del os.environ["VSK_FAULT"]
        else:
            os.environ["VSK_FAULT"] = old


@pytest.mark.parametrize("spec,status", [("alloc:1", OUT_OF_MEMORY),
                                         ("alloc:3", OUT_OF_MEMORY),
                                         ("launch:1", EXECUTION_FAILED),
                                         ("launch:4", EXECUTION_FAILED),
                                         ("sync:1", EXECUTION_FAILED),
                                         ("sync:2", EXECUTION_FAILED)])
def test_injected_fault_maps_and_recovers(spec, status):
    rng = np.random.default_rng(21)
    x = rng.standard_normal((3000, 40)).astype(np.float32)
    q = rng.standard_normal((25, 40)).astype(np.float32)
    ctx = _armed(spec)
    raised = None
    try:
        for _ in range(3):  # enough events for every spec above
            db = VectorDatabase(ctx, x)
            db.search(q, 10, "euclideanSquared")
            db.free()
    except VSKError as e:
        raised = e
    assert raised is not None, "the armed fault did not fire"
    assert raised.status == status, raised
    assert "injected fault" in str(raised)
    # the context recovers: a full upload and search match the oracle
    db = VectorDatabase(ctx, x)
    gd, gi = db.search(q, 10, "euclideanSquared")
    od, oi = O.search_flat(q, x, 10, O.L2SQ)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)
    db.free()
    ctx.close()


def test_unarmed_and_malformed_specs_do_nothing():
    rng = np.random.default_rng(22)
    x = rng.standard_normal((500, 8)).astype(np.float32)
    for spec in ("", "launch", "launch:0", "nothing:3", "sync:-2"):
        ctx = _armed(spec)
        db = VectorDatabase(ctx, x)
        gd, gi = db.search(x[:5], 3, "euclideanSquared")
        od, oi = O.search_flat(x[:5], x, 3, O.L2SQ)
        np.testing.assert_array_equal(gi, oi)
        db.free()
        ctx.close()


@pytest.mark.parametrize("spec", ["launch:3", "sync:2"])
def test_profile_reset_after_failed_profiled_call(spec):
    """With per-kernel timing on, a call that fails after some of its
    timers closed leaves no pending timings behind: vsk_profile_reset and
    the next call see clean statistics (the next call's timings name only
    statistics that exist)."""
    rng = np.random.default_rng(23)
    x = rng.standard_normal((4000, 32)).astype(np.float32)
    q = rng.standard_normal((30, 32)).astype(np.float32)
    ctx = _armed(spec)
    ctx.profile(True)
    db = VectorDatabase(ctx, x)
    raised = None
    try:
        for _ in range(3):
            db.search(q, 10, "euclideanSquared")
    except VSKError as e:
        raised = e
    assert raised is not None, "the armed fault did not fire"
    ctx.profile_reset()
    gd, gi = db.search(q, 10, "euclideanSquared")
    od, oi = O.search_flat(q, x, 10, O.L2SQ)
    np.testing.assert_array_equal(gi, oi)
    stats = ctx.profile_stats()
    assert stats and all(v[0] >= 1 for v in stats.values())
    db.free()
    ctx.close()


def _after_every_fault(kinds, make, search, want):
    """Fails event n = 1, 2, ... of a fresh context in turn until three runs of
    make and search on end meet none; whenever the search is what failed, the
    same call on the same object must then return ``want``, as must a search
    that answers."""
    tried = 0
    for kind in kinds:
        clean = 0
        for n in range(1, 200):
            print(f"fault {kind}:{n}", flush=True)
            ctx = _armed(f"{kind}:{n}")
            obj = None
            try:
                try:
                    obj = make(ctx)
                    gd, gi = search(obj)
                    clean += 1
                except VSKError as e:
                    assert "injected fault" in str(e)
                    clean = 0
                    if obj is None:
                        continue
                    tried += 1
                    gd, gi = search(obj)
                np.testing.assert_array_equal(gi, want[1])
                np.testing.assert_array_equal(gd, want[0])
            finally:
                if obj is not None:
                    obj.free()
                ctx.close()
            if clean == 3:
                break
        else:
            raise AssertionError("every event failed")
    assert tried > 3


def _close_rows(n, nq, d):
    """Rows whose distances differ by less than a 16-bit plane's rounding,
    and by more than fp32's: a screen that took its planes for exact would
    return other rows."""
    rng = np.random.default_rng(n + d)
    return ((1 + 0.05 * rng.standard_normal((n, d))).astype(np.float32),
            (1 + 0.05 * rng.standard_normal((nq, d))).astype(np.float32))


@pytest.mark.parametrize("metric", ["euclideanSquared", "cosine", "cosineNormalized"])
def test_fault_while_the_screen_plane_is_made(metric, monkeypatch):
    """A search that fails while the database's 16-bit plane is made, or
    before the plane's error bound is read back, leaves no plane behind that
    the next search would trust: that one is bit for bit the oracle."""
    monkeypatch.setenv("VSK_FLAT_KERNEL", "screen")
    x, q = _close_rows(30_000, 40, 16)
    if metric == "cosineNormalized":
        x /= np.linalg.norm(x, axis=1, keepdims=True)
        q /= np.linalg.norm(q, axis=1, keepdims=True)
    code = {"euclideanSquared": O.L2SQ, "cosine": O.COSINE,
            "cosineNormalized": O.COSINE_NORMALIZED}[metric]
    _after_every_fault(("launch", "alloc", "sync"), lambda ctx: VectorDatabase(ctx, x),
                       lambda db: db.search(q, 10, metric), O.search_flat(q, x, 10, code))


def test_fault_while_the_probe_plane_is_made(monkeypatch):
    """The same for the centroids' plane of the IVF probe's screen."""
    monkeypatch.setenv("VSK_FLAT_KERNEL", "screen")
    x, q = _close_rows(9000, 40, 16)
    c = _close_rows(3000, 1, 16)[0]
    lists = O.ivf_assign(x, c)
    cfg = IVFConfiguration(dimensions=16, numberOfCentroids=len(c), numberOfProbes=5)
    _after_every_fault(("launch", "alloc", "sync"), lambda ctx: IVFIndex.build(ctx, cfg, c, x),
                       lambda idx: idx.search(q, 10),
                       O.ivf_search(q, x, np.arange(len(x)), lists, c, 5, 10))


@pytest.mark.parametrize("metric", ["euclideanSquared", "cosine", "cosineNormalized"])
def test_no_memory_for_the_screen_plane(metric, monkeypatch):
    """A search whose plane finds no memory (the host reports that allocation
    as failed) answers by the exact scan, bit for bit the oracle; the next
    one makes the plane and screens."""
    monkeypatch.setenv("VSK_FLAT_KERNEL", "screen")
    x, q = _close_rows(20_000, 40, 16)
    code = {"euclideanSquared": O.L2SQ, "cosine": O.COSINE,
            "cosineNormalized": O.COSINE_NORMALIZED}[metric]
    od, oi = O.search_flat(q, x, 10, code)
    answered = 0
    for n in range(1, 60):
        print(f"no memory {metric} alloc:{n}", flush=True)
        ctx = _armed(f"alloc:{n}")
        ctx.profile(True)
        db = None
        try:
            db = VectorDatabase(ctx, x)
            screened = []
            for _ in range(2):
                ctx.profile_reset()
                gd, gi = db.search(q, 10, metric)
                screened.append(any(k.startswith("flat_screen") for k in ctx.profile_stats()))
                np.testing.assert_array_equal(gi, oi)
                np.testing.assert_array_equal(gd, od)
            if screened == [True, True]:
                break  # (no allocation left to fail)
            assert screened == [False, True]
            answered += 1
        except VSKError as e:
            assert "injected fault" in str(e)
        finally:
            if db is not None:
                db.free()
            ctx.close()
    else:
        raise AssertionError("every allocation failed")
    assert answered >= 1
