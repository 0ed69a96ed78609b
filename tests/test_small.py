"""Clouds of at most 16,384 points on the kernels that sort and sample each
with one workgroup (nsfps_small.hip; NSFPS_SMALL=0 takes the general engine):
the oracle's samples at the edges of the kernels' slots (64-point leaves,
1,024-point slots), on shared buckets, ties and crowded buckets, through the
plan and the batched call, and their error paths.  Indices: no tolerance."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

UNIT = (-1.0, 1.0, -1.0, 1.0, -1.0, 1.0)


@pytest.fixture(scope="module")
def lib():
    from ns_fps_amd.capi import Lib
    L = Lib()
    if L.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need an MI355X")
    return L


@pytest.fixture(scope="module")
def hip():
    from ns_fps_amd.capi import Hip
    return Hip()


def lattice(side, take=None):
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3), -1).reshape(-1, 3).astype(np.float32)
    return g[np.random.RandomState(3).permutation(len(g))][:take]


def cloud(kind, n):
    rs = np.random.RandomState(n)
    if kind == "cube":
        return rs.uniform(-1, 1, (n, 3)).astype(np.float32)
    if kind == "crowded":  # few buckets: stored in their own spatial order
        return rs.randn(n, 3).astype(np.float32) * np.float32([1, 1, 0.01])
    if kind == "dups":
        return np.repeat(rs.randn(n // 16, 3), 16, 0)[rs.permutation(n)].astype(np.float32)
    if kind == "line":  # cell boundaries, and an axis of no extent
        return np.stack([rs.randint(-64, 64, n) / 64, np.zeros(n), rs.rand(n)], 1).astype(np.float32)
    return lattice(26, n)


@pytest.mark.parametrize("small", ["0", "1"])
@pytest.mark.parametrize("kind,n,m,rng", [
    *[("cube", n, max(2, n // 3), (*UNIT, 16, 16, 16)) for n in (3, 63, 64, 65, 127, 1024, 1025, 2049,
                                                                4096, 8193, 16383, 16384)],
    ("cube", 1000, 999, (*UNIT, 8, 8, 8)), ("cube", 16384, 16383, (*UNIT, 64, 64, 64)),
    ("cube", 5000, 2000, (*UNIT, 17, 17, 17)), ("cube", 12000, 3000, (*UNIT, 30, 30, 30)),
    ("cube", 3000, 900, (*UNIT, 1, 1, 1)), ("cube", 4000, 900, (*UNIT, 1024, 2, 5)),
    ("crowded", 10000, 1000, (-100, 100, -100, 100, -100, 100, 16, 16, 16)),
    ("crowded", 16384, 2000, (-100, 100, -100, 100, -100, 100, 15, 16, 16)),
    ("dups", 8000, 3000, (-4, 4, -4, 4, -4, 4, 16, 16, 16)),
    ("line", 4000, 1500, (*UNIT, 32, 32, 32)),
    ("lattice", 16384, 5000, (0, 26, 0, 26, 0, 26, 8, 8, 8)),
    ("lattice", 4096, 4000, (0, 26, 0, 26, 0, 26, 26, 26, 26)),
])
def test_small_clouds_match_the_oracle(lib, hip, oracle, monkeypatch, small, kind, n, m, rng):
    P = cloud(kind, n)
    monkeypatch.setenv("NSFPS_SMALL", small)
    want = oracle.fps(P, m, rng)
    assert np.array_equal(lib.fps(P, m, rng), want)
    assert lib.stats()["engine"] == 1 and lib.stats()["rounds"] >= 1
    plan = lib.plan_create(P, len(P), rng)
    d_out = hip.malloc(m * 4)
    try:
        for k in (m, max(2, m // 2)):
            got = lib.plan_sample(plan, k, d_out)
            assert np.array_equal(hip.download(d_out, got, np.int32), want[:k])
    finally:
        lib.plan_destroy(plan)
        hip.free(d_out)


@pytest.mark.parametrize("n,m,batch,one", [
    (8192, 8000, 1, True), (8193, 1024, 1, True), (8193, 1025, 1, False), (12288, 1536, 1, True),
    (12289, 64, 1, False), (16384, 4096, 15, False), (16384, 4096, 16, True), (16385, 64, 16, False),
])
def test_which_calls_one_workgroup_a_cloud_takes(lib, oracle, n, m, batch, one):
    """At each side of the rule's lines.  The statistics tell the two apart:
    a small call's sampling is one launch, so late_ms is all of sample_ms."""
    P = [cloud("cube", n), cloud("cube", n + 1)[:n]]
    rng = (*UNIT, 16, 16, 16)
    if batch == 1:
        got = [lib.fps(P[0], m, rng)]
    else:
        got = lib.fps_batched(np.stack([P[b % 2] for b in range(batch)]), m, [rng] * batch)
    st = lib.stats()
    assert (st["late_ms"] == st["sample_ms"] and st["wide_ms"] == 0.0) == one
    for b in range(min(batch, 2)):
        assert np.array_equal(got[b], oracle.fps(P[b], m, rng))


@pytest.mark.parametrize("scale", [1.0, 1e-21, 3e18, 1e30])
def test_small_clouds_at_the_ends_of_the_number_range(lib, oracle, monkeypatch, scale):
    """Squared distances that are subnormal, or overflow."""
    P = (np.random.RandomState(9).uniform(-1, 1, (700, 3)) * scale).astype(np.float32)
    rng = tuple(float(np.float32(v * scale)) for v in UNIT) + (8, 8, 8)
    monkeypatch.setenv("NSFPS_SMALL", "1")
    assert np.array_equal(lib.fps(P, 200, rng), oracle.fps(P, 200, rng))


@pytest.mark.parametrize("n", [1000, 6000])
def test_small_batches_match_the_oracle(lib, oracle, monkeypatch, n):
    P = np.stack([cloud(k, n) for k in ("cube", "crowded", "line")])
    monkeypatch.setenv("NSFPS_SMALL", "1")
    got = lib.fps_batched(P, n // 4, None, (16, 16, 16))
    for b in range(len(P)):
        assert np.array_equal(got[b], oracle.fps(P[b], n // 4, None)), b


def test_small_clouds_report_what_the_general_engine_reports(lib, monkeypatch):
    from ns_fps_amd.capi import NsfpsError
    said = {}
    for small in ("0", "1"):
        monkeypatch.setenv("NSFPS_SMALL", small)
        for what, value, rng in [("nan", np.nan, (*UNIT, 8, 8, 8)), ("inf", np.inf, None),
                                 ("flat", 1e9, None)]:
            P = np.full((200, 3), 1e9, np.float32) if what == "flat" else cloud("cube", 200)
            P[77, 1] = value
            with pytest.raises(NsfpsError) as e:
                lib.fps(P, 50, rng)
            said.setdefault(what, set()).add((e.value.status, str(e.value)))
    assert all(len(v) == 1 for v in said.values()), said


@pytest.mark.parametrize("small", ["0", "1"])
@pytest.mark.parametrize("what", ["nan", "flat"])
@pytest.mark.parametrize("at", [0, 5, 7])
def test_a_batch_with_a_refused_cloud_writes_no_row(lib, hip, oracle, monkeypatch, small, what, at):
    from ns_fps_amd.capi import NsfpsError
    P = np.stack([cloud("cube", 300 + b)[:300] for b in range(8)])
    good = P.copy()
    if what == "nan":
        P[at, 123, 2] = np.nan
    else:
        P[at] = 1e9
    monkeypatch.setenv("NSFPS_SMALL", small)
    before = np.arange(8 * 60, dtype=np.int32)
    d_xyz, d_out, d_good = hip.upload(P), hip.upload(before), hip.upload(good)
    try:
        with pytest.raises(NsfpsError):
            lib.fps_batched_device(d_xyz, 8, 300, 60, d_out)
        assert np.array_equal(hip.download(d_out, 8 * 60, np.int32), before)
        # and the call after it is sampled
        lib.fps_batched_device(d_good, 8, 300, 60, d_out)
        rows = hip.download(d_out, 8 * 60, np.int32).reshape(8, 60)
        for b in range(8):
            assert np.array_equal(rows[b], oracle.fps(good[b], 60, None)), b
    finally:
        for d in (d_xyz, d_out, d_good):
            hip.free(d)


@pytest.mark.parametrize("kind", ["launch", "copy", "sync", "any"])
def test_every_operation_of_a_small_call_fails_cleanly(lib, oracle, monkeypatch, kind):
    from ns_fps_amd.capi import NsfpsError
    P, rng = cloud("cube", 3000), (*UNIT, 16, 16, 16)
    want = oracle.fps(P, 500, rng)
    monkeypatch.setenv("NSFPS_SMALL", "1")
    assert np.array_equal(lib.fps(P, 500, rng), want)
    failed = 0
    for i in range(1, 100):
        monkeypatch.setenv("NSFPS_INJECT", f"{kind}:{i}")
        try:
            got = lib.fps(P, 500, rng)
            break
        except NsfpsError as e:
            assert "injected failure" in str(e)
            failed += 1
        finally:
            monkeypatch.delenv("NSFPS_INJECT")
        assert np.array_equal(lib.fps(P, 500, rng), want)
    assert np.array_equal(got, want) and failed >= (2 if kind == "launch" else 1)
