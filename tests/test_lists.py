"""The rounds engine's lists and final order at their edges (nsfps_runs.hip):
both list lengths, nodes with more samples a round than fit the LDS at once,
ties, chains of conflicts, nearly all points sampled, shared buckets, split
update passes and batched clouds, against the oracle.  Indices: no tolerance."""

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


def cloud(kind, n):
    rs = np.random.RandomState(n % 1000003)
    if kind == "cube":
        P = rs.uniform(-1, 1, (n, 3))
    elif kind == "lattice":  # ties in every distance
        side = int(np.ceil(n ** (1 / 3)))
        P = np.stack(np.meshgrid(*[np.arange(side)] * 3), -1).reshape(-1, 3) * (2 / side) - 1
        P = P[rs.permutation(len(P))[:n]]
    elif kind == "dups":
        P = np.repeat(rs.uniform(-1, 1, ((n + 7) // 8, 3)), 8, 0)[rs.permutation(n)]
    elif kind == "plane":
        P = rs.uniform(-1, 1, (n, 3)) * [1, 1, 0]
    else:  # rings of halving radius: each sample's rivals are its neighbours
        r = 2.0 ** -(np.arange(n) % 40)
        a = rs.uniform(0, 2 * np.pi, n)
        P = np.stack([r * np.cos(a), r * np.sin(a), r * rs.uniform(-0.1, 0.1, n)], 1)
    return np.ascontiguousarray(P, np.float32)


@pytest.mark.parametrize("kind,n,m,blocks", [
    ("cube", 2, 1, (4, 4, 4)), ("cube", 70, 69, (4, 4, 4)), ("cube", 1025, 1024, (8, 8, 8)),
    ("cube", 32768, 3000, (16, 16, 16)), ("cube", 32769, 3000, (16, 16, 16)),
    ("cube", 40000, 39999, (1, 1, 1)), ("cube", 60000, 30000, (2, 2, 2)),
    ("cube", 50000, 9000, (17, 17, 17)), ("cube", 90000, 20000, (30, 30, 30)),
    ("lattice", 64000, 9000, (16, 16, 16)), ("lattice", 40000, 39990, (8, 8, 8)),
    ("dups", 48000, 20000, (16, 16, 16)), ("plane", 70000, 9000, (32, 32, 2)),
    ("rings", 40000, 9000, (32, 32, 4)), ("rings", 3000, 2990, (4, 4, 4)),
])
def test_lists_match_the_oracle(lib, oracle, monkeypatch, kind, n, m, blocks):
    P = cloud(kind, n)
    monkeypatch.setenv("NSFPS_SMALL", "0")
    want = oracle.fps(P, m, (*UNIT, *blocks))
    assert np.array_equal(lib.fps(P, m, (*UNIT, *blocks)), want)
    if n <= 1025:
        got = lib.fps_batched(np.stack([P] * 9), m, [(*UNIT, *blocks)] * 9)
        assert all(np.array_equal(g, want) for g in got)


def test_a_window_of_coarse_bins_that_ends_above_the_last_keys(lib, oracle):
    """Squared distances over more than 60 octaves give the second round's
    window bins of 2^52 keys; it ends above the keys of the points at distance
    0, which are far more than a list holds and are not to be listed with the
    1,015 inside the window."""
    rs = np.random.RandomState(5)
    d2 = np.concatenate([[2.0 ** 69], rs.uniform(20.5, 38.0, 1000), rs.uniform(18.1, 19.9, 25)])
    u = rs.randn(len(d2), 3)
    far = u / np.linalg.norm(u, axis=1, keepdims=True) * np.sqrt(d2)[:, None]
    far[0] = [2.0 ** 34.5, 0, 0]
    P = np.zeros((40000, 3), np.float32)
    P[1 + rs.permutation(39999)[:len(far)]] = far
    rng = (-1e11, 1e11, -1e11, 1e11, -1e11, 1e11, 4, 4, 4)
    assert np.array_equal(lib.fps(P, 1500, rng), oracle.fps(P, 1500, rng))


@pytest.mark.parametrize("kind,n,blocks", [
    ("cube", 17000, (32, 32, 32)), ("cube", 600, (1, 1, 1)), ("cube", 40000, (17, 17, 17)),
    ("lattice", 20000, (15, 16, 16)), ("dups", 2000, (8, 8, 8)), ("rings", 33000, (32, 32, 4)),
    ("plane", 300000, (32, 32, 2)),
])
def test_first_samples_match_the_oracle(lib, oracle, monkeypatch, kind, n, blocks):
    """Few samples are taken one after another (128 at most: the whole call;
    more: about the first 64, the rest by layers), on every list length."""
    P = cloud(kind, n)
    monkeypatch.setenv("NSFPS_SMALL", "0")
    want = oracle.fps(P, 600 if n > 600 else 599, (*UNIT, *blocks))
    for m in (2, 3, 63, 64, 65, 127, 128, 129, 200, len(want)):
        got = lib.fps(P, m, (*UNIT, *blocks))
        assert np.array_equal(got, want[:m]), (m, len(got))


@pytest.mark.parametrize("batch,n", [(2, 33000), (4, 33000), (16, 33000), (64, 33000), (7, 20000)])
def test_shorter_lists_of_many_clouds_match_the_oracle(lib, oracle, batch, n):
    kinds = ["cube", "lattice", "dups", "rings"]
    P = [cloud(kinds[b % 4], n) for b in range(4)]
    want = [oracle.fps(p, 700, (*UNIT, 16, 16, 16)) for p in P]
    for m in (40, 700):
        got = lib.fps_batched(np.stack([P[b % 4] for b in range(batch)]), m,
                              [(*UNIT, 16, 16, 16)] * batch)
        for b in range(batch):
            assert np.array_equal(got[b], want[b % 4][:m]), (b, m)


@pytest.mark.parametrize("rounds", ["1", "2", "9"])
@pytest.mark.parametrize("kind,n,m", [("cube", 60000, 30000), ("lattice", 30000, 12000),
                                      ("dups", 48000, 5900), ("rings", 600, 500)])
def test_a_full_log_of_rounds_matches_the_oracle(lib, oracle, monkeypatch, rounds, kind, n, m):
    """Rounds beyond the log's entries share its last one, whose samples are
    sorted in pieces of a list's length."""
    P = cloud(kind, n)
    monkeypatch.setenv("NSFPS_LOG_ROUNDS", rounds)
    want = oracle.fps(P, m, (*UNIT, 16, 16, 16))
    assert np.array_equal(lib.fps(P, m, (*UNIT, 16, 16, 16)), want)
    plan = lib.plan_create(P, n, (*UNIT, 16, 16, 16))
    try:
        from ns_fps_amd.capi import Hip
        hip = Hip()
        d_out = hip.malloc(m * 4)
        got = lib.plan_sample(plan, m, d_out)
        assert np.array_equal(hip.download(d_out, got, np.int32), want)
        hip.free(d_out)
    finally:
        lib.plan_destroy(plan)


@pytest.mark.parametrize("scale", [1.0, 1e-21, 3e-20, 3e18, 1e30])
def test_first_samples_at_the_ends_of_the_number_range(lib, oracle, monkeypatch, scale):
    """Squared distances that are subnormal or overflow: the keys of the lists
    sampled one after another are compared as doubles, subnormal ones among
    them."""
    P = (np.random.RandomState(9).uniform(-1, 1, (20000, 3)) * scale).astype(np.float32)
    P[:40] *= np.float32(0.01)
    rng = tuple(float(np.float32(v * scale)) for v in UNIT) + (8, 8, 8)
    monkeypatch.setenv("NSFPS_SMALL", "0")
    want = oracle.fps(P, 400, rng)
    for m in (100, 400):
        assert np.array_equal(lib.fps(P, m, rng), want[:m])
