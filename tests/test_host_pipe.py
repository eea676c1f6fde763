"""Large host copies (host_pipe.h): sizes at the thresholds of the pipe, whole
pieces and a partial last one, bit for bit, on back-to-back calls that reuse
the pinned pieces."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.mark.parametrize("entries", [MB // 2 - 1, MB // 2, 3 * MB - 1, 3 * MB, 3 * MB + 1, 8 * MB, 9 * MB + 12345])
def test_factors_round_trip(entries):
    """W [1][entries] in and back: 4 bytes an entry, so 2 MB (the way back)
    and 12 MB (the way in) are among the sizes, and more than eight pieces."""
    from cdmf_amd import datadir
    from cdmf_amd import solver as S
    ds = datadir.from_triplets(entries, 2, (np.array([0, entries - 1]), np.array([0, 1]), np.ones(2)),
                               (np.array([0]), np.array([0]), np.ones(1)))
    r = np.random.default_rng(entries)
    with S.Solver(0) as s:
        s.upload(ds, with_test=False)
        for _ in range(2):
            W = r.standard_normal((1, entries), dtype=np.float32)
            H = r.standard_normal((1, 2), dtype=np.float32)
            s.set_factors(W, H)
            W[:] = 0.0  # the call is done with the caller's array
            W2, H2 = s.factors()
            s.set_factors(W2, H2)
            W3, H3 = s.factors()
            assert np.array_equal(W2, W3) and np.array_equal(H2, H) and np.array_equal(H3, H)
            assert np.any(W2 != 0.0)


def test_two_threads_two_objects():
    """Each object has its own pipe: two threads solving at once give what
    they give one after the other."""
    import threading

    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = D.gen_powerlaw(300000, 500, 3000000, 10, max_row_degree=500, seed=2)
    k = 8
    W0, H0 = D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32)
    out = {}

    def solve(name):
        with S.Solver(0) as s:
            s.upload(ds, with_test=False)
            s.set_factors(W0, H0)
            s.run(k, 0.05, 1, 1, variant=S.VARIANT_TILED)
            out[name] = s.factors()

    solve("alone")
    ts = [threading.Thread(target=solve, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for i in range(2):
        assert np.array_equal(out[i][0], out["alone"][0]) and np.array_equal(out[i][1], out["alone"][1])


@pytest.mark.parametrize("entries", [3 * MB - 1, 3 * MB, 3 * MB + 1, 8 * MB + 1, 9 * MB + 12345])
def test_factors_come_back_as_given(entries):
    """What comes back is what was handed over, on calls that reuse the pinned
    pieces: sizes with a partial last piece and more pieces than slots."""
    from cdmf_amd import datadir
    from cdmf_amd import solver as S
    ds = datadir.from_triplets(entries, 2, (np.array([0, entries - 1]), np.array([0, 1]), np.ones(2)),
                               (np.array([0]), np.array([0]), np.ones(1)))
    r = np.random.default_rng(entries)
    with S.Solver(0) as s:
        s.upload(ds, with_test=False)
        for _ in range(3):
            W = r.standard_normal((1, entries), dtype=np.float32)
            given = W.copy()
            s.set_factors(W, np.ones((1, 2), np.float32))
            W[:] = 0.0  # the call is done with the caller's array
            assert np.array_equal(s.factors()[0], given)
