"""GPU parity of top-p with a repetition-penalty history on rows longer than
the registers hold (long_path.h, 53245 < V <= 262080; src/sampler.rs:83-101,
118-160).  Every row must match the oracle's sample(); rows the path declines
(more than 2048 distinct ids, non-finite values) are recomputed by the general
path with the same answer.
"""
import numpy as np
import pytest

from parity_util import compare, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sampler():
    import nimbus_sampler as ns
    s = ns.Sampler(0)
    yield s
    s.close()


def _history(rnd, x, V, n):
    """Half the row's own top ids, half random ones, with repeats and (rarely) ids past V."""
    ids, off = [], [0]
    for r in range(x.shape[0]):
        top = np.argsort(-np.nan_to_num(x[r, :V], nan=0.0))[: max(1, n)]
        g = np.concatenate([rnd.choice(top, n // 2), rnd.integers(0, V, n - n // 2)])
        if n >= 4:
            g[-1] = V + 5
        ids.append(rnd.permutation(g))
        off.append(off[-1] + n)
    return np.concatenate(ids).astype(np.uint32), np.array(off, np.int64)


def _check(sampler, x, V, label, hist, ld=None, **kw):
    import nimbus_sampler as ns
    params = ns.SamplingParams(**kw)
    B = x.shape[0]
    gi, go = hist
    print(f"[long penalty] {label} B={B} V={V} {kw} ld={ld}", flush=True)
    gpu = run_gpu(sampler, x, V, params, list(range(B)), gen_ids=gi, gen_offsets=go, ld=ld)
    ref = run_oracle(x, V, params, list(range(B)), gen_ids=gi, gen_offsets=go)
    rep = compare(gpu, ref, greedy=False)
    print(f"[long penalty] {label} -> {rep}", flush=True)
    return gpu[1]


# both ends of the range, rows that start off 16 bytes, nuclei of every size
@pytest.mark.parametrize("V,ld_extra", [(53246, 0), (60001, 2), (128256, 0), (131071, 3), (262080, 1), (262081, 0)])
@pytest.mark.parametrize("pen,n", [(1.2, 1), (1.2, 200), (0.7, 300)])
def test_sizes_and_penalties(sampler, V, ld_extra, pen, n):
    rnd = np.random.Generator(np.random.PCG64(V + n))
    x = (rnd.standard_normal((5, V), dtype=np.float32) * np.float32(2.0)).astype(np.float32)
    hist = _history(rnd, x, V, n)
    for p, T in ((0.3, 0.5), (0.9, 0.8), (0.99, 1.3)):
        st = _check(sampler, x, V, f"pen={pen}", hist, ld=V + ld_extra, temperature=T, top_p=p,
                    repetition_penalty=pen)
        assert (st["kernel"] == (1 if V <= 262080 else 2)).all(), (st["kernel"], st["reject"])


# distinct ids at and past the list's capacity
@pytest.mark.parametrize("n,on", [(2048, True), (2049, False)])
def test_limits_of_the_history(sampler, n, on):
    rnd = np.random.Generator(np.random.PCG64(n))
    V = 100003
    x = (rnd.standard_normal((4, V), dtype=np.float32) * np.float32(2.0)).astype(np.float32)
    ids = np.concatenate([np.tile(rnd.permutation(V)[:n], 2) for _ in range(4)]).astype(np.uint32)
    off = np.arange(5, dtype=np.int64) * 2 * n
    st = _check(sampler, x, V, "limits", (ids, off), temperature=0.9, top_p=0.9, repetition_penalty=1.3)
    assert (st["kernel"] == (1 if on else 2)).all(), (st["kernel"], st["reject"])


@pytest.mark.parametrize("lattice", [1, 8])
@pytest.mark.parametrize("pen", [2.0, 1.1])
def test_ties_at_the_cutoff(sampler, lattice, pen):
    # values on a lattice: the cutoff falls among equal values, penalised
    # (doubled or halved, which lands on the lattice) and plain
    rnd = np.random.Generator(np.random.PCG64(31 + lattice))
    V = 60001
    x = (np.round(rnd.standard_normal((8, V)) * 3.0 * lattice) / lattice).astype(np.float32)
    hist = _history(rnd, x, V, 400)
    for p in (0.2, 0.8, 0.97):
        _check(sampler, x, V, "ties", hist, ld=V + 1, temperature=1.0, top_p=p, repetition_penalty=pen)


def test_head_and_cutoff_penalised(sampler):
    # a small nucleus whose every member is penalised, and many members of the
    # cutoff bucket among them
    rnd = np.random.Generator(np.random.PCG64(5))
    V = 70000
    x = rnd.standard_normal((6, V)).astype(np.float32)
    ids = rnd.permutation(V)[:1500].astype(np.uint32)
    x[:, ids] += np.float32(12.0)
    x[3:, ids] = (np.float32(13.0) + rnd.random((3, 1500)) * 0.01).astype(np.float32)
    hist = (np.tile(ids, 6), np.arange(7, dtype=np.int64) * 1500)
    for p in (0.5, 0.9):
        st = _check(sampler, x, V, "head", hist, temperature=1.0, top_p=p, repetition_penalty=1.1)
        assert (st["kernel"] == 1).all(), (st["kernel"], st["reject"])


@pytest.mark.parametrize("V", [60000, 200003])
def test_masked_and_unusual_rows(sampler, V):
    rnd = np.random.Generator(np.random.PCG64(V))
    B = 12
    x = (rnd.standard_normal((B, V), dtype=np.float32) * np.float32(3.0)).astype(np.float32)
    x[0, rnd.permutation(V)[100:]] = -np.inf
    x[1, rnd.permutation(V)[5:]] = -np.inf
    x[2, : V - 300] = -np.inf
    x[3, 777] = 100.0
    x[4] = 1.5
    x[5, 12] = np.nan
    x[6, V - 1] = np.inf
    x[7] = -np.inf
    x[8, rnd.random(V) < 0.99] = -1e9
    x[9] = np.where(rnd.random(V) < 0.5, np.float32(0.0), np.float32(-0.0))
    x[10] *= 1e-30
    x[11] -= 500.0
    hist = _history(rnd, x, V, 60)
    for p in (0.5, 0.9):
        # (constant rows, 4, 9 and 10, hold more equal members than the cutoff ranks)
        st = _check(sampler, x, V, "rows", hist, ld=V + 2, temperature=0.8, top_p=p, repetition_penalty=1.3)
        assert ((st["kernel"] == 1) & (st["reject"] == 0))[[0, 1, 2, 3, 8, 11]].all(), (st["kernel"], st["reject"])


def test_long_decode_with_a_penalty(sampler):
    import test_gpu_decode as td
    kernels = []
    td._run(sampler, B=12, V=128256, steps=6, cap=8,
            params_kw=dict(temperature=0.8, top_p=0.9, repetition_penalty=1.3), seed=505,
            kernels=kernels, sigma=3.0)
    k = np.concatenate([a for a, _ in kernels])
    assert k.size > 0 and (k == 1).all()
