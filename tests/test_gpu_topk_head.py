"""GPU parity of the top-k path that keeps only a row's head (topk_path.h):
top-k with a repetition-penalty history at any length, and top-k on rows
longer than the registers hold (src/sampler.rs:83-116).  Every row must match
the oracle's sample(); rows the path declines (k past 960, more than 4096
history ids, NaN, more candidates than its lists hold) are recomputed by the
general path with the same answer.
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


def _check(sampler, x, V, label, hist=None, ld=None, **kw):
    import nimbus_sampler as ns
    params = ns.SamplingParams(**kw)
    B = x.shape[0]
    gi, go = hist if hist is not None else (None, None)
    print(f"[top-k head] {label} B={B} V={V} {kw} ld={ld}", flush=True)
    gpu = run_gpu(sampler, x, V, params, list(range(B)), gen_ids=gi, gen_offsets=go, ld=ld)
    ref = run_oracle(x, V, params, list(range(B)), gen_ids=gi, gen_offsets=go)
    rep = compare(gpu, ref, greedy=False)
    print(f"[top-k head] {label} -> {rep}", flush=True)
    return gpu[1], ref[1]


# rows per group size: V + 3 <= 65536 G, both sides of each switch, and short
# rows whose head is the whole row
@pytest.mark.parametrize("V,ld_extra", [(256, 1), (1000, 0), (4100, 3), (50257, 0), (53246, 2), (65533, 3),
                                        (65534, 1), (128256, 0), (131069, 1), (131070, 3), (262141, 3)])
@pytest.mark.parametrize("pen,n", [(1.0, 0), (1.2, 100), (0.7, 300)])
def test_sizes_and_penalties(sampler, V, ld_extra, pen, n):
    rnd = np.random.Generator(np.random.PCG64(V + n))
    x = (rnd.standard_normal((6, V), dtype=np.float32) * np.float32(3.0)).astype(np.float32)
    hist = _history(rnd, x, V, n) if n else None
    for k, p, T in ((1, 0.9, 0.8), (50, 0.9, 0.7), (200, 1.0, 1.3)):
        st, _ = _check(sampler, x, V, f"pen={pen}", hist, ld=V + ld_extra, temperature=T, top_p=p, top_k=k,
                       repetition_penalty=pen)
        if V > 4100:
            assert ((st["kernel"] == 1) & (st["reject"] == 0)).all(), (st["kernel"], st["reject"])


@pytest.mark.parametrize("k,n,on", [(959, 64, True), (960, 4096, True), (961, 64, False), (40, 4097, False)])
def test_limits_of_k_and_history(sampler, k, n, on):
    rnd = np.random.Generator(np.random.PCG64(k + n))
    V = 128256
    x = (rnd.standard_normal((4, V), dtype=np.float32) * np.float32(2.0)).astype(np.float32)
    st, _ = _check(sampler, x, V, "limits", _history(rnd, x, V, n), temperature=0.9, top_p=0.95, top_k=k,
                   repetition_penalty=1.3)
    assert (st["kernel"] == (1 if on else 2)).all(), (st["kernel"], st["reject"])


@pytest.mark.parametrize("k", [1, 7, 64])
@pytest.mark.parametrize("lattice", [1, 8])
def test_ties_at_the_kth(sampler, k, lattice):
    # values on a lattice: the k-th largest shares its value with up to
    # hundreds of others, penalised and plain, and all of them are kept
    rnd = np.random.Generator(np.random.PCG64(k * 31 + lattice))
    V = 60001
    x = (np.round(rnd.standard_normal((8, V)) * 3.0 * lattice) / lattice).astype(np.float32)
    hist = _history(rnd, x, V, 40)
    for p in (0.8, 1.0):
        _check(sampler, x, V, "ties", hist, ld=V + 1, temperature=1.0, top_p=p, top_k=k, repetition_penalty=2.0)
        _check(sampler, x, V, "ties", temperature=1.0, top_p=p, top_k=k)


@pytest.mark.parametrize("V", [60000, 200003])
def test_masked_and_unusual_rows(sampler, V):
    # masked vocabularies (all but a few ids, all but fewer than k ids, a
    # block), one far head, constant rows, NaN / +inf / all -inf rows, -1e9
    # masks, rows of zeros of both signs
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
    for k, p in ((20, 0.9), (300, 1.0)):
        st, _ = _check(sampler, x, V, "rows", hist, ld=V + 2, temperature=0.8, top_p=p, top_k=k,
                       repetition_penalty=1.3)
        ok = [0, 1, 2, 3, 8, 10, 11]
        assert ((st["kernel"] == 1) & (st["reject"] == 0))[ok].all(), (st["kernel"], st["reject"])


def test_long_decode_with_every_knob(sampler):
    import test_gpu_decode as td
    kernels = []
    td._run(sampler, B=12, V=128256, steps=6, cap=8,
            params_kw=dict(temperature=0.8, top_p=0.9, top_k=40, repetition_penalty=1.3), seed=505,
            kernels=kernels, sigma=3.0)
    k = np.concatenate([a for a, _ in kernels])
    assert k.size > 0 and (k == 1).all()
