"""GPU parity of the split-bf16 LM head (lm_head_split.h: B > 1, every f32
operand as the exact sum of three bf16 parts) at the edges of its tiles, the
two ways it reads W, and its limits, against exact f64 sums.

Bar: every logit within the f32 error bound of a length-H sum (as
test_gpu_lm_head.py), and the relative error over all logits (2-norm) at most
2.5e-7: three roundings of 2^-24 would be 1.8e-7, and the f32 matrix-core sums
that this kernel replaced had 3.6e-7 at H = 768.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sampler():
    import nimbus_sampler as ns
    s = ns.Sampler(0)
    yield s
    s.close()


def _case(sampler, fmt, B, H, V, group=None, off=0, edit=None, seed=0):
    """Logits, exact sums and sums of absolute terms; `off`: elements skipped before
    x and W (alignment); edit(x, w or None) changes the operands first."""
    import torch
    from oracle import lm_head_oracle as lh
    rnd = np.random.default_rng(seed + B + H + V)
    x = rnd.standard_normal((B, H)).astype(np.float32)
    w = (rnd.standard_normal((V, H)) * 0.05).astype(np.float32)
    if edit is not None:
        edit(x, w)
    data, scales = (w.reshape(-1), None) if fmt == 0 else lh.quantize(w, V, H, fmt, group)
    dev = torch.device("cuda:0")
    xb = torch.full((B * (H + 5) + off,), float("nan"), device=dev)[off:].view(B, H + 5)
    xb[:, :H] = torch.from_numpy(x).to(dev)
    step = 1 if fmt == 0 else 4  # (rows of W start on 4 bytes)
    raw = np.ascontiguousarray(data)
    d = torch.zeros(raw.size + off * step, dtype=torch.float32 if fmt == 0 else torch.uint8, device=dev)[off * step:]
    d.copy_(torch.from_numpy(raw).to(dev))
    s = torch.from_numpy(scales).to(dev) if scales is not None else None
    print(f"[lm_head split] fmt={fmt} B={B} H={H} V={V} group={group} off={off}", flush=True)
    out = sampler.lm_head_logits(xb[:, :H], fmt, d, V, scales=s, group_size=group or 0)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        exact, absd = lh.lm_head_logits(x, fmt, data, scales, V, H, group)
    return out.cpu().numpy(), exact, absd


def _check(got, exact, absd, H, groups=1):
    from oracle import lm_head_oracle as lh
    err = np.abs(got.astype(np.float64) - exact)
    assert np.all(err <= lh.f32_bound(absd, H, groups)), float((err / lh.f32_bound(absd, H, groups)).max())
    assert np.linalg.norm(err) <= 2.5e-7 * np.linalg.norm(exact), np.linalg.norm(err) / np.linalg.norm(exact)


@pytest.mark.parametrize("B", [2, 32, 33, 64, 65, 128, 129, 256, 257])
@pytest.mark.parametrize("fmt", [0, 8, 4])
def test_batches(sampler, fmt, B):
    got, exact, absd = _case(sampler, fmt, B, 136, 391, off=1)
    _check(got, exact, absd, 136)


@pytest.mark.parametrize("fmt,B,H,V,group", [
    (0, 40, 4, 129, None), (0, 17, 100, 1000, None), (0, 33, 2052, 130, None),  # H % 8, % 32, % 64 != 0
    (0, 3, 64, 98305, None), (8, 3, 64, 98305, None), (4, 60, 96, 100001, None),  # two tiles per wave in v
    (0, 200, 40, 49153, None), (8, 130, 40, 50001, None),                        # 8 waves, one tile
    (8, 20, 8, 77, None), (8, 20, 1176, 300, None), (4, 20, 40, 300, None),      # rows none of 32: by steps
    (8, 20, 96, 300, 32), (8, 70, 192, 300, 96), (4, 200, 128, 300, 32),         # groups by steps
    (8, 20, 128, 300, 64), (8, 150, 384, 300, 128), (4, 40, 256, 300, 128), (4, 256, 192, 300, 192),
    (8, 9, 96, 300, 48),                                                         # left to the f32 kernel
])
def test_lengths_and_groups(sampler, fmt, B, H, V, group):
    got, exact, absd = _case(sampler, fmt, B, H, V, group)
    _check(got, exact, absd, H, H // (group or H))


@pytest.mark.parametrize("fmt", [0, 8])
def test_values_of_every_size(sampler, fmt):
    # rows scaled from 1e-30 to 1e30, and far apart values inside a row
    def edit(x, w):
        x *= (10.0 ** np.linspace(-30, 30, x.shape[0])).astype(np.float32)[:, None]
        x[:, ::7] *= np.float32(1e-6)
        if fmt == 0:
            w[:, ::5] *= np.float32(1e-7)
    got, exact, absd = _case(sampler, fmt, 21, 256, 200, edit=edit)
    from oracle import lm_head_oracle as lh
    err = np.abs(got.astype(np.float64) - exact)
    assert np.all(err <= lh.f32_bound(absd, 256))


@pytest.mark.parametrize("fmt", [0, 8, 4])
def test_infinities_and_nan(sampler, fmt):
    def edit(x, w):
        x[1, 3] = np.inf
        x[2, 5] = np.nan
        x[3, 7], x[3, 8] = np.inf, -np.inf
        # (its bf16 rounding overflows; codes are summed before their scale, and
        # 127 x must stay finite in f32, as in the kernel this one replaced)
        x[4, 9] = 3.4e38 if fmt == 0 else 2e36
        if fmt == 0:
            w[5, 3] = 0.0
            w[6, 0] = -np.inf
            w[7, 1] = np.nan
            w[8, 2] = 3.4e38
            x[:, 2] = np.where(np.abs(x[:, 2]) < 1.0, x[:, 2], 0.5)
    got, exact, absd = _case(sampler, fmt, 6, 64, 40, edit=edit)
    exact32 = np.where(np.abs(exact) > 3.4028235e38, np.sign(exact) * np.inf, exact)
    assert np.array_equal(np.isnan(got), np.isnan(exact32))
    inf = np.isinf(exact32)
    assert np.array_equal(got[inf], exact32[inf].astype(np.float32))
    fin = np.isfinite(exact32)
    from oracle import lm_head_oracle as lh
    assert np.all(np.abs(got[fin] - exact32[fin]) <= lh.f32_bound(absd, 64)[fin])
