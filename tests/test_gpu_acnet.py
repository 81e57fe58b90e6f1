"""The one-kernel minibatch of the reference actor-critic's shape (csrc/acnet.hip) against the plan
that runs it as separate products (TALOS_PLAN_UNFUSED=1), at the edges of its tiling: token tiles of
16, groups of up to 8 samples and 128 tokens, several groups a workgroup, calls of fewer samples
than the plan's batch, either activation, 1 to 8 actions, rows that are not 16-byte aligned.

Bound: both sides are fp32 sums of at most 128 terms a product, about a dozen products deep; each
stays within a few 1e-7 (2-norm) of the f64 result, and 1e-5 of a tensor's norm leaves a dropped row
or column far outside. A tensor whose terms cancel (with one token a sample the whole query path's
gradient is zero, what is left is the rounding of its terms) gets 1e-7 of the whole gradient's norm
instead: 2^-24 of terms as large as the gradient, both sides' roundings.
"""
import numpy as np
import pytest

import talos_hip as th
import workload
from common import f32, gacha_states, ppo_params

pytestmark = pytest.mark.gpu
DA = th.DeviceArray


def net_args(B, S, act=th.ACT_RELU, A=5):
    a = list(workload.REFERENCE_ACTOR_CRITIC)
    a[6], a[8] = A, act
    return (B, S, *a)


def tensor_sizes(A):
    return [512, 64, 64, 2048, 2048, 2048, 4096, 4096, 4096, 4096, 64, 8192, 128, 8192, 64, 64, 4096, 64, 64 * A, A, 64, 1]


def run(cfg, n, p, states, lens, actions, adv, ret, old, shift=0):
    plan = th.Plan("ppo", cfg)
    P = DA.from_numpy(p)
    raw = DA.zeros(states.size + 4)
    th.call("talos_memcpy_h2d", raw.offset(shift), states.ctypes.data, states.nbytes, None)
    dev = [DA.from_numpy(actions, np.int32)] + [DA.from_numpy(v) for v in (adv, ret, old)]
    L = None if lens is None else DA.from_numpy(lens, np.int32)
    lp = None if L is None else L.ptr
    loss, dp, stats = DA.zeros(1), DA.zeros(p.size), DA.from_numpy(np.full(5, 2.0), np.float64)
    lg, vl = DA.zeros((n, cfg.n_actions)), DA.zeros(n)
    th.call("talos_ppo_minibatch_f32", plan.h, n, P.ptr, raw.offset(shift), lp, dev[0].ptr, dev[1].ptr, dev[2].ptr,
            dev[3].ptr, loss.ptr, dp.ptr, stats.ptr, 1, None)
    th.call("talos_ppo_forward_n_f32", plan.h, n, P.ptr, raw.offset(shift), lp, lg.ptr, vl.ptr, None)
    out = [a.numpy().astype(np.float64) for a in (loss, dp, stats, lg, vl)]
    plan.destroy()
    return out


def both(monkeypatch, cfg, *args, **kw):
    got = run(cfg, *args, **kw)
    monkeypatch.setenv("TALOS_PLAN_UNFUSED", "1")
    ref = run(cfg, *args)
    monkeypatch.delenv("TALOS_PLAN_UNFUSED")
    return got, ref


def compare(got, ref, A):
    for name, g, r in zip(("loss", "stats", "logits", "values"), (got[0], got[2], got[3], got[4]),
                          (ref[0], ref[2], ref[3], ref[4])):
        np.testing.assert_allclose(g, r, rtol=2e-5, atol=2e-5, err_msg=name)
    floor, o = 1e-2 * np.linalg.norm(ref[1]), 0
    assert sum(tensor_sizes(A)) == ref[1].size
    for i, s in enumerate(tensor_sizes(A)):
        err = np.linalg.norm(got[1][o:o + s] - ref[1][o:o + s])
        assert err <= 1e-5 * max(np.linalg.norm(ref[1][o:o + s]), floor), (i, err)
        o += s


def inputs(rng, n, S, A, ragged):
    lens = rng.integers(1, S + 1, n).astype(np.int32) if ragged else None
    if ragged:
        lens[0], lens[-1] = S, 1
    return (f32(gacha_states(rng, n, S)).astype(np.float32), lens, rng.integers(0, A, n).astype(np.int32),
            rng.normal(size=n).astype(np.float32), rng.normal(size=n).astype(np.float32),
            rng.normal(-1.5, 0.2, n).astype(np.float32))


@pytest.mark.parametrize("n,batch,S,ragged,act,A,shift", [
    (1, 1, 1, False, th.ACT_RELU, 5, 0), (7, 9, 15, True, th.ACT_GELU, 5, 0), (9, 9, 16, True, th.ACT_GELU, 1, 1),
    (8, 8, 17, False, th.ACT_GELU, 8, 0), (5, 5, 31, True, th.ACT_RELU, 5, 3), (70, 70, 33, True, th.ACT_GELU, 5, 0),
    (3, 4, 127, True, th.ACT_GELU, 2, 0), (2, 2, 128, False, th.ACT_RELU, 5, 0), (2500, 2500, 3, True, th.ACT_GELU, 5, 0),
    (600, 640, 16, True, th.ACT_GELU, 5, 0), (300, 300, 65, False, th.ACT_GELU, 3, 0)])
def test_one_kernel_matches_separate_products(monkeypatch, n, batch, S, ragged, act, A, shift):
    rng = np.random.default_rng(900 + n + S)
    cfg = th.PpoCfg(*net_args(batch, S, act, A))
    p = f32(ppo_params(rng, cfg)).astype(np.float32)
    got, ref = both(monkeypatch, cfg, n, p, *inputs(rng, n, S, A, ragged), shift=shift)
    compare(got, ref, A)


@pytest.mark.parametrize("n,S", [(8, 15), (1, 15), (9, 17), (5, 16)])
def test_eps_zero(monkeypatch, n, S):
    """Token tiles that are not full (a group's tokens no multiple of 16, a last group of one sample) hold
    zero rows, whose 1 / sqrt(0 + eps) must not reach the gradients."""
    rng = np.random.default_rng(31 * n + S)
    a = list(net_args(n, S, th.ACT_GELU))
    assert a[11] == 1e-5
    a[11] = 0.0
    cfg = th.PpoCfg(*a)
    p = f32(ppo_params(rng, cfg)).astype(np.float32)
    got, ref = both(monkeypatch, cfg, n, p, *inputs(rng, n, S, 5, False))
    assert np.all(np.isfinite(got[1]))
    compare(got, ref, 5)


# The flat tensors in order, and those whose terms add in f64 over all samples
TENSORS = "we be g1 wdkv wuk wuv wq wkr wqr wo g2 w1 b1 w2 b2 gf wout bout wa ba wc bc".split()
F64_SUMS = "g1 g2 gf wa ba wc bc".split()


def test_small_terms_after_a_large_one():
    """65536 equal samples, the first with advantage and value error 1, the others with 2^-26: every
    gradient is the one sample's times 1 + 65535 * 2^-26 (all scales are powers of two, so each sample's own
    terms are exactly scaled copies). An fp32 sum that starts with the first sample keeps none of the
    terms after it, and loses 2^-26 a sample: a workgroup's run of at most 32 samples (512 tokens) 31 * 2^-26,
    and the final rounding and the sums over tokens a few 2^-24, below 2^-20 together. (A run over all of a CU's
    256 samples loses 3.8e-6.) The sums that are f64 throughout keep only the 2^-24 or so of their
    own terms and of the result's rounding: 2^-23. Elementwise, relative to the tensor's largest value."""
    n, S = 65536, 16
    a = list(net_args(n, S, th.ACT_GELU))
    a[15] = 0.0  # no entropy term: its gradient would not scale
    rng = np.random.default_rng(5)
    p = f32(ppo_params(rng, th.PpoCfg(*a))).astype(np.float32)
    p[-65:] = 0.0  # value 0 exactly
    small = np.float32(2.0**-26)
    one = f32(gacha_states(rng, 1, S)).astype(np.float32)

    def grads(B, count):
        a[0] = B
        scale = np.full(count, small, np.float32)
        scale[0] = 1.0
        # (a negative advantage and a ratio above 1 + clip: never clipped)
        return run(th.PpoCfg(*a), count, p, np.tile(one, (count, 1, 1)), None, np.full(count, 2, np.int32), -scale, -scale,
                   np.full(count, -6.0, np.float32))[1]

    ref = grads(1, 1) * (1.0 + (n - 1) * float(small)) / n
    got, o = grads(n, n), 0
    for name, size in zip(TENSORS, tensor_sizes(5)):
        g, r = got[o:o + size], ref[o:o + size]
        o += size
        assert np.abs(r).max() > 0, name
        err = np.abs(g - r).max() / np.abs(r).max()
        assert err <= (2.0**-23 if name in F64_SUMS else 2.0**-20), (name, err)


def test_out_of_range_action(monkeypatch):
    """NaN loss, and no gradient from that sample, as on the other path."""
    rng = np.random.default_rng(77)
    cfg = th.PpoCfg(*net_args(12, 16, th.ACT_GELU))
    p = f32(ppo_params(rng, cfg)).astype(np.float32)
    x = list(inputs(rng, 12, 16, 5, True))
    x[2][3], x[2][9] = 5, -1
    got, ref = both(monkeypatch, cfg, 12, p, *x)
    assert np.isnan(got[0][0]) and np.isnan(ref[0][0])
    got[0], ref[0] = np.zeros(1), np.zeros(1)
    compare(got, ref, 5)
