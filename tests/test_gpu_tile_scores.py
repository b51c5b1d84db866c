"""The FP32-exact attention kernels (attention.hip) over the range of finite
scores: rows whose maximum is far from zero, held by several keys in different
tiles and splits, so that the context is the mean of those keys' V exactly
whatever rounds below them; light keys beside a heavy one that has nothing to add;
and scales at the ends of FP32."""

import numpy as np
import pytest

from gpu_util import dev, host, log, stored

pytestmark = pytest.mark.gpu

QUERIES, HQ, HKV = 5, 4, 2


@pytest.fixture(scope="module")
def torch_mod():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a ROCm device"
    return torch


def _exact_kernels(dt, D, diag):
    """Calls that reach attention.hip: bf16/f16 without diagnostics at head sizes
    64, 128 and 256 belong to other kernels."""
    return dt == "f32" or diag or D not in (64, 128, 256)


def _run(torch, orc, q, k, v, dt, scale, softcap=0.0, diag=False, check=True):
    """(got, expected) contexts, scores and probabilities."""
    from toklet_amd import ops

    Q, hq, D = q.shape
    hkv, keys, _ = k.shape
    ref = orc.window_attention(q.reshape(-1), k.reshape(-1), v.reshape(-1), Q, keys, keys, hq, hkv, D, keys - Q, 0, None,
                               scale, softcap=softcap) if check else None
    ctx = ops.Context(0)
    out = torch.full((Q * hq * D,), np.nan, device="cuda")
    sc, pr = (torch.full((hq * Q * keys,), np.nan, device="cuda") if diag else None for _ in range(2))
    try:
        ops.window_attention(ctx, dev(q.reshape(-1), dt), dev(k.reshape(-1), dt), dev(v.reshape(-1), dt), out, sc, pr,
                             ops.WindowAttentionShape(Q, keys, keys, hq, hkv, D, keys - Q, 0, None, scale, softcap))
        return [host(x) if x is not None else None for x in (out, sc, pr)], ref
    finally:
        ctx.close()


@pytest.mark.parametrize("diag", [False, True])
@pytest.mark.parametrize("keys", [15, 700])  # one tile; several splits
@pytest.mark.parametrize("D", [64, 96, 256, 512])
@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
def test_row_maximum_weighs_one(torch_mod, orc, dt, D, keys, diag):
    if not _exact_kernels(dt, D, diag):
        pytest.skip("another kernel's call")
    rng = np.random.default_rng(D + keys)
    sign = np.sign(rng.standard_normal(D)).astype(np.float32)
    v = stored(rng.standard_normal((HKV, keys, D)), dt)
    top = [2, 9] if keys == 15 else [3, 250, 251, 600, 690]
    scale = 1.0 / np.sqrt(D)
    largest = 65504.0 ** 2 * D * scale
    for score in (1e2, 1e5, 1e8, 3e8, 1e9, 1e10, largest) + ((1e30,) if dt != "f16" else ()):
        a = np.sqrt(score * np.sqrt(D) / D)
        q = sign * np.float32(a) * np.where(np.arange(QUERIES * HQ) % 2, 0.5, 1.0).reshape(QUERIES, HQ, 1)
        k = -sign * np.float32(a) * rng.uniform(0.3, 1.0, (HKV, keys, 1))
        k[:, top] = sign * np.float32(a)
        q, k = stored(q, dt), stored(k, dt)
        for softcap in (0.0, 2.0 * score):
            got, ref = _run(torch_mod, orc, q, k, v, dt, scale, softcap, diag)
            worst = np.max(np.abs(got[0] - ref[0]) - 1e-4 * np.abs(ref[0]))
            log(f"{dt} D={D} keys {keys} diag {diag} score {score:.3g} cap {softcap:.3g}: worst excess {worst:.2e}")
            # The reference's gate for FP32 arithmetic (tests/cpu_attention.rs:6-14).
            assert np.all(np.isfinite(got[0])) and worst <= 1e-5
            if diag:
                # An FP32 dot of D products (and the softcap's tanh): D ulps at most.
                assert np.all(np.abs(got[1] - ref[1]) <= D * 2.0 ** -23 * np.abs(ref[1]))
                assert np.max(np.abs(got[2] - ref[2])) <= 1e-5


@pytest.mark.parametrize("diag", [False, True])
@pytest.mark.parametrize("D", [64, 96, 256, 512])
@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
def test_light_keys_keep_their_bits(torch_mod, orc, dt, D, diag):
    """A heavy key whose V is zero, and keys e^-25 and e^-60 as heavy: their sum is
    all of the context, so a weight that lost bits or fell to zero shows at full
    size.  Weights are 2^t with t rounded to FP32 (at most 87, half an ulp 2^-18)
    and V, P and sums as FP32 keeps them: within 1e-5 of the result."""
    if not _exact_kernels(dt, D, diag):
        pytest.skip("another kernel's call")
    rng = np.random.default_rng(D)
    keys = 70
    for nats in (25.0, 60.0):
        v = np.zeros((HKV, keys, D), np.float32)
        k = np.zeros((HKV, keys, D), np.float32)
        k[:, 1:, 0] = -4.0
        v[:, 1:] = rng.uniform(100.0, 400.0, (HKV, keys - 1, D))
        q = np.zeros((QUERIES, HQ, D), np.float32)
        q[:, :, 0] = nats / 4.0
        q, k, v = (stored(x, dt) for x in (q, k, v))
        got, ref = _run(torch_mod, orc, q, k, v, dt, 1.0, diag=diag)
        worst = np.max(np.abs(got[0] / ref[0].astype(np.float64) - 1.0))
        log(f"{dt} D={D} diag {diag} {nats} nats: relative error {worst:.2e}")
        assert worst <= 1e-5


@pytest.mark.parametrize("diag", [False, True])
@pytest.mark.parametrize("D", [64, 256])
def test_scales_at_the_ends(torch_mod, orc, D, diag):
    """Scores of ordinary size from dots near FP32's largest, and from dots as small
    as the scale is large."""
    rng = np.random.default_rng(D)
    keys = 70
    v = stored(rng.standard_normal((HKV, keys, D)), "f32")
    sign = np.sign(rng.standard_normal(D)).astype(np.float32)
    for scale, dot in ((2.0 ** -124, 2.9e38), (2.0 ** -99, 2.0 ** 102), (2.0 ** 99, 2.0 ** -96), (2.0 ** 110, 2.0 ** -107)):
        a = np.sqrt(dot / D)
        q = np.broadcast_to(sign * a, (QUERIES, HQ, D)).astype(np.float32)
        k = (sign * a * rng.uniform(-1.0, 1.0, (HKV, keys, 1))).astype(np.float32)
        got, ref = _run(torch_mod, orc, q, k, v, "f32", np.float32(scale), diag=diag)
        worst = np.max(np.abs(got[0] - ref[0]) - 1e-4 * np.abs(ref[0]))
        log(f"D={D} diag {diag} scale {scale:.3g}: worst excess {worst:.2e}")
        assert np.all(np.isfinite(got[0])) and worst <= 1e-5


@pytest.mark.parametrize("diag", [False, True])
@pytest.mark.parametrize("dt,D", [("f32", 64), ("f32", 256), ("bf16", 96)])
def test_scores_past_the_largest_are_refused(torch_mod, orc, dt, D, diag):
    """Finite operands whose scaled score is not: refused whichever sign it has, also
    where a larger finite score would leave it no weight."""
    from toklet_amd import ops

    q = np.ones((QUERIES, HQ, D), np.float32)
    for sign in (-1.0, 1.0):
        k = np.zeros((HKV, 40, D), np.float32)
        k[:, 7] = sign * 1e9
        with pytest.raises(ops.TkhError) as e:
            _run(torch_mod, orc, q, stored(k, dt), np.ones_like(k), dt, 1e30, diag=diag, check=False)
        assert e.value.name == "NonFinite"


@pytest.mark.parametrize("softcap", [0.0, 30.0])
@pytest.mark.parametrize("dt,D,diag", [("f32", 64, False), ("f32", 256, True), ("bf16", 96, False), ("f16", 128, True)])
def test_nan_operands_are_refused(torch_mod, orc, dt, D, diag, softcap):
    """Also with a softcap, whose tanh saturates for any size of score."""
    from toklet_amd import ops

    for at in range(3):
        operands = [np.ones((QUERIES, HQ, D), np.float32), *(np.ones((HKV, 40, D), np.float32) for _ in range(2))]
        operands[at][1, 3, 5] = np.nan
        with pytest.raises(ops.TkhError) as e:
            _run(torch_mod, orc, *operands, dt, 1.0, softcap, diag, check=False)
        assert e.value.name == "NonFinite"
