"""The guards of the FP16 MFMA refine, checked on the CPU.

The library (hegj_g16_operands, the host build of the device code) gives the
FP16 operands A', B' and the guards w of each point.  A product of two FP16
values is exact in FP32; the order and rounding of the FP32 additions inside
v_mfma_f32_16x16x32_f16 are not published, so s' = A'_q . B'_c is summed under
the adversarial models of the split-BF16 test, and every decision that the
kernel would take is compared with the reference's FP64 chain
(kernel.cu:347-355):
    reject  s' > trej             must imply acc > T
    accept  s' + w_q + w_c <= tacc  must imply acc <= T.

The guard of a point is its own measured rounding error E, used through the
triangle inequality.  `aligned` pairs make that an equality: both rounding
errors lie along the pair's difference, so nothing of the guard is to spare and
a shrunk one decides wrongly."""
import math

import numpy as np
import pytest

from test_mfma_band import mfma_sum, near_threshold_pairs


def f16(b):
    return b.view(np.float16).astype(np.float64)


def aligned(rng, dim, m=400, far=2800):
    """Pairs whose distance is `far` + 0.9 units of the FP16 spacing per
    dimension (times 1 + r, |r| down to 1e-13) while that of their FP16 values
    is a whole number of units: larger by 0.1 or smaller by 0.9.  The ends lie
    on both sides of the centre: then the guard of the FP32 additions, which
    grows with the norms, is small beside that of the rounding."""
    u = 2.0 ** -7  # the spacing in [8, 16)
    sgn = rng.choice([-1.0, 1.0], (m, dim))
    zq = -sgn * rng.integers(1200, 1600, (m, dim)) * u
    want = (far + 0.9) * (1 + rng.choice([-1, 1], m) * 10 ** rng.uniform(-13, -4, m))
    z = np.where(rng.random(m) < 0.5, np.floor(want), np.ceil(want))
    f = (want - z) / 2  # each end's error, in units along the difference
    q = zq - sgn * f[:, None] * u
    c = zq + sgn * z[:, None] * u + sgn * f[:, None] * u
    return q, c, (far + 0.9) * u * math.sqrt(dim)


def decide(H, q, c, eps, scale, mode, order, perm):
    m = len(q)
    A, B, w, kp, trej, tacc = H.g16_operands(np.concatenate([q, c]), np.zeros(q.shape[1]), eps, scale)
    prod = f16(A[:m]) * f16(B[m:])
    if perm is not None:
        prod = prod[:, perm]
    s = mfma_sum(prod, mode, order).astype(np.float64)
    w = w.astype(np.float64)
    return s > trej, s + w[:m] + w[m:] <= tacc


def models(rng, kp):
    for mode in ("rne", "rz", "ru", "rd"):
        for order in ("seq", "block"):
            for perm in (None, np.arange(kp)[::-1], rng.permutation(kp)):
                yield mode, order, perm


@pytest.mark.parametrize("kind", ["aligned", "spread"])
@pytest.mark.parametrize("dim", [16, 18, 28, 29, 60, 61, 90, 124])
def test_decisions_are_sound(oracle, dim, kind):
    import hegjoin_amd as H
    rng = np.random.default_rng(dim)
    kp = H.g16_operands(np.zeros((1, dim)), np.zeros(dim), 0.1)[3]
    assert kp % 32 == 0 and kp >= dim + 4
    if kind == "aligned":
        q, c, eps = aligned(rng, dim)
    else:
        eps = 0.05 * math.sqrt(dim)
        q, c = near_threshold_pairs(oracle, rng, dim, oracle.threshold(eps))
    truth = oracle.chain(q, c) <= oracle.threshold(eps)
    assert truth.any() and (~truth).any()
    for mode, order, perm in models(rng, kp):
        reject, accept = decide(H, q, c, eps, 1.0, mode, order, perm)
        assert not (reject & truth).any(), (mode, order)
        assert not (accept & ~truth).any(), (mode, order)
        assert (~reject & ~accept).any()  # a band exists
    # the check can fail: guards a fifth tighter (spread pairs: none) decide wrongly
    wrong = 0
    for scale in ((0.8,) if kind == "aligned" else (0.0,)):
        for mode in ("ru", "rd"):
            reject, accept = decide(H, q, c, eps, scale, mode, "seq", None)
            wrong += int((reject & truth).sum() + (accept & ~truth).sum())
    assert wrong > 0


@pytest.mark.parametrize("eps", [1.0, 1e-3, 1e-30, 1e-100, 1e-140])
def test_decisions_are_sound_at_every_scale(oracle, eps):
    """The operands are scaled by a power of two: the same decisions at any
    eps whose square is a normal number."""
    import hegjoin_amd as H
    rng = np.random.default_rng(7)
    q, c, e = aligned(rng, 18)
    s = eps / e
    q, c = q * s, c * s
    truth = oracle.chain(q, c) <= oracle.threshold(eps)
    for mode in ("rne", "ru", "rd"):
        reject, accept = decide(H, q, c, eps, 1.0, mode, "seq", None)
        assert not (reject & truth).any() and not (accept & ~truth).any()


@pytest.mark.parametrize("eps", [2.0 ** -500, 2.0 ** -515, 2.0 ** -525, 2.0 ** -530, 2.0 ** -534, 2.0 ** -536])
def test_decisions_where_squares_underflow(oracle, eps):
    """Thresholds down to a few units of the smallest FP64 number, where the
    FP64 chain itself rounds by parts of T.  Points that FP16 holds exactly
    (E = 0), so no other guard hides it."""
    import hegjoin_amd as H
    rng = np.random.default_rng(9)
    dim, m, u = 18, 3000, 2.0 ** -10
    q = rng.integers(-1000, 1000, (m, dim)) * u
    d = rng.standard_normal((m, dim))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    c = np.rint((q + d * (1 + rng.uniform(-0.02, 0.02, (m, 1)))) / u) * u
    q, c = q * eps, c * eps
    truth = oracle.chain(q, c) <= oracle.threshold(eps)
    assert truth.any() and (~truth).any()
    for mode in ("rne", "ru", "rd"):
        reject, accept = decide(H, q, c, eps, 1.0, mode, "seq", None)
        assert not (reject & truth).any() and not (accept & ~truth).any()
