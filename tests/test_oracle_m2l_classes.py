"""The offset classes of the target-stationary M2L, on the oracle's translation.

Offsets of equal |dz| and dx^2 + dy^2 differ by a rotation about z and the
reflection z -> -z, so the translation by any of them is the one by the class
representative (same dx^2 + dy^2, dz >= 0, azimuth 0) between the diagonal
matrices e^{+-i m phi} (-1)^(n+m) that the kernel's phase table holds."""
import numpy as np

import oracle as O


def _offsets():
    for dx in range(-3, 4):
        for dy in range(-3, 4):
            for dz in range(-3, 4):
                if max(abs(dx), abs(dy), abs(dz)) > 1:
                    yield dx, dy, dz


def test_every_offset_is_its_class_translation():
    """All 316 offsets at order 7 against their class's representative, to
    1e-12 of the result (two FP64 evaluations of one expansion)."""
    p, k, side = 7, 9.0, 0.1
    n = np.repeat(np.arange(p), 2 * np.arange(p) + 1)
    m = np.concatenate([np.arange(-q, q + 1) for q in range(p)])
    rng = np.random.default_rng(3)
    x = rng.standard_normal(p * p) + 1j * rng.standard_normal(p * p)
    classes = set()
    for dx, dy, dz in _offsets():
        classes.add((dx * dx + dy * dy, abs(dz)))
        want = O.translate(O.COAX_SR, p, p, k, side * np.array([dx, dy, dz], float), x)
        w = np.exp(1j * m * np.arctan2(dy, dx)) * (np.where((n + m) % 2, -1.0, 1.0) if dz < 0 else 1)
        rep = side * np.array([np.hypot(dx, dy), 0.0, abs(dz)])
        got = np.conj(w) * O.translate(O.COAX_SR, p, p, k, rep, w * x)
        assert np.linalg.norm(got - want) <= 1e-12 * np.linalg.norm(want), (dx, dy, dz)
    assert len(classes) == 34
