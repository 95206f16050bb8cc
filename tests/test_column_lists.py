"""The column kernels' wave-uniform pixel lists, slab bounds and table range,
restated in float64: every (voxel, pixel) pair with nonzero weight in the 25-tap
windows is visited, and no index leaves the pair table."""
import numpy as np
import pytest

CT_LO, CT_HI = -576, 1200  # mgg_kernels.hip: ct_lo, ct_hi of the back projection
ADJ_LO, ADJ_HI = -800, 1416


def frames(count, seed):
    """Rotations: random, with the normal near a diagonal or an edge, and axis permutations."""
    r = np.random.default_rng(seed)
    out = [np.roll(np.eye(3), k, axis=1) for k in range(3)]
    for t in range(count):
        n = r.standard_normal(3)
        if t % 3 == 1:
            n = np.sign(n) * (1 + r.choice([0.0, 0.01, 0.1]) * r.standard_normal(3))
        if t % 6 == 5:
            n[r.integers(3)] = 0.0
        n /= np.linalg.norm(n)
        u = np.cross(r.standard_normal(3), n)
        u /= np.linalg.norm(u)
        out.append(np.stack([u, np.cross(n, u), n]))
    return out


def pixel_list(u, v, a, b):
    di, dj = np.meshgrid(np.arange(-8, 8), np.arange(-8, 8))
    ok = np.ones(di.shape, bool)
    for k in (a, b):
        ok &= np.abs(u[k] * di + v[k] * dj) <= 2.02 + 0.5 * (abs(u[k]) + abs(v[k]))
    return di[ok], dj[ok]


@pytest.mark.parametrize("seed", [0, 1])
def test_lists_cover_the_windows(seed):
    rng = np.random.default_rng(seed + 10)
    for u, v, n in frames(150, seed):
        c = int(np.argmax(np.abs(n)))
        a, b = [k for k in range(3) if k != c]
        di, dj = pixel_list(u, v, a, b)
        assert max(np.abs(di).max(), np.abs(dj).max()) <= 7
        listed = set(zip(di.tolist(), dj.tolist()))
        slab = 2 / abs(n[c])
        slots = 5 if 2 * slab + 1.5e-2 < 5 else 6 if 2 * slab + 1.5e-2 < 6 else 7
        for _ in range(8):
            x = rng.integers(-120, 121, 3).astype(float)
            zc = -(n[a] * x[a] + n[b] * x[b]) / n[c]
            x[c] = zc
            i0, j0 = np.rint(u @ x), np.rint(v @ x)
            v0 = np.ceil(zc - slab - 5e-3)
            pc = (i0 + di) * u[c] + (j0 + dj) * v[c]
            idx = np.floor(125 * (pc - v0) + 250.5)
            if slots < 7:  # longer columns clamp
                assert idx.max() < CT_HI and idx.min() - 250 * ((slots + 1) // 2 - 1) >= CT_LO
            for z in range(int(zc) - 5, int(zc) + 6):
                x[c] = z
                if abs(n @ x) > 2:
                    continue
                assert v0 <= z < v0 + slots
                i, j = np.rint(u @ x), np.rint(v @ x)
                for q in range(int(j) - 2, int(j) + 3):
                    for p in range(int(i) - 2, int(i) + 3):
                        if np.all(np.abs(p * u + q * v - x) < 2):
                            assert (p - i0, q - j0) in listed
                assert abs(i - i0) <= 3 and abs(j - j0) <= 3


@pytest.mark.parametrize("seed", [2, 3])
def test_transposed_columns_cover_the_pixels_windows(seed):
    rng = np.random.default_rng(seed)
    for u, v, n in frames(150, seed):
        c = int(np.argmax(np.abs(n)))
        a, b = [k for k in range(3) if k != c]
        di, dj = pixel_list(u, v, a, b)
        half = 2 * np.abs(n).sum() / abs(n[c])
        slots = next(k for k in (6, 8, 10, 14) if k == 14 or 2 * half + 1.5e-2 < k)
        for _ in range(8):
            p = rng.integers(-90, 91, 2)
            pos = p[0] * u + p[1] * v
            start = np.floor(pos) - 1  # the 4 x 4 x 4 window of the forward gather
            for xa in range(4):
                for xb in range(4):
                    va, vb = start[a] + xa, start[b] + xb
                    x = np.zeros(3)
                    x[a], x[b] = va, vb
                    zc = -(n[a] * va + n[b] * vb) / n[c]
                    x[c] = zc
                    top = np.floor(zc + half + 5e-3)
                    assert start[c] + 3 <= top and start[c] > top - slots
                    i0, j0 = np.rint(u @ x), np.rint(v @ x)
                    assert np.any((di == p[0] - i0) & (dj == p[1] - j0))
                    pc = (i0 + di) * u[c] + (j0 + dj) * v[c]
                    idx = np.floor(125 * (top - pc) + 250.5)
                    if slots < 14:  # longer columns clamp
                        assert idx.max() < ADJ_HI and idx.min() - 250 * (slots // 2 - 1) >= ADJ_LO
