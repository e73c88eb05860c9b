"""The rule that gives a separable table the direct-convolution form
(dir_classify_kernel in vfd_direct.hpp), restated with numpy: inverting a
window's DFT table and transforming it back reproduces the table far inside
the rule's 1e-12, on every box length class and radius the rule accepts, while
wider windows and perturbed tables miss it by orders of magnitude."""
import numpy as np
import pytest

MAX_R, TOL = 31, 1e-12


def _window(radius):
    s2 = ((radius - 0.5) / 6.0) ** 2
    j = np.arange(-radius, radius + 1)
    g = np.exp(-j * j / (2.0 * s2))
    return g / g.sum()


def _table(g, p):
    """DFT of the window on a box of p, entries k <= p/2, as the library's host code forms it."""
    R = (len(g) - 1) // 2
    k = np.arange(p // 2 + 1)
    j = np.arange(-R, R + 1)
    ang = (j[None, :] * k[:, None]) % p
    return (g[None, :].astype(np.longdouble) * np.cos(2 * np.pi * ang.astype(np.longdouble) / p)).sum(1).astype(np.float64)


def _classify(t, p, n):
    """(radius or -1, worst residual relative to the bound of the entries)."""
    K = p // 2
    J = min(MAX_R, (p - 1) // 2)
    w = np.where((np.arange(K + 1) == 0) | (2 * np.arange(K + 1) == p), 1.0, 2.0) * t
    h = np.zeros(MAX_R + 1)
    for j in range(J + 1):
        h[j] = (w * np.cos(2 * np.pi * ((j * np.arange(K + 1)) % p) / p)).sum() / p
    gmax = abs(h[0]) + 2 * np.abs(h[1:]).sum()
    k = np.arange(K + 1)
    c1, s1 = np.cos(2 * np.pi * k / p), np.sin(2 * np.pi * k / p)
    c, s, r = c1.copy(), s1.copy(), np.full(K + 1, h[0])
    for j in range(1, MAX_R + 1):                      # the kernel's rotation
        r += 2.0 * h[j] * c
        c, s = c * c1 - s * s1, s * c1 + c * s1
    res = np.abs(r - t).max() / gmax
    R = np.nonzero(np.abs(h) > 1e-13 * np.abs(h).max())[0].max()
    return (int(R) if res <= TOL and R <= p - n else -1), res


@pytest.mark.parametrize("p,n", [(64, 32), (80, 40), (96, 40), (128, 64), (616, 301), (640, 320), (1152, 560),
                                 (2048, 1024), (3072, 1536)])
def test_windows_are_recognized(p, n):
    for radius in (1, 2, 6, 13, 19, 30, 31):
        if radius > min(MAX_R, (p - 1) // 2):
            continue
        g = _window(radius)
        R, res = _classify(_table(g, p), p, n)
        taps = np.nonzero(g[radius:] > 1e-13 * g[radius])[0].max()   # the narrowest windows end before their radius
        assert R == taps, (p, radius, R, res)
        assert res <= 1e-13                            # ten times inside the rule


@pytest.mark.parametrize("p,n", [(128, 64), (616, 301), (2048, 1024)])
def test_other_tables_are_not(p, n):
    for radius in (32, 36, 60):                        # taps past the largest radius
        R, res = _classify(_table(_window(radius), p), p, n)
        assert R == -1 and res > 1e-9, (p, radius, res)
    t = _table(_window(8), p)
    t[7] += 1e-11                                      # one entry off
    assert _classify(t, p, n)[0] == -1
    assert _classify(np.ones(p // 2 + 1) / (1 + np.arange(p // 2 + 1)), p, n)[0] == -1
    # a box that leaves fewer zeros than the window's radius: the FFT form wraps
    assert _classify(_table(_window(8), p), p, p - 4)[0] == -1
