"""The paired form of one MFT stage, written out in NumPy from the identities
the GEMM relies on, against the direct complex128 sum:

    C[j] = sum_k A[k] cis(alpha x_k (j - N/2 - shift))
         = cis(alpha xc Y) (P +- iQ),  Y = j - c,
    P = sum_k' Ae cos(2 pi alpha x' Y),  Q = sum_k' Ao sin(2 pi alpha x' Y),

with the fold cis(-alpha (shift + N/2 - c) x_k) in A, Ae / Ao the sum /
difference of the samples x' either side of the midpoint xc, and segments with
midpoints of their own joined by turning (P, Q).  Every parity, offset sign,
shift and pairing centre the kernels accept."""
import numpy as np
import pytest


def cis(t):
    return np.exp(2j * np.pi * t)


def grid(shift, N):
    """Slots, pairing columns and centre, by the rule of the planner."""
    h, mid = N // 2, 0.5 * (N - 1)
    core = h + shift
    if abs(core - mid) <= 1:
        c = mid
    else:
        c = np.rint(2 * core) / 2
        if not 0 <= c <= N - 1 or max(N - np.ceil(c), np.floor(c) + 1) > 0.75 * N:
            c = 0.0
    cm, cp = int(np.floor(c)), int(np.ceil(c))
    return max(N - cp, cm + 1), cp, cm, c - cm, c


def pair_index(n, i):
    h = n // 2
    plus = h + i
    minus = (h - i if i else -1) if n % 2 else h - 1 - i
    return (plus if plus < n else -1), minus


def paired(segments, alpha, shift, N):
    """The stage over segments [(A, x0)], each A sampled at x0 + k."""
    slots, cp, cm, y0, c = grid(shift, N)
    Y = y0 + np.arange(slots)
    P = np.zeros(slots, complex)
    Q = np.zeros(slots, complex)
    last = None
    for A, x0 in segments:
        n = len(A)
        xc = x0 + (n - 1) / 2
        if last is not None:  # turn the sum so far to this segment's midpoint
            r = 2 * np.pi * alpha * (last - xc) * Y
            P, Q = np.cos(r) * P - np.sin(r) * Q, np.sin(r) * P + np.cos(r) * Q
        last = xc
        folded = A * cis(-alpha * (shift + N // 2 - c) * (x0 + np.arange(n)))
        for i in range((n + 1) // 2):
            plus, minus = pair_index(n, i)
            a = folded[plus] if plus >= 0 else 0
            b = folded[minus] if minus >= 0 else 0
            xp = i if n % 2 else i + 0.5
            P = P + (a + b) * np.cos(2 * np.pi * alpha * xp * Y)
            Q = Q + (a - b) * np.sin(2 * np.pi * alpha * xp * Y)
    turn = cis(alpha * last * Y)
    out = np.full(N, np.nan, complex)
    for s in range(slots):
        jp, jm = cp + s, cm - s
        if jp < N:
            out[jp] = turn[s] * (P[s] + 1j * Q[s])
        if 0 <= jm < N and jm != jp:
            out[jm] = np.conj(turn[s]) * (P[s] - 1j * Q[s])
    return out


@pytest.mark.parametrize('n', [1, 2, 3, 16, 17, 32, 33])
@pytest.mark.parametrize('N', [1, 2, 5, 16, 31])
@pytest.mark.parametrize('shift, offset', [(0.0, 0), (0.3, -4), (-2.5, 7), (40.0, 1), (-1.25, -60)])
def test_paired_stage_is_the_direct_sum(n, N, shift, offset):
    rng = np.random.default_rng(n * 100 + N)
    for alpha in (0.013, -0.07):
        A = rng.standard_normal(n) + 1j * rng.standard_normal(n)
        x = np.arange(n) - n // 2 + offset
        ref = np.array([np.sum(A * cis(alpha * x * (j - N // 2 - shift))) for j in range(N)])
        # every term is exact in double but for its rounding: n terms of size 1, phases of up to 1e3 turns
        assert np.max(np.abs(paired([(A, x[0])], alpha, shift, N) - ref)) < 1e-9


def test_segments_join_by_turning():
    rng = np.random.default_rng(5)
    alpha, shift, N = 0.011, 3.7, 40
    segs = []
    ref = np.zeros(N, complex)
    for n, x0 in ((17, -40), (24, 3), (5, 61)):
        A = rng.standard_normal(n) + 1j * rng.standard_normal(n)
        x = x0 + np.arange(n)
        ref += np.array([np.sum(A * cis(alpha * x * (j - N // 2 - shift))) for j in range(N)])
        segs.append((A, x0))
    assert np.max(np.abs(paired(segs, alpha, shift, N) - ref)) < 1e-10
