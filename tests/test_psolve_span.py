"""The periodic line solves address a wave's rows by 32-bit offsets from its first lane, and the
launch checks them against the segments that a wave's 64 lanes span: (TI - gcd(64, TI) + 63) // TI for
blocks of TI columns.  Here the span is counted wave by wave for every block the launch can choose,
and the offsets it allows are checked to hold every grid that fits in 288 GB."""
import math

import pytest


def shapes(mixed):
    """(rows m, segment rows, TI, S) of the launch"""
    maxm, timin = (64, 32) if mixed else (32, 16)
    for n in range(3, 1026):
        m = n - 1
        S = -(-m // maxm)
        TI = min(64, max(timin, 512 // S))
        if TI * S <= 512:
            yield n, m, -(-m // S) if mixed else maxm, TI, S


def gspan(TI):
    return (TI - math.gcd(64, TI) + 63) // TI


@pytest.mark.parametrize("mixed", [False, True])
def test_span_of_a_wave(mixed):
    for n, m, seg, TI, S in shapes(mixed):
        g = TI & -TI if TI & -TI & 63 else 64
        assert g == math.gcd(64, TI)
        most = max((min(l + 63, TI * S - 1) // TI) - l // TI for l in range(0, TI * S, 64))
        assert most <= gspan(TI), (n, TI, S)
        if S > 4:
            # not by more than the lanes a last, partly filled wave lacks
            assert most >= gspan(TI) - 1, (n, TI, S)


@pytest.mark.parametrize("mixed", [False, True])
def test_every_grid_that_fits_is_accepted(mixed):
    """z solves: a plane is at most the cells left by the field arrays (FP64: 16 of the four
    fields and their sources, pressure, potential, spectrum and half of it for the radial
    factors, 156 bytes a cell; mixed: 132), and by the longest lines of 1024 and 8192 cells"""
    cells = 288 * 2 ** 30 // (132 if mixed else 156)
    smooth = [n for n in range(3, 1026) if n == math.prod(p ** e for p, e in factors(n))]
    accepted = {n: (gspan(TI) * seg + 8) * 8 for n, m, seg, TI, S in shapes(mixed)}
    for n in smooth:
        if n in accepted:
            plane = min(cells // (n + 2), 1056 * 8194)
            assert accepted[n] * plane < 2 ** 32, n


def factors(n):
    out = []
    for p in (2, 3, 5, 7):
        e = 0
        while n % p == 0:
            n //= p
            e += 1
        out.append((p, e))
    return out
