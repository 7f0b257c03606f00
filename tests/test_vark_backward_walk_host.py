"""CPU model of the backward walk of the rounds deal (make_sched in vark_kernel.h): the workgroups of
the odd XCDs may take their tiles from the last one back."""
import pytest


def _forward(p, num_wg, total):
    out, t, d, d_alt = [], p, 2 * (num_wg - p) - 1, 2 * p + 1
    while 0 <= t < total:
        out.append(t)
        t, d, d_alt = t + d, d_alt, d
    return out


def _backward(p, num_wg, total):
    k = (total - 1) // num_wg
    at_k = (k + 1) * num_wg - 1 - p if k & 1 else k * num_wg + p
    last = k if at_k < total else k - 1
    t = (last + 1) * num_wg - 1 - p if last & 1 else last * num_wg + p
    d0, d1 = 2 * (num_wg - p) - 1, 2 * p + 1
    d, d_alt = (-d0, -d1) if last & 1 else (-d1, -d0)
    out = []
    while 0 <= t < total:                                    # Sched::has: an unsigned comparison
        out.append(t)
        t, d, d_alt = t + d, d_alt, d
    return out


@pytest.mark.parametrize("num_wg", [8, 24, 256, 304])
def test_backward_walk_takes_the_same_tiles(num_wg):
    for total in (1, num_wg - 1, num_wg, num_wg + 1, 2 * num_wg, 2 * num_wg + 7, 5 * num_wg + num_wg // 2, 7 * num_wg - 1):
        for p in range(min(num_wg, total)):
            assert _backward(p, num_wg, total) == _forward(p, num_wg, total)[::-1], (total, p)
