"""CPU model of parts of make_sched (vark_kernel.h): the backward walk of the rounds deal, in which the
workgroups of the odd XCDs may take their tiles from the last one back, and the slices' bounds."""
import random

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


def _bounds(w_slot, tpg):
    """The kernel's form: every slot looks for the targets that its work reaches."""
    total_w, before = sum(w_slot) * tpg, 0
    bounds = [0] * 4 + [len(w_slot) * tpg]
    for sl, w in enumerate(w_slot):
        after = before + w * tpg
        for x in range(1, 4):
            target = total_w * x // 4
            if before < target <= after:
                bounds[x] = sl * tpg + min(-(-(target - before) // w), tpg)
        before = after
    return bounds


def _first_tiles(w_slot, tpg):
    """Slice x starts at the first tile that x / 4 of all work precede."""
    done = [0]
    for w in w_slot:
        done += [done[-1] + w * (i + 1) for i in range(tpg)]
    return [next(t for t, d in enumerate(done) if d >= done[-1] * x // 4) for x in range(4)] + [len(done) - 1]


def test_slice_bounds_also_of_one_tile():
    """The bounds of the smallest launches included, where a quarter of the work rounds to nothing."""
    rng = random.Random(0)
    small = [([w] * G, tpg) for w in (1, 2, 3, 5) for G in (1, 2, 3) for tpg in (1, 2, 3)]
    for w_slot, tpg in small + [([rng.randint(1, 99) for _ in range(rng.randint(1, 40))], rng.randint(1, 50))
                                for _ in range(200)]:
        assert _bounds(w_slot, tpg) == _first_tiles(w_slot, tpg), (w_slot, tpg)


def walks_backwards(lens, tiles_of_group, stage, epi_w, light, num_wg=256):
    """Whether the odd XCDs of an fp32 launch walk back: the rounds deal is strictly the lighter one and the
    stages that the tiles' C stores are worth (``light`` each) are a quarter of the work or more.
    ``tiles_of_group`` tiles in every group, ``stage`` tokens a stage."""
    w = sorted((-(-n // stage) + epi_w for n in lens), reverse=True)
    tpg, total = tiles_of_group, len(lens) * tiles_of_group
    bounds, wpx = _bounds(w, tpg), num_wg // 8

    def heaviest(walk):
        return max(sum(w[t // tpg] for t in walk(wg)) for wg in range(num_wg))

    def slices(wg):
        xcd = wg % 8
        return range(bounds[xcd % 4] + xcd // 4 * wpx + wg // 8, bounds[xcd % 4 + 1], 2 * wpx)

    rounds = heaviest(lambda wg: _forward(wg % 8 * wpx + wg // 8, num_wg, total))
    return rounds < heaviest(slices) and 4 * sum(max(0, light + epi_w - x) for x in w) >= sum(w) and total > num_wg


def test_the_full_size_lengths_walk_as_measured():
    """Zipf lengths of 16384 tokens walk back on the 320 x 320 tiles of [32, 2880, 5760] in both fp32 modes,
    even lengths of 131072 do not."""
    raw = [1 / (i + 1) ** 1.2 for i in range(24)]
    zipf = [int(16384 * r / sum(raw)) for r in raw] + [0] * 8
    for light in (16, 32):
        assert walks_backwards(zipf, 162, 64, 3, light)
        assert not walks_backwards([4096] * 32, 162, 64, 3, light)
