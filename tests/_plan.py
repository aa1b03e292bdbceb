"""The choice of the wide items' height and width restated (launch.h ItemPlan,
capi.hip fused_plan, routing.hip item_plan), for tests of the choice and for
tests that need to know which tiles a case runs."""
import numpy as np

ITEM_COST, HALF_TILE, CUS = 256, 0.7, 32
SHORTER = [256, 224, 192, 160, 128]


def cuts(counts, h, nt):
    """Both cuts of the items over the XCDs, as (items of each XCD [8], time of the slowest in rows of cost)."""
    cost = np.concatenate([[(ITEM_COST * -(-n // h) + n) / -(-n // h)] * (-(-n // h) * nt) for n in counts if n] or [[]])
    total, below = len(cost), np.concatenate([[0.0], np.cumsum(cost)])
    per = -(-total // 8)
    equal = [min(total, x * per) for x in range(9)]
    # (a cut that falls between two items may round either way by one item)
    weighted = [int(np.searchsorted(below, below[-1] * x / 8 * (1 + 1e-12), side="right") - 1) for x in range(8)] + [total]
    for b in (equal, weighted):
        n = np.diff(b)
        s = np.diff(below[b]) if b is equal else below[-1] / 8 * np.ones(8)
        yield n, max([-(-int(k) // CUS) * c / k for k, c in zip(n, s) if k > 0] or [0.0])


def slots(P, E, tall, short, nt, nt_most):
    """The host's workgroups per XCD."""
    bound = lambda h, n: ((P // h + min(P, E)) * 256 + P) * n // (8 * 256) + 2
    return max(bound(tall, nt), min(bound(short, nt_most), CUS))


def options(P, E, H, I, tall):
    """What fused_plan allows: (nt1, nt2, any1, any2, bn2)."""
    used = min(P, E)
    items = used * -(-(-(-P // used)) // tall)
    nt1, nt2 = I // 128, H // 128
    bn2 = 128 if H % 256 else (0 if items * (H // 256) < 256 else 256)
    return nt1, nt2, items * nt1 <= 1024, items * ((nt2 + 1) // 2) <= 1024, bn2


def both_slots(P, E, tall, nt1, nt2, any1, any2, bn2):
    return (slots(P, E, tall, 128 if any1 else tall, nt1, nt1),
            slots(P, E, tall, 128 if any2 else tall, nt2 if bn2 == 128 else nt2 // 2, nt2 // 2 if bn2 == 256 else nt2))


def chosen(counts, H, I, tall):
    """((height of Stage 1's tallest items), (height, features) of Stage 2's) for these routed rows."""
    P, E = int(sum(counts)), len(counts)
    nt1, nt2, any1, any2, bn2 = options(P, E, H, I, tall)
    room = both_slots(P, E, tall, nt1, nt2, any1, any2, bn2)
    out = []
    for nts, shorter, r in (({128: nt1}, any1, room[0]),
                            ({w: nt2 * 128 // w for w in (256, 128) if bn2 in (0, w)}, any2, room[1])):
        est = {(h, w): min([t for k, t in cuts(counts, h, n) if k.max() <= r] or [np.inf]) *
               (HALF_TILE if w == 128 and nts is not None and len(out) == 1 else 1.0)
               for h in [tall] + SHORTER * shorter for w, n in nts.items()}
        out.append(min(est, key=est.get))
    return out[0][0], out[1]
