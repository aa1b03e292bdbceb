"""The plan of a fused launch's wide items (launch.h ItemPlan), read back from
align's own output: for even and skewed routings it covers every item once
within the workgroups that the host launches, uses a height and width that it
may, and takes the one whose slowest XCD, restated here, ends first."""
import ctypes

import numpy as np
import pytest
import torch

from _plan import HALF_TILE, SHORTER, both_slots, cuts

pytestmark = pytest.mark.gpu

LAUNCH_ALIGN = "_ZN3moe12launch_alignEPKiiiiPiS2_S2_S2_S2_S2_P12ihipStream_tiRKNS_8ItemPlanE"


class ItemPlan(ctypes.Structure):
    _fields_ = [("out", ctypes.c_void_p), ("tall", ctypes.c_int), ("nt1", ctypes.c_int), ("nt2", ctypes.c_int),
                ("any1", ctypes.c_bool), ("any2", ctypes.c_bool), ("bn2", ctypes.c_int),
                ("slots1", ctypes.c_int), ("slots2", ctypes.c_int)]


def _plan(counts, tall, nt1, nt2, any1, any2, bn2, slots, bm=64):
    """align's plan for `counts` routed rows per expert, as (istart1, istart2, xb1, xb2, bn)."""
    from muxi_race_amd._lib import lib
    E, P = len(counts), int(sum(counts))
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ids = ids[torch.randperm(P, generator=torch.Generator().manual_seed(P))].to(torch.int32).cuda()
    mk = lambda n: torch.full((n,), -7, dtype=torch.int32, device="cuda")
    bufs = [mk(P + E * bm), mk((P + E * bm) // 32 + 1), mk(E), mk(E + 1), mk(E + 1), mk(4096 * E)]
    out = mk(2 * E + 21 + 16)
    plan = ItemPlan(out.data_ptr(), tall, nt1, nt2, any1, any2, bn2, *slots)
    f = getattr(lib(), LAUNCH_ALIGN)
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int] + [ctypes.c_void_p] * 7 + \
        [ctypes.c_int, ctypes.c_void_p]
    rc = f(ids.data_ptr(), P, E, bm, *[b.data_ptr() for b in bufs], torch.cuda.current_stream().cuda_stream, 0,
           ctypes.addressof(plan))
    torch.cuda.synchronize()
    assert rc == 0
    assert bufs[2].tolist() == list(counts)
    o = out.cpu().numpy()
    assert (o[2 * E + 21:] == -7).all()
    return o[:E + 1], o[E + 1:2 * E + 2], o[2 * E + 2:2 * E + 11], o[2 * E + 11:2 * E + 20], int(o[2 * E + 20])


def _check(counts, tall, nt1, nt2, any1, any2, bn2):
    E, P = len(counts), int(sum(counts))
    slots = both_slots(P, E, tall, nt1, nt2, any1, any2, bn2)
    i1, i2, xb1, xb2, bn = _plan(counts, tall, nt1, nt2, any1, any2, bn2, slots)
    chosen = []
    for istart, xb, heights, nts, room in (
            (i1, xb1, [tall] + SHORTER * any1, {128: nt1}, slots[0]),
            (i2, xb2, [tall] + SHORTER * any2, {w: nt2 * 128 // w for w in (128, 256) if bn2 in (0, w)}, slots[1])):
        w = bn if istart is i2 else 128
        assert w in nts
        match = [h for h in heights if (np.diff(istart) == [-(-n // h) for n in counts]).all()]
        assert istart[0] == 0 and match, (counts, istart)
        total = int(istart[E]) * nts[w]
        assert xb[0] == 0 and xb[8] == total and (np.diff(xb) >= 0).all()
        assert np.diff(xb).max() <= room
        # what fits, and what a cut that rounds one item further would still let fit
        est = {(h, v): [t * (HALF_TILE if v == 128 and istart is i2 else 1.0) for k, t in cuts(counts, h, n) if k.max() < room]
               for h in heights for v, n in nts.items()}
        mine = min([t for h in match for k, t in cuts(counts, h, nts[w]) if k.max() <= room + 1]) * \
            (HALF_TILE if w == 128 and istart is i2 else 1.0)
        assert mine <= min([t for e in est.values() for t in e] or [np.inf]) * 1.02 + 1, (est, match, w)
        chosen.append((match, w))
    return chosen


@pytest.mark.parametrize("E", [1, 2, 7, 24, 25, 64, 65, 200, 768, 1024])
@pytest.mark.parametrize("tall", [256, 288])
def test_plan_over_expert_counts(E, tall):
    """E from one to the most: the plan's LDS beside the histograms (E below
    25) and over them, 16 waves (E up to 768) and 8, one workgroup and many."""
    rng = np.random.default_rng(E)
    for k in range(3):
        n = rng.integers(0, 400, E) if k == 0 else (rng.zipf(1.5, E) * 20).clip(0, 3000) if k == 1 else np.zeros(E, int)
        n[rng.integers(0, E)] += 1
        _check([int(v) for v in n], tall, 16, 56, True, True, 0)
        _check([int(v) for v in n], tall, 3, 7, False, True, 128)
        _check([int(v) for v in n], tall, 11, 2, True, False, 256)


def test_plan_follows_the_routing():
    """Experts of like counts that fill one round keep the tallest items; one
    popular expert among them makes both stages take shorter ones."""
    even = [256] * 16
    assert all(288 in m and 128 not in m for m, _ in _check(even, 288, 16, 32, True, True, 0))
    zipf = [1120, 610, 380, 250, 160, 110, 80, 70, 60, 40, 35, 30, 20, 15, 12, 8]
    assert all(288 not in m for m, _ in _check(zipf, 288, 16, 32, True, True, 0))
    # few items: a launch that leaves CUs idle takes 128 rows and 128 features
    assert _check([1024] * 2, 288, 4, 8, True, True, 0) == [([128], 128)] * 2
