"""GPU parity of absorbed rows: an fp16 wide item of more than 256 rows takes up
to 32 of them along as extra token rows of its 256-row tile (grouped_gemm.hip
Ring, ABS).  Row counts straddle the tile: 257 to 288 rows are one item with 1
to 32 absorbed rows, 545 two (288 and 257), 576 two with 32 each, 256 and fewer
none.  The shapes are ones where the plan takes 288-row items in both stages
(asserted against the restated rule), with 256 features in Stage 2 (H 2048) and
128 (H 1152, no multiple of 256).  Every output is compared whole with the
oracle, from a NaN-poisoned buffer."""
import numpy as np
import pytest
import torch

from _cases import exact_routing_inputs
from _plan import chosen
from conftest import assert_close
from oracle import fused_moe_forward

pytestmark = pytest.mark.gpu

# per-expert routed rows
COUNTS = [257, 288, 545, 576, 270, 287, 256, 1, 0, 33, 160, 161, 257, 280, 288, 265, 284, 272, 288, 260, 259, 287]
I = 1024
SHAPES = [(2048, 256), (1152, 128)]  # H, Stage 2's features per item


def _inputs(k, seed, counts=COUNTS, H=2048, I=I):
    return exact_routing_inputs(k, seed, counts, H, I)


@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("H,bn", SHAPES)
def test_absorbed_rows_full_output(k, H, bn):
    from muxi_race_amd import fused_moe
    assert chosen(COUNTS, H, I, 288) == (288, (288, bn))
    x, logits, wg, wu, wd = _inputs(k, 31 + k, H=H)
    out = torch.full((x.shape[0], H), float("nan"), dtype=torch.float16, device="cuda")
    out = fused_moe(x.cuda(), logits.cuda(), wg.cuda(), wu.cuda(), wd.cuda(), k, out=out)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out).all()), "non-finite values left in the NaN-poisoned output"
    assert_close(out, fused_moe_forward(x, logits, wg, wu, wd, k), what=f"absorbed rows k={k} H={H}")


@pytest.mark.parametrize("E,mean", [(80, 270), (150, 140)])
def test_absorbed_rows_many_experts(E, mean):
    """The expert scans over two and three chunks of 64, top-2, with experts of
    257 to 288 and 513 to 544 rows among shorter ones and empty ones."""
    from muxi_race_amd import fused_moe
    rng = np.random.default_rng(5)
    if mean > 200:
        counts = [int(rng.choice([rng.integers(257, 289), rng.integers(289, 400), rng.integers(513, 545),
                                  rng.integers(100, 256), 0])) for _ in range(E)]
    else:
        counts = [int(rng.choice([0, rng.integers(1, 40), rng.integers(129, 161), rng.integers(161, 257),
                                  rng.integers(257, 289)])) for _ in range(E)]
    counts[-1] += sum(counts) % 2
    x, logits, wg, wu, wd = _inputs(2, 41, counts, 256, 1024)
    assert chosen(counts, 256, 1024, 288)[0] == 288
    out = torch.full((x.shape[0], 256), float("nan"), dtype=torch.float16, device="cuda")
    out = fused_moe(x.cuda(), logits.cuda(), wg.cuda(), wu.cuda(), wd.cuda(), 2, out=out)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out).all()), "non-finite values left in the NaN-poisoned output"
    assert_close(out, fused_moe_forward(x, logits, wg, wu, wd, 2), what=f"absorbed rows E={E}")


def test_absorbed_rows_repeatable():
    """Two calls give bitwise the same output (the items are fixed by the routing
    alone)."""
    from muxi_race_amd import fused_moe
    x, logits, wg, wu, wd = (t.cuda() for t in _inputs(2, seed=40))
    a = fused_moe(x, logits, wg, wu, wd, 2)
    b = fused_moe(x, logits, wg, wu, wd, 2)
    torch.cuda.synchronize()
    assert torch.equal(a, b)


@pytest.mark.parametrize("H", [2048, 1152])
def test_absorbed_rows_prerouted_padding_zero(H):
    """run_kernel on 32 experts, enough to take 288-row items (more than 112 rows
    on average, more than a quarter of them taller than a block, 256 Stage 1
    items), in both of Stage 2's widths.  The padding rows behind the absorbed
    ones must come back exactly 0 from a NaN-poisoned output, with NaN in x's
    padding rows (problem_detail.json:50 note 4)."""
    from _cases import prerouted_inputs
    from muxi_race_amd import run_kernel
    from oracle import prerouted_forward
    sizes = COUNTS + [257, 288, 3, 0, 385, 130, 160, 289, 513, 12]
    blocks = sum(-(-n // 128) for n in sizes)
    assert len(sizes) == 32 and sum(sizes) > 112 * 32 and 4 * (blocks - 32) > 32
    args = list(prerouted_inputs(sizes, H, I, seed=77))
    x, gpo = args[0], args[7].cpu().tolist()
    pad = torch.ones(x.shape[0], dtype=torch.bool)
    for e, n in enumerate(sizes):
        pad[gpo[e]:gpo[e] + n] = False
    x[pad.to(x.device)] = float("nan")
    out = torch.full(x.shape, float("nan"), dtype=torch.float16, device=x.device)
    run_kernel(*args, out)
    torch.cuda.synchronize()
    assert_close(out, prerouted_forward(*args), what="prerouted absorbed rows")
    assert (out[pad.to(out.device)] == 0).all()


@pytest.mark.parametrize("bm", [0, 128])
def test_last_blocks_beyond_absorption(bm):
    """Row counts past what one tall item takes, split over two or more: 424, 572,
    562, 296, 600 and others, top-1, with the library's padding and 128 rows;
    pre-routed too, with NaN-poisoned padding."""
    from muxi_race_amd import fused_moe
    counts = [424, 572, 562, 296, 600, 250, 0, 31, 200]
    H = I = 256
    x, logits, wg, wu, wd = _inputs(1, 44, counts, H, I)
    T = x.shape[0]
    out = torch.full((T, H), float("nan"), dtype=torch.float16, device="cuda")
    out = fused_moe(x.cuda(), logits.cuda(), wg.cuda(), wu.cuda(), wd.cuda(), 1, block_m=bm, out=out)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out).all()), "non-finite values left in the NaN-poisoned output"
    assert_close(out, fused_moe_forward(x, logits, wg, wu, wd, 1), what=f"rows past a tall item bm={bm}")
    if bm == 128:
        from _cases import prerouted_inputs
        from muxi_race_amd import run_kernel
        from oracle import prerouted_forward
        sizes = [424, 572, 296, 3, 0, 562]
        args = list(prerouted_inputs(sizes, 512, 256, seed=45))
        xp, gpo = args[0], args[7].cpu().tolist()
        pad = torch.ones(xp.shape[0], dtype=torch.bool)
        for e, n in enumerate(sizes):
            pad[gpo[e]:gpo[e] + n] = False
        xp[pad.to(xp.device)] = float("nan")
        o = torch.full(xp.shape, float("nan"), dtype=torch.float16, device=xp.device)
        run_kernel(*args, o)
        torch.cuda.synchronize()
        assert_close(o, prerouted_forward(*args), what="prerouted rows past a tall item")
        assert (o[pad.to(o.device)] == 0).all()
