"""Which items a fused call with block_m = 0 runs, read off its bits: fp16
32-row items sum two halves of K, wide ones the whole of it, so the call equals
either block_m = 32 or block_m = 64 and the other differs.  The line lies where
the expected 32-row blocks over the experts held here take about one item per
CU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(T, E, held, k, I):
    g = torch.Generator(device="cuda").manual_seed(T + E)
    mk = lambda *sh: torch.randn(sh, generator=g, device="cuda")
    x, lg = mk(T, 1024).half(), mk(T, E)
    return x, lg, [(mk(*sh) * 0.05).half() for sh in ((held, I, 1024), (held, I, 1024), (held, 1024, I))]


# (tokens, experts routed over, held, k, I, narrow): 200 pairs of a block and a
# tile are 8 experts of 84 rows at I 1024, of 184 at I 512
@pytest.mark.parametrize("T,E,held,k,I,narrow", [
    (336, 8, 8, 2, 1024, True), (400, 8, 8, 2, 1024, False), (512, 8, 8, 2, 1024, False),
    (736, 8, 8, 2, 512, True), (800, 8, 8, 2, 512, False),
    (96, 8, 8, 2, 2048, True), (128, 8, 8, 2, 2048, True), (160, 8, 8, 2, 2048, False),
    # an expert shard counts the experts that it holds: 4 of 64 at 100 rows
    (3200, 64, 4, 2, 512, True), (3200, 64, 64, 2, 512, False), (8000, 64, 4, 2, 512, True), (16000, 64, 4, 2, 512, False),
])
def test_library_picks(T, E, held, k, I, narrow):
    from muxi_race_amd import fused_moe
    x, lg, w = _case(T, E, held, k, I)
    more = {} if held == E else dict(expert_range=(8, held))
    got, n, wide = (fused_moe(x, lg, *w, k, block_m=bm, **more) for bm in (0, 32, 64))
    torch.cuda.synchronize()
    assert not torch.equal(n, wide), "the sums do not tell the items apart"
    assert torch.equal(got, n if narrow else wide)


@pytest.mark.parametrize("T,E,held,k,I,narrow", [(800, 64, 4, 2, 512, False), (600, 64, 4, 2, 512, True)])
def test_library_picks_for_dispatched_tokens(T, E, held, k, I, narrow):
    """Each token has a choice here, so the experts held here get more rows than
    the average over all (25 of 800 tokens, above the line; 200 here), and the
    workspace that the size function asks for holds the wide items."""
    from muxi_race_amd import fused_moe_routed
    x, lg, w = _case(T, E, held, k, I)
    ids = torch.stack([8 + torch.arange(T) % held, torch.full((T,), 40)], 1).int().cuda()
    wts = torch.softmax(lg[:, :k], 1).contiguous()
    got, n, wide = (fused_moe_routed(x, ids, wts, *w, expert_begin=8, num_experts=E, block_m=bm) for bm in (0, 32, 64))
    torch.cuda.synchronize()
    assert not torch.equal(n, wide), "the sums do not tell the items apart"
    assert torch.equal(got, n if narrow else wide)


@pytest.mark.parametrize("bm", [32, 64, 128])
def test_workspace_sized_without_block_m_serves_explicit_blocks(bm):
    """A C caller's workspace sized with block_m = 0 also holds the call with
    an explicit block_m up to the one that the rows per expert suggest."""
    from muxi_race_amd._lib import lib
    L = lib()
    T, H, I, E, k = 400, 1024, 512, 8, 2   # 100 rows per expert: moe_pick_block_m says 128
    assert L.moe_pick_block_m(T, E, k) == 128
    x, lg, w = _case(T, E, E, k, I)
    outs = []
    for b in (bm, 0):
        ws = torch.empty(L.moe_fused_workspace_bytes(T, H, I, E, k, 0, 0), dtype=torch.uint8, device="cuda")
        out = torch.full((T, H), float("nan"), dtype=torch.float16, device="cuda")
        rc = L.moe_fused_forward(x.data_ptr(), lg.data_ptr(), None, *(m.data_ptr() for m in w), out.data_ptr(), T, H, I, E,
                                 k, b, ws.data_ptr(), ws.numel(), None, None, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, L.moe_last_error_string()
        torch.cuda.synchronize()
        outs.append(out.float())
    # K sums in another order: one fp16 rounding of h and of the output each
    assert torch.isfinite(outs[0]).all()
    assert float((outs[0] - outs[1]).norm() / outs[1].norm()) < 2e-3
