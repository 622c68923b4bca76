"""A launch whose own tiles would leave CUs idle runs in smaller ones; which tiles compute an element must
not change its bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# edges of the 64-, 128- and 256-wide tiles, one and several k-blocks (ring of four), split reductions,
# more jobs than the GPU holds at once, and tall matrices
SHAPES = [(1, 1, 1), (1, 64, 64), (1, 65, 129), (1, 63, 577), (1, 128, 320), (3, 192, 260), (1, 250, 250), (1, 512, 2048),
          (2, 2304, 256), (1, 128, 16384), (1, 1027, 1100), (40, 100, 1000), (1, 1500, 1100)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("rounding", ["reference", "fused"])
def test_tile_class_of_a_launch_does_not_change_the_bits(shape, rounding, monkeypatch):
    import muon_amd
    from muon_amd import plan
    monkeypatch.setattr(plan, "SMALL", False)
    torch.manual_seed(sum(shape))
    G = torch.randn(*shape, device="cuda")
    outs, classes = [], []
    for forced in ("1,1,1", "0,0,0", "2,2,2", "2,0,2", "0,2,0"):
        monkeypatch.setattr(plan, "LAUNCH_CLASS", forced)
        muon_amd.functional.clear_engine_cache()
        outs.append(muon_amd.zeropower_via_newtonschulz5(G, rounding=rounding))
        eng = next(iter(muon_amd.functional._ENGINE_CACHE.values()))
        classes.append(tuple(eng.chunks[0].launches[k].tile_class for k in ("gram", "poly", "update")))
    muon_amd.functional.clear_engine_cache()
    assert classes[2] == (2, 2, 2) and len(set(classes)) >= 4
    assert torch.isfinite(outs[0].float()).all()
    for other in outs[1:]:
        assert torch.equal(outs[0], other)


def test_fused_parameter_step_in_small_tiles_gives_the_bits_of_large_ones(monkeypatch):
    import muon_amd
    from muon_amd import plan
    monkeypatch.setattr(plan, "SMALL", False)
    shapes = [(70, 200), (200, 70), (64, 64), (33, 500), (300, 257)]
    results = []
    for forced in ("0,0,0", "2,2,2"):
        monkeypatch.setattr(plan, "LAUNCH_CLASS", forced)
        torch.manual_seed(3)
        ps = [torch.nn.Parameter(torch.randn(*s, device="cuda", dtype=dt)) for s in shapes for dt in (torch.float32,)]
        ps += [torch.nn.Parameter(torch.randn(*s, device="cuda", dtype=torch.bfloat16)) for s in shapes]
        for p in ps:
            p.grad = torch.randn_like(p)
        opt = muon_amd.SingleDeviceMuon(ps, weight_decay=0.1)
        for _ in range(2):
            opt.step()
        results.append([p.detach().clone() for p in ps])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("rescale", ["symmetric", "rows"])
@pytest.mark.parametrize("shape", [(1, 40, 65), (3, 65, 129), (1, 128, 320), (2, 250, 250), (2, 600, 130), (1, 1027, 1100), (1, 1100, 1500)])
def test_tile_classes_mixed_in_the_aol_variant(shape, rescale, monkeypatch):
    """Its first X X^T, which leaves the row sums, keeps the matrix's own class while the others take smaller tiles, over
    buffers whose padding holds NaNs (nothing of it may reach a result)."""
    import muon_amd
    from muon_amd import plan
    torch.manual_seed(sum(shape))
    G = torch.randn(*shape, device="cuda")
    outs = []
    for forced in ("1,1,1", "0,0,0", "2,2,2", "2,0,2", "0,2,0"):
        monkeypatch.setattr(plan, "LAUNCH_CLASS", forced)
        muon_amd.clear_engine_cache()
        muon_amd.zeropower_via_aol4(G, rescale=rescale)
        eng = next(iter(muon_amd.functional._ENGINE_CACHE.values()))
        assert eng.chunks[0].launches["gram_rowsum"].tile_class == eng.chunks[0].tile_class
        assert forced != "2,2,2" or {eng.chunks[0].launches[k].tile_class for k in ("gram", "poly", "update")} == {2}
        for ws in eng.workspaces:
            ws.fill_(0xff)
        outs.append(muon_amd.zeropower_via_aol4(G, rescale=rescale))
    muon_amd.clear_engine_cache()
    assert torch.isfinite(outs[0].float()).all()
    for other in outs[1:]:
        assert torch.equal(outs[0], other)
