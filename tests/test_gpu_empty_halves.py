"""256 x 256 tiles at the edge of a matrix leave out the half that lies in the padding; that must not change a bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# one to four k-blocks (the ring holds two and a half) and more, data ending at, just before and just behind the middle of a
# tile in rows, columns or both, tall and wide, several matrices
SHAPES = [(1, 1, 1), (1, 60, 100), (1, 100, 128), (1, 127, 129), (1, 128, 384), (2, 129, 190), (1, 320, 256), (3, 200, 260),
          (1, 385, 640), (2, 1025, 1152), (1, 1153, 1090), (1, 1280, 1300), (40, 300, 400)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("variant", ["reference", "fused", "aol4", "step"])
def test_empty_halves_are_products_of_zero(shape, variant, monkeypatch):
    import muon_amd
    from muon_amd import plan
    monkeypatch.setattr(plan, "SMALL", False)
    monkeypatch.setattr(plan, "BIG_TILE_MIN_M", 1)
    monkeypatch.setattr(plan, "LAUNCH_CLASS", "1,1,1")
    torch.manual_seed(sum(shape))
    G = torch.randn(*shape, device="cuda")
    outs = []
    for skip in (False, True):
        monkeypatch.setattr(plan, "SKIP_EMPTY", skip)
        muon_amd.clear_engine_cache()
        if variant == "step":
            ps = [torch.nn.Parameter(g.clone()) for g in G]
            for p, g in zip(ps, G):
                p.grad = g.flip(0)
            opt = muon_amd.SingleDeviceMuon(ps, weight_decay=0.1)
            opt.step()
            opt.step()
            outs.append(torch.stack([p.detach() for p in ps]))
        elif variant == "aol4":
            outs.append(muon_amd.zeropower_via_aol4(G))
        else:
            outs.append(muon_amd.zeropower_via_newtonschulz5(G, rounding=variant))
    muon_amd.clear_engine_cache()
    assert torch.isfinite(outs[0].float()).all()
    assert torch.equal(*outs)


# the rows-only rescaling multiplies the polynomial over every tile, stored in one orientation; the long shapes would be split
# (their X X^T) in the class that their sizes ask for
ROWS_SHAPES = [s for s in SHAPES if min(s[1:]) >= 32] + [(1, 300, 4096), (2, 4160, 260)]


@pytest.mark.parametrize("shape", ROWS_SHAPES)
def test_empty_halves_of_the_unmirrored_polynomial(shape, monkeypatch):
    import muon_amd
    from muon_amd import plan
    monkeypatch.setattr(plan, "SMALL", False)
    monkeypatch.setattr(plan, "BIG_TILE_MIN_M", 1)
    monkeypatch.setattr(plan, "LAUNCH_CLASS", "1,1,1")
    torch.manual_seed(sum(shape))
    G = torch.randn(*shape, device="cuda")
    outs = []
    for skip in (False, True):
        monkeypatch.setattr(plan, "SKIP_EMPTY", skip)
        muon_amd.clear_engine_cache()
        outs.append(muon_amd.zeropower_via_aol4(G, rescale="rows"))
    muon_amd.clear_engine_cache()
    assert torch.isfinite(outs[0].float()).all()
    assert torch.equal(*outs)
