"""The normalise launch alone (a run without iterations): rows that start at any 2-byte address, tiles and chunks
cut by the edge of the matrix, both orientations, and norms out of the range of the short division."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _normalised(G):
    import muon_amd
    return muon_amd.zeropower_via_newtonschulz5(G, steps=0)


@pytest.mark.parametrize("cols", [128, 129, 1100, 1101, 1102, 1104])
@pytest.mark.parametrize("rows", [1, 127, 300, 1500])
def test_normalise_divides_as_the_specification(rows, cols, monkeypatch):
    from muon_amd import plan
    monkeypatch.setattr(plan, "SMALL", False)
    torch.manual_seed(rows + cols)
    G = torch.randn(rows, cols, device="cuda")
    X = G.bfloat16()
    norm = X.double().norm().to(torch.bfloat16)         # the kernel's fp32 sum may land on a neighbouring bf16 value
    step = torch.tensor([0, 1, -1], dtype=torch.int16, device="cuda")
    candidates = [(norm.view(torch.int16) + s).view(torch.bfloat16) + 1e-7 for s in step]
    got = _normalised(G)
    assert any(torch.equal(got, X / c) for c in candidates)


@pytest.mark.parametrize("shape", [(200, 330), (330, 200)])
def test_normalise_beyond_the_range_of_the_short_division(shape, monkeypatch):
    from muon_amd import plan
    monkeypatch.setattr(plan, "SMALL", False)
    torch.manual_seed(1)
    G = torch.randn(*shape, device="cuda")
    tiny = (G * 1e-30).bfloat16()                       # the squares underflow: the denominator is epsilon
    assert torch.equal(_normalised(tiny), tiny / torch.tensor(1e-7, device="cuda").bfloat16())
    assert (_normalised(G * 1e30) == 0).all()           # the squares overflow: every element over infinity
    assert (_normalised(torch.zeros_like(G)) == 0).all()
    G[3, 5] = float("nan")
    assert _normalised(G).isnan().all()


@pytest.mark.parametrize("shapes", [[(1, 9)], [(130, 700)], [(1000, 520), (520, 1000), (128, 8192)]])
def test_norms_formed_in_the_normalise_launch(shapes, monkeypatch):
    """Norms from the normalise launch itself and from a launch of their own: the same bits (one to 64 partial sums;
    128 x 8192 has a split reduction, whose counters either launch clears)."""
    import muon_amd
    from muon_amd import plan
    monkeypatch.setattr(plan, "SMALL", False)
    results = []
    for blocks in ((0, 0), (512, 4096)):
        monkeypatch.setattr(plan, "NORM_IN_NORMALIZE_BLOCKS", blocks)
        torch.manual_seed(3)
        params = [torch.nn.Parameter(torch.randn(*s, device="cuda")) for s in shapes]
        opt = muon_amd.SingleDeviceMuon(params, lr=0.02)
        for _ in range(2):
            for p in params:
                p.grad = torch.randn_like(p)
            opt.step()
        results.append([p.detach().clone() for p in params])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("small", [True, False])
@pytest.mark.parametrize("transposed", [False, True])
def test_elements_too_small_for_the_short_division(small, transposed, monkeypatch):
    """Every bf16 value below 2^-60, zeros of either sign among them, over fp32 denominators: the bits of the ordinary
    division.  One element per matrix makes the norm, exactly; the squares of the others vanish beside its own."""
    import muon_amd
    from muon_amd import plan
    monkeypatch.setattr(plan, "SMALL", small)
    muon_amd.clear_engine_cache()
    bits = torch.arange((127 - 60) << 7, dtype=torch.int32)
    values = torch.cat([bits, bits | 0x8000]).to(torch.int16).view(torch.bfloat16)
    rows, cols = 68, 256
    assert values.numel() <= rows * cols - 1 < values.numel() + cols
    # 0.25 .. some hundreds, and two norms for which the short division of such values misses the bf16 result
    for norm in [0x3E80 + 37 * k for k in range(24)] + [0x38E3, 0x3ABC]:
        top = torch.tensor([norm], dtype=torch.int16).view(torch.bfloat16)
        x = torch.zeros(rows * cols, dtype=torch.bfloat16)
        x[:values.numel()] = values
        x[-1] = top
        x = x.view(rows, cols)
        x = x.T.contiguous() if transposed else x
        got = muon_amd.zeropower_via_newtonschulz5(x.cuda(), steps=0, rounding="fused").cpu()
        want = (x.float() / (top.float() + 1e-7)).bfloat16()
        differ = got.view(torch.int16) != want.view(torch.int16)
        assert not differ.any(), (float(top), int(differ.sum()), x[differ][:4], got[differ][:4], want[differ][:4])
    muon_amd.clear_engine_cache()
