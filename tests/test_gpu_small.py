"""The whole step of a small matrix in one workgroup: the bits of the separate launches, at the edges of its
classes (short side 32, 64, 128), of a k-block (64), of a block of the sum of squares (8192 elements)
and of what fits LDS."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (1, 7), (5, 3), (31, 65), (32, 2304), (33, 33), (64, 64), (64, 576), (1024, 64), (65, 320), (127, 127),
          (128, 64), (320, 128), (128, 257), (2000, 16), (48, 171), (128, 320)]


def _engine(rows, cols):
    from muon_amd import functional
    return [e for k, e in functional._ENGINE_CACHE.items() if k[2:4] == (rows, cols)][0]


@pytest.mark.parametrize("rounding", ["reference", "fused"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_small_step_gives_the_bits_of_the_general_path(rounding, dtype, monkeypatch):
    import muon_amd
    from muon_amd import plan
    for rows, cols in SHAPES:
        for batch, steps in ((1, 5), (3, 5), (1, 0), (1, 2)):
            torch.manual_seed(rows * 1000 + cols)
            g0 = torch.randn(batch, rows, cols, device="cuda").to(dtype)
            m0 = (torch.randn(batch, rows, cols, device="cuda") * 0.3).to(dtype)
            got = []
            for small in (True, False):
                monkeypatch.setattr(plan, "SMALL", small)
                muon_amd.clear_engine_cache()
                g, m = g0.clone(), m0.clone()
                up = muon_amd.muon_update(g, m, ns_steps=steps, rounding=rounding)
                assert bool(_engine(rows, cols).small) == small, (rows, cols)
                got.append((up, g, m, muon_amd.zeropower_via_newtonschulz5(g0, steps=steps, rounding=rounding)))
            for a, b in zip(*got):
                assert torch.equal(a, b), (rows, cols, batch, steps)
    muon_amd.clear_engine_cache()


def test_optimizer_over_small_matrices_matches_the_general_path_eagerly_and_replayed(monkeypatch):
    """Parameters off the 16-byte grid, several classes in one group, decay, a changing learning rate."""
    import muon_amd
    from muon_amd import plan
    shapes = [(64, 64, 3, 3), (10, 64), (128, 300), (3, 5), (300, 100)]
    finals = []
    for small, graph in ((True, False), (True, True), (False, False)):
        monkeypatch.setattr(plan, "SMALL", small)
        torch.manual_seed(5)
        flat = torch.randn(3 + sum(torch.Size(s).numel() for s in shapes), device="cuda")
        off, ps = 3, []
        for s in shapes:
            n = torch.Size(s).numel()
            ps.append(torch.nn.Parameter(flat[off:off + n].view(s)))
            off += n
        opt = muon_amd.SingleDeviceMuon(ps, weight_decay=0.1, use_graph=graph)
        for step in range(4):
            for p in ps:
                p.grad = torch.randn_like(p)
            opt.param_groups[0]["lr"] = 0.02 / (step + 1)
            opt.step()
        eng = next(iter(opt._muon_engines.values()))
        assert bool(eng.small) == small
        finals.append([p.detach().clone() for p in ps] + [opt.state[p]["momentum_buffer"].clone() for p in ps])
    for other in finals[1:]:
        assert all(torch.equal(a, b) for a, b in zip(finals[0], other))


def test_what_does_not_fit_one_workgroup_takes_the_general_path():
    from muon_amd import _lib, plan
    lib = _lib.load()
    assert [lib.muon_amd_small_class(*s) for s in ((129, 129), (128, 321), (64, 1089), (32, 5000), (1, 200000))] == [0] * 5
    assert [lib.muon_amd_small_class(*s) for s in ((128, 320), (320, 128), (64, 1088), (20, 2000))] == [128, 128, 64, 32]
    assert plan.small_groups([(64, 64), (256, 256)]) is None and plan.small_groups([(64, 64)], "aol4") is None


@pytest.mark.parametrize("rounding", ["reference", "fused"])
@pytest.mark.parametrize("steps", [1, 2, 5])
def test_small_step_gives_the_signs_of_zeros_of_the_general_path(rounding, steps, monkeypatch):
    """Terms that round to negative zeros: rows that are orthogonal up to products near the smallest bf16 value, and
    elements that are negative zeros themselves.  Compared as bit patterns."""
    import muon_amd
    from muon_amd import plan
    torch.manual_seed(11)
    G = torch.zeros(200, 8, 40)
    sign = torch.randint(0, 2, G.shape) * 2.0 - 1
    G = torch.where(torch.rand(G.shape) < 0.3, 10.0 ** (torch.rand(G.shape) * 24 - 44), G) * sign     # signed zeros among them
    G[:, torch.arange(8), torch.arange(8)] = 1.0
    G[:, 1::3, 20:] *= 1e21                              # some factors whose products with those are subnormal
    G = G.cuda()
    got = []
    for small in (True, False):
        monkeypatch.setattr(plan, "SMALL", small)
        muon_amd.clear_engine_cache()
        got.append(muon_amd.zeropower_via_newtonschulz5(G, steps=steps, rounding=rounding).view(torch.int16))
    muon_amd.clear_engine_cache()
    assert (got[1] == -0x8000).any() and (got[1] == 0).any()
    assert torch.equal(*got)


@pytest.mark.parametrize("rounding", ["reference", "fused"])
def test_classes_mixed_in_one_launch_give_the_bits_of_the_general_path(rounding, monkeypatch):
    """Every shape of the list beside the others, the largest of each class among them, in two storage types."""
    import muon_amd
    from muon_amd import plan
    for dtype in (torch.float32, torch.bfloat16):
        finals = []
        for small in (True, False):
            monkeypatch.setattr(plan, "SMALL", small)
            torch.manual_seed(8)
            ps = [torch.nn.Parameter(torch.randn(s, device="cuda").to(dtype)) for s in SHAPES + [(32, 2432), (64, 1088)]]
            opt = muon_amd.SingleDeviceMuon(ps, weight_decay=0.1, ns_rounding=rounding)
            for _ in range(2):
                for p in ps:
                    p.grad = torch.randn(p.shape, device="cuda").to(dtype)
                opt.step()
            eng = next(iter(opt._muon_engines.values()))
            assert [rt.small_class for rt in eng.small] == ([0] if small else [])
            finals.append([p.detach().clone() for p in ps] + [opt.state[p]["momentum_buffer"].clone() for p in ps])
        assert all(torch.equal(a, b) for a, b in zip(*finals))
