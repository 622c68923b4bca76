"""The streaming launches and the fused parameter step on tensors that start at any element and end inside a group of
four or eight: the same bits as the same tensors at an aligned address, and nothing written around them."""
import pytest
import torch

from oracle import muon_oracle as O

pytestmark = pytest.mark.gpu

GUARD = 64


def _placed(values, offset):
    """-> (buffer, view of it that holds `values` at an address `offset` elements off 16 bytes)"""
    buf = torch.full((values.numel() + offset + 2 * GUARD,), 7.0, dtype=values.dtype, device="cuda")
    view = buf[GUARD + offset:GUARD + offset + values.numel()].view(values.shape)
    view.copy_(values)
    return buf, view


def _guards_intact(buf, view, offset):
    return bool((buf[:GUARD + offset] == 7).all() and (buf[GUARD + offset + view.numel():] == 7).all())


def _muon_step(shape, dtype, offset, mutate):
    import muon_amd
    gen = torch.Generator(device="cuda").manual_seed(sum(shape))
    draw = lambda std: torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)
    placed = [_placed(t, offset) for t in (draw(0.02), draw(1e-3), draw(3e-4))]
    (_, p), (_, g), (_, m) = placed
    q = torch.nn.Parameter(p)
    q.grad = g
    before = m.clone(), g.clone()
    opt = muon_amd.SingleDeviceMuon([q], lr=0.02, weight_decay=0.01, mutate_grad=mutate)
    opt.state[q]["momentum_buffer"] = m
    opt.step()
    assert all(_guards_intact(buf, view, offset) for buf, view in placed)
    return q.detach().clone(), m.clone(), g.clone(), before


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(300, 333), (333, 300), (131, 1501), (1102, 257), (3, 151, 201), (256, 1024)])
def test_muon_step_at_any_address(shape, dtype, monkeypatch):
    from muon_amd import plan
    monkeypatch.setattr(plan, "SMALL", False)
    mutate = shape[0] != 300
    p0, m0, g0, (m_in, g_in) = _muon_step(shape, dtype, 0, mutate)
    # lerp: one product, one sum; a contraction may leave out the rounding between them
    eps = 2.0 ** (-23 if dtype == torch.float32 else -7)
    want = m_in.double() + (g_in.double() - m_in.double()) * (1 - 0.95)
    assert ((m0.double() - want).abs() <= 2 * eps * (m_in.double().abs() + g_in.double().abs())).all()
    assert torch.equal(g0, g_in) != mutate
    for offset in (1, 2, 3):
        p, m, g, _ = _muon_step(shape, dtype, offset, mutate)
        assert torch.equal(p, p0) and torch.equal(m, m0) and torch.equal(g, g0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("numel", [1, 2, 3, 5, 768, 1021, 1024, 8191, 8192, 8193, 9217, 16387])
def test_adam_at_any_address(numel, dtype):
    import muon_amd
    gen = torch.Generator(device="cuda").manual_seed(numel)
    draw = lambda std: torch.empty(numel, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)
    g, m, v = draw(1e-3), draw(3e-4), draw(1e-3).square()
    first = None
    for offset in (0, 1, 2, 3):
        placed = [_placed(t, offset) for t in (g, m, v)]
        got = [muon_amd.adam_update(*(view for _, view in placed), 100, (0.9, 0.95), 1e-10).clone()]
        got += [view.clone() for _, view in placed]
        assert all(_guards_intact(buf, view, offset) for buf, view in placed)
        first = first or got
        assert all(torch.equal(a, b) for a, b in zip(got, first))
    if dtype == torch.float32:
        mc, vc = m.cpu().clone(), v.cpu().clone()
        want = O.adam_update(g.cpu(), mc, vc, 100, (0.9, 0.95), 1e-10)
        for a, b in zip(first, (want, g.cpu(), mc, vc)):
            assert torch.allclose(a.cpu(), b, rtol=1e-5, atol=1e-8)
