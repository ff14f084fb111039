"""Routed experts of large steps (GPU): rows sorted without padding and gathered by the 256 x 256 tiles,
the sort's one and 64 workgroups, and the logits of four rows at a time, against the same ops on
CPU tensors."""
import pytest
import torch

from aws_k8s_ansible_provisioner_amd import ops
from aws_k8s_ansible_provisioner_amd.ops import reference as ref
from aws_k8s_ansible_provisioner_amd.ops import stream as sops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,E,block", [(1, 1, 1), (63, 3, 64), (8191, 8, 1), (8192, 8, 1),
                                       (8300, 32, 64), (20011, 5, 1), (70001, 17, 32),
                                       (8192, 1, 1), (12001, 4, 64), (70001, 2, 1)])
def test_align(n, E, block):
    """Every id in its expert's segment, from 8192 ids on in order; ids that name no expert skipped."""
    g = torch.Generator().manual_seed(n)
    ids = torch.randint(-1, E + 1, (n,), generator=g, dtype=torch.int32)
    cap = ops.moe_capacity(n, E, block)
    inv = torch.empty(n, dtype=torch.int32, device=DEV)
    tiles = torch.empty(cap // block, dtype=torch.int32, device=DEV)
    s, offs, total = ops.moe_align(ids.to(DEV), E, block, inv=inv, tile_expert=tiles)
    s, offs, inv, tiles = s.cpu(), offs.cpu(), inv.cpu(), tiles.cpu()
    at = 0
    for e in range(E):
        want = (ids == e).nonzero().flatten().int()
        end = at + -(-len(want) // block) * block
        assert int(offs[e]) == at
        got = s[at:at + len(want)]
        assert torch.equal(inv[got.long()], torch.arange(at, at + len(want), dtype=torch.int32))
        assert torch.equal(got if n >= 8192 else got.sort().values, want)
        assert bool((s[at + len(want):end] == n).all())
        assert bool((tiles[at // block:end // block] == e).all())
        at = end
    assert int(offs[E]) == at == int(total)
    assert bool((tiles[at // block:] == -1).all())
    assert bool((inv[(ids < 0) | (ids >= E)] == -1).all())


@pytest.mark.parametrize("T,d,F,pad", [(1024, 256, 128, 0), (1500, 512, 384, 8)])
def test_large_steps(T, d, F, pad):
    """One expert without rows, one with few, rows of a wider tensor.  Both sides round the gated
    units to bf16 (2^-9 relative) and sum the rest in fp32: as the smaller tiles' test."""
    g = torch.Generator().manual_seed(T)
    E = 8
    h = torch.randn(T, d + pad, generator=g).bfloat16()
    w13 = (torch.randn(E, 2 * F, d, generator=g) * d ** -0.5).bfloat16()
    w2 = (torch.randn(E, d, F, generator=g) * F ** -0.5).bfloat16()
    ids = torch.stack([torch.randperm(6, generator=g)[:2] for _ in range(T)]).int()
    ids[:3, 0] = 6
    w = torch.rand(T, 2, generator=g)
    hd = h.to(DEV)[:, :d]
    assert ops._moe_large(2 * T, E, hd, w13, w2)
    out = ops.fused_moe(hd, w13.to(DEV), w2.to(DEV), w.to(DEV), ids.to(DEV)).float().cpu()
    exp = ref.fused_moe(h[:, :d].contiguous(), w13, w2, w, ids).float()
    assert bool(((out - exp).abs() <= 3e-2 + 3e-2 * exp.abs()).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,d,n,top", [(1023, 256, 8, 2), (1024, 260, 9, 3), (1025, 1000, 3, 1),
                                       (2559, 512, 8, 2), (2561, 516, 17, 4), (2563, 4, 2, 1),
                                       (2560, 768, 40, 8)])
def test_routing(T, d, n, top, dt):
    """Sums of d products in fp32 on both sides: logits within d 2^-24 of the products' sum of
    magnitudes; the winners agree where the logits differ by more."""
    g = torch.Generator().manual_seed(T + n)
    h = torch.randn(T, d, generator=g).to(dt)
    r, b = torch.randn(n, d, generator=g) * d ** -0.5, torch.randn(n, generator=g)
    z = h.double() @ r.double().T + b.double()
    ids, w = sops.route_topk(h.to(DEV), r.to(DEV), b.to(DEV), top)
    ids, w = ids.cpu().long(), w.cpu()
    tol = d * 2.0 ** -24 * float((h.double().abs() @ r.double().abs().T).max())
    val = z.topk(top, dim=-1).values
    assert float((z.gather(1, ids) - val).abs().max()) <= 2 * tol
    assert float((w - torch.softmax(val, -1)).abs().max()) <= 4 * tol + 1e-6
    few = sops.route_topk(h[:100].to(DEV), r.to(DEV), b.to(DEV), top)      # a row at a time: same sums
    assert torch.equal(few[0].cpu().long(), ids[:100]) and torch.equal(few[1].cpu(), w[:100])


@pytest.mark.parametrize("n,E,run", [(8192, 32, 1), (9000, 8, 64), (16500, 3, 4000), (8193, 1, 7),
                                     (70001, 17, 3)])
def test_align_runs(n, E, run):
    """Ids by turns in runs: a counter goes from lane to lane of a wave, or stays with one for long."""
    ids = (torch.arange(n) // run % E).to(torch.int32)
    inv = torch.empty(n, dtype=torch.int32, device=DEV)
    s, offs, total = ops.moe_align(ids.to(DEV), E, 1, inv=inv)
    order = ids.sort(stable=True).indices.to(torch.int32)
    assert int(total) == n and torch.equal(s.cpu()[:n], order)
    assert torch.equal(inv.cpu()[order.long()], torch.arange(n, dtype=torch.int32))
    assert torch.equal(offs.cpu(), torch.tensor([0] + torch.bincount(ids, minlength=E).cumsum(0).tolist(),
                                                dtype=torch.int32))
