"""Head-mixed attention of prompt chunks with keys staged through LDS (GPU) against the same op on CPU
tensors: both head sizes, value sizes that fill one, several and two grid rows of 32-entry tiles (also
with a last wave that has none), chunks that end inside 32-key pieces, 64-key steps and 128-query
tiles, cached tokens before them, pages of 32, 64 and 96 tokens, single rows that lead the step, rows
that are not 16-byte aligned, no mixing and no gate.

Tolerance: weights and outputs are rounded to bf16 (relative 2^-9 each, on either side for the
outputs): the 2-norm of the difference stays under 3 * 2^-9 of the result's; mixing sums up to H heads'
rounded weights, whose errors are independent."""
import pytest
import torch

from aws_k8s_ansible_provisioner_amd.ops import stream as sops

pytestmark = pytest.mark.gpu
DEV, TOL = "cuda", 3 * 2.0 ** -9


@pytest.mark.parametrize("H,G,D,Dv,BS,shape,nd,extra", [
    (4, 2, 64, 64, 32, [(0, 33)], 0, "gate talk"),
    (2, 1, 128, 32, 64, [(0, 128), (5, 1), (64, 129)], 0, "talk"),
    (16, 4, 128, 128, 64, [(70, 131), (0, 64), (191, 300)], 0, "gate talk"),
    (32, 8, 128, 128, 64, [(3, 200), (0, 61)], 0, "gate talk"),
    (6, 3, 64, 96, 96, [(95, 97), (0, 31), (1, 96)], 0, "gate"),
    (9, 3, 64, 160, 32, [(0, 127), (31, 66)], 0, ""),
    (8, 4, 128, 64, 64, [(200, 1), (17, 1), (9, 150)], 2, "gate talk odd"),
])
def test_chunks(H, G, D, Dv, BS, shape, nd, extra):
    g = torch.Generator().manual_seed(H * D + Dv)
    pages = [-(-(p + n) // BS) for p, n in shape]
    NB = sum(pages) + 1
    perm, at = torch.randperm(NB, generator=g), 0
    bt = torch.zeros(len(shape), max(pages), dtype=torch.int32)
    tiles, start = [], [0]
    for b, (p, n) in enumerate(shape):
        bt[b, :pages[b]] = perm[at:at + pages[b]].to(torch.int32)
        at += pages[b]
        start.append(start[-1] + n)
        if b >= nd:
            tiles += [(p + min(n, r + 256), b, r) for r in range(0, n, 256)]
    tiles.sort()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)
    T, pad = start[-1], 3 if "odd" in extra else 0
    pos = torch.cat([torch.arange(p, p + n) for p, n in shape])
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16()
    q, k, v = rnd(T, H, D), rnd(NB, G, BS, D), rnd(NB, G, BS // 8, Dv, 8)
    gate = rnd(T, H * Dv + pad) if "gate" in extra else None
    talk = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g) if "talk" in extra else None
    lens, qs = i32([p + n for p, n in shape]), i32(start)
    ts, tr = i32([t[1] for t in tiles]), i32([t[2] for t in tiles])

    def run(dev):
        m = lambda x: None if x is None else x.to(dev)
        out = torch.zeros(T, H * Dv + pad, dtype=torch.bfloat16, device=dev)
        w = (lambda x: x[:, pad:]) if pad else (lambda x: x)
        sops.talking_attention_prefill(w(out), m(q), m(k), m(v), m(bt), m(lens), m(qs), m(pos),
                                       m(ts), m(tr), 256, m(talk),
                                       w(m(gate)) if gate is not None else None, D ** -0.5, nd)
        return out.float().cpu()

    a, b = run(DEV), run("cpu")
    assert float((a - b).norm() / b.norm()) <= TOL
    assert float((a - b).abs().max()) <= 8 * TOL * float(b.abs().max())


def _two_prompts(g, H=8, G=4, D=128, Dv=64, BS=32):
    """Two sequences, the second continued at an odd position: (arguments, run)."""
    shape = [(0, 200), (77, 150)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16()
    a = dict(q=rnd(350, H, D), k=rnd(16, G, BS, D), v=rnd(16, G, BS // 8, Dv, 8),
             bt=torch.randperm(16, generator=g).view(2, 8).to(torch.int32), lens=i32([200, 227]),
             qs=i32([0, 200, 350]), pos=torch.cat([torch.arange(p, p + n) for p, n in shape]),
             ts=i32([0, 0, 1, 1]), tr=i32([0, 128, 0, 128]))
    talk = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)

    def run(dev):
        out = torch.zeros(350, H * Dv, dtype=torch.bfloat16, device=dev)
        sops.talking_attention_prefill(
            out, *(a[n].to(dev) for n in ("q", "k", "v", "bt", "lens", "qs", "pos", "ts", "tr")), 128,
            talk.to(dev), None, D ** -0.5, 0)
        return out.float().cpu()

    return a, run


@pytest.mark.parametrize("size,place", [(2.0 ** 17, 0.0), (2.0 ** 55, 0.0), (1.0, -2.0 ** 103)])
def test_scores_of_any_size(size, place):
    """Finite scores of any size: far apart (one weight is 1, the others 0), or all at one place far below
    zero (equal weights)."""
    a, run = _two_prompts(torch.Generator().manual_seed(5))
    a["q"], a["k"] = (a["q"].float() * size).bfloat16(), (a["k"].float() * size).bfloat16()
    if place:
        a["q"][:], a["k"][:] = 2.0 ** 10, place
    got, want = run(DEV), run("cpu")
    assert want.isfinite().all() and got.isfinite().all()
    assert float((got - want).norm() / want.norm()) <= TOL


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("Dv", [64, 128])
def test_values_that_are_not_finite_stay_where_they_are_seen(Dv, bad):
    """A value that is not finite reaches the rows that see it and at most those of their 32-row piece that
    share its 32-key piece; what lies behind a sequence's last 8-token group in its page reaches none."""
    a, run = _two_prompts(torch.Generator().manual_seed(7), Dv=Dv)
    clean, v = run(DEV), a["v"].clone()
    for b, end in ((0, 200), (1, 232)):
        a["k"][a["bt"][b, end // 32], :, end % 32:] = bad
        a["v"][a["bt"][b, end // 32], :, end % 32 // 8:] = bad
    assert torch.equal(run(DEV), clean)
    row = torch.arange(150)
    last = 77 + (row | 31).clamp_max(149)
    for j in (3, 80, 110, 141, 200, 226):
        a["v"] = v.clone()
        a["v"][a["bt"][1, j // 32], 1, j % 32 // 8, 5, j % 8] = bad
        got = run(DEV)
        assert torch.equal(got[:200], clean[:200])
        out_of_reach = last < (j & ~31)
        assert torch.equal(got[200:][out_of_reach], clean[200:][out_of_reach])
        assert not got[200:][row + 77 >= j].view(-1, 8, Dv)[:, 2:4, 5].isfinite().any()


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("D,Dv", [(128, 64), (128, 128), (64, 64)])
def test_values_that_are_not_finite_in_a_prompt_from_its_start(D, Dv, bad):
    """The same for a prompt at position 0: its first 32 rows see half of the first step's 64 keys."""
    a, run = _two_prompts(torch.Generator().manual_seed(8), D=D, Dv=Dv)
    clean, v = run(DEV), a["v"].clone()
    row = torch.arange(200)
    for j in (3, 31, 32, 40, 63, 64, 100, 131, 199):
        a["v"] = v.clone()
        a["v"][a["bt"][0, j // 32], 1, j % 32 // 8, 5, j % 8] = bad
        got = run(DEV)
        assert torch.equal(got[200:], clean[200:])
        out_of_reach = (row | 31) < (j & ~31)
        assert torch.equal(got[:200][out_of_reach], clean[:200][out_of_reach]), j
        assert not got[:200][row >= j].view(-1, 8, Dv)[:, 2:4, 5].isfinite().any()
