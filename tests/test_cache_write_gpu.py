"""The cache-writing kernels in 16-byte pieces (GPU) against the same ops on CPU tensors: steps on both
sides of 512 rows, a last group of rows that is not full, chunks whose slots start inside an 8-token
group, rows that write nothing, several sequences whose rows meet inside one group, and blocks of
pooled entries that cross pages.

Tolerance: both sides compute in fp32 and round once.  Sums in another order and the two square roots
differ by a few 2^-24 relative, and a rotation adds two products of at most about 8 with that error
each: at most 2^-18 absolute also where they cancel.  On top a bf16 rounding can move by one step
(8 significant bits: at most 2^-7 of the value)."""
import pytest
import torch

from aws_k8s_ansible_provisioner_amd.ops import stream as sops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _step(n, BS, seed):
    """Slots of sequences of uneven lengths that begin at any token of a group, a few rows -1."""
    g = torch.Generator().manual_seed(seed)
    slots, pos, page = [], [], 0
    while len(slots) < n:
        ln = min(int(torch.randint(1, 200, (1,), generator=g)), n - len(slots))
        p0 = int(torch.randint(0, 2 * BS, (1,), generator=g))
        slots += [page * BS + p for p in range(p0, p0 + ln)]
        pos += range(p0, p0 + ln)
        page += -(-(p0 + ln) // BS)
    slots, pos = torch.tensor(slots), torch.tensor(pos)
    slots[torch.randperm(n, generator=g)[:max(1, n // 50)]] = -1
    perm = torch.randperm(page + 1, generator=g)
    return torch.where(slots >= 0, perm[slots.clamp(min=0) // BS] * BS + slots % BS, slots), pos, \
        page + 1


def _same(a, b, dt):
    a, b = a.float(), b.float()
    step = 2.0 ** -7 if dt == torch.bfloat16 else 0.0
    over = (a - b).abs() - step * b.abs()
    assert float(over.max()) <= 2.0 ** -18, float(over.max())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 511, 512, 515])
@pytest.mark.parametrize("form", ["normed", "biased", "whole"])
def test_head_caches(form, n, dt):
    g = torch.Generator().manual_seed(n)
    H, G, D, Dv, BS = 4, 2, 64, 64 if form == "whole" else 128, 32
    slots, pos, NB = _step(n, BS, n)
    N = (H + G) * D + G * Dv + 8
    proj = torch.randn(n, N, generator=g).to(dt)
    cs = sops.rotary_table(4 * BS + 200, 32, 1e4, None, "cpu")
    bias = torch.randn(N, generator=g)
    qw, kw = torch.rand(H * D, generator=g) + 0.5, torch.rand(G * D, generator=g) + 0.5
    qb, kb = torch.randn(H * D, generator=g).to(dt), torch.randn(G * D, generator=g).to(dt)

    def run(dev):
        c = lambda t: t.clone().to(dev)
        q = torch.zeros(n, H, D, dtype=dt, device=dev)
        kc = torch.zeros(NB, G, BS, D, dtype=dt, device=dev)
        vc = torch.zeros(NB, G, BS // 8, Dv, 8, dtype=dt, device=dev)
        if form == "normed":
            sops.head_norm_cache(c(proj), q, kc, vc, c(slots), H, G, D, Dv, 8, 8 + H * D,
                                 8 + (H + G) * D, 1e-5, q_w=c(qw[:D]), k_w=c(kw[:D]),
                                 cos_sin=c(cs), positions=c(pos))
        elif form == "biased":
            sops.bias_rope_cache(c(proj), q, kc, vc, c(pos), c(slots), c(cs), c(bias), H, G, D, Dv,
                                 8, 8 + H * D, 8 + (H + G) * D)
        else:
            sops.proj_norm_rope_cache(c(proj), q, kc, vc, c(pos), c(slots), c(cs), c(qw), c(kw),
                                      H, G, D, 8, 8 + H * D, 1e-5, c(qb), c(kb))
        return q, kc, vc

    for a, b in zip(run(DEV), run("cpu")):
        _same(a.cpu(), b, dt)


@pytest.mark.parametrize("form,n,H,G,D,rot,BS", [
    ("normed", 6601, 16, 4, 128, 128, 32),      # two rows and four heads to a thread
    ("normed", 1703, 17, 3, 128, 64, 40),       # one row and two heads, the last ones missing
    ("biased", 3301, 32, 8, 128, 128, 32), ("biased", 1650, 16, 5, 64, 64, 24),
    ("biased", 700, 6, 2, 256, 128, 32),
    ("whole", 767, 16, 4, 128, 128, 32), ("whole", 768, 16, 4, 128, 64, 32),   # a workgroup, a wave
    ("whole", 771, 24, 8, 64, 64, 40), ("whole", 1027, 32, 8, 128, 128, 32),
    ("whole", 800, 3, 1, 512, 16, 32), ("whole", 801, 5, 1, 96, 32, 32)])
def test_large_steps(form, n, H, G, D, rot, BS):
    """Both sides of the sizes from which a thread takes several rows and heads and a wave a whole
    token; pages that are no power of two, heads and rows left over."""
    g = torch.Generator().manual_seed(n)
    dt = torch.bfloat16
    slots, pos, NB = _step(n, BS, n)
    N = (H + 2 * G) * D + 8
    proj = torch.randn(n, N, generator=g).to(dt)
    cs = sops.rotary_table(4 * BS + 200, rot, 1e4, None, "cpu")
    bias = torch.randn(N, generator=g)
    qw, kw = torch.rand(H * D, generator=g) + 0.5, torch.rand(G * D, generator=g) + 0.5
    qb, kb = torch.randn(H * D, generator=g).to(dt), torch.randn(G * D, generator=g).to(dt)

    def run(dev):
        c = lambda t: t.clone().to(dev)
        q = torch.zeros(n, H, D, dtype=dt, device=dev)
        kc = torch.zeros(NB, G, BS, D, dtype=dt, device=dev)
        vc = torch.zeros(NB, G, BS // 8, D, 8, dtype=dt, device=dev)
        o = (8, 8 + H * D, 8 + (H + G) * D)
        if form == "normed":
            sops.head_norm_cache(c(proj), q, kc, vc, c(slots), H, G, D, D, *o, 1e-5, q_w=c(qw[:D]),
                                 k_w=c(kw[:D]), cos_sin=c(cs), positions=c(pos))
        elif form == "biased":
            sops.bias_rope_cache(c(proj), q, kc, vc, c(pos), c(slots), c(cs), c(bias), H, G, D, D, *o)
        else:
            sops.proj_norm_rope_cache(c(proj), q, kc, vc, c(pos), c(slots), c(cs), c(qw), c(kw), H, G,
                                      D, *o[:2], 1e-5, c(qb), c(kb))
        return q, kc, vc

    for a, b in zip(run(DEV), run("cpu")):
        _same(a.cpu(), b, dt)


@pytest.mark.parametrize("n,q_rank,kv_rank,rot,form", [
    (2047, 768, 512, 64, ""), (2048, 768, 512, 64, ""), (2077, 1536, 512, 64, "half"),
    (2050, 1032, 96, 16, ""), (2049, 64, 256, 32, "rows"), (2051, 768, 512, 64, "queries"),
    (70, 768, 512, 64, ""), (300, 8, 8, 8, "half"), (65, 1536, 504, 128, "half"), (71, 520, 64, 32, "rows"),
    (64, 2048, 512, 64, "queries"), (66, 1032, 512, 136, ""), (576, 64, 512, 64, ""), (577, 64, 512, 64, ""),
    (2047, 64, 256, 32, "half"), (2047, 64, 512, 64, "rows")])
def test_latent_rows(n, q_rank, kv_rank, rot, form):
    """Both sides of 2048 rows (32 to a workgroup) and of 512 + q_rank (one to a wave); rows without the grouped copy, and
    without any; ranks of one 16-byte piece, of one piece more and less than whole waves."""
    g = torch.Generator().manual_seed(n)
    BS, dt = 64, torch.bfloat16
    slots, pos, NB = _step(n, BS, n)
    proj = torch.randn(n, 8 + q_rank + kv_rank + rot, generator=g).to(dt)
    cs = sops.rotary_table(4 * BS + 200, rot, 1e4, None, "cpu")
    qw, kw = torch.rand(q_rank, generator=g) + 0.5, torch.rand(kv_rank, generator=g) + 0.5

    def run(dev):
        c = lambda t: t.clone().to(dev)
        cq = torch.zeros(n, q_rank, dtype=dt, device=dev)
        rows = torch.zeros(NB, BS, kv_rank + rot, dtype=dt, device=dev)
        groups = torch.zeros(NB, BS // 8, kv_rank, 8, dtype=dt, device=dev)
        sops.latent_prep(c(proj), cq, None if form == "queries" else rows, c(pos), c(slots), c(cs),
                         c(qw), c(kw), q_rank, kv_rank, rot, 8, 8 + q_rank, 1e-5,
                         vgroups=None if form in ("rows", "queries") else groups,
                         half=form == "half")
        return cq, rows, groups

    for a, b in zip(run(DEV), run("cpu")):
        _same(a.cpu(), b, dt)


@pytest.mark.parametrize("D,Dv,pool,BS", [(64, 128, 64, 64), (128, 64, 32, 64), (64, 32, 16, 16),
                                          (256, 256, 64, 64), (72, 64, 64, 64)])
def test_pooled_blocks(D, Dv, pool, BS):
    """(D of 72: the form row by row.)  Sums of `pool` fp32 values in another order: within
    pool 2^-24 of the largest."""
    g = torch.Generator().manual_seed(D + pool)
    G, shape = 2, [(0, 300), (37, 211), (63, 1), (5, 90)]
    pages = [-(-(p + m) // BS) for p, m in shape]
    NB = sum(pages) + 1
    perm, at = torch.randperm(NB, generator=g), 0
    bt = torch.zeros(len(shape), max(pages), dtype=torch.int32)
    for b, k in enumerate(pages):
        bt[b, :k] = perm[at:at + k].to(torch.int32)
        at += k
    qs = torch.tensor([0] + [m for _, m in shape]).cumsum(0).to(torch.int32)
    pos = torch.cat([torch.arange(p, p + m) for p, m in shape])
    seq = torch.repeat_interleave(torch.arange(len(shape)), torch.tensor([m for _, m in shape]))
    slots = bt[seq, pos // BS].long() * BS + pos % BS
    slots[63] = -1
    kc = torch.randn(NB, G, BS, D, generator=g).bfloat16()
    vc = torch.randn(NB, G, BS // 8, Dv, 8, generator=g).bfloat16()

    def run(dev):
        kp = torch.zeros(NB, G, BS // pool, D, device=dev)
        vp = torch.zeros(NB, G, BS // pool, Dv, device=dev)
        sops.pool_cache_blocks(kc.to(dev), vc.to(dev), kp, vp, pos.to(dev), slots.to(dev),
                               bt.to(dev), qs.to(dev), pool)
        return kp, vp

    for a, b in zip(run(DEV), run("cpu")):
        assert float((a.cpu() - b).abs().max()) <= pool * 2.0 ** -24 * 5


def test_fp32_rows_take_no_longer_than_head_by_head():
    """The norm over whole rows moves a sixth less than the norm per head with values of their own."""
    T, H, G, D, BS = 13000, 16, 4, 128, 32
    slots, pos = torch.arange(T, device=DEV), torch.arange(T, device=DEV) % 2000
    cs = sops.rotary_table(2048, D, 1e4, None, "cpu").to(DEV)
    proj = torch.randn(T, (H + 2 * G) * D, device=DEV)
    q, kc = torch.empty(T, H, D, device=DEV), torch.zeros(T // BS + 1, G, BS, D, device=DEV)
    vc = torch.zeros(T // BS + 1, G, BS // 8, D, 8, device=DEV)
    qw, kw = torch.ones(H * D, device=DEV), torch.ones(G * D, device=DEV)

    def time(step):
        spent = []
        for _ in range(9):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(10):
                step()
            b.record()
            b.synchronize()
            spent.append(a.elapsed_time(b))
        return min(spent)
    whole = time(lambda: sops.proj_norm_rope_cache(proj, q, kc, vc, pos, slots, cs, qw, kw, H, G, D, 0,
                                                   H * D, 1e-5))
    heads = time(lambda: sops.head_norm_cache(proj, q, kc, vc, slots, H, G, D, D, 0, H * D, (H + G) * D,
                                              1e-5, cos_sin=cs, positions=pos))
    assert whole < 1.12 * heads
