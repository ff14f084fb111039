"""Latent attention of prompt chunks at 512 latent and 64 rotated dimensions (GPU) against the same op
on CPU tensors: odd and even heads, chunks that end inside 32-token units, 32-key pieces and 64-key
steps, cached tokens before them, pages of 32, 64 and 96 tokens, a sequence without rows, rows that lead
the step and stay as they are.

Tolerance: weights and outputs are rounded to bf16 (relative 2^-9 each, on either side for the
outputs): the 2-norm of the difference stays under 3 * 2^-9 of the result's."""
import pytest
import torch

from aws_k8s_ansible_provisioner_amd.ops import stream as sops

pytestmark = pytest.mark.gpu
DEV, TOL, R, ROT = "cuda", 3 * 2.0 ** -9, 512, 64


@pytest.mark.parametrize("H,BS,shape,lead,tile_rows", [
    (1, 32, [(0, 1)], 0, 128),
    (3, 64, [(0, 33), (63, 64), (0, 130)], 0, 128),
    (2, 96, [(95, 97), (1, 31), (0, 0), (64, 65)], 0, 256),
    (16, 64, [(0, 200), (500, 70)], 0, 128),
    (5, 32, [(40, 1), (70, 1), (31, 161)], 2, 128),
])
def test_chunks(H, BS, shape, lead, tile_rows):
    g = torch.Generator().manual_seed(H * BS)
    pages = [-(-(p + n) // BS) for p, n in shape]
    NB = sum(pages) + 1
    perm, at = torch.randperm(NB, generator=g), 0
    bt = torch.zeros(len(shape), max(pages), dtype=torch.int32)
    tiles, start = [], [0]
    for b, (p, n) in enumerate(shape):
        bt[b, :pages[b]] = perm[at:at + pages[b]].to(torch.int32)
        at += pages[b]
        start.append(start[-1] + n)
        if b >= lead:
            tiles += [(p + min(n, r + tile_rows), b, r) for r in range(0, n, tile_rows)]
    tiles.sort()
    T, i32 = start[-1], lambda x: torch.tensor(x, dtype=torch.int32)
    pos = torch.cat([torch.arange(p, p + n) for p, n in shape])
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16()
    cache = rnd(NB, BS, R + ROT)
    groups = cache[..., :R].reshape(NB, BS // 8, 8, R).transpose(2, 3).contiguous()
    q_lat, q = rnd(H, T, R), rnd(T, H, 128 + ROT)
    lens, qs = i32([p + n for p, n in shape]), i32(start)
    ts, tr = i32([t[1] for t in tiles]), i32([t[2] for t in tiles])

    def run(dev):
        m = lambda x: x.to(dev)
        out = torch.zeros(H, T, R, dtype=torch.bfloat16, device=dev)
        sops.latent_attention_prefill(out, m(q_lat), m(q), 128, m(cache), m(groups), m(bt), m(lens),
                                      m(qs), m(pos), m(ts), m(tr), tile_rows, (R + ROT) ** -0.5,
                                      first_seq=lead)
        return out.float().cpu()

    a, b = run(DEV), run("cpu")
    assert bool((a[:, :start[lead]] == 0).all())
    a, b = a[:, start[lead]:], b[:, start[lead]:]
    assert float((a - b).norm() / b.norm()) <= TOL
    assert float((a - b).abs().max()) <= 8 * TOL * float(b.abs().max())


def test_scores_far_below_zero():
    """All keys at one place whose scores lie below -1e30 (a power of two: exact): equal weights, so every row is
    that place again."""
    H, T = 3, 70
    q_lat, q = torch.full((H, T, R), 2.0 ** 10), torch.zeros(T, H, 128 + ROT)
    cache = torch.full((4, 32, R + ROT), -2.0 ** 103)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    out = torch.zeros(H, T, R, dtype=torch.bfloat16, device=DEV)
    bf = lambda x: x.bfloat16().to(DEV)
    sops.latent_attention_prefill(out, bf(q_lat), bf(q), 128, bf(cache),
                                  bf(cache[..., :R].reshape(4, 4, R, 8)), i32([[2, 0, 3]]), i32([T]),
                                  i32([0, T]), torch.arange(T, device=DEV), i32([0]), i32([0]), 128,
                                  (R + ROT) ** -0.5)
    assert float((out.double().cpu() / -2.0 ** 103 - 1).abs().max()) <= 2.0 ** -8
