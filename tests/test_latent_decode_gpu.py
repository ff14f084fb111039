"""Latent attention of decode rows (R = 512, r = 64), rows read once: lengths around the blocks of 32
keys and the steps of 32 and 64, tables longer than a batch of 64 blocks, both workgroup sizes, one and two
tiles of heads, unsplit and split, rows behind a sequence's end that are not finite."""
import pytest
import torch

from aws_k8s_ansible_provisioner_amd.ops import stream as sops

pytestmark = pytest.mark.gpu
R, ROT = 512, 64


@pytest.mark.parametrize("H,BS,lens,parts", [
    (16, 32, [1, 31, 32, 33, 63, 64, 65, 0, 97], 1),
    (5, 64, [200, 129, 1, 96], 3),
    (33, 32, [70, 5, 64], 2),
    (16, 32, [2049, 2300, 64], 1),                       # more than 64 blocks in a partition
    (16, 128, [2111, 40], 5),
    (32, 32, [(37 * i) % 150 for i in range(150)], 2),   # more workgroups than CUs
    (33, 64, [4200] + [66] * 130, 1),                    # the same, and more than 64 blocks in a partition
    (16, 32, [4300, 0] + [70] * 130, 2),
])
def test_against_rows(H, BS, lens, parts):
    g = torch.Generator().manual_seed(H * 1000 + parts)
    B, bf = len(lens), torch.bfloat16
    pages = [-(-n // BS) for n in lens]
    NB = sum(pages) + 1
    order = torch.randperm(NB, generator=g).to(torch.int32)
    bt = torch.zeros(B, max(pages), dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        bt[b, :n] = order[at:at + n]
        at += n
    sl = torch.tensor(lens, dtype=torch.int32)
    cache = torch.randn(NB, BS, R + ROT, generator=g).to(bf)
    for b, n in enumerate(lens):                        # behind the end: infinities and NaN
        if n % BS:
            cache[int(bt[b, n // BS]), n % BS:] = float("nan") if b % 2 else float("inf")
    vg = cache[:, :, :R].reshape(NB, BS // 8, 8, R).transpose(2, 3).contiguous()
    ql = (0.3 * torch.randn(H, B, R, generator=g)).to(bf)
    q = torch.randn(B, H, ROT, generator=g).to(bf)
    pos = (sl - 1).clamp(min=0).long()
    scale = 2.0 * (R + ROT) ** -0.5
    want = torch.zeros(H, B, R, dtype=bf)
    sops.latent_attention(want, ql, q, 0, cache, bt, sl, None, pos, scale)
    ws = sops.latent_decode_workspace(B, H, R, parts, "cuda") if parts > 1 else None
    for t in ws or ():
        t.fill_(float("nan"))
    got = torch.zeros(H, B, R, dtype=bf, device="cuda")
    sops.latent_attention_decode(got, ql.cuda(), q.cuda(), 0, cache.cuda(), vg.cuda(), bt.cuda(),
                                 sl.cuda(), pos.cuda(), scale, ws, parts)
    got, want = got.cpu().float(), want.float()
    # an output is a mean of latents: its weights are rounded to bf16 (2^-9 of each, so of the mean of
    # |c|), and so are it and the reference
    seen = torch.cat([cache[bt[b, j // BS].long(), j % BS, :R].float().abs().max()[None]
                      for b, n in enumerate(lens) for j in range(0, n, 7)] or [torch.ones(1)]).max()
    assert (got - want).abs().max() <= 3 * 2.0 ** -9 * max(float(seen), 6.0)
    for b, n in enumerate(lens):
        assert (got[:, b] - want[:, b]).norm() <= 1.2e-2 * want[:, b].norm(), (b, n)
    assert all(bool((got[:, b] == 0).all()) for b, n in enumerate(lens) if n == 0)
