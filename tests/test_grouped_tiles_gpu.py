"""Grouped products on 256 x 256 tiles whose last round goes in quarters: one to six K tiles (the quarters
hold three ahead), groups that are empty, shorter than a quarter and longer than a tile, a step that is all
quarters, one of whole tiles and quarters and one whose last round is too full to cut, gathered rows."""
import pytest
import torch

from aws_k8s_ansible_provisioner_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("lens,N,K,gather", [
    ([5], 256, 64, False), ([0, 300, 64, 0, 129], 512, 128, True), ([65, 1, 513], 256, 192, False),
    ([255, 257], 768, 256, True), ([700, 0, 31], 512, 384, False),
    ([256 * 60, 256 * 70 + 1], 512, 64, True),            # 262 tiles: 256 whole, 6 in quarters
    ([256 * 200, 10], 256, 64, False),                    # 201: whole
])
def test_last_round(lens, N, K, gather, silu):
    ops.load_native(required=True)
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + K)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()
    M, E = sum(lens), len(lens)
    offs = torch.tensor(lens, device="cuda").cumsum(0).to(torch.int32)
    rows = torch.randperm(M, device="cuda", generator=g).to(torch.int32) if gather else None
    x, w = rnd((M + 1) // 2 if gather else M, K), rnd(E, N, K)
    out = torch.full((M, N // 2 if silu else N), 7.0, device="cuda", dtype=torch.bfloat16)
    torch.ops.akap.pgemm(out, x, w, 2 if silu else 0, offs, rows, 2 if gather else 1)
    xs = (x[(rows // 2).long()] if gather else x).float()
    at = 0
    for e, n in enumerate(lens):
        if n == 0:
            continue
        y = xs[at:at + n] @ w[e].float().t()
        mag = xs[at:at + n].abs() @ w[e].float().abs().t()
        got = out[at:at + n].float()
        at += n
        if not silu:      # one rounding to bf16 and K products summed in fp32 on either side
            assert bool(((got - y).abs() <= 2.0 ** -8 * y.abs() + K * 2.0 ** -22 * mag).all())
            continue
        # gate, up and their sigmoid form are rounded in turn: 3 * 2^-8 of the product, and what the
        # rounding of the gate (2^-8 of it, slope of the silu at most 1.1) makes of it
        a, b = y[:, :N // 2].bfloat16().float(), y[:, N // 2:].bfloat16().float()
        want = torch.nn.functional.silu(a) * b
        lim = 3 * 2.0 ** -8 * want.abs() + 1.1 * 2.0 ** -8 * (a.abs() * b.abs()) + 1e-3
        assert bool(((got - want).abs() <= lim).all())
