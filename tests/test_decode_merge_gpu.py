"""Split decode attention: partitions without keys are neither written nor read, at few and many
partitions (past a wave's 64 lanes), whole and ragged pieces, heads and columns that do not fill a
workgroup."""
import pytest
import torch

from aws_k8s_ansible_provisioner_amd.ops import stream as sops

pytestmark = pytest.mark.gpu
BS = 32
LENS = [1, 2250, 0, 333, 128, 40]


def _table(g):
    pages = [-(-n // BS) for n in LENS]
    bt = torch.zeros(len(LENS), max(pages), dtype=torch.int32)
    order, at = torch.randperm(sum(pages), generator=g).int(), 0
    for b, n in enumerate(pages):
        bt[b, :n] = order[at:at + n]
        at += n
    return bt, torch.tensor(LENS, dtype=torch.int32), sum(pages)


def _close(got, want, dtype):
    """bf16: weights and outputs are rounded once each, 2^-9 of a value at most; the roundings of the
    keys are independent, so a row's error stays below 2^-8 of its norm, with half as much again for
    the reference's own rounding."""
    bound = 6e-3 if dtype == torch.bfloat16 else 2e-5
    for b, n in enumerate(LENS):
        if n:
            err = (got[b].float().cpu() - want[b].float()).norm() / want[b].float().norm()
            assert err < bound, (b, n, float(err))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("parts", [2, 5, 70])
@pytest.mark.parametrize("H,G,D", [(6, 2, 64), (4, 4, 128), (3, 1, 32)])
def test_sink_attention(dtype, parts, H, G, D):
    g = torch.Generator().manual_seed(parts * D)
    bt, sl, NB = _table(g)
    q = torch.randn(len(LENS), H, D, generator=g).to(dtype)
    kc = torch.randn(NB, G, BS, D, generator=g).to(dtype)
    vc = torch.randn(NB, G, BS // 8, D, 8, generator=g).to(dtype)
    gate, sink = torch.randn(len(LENS), H, generator=g).to(dtype), torch.randn(H, generator=g)
    want = torch.zeros(len(LENS), H * D, dtype=dtype)
    for window in (0, 600):
        sops.sink_attention_decode(want, q, kc, vc, bt, sl, gate, sink, D ** -0.5, 0, window)
        ws = sops.decode_workspace(len(LENS), H, D, parts, "cuda")
        for t in ws:
            t.fill_(float("nan"))
        got = torch.zeros_like(want, device="cuda")
        sops.sink_attention_decode(got, *(t.cuda() for t in (q, kc, vc, bt, sl, gate, sink)), D ** -0.5,
                                   0, window, ws, parts)
        _close(got, want, dtype)


@pytest.mark.parametrize("parts", [2, 5, 70])
@pytest.mark.parametrize("H,R,r", [(5, 512, 64), (16, 256, 32), (3, 96, 16)])
def test_latent_attention(parts, H, R, r):
    g = torch.Generator().manual_seed(parts * R)
    bt, sl, NB = _table(g)
    T, bf = len(LENS), torch.bfloat16
    cache = torch.randn(NB, BS, R + r, generator=g).to(bf)
    vg = cache[:, :, :R].reshape(-1, BS // 8, 8, R).transpose(2, 3).contiguous()
    ql = (0.3 * torch.randn(H, T, R, generator=g)).to(bf)
    q = torch.randn(T, H, r, generator=g).to(bf)
    pos = (sl - 1).clamp(min=0).long()
    want = torch.zeros(H, T, R, dtype=bf)
    sops.latent_attention(want, ql, q, 0, cache, bt, sl, None, pos, (R + r) ** -0.5)
    ws = sops.latent_decode_workspace(T, H, R, parts, "cuda")
    for t in ws:
        t.fill_(float("nan"))
    got = torch.zeros_like(want, device="cuda")
    ql, q, cache, vg, bt, sl, pos = (t.cuda() for t in (ql, q, cache, vg, bt, sl, pos))
    sops.latent_attention_decode(got, ql, q, 0, cache, vg, bt, sl, pos, (R + r) ** -0.5, ws, parts)
    _close(got.transpose(0, 1), want.transpose(0, 1), bf)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("parts", [2, 5, 70])
@pytest.mark.parametrize("H,G,D,Dv", [(16, 4, 64, 128), (32, 8, 32, 64), (6, 2, 32, 96), (3, 3, 16, 32)])
def test_talking_attention(dtype, parts, H, G, D, Dv):
    g = torch.Generator().manual_seed(parts * Dv + H)
    bt, sl, NB = _table(g)
    T = len(LENS)
    q = torch.randn(T, H, D, generator=g).to(dtype)
    kc = torch.randn(NB, G, BS, D, generator=g).to(dtype)
    vc = torch.randn(NB, G, BS // 8, Dv, 8, generator=g).to(dtype)
    talk = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)
    gate = torch.randn(T, H * Dv, generator=g).to(dtype)
    pos = (sl - 1).clamp(min=0).long()
    for mix in (talk, None):
        want = torch.zeros(T, H * Dv, dtype=dtype)
        sops.talking_attention(want, q, kc, vc, bt, sl, None, pos, mix, gate, D ** -0.5)
        ws = sops.talking_attention_workspace(T, H, G, Dv, parts, "cuda")
        for t in ws:
            t.fill_(float("nan"))
        got = torch.zeros_like(want, device="cuda")
        dev = [t.cuda() for t in (q, kc, vc, bt, sl, pos)]
        sops.talking_attention_decode(got, *dev, mix.cuda() if mix is not None else None, gate.cuda(),
                                      D ** -0.5, ws, parts)
        _close(got, want, dtype)


@pytest.mark.parametrize("part_size,parts", [(768, 3), (256, 9), (128, 18), (128, 33), (512, 64)])
@pytest.mark.parametrize("G", [1, 2, 4])
def test_paged_attention(part_size, parts, G):
    """Against the same kernel unsplit.  A weight is rounded to bf16 against its partition's maximum, so to
    other bits than unsplit: at most 2^-9 of it on either side, 2^-8 of the weighted mean of |v| in all;
    the outputs are rounded once on either side."""
    from aws_k8s_ansible_provisioner_amd import ops

    g = torch.Generator().manual_seed(parts)
    bt, sl, NB = _table(g)
    H, D, T, bf = 3, 128, len(LENS), torch.bfloat16
    k = torch.randn(NB, H, BS, D, generator=g).to(bf).cuda()
    v = torch.randn(NB, H, BS // 8, D, 8, generator=g).to(bf).cuda()
    q = torch.randn(T, H * G, D, generator=g).to(bf).cuda()
    bt, sl = bt.cuda(), sl.cuda()
    got, want = (torch.full((T, H * G, D), 7.0, dtype=bf, device="cuda") for _ in range(2))
    ops.paged_attention_decode(want, q, k, v, bt, sl, G, D ** -0.5, part_size=2304)
    ws = ops.decode_workspace(T, H, G, parts, "cuda")
    for t in ws:
        t.fill_(float("nan"))
    ops.paged_attention_decode(got, q, k, v, bt, sl, G, D ** -0.5, ws, parts, part_size)
    got, want = got.float(), want.float()
    assert bool((got[2] == 0).all()) and bool((want[2] == 0).all())       # a row without keys
    mag = torch.empty_like(q)
    ops.paged_attention_decode(mag, q, k, v.abs(), bt, sl, G, D ** -0.5, part_size=2304)
    assert bool(((got - want).abs() <= 2.0 ** -8 * (1.02 * mag.float() + want.abs())).all())
    assert (got - want).norm() <= 6e-3 * want.norm()      # independent roundings, as above


@pytest.mark.parametrize("part_size,parts,G", [(128, 18, 2), (256, 9, 4), (1024, 3, 1), (768, 2, 16)])
def test_paged_attention_tickets(part_size, parts, G):
    """The merge within the launch: the values of the second launch (a workspace without tickets) but for
    the order of one fp32 product, so at most one bf16 step apart; tickets that are zeros again after every
    launch; and the same bits from every replay of a captured step, whoever comes last."""
    from aws_k8s_ansible_provisioner_amd import ops

    g = torch.Generator().manual_seed(parts)
    bt, sl, NB = _table(g)
    H, D, T, bf = 3, 128, len(LENS), torch.bfloat16
    k = torch.randn(NB, H, BS, D, generator=g).to(bf).cuda()
    v = torch.randn(NB, H, BS // 8, D, 8, generator=g).to(bf).cuda()
    q = torch.randn(T, H * G, D, generator=g).to(bf).cuda()
    bt, sl = bt.cuda(), sl.cuda()
    want, got = (torch.full((T, H * G, D), 7.0, dtype=bf, device="cuda") for _ in range(2))
    ws = ops.decode_workspace(T, H, G, parts, "cuda")
    ops.paged_attention_decode(want, q, k, v, bt, sl, G, D ** -0.5, tuple(ws), parts, part_size)

    def step():
        ops.paged_attention_decode(got, q, k, v, bt, sl, G, D ** -0.5, ws, parts, part_size)

    step()
    assert not bool(ws.tickets.any())
    d = (got.float() - want.float()).abs()
    assert bool((d <= 2.0 ** -7 * want.float().abs()).all())
    first = got.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for _ in range(4):
        got.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, first) and not bool(ws.tickets.any())


def test_paged_attention_tickets_are_left_as_found():
    """A whole step adds nothing to its tickets, whatever stands in them when it starts and however many
    partitions its rows have: one whose tickets another step was using (with outputs that mean nothing) leaves
    them to that one, and the step after both finds zeros."""
    from aws_k8s_ansible_provisioner_amd import ops

    g = torch.Generator().manual_seed(3)
    bt, sl, NB = _table(g)
    H, G, D, T, bf = 3, 2, 128, len(LENS), torch.bfloat16
    k = torch.randn(NB, H, BS, D, generator=g).to(bf).cuda()
    v = torch.randn(NB, H, BS // 8, D, 8, generator=g).to(bf).cuda()
    q = torch.randn(T, H * G, D, generator=g).to(bf).cuda()
    bt, sl = bt.cuda(), sl.cuda()
    ws = ops.decode_workspace(T, H, G, 18, "cuda")
    first, out = (torch.empty(T, H * G, D, dtype=bf, device="cuda") for _ in range(2))
    ops.paged_attention_decode(first, q, k, v, bt, sl, G, D ** -0.5, ws, 18, 128)
    for parts, size in ((18, 128), (9, 256), (2, 1152)):
        ws.tickets.fill_(3)
        ops.paged_attention_decode(out, q, k, v, bt, sl, G, D ** -0.5, ws, parts, size)
        assert bool((ws.tickets == 3).all())
    ws.tickets.fill_(0)
    ops.paged_attention_decode(out, q, k, v, bt, sl, G, D ** -0.5, ws, 18, 128)
    assert torch.equal(out, first)


def test_paged_attention_workspace_of_another_stream():
    """A workspace made on a stream with much to do, used on another one at once: its tickets are there.  One
    made while a graph is captured has none, and merges by the second launch."""
    from aws_k8s_ansible_provisioner_amd import ops

    g = torch.Generator().manual_seed(4)
    bt, sl, NB = _table(g)
    H, G, D, T, bf = 3, 2, 128, len(LENS), torch.bfloat16
    k = torch.randn(NB, H, BS, D, generator=g).to(bf).cuda()
    v = torch.randn(NB, H, BS // 8, D, 8, generator=g).to(bf).cuda()
    q = torch.randn(T, H * G, D, generator=g).to(bf).cuda()
    bt, sl = bt.cuda(), sl.cuda()
    want, got = (torch.full((T, H * G, D), 7.0, dtype=bf, device="cuda") for _ in range(2))
    ops.paged_attention_decode(want, q, k, v, bt, sl, G, D ** -0.5,
                               ops.decode_workspace(T, H, G, 9, "cuda"), 9, 256)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        a = torch.randn(4096, 4096, device="cuda")
        left = torch.full((T * H * ops.DECODE_TICKET_INTS,), 5, dtype=torch.int32, device="cuda")
        del left                                   # (the tickets may be given this memory)
        for _ in range(20):
            a = (a @ a).clamp_(-1, 1)
        ws = ops.decode_workspace(T, H, G, 9, "cuda")
    ops.paged_attention_decode(got, q, k, v, bt, sl, G, D ** -0.5, ws, 9, 256)
    assert ws.tickets is not None and torch.equal(got, want)

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ws = ops.decode_workspace(T, H, G, 9, "cuda")
        ops.paged_attention_decode(got, q, k, v, bt, sl, G, D ** -0.5, ws, 9, 256)
    assert ws.tickets is None
    plain = torch.empty_like(want)
    ops.paged_attention_decode(plain, q, k, v, bt, sl, G, D ** -0.5,
                               tuple(ops.decode_workspace(T, H, G, 9, "cuda")), 9, 256)
    for _ in range(3):
        got.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, plain)


@pytest.mark.parametrize("T,H,G,parts,size,fp8", [
    (4, 8, 2, 16, 128, False), (3, 1, 8, 70, 128, False), (1, 2, 16, 140, 128, False), (2, 1, 4, 513, 128, True),
    (9, 4, 5, 3, 1024, True)])
def test_paged_attention_merge_of_many_partitions(T, H, G, parts, size, fp8):
    """Rows of all partitions, all but a key, one key, one whole partition, one key more and none: the values of the
    second launch but for the order of one fp32 product; its own where there are tickets for fewer rows or the
    partial rows lie off 16 bytes, whatever the tickets hold."""
    from aws_k8s_ansible_provisioner_amd import ops

    g = torch.Generator().manual_seed(T + parts)
    D, bf, most = 128, torch.bfloat16, parts * size
    lens = [most, size + 1, most - 1, 1, 0, size, most // 2, 3, most][:T]
    NB = most // BS
    bt = torch.stack([torch.randperm(NB, generator=g) for _ in range(T)]).int().cuda()
    k = torch.randn(NB, H, BS, D, generator=g).to(bf).cuda()
    v = torch.randn(NB, H, BS // 8, D, 8, generator=g).to(bf).cuda()
    if fp8:
        k, v = (t.to(torch.float8_e4m3fn).view(torch.uint8) for t in (k, v))
    q = torch.randn(T, H * G, D, generator=g).to(bf).cuda()
    sl = torch.tensor(lens, dtype=torch.int32).cuda()
    want, got = (torch.full((T, H * G, D), 7.0, dtype=bf, device="cuda") for _ in range(2))
    ws = ops.decode_workspace(T, H, G, parts, "cuda")
    ops.paged_attention_decode(want, q, k, v, bt, sl, G, D ** -0.5, tuple(ws), parts, size)
    ops.paged_attention_decode(got, q, k, v, bt, sl, G, D ** -0.5, ws, parts, size)
    assert bool(((got.float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs()).all())
    assert not bool(ws.tickets.any())
    short = ops.DecodeWorkspace(tuple(ws))
    short.tickets = torch.full((T * H * ops.DECODE_TICKET_INTS - 1,), 5, dtype=torch.int32, device="cuda")
    odd = ops.DecodeWorkspace((ws[0], ws[1], torch.empty(ws[2].numel() + 1, device="cuda")[1:]))
    odd.tickets = torch.full_like(ws.tickets, 5)
    for w in (short, odd):
        got.fill_(7.0)
        ops.paged_attention_decode(got, q, k, v, bt, sl, G, D ** -0.5, w, parts, size)
        assert torch.equal(got, want) and bool((w.tickets == 5).all())
