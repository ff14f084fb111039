"""Attention of prompt chunks with keys and values staged through LDS (GPU) against the same ops on
CPU tensors: both head sizes, every split of the query heads over the waves (1, 2, 3, 4, 8 heads to a
key/value head), chunks that end inside 32-token pieces and 128-token tiles, cached tokens before them,
chunk and window edges, sinks, gates, pooled entries past one step of 64, rows that are not 16-byte
aligned, and pages of 32 and 64 tokens.

Tolerance: weights and outputs are rounded to bf16 (relative 2^-9 each, on either side for the
outputs): the 2-norm of the difference stays under 3 * 2^-9 of the result's."""
import math

import pytest
import torch

from aws_k8s_ansible_provisioner_amd.ops import stream as sops

pytestmark = pytest.mark.gpu
DEV, TOL = "cuda", 3 * 2.0 ** -9


def _step(shape, G, D, BS, rows, seed):
    """(cached, new) per sequence -> staged arrays and random caches (CPU)."""
    g = torch.Generator().manual_seed(seed)
    pages = [-(-(p + n) // BS) for p, n in shape]
    perm = torch.randperm(sum(pages) + 2, generator=g)
    bt = torch.zeros(len(shape), max(pages) + 1, dtype=torch.int32)
    at, tiles, start, pos = 0, [], [0], []
    for b, (p, n) in enumerate(shape):
        bt[b, :pages[b]] = perm[at:at + pages[b]].to(torch.int32)
        at += pages[b]
        start.append(start[-1] + n)
        pos.append(torch.arange(p, p + n))
        tiles += [(p + min(n, r + rows), b, r) for r in range(0, n, rows)]
    tiles.sort(key=lambda t: t[0])
    pos = torch.cat(pos)
    seq = torch.repeat_interleave(torch.arange(len(shape)), torch.tensor([n for _, n in shape]))
    slots = bt[seq, pos // BS].long() * BS + pos % BS
    NB = len(perm)
    return dict(bt=bt, q_start=torch.tensor(start, dtype=torch.int32), pos=pos, slots=slots,
                lens=torch.tensor([p + n for p, n in shape], dtype=torch.int32),
                ts=torch.tensor([t[1] for t in tiles], dtype=torch.int32),
                tr=torch.tensor([t[2] for t in tiles], dtype=torch.int32), rows=rows,
                k=torch.randn(NB, G, BS, D, generator=g).bfloat16(),
                v=torch.randn(NB, G, BS // 8, D, 8, generator=g).bfloat16(), gen=g)


def _close(got, want):
    got, want = got.cpu().double(), want.double()
    assert float((got - want).norm() / want.norm()) < TOL
    assert float((got - want).abs().max()) < 16 * 2.0 ** -9 * float(want.abs().max())


SHAPES = [[(0, 1), (0, 33), (70, 64)], [(0, 300), (5, 129), (190, 31)], [(130, 257), (0, 128)]]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("H,G,D,BS,rows", [(4, 4, 128, 32, 128), (4, 2, 64, 64, 128), (6, 2, 128, 32, 128),
                                           (8, 2, 128, 64, 256), (8, 1, 64, 32, 128),
                                           (3, 1, 64, 32, 256)])
@pytest.mark.parametrize("chunk,window", [(0, 0), (64, 0), (0, 45), (100, 70)])
def test_sink_prefill_staged(shape, H, G, D, BS, rows, chunk, window):
    s = _step(shape, G, D, BS, rows, seed=H * D + chunk)
    T = int(s["q_start"][-1])
    q = torch.randn(T, H, D, generator=s["gen"]).bfloat16()
    odd = window > 0                      # rows that start at odd elements / 16-byte pieces
    proj = torch.randn(T, H + 3, generator=s["gen"]).bfloat16()
    gate = proj[:, 2:2 + H] if chunk else None
    sink = torch.randn(H, generator=s["gen"]) * 3 if chunk or window else None
    args = (s["bt"], s["lens"], s["q_start"], s["ts"], s["tr"])
    outs = []
    for dev in ("cpu", DEV):
        wide = torch.zeros(T, H * D + (5 if odd else 8), dtype=torch.bfloat16, device=dev)
        out = wide[:, 1 if odd else 0:][:, :H * D]
        sops.sink_attention_prefill(out, q.to(dev), s["k"].to(dev), s["v"].to(dev),
                                    *(a.to(dev) for a in args), rows,
                                    proj.to(dev)[:, 2:2 + H] if gate is not None else None,
                                    sink.to(dev) if sink is not None else None, D ** -0.5, chunk,
                                    window)
        outs.append(out)
    _close(outs[1], outs[0])


@pytest.mark.parametrize("H,G,D,window,pool", [(4, 2, 128, 40, 4), (8, 2, 64, 70, 1), (3, 1, 64, 64, 16),
                                               (2, 2, 128, 33, 40)])
@pytest.mark.parametrize("shape", [[(0, 150), (260, 70)], [(500, 33), (0, 40), (37, 129)]])
def test_pooled_prefill_staged(shape, H, G, D, window, pool):
    BS = 32
    s = _step(shape, G, D, BS, 128, seed=H + D + window)
    T = int(s["q_start"][-1])
    q = torch.randn(T, H, D, generator=s["gen"]).bfloat16()
    n = sops.pool_slots(BS, pool)
    NB = s["k"].shape[0]
    kp, vp = (torch.randn(NB, G, n, D, generator=s["gen"]) for _ in range(2))
    outs = []
    for dev in ("cpu", DEV):
        out = torch.zeros(T, H * D, dtype=torch.bfloat16, device=dev)
        sops.pooled_window_attention_prefill(
            out, q.to(dev), s["k"].to(dev), s["v"].to(dev), kp.to(dev), vp.to(dev), s["bt"].to(dev),
            s["q_start"].to(dev), s["pos"].to(dev), s["slots"].to(dev), s["ts"].to(dev),
            s["tr"].to(dev), 128, D ** -0.5, window, pool, True)
        outs.append(out)
    _close(outs[1], outs[0])


@pytest.mark.parametrize("D", [32, 64, 128])
def test_sink_prefill_ranges(D):
    """Tiles that name no sequence and sequences with fewer keys than rows are passed over; block-table
    entries outside the cache or past the table's end are page 0.  The same at every head size."""
    H, G, BS, rows = 8, 2, 32, 128
    s = _step([(0, 150), (40, 90), (0, 70)], G, D, BS, rows, seed=D)
    q = torch.randn(310, H, D, generator=s["gen"]).bfloat16()

    def run(bt, lens, ts):
        out = torch.full((310, H * D), 7.0, dtype=torch.bfloat16, device=DEV)
        sops.sink_attention_prefill(out, *(t.to(DEV) for t in (q, s["k"], s["v"], bt, lens, s["q_start"],
                                                              ts, s["tr"])), rows, None, None,
                                    D ** -0.5)
        torch.cuda.synchronize()
        return out.cpu()

    whole = run(s["bt"], s["lens"], s["ts"])
    lens = s["lens"].clone()
    lens[1] = 0
    got = run(s["bt"], lens, s["ts"])
    assert (got[150:240] == 7).all()
    assert torch.equal(got[:150], whole[:150]) and torch.equal(got[240:], whole[240:])
    for bad in (-1, 3):
        got = run(s["bt"], s["lens"], torch.where(s["ts"] == 2, bad, s["ts"]).to(torch.int32))
        assert (got[240:] == 7).all() and torch.equal(got[:240], whole[:240])
    zero, out_of_range = s["bt"].clone(), s["bt"].clone()
    zero[0, 2], out_of_range[0, 2] = 0, -1
    zero[1, 1], out_of_range[1, 1] = 0, s["k"].shape[0]
    assert torch.equal(run(out_of_range, s["lens"], s["ts"]), run(zero, s["lens"], s["ts"]))
    cut = s["bt"].clone()
    cut[:, 3:] = 0
    assert torch.equal(run(s["bt"][:, :3].contiguous(), s["lens"], s["ts"]),
                       run(cut, s["lens"], s["ts"]))


@pytest.mark.parametrize("sink", [0.0, 6.0, 12.0])
def test_sink_prefill_error_does_not_grow_with_the_sink(sink):
    """A sink scales a row's weights and sums alike, so the weights' rounding (2^-9, the largest exactly 1)
    must not depend on it.  For scores of deviation 2 a float64 model of both forms gives, averaged over
    these 3584 rows, 1.00 of the error without a sink where the sink enters at the end, and 1.12 and 1.17
    (sinks of 6 and 12) where maximum and sum start from it."""
    H, G, D, T = 16, 2, 128, 256
    scale = 2 * D ** -0.5
    s = _step([(0, T)], G, D, 32, 128, seed=3)
    q = torch.randn(T, H, D, generator=s["gen"]).bfloat16()
    K = s["k"][s["bt"][0, :8].long()].transpose(0, 1).reshape(G, T, D).double()
    V = s["v"][s["bt"][0, :8].long()].transpose(3, 4).transpose(0, 1).reshape(G, T, D).double()
    x = torch.einsum("thd,hjd->htj", q.double(), K.repeat_interleave(H // G, 0)) * scale
    x = x.masked_fill(torch.ones(T, T).triu(1).bool(), float("-inf"))
    errs = []
    for sk in (None, sink):
        out = torch.empty(T, H * D, dtype=torch.bfloat16, device=DEV)
        sops.sink_attention_prefill(
            out, *(s[n].to(DEV) if isinstance(n, str) else n for n in
                   (q.to(DEV), "k", "v", "bt", "lens", "q_start", "ts", "tr")), 128, None,
            None if sk is None else torch.full((H,), sk, device=DEV), scale)
        z = torch.full((H, T, 1), float("-inf") if sk is None else sk, dtype=torch.float64)
        want = torch.matmul(torch.softmax(torch.cat([x, z], 2), 2)[..., :-1],
                            V.repeat_interleave(H // G, 0)).transpose(0, 1)
        got = out.cpu().double().view(T, H, D)
        errs.append(float(((got - want).norm(dim=2) / want.norm(dim=2))[32:].mean()))
    assert errs[1] < 1.03 * errs[0], errs


def test_sink_prefill_gate_is_exact_to_fp32():
    """Gates far below zero: a row that sees one key has its value times sigmoid(z) as the result, which
    must round to the bf16 that the exact product rounds to but for fp32 errors.  An error of e times the
    value turns a share e / 2^-7.5 of the roundings over.  Exponential, sum, division and product err by
    1.5 * 2^-24 on average: 1.6e-5; an exponential whose argument z log2(e) is rounded to fp32 first errs
    by some 20 * 2^-24: 2e-4.  The line is at five times the former."""
    H, G, D, T = 16, 16, 128, 512
    s = _step([(0, T)], G, D, 32, 128, seed=9)
    z = (-60 - 25 * torch.rand(T, H, generator=s["gen"])).bfloat16()
    out = torch.empty(T, H * D, dtype=torch.bfloat16, device=DEV)
    q = torch.randn(T, H, D, generator=s["gen"]).bfloat16()
    sops.sink_attention_prefill(
        out, q.to(DEV), *(s[n].to(DEV) for n in ("k", "v", "bt", "lens", "q_start", "ts", "tr")), 128,
        z.to(DEV), None, D ** -0.5, 1)                  # chunks of one position: a row sees its own key
    v = s["v"][s["bt"][0, :16].long()].transpose(3, 4).transpose(1, 2).reshape(16 * 4, G, 8, D)
    v = v.transpose(1, 2).reshape(T, G, D).double()
    want = (v * torch.sigmoid(z.double())[:, :, None]).view(T, H * D)
    assert float((out.cpu() != want.bfloat16()).float().mean()) < 8e-5


@pytest.mark.parametrize("D", [64, 128])
def test_pooled_prefill_small_weights(D):
    """Weights that only a denormal bf16 holds: keys `e` log2 units below the sink of score 0, with values
    of 2^126, add up to i + 1 times 2^(126 - e) at row i (all powers of two but the count: exact but for the
    rounding of the result)."""
    H, G, T = 4, 2, 64
    s = _step([(0, T)], G, D, 32, 128, seed=1)
    q, k = torch.zeros(T, H, D, dtype=torch.bfloat16), torch.zeros_like(s["k"])
    q[..., 0] = 1.0
    v = torch.full_like(s["v"], 2.0 ** 126)
    for e in (0, 100, 126, 128, 133):
        k[..., 0] = -float(e)
        out = torch.empty(T, H * D, dtype=torch.bfloat16, device=DEV)
        sops.pooled_window_attention_prefill(
            out, *(t.to(DEV) for t in (q, k, v)), None, None,
            *(s[n].to(DEV) for n in ("bt", "q_start", "pos", "slots", "ts", "tr")), 128,
            math.log(2.0), 0, 0, True)
        n = torch.arange(1, T + 1).double()[:, None]
        want = n * 2.0 ** (126 - e) / (1 + (n if e == 0 else 0))
        rows = 3 if e == 0 else T            # (sums of four such values with weight 1 are not finite)
        # (log2(e) ln 2 in fp32 is 1 to 2^-24, times the score)
        assert float((out.cpu().double() / want - 1)[:rows].abs().max()) < 2.0 ** -8


@pytest.mark.parametrize("unit_sink", [True, False])
@pytest.mark.parametrize("size,shift", [(2.0 ** 17, 0.0), (2.0 ** 55, 0.0), (2.0 ** 17, -2.0 ** 103)])
def test_pooled_prefill_scores_of_any_size(unit_sink, size, shift):
    """Finite scores of any size: far apart (one weight is 1, the others 0), or all far below zero."""
    H, G, D, T, window, pool = 4, 2, 128, 200, 70, 16
    s = _step([(0, T)], G, D, 32, 128, seed=2)
    q = (torch.randn(T, H, D, generator=s["gen"]) * size).bfloat16()
    k = (s["k"].float() * size).bfloat16()
    n = sops.pool_slots(32, pool)
    kp = (torch.randn(len(k), G, n, D, generator=s["gen"]) * size).bfloat16().float()   # (as operands)
    vp = torch.randn(len(k), G, n, D, generator=s["gen"])
    if shift:                               # every key at the same place, far below
        q[:], k[:], kp[:] = 2.0 ** 10, shift, shift
    outs = []
    for dev in ("cpu", DEV):
        out = torch.zeros(T, H * D, dtype=torch.bfloat16, device=dev)
        sops.pooled_window_attention_prefill(
            out, *(t.to(dev) for t in (q, k, s["v"], kp, vp)),
            *(s[a].to(dev) for a in ("bt", "q_start", "pos", "slots", "ts", "tr")), 128, D ** -0.5,
            window, pool, unit_sink)
        outs.append(out.cpu())
    assert outs[0].isfinite().all() and outs[1].isfinite().all()
    if outs[0].any():
        _close(outs[1], outs[0])
    else:
        assert not outs[1].any()


@pytest.mark.parametrize("D", [64, 128])
def test_sink_prefill_scores_far_below_zero(D):
    """Equal scores below -1e30 (a power of two: exact in fp32) are equal weights."""
    H, G, T = 8, 2, 200
    s = _step([(0, T)], G, D, 32, 128, seed=6)
    q, k = torch.full((T, H, D), 2.0 ** 10).bfloat16(), torch.full_like(s["k"], -2.0 ** 103)
    outs = []
    for dev in ("cpu", DEV):
        out = torch.zeros(T, H * D, dtype=torch.bfloat16, device=dev)
        sops.sink_attention_prefill(out, *(t.to(dev) for t in (q, k, s["v"])),
                                    *(s[n].to(dev) for n in ("bt", "lens", "q_start", "ts", "tr")), 128,
                                    None, None, D ** -0.5)
        outs.append(out)
    _close(outs[1], outs[0])


@pytest.mark.parametrize("pooled", [False, True])
@pytest.mark.parametrize("D,window", [(64, 45), (128, 70), (128, 0)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_values_that_are_not_finite_stay_where_they_are_seen(pooled, D, window, bad):
    """A value that is not finite reaches the rows that see it and at most the others of their 32-token
    piece (and 8-token group); what lies behind a sequence's last group in its page reaches none."""
    H, G, BS, pool = 8, 2, 32, 8
    shape = [(0, 150), (37, 171)]
    s = _step(shape, G, D, BS, 128, seed=D + window)
    q = torch.randn(321, H, D, generator=s["gen"]).bfloat16()
    n = sops.pool_slots(BS, pool)
    kp, vp = (torch.randn(len(s["k"]), G, n, D, generator=s["gen"]) for _ in range(2))

    def run(k, v, vp):
        out = torch.zeros(321, H * D, dtype=torch.bfloat16, device=DEV)
        m = lambda *names: [s[a].to(DEV) for a in names]
        if pooled:
            sops.pooled_window_attention_prefill(
                out, q.to(DEV), k.to(DEV), v.to(DEV), kp.to(DEV), vp.to(DEV),
                *m("bt", "q_start", "pos", "slots", "ts", "tr"), 128, D ** -0.5, window, pool, True)
        else:
            sops.sink_attention_prefill(out, q.to(DEV), k.to(DEV), v.to(DEV),
                                        *m("bt", "lens", "q_start", "ts", "tr"), 128, None, None,
                                        D ** -0.5, 0, window)
        return out.cpu()

    clean = run(s["k"], s["v"], vp)
    # behind the sequences' last groups
    k, v = s["k"].clone(), s["v"].clone()
    for b, (p, c) in enumerate(shape):
        end = -(-(p + c) // 8) * 8
        k[s["bt"][b, end // BS], :, end % BS:] = bad
        v[s["bt"][b, end // BS], :, end % BS // 8:] = bad
    assert torch.equal(run(k, v, vp), clean)
    # one value of the second sequence
    i = torch.arange(37, 208)
    piece = (i - 37) // 32 * 32 + 37
    last = (piece + 31).clamp_max(207)
    lo = (lambda x: (x - window + 1).clamp_min(0)) if window else torch.zeros_like
    for j in (3, 39, 100, 166, 200):
        v = s["v"].clone()
        v[s["bt"][1, j // BS], 1, j % BS // 8, 5, j % 8] = bad
        got = run(s["k"], v, vp)
        assert torch.equal(got[:150], clean[:150])
        got, want = (x[150:].view(171, H, D) for x in (got, clean))
        out_of_reach = ((last | 7) < j) | ((lo(piece) & ~7) > j)
        assert torch.equal(got[out_of_reach], want[out_of_reach])
        assert not got[(i >= j) & (lo(i) <= j)][:, H // 2:, 5].isfinite().any()
    # one pooled entry
    if pooled and window:
        for c in (0, 7, 13):
            bad_vp = vp.clone()
            bad_vp[s["bt"][1, c * pool // BS], 1, c * pool % BS // pool, 5] = bad
            got = run(s["k"], s["v"], bad_vp)[150:].view(171, H, D)
            unseen = c * pool + pool - 1 > last - window
            assert torch.equal(got[unseen], clean[150:].view(171, H, D)[unseen])
            assert not got[c * pool + pool - 1 <= i - window][:, H // 2:, 5].isfinite().any()


@pytest.mark.parametrize("shape,H,G", [([(0, 256)], 8, 2), ([(0, 257)], 4, 4), ([(200, 121)], 8, 2),
                                       ([(0, 700), (333, 90), (0, 40)], 4, 1), ([(0, 130)] * 20, 8, 4)])
@pytest.mark.parametrize("D,window,pool", [(128, 0, 0), (64, 290, 0), (128, 300, 8), (64, 330, 16)])
def test_two_teams(shape, H, G, D, window, pool):
    """Steps around the number from which two teams share them, odd and even, a pooled part of more than 64
    entries, and a grid that one team takes whatever its steps; values that no query sees are not finite."""
    s = _step(shape, G, D, 32, 128, seed=H * D + window)
    T = int(s["q_start"][-1])
    q = torch.randn(T, H, D, generator=s["gen"]).bfloat16()
    for b, (p, n) in enumerate(shape):
        if (p + n) % 32:
            s["v"][int(s["bt"][b, (p + n) // 32]), :, ((p + n) % 32 + 7) // 8:] = float("nan")
    outs = []
    for dev in ("cpu", DEV):
        m = {k: v.to(dev) for k, v in s.items() if torch.is_tensor(v)}
        out = torch.zeros(T, H * D, dtype=torch.bfloat16, device=dev)
        if pool:
            g = torch.Generator().manual_seed(T)
            kp, vp = (torch.randn(s["k"].shape[0], G, sops.pool_slots(32, pool), D, generator=g).to(dev)
                      for _ in range(2))
            sops.pooled_window_attention_prefill(out, q.to(dev), m["k"], m["v"], kp, vp, m["bt"],
                                                 m["q_start"], m["pos"], m["slots"], m["ts"], m["tr"],
                                                 128, D ** -0.5, window, pool, True)
        else:
            sops.sink_attention_prefill(out, q.to(dev), m["k"], m["v"], m["bt"], m["lens"],
                                        m["q_start"], m["ts"], m["tr"], 128, None,
                                        torch.linspace(-2, 3, H).to(dev), D ** -0.5, 0, window)
        outs.append(out)
    _close(outs[1], outs[0])
