"""Prompt chunks of the selective scan and the retention in matrix form (GPU) against the same
ops on CPU tensors: sequences around the chunk size of 32 rows and the segment size of 256, several
sequences per step (some continued from their slots, one a padding sequence), steps whose long
sequences are cut into segments and such that are walked whole, every head size of the matrix form, projections that are column slices of wider rows, and values that are not finite.

Tolerance: both sides sum at most N + 32 products per entry in fp32 in different orders; the
relative 2-norm error of such sums is a few times 2^-24, 2e-6 leaves a factor of ten."""
import math

import pytest
import torch

from aws_k8s_ansible_provisioner_amd.ops import stream as sops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rel(a, b):
    return float((a.double().cpu() - b.double()).norm() / b.double().norm().clamp_min(1e-30))


def _step(lens, starts, seed=0):
    q_start = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    pos = torch.cat([torch.arange(s, s + n) for n, s in zip(lens, starts)]).to(torch.int64)
    slot = torch.cat([torch.full((n,), b if s >= 0 else -1, dtype=torch.int32)
                      for b, (n, s) in enumerate(zip(lens, starts))])
    return q_start, pos.clamp_min(0), slot


# (rows per sequence, first position; -1: a padding sequence without a slot)
STEPS = [([5], [0]), ([32], [7]), ([33, 31, 64], [0, 3, 0]), ([1, 65, 40, 90], [9, 0, -1, 11]),
         ([300, 257, 256, 40], [0, 5, 0, 2]), ([1100], [0])]


def _scan_inputs(T, B, H, V, N, G, dt, wide, seed):
    g = torch.Generator().manual_seed(seed)
    C = H * V + 2 * G * N
    xbc = torch.randn(T, C, generator=g)
    proj = torch.randn(T, H + wide, generator=g).to(dt)[:, wide // 2:]
    state = torch.randn(B, H, N, V, generator=g)
    return (xbc, proj, torch.randn(H, generator=g) * 0.5 - 1.0, torch.randn(H, generator=g) * 0.5,
            torch.randn(H, generator=g) * 0.2 + 1.0, state)


def _run_scan(inp, step, H, V, N, G, dev):
    xbc, proj, bias, a_log, d_skip, state = inp
    wide = proj.stride(0)
    full = torch.zeros(proj.shape[0], wide, dtype=proj.dtype, device=dev)
    off = wide - proj.shape[1] if wide > proj.shape[1] else 0
    full[:, off:off + proj.shape[1]] = proj.to(dev)
    q_start, pos, slot = (t.to(dev) for t in step)
    st = state.clone().to(dev)
    y = torch.zeros(xbc.shape[0], H * V, device=dev)
    sops.selective_scan(y, xbc.to(dev), full[:, off:], 0, bias.to(dev), a_log.to(dev),
                        d_skip.to(dev), st, slot, pos, q_start, H, V, N, G)
    return y, st


@pytest.mark.parametrize("H,V,N,G,dt", [(4, 64, 128, 1, torch.bfloat16), (6, 64, 64, 2, torch.float32),
                                        (2, 128, 128, 2, torch.bfloat16),
                                        (3, 128, 64, 1, torch.float32), (3, 64, 128, 1, torch.float32)])
@pytest.mark.parametrize("lens,starts", STEPS)
def test_selective_scan_chunks(lens, starts, H, V, N, G, dt):
    step = _step(lens, starts)
    inp = _scan_inputs(sum(lens), len(lens), H, V, N, G, dt, 6, seed=sum(lens) + V)
    want = _run_scan(inp, step, H, V, N, G, "cpu")
    got = _run_scan(inp, step, H, V, N, G, DEV)
    live = (step[2] >= 0)
    assert _rel(got[0][live.to(DEV)], want[0][live]) < 2e-6
    assert _rel(got[1], want[1]) < 2e-6
    assert torch.equal(got[1].cpu()[[b for b, s in enumerate(starts) if s < 0]],
                       inp[5][[b for b, s in enumerate(starts) if s < 0]])


# lens, starts, heads of the scan and of the retention (V 64): two cut sequences of five, one continued, a
# padding sequence; one long continued one; a prompt among rows of one token (whose number alone would
# fill the chip); as many long sequences as fill it, so that none is cut; more sequences than a wave has lanes
CUT = [([700, 600, 1, 3, 257], [0, 10, 0, -1, 4], 4, 4), ([1100], [9], 4, 4),
       ([1] * 50 + [1100] + [1] * 10 + [300], [7] * 50 + [0] + [5] * 10 + [40], 8, 8),
       ([300] * 24 + [1] * 10, [0, 3] * 12 + [9] * 10, 16, 16),
       # cut sequences on both sides of the 64th, sequences without rows among them and at the ends
       ([0, 1100, 0, 2] + [1] * 58 + [0, 520, 700] + [3] * 5 + [300, 0], [0, 4, 0, 9] + [6] * 58 + [0, 0, 8]
        + [2] * 5 + [0, 0], 2, 2),
       # 64 and 65 sequences, which are counted and looked at one by one; 70 that are long, too many to be cut
       ([900] + [2] * 62 + [400], [0] + [4] * 62 + [7], 2, 2), ([400] + [2] * 63 + [900], [3] + [4] * 63 + [0], 2, 2),
       ([260] * 70 + [3] * 40, [0, 5] * 35 + [1] * 40, 6, 6)]


@pytest.mark.parametrize("lens,starts,H,_", CUT)
def test_selective_scan_segments(lens, starts, H, _):
    V, N, G = 64, 64, 2
    T, B = sum(lens), len(lens)
    assert torch.ops.akap_stream.chunk_scan_segment(0, T, B, H, V) == 256
    step = _step(lens, starts)
    inp = _scan_inputs(T, B, H, V, N, G, torch.bfloat16, 0, seed=T)
    want = _run_scan(inp, step, H, V, N, G, "cpu")
    got = _run_scan(inp, step, H, V, N, G, DEV)
    live = step[2] >= 0
    assert _rel(got[0][live.to(DEV)], want[0][live]) < 2e-6
    assert _rel(got[1], want[1]) < 2e-6
    for b in range(B):                     # (each sequence for itself: a lost one is small beside the rest)
        if starts[b] >= 0:
            assert _rel(got[1][b], want[1][b]) < 1e-5
        else:
            assert torch.equal(got[1][b].cpu(), inp[5][b])


@pytest.mark.parametrize("lens", [[40, 33], [1100]])
def test_selective_scan_before_position_zero(lens):
    """A live sequence whose rows' positions are below 0 starts anew, whole and in segments, as in the
    row form (steps of fewer than 16 rows a sequence)."""
    H, V, N, G, B = 4, 64, 64, 2, len(lens)
    inp = _scan_inputs(sum(lens), B, H, V, N, G, torch.bfloat16, 0, seed=sum(lens))
    q_start, pos, slot = _step(lens, [0] * B)
    step = (q_start, pos - 5, slot)
    want = _run_scan(inp, step, H, V, N, G, "cpu")
    got = _run_scan(inp, step, H, V, N, G, DEV)
    assert _rel(got[0], want[0]) < 2e-6 and _rel(got[1], want[1]) < 2e-6


def _run_retention(inp, step, H, D, V, offs, cs, l2, dev):
    proj, state = inp
    q_start, pos, slot = (t.to(dev) for t in step)
    st = state.clone().to(dev)
    buf = torch.zeros(proj.shape[0], H * V + 8, dtype=proj.dtype, device=dev)
    sops.retention(buf[:, :H * V], proj.to(dev), *offs, st, slot, pos, q_start,
                   None if cs is None else cs.to(dev), l2.to(dev), H, D, V, 1e-5)
    return buf[:, :H * V], st


@pytest.mark.parametrize("H,D,V,rot,dt", [(2, 128, 128, 64, torch.float32), (3, 64, 128, 0, torch.float32),
                                          (2, 128, 64, 128, torch.bfloat16),
                                          (4, 64, 64, 16, torch.bfloat16)])
@pytest.mark.parametrize("lens,starts", STEPS)
def test_retention_chunks(lens, starts, H, D, V, rot, dt):
    step = _step(lens, starts)
    T, B = sum(lens), len(lens)
    g = torch.Generator().manual_seed(T + D)
    # gate first, then q, k, v behind a few unused columns
    offs = (H * V + 8, H * V + 8 + H * D, H * V + 8 + 2 * H * D, 0)
    proj = torch.randn(T, 2 * H * V + 2 * H * D + 12, generator=g).to(dt)
    state = torch.randn(B, H, V, D, generator=g)
    l2 = torch.log2(torch.tensor([1.0, 0.97, 0.5, 0.999][:H]))
    ang = torch.arange(2048)[:, None] * (0.5 ** torch.arange(max(1, rot // 2)))[None, :]
    cs = torch.cat([torch.cos(ang), torch.sin(ang)], 1) if rot else None
    args = (step, H, D, V, (offs[0], offs[1], offs[2], offs[3]), cs, l2)
    want = _run_retention((proj, state), *args, "cpu")
    got = _run_retention((proj, state), *args, DEV)
    live = (step[2] >= 0)
    # bf16 outputs: one rounding to 8 bits (2^-9 relative) on either side
    assert _rel(got[0][live.to(DEV)].float(), want[0][live].float()) < (6e-3 if dt == torch.bfloat16
                                                                        else 4e-6)
    assert _rel(got[1], want[1]) < 2e-6


@pytest.mark.parametrize("lens,starts,_,H", CUT)
def test_retention_segments(lens, starts, _, H):
    D = V = 64
    T, B = sum(lens), len(lens)
    assert torch.ops.akap_stream.chunk_scan_segment(1, T, B, H, V) == 256
    step = _step(lens, starts)
    g = torch.Generator().manual_seed(T)
    proj, state = torch.randn(T, 4 * H * V, generator=g), torch.randn(B, H, V, D, generator=g)
    args = (step, H, D, V, (0, H * D, 2 * H * D, 3 * H * D), None,
            torch.log2(torch.linspace(0.9, 0.999, H)))
    want = _run_retention((proj, state), *args, "cpu")
    got = _run_retention((proj, state), *args, DEV)
    live = step[2] >= 0
    assert _rel(got[0][live.to(DEV)], want[0][live]) < 4e-6
    for b in range(B):
        if starts[b] >= 0:
            assert _rel(got[1][b], want[1][b]) < 1e-5
        else:
            assert torch.equal(got[1][b].cpu(), state[b])


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_chunks_values_not_finite(bad):
    """A value that is not finite reaches the rows from its own on and no row before it, in its
    column of its head alone."""
    H, V, N, G = 2, 64, 64, 1
    lens, starts = [70, 40], [0, 0]
    step = _step(lens, starts)
    inp = _scan_inputs(110, 2, H, V, N, G, torch.float32, 0, seed=3)
    inp[0][45, 10] = bad
    want = _run_scan(inp, step, H, V, N, G, "cpu")[0]
    got = _run_scan(inp, step, H, V, N, G, DEV)[0].cpu()
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    ok = torch.isfinite(want)
    assert _rel(got[ok], want[ok]) < 2e-6
    proj = torch.randn(110, 4 * H * V, generator=torch.Generator().manual_seed(4))
    proj[45, 2 * H * V + 10] = bad
    args = (step, H, V, V, (0, H * V, 2 * H * V, 3 * H * V), None, torch.log2(torch.tensor([0.9, 0.5])))
    st = torch.zeros(2, H, V, V)
    want = _run_retention((proj, st), *args, "cpu")[0]
    got = _run_retention((proj, st), *args, DEV)[0].cpu()
    # (the head's norm spreads it over the head's row, as zeros or as NaN: which of the two hangs on
    # whether the product of the row with itself is formed before or after the state's)
    ok = torch.ones(110, H * V, dtype=torch.bool)
    ok[45:70, :V] = False
    assert bool(torch.isfinite(got[ok]).all()) and not bool(torch.isfinite(got[45:70, 10]).any())
    assert _rel(got[ok], want[ok]) < 4e-6


def test_scan_decays_to_zero():
    """Step sizes that take a decay to zero inside a chunk (its logarithm far below fp32's range)."""
    H, V, N, G = 2, 64, 64, 1
    step = _step([96], [4])
    inp = list(_scan_inputs(96, 1, H, V, N, G, torch.float32, 0, seed=8))
    inp[1] = inp[1].clone()
    inp[1][40] = 3000.0
    inp[1][41] = 3.0e4
    inp[3] = torch.tensor([3.0, math.log(1e5)])
    want = _run_scan(tuple(inp), step, H, V, N, G, "cpu")
    got = _run_scan(tuple(inp), step, H, V, N, G, DEV)
    # (outputs grow by the step sizes: compared row by row, the largest relative to its row)
    d = (got[0].cpu() - want[0]).norm(dim=1) / want[0].norm(dim=1)
    assert float(d.max()) < 5e-6
    assert _rel(got[1], want[1]) < 5e-6


def test_scan_output_error():
    """Outputs against float64 from the same fp32 inputs, keys and queries of mostly one sign (as they come
    out of the convolution's silu).  A float32 model of the sums, each with its own rounding, gives 8.5e-8
    with the 128 products of q . k in short chains that meet in fp64, 1.2e-7 in chains of 32 that meet in
    fp32; the row-by-row form has 9.4e-8."""
    H, V, N, T = 32, 64, 128, 256
    g = torch.Generator().manual_seed(12)
    xbc = torch.nn.functional.silu(torch.randn(T, H * V + 2 * N, generator=g) * 0.6)
    inp = (xbc, torch.randn(T, H, generator=g), torch.randn(H, generator=g) * 0.5 - 1.0,
           torch.randn(H, generator=g) * 0.5, torch.zeros(H), torch.randn(1, H, N, V, generator=g) * 0.3)
    y, state = _run_scan(inp, _step([T], [5]), H, V, N, 1, DEV)
    x, k, q = (t.double() for t in xbc.split([H * V, N, N], 1))
    dt = torch.nn.functional.softplus(inp[1].double() + inp[2].double(), threshold=1000.0)
    decay = torch.exp(-torch.exp(inp[3].double()) * dt)
    S, want = inp[5][0].double(), []
    for t in range(T):
        S = decay[t, :, None, None] * S + \
            (dt[t, :, None] * k[t])[:, :, None] * x[t].view(H, 1, V)
        want.append((q[t] @ S).view(-1))
    assert _rel(y, torch.stack(want)) < 1.02e-7
    assert _rel(state[0], S) < 1e-7


@pytest.mark.parametrize("lens", [[700], [64] * 8, [2100], [300] * 5, [1] * 60 + [1500], [1] * 150 + [1600],
                                  [16] * 40])
@pytest.mark.parametrize("H,KH", [(8, 1), (64, 8)])
def test_scratch_stays_below_what_the_cache_leaves(lens, H, KH):
    """What a call asks the allocator for is within the bound that the cache's size leaves room for, and a
    matrix-form step takes more than an eighth of that (segments or not)."""
    V, N, T, B = 64, 64, sum(lens), len(lens)
    q_start, pos, slot = (t.to(DEV) for t in _step(lens, [0] * B))
    xbc, proj = torch.zeros(T, H * V + 2 * KH * N, device=DEV), torch.zeros(T, 4 * H * V, device=DEV)
    state, one, y = torch.zeros(B, H, V, N, device=DEV), torch.ones(H, device=DEV), torch.empty(T, H * V, device=DEV)

    def took(f):
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_stats()["requested_bytes.all.current"]
        f()
        return torch.cuda.memory_stats()["requested_bytes.all.peak"] - before

    n = took(lambda: sops.selective_scan(y, xbc, proj, 0, one, one, one, state, slot, pos, q_start, H, V,
                                         N, KH))
    most = sops.recurrence_scratch_bytes(T, B, H, KH, V, N, True)
    assert n <= most and (T < 16 * B or n > most / 8)
    decay = -one
    n = took(lambda: sops.retention(y, proj, 0, H * V, 2 * H * V, 3 * H * V, state, slot, pos, q_start,
                                    None, decay, H, N, V, 1e-5))
    most = sops.recurrence_scratch_bytes(T, B, H, H, V, N, False)
    assert n <= most and (T < 16 * B or n > most / 8)


def _marked(rows, what):
    """Scan inputs over `rows` rows, one operand with entries that do not split into three bf16 parts."""
    H, V, N = 2, 64, 128
    inp = list(_scan_inputs(rows, 1, H, V, N, 1, torch.float32, 0, seed=11))
    xbc, state = inp[0].clone(), inp[5].clone()
    inp[2] = inp[2] - 3.0                              # steps below 1: no product with one overflows
    x, k, q = xbc.split([H * V, N, N], 1)
    big = 3.395e38                                     # above bf16's largest, finite
    if what == "keys":
        k[:, 5], q[:, 5] = big, 1e-30
        x *= 1e-30
    elif what == "queries":
        q[40, 7], k[:, 7] = big, 1e-36
        state[:, :, 7] *= 1e-36
    elif what == "values":
        x[:, 9], k[:] = big, k * 1e-36
    elif what == "state":
        state[0, 0, 3, 8], q[:, 3] = big, 1e-36
    elif what == "small":
        x *= 1e-36
        state *= 1e-36
    else:                                              # an entry of that operand is not finite
        name, v = what.split()
        {"keys": k, "queries": q}.get(name, x)[40, 6] = float(v)
        if name == "state":
            x[40, 6] = 0.5
            state[0, 1, 4, 9] = float(v)
    inp[0], inp[5] = xbc, state
    return tuple(inp), H, V, N


@pytest.mark.parametrize("rows", [49, 300, 1100])
@pytest.mark.parametrize("what", ["keys", "queries", "values", "state", "small", "keys inf", "keys nan",
                                  "queries -inf", "state inf", "state nan"])
def test_operands_that_do_not_split(what, rows):
    """Magnitudes past bf16's, values that are not finite, and values whose parts are denormal: the same
    numbers as row by row, and the same entries not finite.  Sums in another order over about 150 fp32
    terms: 2e-6 of a head's row; of the small ones 1e-5, as their last bits are denormal."""
    inp, H, V, N = _marked(rows, what)
    step = _step([rows], [6])
    want = _run_scan(inp, step, H, V, N, 1, "cpu")
    got = _run_scan(inp, step, H, V, N, 1, DEV)
    for a, b in zip(got[:2], want[:2]):
        a, ok = a.cpu(), torch.isfinite(b)
        assert torch.equal(torch.isfinite(a), ok)
        scale = float(b[ok].abs().max())
        assert _rel(a[ok].double() / scale, b[ok].double() / scale) < (1e-5 if what == "small" else 4e-6)


@pytest.mark.parametrize("what", ["values inf", "values nan", "keys inf", "keys large"])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_retention_operands_that_do_not_split(what, dt):
    """The state after the step, whose entries no norm mixes: a key that is not finite spoils its row of
    the state, a value its column."""
    H, V, T = 2, 128, 100
    g = torch.Generator().manual_seed(5)
    proj = torch.randn(T, 4 * H * V, generator=g).to(dt)
    name, v = what.split()
    proj[37, (2 if name == "values" else 1) * H * V + 11] = {"large": 3e38}.get(v) or float(v)
    args = (_step([T], [3]), H, V, V, (0, H * V, 2 * H * V, 3 * H * V), None,
            torch.log2(torch.tensor([0.97, 0.5])))
    st = torch.randn(1, H, V, V, generator=g)
    want = _run_retention((proj, st), *args, "cpu")[1]
    got = _run_retention((proj, st), *args, DEV)[1].cpu()
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), ok)
    scale = float(want[ok].abs().max())
    assert _rel(got[ok].double() / scale, want[ok].double() / scale) < 4e-6


# lengths at whole segments of 64 and 128 rows and one beside them, continued and not; heads that take each
@pytest.mark.parametrize("lens,starts", [([384, 1, 257, 420], [3, 0, 0, 8]), ([1025, 512, 63], [0, 5, 2])])
@pytest.mark.parametrize("mode,H,piece", [(0, 8, 64), (0, 56, 128), (1, 4, 64), (1, 28, 128), (1, 64, 256)])
def test_shorter_segments(lens, starts, mode, H, piece):
    V = N = 64
    T, B = sum(lens), len(lens)
    step = _step(lens, starts)
    assert torch.ops.akap_stream.chunk_scan_piece(mode, T, B, H, V) == piece
    g = torch.Generator().manual_seed(T + H)
    if mode == 0:
        inp = _scan_inputs(T, B, H, V, N, 2, torch.bfloat16, 0, seed=T)
        want = _run_scan(inp, step, H, V, N, 2, "cpu")
        got = _run_scan(inp, step, H, V, N, 2, DEV)
    else:
        proj, state = torch.randn(T, 4 * H * V, generator=g), torch.randn(B, H, V, N, generator=g)
        args = (step, H, N, V, (0, H * V, 2 * H * V, 3 * H * V), None,
                torch.log2(torch.linspace(0.9, 0.999, H)))
        want = _run_retention((proj, state), *args, "cpu")
        got = _run_retention((proj, state), *args, DEV)
    assert _rel(got[0], want[0]) < (2e-6 if mode == 0 else 4e-6)
    for b in range(B):
        assert _rel(got[1][b], want[1][b]) < 1e-5


@pytest.mark.parametrize("T", [5, 130, 1500, 3300])
@pytest.mark.parametrize("C,taps", [(1040, 4), (6200, 2)])
def test_convolution_rows(T, C, taps):
    """Every number of rows that a workgroup of the convolution takes, over sequence ends."""
    lens = [T - T // 3 - 1, 1, T // 3]
    q_start, pos, slot = _step(lens, [3, 0, 4])
    g = torch.Generator().manual_seed(T)
    proj = torch.randn(T, C + 8, generator=g).to(torch.bfloat16)
    w, b = torch.randn(C, taps, generator=g), torch.randn(C, generator=g)
    state = torch.randn(3, taps - 1, C, generator=g).to(torch.bfloat16)
    got = []
    for dev in ("cpu", DEV):
        st, out = state.clone().to(dev), torch.zeros(T, C, device=dev)
        sops.conv_silu(out, proj.to(dev), 8, w.to(dev), b.to(dev), st, slot.to(dev), pos.to(dev),
                       q_start.to(dev))
        got.append((out.cpu(), st.cpu()))
    assert _rel(got[1][0], got[0][0]) < 1e-6        # four products in fp32 and an exponential
    assert torch.equal(got[1][1], got[0][1])


@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C,first", [(8, 5), (1016, 509), (1024, 600), (1032, 1027), (3080, 0)])
def test_convolution_columns(C, first, out):
    """Columns of a workgroup that is not full, and the first one with an activation in either half."""
    T, taps = 45, 4
    q_start, pos, slot = _step([40, 5], [0, 7])
    g = torch.Generator().manual_seed(C)
    proj = torch.randn(T, C + 16, generator=g).to(torch.bfloat16)
    w, b = torch.randn(C, taps, generator=g), torch.randn(C, generator=g)
    state = torch.randn(2, taps - 1, C, generator=g).to(torch.bfloat16)
    got = []
    for dev in ("cpu", DEV):
        st, o = state.clone().to(dev), torch.zeros(T, C, dtype=out, device=dev)
        sops.conv_silu(o, proj.to(dev), 8, w.to(dev), b.to(dev), st, slot.to(dev), pos.to(dev),
                       q_start.to(dev), first)
        got.append((o.cpu(), st.cpu()))
    # four products in fp32 and an exponential; bf16 neighbours differ by up to 2^-7
    d = (got[1][0].double() - got[0][0].double()).abs()
    ulp = 2e-6 if out == torch.float32 else 2.0 ** -7
    assert (d <= ulp * (got[0][0].double().abs() + 1)).all()
    assert torch.equal(got[1][1], got[0][1])


def _beside(rows, what):
    """Scan inputs of ordinary sizes where one operand has entries of 1e-36 between larger ones, whose last
    bits are denormal, and the other has ones large enough to make them count, in one row of the state."""
    H, V, N = 2, 64, 128
    inp = list(_scan_inputs(rows, 1, H, V, N, 1, torch.float32, 0, seed=12))
    xbc, state, t = inp[0].clone(), inp[5].clone(), rows - 5
    inp[2] = inp[2] - 3.0
    x, k, q = xbc.split([H * V, N, N], 1)
    if what == "state":
        state[:, :, 3] *= 1e-36
        k[:, 3] = 0.0
        q[:, 3] *= 3e37
    elif what == "queries":
        state[:, :, 3] *= 3e37
        k[:, 3] = 0.0
        q[:, 3] = 0.0
        q[1, 3] = 1.2345e-36
    elif what == "keys":
        k[t] = 0.0
        k[t, 3], x[t] = 1.2345e-36, x[t] * 1e37
    else:                                              # the values of a token
        k[t] = 0.0
        k[t, 3], x[t] = 1e37, x[t] * 1e-36
    inp[0], inp[5] = xbc, state
    return tuple(inp), H, V, N


@pytest.mark.parametrize("rows", [49, 300, 1100])
@pytest.mark.parametrize("what", ["state", "queries", "keys", "values"])
def test_small_operands_beside_larger_ones(what, rows):
    """A part that is denormal is not lost where the other operand is large: every operand as exact as in
    fp32, row by row of the state and of the outputs (sums of 160 fp32 terms in another order)."""
    inp, H, V, N = _beside(rows, what)
    step = _step([rows], [6])
    want = _run_scan(inp, step, H, V, N, 1, "cpu")
    got = _run_scan(inp, step, H, V, N, 1, DEV)
    err = (got[0].cpu() - want[0]).norm(dim=1) / want[0].norm(dim=1)
    assert float(err.max()) < 1e-5
    assert _rel(got[1][:, :, 3], want[1][:, :, 3]) < 4e-6
    assert _rel(got[1], want[1]) < 4e-6


@pytest.mark.parametrize("what", ["keys", "values", "denormal values"])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_retention_small_operands_beside_larger_ones(what, dt):
    """The same of the retention, whose values may be of one part alone, by the state's row of the key."""
    H, V, T = 2, 128, 96
    proj = torch.randn(T, 4 * H * V, generator=torch.Generator().manual_seed(6)).to(dt)
    k, v = proj[:, H * V:2 * H * V], proj[:, 2 * H * V:3 * H * V]
    k[80].zero_()
    if what == "keys":
        k[80, 11], v[80] = 1.2345e-36, v[80] * 1e37
    else:
        k[80, 11], v[80] = 1e37, v[80] * (1e-36 if what == "values" else 3e-39)
    args = (_step([T], [3]), H, V, V, (0, H * V, 2 * H * V, 3 * H * V), None,
            torch.log2(torch.tensor([0.97, 0.9])))
    st = torch.randn(1, H, V, V, generator=torch.Generator().manual_seed(7))
    want = _run_retention((proj, st), *args, "cpu")[1]
    got = _run_retention((proj, st), *args, DEV)[1].cpu()
    assert _rel(got, want) < 4e-6
    assert _rel(got[0, 0, :, 11], want[0, 0, :, 11]) < 4e-6


@pytest.mark.parametrize("a_log", [1.5, 2.5, 3.5])
def test_scan_weights_that_decay_far(a_log):
    """Decays that take the first rows of a chunk down to denormal weights in the state after it, with a
    value large enough to count among them."""
    H, V, N, rows = 2, 64, 128, 64
    inp = list(_scan_inputs(rows, 1, H, V, N, 1, torch.float32, 0, seed=13))
    inp[1], inp[2] = torch.zeros_like(inp[1]), torch.zeros(H)      # steps of log 2
    inp[3] = torch.full((H,), a_log)
    inp[0] = inp[0].clone()
    inp[0][rows - 9, :H * V] *= 1e15
    step = _step([rows], [6])
    want = _run_scan(tuple(inp), step, H, V, N, 1, "cpu")
    got = _run_scan(tuple(inp), step, H, V, N, 1, DEV)
    err = (got[0].cpu() - want[0]).norm(dim=1) / want[0].norm(dim=1)
    assert float(err.max()) < 1e-5 and _rel(got[1], want[1]) < 4e-6


# decays on both sides of the one from which keys times weights are scaled, ones whose weights run out, zero
@pytest.mark.parametrize("dt,V", [(torch.float32, 64), (torch.bfloat16, 128)])
@pytest.mark.parametrize("lens,starts", [([64, 33], [0, 5]), ([1100], [3])])
def test_retention_strong_decays(lens, starts, dt, V):
    """Tokens whose weight in the state is far below the last ones'.  Then a value among them so large that
    it counts all the same, for the states alone: rows that it rules and rows where it fades are normed, so
    their outputs say nothing about a single product."""
    H, D, T, B = 5, 128, sum(lens), len(lens)
    g = torch.Generator().manual_seed(T + V)
    proj = torch.randn(T, 2 * H * D + 2 * H * V, generator=g)
    state = torch.randn(B, H, V, D, generator=g)
    l2 = torch.log2(torch.tensor([0.42, 0.4, 0.05, 0.01, 0.0]))
    args = (_step(lens, starts), H, D, V, (0, H * D, 2 * H * D, 2 * H * D + H * V), None, l2)
    for large in (False, True):
        if large:
            proj[torch.tensor(lens).cumsum(0) - 17, 2 * H * D:2 * H * D + H * V] *= 3e30
        want = _run_retention((proj.to(dt), state), *args, "cpu")
        got = _run_retention((proj.to(dt), state), *args, DEV)
        for h in range(H):
            a, b = (y[0][:, h * V:(h + 1) * V].float() for y in (got, want))
            assert large or _rel(a, b) < (6e-3 if dt == torch.bfloat16 else 4e-6)
            assert _rel(got[1][:, h], want[1][:, h]) < 2e-6


def test_retention_strong_decays_take_no_longer():
    """Keys times weights split however small the weights are."""
    H, D, T = 8, 128, 4096
    g = torch.Generator(device=DEV).manual_seed(1)
    proj = torch.randn(T, 4 * H * D, device=DEV, generator=g).bfloat16()
    state, out = torch.randn(4, H, D, D, device=DEV, generator=g), proj.new_empty(T, H * D)
    q_start, pos, slot = (t.to(DEV) for t in _step([T // 4] * 4, [0] * 4))

    def time(decay):
        l2 = torch.full((H,), math.log2(decay), device=DEV)
        spent = []
        for _ in range(9):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                sops.retention(out, proj, 0, H * D, 2 * H * D, 3 * H * D, state, slot, pos, q_start, None,
                               l2, H, D, D, 1e-5)
            b.record()
            b.synchronize()
            spent.append(a.elapsed_time(b))
        return min(spent)
    usual = time(0.97)
    for decay in (0.2, 0.05, 0.01, 0.003):
        assert time(decay) < 1.3 * usual       # (3.6 times as long with its products in fp32)


@pytest.mark.parametrize("what", ["large values", "small pairs", "both"])
def test_retention_pair_weights_of_any_size(what):
    """bf16 values meet the products of queries and keys in three parts, which lose 2^-125 of a small one:
    outputs against 64 bits, with values of 1e12, products of 1e-30 and both, no further off than a rounding
    to bf16 on either side of the norm."""
    H, V, T = 2, 128, 70
    proj = torch.randn(T, 4 * H * V, generator=torch.Generator().manual_seed(8))
    if what != "large values":
        proj[:, :2 * H * V] *= 1e-15
    if what != "small pairs":
        proj[:, 2 * H * V:3 * H * V] *= 3e11
    proj = proj.bfloat16()
    l2 = torch.log2(torch.tensor([0.97, 0.3]))
    args = (_step([T], [0]), H, V, V, (0, H * V, 2 * H * V, 3 * H * V), None, l2)
    got = _run_retention((proj, torch.zeros(1, H, V, V)), *args, DEV)[0].cpu().double().view(T, H, V)
    q, k, v, gate = (t.view(T, H, V).transpose(0, 1) for t in proj.double().split(H * V, 1))
    i = torch.arange(T)
    w = torch.exp2((i[:, None] - i).clamp_min(0) * l2.double()[:, None, None]).tril()
    o = ((q @ k.transpose(1, 2)) * V ** -0.5 * w) @ v
    o = o / torch.sqrt((o * o).mean(2, keepdim=True) + 1e-5) * torch.nn.functional.silu(gate)
    assert _rel(got.transpose(0, 1), o) < 3e-3


@pytest.mark.parametrize("mode,lens,starts", [
    (0, [383, 129], [0, 7]), (0, [253], [3]), (1, [320, 129, 128, 257], [0, 4, 9, 0]), (1, [161], [0])])
def test_few_short_prompts_in_segments(mode, lens, starts):
    """Sequences of 129 rows and more in segments of 64 where all are short, beside one of 128, whole."""
    H, V, N, T, B = 4, 64, 64, sum(lens), len(lens)
    assert torch.ops.akap_stream.chunk_scan_segment(mode, T, B, H, V) == 128
    step = _step(lens, starts)
    if mode == 0:
        inp = _scan_inputs(T, B, H, V, N, 2, torch.bfloat16, 0, seed=T)
        want, got = (_run_scan(inp, step, H, V, N, 2, d) for d in ("cpu", DEV))
    else:
        g = torch.Generator().manual_seed(T)
        proj, state = torch.randn(T, 4 * H * V, generator=g), torch.randn(B, H, V, N, generator=g)
        args = (step, H, N, V, (0, H * V, 2 * H * V, 3 * H * V), None,
                torch.log2(torch.linspace(0.9, 0.999, H)))
        want, got = (_run_retention((proj, state), *args, d) for d in ("cpu", DEV))
    assert _rel(got[0], want[0]) < 4e-6
    for b in range(B):
        assert _rel(got[1][b], want[1][b]) < 1e-5


@pytest.mark.parametrize("D,V,rot", [(128, 128, 64), (128, 64, 40), (64, 128, 32), (64, 64, 8)])
@pytest.mark.parametrize("what", ["usual", "small keys", "odd key", "odd query"])
def test_retention_entries_that_do_not_turn(D, V, rot, what):
    """bf16 rows of which at most half the entries turn keep the others in one part, with a power of two of their
    weights; the same rows in fp32 go the general way.  Keys of 2^-100 are too small for that and infinite ones do
    not split; those of 2^-60 and of 3e38 do.  Outputs: a rounding to bf16; states: both sides sum in fp32 (module
    comment)."""
    H, lens, starts = 4, [1, 33, 300, 64], [9, 0, 5, 0]
    T, B = sum(lens), len(lens)
    g = torch.Generator().manual_seed(D + V + rot)
    proj = torch.randn(T, 2 * H * D + 2 * H * V, generator=g)
    q, k = (proj[:, i * H * D:(i + 1) * H * D].view(T, H, D) for i in range(2))
    if what == "small keys":
        k[:, 0, rot:] *= 2.0 ** -60
        k[::3, 1, D - 1] *= 2.0 ** -100
    elif what == "odd key":
        k[-3, 0, D - 1], k[40, 1, rot] = float("inf"), 3e38
    elif what == "odd query":
        q[-3, 0, D - 1], q[40, 1, rot] = float("nan"), 2.0 ** -110
    proj = proj.bfloat16()
    state = torch.randn(B, H, V, D, generator=g)
    ang = torch.arange(2048)[:, None] * (0.5 ** torch.arange(rot // 2))[None, :]
    args = (_step(lens, starts), H, D, V, (0, H * D, 2 * H * D, 2 * H * D + H * V),
            torch.cat([torch.cos(ang), torch.sin(ang)], 1), torch.log2(torch.tensor([0.97, 0.42, 0.2, 0.999])), DEV)
    got, want = _run_retention((proj, state), *args), _run_retention((proj.float(), state), *args)
    for a, b, limit in zip((got[0].float(), got[1]), want, (3e-3, 2e-6)):
        ok = torch.isfinite(b)
        assert torch.equal(torch.isfinite(a), ok)
        # (a product of 3e38 rules its head's sums: heads apart)
        for h in range(H):
            part = (slice(None), slice(h * V, (h + 1) * V)) if a.dim() == 2 else (slice(None), h)
            assert _rel(torch.where(ok, a, 0.)[part], torch.where(ok, b, 0.)[part].cpu()) < limit


@pytest.mark.parametrize("what,decay,size", [
    ("values", 0.42, 1.2e-36), ("values", 0.06, 1.3e-9),
    ("denormal values", 0.97, 3e-39), ("large values", 0.42, 1e13), ("large values", 0.06, 1e13),
    ("small keys", 0.42, 1e-25), ("small keys", 0.06, 1e-17), ("odd", 0.42, 1.2e-36)])
@pytest.mark.parametrize("V", [64, 128])
@pytest.mark.parametrize("T", [96, 1120])
def test_retention_small_operands_that_do_not_turn(T, V, what, decay, size):
    """The oldest row of a chunk of bf16, whose weight in the state is the smallest, with a value or a key of
    any size, alone in one row of the state of an entry that does not turn, beside a key or a value that makes
    it count: as exact as the operands in fp32.  (The row form rounds the entry 31 times and has the decay's own
    rounding 31 times, 3.7e-6 in all; a weight's exponent of up to 126 is rounded to 2^-18, 2.6e-6 of the weight;
    some roundings of the products besides.)"""
    H, row, at = 2, T - 32, 3 * V // 4 + 4
    proj = torch.randn(T, 4 * H * V, generator=torch.Generator().manual_seed(16)).bfloat16()
    k, v = proj[:, H * V:2 * H * V], proj[:, 2 * H * V:3 * H * V]
    k[:, at] = 0.0
    k[row, at], v[row] = (size, v[row] * 1e30) if what == "small keys" else (1e37, v[row] * size)
    if what == "large values":
        k[row, at] = 1.0
    elif what == "odd":
        k[row + 1, at - 1] = float("inf")
    args = (_step([T], [0]), H, V, V, (0, H * V, 2 * H * V, 3 * H * V), None,
            torch.log2(torch.tensor([decay, 0.9])))
    st = torch.zeros(1, H, V, V)
    want = _run_retention((proj, st), *args, "cpu")[1][0, 0, :, at]
    got = _run_retention((proj, st), *args, DEV)[1].cpu()[0, 0, :, at]
    assert float(want.abs().max()) > 0
    assert float(((got - want).abs() - 8e-6 * want.abs()).max()) <= 0


def test_retention_small_keys_take_no_longer():
    """Keys that one bf16 part holds do not send a chunk through the fp32 products, however small they are."""
    H, D, T = 8, 128, 4096
    g = torch.Generator(device=DEV).manual_seed(1)
    proj = torch.randn(T, 4 * H * D, device=DEV, generator=g)
    state, out = torch.randn(4, H, D, D, device=DEV, generator=g), proj.new_empty(T, H * D).bfloat16()
    q_start, pos, slot = (t.to(DEV) for t in _step([T // 4] * 4, [0] * 4))
    l2 = torch.full((H,), math.log2(0.97), device=DEV)

    def time(rows):
        spent = []
        for _ in range(9):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                sops.retention(out, rows, 0, H * D, 2 * H * D, 3 * H * D, state, slot, pos, q_start, None,
                               l2, H, D, D, 1e-5)
            b.record()
            b.synchronize()
            spent.append(a.elapsed_time(b))
        return min(spent)
    usual = time(proj.bfloat16())
    for size in (2.0 ** -60, 2.0 ** -90):
        proj[:, H * D:2 * H * D].view(T, H, D)[::7, :, D - 3] = size
        assert time(proj.bfloat16()) < 1.3 * usual      # (3.6 times as long with its products in fp32)


@pytest.mark.parametrize("D,V,rot", [(128, 128, 64), (64, 64, 32), (128, 64, 128), (64, 128, 64), (128, 128, 96)])
@pytest.mark.parametrize("lens,starts", [([700, 420], [5, 0]), ([300, 161, 33], [0, 4, 2])])
def test_retention_segments_of_turned_rows(D, V, rot, lens, starts):
    """bf16 rows in segments, half of the entries turned and more, against the same rows in fp32."""
    H, T, B = 4, sum(lens), len(lens)
    assert torch.ops.akap_stream.chunk_scan_segment(1, T, B, H, V) > 0
    g = torch.Generator().manual_seed(D + V + rot)
    proj = torch.randn(T, 2 * H * D + 2 * H * V, generator=g).bfloat16()
    state = torch.randn(B, H, V, D, generator=g)
    ang = torch.arange(2048)[:, None] * (0.5 ** torch.arange(rot // 2))[None, :]
    args = (_step(lens, starts), H, D, V, (0, H * D, 2 * H * D, 2 * H * D + H * V),
            torch.cat([torch.cos(ang), torch.sin(ang)], 1), torch.log2(torch.tensor([0.97, 0.42, 0.2, 0.999])), DEV)
    got, want = _run_retention((proj, state), *args), _run_retention((proj.float(), state), *args)
    for h in range(H):
        part = slice(h * V, (h + 1) * V)
        assert _rel(got[0].float()[:, part], want[0][:, part].cpu()) < 3e-3
        assert _rel(got[1][:, h], want[1][:, h].cpu()) < 2e-6
