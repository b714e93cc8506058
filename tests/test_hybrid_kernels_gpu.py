"""HIP kernels of the hybrid decoders against their fp32 PyTorch references
(``ops.reference``), op by op, in bf16 and fp32, on sizes that are not multiples of the
wave (odd head sizes, several norm groups, chunks that continue a slot's state)."""
import math
import re
import types

import pytest
import torch

from kubernetes_gpu_cluster_amd import ops
from kubernetes_gpu_cluster_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DT = [torch.bfloat16, torch.float32]


def _tol(dt):
    return dict(rtol=2e-2, atol=2e-2) if dt == torch.bfloat16 else dict(rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("W,G", [(352, 2), (384, 3), (1024, 1)])
def test_group_norm_and_add(gpu, dt, W, G):
    torch.manual_seed(0)
    x = torch.randn(37, W) * 3
    y = torch.randn(37, W).to(dt)
    w = torch.rand(W) + 0.5
    want_x = x + y.float()
    want = ref.group_rms_norm(want_x, w, G, 1e-5, dt)
    xg = x.to(gpu)
    got = ops.group_rms_norm(xg, w.to(gpu), G, 1e-5, dt, add=y.to(gpu))
    torch.testing.assert_close(xg.cpu(), want_x)
    torch.testing.assert_close(got.cpu().float(), want.float(), **_tol(dt))
    got2 = ops.group_rms_norm(xg, w.to(gpu), G, 1e-5, dt)
    torch.testing.assert_close(got2.cpu().float(), want.float(), **_tol(dt))


@pytest.mark.parametrize("dt", DT)
def test_depth_mix_norm(gpu, dt):
    torch.manual_seed(1)
    L, cap, T, W, G, layer = 5, 16, 11, 192, 3, 3
    hist = torch.randn(L + 1, cap, W)
    x = torch.randn(T, W)
    y = torch.randn(T, W).to(dt)
    coef = torch.randn(layer + 2)
    w = torch.rand(W) + 0.5
    h_ref, x_ref = hist.clone(), x.clone()
    want = ops.depth_mix_norm(x_ref, h_ref, layer, y, coef, w, G, 1e-5, dt)
    hg, xg = hist.to(gpu), x.to(gpu)
    got = ops.depth_mix_norm(xg, hg, layer, y.to(gpu), coef.to(gpu), w.to(gpu), G, 1e-5, dt)
    torch.testing.assert_close(hg.cpu(), h_ref, rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(xg.cpu(), x_ref, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(got.cpu().float(), want.float(), **_tol(dt))


@pytest.mark.parametrize("W,G", [(192, 3), (512, 2), (2044, 1), (2048, 1), (4352, 1), (8192, 4)])
@pytest.mark.parametrize("layers", [3, 7, 12])
def test_depth_mix_sums_begun_ahead(gpu, W, G, layers):
    """The same rows, results and normed rows to the bit, whichever layer began a sum."""
    torch.manual_seed(layers)
    T, cap, dt = 5, 9, torch.bfloat16
    ys = [torch.randn(T, W).to(dt).to(gpu) for _ in range(layers)]
    dwa = [torch.randn(i + 2).to(gpu) for i in range(layers)]
    w = (torch.rand(W) + 0.5).to(gpu)
    start = torch.randn(T, W).to(gpu)
    out = []
    for plan in ([(None, 0)] * layers, ops.depth_mix_plan(layers)):
        hist, x, rows = torch.full((layers + 1, cap, W), 7.0, device=gpu), start.clone(), []
        sums = torch.full((3, cap, W), 7.0, device=gpu)
        hist[0, :T] = start
        for i, (take, n) in enumerate(plan):
            h = ops.depth_mix_norm(x, hist, i, ys[i], dwa[i], w, G, 1e-5, dt, sums, take, dwa[i + 1: i + 1 + n])
            rows += [h, x.clone()]
        assert (hist[:, T:] == 7).all() and (sums[:, T:] == 7).all()
        out.append(rows + [hist])
    assert any(n for _, n in plan)
    for a, b in zip(*out):
        assert torch.equal(a, b)
    # and the sums themselves, from fp32 on the CPU
    hc, sc, xc = hist.cpu(), torch.zeros(3, cap, W), start.cpu()
    for i, (take, n) in enumerate(plan):
        h = ops.depth_mix_norm(xc, hc, i, ys[i].cpu(), dwa[i].cpu(), w.cpu(), G, 1e-5, dt, sc, take,
                               [c.cpu() for c in dwa[i + 1: i + 1 + n]])
        bound = 2.0 ** -22 * (i + 2) * sum(c.abs() * r.abs() for c, r in zip(dwa[i].cpu(), hc[:, :T]))
        assert ((out[1][2 * i + 1].cpu() - xc).abs() <= bound + 2.0 ** -20).all()
        xc = out[1][2 * i + 1].cpu().clone()


def test_depth_mix_registered_op(gpu):
    """The registered op without sums of following layers takes the arguments that it always took."""
    torch.manual_seed(5)
    W, T, dt = 256, 3, torch.bfloat16
    start, hist, y = torch.randn(T, W).to(gpu), torch.randn(4, T, W).to(gpu), torch.randn(T, W).to(dt).to(gpu)
    c, w, x, out = torch.randn(3).to(gpu), torch.rand(W).to(gpu), start.clone(), torch.empty(T, W, dtype=dt, device=gpu)
    h, r = hist.clone(), start.clone()
    torch.ops.kgc.depth_mix_norm(out, x, hist, y, c, w, 1, 1, 1e-5)
    assert torch.equal(out, ops.depth_mix_norm(r, h, 1, y, c, w, 1, 1e-5, dt))
    assert torch.equal(x, r) and torch.equal(hist, h) and not torch.equal(x, start)


def test_depth_mix_refuses_sums_that_do_not_fit(gpu):
    W, T, dt = 256, 3, torch.bfloat16
    x, hist, w = torch.zeros(T, W, device=gpu), torch.zeros(4, T, W, device=gpu), torch.ones(W, device=gpu)
    y, c, sums = torch.zeros(T, W, dtype=dt, device=gpu), torch.ones(5, device=gpu), torch.zeros(1, T, W, device=gpu)
    call = lambda *a: ops.depth_mix_norm(x, hist, 1, y, c[:3], w, 1, 1e-5, dt, *a)   # noqa: E731
    call(sums, (0, 2))
    for bad in ((sums, (1, 2)), (sums, (0, 3)), (sums, (0, 2), [c]), (sums, None, [c, c]), (sums, None, [c[:2]]),
                (sums[:, :2], None, [c]), (sums[..., :128], None, [c]), (sums.double(), (0, 2))):
        with pytest.raises(RuntimeError):
            call(*bad)


@pytest.mark.parametrize("dt", DT)
def test_xielu_gate_proj_head_norm(gpu, dt):
    torch.manual_seed(2)
    z = (torch.randn(9, 200) * 3).to(dt)
    ab = torch.tensor([0.7, 1.3])
    torch.testing.assert_close(ops.xielu(z.to(gpu), ab.to(gpu)).cpu().float(),
                               ref.xielu(z, ab).float(), **_tol(dt))
    h = torch.randn(13, 288).to(dt)
    w = (torch.randn(10, 288) * 0.2).to(dt)
    b = torch.randn(10)
    want = ref.gate_proj(h, w, b, ops.GATE_CAP_TANH, ops.GATE_LOGSIG_CAP_TANH, 5, 15.0)
    got = ops.gate_proj(h.to(gpu), w.to(gpu), b.to(gpu), ops.GATE_CAP_TANH,
                        ops.GATE_LOGSIG_CAP_TANH, 5, 15.0)
    torch.testing.assert_close(got.cpu(), want, rtol=1e-4, atol=1e-4)
    got = ops.gate_proj(h.to(gpu), w.to(gpu), None, ops.GATE_SIGMOID)
    torch.testing.assert_close(got.cpu(), ref.gate_proj(h, w, None, 0, 0, 10, 1.0), rtol=1e-4,
                               atol=1e-4)
    H, dv = 3, 40
    o = torch.randn(7, H * dv) * 5
    big = torch.randn(7, 300).to(dt)
    g = big[:, 100:100 + H * dv]
    nw = torch.rand(H * dv) + 0.5
    want = ref.head_norm_gate(o, g, nw, H, 1e-5, dt)
    got = ops.head_norm_gate(o.to(gpu), big.to(gpu)[:, 100:100 + H * dv], nw.to(gpu), H, 1e-5, dt)
    torch.testing.assert_close(got.cpu().float(), want.float(), **_tol(dt))


def _meta(P_q, P_sl, D_ctx, tables, slots=None):
    """AttnMetadata stand-in: prefill chunks (query lens, seq lens) then decode rows."""
    m = types.SimpleNamespace()
    P, D = len(P_q), len(D_ctx)
    m.num_prefills, m.num_decodes, m.num_prefill_tokens = P, D, sum(P_q)
    qsl = [0]
    for q in P_q:
        qsl.append(qsl[-1] + q)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32)   # noqa: E731
    m.query_start_loc = i32(qsl) if P else None
    m.prefill_seq_lens = i32(P_sl) if P else None
    m.prefill_block_tables = tables[:P].contiguous() if P else None
    m.decode_ctx_lens = i32(D_ctx) if D else None
    m.decode_block_tables = tables[P:P + D].contiguous() if D else None
    m.state_slots = i32(slots) if slots is not None else None
    return m


def _to(m, dev):
    out = types.SimpleNamespace(**vars(m))
    for k, v in vars(m).items():
        if torch.is_tensor(v):
            setattr(out, k, v.to(dev))
    return out


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,G,dk,dv,rot,window,keep", [(6, 2, 40, 24, 16, 9, 3), (4, 4, 64, 64, 64, 0, 0),
                                                        (8, 1, 96, 128, 32, 70, 5)])
def test_rope_store_and_window_attention(gpu, dt, H, G, dk, dv, rot, window, keep):
    torch.manual_seed(3)
    bs, nb = 8, 64
    # two prefill chunks (one continuing at position 50, one fresh) and two decode rows
    P_q, P_sl, D_ctx = [13, 21], [63, 21], [90, 7]
    T = sum(P_q) + len(D_ctx)
    perm = torch.randperm(nb - 1)[:4 * 12].view(4, 12) + 1
    tables = perm.to(torch.int32)
    kc = torch.randn(nb, G, bs, dk).to(dt)
    vc = torch.randn(nb, G, bs, dv).to(dt)
    m = _meta(P_q, P_sl, D_ctx, tables)
    pos = torch.cat([torch.arange(50, 63), torch.arange(0, 21), torch.tensor([89, 6])])
    seq_of = [0] * 13 + [1] * 21 + [2, 3]
    slots = torch.tensor([int(tables[s, p // bs]) * bs + p % bs for s, p in zip(seq_of, pos.tolist())])
    qkv = torch.randn(T, (H + G) * dk + G * dv).to(dt)
    table = ref.rope_table(rot, 128, 10000.0)
    gate = torch.rand(T, H)
    kc_r, vc_r = kc.clone(), vc.clone()
    q_r = ops.rope_kv_store(qkv, pos, table, kc_r, vc_r, slots, H, G, dk, dv)
    want = ops.window_attention(q_r, kc_r, vc_r, pos, m, 0.11, window, keep, gate)
    kc_g, vc_g = kc.to(gpu), vc.to(gpu)
    q_g = ops.rope_kv_store(qkv.to(gpu), pos.to(gpu), table.to(gpu), kc_g, vc_g, slots.to(gpu),
                            H, G, dk, dv)
    tol = _tol(dt)
    torch.testing.assert_close(q_g.cpu().float(), q_r.float(), **tol)
    torch.testing.assert_close(kc_g.cpu().float(), kc_r.float(), **tol)
    torch.testing.assert_close(vc_g.cpu().float(), vc_r.float(), rtol=0, atol=0)
    got = ops.window_attention(q_r.to(gpu), kc_r.to(gpu), vc_r.to(gpu), pos.to(gpu), _to(m, gpu),
                               0.11, window, keep, gate.to(gpu))
    torch.testing.assert_close(got.cpu().float(), want.float(), **tol)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,d,dv", [(3, 24, 40), (2, 80, 64), (1, 136, 200)])
def test_mlstm_scan(gpu, dt, H, d, dv):
    torch.manual_seed(4)
    slots_n = 5
    # chunk continuing slot 3 (position 17), fresh chunk in slot 0, a padding sequence
    # (slot -1), decode rows continuing slots 4 and 1 (one of them at position 0)
    P_q, P_sl, D_ctx = [9, 14, 4], [26, 14, 4], [31, 1]
    slot_ids = [3, 0, -1, 4, 1]
    T = sum(P_q) + len(D_ctx)
    m = _meta(P_q, P_sl, D_ctx, torch.zeros(5, 1, dtype=torch.int32), slot_ids)
    S = torch.randn(slots_n, H, d, dv) * 0.3
    n = torch.randn(slots_n, H, d) * 0.3
    mm = torch.rand(slots_n, H) * 2
    qkvg = torch.randn(T, 2 * H * d + 2 * H * dv).to(dt)
    gates = torch.cat([torch.randn(T, H) * 2, -torch.rand(T, H) * 2], dim=1)
    st_r = (S.clone(), n.clone(), mm.clone())
    want = ops.mlstm_scan(qkvg, gates, st_r, m, H, d, dv)
    st_g = (S.to(gpu), n.to(gpu), mm.to(gpu))
    got = ops.mlstm_scan(qkvg.to(gpu), gates.to(gpu), st_g, _to(m, gpu), H, d, dv)
    torch.testing.assert_close(got.cpu(), want, rtol=2e-4, atol=2e-4)
    for a, b in zip(st_g, st_r):
        torch.testing.assert_close(a.cpu(), b, rtol=2e-4, atol=2e-4)


def test_mlstm_scan_many_workgroups(gpu):
    """More workgroups than the chip holds at once: those of a head's later columns begin after
    the first one has written n and m back, and still start from the incoming ones."""
    torch.manual_seed(14)
    B, H, d, dv = 192, 4, 64, 512
    m = _meta([], [], [50] * B, torch.zeros(B, 1, dtype=torch.int32), torch.randperm(B).tolist())
    st = (torch.randn(B, H, d, dv) * 0.3, torch.randn(B, H, d) * 0.3, torch.rand(B, H) * 2)
    qkvg = torch.randn(B, 2 * H * d + 2 * H * dv)
    gates = torch.cat([torch.randn(B, H) * 2, -torch.rand(B, H) * 2], dim=1)
    st_g = tuple(x.to(gpu) for x in st)
    want = ops.mlstm_scan(qkvg, gates, st, m, H, d, dv)
    got = ops.mlstm_scan(qkvg.to(gpu), gates.to(gpu), st_g, _to(m, gpu), H, d, dv)
    torch.testing.assert_close(got.cpu(), want, rtol=2e-4, atol=2e-4)
    for a, b in zip(st_g, st):
        torch.testing.assert_close(a.cpu(), b, rtol=2e-4, atol=2e-4)


def _mlstm64(qkvg, gates, st, m, H, d, dv):
    """The recurrence in float64, and a bound of what fp32 rounding can do to each result: the
    sums of absolute values behind numerator and denominator (the same recurrence over |k|,
    |v|, |q|) in units of 2^-24."""
    T = qkvg.shape[0]
    out, unit = torch.zeros(T, H, dv).double(), torch.zeros(T, H, dv).double()
    S, n, mm = (x.double().clone() for x in st)
    SA, nA = S.abs(), n.abs()
    for (a, ln, p0), slot in zip(_step_rows(m), m.state_slots.tolist()):
        if slot < 0:
            continue
        if p0 == 0:
            for x in (S, n, mm, SA, nA):
                x[slot] = 0
        for t in range(a, a + ln):
            row = qkvg[t].double()
            q, k = row[: H * d].view(H, d) * d ** -0.5, row[H * d: 2 * H * d].view(H, d)
            v = row[2 * H * d: 2 * H * d + H * dv].view(H, dv)
            ig, fg = gates[t, :H].double(), gates[t, H:].double()
            mn = torch.maximum(fg + mm[slot], ig)
            f, i = torch.exp(fg + mm[slot] - mn)[:, None], torch.exp(ig - mn)[:, None]
            mm[slot] = mn
            S[slot] = f[..., None] * S[slot] + (i * k)[..., None] * v[:, None]
            SA[slot] = f[..., None] * SA[slot] + (i * k).abs()[..., None] * v.abs()[:, None]
            n[slot], nA[slot] = f * n[slot] + i * k, f * nA[slot] + (i * k).abs()
            den = torch.maximum((n[slot] * q).sum(-1).abs(), torch.exp(-mn))[:, None] + 1e-6
            out[t] = (S[slot] * q[..., None]).sum(1) / den
            unit[t] = ((SA[slot] * q.abs()[..., None]).sum(1) +
                       out[t].abs() * (nA[slot] * q.abs()).sum(-1, keepdim=True)) / den
    return out.view(T, -1), unit.view(T, -1) * 2.0 ** -24, (S, n, mm), (SA, nA, mm.abs() + 16)


# (chunk lengths, tokens before them): around the chunk (32 / 64 tokens) and tile (16) edges, a
# padding sequence, decode rows behind the chunks, long chunks that are cut into segments, and
# one and two rows among longer chunks
CHUNKS = [([1, 15, 16, 17, 31, 33], [0, 5, 0, 40, 0, 0], [9, 1]), ([63, 64, 65, 129], [0, 7, 0, 0], []),
          ([700], [0], []), ([33, 1300], [3, 11], [30]), ([1, 96, 2, 90, 31, 5], [0, 3, 9, 0, 0, 1], [4])]


def _whole(got, want):
    """All 24 bits of every operand reach the result: the norm of the difference within 5e-7 of the
    result's, four times what three bf16 parts per operand show (an operand of two parts is off by
    2.4e-6, which bounds on single elements let pass: its errors average out in their sums)."""
    return float((got.double().cpu() - want).norm()) <= 5e-7 * float(want.norm())


def _chunk_step(lens, before, D_ctx):
    n = len(lens) + len(D_ctx)
    slots = list(range(n))[::-1]
    if len(lens) > 2:
        slots[2] = -1                       # a padding sequence
    return _meta(lens, [a + b for a, b in zip(lens, before)], D_ctx, torch.zeros(n, 1, dtype=torch.int32),
                 slots), sum(lens) + len(D_ctx), n


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,d,dv", [(2, 128, 40), (1, 128, 128), (1, 256, 144)])
@pytest.mark.parametrize("lens,before,D_ctx", CHUNKS)
def test_mlstm_scan_chunkwise(gpu, dt, H, d, dv, lens, before, D_ctx):
    """Prompt rows on the chunkwise kernel against float64: within 16 units of fp32 rounding of
    the absolute sums (a chain of n additions comes to about sqrt(n) / 2 of them, and its largest
    terms are few)."""
    torch.manual_seed(24)
    m, T, n = _chunk_step(lens, before, D_ctx)
    st = (torch.randn(n, H, d, dv) * 0.3, torch.randn(n, H, d) * 0.3, torch.rand(n, H) * 2)
    qkvg = torch.randn(T, 2 * H * d + 2 * H * dv).to(dt)
    lf = torch.nn.functional.logsigmoid(torch.randn(T, H) * 2 + 2)
    lf[::29] = -40.0                        # gates that close
    gates = torch.cat([torch.randn(T, H) * 3, lf], dim=1)
    st_g = tuple(x.to(gpu) for x in st)
    want, unit, st_w, st_u = _mlstm64(qkvg, gates, st, m, H, d, dv)
    got = ops.mlstm_scan(qkvg.to(gpu), gates.to(gpu), st_g, _to(m, gpu), H, d, dv)
    assert ((got.double().cpu() - want).abs() <= 16 * unit).all()
    assert _whole(st_g[0], st_w[0])         # (outputs: the denominators' cancellation is in `unit`)
    for a, b, u in zip(st_g, st_w, st_u):
        assert ((a.double().cpu() - b).abs() <= 16 * 2.0 ** -24 * u).all()


@pytest.mark.parametrize("H,d,dv", [(2, 128, 40), (1, 128, 264), (1, 256, 144), (1, 256, 272), (1, 128, 36)])
@pytest.mark.parametrize("lens,before,D_ctx", [([1, 15, 16, 17, 63, 64, 65, 129, 660], [0, 5, 0, 40, 0, 0, 9, 0, 3], [9, 1]),
                                               ([384], [7], []), ([1300, 33, 2], [0, 11, 0], [30])])
def test_mlstm_scan_rows_by_dma(gpu, H, d, dv, lens, before, D_ctx):
    """Many rows, and sequences that are cut: whole and ragged chunks, a padding sequence, one and two workgroups
    per head, the last one's columns in part, segments of two chunks; values not in 16-byte units."""
    test_mlstm_scan_chunkwise(gpu, torch.bfloat16, H, d, dv, lens, before, D_ctx)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,d,dv", [(2, 128, 40), (1, 256, 144)])
@pytest.mark.parametrize("lens", [[4] * 9, [3] * 9, [5, 7, 6, 6, 7, 6, 6], [8], [7]])
def test_mlstm_scan_short_prompts(gpu, dt, H, d, dv, lens):
    """Rows few enough that the costs decide, on both sides of the rule, some in one chunk that is nearly empty."""
    test_mlstm_scan_chunkwise(gpu, dt, H, d, dv, lens, [3 * i for i in range(len(lens))], [5])


@pytest.mark.parametrize("H,d,dv", [(10, 128, 264), (15, 128, 144)])
def test_mlstm_scan_rows_by_dma_many_heads(gpu, H, d, dv):
    """Whole sequences with 128 key channels, which take heads enough to fill the CUs."""
    test_mlstm_scan_chunkwise(gpu, torch.bfloat16, H, d, dv, [1, 15, 16, 17, 63, 64, 65, 129, 660], [0, 5, 0, 40, 0, 0, 9, 0, 3], [9, 1])


@pytest.mark.parametrize("H,d,dv,P,n,own", [(4, 128, 512, 16, 300, False), (4, 128, 512, 32, 64, True), (4, 256, 512, 16, 100, True),
                                            (2, 128, 128, 64, 40, False), (4, 256, 128, 1, 600, True), (4, 256, 128, 8, 1500, False)])
def test_mlstm_scan_routes(gpu, H, d, dv, P, n, own):
    """Steps whose rows come by DMA and steps that stay in the general walk (csrc/kernels/chunk_scan.hip has the times)."""
    m = _to(_meta([n] * P, [n] * P, [], torch.zeros(P, 1, dtype=torch.int32), list(range(P))), gpu)
    x, g = torch.zeros(P * n, 2 * H * (d + dv), device=gpu).bfloat16(), torch.zeros(P * n, 2 * H, device=gpu)
    st = tuple(torch.zeros(P, H, *y, device=gpu) for y in ((d, dv), (d,), ()))
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        ops.mlstm_scan(x, g, st, m, H, d, dv)
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages()]
    assert any("mlstm_walk_kernel" in k for k in names) == own and any("chunk_scan_kernel" in k for k in names) != own


@pytest.mark.parametrize("lens,bad", [([45, 700, 400], (1, 333)), ([45, 700, 400], (0, 0)), ([45, 700, 400], (2, 399)),
                                      ([700, 33], (0, 130)), ([700, 33], (0, 698)), ([780, 33], (0, 130)), ([780, 33], (0, 778))])
def test_mlstm_scan_rows_by_dma_not_finite(gpu, lens, bad):
    """A value that is not finite reaches its own column from its row on, and nothing else changes by a bit; whole
    sequences (1145 rows) and segments (780 and 33; 700 and 33 stay in the general walk)."""
    torch.manual_seed(92)
    H, d, dv, (seq, tok), c = 2, 128, 272, bad, 261
    m, T, n = _chunk_step(lens, [0, 7, 0][:len(lens)], [])
    m.state_slots = torch.arange(n, dtype=torch.int32)
    x, g = torch.randn(T, 2 * H * d + 2 * H * dv).to(torch.bfloat16), torch.cat([torch.randn(T, H), -torch.rand(T, H)], dim=1)
    st = [torch.randn(n, H, d, dv), torch.randn(n, H, d), torch.rand(n, H)]

    def run():
        s = tuple(y.to(gpu) for y in st)
        return ops.mlstm_scan(x.to(gpu), g.to(gpu), s, _to(m, gpu), H, d, dv).cpu().view(T, H, dv), s[0].cpu()
    want, S_w = run()
    assert want.isfinite().all() and S_w.isfinite().all()
    t, end = sum(lens[:seq]) + tok, sum(lens[:seq + 1])
    x[t, 2 * H * d + dv + c] = float("-inf")
    got, S = run()
    hit, hit_S = torch.zeros(T, H, dv, dtype=torch.bool), torch.zeros(n, H, d, dv, dtype=torch.bool)
    hit[t:end, 1, c] = True
    hit_S[seq, 1, :, c] = True
    assert not got[hit].isfinite().any() and torch.equal(got[~hit], want[~hit])
    assert not S[hit_S].isfinite().any() and torch.equal(S[~hit_S], S_w[~hit_S])


def _step_rows(m):
    """(first row, rows, position of the first) of every step sequence."""
    qsl = m.query_start_loc.tolist() if m.num_prefills else [0]
    seqs = [(qsl[i], qsl[i + 1] - qsl[i], int(m.prefill_seq_lens[i]) - (qsl[i + 1] - qsl[i]))
            for i in range(m.num_prefills)]
    return seqs + [(qsl[-1] + i, 1, c - 1) for i, c in
                   enumerate(m.decode_ctx_lens.tolist() if m.num_decodes else [])]


def _matrix64(m, S, q, k, v, decay, beta=None):
    """S_t = decay_t S + k u^T, o = S^T q in float64 (u = v, or beta (v - S^T k) of the decayed S)
    with the sums of absolute values behind o and S in units of 2^-24: q, k [T, H, d], v [T, H, dv],
    decay [T, H, 1 or d], S [slots, H, d, dv]."""
    out, unit = torch.zeros_like(v), torch.zeros_like(v)
    S = S.double().clone()
    SA = S.abs()
    for (a, ln, p0), slot in zip(_step_rows(m), m.state_slots.tolist()):
        if slot < 0:
            continue
        if p0 == 0:
            S[slot], SA[slot] = 0, 0
        for t in range(a, a + ln):
            x, xa = decay[t][..., None] * S[slot], decay[t][..., None] * SA[slot]
            u, ua = v[t], v[t].abs()
            if beta is not None:
                u = beta[t][:, None] * (u - (x * k[t][..., None]).sum(1))
                ua = beta[t][:, None] * (ua + (xa * k[t].abs()[..., None]).sum(1))
            S[slot], SA[slot] = x + k[t][..., None] * u[:, None], xa + k[t].abs()[..., None] * ua[:, None]
            out[t] = (S[slot] * q[t][..., None]).sum(1)
            unit[t] = (SA[slot] * q[t].abs()[..., None]).sum(1)
    return out.flatten(1), unit.flatten(1) * 2.0 ** -24, S, SA * 2.0 ** -24


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,G,V", [(2, 1, 64), (4, 2, 40), (3, 3, 144)])
@pytest.mark.parametrize("lens,before,D_ctx", CHUNKS)
def test_ssd_scan_chunkwise(gpu, dt, H, G, V, lens, before, D_ctx):
    """Prompt rows on the chunkwise kernel against float64 (the bound: see the mLSTM's test); two
    heads per workgroup, heads of odd widths and heads that do not pair up."""
    torch.manual_seed(25)
    N = 128
    m, T, n = _chunk_step(lens, before, D_ctx)
    S = torch.randn(n, H, N, V) * 0.3
    xbc, dtv = torch.randn(T, H * V + 2 * G * N), torch.randn(T, H + 5).to(dt)[:, 5:]
    a_log, dtb, skip = torch.rand(H) * 2, torch.randn(H) - 2, torch.randn(H)
    a_log[0] = 12.0                         # decays that forget everything at every token
    x, B, C = (y.double() for y in xbc.split([H * V, G * N, G * N], 1))
    size = torch.nn.functional.softplus(dtv.double() + dtb.double())
    each = lambda y: y.view(T, G, N).repeat_interleave(H // G, 1)   # noqa: E731
    x = x.view(T, H, V)
    want, unit, S_w, S_u = _matrix64(m, S, each(C), each(B) * size[..., None], x,
                                     torch.exp(-torch.exp(a_log.double()) * size)[..., None])
    live = torch.zeros(T, 1)
    for (a, ln, _), slot in zip(_step_rows(m), m.state_slots.tolist()):
        live[a: a + ln] = slot >= 0
    add = (skip.double()[:, None] * x).flatten(1) * live
    S_g = S.to(gpu)
    got = ops.ssd_scan(xbc.to(gpu), dtv.to(gpu), a_log.to(gpu), dtb.to(gpu), skip.to(gpu), S_g, _to(m, gpu),
                       H, V, N, G)
    assert ((got.double().cpu() - want - add).abs() <= 16 * (unit + add.abs() * 2.0 ** -24)).all()
    assert ((S_g.double().cpu() - S_w).abs() <= 16 * S_u).all()
    assert _whole(got, want + add) and _whole(S_g, S_w)


@pytest.mark.parametrize("H,G,V", [(4, 1, 64), (8, 2, 40), (4, 1, 144), (8, 1, 33), (4, 1, 131), (4, 1, 16)])
@pytest.mark.parametrize("lens,before,D_ctx", [([400, 129, 250, 33, 31, 1, 96], [0, 7, 0, 0, 9, 0, 64], [5]),
                                               ([1025, 449], [33, 0], []), ([1000, 28, 1500], [0, 7, 9], [2])])
def test_ssd_scan_shared_images(gpu, H, G, V, lens, before, D_ctx):
    """Prompt rows of heads that share B and C: whole sequences and segments that end inside a chunk, a
    padding sequence, pairs of heads, one head over two workgroups, an odd number of columns."""
    test_ssd_scan_chunkwise(gpu, torch.bfloat16, H, G, V, lens, before, D_ctx)


@pytest.mark.parametrize("H,G,V", [(4, 1, 144), (4, 1, 131), (8, 1, 200), (8, 2, 33)])
@pytest.mark.parametrize("lens,before,D_ctx", [([256, 250, 0, 33, 255, 256, 254], [0, 7, 0, 0, 9, 0, 64], [5]),
                                               ([1500, 1001], [33, 0], []), ([300], [2], []), ([335, 290], [0, 70], [])])
def test_ssd_scan_shared_images_long(gpu, H, G, V, lens, before, D_ctx):
    """The same for heads of more than 64 columns, which take longer prompts there, and for prompts that are
    cut into two segments and a rest."""
    test_ssd_scan_chunkwise(gpu, torch.bfloat16, H, G, V, lens, before, D_ctx)


@pytest.mark.parametrize("G,P,n,allocs", [(1, 1, 113, 1), (1, 20, 20, 0), (8, 20, 20, 0), (8, 256, 20, 0), (1, 33, 20, 1), (4, 17, 33, 1),
                                          (8, 4, 128, 0), (8, 16, 500, 0), (8, 33, 100, 1), (1, 1, 300, 1), (8, 1, 300, 2),
                                          (1, 4, 300, 2), (8, 1, 1000, 1)])
def test_ssd_scan_routes(gpu, G, P, n, allocs):
    """Steps that pay for images of their chunks and steps that do not (csrc/kernels/chunk_ssd.hip has the times), told
    by their workspaces: none, one for the images and segments, two for segments alone."""
    H, V, d = 32, 64, 128
    m = _to(_meta([n] * P, [n] * P, [], torch.zeros(P, 1, dtype=torch.int32), list(range(P))), gpu)
    x, g = torch.zeros(P * n, H * V + 2 * G * d, device=gpu), torch.zeros(P * n, H, device=gpu).bfloat16()
    z, S = torch.zeros(H, device=gpu), torch.zeros(P, H, d, V, device=gpu)
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]   # noqa: E731
    before = count()
    ops.ssd_scan(x, g, z, z, z, S, m, H, V, d, G)
    assert count() - before == 1 + allocs                # (and the outputs)


@pytest.mark.parametrize("op,dt", [("mlstm", torch.bfloat16), ("mlstm", torch.float16), ("ssd", torch.bfloat16)])
def test_scan_segments_start_from_the_incoming_state(gpu, op, dt):
    """Continued prompts that are cut into segments, while products on another stream hold
    workgroups back: a segment that starts after its sequence's last one has ended still walks
    from the state the slot held before the call.  The bits of the same call alone, which the
    tests above compare with float64; the last segments are short."""
    torch.manual_seed(27)
    m, T, n = _chunk_step([1025, 449], [700, 33], [5])
    m = _to(m, gpu)
    if op == "mlstm":
        H, d, dv = 4, 128, 256
        st = [torch.randn(n, H, d, dv), torch.randn(n, H, d), torch.rand(n, H) * 2]
        x = torch.randn(T, 2 * H * d + 2 * H * dv).to(dt).to(gpu)
        gates = torch.cat([torch.randn(T, H), torch.full((T, H), -1e-3)], dim=1).to(gpu)
        run = lambda s: ops.mlstm_scan(x, gates, s, m, H, d, dv)   # noqa: E731
    else:
        H, V, N = 48, 64, 128
        st = [torch.randn(n, H, N, V)]
        x, dtv = torch.randn(T, H * V + 2 * N).to(gpu), torch.randn(T, H).to(dt).to(gpu)
        par = [torch.full((H,), -6.0), torch.zeros(H), torch.randn(H)]
        par = [y.to(gpu) for y in par]
        run = lambda s: ops.ssd_scan(x, dtv, *par, s[0], m, H, V, N, 1)   # noqa: E731
    alone = [y.to(gpu) for y in st]
    want = run(alone)
    a, side = torch.randn(4096, 4096, device=gpu, dtype=torch.bfloat16), torch.cuda.Stream()
    for _ in range(8):
        s = [y.to(gpu) for y in st]
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            for _ in range(6):
                torch.mm(a, a)
        got = run(s)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and all(torch.equal(y, z) for y, z in zip(s, alone))


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,G,V", [(2, 1, 128), (3, 3, 40), (3, 1, 144)])
@pytest.mark.parametrize("lens,before,D_ctx", CHUNKS)
def test_gated_delta_scan_chunkwise(gpu, dt, H, G, V, lens, before, D_ctx):
    """Prompt rows on the chunkwise kernel against float64: keys that are nearly parallel (the
    triangular systems are then as large as they get), heads that share keys in twos, threes and
    not at all.  The bound is that of the mLSTM's test, doubled for the value that is read before
    the write."""
    torch.manual_seed(26)
    d = 128
    m, T, n = _chunk_step(lens, before, D_ctx)
    S = torch.randn(n, H, d, V) * 0.3
    qkv = torch.randn(T, 2 * G * d + H * V)
    qkv[:, G * d: 2 * G * d] += 2 * torch.randn(G * d)
    ba = torch.randn(T, 2 * H + 5).to(dt)[:, 5:]
    a_log, dtb = torch.rand(H) * 2, torch.randn(H) - 2
    a_log[-1] = 12.0                        # decays that forget everything at every token
    q, k, v = (y.double() for y in qkv.split([G * d, G * d, H * V], 1))
    unit = lambda y: y * torch.rsqrt(y.pow(2).sum(-1, keepdim=True) + 1e-6)   # noqa: E731
    each = lambda y: unit(y.view(T, G, d)).repeat_interleave(H // G, 1)   # noqa: E731
    size = torch.nn.functional.softplus(ba[:, H:].double() + dtb.double())
    want, bound, S_w, S_u = _matrix64(m, S, each(q) * d ** -0.5, each(k), v.view(T, H, V),
                                      torch.exp(-torch.exp(a_log.double()) * size)[..., None],
                                      torch.sigmoid(ba[:, :H].double()))
    S_g = S.to(gpu)
    got = ops.gated_delta_scan(qkv.to(gpu), ba.to(gpu), a_log.to(gpu), dtb.to(gpu), S_g, _to(m, gpu), H, G, d, V)
    assert ((got.double().cpu() - want).abs() <= 32 * bound).all()
    assert ((S_g.double().cpu() - S_w).abs() <= 32 * S_u).all()
    assert _whole(got, want) and _whole(S_g, S_w)


@pytest.mark.parametrize("H,G,V,lens,before", [
    (16, 8, 128, [400], [0]), (2, 1, 130, [289, 520], [0, 31]), (8, 8, 22, [96 * 4], [5]), (4, 2, 128, [1, 700], [0, 0])])
def test_gated_delta_scan_short_segments(gpu, H, G, V, lens, before):
    """Few sequences in segments of three chunks: one that ends with a segment, one that is shorter than a segment,
    columns that are no multiple of 4, 16 or 128, states that enter."""
    test_gated_delta_scan_chunkwise(gpu, torch.bfloat16, H, G, V, lens, before, [])


@pytest.mark.parametrize("path", ["fast", "simple"])
@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,G,dk,dv,window,keep", [(4, 2, 96, 64, 70, 5), (4, 1, 128, 128, 150, 3),
                                                   (4, 2, 64, 32, 0, 0), (2, 1, 160, 96, 64, 70),
                                                   (3, 3, 32, 16, 1, 0), (6, 1, 64, 48, 129, 1)])
def test_window_attention_long_chunks(gpu, dt, path, H, G, dk, dv, window, keep, monkeypatch):
    """Chunks that span several 64-key tiles and 64-row blocks, continue long contexts and
    start mid-page, next to decode rows (one of them the first token of its sequence): the
    MFMA tile kernel and the 8-wave decode kernel (and, with KGC_WINDOW_ATTN=simple, the
    one-wave kernel alone) against the fp32 reference."""
    monkeypatch.setenv("KGC_WINDOW_ATTN", path)
    torch.manual_seed(5)
    bs = 8
    P_q, P_sl, D_ctx = [200, 77, 130], [300, 77, 513], [400, 65, 1]
    lens = P_sl + D_ctx
    mb = max(lens) // bs + 1
    nb = len(lens) * mb + 1
    tables = (torch.randperm(nb - 1)[: len(lens) * mb].view(len(lens), mb) + 1).to(torch.int32)
    kc = (torch.randn(nb, G, bs, dk) * 0.7).to(dt)
    vc = torch.randn(nb, G, bs, dv).to(dt)
    m = _meta(P_q, P_sl, D_ctx, tables)
    T = sum(P_q) + len(D_ctx)
    q = torch.randn(T, H, dk).to(dt)
    pos = torch.cat([torch.arange(sl - ql, sl) for ql, sl in zip(P_q, P_sl)] +
                    [torch.tensor([c - 1 for c in D_ctx])])
    gate = torch.rand(T, H)
    want = ops.window_attention(q, kc, vc, pos, m, 0.13, window, keep, gate)
    got = ops.window_attention(q.to(gpu), kc.to(gpu), vc.to(gpu), pos.to(gpu), _to(m, gpu), 0.13,
                               window, keep, gate.to(gpu))
    torch.testing.assert_close(got.cpu().float(), want.float(), **_tol(dt))


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("rows,W,N", [(1500, 288, 10), (2048, 1536, 8), (1100, 2304, 19)])
def test_gate_proj_many_rows(gpu, dt, rows, W, N):
    """The row-blocked kernel (weights held in registers, >= 1024 rows)."""
    torch.manual_seed(6)
    h = torch.randn(rows, W).to(dt)
    w = (torch.randn(N, W) * 0.1).to(dt)
    b = torch.randn(N)
    want = ref.gate_proj(h, w, b, ops.GATE_CAP_TANH, ops.GATE_LOGSIG_CAP_TANH, N // 2, 9.0)
    got = ops.gate_proj(h.to(gpu), w.to(gpu), b.to(gpu), ops.GATE_CAP_TANH,
                        ops.GATE_LOGSIG_CAP_TANH, N // 2, 9.0)
    torch.testing.assert_close(got.cpu(), want, rtol=2e-4, atol=2e-4)


@pytest.mark.parametrize("dt", DT)
def test_window_attention_many_decode_rows(gpu, dt):
    """A decode batch large enough (rows x kv heads >= 512) for the 4-wave workgroups."""
    torch.manual_seed(8)
    H, G, dk, dv, bs, window, keep = 4, 2, 64, 32, 8, 50, 3
    g = torch.Generator().manual_seed(9)
    D_ctx = torch.randint(1, 200, (300,), generator=g).tolist()
    mb = max(D_ctx) // bs + 1
    nb = 64
    tables = torch.randint(1, nb, (len(D_ctx), mb), generator=g).to(torch.int32)
    kc = (torch.randn(nb, G, bs, dk) * 0.7).to(dt)
    vc = torch.randn(nb, G, bs, dv).to(dt)
    m = _meta([], [], D_ctx, tables)
    q = torch.randn(len(D_ctx), H, dk).to(dt)
    pos = torch.tensor([c - 1 for c in D_ctx])
    want = ops.window_attention(q, kc, vc, pos, m, 0.2, window, keep, None)
    got = ops.window_attention(q.to(gpu), kc.to(gpu), vc.to(gpu), pos.to(gpu), _to(m, gpu), 0.2,
                               window, keep, None)
    torch.testing.assert_close(got.cpu().float(), want.float(), **_tol(dt))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,latent,bs,kw", [
    (8, 2, False, 8, dict(window=0, keep=0, softcap=20.0)), (4, 1, False, 16, dict(window=70, keep=5)),
    (8, 1, False, 8, dict(window=64, keep=70)), (4, 1, False, 24, dict(window=48, keep=0, chunked=True, sink=0.4)),
    (8, 1, True, 8, dict(window=100, keep=0)), (4, 1, True, 32, dict(window=0, keep=0))])
def test_window_attention_shared_tiles(gpu, dt, H, G, latent, bs, kw):
    """Prompt rows where four heads share a key/value head: row counts around the wave (32), block
    (64) and work item (128) edges, contexts that start inside a page and a tile, rows with one
    visible key, kept tokens in tiles of their own and inside the window, pages of no power of two;
    latent rows hold keys and values.  One rounding of the result to 16 bits (and of the weights'
    pairs: 2^-17 of sums of values around 1)."""
    torch.manual_seed(31)
    dk, dv = (256, 192) if latent else (128, 128)
    P_q, old = [1, 31, 33, 64, 65, 129, 150], [0, 90, 7, 0, 130, 0, 63]
    P_sl, T = [a + b for a, b in zip(P_q, old)], sum(P_q)
    width = max(P_sl) // bs + 1
    nb = len(P_q) * width + 1
    tables = (torch.randperm(nb - 1) + 1).view(len(P_q), width).int()
    kc = torch.randn(nb, G, bs, dk).to(dt)
    vc = kc[..., :dv] if latent else torch.randn(nb, G, bs, dv).to(dt)
    m = _meta(P_q, P_sl, [], tables)
    pos = torch.cat([torch.arange(o, o + a) for a, o in zip(P_q, old)])
    q = torch.randn(T, H, dk).to(dt)
    gate, eg = torch.rand(T, H), torch.randn(T, H * dv + 8).to(dt)[:, 8:]
    kw = dict(kw)
    args = (0.08, kw.pop("window"), kw.pop("keep"), gate)
    want = ops.window_attention(q, kc, vc, pos, m, *args, elem_gate=eg, out_scale=1.3, **kw)
    kg = kc.to(gpu)
    got = ops.window_attention(q.to(gpu), kg, kg[..., :dv] if latent else vc.to(gpu), pos.to(gpu), _to(m, gpu),
                               0.08, args[1], args[2], gate.to(gpu), elem_gate=eg.to(gpu), out_scale=1.3, **kw)
    ulp = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -10       # neighbours where rounding differs
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=1.01 * ulp, atol=2e-4)


def _window_forms(f):
    """Forms of the shared-tile prompt kernel (0: 64 rows, 1: 32 rows, 2: 32 rows and two groups of waves) in a call."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        f()
        torch.cuda.synchronize()
    keys = [e.key for e in prof.key_averages() if "window_prefill_gqa_kernel" in e.key]
    return [int(re.search(r"(?:ELi|, )(\d)(?:EE|>)", k).group(1)) for k in keys]


@pytest.mark.parametrize("latent", [False, True])
@pytest.mark.parametrize("n,L,old,window,form", [
    (1, 30, 0, 0, (0, 1)), (4, 64, 0, 0, (1, 1)), (2, 150, 0, 1024, (0, 1)), (1, 20, 300, 0, (2, 2)),       # up to one round of 32 rows
    (16, 140, 0, 0, (0, 0)), (5, 700, 0, 0, (2, 2)), (4, 700, 0, 1024, (0, 0)),                            # up to two
    (40, 100, 0, 0, (1, 1)), (24, 300, 0, 1024, (0, 1)), (10, 512, 0, 0, (0, 1)), (12, 300, 0, 1024, (1, 1))])
def test_window_attention_forms_by_length(gpu, latent, n, L, old, window, form):
    """Tables as wide as a service's longest request take no other form than tables of the sequences' own width where
    the step's longest sequence is named; form: of heads with keys and values of their own, of latent rows."""
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("forms for 256 CUs")
    bs, H, G, dk, dv = 32, 16, *((1, 256, 192) if latent else (4, 128, 128))
    width = -(-(L + old) // bs)
    kc = torch.zeros(n * width, G, bs, dk, dtype=torch.bfloat16, device=gpu)
    vc = kc[..., :dv] if latent else torch.zeros_like(kc)
    tables = torch.arange(n * width, dtype=torch.int32).view(n, width)
    wide = torch.cat([tables, tables[:, :1].expand(-1, 256)], 1).contiguous()
    q = torch.zeros(n * L, H, dk, dtype=torch.bfloat16, device=gpu)
    pos = torch.arange(old, old + L, device=gpu).repeat(n)

    def run(t, longest):
        m = _to(_meta([L] * n, [L + old] * n, [], t), gpu)
        m.prefill_max_len = longest
        m.work_seq, m.work_mblk = (torch.tensor(x, dtype=torch.int32, device=gpu) for x in ops.prefill_work_list([L] * n, [L + old] * n))
        return _window_forms(lambda: ops.window_attention(q, kc, vc, pos, m, 0.08, window, 0))
    assert run(tables, 0) == run(wide, L + old) == [form[latent]]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent", [False, True])
@pytest.mark.parametrize("n,bs,kw,forms", [
    (9, 4, dict(window=200, keep=70), (2, 2)), (9, 32, dict(window=0, keep=0, softcap=20.0), (2, 2)),      # every other tile each
    (9, 12, dict(window=256, keep=0, chunked=True, sink=0.4), (2, 2)),
    (4, 32, dict(window=60, keep=3), (0, 1)), (4, 32, dict(window=60, keep=3, rows=60), (1, 1)),           # 32 rows, few tiles
    (130, 4, dict(window=90, keep=66, rows=60), (1, 1)), (130, 20, dict(window=0, keep=0), (0, 1))])       # two workgroups to a CU
def test_window_attention_forms(gpu, dt, latent, n, bs, kw, forms):
    """Prompt rows where workgroups own 32 rows, two groups of waves share the tiles or one has them all: windows
    that begin between the rows that are copied together, tiles of kept tokens, odd and even numbers of tiles,
    one row to 70, tables that end inside a tile (what lay in LDS there before is not finite).  Calls in
    pages of a row less, which are of 64 rows for want of whole copies, have the same bits where no two groups share
    the tiles; the bound is the shared tiles'."""
    torch.manual_seed(41)
    H, dk, dv = 4, *((256, 192) if latent else (128, 128))
    q_rows, kw = kw.get("rows"), {k: v for k, v in kw.items() if k != "rows"}
    P_q = [q_rows + i % 3 if q_rows else 1 + (i * 23) % (70 if n < 100 else 7) for i in range(n)]
    old = [(i * 61) % (600 if n == 9 else 130) for i in range(n)]
    P_sl, T = [a + b for a, b in zip(P_q, old)], sum(P_q)
    pos = torch.cat([torch.arange(o, o + a) for a, o in zip(P_q, old)])
    q, kw = torch.randn(T, H, dk).to(dt), dict(kw)
    args = (0.08, kw.pop("window"), kw.pop("keep"))
    keys = [torch.randn(s, dk).to(dt) for s in P_sl]
    vals = [k[:, :dv] if latent else torch.randn(k.shape[0], dv).to(dt) for k in keys]

    def pack(bs, dev):
        width = max(P_sl) // bs + 1
        tables = torch.randperm(n * width).view(n, width)
        kc = torch.zeros(n * width, 1, bs, dk, dtype=dt)
        vc = torch.zeros(n * width, 1, bs, dv, dtype=dt)
        for t, k, v in zip(tables, keys, vals):
            j = torch.arange(k.shape[0])
            kc[t[j // bs], 0, j % bs] = k
            vc[t[j // bs], 0, j % bs] = v
        kc = kc.to(dev)
        return kc, kc[..., :dv] if latent else vc.to(dev), _to(_meta(P_q, P_sl, [], tables.int()), dev)

    def run(bs, dev):
        kc, vc, m = pack(bs, dev)
        return ops.window_attention(q.to(dev), kc, vc, pos.to(dev), m, *args, None, **kw)

    want = run(bs, "cpu")
    kc, vc, m = pack(bs, gpu)
    for c in (kc, vc):                       # every CU's LDS
        c.fill_(float("nan"))
    ops.window_attention(q.to(gpu), kc, vc, pos.to(gpu), m, *args, None, **kw)
    got = run(bs, gpu)
    ulp = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -10       # neighbours where rounding differs
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=1.01 * ulp, atol=2e-4)
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        assert _window_forms(lambda: run(bs, gpu)) == [forms[latent]]
    if n != 9:
        assert _window_forms(lambda: run(bs - 1, gpu)) == [0]
        assert torch.equal(got, run(bs - 1, gpu))


def _rounded_once(got, want, unit, eps):
    """got (16 bits) within half a unit in its last place of want (float64), and eps of ``unit`` for the arithmetic."""
    bits, low = (7, -126) if got.dtype == torch.bfloat16 else (10, -14)
    half = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(2.0 ** low))) - bits - 1)
    return ((got.double().cpu() - want).abs() <= half + eps * unit).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent", [False, True])
@pytest.mark.parametrize("lo,hi", [(6.0, 7.9), (8.5, 12.0)])
def test_window_attention_later_maximum(gpu, dt, latent, lo, hi):
    """Prompt rows that see one key of score 0 in their first tile, one of 2^lo to 2^hi times its weight in a later
    one, and no others to speak of: sums that are not zero move to a new maximum, and the weight that decides
    the result is exact (a pair of bf16 holds 17 bits of any other: 2^-18).  16 units of 2^-24 cover the
    fp32 steps: sums, exponents of the first key (its share is at most 2^-6), division, gate, scale."""
    torch.manual_seed(38)
    H, dk, dv, n, rows, old, bs = 4, 256 if latent else 128, 192 if latent else 128, 8, 128, 130, 16
    width = (rows + old) // bs + 1
    tables = torch.randperm(n * width).view(n, width).int()
    k, v = torch.zeros(n, width * bs, dk), torch.randn(n, width * bs, dv).to(dt)
    k[..., -1] = -16.0
    k[:, 0, -1], k[:, 100, -1] = 0.0, 1.0
    if latent:
        k[..., :dv] = v.float()
    kc = torch.empty(n * width, 1, bs, dk, dtype=dt)
    kc[tables.long(), 0] = k.to(dt).view(n, width, bs, dk)
    vc = torch.empty(n * width, 1, bs, dv, dtype=dt)
    vc[tables.long(), 0] = v.view(n, width, bs, dv)
    q, scale = torch.zeros(n * rows, H, dk).to(dt), 0.5
    q[..., -1] = ((lo + torch.rand(n * rows, H) * (hi - lo)) * math.log(2) / scale).to(dt)
    w = torch.exp(scale * q[..., -1].double())[..., None]
    v0, v1 = (v[:, j].double().repeat_interleave(rows, 0)[:, None] for j in (0, 100))
    want, unit = (v0 + w * v1) / (1 + w), (v0.abs() + w * v1.abs()) / (1 + w)
    m = _to(_meta([rows] * n, [rows + old] * n, [], tables), gpu)
    pos = torch.arange(old, old + rows).repeat(n).to(gpu)
    kg = kc.to(gpu)
    got = ops.window_attention(q.to(gpu), kg, kg[..., :dv] if latent else vc.to(gpu), pos, m, scale, 0, 0)
    assert _rounded_once(got.view(-1, H, dv), want, unit, 16 * 2.0 ** -24)


@pytest.mark.parametrize("dt,low,mag", [(torch.bfloat16, -60.0, 1.0), (torch.float16, -10.0, 1024.0)])
@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("at", [8, 1])
def test_window_attention_one_gate(gpu, dt, low, mag, decode, at):
    """Rows that see themselves only give their value times the gate's sigmoid, in prompt and decode rows, from gates
    that can be read four at a time and not: 6 units of 2^-24 (the sigmoid's 3, three products) and one rounding
    to 16 bits.  A gate per head spreads the results between 16-bit values."""
    torch.manual_seed(39)
    H, d, T, bs = 4, 128, 2048, 16
    v = (torch.randn(T, d) * mag).to(dt)
    kc, vc = torch.zeros(T // bs, 1, bs, d, dtype=dt), v.view(T // bs, 1, bs, d)
    eg, gate = (torch.rand(T, H * d + at) * (3 - low) + low).to(dt), torch.rand(T, H) + 0.5
    tables = torch.arange(T // bs).view(1, -1).int()
    m = _meta([], [], list(range(1, T + 1)), tables.expand(T, -1)) if decode else _meta([T], [T], [], tables)
    got = ops.window_attention(torch.zeros(T, H, d, device=gpu, dtype=dt), kc.to(gpu), vc.to(gpu),
                               torch.arange(T, device=gpu), _to(m, gpu), 1.0, 1, 0, gate.to(gpu),
                               elem_gate=eg.to(gpu)[:, at:])
    want = v.double()[:, None] * torch.sigmoid(eg[:, at:].double()).view(T, H, d) * gate.double()[..., None]
    assert _rounded_once(got.view(T, H, d), want, want.abs(), 6 * 2.0 ** -24)


def test_window_attention_gate_ends(gpu):
    """Gates at the ends of the range: one, zero, the smallest sigmoids and NaN."""
    x = torch.tensor([200.0, 88.0, 0.0, -87.5, -100.0, -103.0, -105.0, -3e38, float("inf"), float("-inf"), float("nan")])
    H, d, T = 4, 128, 128
    eg = x.bfloat16().repeat(T * H * d // len(x) + 1)[: T * H * d].view(T, H * d)
    v = torch.full((T // 16, 1, 16, d), 2.0 ** 100).bfloat16().to(gpu)
    m = _to(_meta([T], [T], [], torch.arange(T // 16).view(1, -1).int()), gpu)
    got = ops.window_attention(torch.zeros(T, H, d, device=gpu).bfloat16(), torch.zeros_like(v), v,
                               torch.arange(T, device=gpu), m, 1.0, 1, 0, elem_gate=eg.to(gpu)).cpu()
    want = torch.sigmoid(eg.double()) * 2.0 ** 100
    assert (got.isnan() == eg.isnan()).all()
    # (below 2^-126 a sigmoid has 2^-149 as its unit)
    ok = (got.double() - want).abs() <= want * 2.0 ** -8 * 1.001 + 2.0 ** -49
    assert ok[~eg.isnan()].all()


@pytest.mark.parametrize("latent", [False, True])
@pytest.mark.parametrize("at", [0, 4, 8])
@pytest.mark.parametrize("bs", [1, 7, 32])
def test_window_attention_output_slices_and_pages(gpu, latent, at, bs):
    """Prompt rows of shared tiles into column slices of a wider buffer (stores of 16 bytes where the rows
    allow it, else of 8), pages of one token, of no power of two and of 32: the bits of the plain call on
    the same keys in pages of 16."""
    torch.manual_seed(37)
    H, dk, dv, lens, old = 4, 256 if latent else 128, 192 if latent else 128, [70, 3, 130], [0, 40, 25]
    T, q = sum(lens), torch.randn(203, H, dk).bfloat16().to(gpu)
    keys = [torch.randn(a + b, dk).bfloat16().to(gpu) for a, b in zip(lens, old)]
    vals = [k[:, :dv] if latent else torch.randn(k.shape[0], dv).bfloat16().to(gpu) for k in keys]
    pos = torch.cat([torch.arange(o, o + a) for a, o in zip(lens, old)]).to(gpu)

    def run(bs, out=None):
        width = max(k.shape[0] for k in keys) // bs + 1
        tables = (torch.randperm(3 * width, generator=torch.Generator().manual_seed(bs))).view(3, width)
        kc = torch.zeros(3 * width, 1, bs, dk, device=gpu, dtype=torch.bfloat16)
        vc = kc[..., :dv] if latent else torch.zeros(3 * width, 1, bs, dv, device=gpu, dtype=torch.bfloat16)
        for t, k, v in zip(tables.to(gpu), keys, vals):
            j = torch.arange(k.shape[0], device=gpu)
            kc[t[j // bs], 0, j % bs] = k
            if not latent:
                vc[t[j // bs], 0, j % bs] = v
        m = _to(_meta(lens, [a + b for a, b in zip(lens, old)], [], tables.int()), gpu)
        return ops.window_attention(q, kc, vc, pos, m, 0.08, 50, 3, None, out=out)

    buf = torch.full((T, H * dv + 16), 7.0, device=gpu, dtype=torch.bfloat16)
    got = run(bs, buf[:, at: at + H * dv])
    assert torch.equal(got, run(16))
    rest = torch.ones(H * dv + 16, dtype=torch.bool, device=gpu)
    rest[at: at + H * dv] = False
    assert (buf[:, rest] == 7).all()


def test_window_attention_largest_pages(gpu):
    """Latent rows in pages of 2^24 tokens, 2^32 elements each: rows of the second page are not the first's."""
    torch.manual_seed(40)
    H, dk, dv, T, bs = 4, 256, 192, 70, 1 << 24
    q, rows, pos = torch.randn(T, H, dk).bfloat16().to(gpu), torch.randn(T, dk).bfloat16().to(gpu), torch.arange(T, device=gpu)

    def run(bs, table):
        kc = torch.empty(2, 1, bs, dk, device=gpu, dtype=torch.bfloat16)
        kc[0, 0, :T] = 3.0
        kc[1, 0, :T] = rows
        return ops.window_attention(q, kc, kc[..., :dv], pos, _to(_meta([T], [T], [], torch.tensor([[table]]).int()), gpu), 0.08, 0, 0)
    got, want = run(bs, 1).float(), run(128, 1).float()
    torch.cuda.empty_cache()
    torch.testing.assert_close(got, want, rtol=1.01 * 2.0 ** -7, atol=2e-4)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent", [False, True])
@pytest.mark.parametrize("cap", [1e6, 1.5])
def test_window_attention_capped_scores(gpu, dt, latent, cap):
    """Capped scores keep fp32's relative precision where the cap is far above them (a difference
    of numbers near the cap would be off by 1e6 2^-24 and more, whole units of the weights'
    exponents), and take both ends of tanh where it is not.  The bound is the shared tiles'."""
    torch.manual_seed(32)
    G, H, bs, (dk, dv) = 1, 4, 16, (256, 192) if latent else (128, 128)
    lens = [130, 33]
    width = 9
    tables = (torch.randperm(2 * width) + 1).view(2, width).int()
    kc = torch.randn(2 * width + 1, G, bs, dk).to(dt)
    vc = kc[..., :dv] if latent else torch.randn(2 * width + 1, G, bs, dv).to(dt)
    m, T = _meta(lens, lens, [], tables), sum(lens)
    pos, q = torch.cat([torch.arange(n) for n in lens]), torch.randn(T, H, dk).to(dt)
    args = (1.5 / dk ** 0.5, 0, 0, torch.ones(T, H))
    want = ops.window_attention(q, kc, vc, pos, m, *args, softcap=cap)
    kg = kc.to(gpu)
    got = ops.window_attention(q.to(gpu), kg, kg[..., :dv] if latent else vc.to(gpu), pos.to(gpu), _to(m, gpu),
                               *args[:3], args[3].to(gpu), softcap=cap)
    ulp = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -10       # neighbours where rounding differs
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=1.01 * ulp, atol=2e-4)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("latent", [False, True])
@pytest.mark.parametrize("ctx,bad,clean,kw", [
    (10, 70, [(0, 48)], {}),                                         # only the last 16 of the 64 rows see its tile
    (16, 20, [(48, 64)], dict(window=64, chunked=True)),             # a chunk before these rows'
    (10, 20, [], {})])                                               # every group sees its tile
def test_window_attention_values_not_finite(gpu, dt, latent, ctx, bad, clean, kw):
    """A value that is not finite: rows whose 16 rows see nothing of its 64 keys keep the bits of the call
    without it (as in the kernel of one head per workgroup), every row keeps its other columns, and rows that
    see it do not hide it."""
    torch.manual_seed(33)
    H, bs, n, (dk, dv) = 4, 16, 64, (256, 192) if latent else (128, 128)
    total = n + ctx
    width = (total + bs - 1) // bs
    tables = (torch.randperm(width) + 1).view(1, width).int()
    m, q = _meta([n], [total], [], tables), torch.randn(n, H, dk).to(dt)
    kc = torch.randn(width + 1, 1, bs, dk).to(dt)
    kw = dict(kw)
    window = kw.pop("window", 0)
    row, col = (int(tables[0, bad // bs]), 0, bad % bs), 100

    def run(vc):
        vg = vc.to(gpu)
        kg = vg if latent else kc.to(gpu)
        return ops.window_attention(q.to(gpu), kg, vg[..., :dv], torch.arange(ctx, total).to(gpu), _to(m, gpu),
                                    dk ** -0.5, window, 0, torch.ones(n, H).to(gpu), **kw).cpu().view(n, H, dv)
    vc = kc if latent else torch.randn(width + 1, 1, bs, dv).to(dt)
    want = run(vc)
    vb = vc.clone()
    vb[row][col] = float("inf")
    got = run(vb)
    pos = torch.arange(ctx, total)
    sees = pos >= bad
    if window:
        sees &= pos // window == bad // window
    assert sees.any() and not got[sees][..., col].isfinite().any()
    if not latent:                           # (a latent row is the key, too)
        keep = torch.arange(dv) != col
        assert torch.equal(got[..., keep], want[..., keep])
    for a, b in clean:
        assert torch.equal(got[a:b], want[a:b])


def _gla_case(T, slots, H, d, V, R, dt, tau, dev, open_=3.0):
    """Inputs of gla_scan and its terms for ``_matrix64``."""
    proj = (torch.randn(T, 2 * H * d + H * V + R) * 0.7).to(dt)
    a2, bias, S = torch.randn(H * d, R) * 0.3, torch.randn(H * d) + open_, torch.randn(slots, H, d, V)
    z = proj[:, -R:].double() @ a2.double().T + bias.double()
    decay = torch.exp(torch.nn.functional.logsigmoid(z) / tau).view(T, H, d)
    q, k, v = proj[:, : 2 * H * d + H * V].double().split([H * d, H * d, H * V], 1)
    terms = (S, q.view(T, H, d) * d ** -0.5, k.view(T, H, d), v.reshape(T, H, V), decay)
    dp = proj.to(dev)
    return terms, lambda st, m: ops.gla_scan(dp, dp[:, -R:], a2.to(dev), bias.to(dev), st, m, H, d, V, tau)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,d,V,R", [(2, 12, 4, 1), (1, 64, 60, 5), (3, 65, 64, 16), (2, 128, 68, 16),
                                     (1, 129, 256, 37), (1, 256, 132, 128)])
def test_gla_decode_rows(gpu, dt, H, d, V, R):
    """A step of decode rows only: state rows around the 16, 64, 128 row edges, columns around a
    workgroup's 64, a fresh row and a padding row.  The decay's logarithm is a sum of R + 1 terms
    (below 64 in all here) over tau."""
    torch.manual_seed(5)
    n, tau = 5, 4.0
    terms, run = _gla_case(n, n, H, d, V, R, dt, tau, gpu)
    m = _meta([], [], [7, 1, 300, 4, 2], torch.zeros(n, 1, dtype=torch.int32), slots=[3, 0, -1, 1, 4])
    want, unit, S, SA = _matrix64(m, *terms)
    st = terms[0].to(gpu)
    got = run(st, _to(m, gpu))
    rel = 16 + 64 / tau
    assert ((got.cpu() - want).abs() <= (d + rel) * unit + 1e-30).all()
    assert ((st.cpu() - S).abs() <= rel * SA).all()
    assert (got.cpu()[2] == 0).all() and (st.cpu()[2] == terms[0][2]).all()


@pytest.mark.parametrize("op", ["gla", "ssd", "delta"])
def test_decode_states_beyond_the_caches(gpu, op):
    """Decode rows whose states are 128 MB and more, which are read and written past the caches: the bits of the
    same rows in two steps of half as many, of a fresh row and of a padding row too."""
    torch.manual_seed(43)
    n, H, d, V, R = 130, *dict(gla=(8, 128, 256, 16), ssd=(32, 128, 64, 0), delta=(16, 128, 128, 0))[op]
    S = torch.randn(n, H, d, V, device=gpu)
    assert S.numel() * 4 >= 128 << 20 > S[:n // 2].numel() * 4
    rnd = lambda *s: torch.randn(*s, device=gpu)   # noqa: E731
    ctx, slots = [2 + i for i in range(n)], [(i * 7) % n for i in range(n)]
    ctx[3], slots[70] = 1, -1
    if op == "gla":
        x, y, a2, b = rnd(n, 2 * H * d + H * V).bfloat16(), rnd(n, R).bfloat16(), rnd(H * d, R), rnd(H * d)
        run = lambda r, s, m: ops.gla_scan(x[r], y[r], a2, b, s, m, H, d, V, 16.0)   # noqa: E731
    elif op == "ssd":
        x, y, p = rnd(n, H * V + 2 * d), rnd(n, H).bfloat16(), [rnd(H) - 2 for _ in range(3)]
        run = lambda r, s, m: ops.ssd_scan(x[r], y[r], *p, s, m, H, V, d, 1)   # noqa: E731
    else:
        x, y, p = rnd(n, H * d + H * V), rnd(n, 2 * H).bfloat16(), [rnd(H) - 2 for _ in range(2)]
        run = lambda r, s, m: ops.gated_delta_scan(x[r], y[r], *p, s, m, H, H // 2, d, V)   # noqa: E731

    def step(r, s):
        t = torch.zeros(len(ctx[r]), 1, dtype=torch.int32)
        return run(r, s, _to(_meta([], [], ctx[r], t, slots=slots[r]), gpu))
    once, twice = S.clone(), S.clone()
    got = step(slice(0, n), once)
    want = torch.cat([step(slice(0, n // 2), twice), step(slice(n // 2, n), twice)])
    assert torch.equal(got, want) and torch.equal(once, twice) and not torch.equal(once, S)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,W,N", [(64, 128, 1), (65, 1024, 17), (79, 1152, 8), (1000, 2048, 16), (64, 2304, 33),
                                      (100, 4096, 5), (8200, 256, 8)])
def test_gate_proj_matrix_cores(gpu, dt, rows, W, N):
    """Rows from the matrix-core kernel's least, around its blocks of 16 rows and 16 outputs, widths of
    every register form, more blocks than workgroups; a row of NaN stays alone.  Sums of W fp32 terms
    in parts: 2^-24 of the sum of absolute products, times the sums' depth (below 24)."""
    torch.manual_seed(41)
    h, w = torch.randn(rows, W).to(dt), (torch.randn(N, W) * 0.05).to(dt)
    b = torch.randn(N)
    h[3] = float("nan")
    got = ops.gate_proj(h.to(gpu), w.to(gpu), b.to(gpu), ops.GATE_NONE).cpu()
    assert got[3].isnan().all()
    keep = torch.arange(rows) != 3
    want = h[keep].double() @ w.double().T + b.double()
    unit = (h[keep].double().abs() @ w.double().abs().T + b.double().abs()) * 2.0 ** -24
    assert ((got[keep] - want).abs() <= 24 * unit).all()
    got = ops.gate_proj(h.to(gpu), w.to(gpu), None, ops.GATE_CAP_TANH, ops.GATE_LOGSIG_CAP_TANH, N // 2, 15.0).cpu()
    want = ref.gate_proj(h[keep], w, None, ops.GATE_CAP_TANH, ops.GATE_LOGSIG_CAP_TANH, N // 2, 15.0)
    torch.testing.assert_close(got[keep], want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("rows,W,G", [(1, 256, 1), (3, 1280, 5), (2, 2048, 1), (5, 2560, 2), (2, 4096, 16), (3, 8192, 1)])
def test_row_kernels_by_vectors(gpu, dt, rows, W, G):
    """Rows held in registers: one to eight float4 per thread, threads without columns, groups of
    one wave up to the whole row, head vectors of no multiple of 256, xIELU around the ends of its
    series.  Against float64: sums of W squares and quotients (32 units of 2^-24), one rounding to
    the activation type."""
    torch.manual_seed(51)
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[dt] * 1.01 + 32 * 2.0 ** -24
    x, y, w = torch.randn(rows, W) * 3, torch.randn(rows, W).to(dt), torch.rand(W) + 0.5

    def close(got, want, unit=None):
        err = (got.cpu().double() - want).abs()
        assert (err <= ulp * (want.abs() if unit is None else unit) + 1e-7).all()

    def norm(v, n):
        v = v.view(rows, n, -1)
        return (v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-5)).view(rows, W)
    x1 = x.clone().to(gpu)
    s = (x + y.float()).double()
    got = ops.group_rms_norm(x1, w.to(gpu), G, 1e-5, dt, add=y.to(gpu))
    close(got, norm(s, G) * w.double())
    assert torch.equal(x1.cpu().double(), s)
    hist, coef = torch.randn(6, rows + 1, W), torch.randn(6)
    hg, x1 = hist.to(gpu), x.clone().to(gpu)
    for layer in (0, 4):
        h64, x0 = hg.cpu().double()[:, :rows], x1.cpu()
        h64[layer + 1] = (x0 + y.float()).double()
        terms = coef[: layer + 2].double()[:, None, None] * h64[: layer + 2]
        got = ops.depth_mix_norm(x1, hg, layer, y.to(gpu), coef[: layer + 2].to(gpu), w.to(gpu), G, 1e-5, dt)
        assert torch.equal(hg[layer + 1, :rows].cpu().double(), h64[layer + 1])
        assert ((x1.cpu().double() - terms.sum(0)).abs() <= 8 * 2.0 ** -24 * terms.abs().sum(0)).all()
        close(got, norm(x1.cpu().double(), G) * w.double())
    for H, dv in ((1, W if W <= 1024 else 1024), (3, 68), (2, 516)):
        o, big, nw = torch.randn(rows, H * dv), torch.randn(rows, H * dv + 16).to(dt), torch.rand(H * dv) + 0.5
        v = o.double().view(rows, H, dv)
        want = (v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-5)).view(rows, -1) * nw.double()
        got = ops.head_norm_gate(o.to(gpu), big.to(gpu)[:, 8: 8 + H * dv], nw.to(gpu), H, 1e-5, dt)
        close(got, want * torch.sigmoid(big[:, 8: 8 + H * dv].double()))
    z = torch.cat([torch.randn(rows * W - 8) * 2, torch.tensor([-0.5, -0.5001, -0.4999, -1e-3, 0.0, 1e-3, -30.0, 9.0])]).to(dt)
    z64 = z.double()
    want = torch.where(z64 > 0, 0.7 * z64 * z64 + 0.5 * z64, 1.3 * (torch.expm1(z64) - z64) + 0.5 * z64)
    unit = torch.where(z64 > 0, want, 1.3 * (torch.expm1(z64) - z64).abs() + 0.5 * z64.abs())
    close(ops.xielu(z.to(gpu), torch.tensor([0.7, 1.3]).to(gpu)), want, unit)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("T,H,G,dk,dv,rot", [(1, 4, 1, 64, 64, 64), (37, 6, 2, 40, 24, 16), (130, 16, 4, 128, 128, 64),
                                             (9, 3, 3, 24, 8, 0), (65, 2, 1, 192, 128, 192)])
def test_rope_kv_store_by_chunks(gpu, dt, interleaved, T, H, G, dk, dv, rot):
    """16-byte chunks against single elements (which rows at an odd address take): the same bytes, with
    padding slots, slots past the cache and positions outside the table."""
    torch.manual_seed(61)
    n, bs, nb = (H + G) * dk + G * dv, 8, T // 8 + 3
    wide = torch.randn(T, n + 9, device=gpu).to(dt)
    qkv = torch.empty(T, n + 8, device=gpu, dtype=dt)[:, :n]
    qkv.copy_(wide[:, 1: n + 1])
    table = torch.randn(50, rot, device=gpu) if rot else None
    pos, slots = torch.randint(-2, 60, (T,), device=gpu), torch.randperm(nb * bs, device=gpu)[:T]
    if T > 2:
        slots[1], slots[2] = -1, nb * bs
    got = []
    for x in (wide[:, 1: n + 1], qkv):
        kc, vc = (torch.zeros(nb, G, bs, d, device=gpu, dtype=dt) for d in (dk, dv))
        got.append((ops.rope_kv_store(x, pos, table, kc, vc, slots, H, G, dk, dv, interleaved), kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and bool(got[0][2].any())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,rows", [(8, 2, 9), (16, 1, 40), (12, 4, 140), (16, 4, 17), (16, 4, 100)])
@pytest.mark.parametrize("kw", [dict(window=0, keep=0), dict(window=300, keep=5), dict(window=128, keep=0, chunked=True, sink=0.3),
                                dict(window=0, keep=0, softcap=15.0)])
def test_window_decode_many_waves(gpu, dt, H, G, rows, kw):
    """Decode rows of 128/128 heads on 16 waves (68 and 400 workgroups, and windows of 128 keys), on 4 (560
    workgroups) and in pieces (18 and 40): one key, chunks around 32 and the 16 x 32 of a round, several rounds, a
    padding row."""
    torch.manual_seed(71)
    lens = [1, 31, 32, 33, 511, 513, 1025, 700, 0] + [5 + 13 * i for i in range(rows - 9)]
    bs, width = 16, 70
    nb = 400
    tables = torch.randint(0, nb, (rows, width), dtype=torch.int32)
    kc, vc = torch.randn(nb, G, bs, 128).to(dt), torch.randn(nb, G, bs, 128).to(dt)
    q, gate = torch.randn(rows, H, 128).to(dt), torch.rand(rows, H)
    lens = [min(n, width * bs) for n in lens]
    m = _meta([], [], lens, tables)
    pos, kw = torch.tensor(lens) - 1, dict(kw)
    args = (0.09, kw.pop("window"), kw.pop("keep"))
    want = ops.window_attention(q, kc, vc, pos, m, *args, gate, **kw)
    got = ops.window_attention(q.to(gpu), kc.to(gpu), vc.to(gpu), pos.to(gpu), _to(m, gpu), *args, gate.to(gpu), **kw)
    assert (got[8] == 0).all()
    ulp = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -10       # neighbours where rounding differs
    keep = torch.arange(rows) != 8
    torch.testing.assert_close(got.cpu().float()[keep], want.float()[keep], rtol=1.01 * ulp, atol=2e-4)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,rows", [(16, 66), (20, 40), (16, 520)])
@pytest.mark.parametrize("kw", [dict(window=0, keep=0), dict(window=300, keep=5, sink=0.3)])
def test_window_decode_latent_many_rows(gpu, dt, H, rows, kw):
    """Latent decode rows of steps that are not split: 66 and 80 workgroups of 8 waves (20 heads take two), 520 of 4;
    one key, chunks around 32 and the 8 x 32 of a round, several rounds, a padding row."""
    torch.manual_seed(72)
    lens = [1, 31, 32, 33, 255, 257, 513, 1000, 0] + [5 + 13 * i % 700 for i in range(rows - 9)]
    bs, nb, width = 16, 300, 63
    tables = torch.randint(0, nb, (rows, width), dtype=torch.int32)
    kc, q, gate = torch.randn(nb, 1, bs, 256).to(dt), torch.randn(rows, H, 256).to(dt), torch.rand(rows, H)
    m, pos, kw = _meta([], [], lens, tables), torch.tensor(lens) - 1, dict(kw)
    args = (0.06, kw.pop("window"), kw.pop("keep"))
    want = ops.window_attention(q, kc, kc[..., :192], pos, m, *args, gate, **kw)
    kg = kc.to(gpu)
    got = ops.window_attention(q.to(gpu), kg, kg[..., :192], pos.to(gpu), _to(m, gpu), *args, gate.to(gpu), **kw)
    assert (got[8] == 0).all()
    ulp = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -10       # neighbours where rounding differs
    keep = torch.arange(rows) != 8
    torch.testing.assert_close(got.cpu().float()[keep], want.float()[keep], rtol=1.01 * ulp, atol=2e-4)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,dk,dv,latent", [(16, 4, 128, 128, False), (6, 2, 72, 40, False), (40, 1, 256, 192, True),
                                              (3, 1, 200, 248, False), (20, 1, 128, 64, True)])
@pytest.mark.parametrize("lens,kw", [([2100], dict(window=0, keep=0)), ([0, 1, 33, 300, 2100, 511], dict(window=0, keep=0, softcap=5.0)),
                                     ([2100, 40, 1024], dict(window=300, keep=5, sink=0.4)), ([2081, 2048, 2047], dict(window=1024, keep=0, chunked=True))])
def test_window_decode_in_pieces(gpu, dt, H, G, dk, dv, latent, lens, kw):
    """Steps of few rows, their keys over many workgroups: rows with fewer chunks than pieces, several chunks
    per piece, one key, a padding row, a sink, values of their own and as columns of the keys."""
    torch.manual_seed(73)
    n, bs, width, nb = len(lens), 16, 132, 300
    tables = torch.randint(0, nb, (n, width), dtype=torch.int32)
    kc = torch.randn(nb, G, bs, dk).to(dt)
    vc = kc[..., :dv] if latent else torch.randn(nb, G, bs, dv).to(dt)
    q, gate = torch.randn(n, H, dk).to(dt), torch.rand(n, H)
    eg = torch.randn(n, H * dv + 8).to(dt)
    m = _meta([], [], lens, tables)
    pos, kw = torch.tensor(lens) - 1, dict(kw)
    args = (0.09, kw.pop("window"), kw.pop("keep"))
    want = ops.window_attention(q, kc, vc, pos, m, *args, gate, elem_gate=eg[:, 8:], **kw).float()
    kg = kc.to(gpu)
    vg = kg[..., :dv] if latent else vc.to(gpu)
    got = ops.window_attention(q.to(gpu), kg, vg, pos.to(gpu), _to(m, gpu), *args, gate.to(gpu),
                               elem_gate=eg.to(gpu)[:, 8:], **kw).cpu().float()
    live = torch.tensor(lens) > 0
    assert (got[~live] == 0).all()
    ulp = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -10       # neighbours where rounding differs
    torch.testing.assert_close(got[live], want[live], rtol=1.01 * ulp, atol=2e-4)


@pytest.mark.parametrize("rows,longest,pieces,latent", [
    (1, 192, 0, False), (1, 193, 7, False), (8, 256, 8, False), (12, 1000, 32, False), (16, 192, 0, False),
    (16, 384, 12, False), (16, 0, 32, False), (17, 4000, 0, False), (3, 30, 1, True), (64, 70, 3, True)])
def test_window_decode_pieces_follow_the_longest_context(gpu, rows, longest, pieces, latent):
    """A step whose longest context is known is split by it, not by tables that hold 4096 keys: one launch and no
    workspace up to six chunks (four key/value heads a row; latent rows always); the results are those of a table as long as the
    contexts, whichever route they take."""
    torch.manual_seed(74)
    H, G, dk, d, bs, width, dt = (16, 1, 256, 192, 32, 128, torch.bfloat16) if latent else (16, 4, 128, 128, 32, 128, torch.bfloat16)
    lens = [max(1, min(longest or 300, 4000) - 7 * i) for i in range(rows)]
    tables = torch.randint(0, 200, (rows, width), dtype=torch.int32)
    kc, vc = (torch.randn(200, G, bs, dk).to(dt).to(gpu) for _ in range(2))
    vc = kc[..., :d] if latent else vc
    q, pos = torch.randn(rows, H, dk).to(dt).to(gpu), (torch.tensor(lens) - 1).to(gpu)

    def run(m, out):
        m = _to(m, gpu)
        count = lambda: torch.cuda.memory_stats()["requested_bytes.all.allocated"]   # noqa: E731
        before = count()
        ops.window_attention(q, kc, vc, pos, m, 0.09, 1024, 0, out=out)
        return count() - before
    m = _meta([], [], lens, tables)
    m.decode_max_ctx = longest
    got, want = torch.empty(rows, H * d, dtype=dt, device=gpu), torch.empty(rows, H * d, dtype=dt, device=gpu)
    assert run(m, got) == rows * H * pieces * (d + 2) * 4
    run(_meta([], [], lens, tables[:, : max(lens) // bs + 1].contiguous()), want)
    torch.testing.assert_close(got.float(), want.float(), rtol=1.01 * 2.0 ** -7, atol=2e-4)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,V,R", [(2, 64, 5), (1, 144, 16), (3, 40, 1)])
@pytest.mark.parametrize("lens,before,D_ctx", CHUNKS)
def test_gla_scan_chunkwise(gpu, dt, H, V, R, lens, before, D_ctx):
    """Prompt rows in chunks of 32 (and decode rows behind them): ends inside a chunk, continued and
    fresh states, a padding sequence, value columns off a wave's 16 and a workgroup's 128; decays from
    none at all to all but zero.  Products of up to 32 decays (R + 1 terms over tau each) and
    sums of d + 32 terms, in units of 2^-24 of the sums of absolute values."""
    torch.manual_seed(81)
    d, tau = 128, 4.0
    m, T, n = _chunk_step(lens, before, D_ctx)
    for open_ in (3.0, -12.0, 100.0):
        terms, run = _gla_case(T, n, H, d, V, R, dt, tau, gpu, open_)
        want, unit, S, SA = _matrix64(m, *terms)
        st = terms[0].to(gpu)
        got = run(st, _to(m, gpu))
        assert ((got.cpu() - want).abs() <= (d + 64) * unit + 1e-30).all()
        assert ((st.cpu() - S).abs() <= 128 * SA + 1e-30).all()
        if open_ == 100.0:                  # every decay is 1: no error of theirs
            assert _whole(got, want) and _whole(st, S)


@pytest.mark.parametrize("V", [30, 32])
@pytest.mark.parametrize("lens,before", [([2100], [7]), ([700, 330], [0, 40])])
def test_gla_scan_segments_of_odd_rows(gpu, V, lens, before):
    """Few sequences in segments, more and fewer than four of them: state rows of a multiple of 4 elements, which the
    chain over the segments takes at a time, and of none."""
    test_gla_scan_chunkwise(gpu, torch.bfloat16, 2, V, 5, lens, before, [])


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("R", [4, 20, 128])
def test_gla_rows_off_their_alignment(gpu, dt, R):
    """Ranks of a part of, one and several sixteens: rows read in pairs and fours, and the same values in rows of an
    odd stride, from an odd address or with the projection off its 16 bytes, one by one: the same bits.  Units as
    below, and the R + 1 terms of a decay's argument."""
    torch.manual_seed(83)
    H, d, V, tau = 2, 128, 48, 4.0
    m, T, n = _chunk_step([33, 64, 47], [3, 0, 0], [])
    W = 2 * H * d + H * V
    x, low = (torch.randn(T, W) * 0.7).to(dt), (torch.randn(T, R) * 0.7).to(dt)
    a2, bias, S0 = torch.randn(H * d, R) * 0.3 * (16 / max(R, 16)) ** 0.5, torch.randn(H * d) + 3.0, torch.randn(n, H, d, V)
    z = low.double() @ a2.double().T + bias.double()
    decay = torch.exp(torch.nn.functional.logsigmoid(z) / tau).view(T, H, d)
    q, k, v = x.double().split([H * d, H * d, H * V], 1)
    want, unit, S, SA = _matrix64(m, S0, q.view(T, H, d) * d ** -0.5, k.view(T, H, d), v.reshape(T, H, V), decay)

    def run(x, low, a2):
        st = S0.to(gpu)
        return ops.gla_scan(x, low, a2, bias.to(gpu), st, _to(m, gpu), H, d, V, tau), st
    def wider(t, off):                       # rows of an odd stride, `off` elements into them
        w = torch.zeros(t.shape[0], t.shape[1] + 8 + (t.shape[1] + 1) % 2, dtype=t.dtype)
        w[:, off:off + t.shape[1]] = t
        return w.to(gpu)[:, off:off + t.shape[1]]
    a2o = torch.zeros(a2.numel() + 1)
    a2o[1:] = a2.flatten()
    a2o = a2o.to(gpu)[1:].view_as(a2)
    x, low, a2 = x.to(gpu), low.to(gpu), a2.to(gpu)
    got, st = run(x, low, a2)
    assert ((got.cpu() - want).abs() <= (d + 64 + R) * unit + 1e-30).all()
    assert ((st.cpu() - S).abs() <= (128 + R) * SA + 1e-30).all()
    for args in ((wider(x, 0), low, a2), (wider(x, 3), low, a2), (x, wider(low, 1), a2), (x, low, a2o)):
        other, st2 = run(*args)
        assert torch.equal(other, got) and torch.equal(st2, st)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("tau", [16.0, 0.5])
def test_gla_prompt_decays(gpu, dt, tau):
    """One token's decay per channel, arguments from -60 to 100, seen as what it leaves of a state of ones: the others'
    are 1 and the keys 0.  With g the exponent, in units of 2^-24: half of one for the result, 1 for
    its series, and 4 |g| for the logarithm, the difference and the product of which g is rounded."""
    H, d, V, T = 1, 128, 16, 40
    m, _, n = _chunk_step([T], [3], [])
    a2 = torch.zeros(H * d, 4)
    a2[:, 0] = torch.cat([torch.linspace(-60, 100, 64), torch.linspace(-3, 3, 64)])
    a2[:, 1] = 100.0
    x, low = torch.zeros(T, 2 * H * d + H * V, dtype=dt), torch.zeros(T, 4, dtype=dt)
    low[:, 1] = 1.0
    low[17] = torch.tensor([1.0, 0, 0, 0])
    st = torch.ones(n, H, d, V).to(gpu)
    ops.gla_scan(x.to(gpu), low.to(gpu), a2.to(gpu), torch.zeros(H * d).to(gpu), st, _to(m, gpu), H, d, V, tau)
    g = torch.nn.functional.logsigmoid(a2[:, 0].double()) / tau
    want = g.exp()
    got = st[0, 0].cpu().double()
    assert torch.equal(got, got[:, :1].expand_as(got))
    assert ((got[:, 0] - want).abs() <= (2 + 4 * g.abs()) * want * 2.0 ** -24 + 2.0 ** -149).all()


@pytest.mark.parametrize("dt,R", [(torch.bfloat16, 16), (torch.float16, 7), (torch.float32, 4)])
def test_gla_scan_long_segments(gpu, dt, R):
    """Segments of seven chunks, the last one short, beside a sequence that is not cut, on two workgroups per
    head; ranks in and out of fours, rows in 16-byte units and not.  Decays near one: what the segments hand on
    stays in the sums."""
    torch.manual_seed(82)
    H, d, V = 8, 128, 144
    m, T, n = _chunk_step([3000, 40], [5, 0], [3])
    terms, run = _gla_case(T, n, H, d, V, R, dt, 4.0, gpu, 8.0)
    want, unit, S, SA = _matrix64(m, *terms)
    st = terms[0].to(gpu)
    got = run(st, _to(m, gpu))
    assert ((got.cpu() - want).abs() <= (d + 64) * unit + 1e-30).all()
    assert ((st.cpu() - S).abs() <= 128 * SA + 1e-30).all()


@pytest.mark.parametrize("op,dt", [("mlstm", torch.bfloat16), ("mlstm", torch.float16), ("ssd", torch.bfloat16),
                                   ("delta", torch.bfloat16), ("gla", torch.bfloat16), ("gla", torch.float32)])
@pytest.mark.parametrize("where,val", [("v", float("nan")), ("v", float("-inf")), ("k", float("nan")), ("gate", float("nan"))])
@pytest.mark.parametrize("bad", [(0, 20), (0, 44), (1, 0), (1, 333), (1, 698), (2, 32)])
def test_chunkwise_scans_keep_what_is_not_finite_to_later_rows(gpu, op, dt, where, val, bad):
    """One value, key channel or gate that is not finite, at tokens inside, at the ends of and alone
    in a chunk and in a prompt cut into segments: the rows before it, other sequences, and for a
    value the other columns have the bits of the call without it; it reaches every row from its own
    on and the state, as token by token."""
    torch.manual_seed(91)
    lens = [45, 700, 33]
    m, T, n = _chunk_step(lens, [3, 0, 7], [])
    m.state_slots = torch.tensor([2, 0, 1], dtype=torch.int32)
    mg, d, H, G = _to(m, gpu), 128, 2, 2 if op in ("mlstm", "gla") else 1
    V = 144
    a, b = torch.full((H,), -1.0).to(gpu), torch.zeros(H).to(gpu)
    if op == "mlstm":
        x, g = torch.randn(T, 2 * H * d + 2 * H * V).to(dt), torch.cat([torch.randn(T, H), -torch.rand(T, H)], dim=1)
        st = [torch.randn(n, H, d, V), torch.randn(n, H, d), torch.rand(n, H)]
        koff, voff = H * d, 2 * H * d
        run = lambda x, g, s: ops.mlstm_scan(x, g, s, mg, H, d, V)   # noqa: E731
    elif op == "ssd":
        x, g, st, koff, voff = torch.randn(T, H * V + 2 * G * d), torch.randn(T, H).to(dt), [torch.randn(n, H, d, V)], H * V, 0
        run = lambda x, g, s: ops.ssd_scan(x, g, a, b, b, s[0], mg, H, V, d, G)   # noqa: E731
    elif op == "delta":
        x, g, st = torch.randn(T, 2 * G * d + H * V), torch.randn(T, 2 * H).to(dt), [torch.randn(n, H, d, V)]
        koff, voff = G * d, 2 * G * d
        run = lambda x, g, s: ops.gated_delta_scan(x, g, a, b, s[0], mg, H, G, d, V)   # noqa: E731
    else:
        R = 3
        x, g, st = torch.randn(T, 2 * H * d + H * V).to(dt), torch.randn(T, R).to(dt), [torch.randn(n, H, d, V)]
        koff, voff, a2, ab = H * d, 2 * H * d, torch.randn(H * d, R).to(gpu), torch.ones(H * d).to(gpu)
        run = lambda x, g, s: ops.gla_scan(x, g, a2, ab, s[0], mg, H, d, V, 4.0)   # noqa: E731

    def both(x, g):
        s = [y.to(gpu) for y in st]
        return run(x.to(gpu), g.to(gpu), s).cpu().view(T, H, V), s[0].cpu()
    want, S_w = both(x, g)
    assert want.isfinite().all() and S_w.isfinite().all()
    seq, tok = bad
    t, end, h, c = sum(lens[:seq]) + tok, sum(lens[:seq + 1]), H - 1, 77
    if where == "v":
        x[t, voff + h * V + c] = val
    elif where == "k":
        x[t, koff + (h if G == H else 0) * d + 100] = val
    else:
        g[t, h if op != "gla" else 0] = val
    got, S = both(x, g)
    hit = torch.zeros(T, H, V, dtype=torch.bool)
    heads = slice(h, h + 1) if where == "v" or (where == "k" and G == H) or (where == "gate" and op != "gla") else slice(0, H)
    hit[t:end, heads, slice(c, c + 1) if where == "v" else slice(0, V)] = True
    assert not got[hit].isfinite().any() and torch.equal(got[~hit], want[~hit])
    hit = torch.zeros(n, H, d, V, dtype=torch.bool)
    slot = int(m.state_slots[seq])
    if where == "k" and op in ("mlstm", "ssd", "gla"):      # only the channel's row of the state
        hit[slot, heads, 100] = True
    else:
        hit[slot, heads, :, slice(c, c + 1) if where == "v" else slice(0, V)] = True
    assert not S[hit].isfinite().any() and torch.equal(S[~hit], S_w[~hit])


@pytest.mark.parametrize("gate", ["strength", "decay"])
@pytest.mark.parametrize("tok", [0, 1, 15, 16, 17, 31, 32, 62])
def test_delta_systems_keep_gates_that_are_not_finite_to_later_rows(gpu, gate, tok):
    """The triangular systems go by blocks of 16 tokens, two heads at a time: a write strength or decay that is NaN
    in either block, of the middle one of three heads that share a key."""
    torch.manual_seed(97)
    H, G, d, V, lens = 6, 2, 128, 24, [63, 64]
    m, T, n = _chunk_step(lens, [0, 5], [])
    x, g, S0 = torch.randn(T, 2 * G * d + H * V), torch.randn(T, 2 * H), torch.randn(n, H, d, V)
    x[:, G * d: 2 * G * d] += 2 * torch.randn(G * d)
    a, b, mg = torch.full((H,), -1.0).to(gpu), torch.zeros(H).to(gpu), _to(m, gpu)

    def both():
        S = S0.to(gpu)
        return ops.gated_delta_scan(x.to(gpu), g.to(gpu), a, b, S, mg, H, G, d, V).cpu().view(T, H, V), S.cpu()
    want, S_w = both()
    assert want.isfinite().all() and S_w.isfinite().all()
    h, t = 4, lens[0] + tok
    g[t, h + (H if gate == "decay" else 0)] = float("nan")
    got, S = both()
    hit, hit_S = torch.zeros(T, H, V, dtype=torch.bool), torch.zeros(n, H, d, V, dtype=torch.bool)
    hit[t:, h] = True
    hit_S[int(m.state_slots[1]), h] = True
    assert not got[hit].isfinite().any() and torch.equal(got[~hit], want[~hit])
    assert not S[hit_S].isfinite().any() and torch.equal(S[~hit_S], S_w[~hit_S])


@pytest.mark.parametrize("op,P,V,Tp", [("delta", 1, 32, 21), ("delta", 8, 512, 158), ("delta", 8, 32, 164), ("delta", 90, 32, 1080),
                                       ("gla", 1, 32, 11), ("gla", 8, 512, 83), ("gla", 100, 512, 300), ("gla", 90, 32, 1080)])
def test_short_prompts_on_both_sides_of_the_chunkwise_rule(gpu, op, P, V, Tp):
    """The fewest rows that go chunkwise -- by the costs, and by the rows in steps of 1024 -- seen by their workspace, and
    a row less, which goes token by token: float64 within the bounds of the tests above."""
    torch.manual_seed(98)
    d, H = 128, 2
    for less in (0, 1):
        m, T, n = _chunk_step([(Tp - less + i) // P for i in range(P)], [0] * P, [])
        m.state_slots = torch.arange(n, dtype=torch.int32)
        x, S = torch.randn(T, 2 * H * d + H * V), torch.randn(n, H, d, V) * 0.3
        q, k, v = x.double().split([H * d, H * d, H * V], 1)
        q, k, v, S_g, mg = q.view(T, H, d), k.view(T, H, d), v.reshape(T, H, V), S.to(gpu), _to(m, gpu)
        if op == "delta":
            g, a, b = torch.randn(T, 2 * H), torch.zeros(H), torch.full((H,), -2.0)
            unit = lambda y: y * torch.rsqrt(y.pow(2).sum(-1, keepdim=True) + 1e-6)   # noqa: E731
            decay = torch.exp(-torch.nn.functional.softplus(g[:, H:].double() - 2.0))[..., None]
            terms, f, fs = (unit(q) * d ** -0.5, unit(k), v, decay, torch.sigmoid(g[:, :H].double())), 32, 32
            args = (x.to(gpu), g.to(gpu), a.to(gpu), b.to(gpu), S_g, mg, H, H, d, V)
        else:
            g, a, b = torch.randn(T, 4), torch.randn(H * d, 4) * 0.3, torch.randn(H * d) + 3.0
            decay = torch.exp(torch.nn.functional.logsigmoid(g.double() @ a.double().T + b.double()) / 4.0).view(T, H, d)
            terms, f, fs = (q * d ** -0.5, k, v, decay), d + 64, 128
            args = (x.to(gpu), g.to(gpu), a.to(gpu), b.to(gpu), S_g, mg, H, d, V, 4.0)
        want, unit, S_w, S_u = _matrix64(m, S, *terms)
        torch.cuda.synchronize()
        before = torch.cuda.memory_stats()["requested_bytes.all.allocated"]
        got = (ops.gated_delta_scan if op == "delta" else ops.gla_scan)(*args)
        asked = torch.cuda.memory_stats()["requested_bytes.all.allocated"] - before
        assert (asked > got.numel() * got.element_size()) == (less == 0)
        assert ((got.double().cpu() - want).abs() <= f * unit + 1e-30).all()
        assert ((S_g.double().cpu() - S_w).abs() <= fs * S_u + 1e-30).all()


@pytest.mark.parametrize("where,val", [("v", float("nan")), ("v", float("-inf")), ("k", float("nan")), ("gate", float("nan"))])
@pytest.mark.parametrize("op,lens,before,at", [
    (op, lens, before, at) for op, lens, before in (("mlstm", [45, 700, 400], [0, 7, 0]), ("mlstm", [780, 33], [0, 5]),
                                                    ("ssd", [45, 300, 33], [3, 0, 7]), ("ssd", [700, 420], [0, 5]))
    for at in ((0, 20), (0, 44), (0, 333), (0, 698), (1, 0), (1, 29), (1, 128), (1, 299), (1, 399)) if at[1] < lens[at[0]]])
def test_own_walks_keep_what_is_not_finite_to_later_rows(gpu, op, lens, before, where, val, at):
    """As the test of the general walk above, in the walks that bf16 mLSTM rows (256 key channels, two workgroups per
    head) and heads that share B and C take: whole sequences and segments (of 128 rows), the first, a middle and
    the last one; two groups of four heads, of which one shows what the other keeps."""
    seq, tok = at
    torch.manual_seed(93)
    m, T, n = _chunk_step(lens, before, [])
    m.state_slots = torch.tensor([n - 1, *range(n - 1)], dtype=torch.int32)
    mg = _to(m, gpu)
    if op == "mlstm":
        H, G, d, V = 2, 2, 256, 272
        x, g = torch.randn(T, 2 * H * d + 2 * H * V).bfloat16(), torch.cat([torch.randn(T, H), -torch.rand(T, H)], dim=1)
        st, koff, voff = [torch.randn(n, H, d, V), torch.randn(n, H, d), torch.rand(n, H)], H * d, 2 * H * d
        run = lambda x, g, s: ops.mlstm_scan(x, g, s, mg, H, d, V)   # noqa: E731
    else:
        H, G, d, V = 8, 2, 128, 40
        x, g, st, koff, voff = torch.randn(T, H * V + 2 * G * d), torch.randn(T, H).bfloat16(), [torch.randn(n, H, d, V)], H * V, 0
        a, b = torch.full((H,), -1.0).to(gpu), torch.zeros(H).to(gpu)
        run = lambda x, g, s: ops.ssd_scan(x, g, a, b, b, s[0], mg, H, V, d, G)   # noqa: E731

    def both():
        s = [y.to(gpu) for y in st]
        return run(x.to(gpu), g.to(gpu), s).cpu().view(T, H, V), s[0].cpu()
    want, S_w = both()
    assert want.isfinite().all() and S_w.isfinite().all()
    t, end, h, c, grp = sum(lens[:seq]) + tok, sum(lens[:seq + 1]), H - 1, V - 3, G - 1
    if where == "v":
        x[t, voff + h * V + c] = val
    elif where == "k":
        x[t, koff + grp * d + 100] = val
    else:
        g[t, h] = val
    got, S = both()
    heads = slice(grp * (H // G), H) if where == "k" else slice(h, h + 1)
    cols = slice(c, c + 1) if where == "v" else slice(0, V)
    hit, hit_S = torch.zeros(T, H, V, dtype=torch.bool), torch.zeros(n, H, d, V, dtype=torch.bool)
    hit[t:end, heads, cols] = True
    hit_S[int(m.state_slots[seq]), heads, 100 if where == "k" else slice(0, d), cols] = True
    assert not got[hit].isfinite().any() and torch.equal(got[~hit], want[~hit])
    assert not S[hit_S].isfinite().any() and torch.equal(S[~hit_S], S_w[~hit_S])
