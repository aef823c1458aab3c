"""GPU parity of the segmented state pass: long sequences cut into segments
that run in parallel (first segment from h0; middle segments as their
zero-start result R and transition P; scan S_{s+1} = P_s S_s + R_s; later
segments again with outputs).  Checked against the CPU oracle and against the
unsegmented kernel on the same inputs."""
import pytest
import torch

from helpers import BF16, assert_out, assert_state, cu_of, rule_inputs, state_rel, STATE_REL
from oracle import gdn_ref

pytestmark = pytest.mark.gpu


CASES = [
    # Hk, Hv, D, lens, max_segments
    (2, 2, 128, [1000], 2),
    (2, 2, 128, [1000], 3),
    (2, 2, 128, [1000], 5),
    (2, 4, 128, [700, 3, 450], 4),
    (4, 4, 64, [129, 900], 12),
    (2, 2, 128, [130], 3),          # 3 chunks into 3 one-chunk segments, the last partial
]


@pytest.mark.parametrize("with_h0", [False, True])
@pytest.mark.parametrize("Hk,Hv,D,lens,segs", CASES, ids=lambda c: str(c))
def test_segmented_chunk_rule(pkg, dev, Hk, Hv, D, lens, segs, with_h0):
    gen = torch.Generator().manual_seed(51)
    N = sum(lens)
    q, k, v, g, beta = rule_inputs(gen, N, Hk, Hv, D)
    cu = cu_of(lens)
    n = len(lens)
    h0 = torch.randn(n, Hv, D, D, generator=gen) * 0.1 if with_h0 else None
    ro, rS = gdn_ref.chunk_varlen(q, k, v, g, beta.float(), cu, h0)
    cu_d = torch.tensor(cu, device=dev)
    cu_h = torch.tensor(cu, dtype=torch.int64)
    args = (q.to(dev), k.to(dev), v.to(dev), g.to(dev), beta.to(dev), cu_d, None if h0 is None else h0.to(dev))
    o_s, S_s = pkg.ops.chunk_gated_delta_rule_varlen(*args, cu_seqlens_cpu=cu_h, max_segments=segs)
    o_1, S_1 = pkg.ops.chunk_gated_delta_rule_varlen(*args, cu_seqlens_cpu=cu_h, max_segments=1)
    assert_out(o_s.cpu(), ro.to(BF16), "segmented out")
    assert_state(S_s.cpu(), rS, "segmented final")
    # against the unsegmented kernel: the same up to rounding
    assert_out(o_s.cpu(), o_1.cpu(), "segmented vs one pass")
    assert state_rel(S_s.cpu(), S_1.cpu()) < STATE_REL


def test_segmented_pool_in_place(pkg, dev):
    """Pool-indexed in-place states (h0 == hT at the slot ids): the first segment
    reads the slot, the last writes it, other slots untouched."""
    gen = torch.Generator().manual_seed(52)
    Hk = Hv = 2
    D = 128
    lens = [800, 64]
    N = sum(lens)
    q, k, v, g, beta = rule_inputs(gen, N, Hk, Hv, D)
    cu = cu_of(lens)
    pool = torch.randn(5, Hv, D, D, generator=gen) * 0.1
    ids = [3, 1]
    ro, rS = gdn_ref.chunk_varlen(q, k, v, g, beta.float(), cu, pool[ids])
    pd = pool.to(dev)
    o, _ = pkg.ops.chunk_gated_delta_rule_varlen(q.to(dev), k.to(dev), v.to(dev), g.to(dev), beta.to(dev),
                                                 torch.tensor(cu, device=dev), pd,
                                                 state_ids=torch.tensor(ids, device=dev), final_state=pd,
                                                 cu_seqlens_cpu=torch.tensor(cu), max_segments=4)
    assert_out(o.cpu(), ro.to(BF16), "pool segmented out")
    assert_state(pd.cpu()[ids], rS, "pool segmented final")
    assert torch.equal(pd.cpu()[[0, 2, 4]], pool[[0, 2, 4]])


def test_segmented_fused_prefill(pkg, dev):
    """The fused gates + conv + chunk call with segments equals the one-pass
    fused call up to rounding, with the conv states rolled once."""
    gen = torch.Generator().manual_seed(53)
    Hk, Hv, D = 2, 4, 128
    lens = [900, 5]
    N = sum(lens)
    C = 2 * Hk * D + Hv * D
    mixed = torch.randn(N, C, generator=gen).to(BF16).to(dev)
    conv_w = (torch.randn(C, 4, generator=gen) * 0.5).to(BF16).to(dev)
    A_log = (torch.rand(Hv, generator=gen) * 2.7).to(BF16).to(dev)
    dt_bias = (torch.rand(Hv, generator=gen) * 2 - 1).to(BF16).to(dev)
    a = torch.randn(N, Hv, generator=gen).to(BF16).to(dev)
    b = torch.randn(N, Hv, generator=gen).to(BF16).to(dev)
    conv0 = torch.randn(4, C, 3, generator=gen).to(BF16).to(dev)
    s0 = (torch.randn(4, Hv, D, D, generator=gen) * 0.1).to(dev)
    ids = torch.tensor([2, 0], device=dev)
    cu = torch.tensor(cu_of(lens), dtype=torch.int64)
    outs = []
    for segs in (1, 6):
        cp, sp = conv0.clone(), s0.clone()
        o = pkg.ops.conv_chunk_prefill_varlen(mixed, cp, conv_w, b, a, A_log, dt_bias, cu.to(dev), sp, ids,
                                              Hk, Hv, D, cu_seqlens_cpu=cu, max_segments=segs)
        outs.append((o.cpu(), cp.cpu(), sp.cpu()))
    (o1, c1, s1), (o6, c6, s6) = outs
    assert_out(o6, o1, "fused segmented vs one pass")
    assert state_rel(s6, s1) < STATE_REL
    assert torch.equal(c6.view(torch.int16), c1.view(torch.int16)), "conv states"


# the automatic plan: one pass (a short sequence), 30 chunks in segments, a
# second sequence cut in fewer beside one that is not, and every sequence cut
@pytest.mark.parametrize("lens", [[300], [1900], [4000, 1500, 70], [2600, 2500]], ids=str)
def test_automatic_segments(pkg, dev, lens):
    """Slowly decaying states (g of a few hundredths), so that the scan's
    transitions matter: the automatic plan against one pass and the oracle."""
    gen = torch.Generator().manual_seed(53)
    Hk, Hv, D = 2, 4, 128
    N = sum(lens)
    q, k, v, g, beta = rule_inputs(gen, N, Hk, Hv, D)
    g = g * 0.02
    cu = cu_of(lens)
    h0 = torch.randn(len(lens), Hv, D, D, generator=gen) * 0.1
    ro, rS = gdn_ref.chunk_varlen(q, k, v, g, beta.float(), cu, h0)
    cu_h = torch.tensor(cu, dtype=torch.int64)
    args = (q.to(dev), k.to(dev), v.to(dev), g.to(dev), beta.to(dev), cu_h.to(dev), h0.to(dev))
    o_s, S_s = pkg.ops.chunk_gated_delta_rule_varlen(*args, cu_seqlens_cpu=cu_h)
    o_1, S_1 = pkg.ops.chunk_gated_delta_rule_varlen(*args, cu_seqlens_cpu=cu_h, max_segments=1)
    assert_out(o_s.cpu(), ro.to(BF16), "automatic segments out")
    assert_state(S_s.cpu(), rS, "automatic segments final")
    assert_out(o_s.cpu(), o_1.cpu(), "automatic segments vs one pass")
    assert state_rel(S_s.cpu(), S_1.cpu()) < STATE_REL


# lengths that one pass runs faster than any cut: 26 chunks at 16 heads, 24 and 18
# at 8; lengths that segments run faster: 32 and 48 chunks
@pytest.mark.parametrize("Hk,Hv,D,lens,cut", [(16, 16, 128, [1661], False), (16, 32, 64, [1661], False),
                                              (4, 8, 128, [1533, 1132], False), (16, 16, 128, [2045], True),
                                              (16, 16, 64, [3070], True)], ids=str)
def test_automatic_plan_lengths(pkg, dev, Hk, Hv, D, lens, cut):
    """Whether the automatic plan cuts: its bits are the one-pass call's or not
    (slowly decaying states, whose roundings differ between the two)."""
    gen = torch.Generator().manual_seed(56)
    q, k, v, g, beta = rule_inputs(gen, sum(lens), Hk, Hv, D, slow_decay=True)
    cu = torch.tensor(cu_of(lens), dtype=torch.int64)
    h0 = torch.randn(len(lens), Hv, D, D, generator=gen) * 0.1
    args = (q.to(dev), k.to(dev), v.to(dev), g.to(dev), beta.to(dev), cu.to(dev), h0.to(dev))
    S_a = pkg.ops.chunk_gated_delta_rule_varlen(*args, cu_seqlens_cpu=cu)[1]
    S_1 = pkg.ops.chunk_gated_delta_rule_varlen(*args, cu_seqlens_cpu=cu, max_segments=1)[1]
    assert torch.equal(S_a, S_1) != cut


# (float64 on the GPU: 16 or 8 heads, one long sequence or two)
@pytest.mark.parametrize("Hk,Hv,D,lens", [(16, 16, 128, [2000]), (4, 8, 128, [3500]), (16, 16, 64, [2500, 1900]),
                                          (16, 16, 128, [5000])], ids=str)
@pytest.mark.parametrize("decay", [0.02, 0.0])
def test_automatic_segments_lose_no_precision(pkg, dev, Hk, Hv, D, lens, decay):
    """Segments move the state through the fp16-operand transitions P; with states
    that decay slowly or not at all they stay as close to float64 as one pass.
    (Measured over 1,700 to 16,000 tokens: both 2.2e-4 of the states at a decay of
    0.02, 3.7e-4 to 4.0e-4 without; the two differ by at most 1.5 %, to either
    side, so a factor of 1.05 is allowed.)"""
    gen = torch.Generator().manual_seed(57)
    q, k, v, g, beta = rule_inputs(gen, sum(lens), Hk, Hv, D)
    g = g * decay
    cu = torch.tensor(cu_of(lens), dtype=torch.int64)
    h0 = torch.randn(len(lens), Hv, D, D, generator=gen) * 0.1
    q, k, v, g, beta, h0 = (t.to(dev) for t in (q, k, v, g, beta, h0))
    unit = lambda t: (t * (t.square().sum(-1, keepdim=True) + 1e-6).rsqrt()).repeat_interleave(Hv // Hk, 1)
    qd, kd, vd, gd, bd = unit(q.double()) * D ** -0.5, unit(k.double()), v.double(), g.double().exp(), beta.double()
    ro, rS = torch.empty_like(vd), h0.double()
    for r in range(len(lens)):
        S = rS[r]
        for t in range(int(cu[r]), int(cu[r + 1])):
            S = S * gd[t, :, None, None]
            delta = (vd[t] - (S * kd[t, :, :, None]).sum(-2)) * bd[t, :, None]
            S = S + kd[t, :, :, None] * delta[:, None, :]
            ro[t] = (S * qd[t, :, :, None]).sum(-2)
        rS[r] = S
    rel = lambda x, y: float((x.double() - y).norm() / y.norm())
    args = (q, k, v, g, beta, cu.to(dev), h0)
    o_a, S_a = pkg.ops.chunk_gated_delta_rule_varlen(*args, cu_seqlens_cpu=cu)
    o_1, S_1 = pkg.ops.chunk_gated_delta_rule_varlen(*args, cu_seqlens_cpu=cu, max_segments=1)
    print(f"states {rel(S_a, rS):.3e} / one pass {rel(S_1, rS):.3e}, outputs {rel(o_a, ro):.3e} / {rel(o_1, ro):.3e}")
    assert not torch.equal(S_a, S_1), "these lengths are cut"
    assert rel(S_a, rS) <= 1.05 * rel(S_1, rS) and rel(o_a, ro) <= 1.05 * rel(o_1, ro)


# empty sequences at the start, between others and at the end; lengths around a
# chunk; the most sequences that the host's list holds, and one more
@pytest.mark.parametrize("D,lens", [(128, [0, 1, 64, 0, 0, 65, 130, 3, 63, 128, 5, 200, 0]),
                                    (64, [70, 0, 1, 129] * 5), (128, [17, 0, 66, 64] * 16), (128, [17, 0, 66, 64] * 16 + [9])],
                         ids=lambda c: str(len(c)) if isinstance(c, list) else str(c))
def test_listed_chunks(pkg, dev, D, lens):
    """Chunks located from the host's list: the same bits as from the device's
    offsets alone."""
    gen = torch.Generator().manual_seed(54)
    Hk = Hv = 16
    q, k, v, g, beta = rule_inputs(gen, sum(lens), Hk, Hv, D)
    cu = torch.tensor(cu_of(lens), dtype=torch.int64)
    h0 = torch.randn(len(lens), Hv, D, D, generator=gen) * 0.1
    args = (q.to(dev), k.to(dev), v.to(dev), g.to(dev), beta.to(dev), cu.to(dev), h0.to(dev))
    o_h, S_h = pkg.ops.chunk_gated_delta_rule_varlen(*args, cu_seqlens_cpu=cu)
    o_d, S_d = pkg.ops.chunk_gated_delta_rule_varlen(*args)
    assert torch.equal(o_h.view(torch.int16), o_d.view(torch.int16)), "outputs"
    assert torch.equal(S_h, S_d), "states"


# both selections cut into several segments; one of a very long sequence; D = 64
@pytest.mark.parametrize("Hk,Hv,D,lens,late", [(2, 4, 128, [2600, 2300, 70], [True, False, False]),
                                               (2, 2, 64, [70, 3300, 0, 2500], [False, True, False, False]),
                                               (16, 16, 128, [49675, 1893, 573], [True, False, False])], ids=str)
def test_split_state_pass_segments(pkg, dev, Hk, Hv, D, lens, late):
    """The state pass of a segmented call split over two launches, whose segment
    states have their own places: the same launches in order on one stream, and
    the whole call, give the same bits (slowly decaying states, so that every
    segment state matters)."""
    gen = torch.Generator(device=dev).manual_seed(55)
    N, n = sum(lens), len(lens)
    C = 2 * Hk * D + Hv * D
    rand = lambda *shape: torch.randn(*shape, generator=gen, device=dev)
    mixed, conv_w = rand(N, C).to(BF16), (rand(C, 4) * 0.5).to(BF16)
    a, b = rand(N, Hv).to(BF16), rand(N, Hv).to(BF16)
    A_log, dt_bias = (rand(Hv) * 0.3 - 4).to(BF16), rand(Hv).to(BF16)
    conv0, s0 = rand(n + 1, C, 3).to(BF16), rand(n + 1, Hv, D, D) * 0.1
    ids = torch.randperm(n + 1, generator=gen, device=dev)[:n]
    cu = torch.tensor(cu_of(lens), dtype=torch.int64)
    outs = []
    for side in (None, torch.cuda.current_stream(dev), torch.cuda.Stream(dev)):
        cp, sp, keep = conv0.clone(), s0.clone(), []
        res = pkg.ops.conv_chunk_prefill_varlen(mixed, cp, conv_w, b, a, A_log, dt_bias, cu.to(dev), sp, ids, Hk, Hv,
                                                D, cu_seqlens_cpu=cu, late=None if side is None else late,
                                                side_stream=side, keep=keep)
        torch.cuda.synchronize()
        outs.append((res if side is None else res[0], cp, sp))
    for name, (o, cp, sp) in zip(("in order", "two streams"), outs[1:]):
        assert torch.equal(o.view(torch.int16), outs[0][0].view(torch.int16)), f"{name}: outputs"
        assert torch.equal(cp.view(torch.int16), outs[0][1].view(torch.int16)), f"{name}: conv states"
        assert torch.equal(sp, outs[0][2]), f"{name}: states"
