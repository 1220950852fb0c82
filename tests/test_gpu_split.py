"""GPU: scans over sequences cut into segments (few (sequence, head) pairs, long time axis) against the fp32
recurrences.  The gates are weak, so that the state entering a segment decides its output, and the lengths leave short
last chunks, short last segments and, in packed batches, sequences shorter than a segment.  Tolerances are those of the
uncut operators (16-bit operands, fp32 sums): 1e-2 on o, 5e-3 on the final state, 2e-2 on the gradients."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from helpers import assert_close, gdr_inputs, gla_inputs
from oracle.recurrent import naive_recurrent_gated_delta_rule, naive_recurrent_gla

pytestmark = pytest.mark.gpu


def _delta(kind, K):
    """The delta rule's kinds go by their key channels."""
    return kind | (8 if K == 64 else 0)


def _cut(N, T, H, slabs, reverse, bounds, kind=0):
    """Whether the launches cut this batch."""
    from fla_amd import _backend as be
    sp = be.Split()
    arr = None if bounds is None else (ctypes.c_int64 * len(bounds))(*bounds)
    return be.lib().fla_scan_split(arr, N, T, H, slabs, int(reverse), kind, ctypes.byref(sp), None, None, None)


CASES = [
    # B, T, H, K, V, boundaries of a packed batch, dtype
    (1, 833, 1, 64, 64, None, torch.bfloat16),        # 14 chunks, the last of one token
    (2, 1087, 2, 128, 128, None, torch.bfloat16),     # 17 chunks, the last of 63 tokens
    (1, 1024, 3, 128, 64, None, torch.float16),
    (1, 1500, 2, 64, 128, [0, 1, 1, 900, 964, 1500], torch.bfloat16),
    (1, 2200, 1, 128, 128, [0, 1290, 1354, 2200], torch.bfloat16),
]


@pytest.mark.parametrize("B,T,H,K,V,bounds,dtype", CASES)
@pytest.mark.parametrize("heads", [False, True])
def test_gla_cut_sequences(device, B, T, H, K, V, bounds, dtype, heads):
    from fla_amd.ops.gla import chunk_gla
    from fla_amd.ops.simple_gla import chunk_simple_gla
    N = B if bounds is None else len(bounds) - 1
    offs = None if bounds is None else torch.tensor(bounds, device=device)
    assert _cut(N, T, H, V // 64, False, bounds)   # (the reverse scan runs uncut: test_gla_cut_state_gradients)
    print("cut", B, T, H, K, V, bounds, dtype, heads, flush=True)
    q, k, v, g, h0 = gla_inputs(B, T, H, K, V, seed=T, dtype=dtype, normalizer=600.0, N=N)
    if heads:
        g = g[..., 0].contiguous()
    do, dht = torch.randn(B, T, H, V).to(dtype), torch.randn(N, H, K, V) * 0.1
    op = chunk_simple_gla if heads else chunk_gla
    dev = [x.to(device) for x in (q, k, v, g, h0)]
    with torch.no_grad():
        o1, ht1 = op(*dev[:4], initial_state=dev[4], output_final_state=True, cu_seqlens=offs, head_first=False)
    leaves = [x.requires_grad_() for x in dev]
    o, ht = op(*leaves[:4], initial_state=leaves[4], output_final_state=True, cu_seqlens=offs, head_first=False)
    torch.autograd.backward((o, ht), (do.to(device), dht.to(device)))
    refs = [x.float().requires_grad_() for x in (q, k, v, g, h0)]
    ro, rht = naive_recurrent_gla(*refs[:3], None if heads else refs[3], initial_state=refs[4], output_final_state=True,
                                  offsets=bounds, g=refs[3] if heads else None)
    torch.autograd.backward((ro, rht), (do.float(), dht))
    for a, b in ((o1, ht1), (o, ht)):
        assert_close("o", ro, a, 1e-2)
        assert_close("ht", rht, b, 5e-3)
    for name, r, d in zip(("dq", "dk", "dv", "dg", "dh0"), refs, leaves):
        assert_close(name, r.grad, d.grad, 2e-2)


def test_gla_cut_gate_logits_and_strong_gates(device):
    """Gates formed from pre-activations, some of them far outside the range of the chunk's single reference point."""
    from fla_amd.ops.gla import chunk_gla
    q, k, v, _, h0 = gla_inputs(1, 1100, 2, 128, 128, seed=5)
    x = torch.randn(1, 1100, 2, 128)
    x[:, 300:330] -= 40.0
    assert _cut(1, 1100, 2, 2, False, None)
    print("cut, gate logits", flush=True)
    with torch.no_grad():
        o, ht = chunk_gla(*(t.to(device) for t in (q, k, v, x)), initial_state=h0.to(device), output_final_state=True,
                          head_first=False, gate_logit_normalizer=8.0)
    ro, rht = naive_recurrent_gla(q, k, v, F.logsigmoid(x) / 8.0, initial_state=h0, output_final_state=True)
    assert_close("o", ro, o, 1e-2)
    assert_close("ht", rht, ht, 5e-3)


GDR_CASES = [
    (1, 1601, 1, 64, 64, None, torch.bfloat16),      # 26 chunks, the last of one token
    (2, 2047, 2, 128, 128, None, torch.bfloat16),    # the last chunk of 63 tokens
    (1, 1856, 3, 128, 64, None, torch.float16),
    (1, 2500, 2, 64, 128, [0, 1, 1, 1900, 1964, 2500], torch.bfloat16),
    (1, 3200, 1, 128, 128, [0, 1790, 1854, 3200], torch.bfloat16),
]


@pytest.mark.parametrize("B,T,H,K,V,bounds,dtype", GDR_CASES)
@pytest.mark.parametrize("gated", [True, False])
def test_gdr_cut_sequences(device, B, T, H, K, V, bounds, dtype, gated):
    """A quarter of the keys' corrections and almost no decay: the transition of a segment is far from zero."""
    from fla_amd.ops.delta_rule import chunk_delta_rule
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule
    N = B if bounds is None else len(bounds) - 1
    offs = None if bounds is None else torch.tensor(bounds, device=device)
    assert _cut(N, T, H, V // 64, False, bounds, _delta(1, K)) and _cut(N, T, H, V // 64, True, bounds, _delta(2, K))
    print("cut delta rule", B, T, H, K, V, bounds, dtype, gated, flush=True)
    q, k, v, g, beta, h0 = gdr_inputs(B, T, H, K, V, seed=T, dtype=dtype, normalizer=2000.0, N=N)
    beta = beta * 0.02
    dev = [x.to(device) for x in (q, k, v, g, beta, h0)]

    def op(q, k, v, g, beta, h0, **kw):
        kw.update(initial_state=h0, output_final_state=True, cu_seqlens=offs, head_first=False)
        return chunk_gated_delta_rule(q, k, v, g, beta, **kw) if gated else chunk_delta_rule(q, k, v, beta, **kw)

    with torch.no_grad():
        o1, ht1 = op(*dev)
    leaves = [x.requires_grad_() for x in dev]
    o, ht = op(*leaves)
    do, dht = torch.randn(B, T, H, V).to(dtype), torch.randn(N, H, K, V) * 0.1
    torch.autograd.backward((o, ht), (do.to(device), dht.to(device)))
    refs = [x.float().requires_grad_() for x in (q, k, v, g, beta, h0)]
    ro, rht = naive_recurrent_gated_delta_rule(*refs[:3], refs[3] if gated else torch.zeros_like(refs[3]), refs[4],
                                               initial_state=refs[5], output_final_state=True, offsets=bounds)
    torch.autograd.backward((ro, rht), (do.float(), dht))
    for a, b in ((o1, ht1), (o, ht)):
        assert_close("o", ro, a, 1e-2)
        assert_close("ht", rht, b, 5e-3)
    for name, r, d in zip(("dq", "dk", "dv", "dg", "dbeta", "dh0"), refs, leaves):
        if name != "dg" or gated:
            assert_close(name, r.grad, d.grad, 2e-2)


@pytest.mark.parametrize("K,V", [(64, 64), (128, 128)])
def test_gdr_cut_l2norm_in_kernel(device, K, V):
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule
    from oracle.modules import l2norm
    q, k, v, g, beta, h0 = gdr_inputs(1, 1700, 2, K, V, seed=3, normalizer=2000.0)
    k = torch.randn(k.shape).to(k.dtype) * 3
    beta = beta * 0.02
    assert _cut(1, 1700, 2, V // 64, False, None, _delta(1, K))
    print("cut delta rule, raw q and k", K, V, flush=True)
    with torch.no_grad():
        o, ht = chunk_gated_delta_rule(*(t.to(device) for t in (q, k, v, g, beta)), initial_state=h0.to(device),
                                       output_final_state=True, head_first=False, use_qk_l2norm_in_kernel=True)
    ro, rht = naive_recurrent_gated_delta_rule(l2norm(q), l2norm(k), v, g, beta, initial_state=h0, output_final_state=True)
    assert_close("o", ro, o, 1e-2)
    assert_close("ht", rht, ht, 5e-3)


GRADIENT_CASES = [
    (1, 1985, 1, 64, 64, None, torch.bfloat16),                     # 32 chunks, the last of one token
    (2, 2303, 2, 128, 128, None, torch.float16),                    # 36 chunks, the last of 63 tokens
    (1, 2500, 2, 128, 64, [0, 0, 2111, 2112, 2500], torch.bfloat16),    # an empty sequence, one of a token, uneven ones
    (1, 2300, 2, 64, 128, [0, 2100, 2300], torch.float16),
]


@pytest.mark.parametrize("heads", [False, True])
@pytest.mark.parametrize("B,T,H,K,V,bounds,dtype", GRADIENT_CASES)
def test_gla_cut_state_gradients(device, B, T, H, K, V, bounds, dtype, heads):
    """A reverse scan over cut sequences against the fp32 recurrence (the cases above are cut in the forward only).  The
    tolerances are those of the cases above."""
    from fla_amd.ops.gla import chunk_gla
    from fla_amd.ops.simple_gla import chunk_simple_gla
    N = B if bounds is None else len(bounds) - 1
    assert _cut(N, T, H, K // 64 * (V // 64), True, bounds, 4)
    print("cut state gradients", B, T, H, K, V, bounds, dtype, heads, flush=True)
    q, k, v, g, h0 = gla_inputs(B, T, H, K, V, seed=T, dtype=dtype, normalizer=600.0, N=N)
    if heads:
        g = g[..., 0].contiguous()
    do, dht = torch.randn(B, T, H, V).to(dtype), torch.randn(N, H, K, V) * 0.1
    leaves = [x.to(device).requires_grad_() for x in (q, k, v, g, h0)]
    o, ht = (chunk_simple_gla if heads else chunk_gla)(
        *leaves[:4], initial_state=leaves[4], output_final_state=True, head_first=False,
        cu_seqlens=None if bounds is None else torch.tensor(bounds, device=device))
    torch.autograd.backward((o, ht), (do.to(device), dht.to(device)))
    refs = [x.float().requires_grad_() for x in (q, k, v, g, h0)]
    ro, rht = naive_recurrent_gla(*refs[:3], **{"g" if heads else "gk": refs[3]}, initial_state=refs[4],
                                  output_final_state=True, offsets=bounds)
    torch.autograd.backward((ro, rht), (do.float(), dht))
    for name, a, r in zip(("dq", "dk", "dv", "dg", "dh0"), leaves, refs):
        assert_close(name, r.grad, a.grad, 2e-2)


@pytest.mark.parametrize("B,T,H,K,V,bounds,dtype", GRADIENT_CASES)
def test_gla_cut_state_gradients_16bit_gates(device, B, T, H, K, V, bounds, dtype):
    """The same with gates in the dtype of q, k and v."""
    from fla_amd.ops.gla import chunk_gla
    N = B if bounds is None else len(bounds) - 1
    assert _cut(N, T, H, K // 64 * (V // 64), True, bounds, 4)
    print("cut state gradients, 16-bit gates", B, T, H, K, V, bounds, dtype, flush=True)
    q, k, v, g, h0 = gla_inputs(B, T, H, K, V, seed=T + 1, dtype=dtype, normalizer=600.0, N=N)
    g, do, dht = g.to(dtype), torch.randn(B, T, H, V).to(dtype), torch.randn(N, H, K, V) * 0.1
    leaves = [x.to(device).requires_grad_() for x in (q, k, v, g, h0)]
    o, ht = chunk_gla(*leaves[:4], initial_state=leaves[4], output_final_state=True, head_first=False,
                      cu_seqlens=None if bounds is None else torch.tensor(bounds, device=device))
    torch.autograd.backward((o, ht), (do.to(device), dht.to(device)))
    refs = [x.float().requires_grad_() for x in (q, k, v, g, h0)]
    ro, rht = naive_recurrent_gla(*refs[:4], initial_state=refs[4], output_final_state=True, offsets=bounds)
    torch.autograd.backward((ro, rht), (do.float(), dht))
    for name, a, r in zip(("dq", "dk", "dv", "dg", "dh0"), leaves, refs):
        assert_close(name, r.grad, a.grad, 2e-2)


@pytest.mark.parametrize("K,V,dtype", [(64, 64, torch.float16), (128, 128, torch.bfloat16), (64, 128, torch.bfloat16),
                                       (128, 64, torch.float16)])
@pytest.mark.parametrize("gated", [True, False])
def test_gdr_cut_backward_that_reads_w(device, K, V, dtype, gated):
    """The cut form of the entry that takes w (the operator's own backward reads the tiles) against its uncut form on the
    same kept tensors.  Where nothing enters from the right, the last segment, they run the same instructions (equal bits).
    Ahead of it the gradients that enter differ by the order of their fp32 sums and the rounding of the operands; either
    form may be off the recurrence by 2e-2 (bf16) or an eighth of it, twice that bounds their difference."""
    from fla_amd import _backend as be
    from fla_amd.ops.gated_delta_rule.wy_fast import fwd_prepare_scan_operands
    B, T, H = 2, 2020, 2
    q, k, v, g, beta, h0 = (x.to(device) for x in gdr_inputs(B, T, H, K, V, seed=5, dtype=dtype, normalizer=200.0))
    do, dht = torch.randn_like(v), torch.randn_like(h0)
    lib, p, scale, st, dims = be.lib(), be.ptr, K ** -0.5, be.stream_of(q), (B, T, H, K, V, B)
    AT, gc, w, Aw = fwd_prepare_scan_operands(k, beta, g if gated else None, keep_w=True)
    chunks = AT.shape[0]
    new = lambda *shape: q.new_empty(*shape)
    o, ht, v_new, hT, Aqk = torch.empty_like(v), torch.empty_like(h0), torch.empty_like(v), new(chunks, H, K * V), torch.empty_like(AT)
    sp, bufs = _split(q, B, T, H, V // 64, _delta(2, K), K * V, K * K)
    back = be.Split()
    assert lib.fla_scan_split(None, B, T, H, V // 64, 1, _delta(2, K), ctypes.byref(back), None, None, None)
    assert (back.nseg, back.sub_chunks, back.ratio, back.slots) == (sp.nseg, sp.sub_chunks, 1, sp.slots) and sp.nseg > 1
    Mt = torch.empty_like(bufs[1])
    sp.transitions_t = Mt.data_ptr()
    print("cut backward from w", K, V, dtype, gated, sp.nseg, sp.sub_chunks, flush=True)
    be.check(lib.fla_chunk_gated_delta_rule_fwd_scan_split(
        *map(p, (q, k, v, AT, gc)), None, *map(p, (h0, o, ht, v_new, hT, Aqk)), None, None, ctypes.byref(sp), be.dt(q), *dims, scale,
        0.0, st), "scan_split")
    states = torch.empty_like(bufs[0])
    back.states, back.decays = states.data_ptr(), Mt.data_ptr()
    results = []
    for split in (None, back):
        out = [torch.empty_like(x) for x in (q, k, v, beta, beta, h0)]
        dv2, dh = torch.empty_like(v), torch.empty_like(hT)
        head = (*map(p, (q, k, v, w, v_new, beta, gc, Aw, do, dht, hT, Aqk)),)
        tail = (p(dv2), p(dh), None, None, None, *map(p, out), None, None, None)
        if split is None:
            be.check(lib.fla_chunk_gated_delta_rule_bwd(*head, None, *tail, 0, be.dt(q), *dims, scale, st), "bwd")
        else:
            be.check(lib.fla_chunk_gated_delta_rule_bwd_split(*head, *tail, ctypes.byref(split), 0, be.dt(q), *dims, scale, st),
                     "bwd_split")
        results.append(dict(zip(("dq", "dk", "dv", "dbeta", "dg", "dh0"), out)))
    torch.cuda.synchronize()
    last = 64 * sp.sub_chunks * (sp.nseg - 1)
    assert last < T
    tol = 4e-2 / (1 if dtype == torch.bfloat16 else 8)
    for name, a in results[0].items():
        b = results[1][name]
        if name == "dg" and not gated:
            continue
        if name != "dh0":
            assert torch.equal(a[:, last:], b[:, last:]), name
        assert_close(name, a.float().cpu(), b.cpu(), tol)
    assert not torch.equal(results[0]["dh0"], results[1]["dh0"])   # (so that the comparison tells the two apart)


@pytest.mark.parametrize("heads", [False, True])
def test_gla_cut_state_behind_a_reset(device, heads):
    """A gate of -1e30 drops the state.  The tokens behind it inside its chunk keep their own decays, which a difference
    of sums that contain the reset would lose; what enters the next segment is made of them."""
    from fla_amd import _backend as be
    from fla_amd.ops.gla import chunk_gla
    T = 1000
    sp = be.Split()
    assert be.lib().fla_scan_split(None, 1, T, 2, 1, 0, 0, ctypes.byref(sp), None, None, None)
    seg = 64 * sp.sub_chunks * sp.ratio
    q, k, v, g, h0 = gla_inputs(1, T, 2, 64, 64, seed=9, normalizer=16.0)
    g[:, seg - 64 + 8] = -1e30          # the first row of a group of four, 55 tokens ahead of the next segment
    if heads:
        g = g[..., :1].expand(-1, -1, -1, 64).contiguous()
    print("cut, reset", heads, sp.sub_chunks, sp.ratio, flush=True)
    with torch.no_grad():
        o, ht = chunk_gla(*(t.to(device) for t in (q, k, v, g)), initial_state=h0.to(device), output_final_state=True,
                          head_first=False)
    ro, rht = naive_recurrent_gla(q, k, v, g, initial_state=h0, output_final_state=True)
    assert_close("o of the segments behind", ro[:, seg:], o[:, seg:], 1e-2)
    assert_close("ht", rht, ht, 5e-3)


def test_packed_batch_first_met_under_capture(device):
    """The tables of a cut are copied to the device by the first call that needs them, which a stream being captured does
    not take: such a call runs uncut, and one on another stream is cut with the same result."""
    from fla_amd.ops.gla import chunk_gla
    from fla_amd.utils import VarlenPlan
    bounds = [0, 1290, 1354, 2200]
    q, k, v, g, _ = (x.to(device) for x in gla_inputs(1, 2200, 1, 64, 64, seed=2, normalizer=600.0))
    offs = torch.tensor(bounds, device=device)
    VarlenPlan(offs, 64).native
    assert _cut(3, 2200, 1, 1, False, bounds)
    print("capture", flush=True)
    with torch.no_grad():
        chunk_gla(q, k, v, g, head_first=False)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            o, _ = chunk_gla(q, k, v, g, cu_seqlens=offs, head_first=False)
        side = torch.cuda.Stream()
        eager, _ = chunk_gla(q, k, v, g, cu_seqlens=offs, head_first=False)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            other, _ = chunk_gla(q, k, v, g, cu_seqlens=offs, head_first=False)
        torch.cuda.synchronize()
        assert torch.equal(eager, other)
        for _ in range(3):
            o.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert_close("o", eager.float().cpu(), o.cpu(), 1e-2)


@pytest.mark.parametrize("op", ["chunk_gla", "chunk_gla fp32", "chunk_gla head-first", "chunk_simple_gla",
                                "chunk_simple_gla, 16-bit state", "chunk_gated_delta_rule", "fused_recurrent_gla",
                                "fused_recurrent_gated_delta_rule", "fused_recurrent_gated_delta_rule, packed", "l2_norm",
                                "causal_conv1d", "causal_conv1d_update", "rms_norm_swish_gate", "gla_gate"])
@pytest.mark.parametrize("grad", [True, False])
def test_forward_mode_is_refused(device, op, grad):
    """No operator has a forward-mode derivative: a tangent is an error, not dropped."""
    import torch.autograd.forward_ad as fw
    from fla_amd import modules as m
    from fla_amd.modules.convolution import causal_conv1d, causal_conv1d_update
    from fla_amd.modules.fused_norm_gate import rms_norm_swish_gate_fn
    from fla_amd.modules.gate_activations import gla_gate
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule
    from fla_amd.ops.gla import chunk_gla, fused_recurrent_gla
    from fla_amd.ops.simple_gla import chunk_simple_gla
    q, k, v, g, beta, h0 = (x.to(device) for x in gdr_inputs(1, 70, 1, 64, 64, seed=1))
    gk, w, kw = g[..., None].expand(-1, -1, -1, 64).contiguous(), torch.randn(64, 4, device=device), dict(head_first=False)
    offs = torch.tensor([0, 30, 70], device=device)
    calls = {
        "chunk_gla": lambda x: chunk_gla(x, k, v, gk, **kw),
        "chunk_gla fp32": lambda x: chunk_gla(x.float(), k.float(), v.float(), gk, **kw),
        "chunk_gla head-first": lambda x: chunk_gla(x, k, v, gk),
        "chunk_simple_gla": lambda x: chunk_simple_gla(x, k, v, g, **kw),
        "chunk_simple_gla, 16-bit state": lambda x: chunk_simple_gla(x, k, v, g, initial_state=h0.bfloat16(), **kw),
        "chunk_gated_delta_rule": lambda x: chunk_gated_delta_rule(x, k, v, g, beta, **kw),
        "fused_recurrent_gla": lambda x: fused_recurrent_gla(x, k, v, gk, **kw),
        "fused_recurrent_gated_delta_rule": lambda x: fused_recurrent_gated_delta_rule(x, k, v, g, beta, **kw),
        "fused_recurrent_gated_delta_rule, packed":
            lambda x: fused_recurrent_gated_delta_rule(x, k, v, g, beta, cu_seqlens=offs, **kw),
        "l2_norm": m.l2_norm,
        "causal_conv1d": lambda x: causal_conv1d(x[:, :, 0], w),
        "causal_conv1d_update": lambda x: causal_conv1d_update(x[:, 0, 0], torch.zeros_like(w)[None].to(x.dtype), w),
        "rms_norm_swish_gate": lambda x: rms_norm_swish_gate_fn(x, v, None, None),
        "gla_gate": lambda x: gla_gate(x, 16.0),
    }
    with fw.dual_level(), torch.set_grad_enabled(grad):
        x = fw.make_dual(q, torch.ones_like(q))
        print("forward mode", op, flush=True)
        with pytest.raises(RuntimeError):
            calls[op](x)


@pytest.mark.parametrize("dtype,heads", [(torch.float16, False), (torch.float16, True), (torch.float32, False)])
def test_gla_cut_keeps_decayed_keys(device, dtype, heads):
    """Keys whose weight has decayed by e^-14 when their sub-block ends are all that its state is made of (the rest of the
    keys is zero, as behind a mask).  The decays of whole chunks multiply fp32 numbers: only the rounding of the 16-bit
    operands k e^{E} (E within a chunk) is left, 2^-11 of each at most and 2^-11 / sqrt(3) of their sum; fp32 inputs
    round v too."""
    from fla_amd import _backend as be
    from fla_amd.ops.gla import chunk_gla
    from fla_amd.ops.simple_gla import chunk_simple_gla
    T, H, D = 2048, 64, 64
    sp = be.Split()
    assert be.lib().fla_scan_split(None, 1, T, H, 1, 0, 0, ctypes.byref(sp), None, None, None)
    sub = 64 * sp.sub_chunks
    assert sub >= 512 and sub < T
    q, k, v, g, _ = gla_inputs(1, T, H, D, D, seed=4, dtype=dtype, h0=False)
    k[:, sub - 280:] = 0
    g[:, :sub], g[:, sub:] = -0.05, 0.0
    print("cut, decayed keys", dtype, heads, sub, flush=True)
    with torch.no_grad():
        x = [t.to(device) for t in (q, k, v, g)]
        if heads:
            o, ht = chunk_simple_gla(*x[:3], x[3][..., 0].contiguous(), output_final_state=True, head_first=False)
        else:
            o, ht = chunk_gla(*x, output_final_state=True, head_first=False)
    w = torch.exp(torch.flip(torch.cumsum(torch.flip(g.double(), [1]), 1), [1]) - g.double())
    ref = torch.einsum("bthk,bthv->bhkv", k.double() * w, v.double())
    assert_close("ht", ref, ht, 5e-4)


@pytest.mark.parametrize("K,V,dtype", [(64, 64, torch.bfloat16), (128, 128, torch.float16), (64, 128, torch.bfloat16),
                                       (128, 64, torch.bfloat16)])
@pytest.mark.parametrize("bounds", [None, [0, 1, 1, 2460, 2500]])
def test_gdr_cut_state_passes_in_fp32(device, K, V, dtype, bounds):
    """Tokens without a correction (beta = 0) and without decay leave the state, and from the right its gradient, as they
    are, bit by bit: every segment's transition is the identity and no bit of a state may be lost between them.  An entry
    that is not finite stays in its value column."""
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule
    T, H = 2500, 2
    N = 1 if bounds is None else len(bounds) - 1
    assert _cut(N, T, H, V // 64, False, bounds, _delta(1, K)) and _cut(N, T, H, V // 64, True, bounds, _delta(2, K))
    q, k, v, g, beta, h0 = (x.to(device) for x in gdr_inputs(1, T, H, K, V, seed=6, dtype=dtype, N=N))
    kw = dict(output_final_state=True, head_first=False,
              cu_seqlens=None if bounds is None else torch.tensor(bounds, device=device))
    print("cut, state passes", K, V, dtype, bounds, flush=True)
    with torch.no_grad():
        _, ht = chunk_gated_delta_rule(q, k, v, g * 0, beta * 0, initial_state=h0, **kw)
        assert torch.equal(ht, h0)
        h0[..., 3, 5] = float("inf")
        _, ht = chunk_gated_delta_rule(q, k, v, g * 0, beta * 0, initial_state=h0, **kw)
        rest = torch.arange(V, device=device) != 5
        assert torch.equal(ht[..., rest], h0[..., rest])
        h0[..., 3, 5] = 0.0
    h0.requires_grad_()
    o, ht = chunk_gated_delta_rule(q, k, v, g * 0, beta * 0, initial_state=h0, **kw)
    dht = torch.randn(ht.shape, device=device)
    torch.autograd.backward((o, ht), (torch.zeros_like(o), dht))
    assert torch.equal(ht, h0) and torch.equal(h0.grad, dht)


@pytest.mark.parametrize("op", ["chunk_gla", "chunk_simple_gla", "chunk_gated_delta_rule", "fp32", "K=96"])
def test_offsets_written_before_the_backward(device, op):
    """A cu_seqlens buffer that is filled again between a forward and its backward: refused, as for any saved tensor."""
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule
    from fla_amd.ops.gla import chunk_gla
    from fla_amd.ops.simple_gla import chunk_simple_gla
    dtype, K = torch.float32 if op == "fp32" else torch.bfloat16, 96 if op == "K=96" else 64
    q, k, v, g, beta, _ = (x.to(device) for x in gdr_inputs(1, 300, 2, K, K, seed=8, dtype=dtype, N=2))
    leaves = [x.requires_grad_() for x in (q, k, v)]
    offs = torch.tensor([0, 100, 300], device=device)
    print("offsets written", op, flush=True)
    kw = dict(head_first=False, cu_seqlens=offs)
    if op == "chunk_gated_delta_rule":
        o, _ = chunk_gated_delta_rule(*leaves, g, beta, **kw)
    elif op == "chunk_simple_gla":
        o, _ = chunk_simple_gla(*leaves, g, **kw)
    else:
        o, _ = chunk_gla(*leaves, g[..., None].expand(-1, -1, -1, K).contiguous(), **kw)
    offs.copy_(torch.tensor([0, 200, 300]))
    with pytest.raises(RuntimeError, match="inplace operation"):
        o.sum().backward()


@pytest.mark.parametrize("delta", [False, True])
def test_tables_of_a_cut_do_not_wait_for_the_device(device, delta):
    """New boundaries behind a queue of work: neither the forward nor the backward waits until it is done."""
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule
    from fla_amd.ops.gla import chunk_gla
    from fla_amd.utils import VarlenPlan
    T, bounds = 3200, [0, 1790, 1854, 3200]
    assert _cut(3, T, 1, 1, False, bounds, _delta(2, 64) * delta) and _cut(3, T, 1, 1, True, bounds, _delta(2, 64) if delta else 4)
    q, k, v, g, beta, _ = (x.to(device) for x in gdr_inputs(1, T, 1, 64, 64, seed=2, normalizer=600.0))
    gk = g[..., None].expand(-1, -1, -1, 64).contiguous()
    q.requires_grad_()
    do, a = torch.randn_like(v), torch.randn(8192, 8192, device=device, dtype=torch.bfloat16)

    def busy():
        for _ in range(40):
            torch.mm(a, a)
        done = torch.cuda.Event()
        done.record()
        return done

    for turn in range(3):   # the first two fill the allocators' pools
        q.grad = None
        offs = torch.tensor(bounds, device=device)
        VarlenPlan(offs, 64).native
        torch.cuda.synchronize()
        print("busy, forward", delta, flush=True)
        done = busy()
        kw = dict(head_first=False, cu_seqlens=offs)
        o, _ = chunk_gated_delta_rule(q, k, v, g, beta, **kw) if delta else chunk_gla(q, k, v, gk, **kw)
        assert turn < 2 or not done.query()
        torch.cuda.synchronize()
        done = busy()
        o.backward(do)
        assert turn < 2 or not done.query()
        torch.cuda.synchronize()


@pytest.mark.parametrize("B,T,H,K,V,bounds,dtype", CASES)
def test_gla_cut_16bit_gates(device, B, T, H, K, V, bounds, dtype):
    """Gates in the dtype of q, k and v: log-gates forward and backward, and pre-activations."""
    from fla_amd.ops.gla import chunk_gla
    N = B if bounds is None else len(bounds) - 1
    offs = None if bounds is None else torch.tensor(bounds, device=device)
    assert _cut(N, T, H, V // 64, False, bounds)   # (the reverse scan runs uncut: test_gla_cut_state_gradients)
    print("cut, 16-bit gates", B, T, H, K, V, bounds, dtype, flush=True)
    q, k, v, g, h0 = gla_inputs(B, T, H, K, V, seed=T, dtype=dtype, normalizer=600.0, N=N)
    g, do = g.to(dtype), torch.randn(B, T, H, V).to(dtype)
    kw = dict(output_final_state=True, cu_seqlens=offs, head_first=False)
    leaves = [x.to(device).requires_grad_() for x in (q, k, v, g, h0)]
    o, ht = chunk_gla(*leaves[:4], initial_state=leaves[4], **kw)
    torch.autograd.backward((o, ht), (do.to(device), torch.zeros_like(ht)))
    refs = [x.float().requires_grad_() for x in (q, k, v, g, h0)]
    ro, rht = naive_recurrent_gla(*refs[:4], initial_state=refs[4], output_final_state=True, offsets=bounds)
    ro.backward(do.float())
    assert_close("o", ro, o, 1e-2)
    assert_close("ht", rht, ht, 5e-3)
    for name, r, d in zip(("dq", "dk", "dv", "dg", "dh0"), refs, leaves):
        assert_close(name, r.grad, d.grad, 2e-2)
    x = torch.randn(g.shape).to(dtype)
    with torch.no_grad():
        o, ht = chunk_gla(*leaves[:3], x.to(device), gate_logit_normalizer=600.0, **kw)
        ro, rht = naive_recurrent_gla(*refs[:3], F.logsigmoid(x.float()) / 600.0, output_final_state=True, offsets=bounds)
    assert_close("o from logits", ro, o, 1e-2)
    assert_close("ht from logits", rht, ht, 5e-3)


@pytest.mark.parametrize("B,T,H,K,V,bounds,dtype", GDR_CASES)
@pytest.mark.parametrize("normalizer,states", [(1.0, True), (200.0, False), (200.0, True)])
def test_gdr_cut_ordinary_corrections(device, B, T, H, K, V, bounds, dtype, normalizer, states):
    """beta = sigmoid with ordinary and with weak gates, with and without states given from outside: the transition of a
    segment is far from the identity, and the folds start from zero."""
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule
    N = B if bounds is None else len(bounds) - 1
    offs = None if bounds is None else torch.tensor(bounds, device=device)
    assert _cut(N, T, H, V // 64, False, bounds, _delta(1, K)) and _cut(N, T, H, V // 64, True, bounds, _delta(2, K))
    print("cut, ordinary beta", B, T, H, K, V, bounds, dtype, normalizer, states, flush=True)
    q, k, v, g, beta, h0 = gdr_inputs(B, T, H, K, V, seed=T, dtype=dtype, normalizer=normalizer, N=N, h0=states)
    kw = dict(output_final_state=states, cu_seqlens=offs, head_first=False)
    leaves = [None if x is None else x.to(device).requires_grad_() for x in (q, k, v, g, beta, h0)]
    with torch.no_grad():
        o1, ht1 = chunk_gated_delta_rule(*leaves[:5], initial_state=leaves[5], **kw)
    o, ht = chunk_gated_delta_rule(*leaves[:5], initial_state=leaves[5], **kw)
    do, dht = torch.randn(B, T, H, V).to(dtype), torch.randn(N, H, K, V) * 0.1
    torch.autograd.backward((o, ht) if states else (o,), (do.to(device), dht.to(device)) if states else (do.to(device),))
    refs = [None if x is None else x.float().requires_grad_() for x in (q, k, v, g, beta, h0)]
    ro, rht = naive_recurrent_gated_delta_rule(*refs[:5], initial_state=refs[5], output_final_state=True, offsets=bounds)
    torch.autograd.backward((ro, rht) if states else (ro,), (do.float(), dht) if states else (do.float(),))
    for a, b in ((o1, ht1), (o, ht)):
        assert_close("o", ro, a, 1e-2)
        if states:
            assert_close("ht", rht, b, 5e-3)
    for name, r, d in zip(("dq", "dk", "dv", "dg", "dbeta", "dh0"), refs, leaves):
        if r is not None:
            assert_close(name, r.grad, d.grad, 2e-2)


def _split(like, N, T, H, slabs, kind, state, transition):
    """A cut of sequences of equal length with its workspaces."""
    from fla_amd import _backend as be
    sp = be.Split()
    assert be.lib().fla_scan_split(None, N, T, H, slabs, 0, kind, ctypes.byref(sp), None, None, None)
    bufs = [torch.empty(sp.slots * H * n, device=like.device) for n in (state, transition)]
    sp.states, sp.decays = (b.data_ptr() for b in bufs)
    return sp, bufs


@pytest.mark.parametrize("K,V,dtype", [(64, 64, torch.float16), (128, 128, torch.bfloat16), (64, 128, torch.bfloat16),
                                       (128, 64, torch.bfloat16)])
@pytest.mark.parametrize("op", ["gla", "gated_delta_rule"])
def test_cut_entry_against_the_uncut_one(device, K, V, dtype, op):
    """The same inputs through both entry points of the library, and the operator, which takes the cut one.  In the first
    segment they run the same instructions (equal bits).  Behind it the states that enter differ by the order of their fp32
    sums and by the rounding of their operands, 2^-9 (bf16) or 2^-12 of each at most; four times that bounds o and ht, which
    round by as much themselves."""
    from fla_amd import _backend as be
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule
    from fla_amd.ops.gla import chunk_gla
    B, T, H, delta = 2, 2020, 2, op != "gla"
    q, k, v, g, beta, h0 = (x.to(device) for x in gdr_inputs(B, T, H, K, V, seed=3, dtype=dtype, normalizer=200.0))
    if not delta:
        g = gla_inputs(B, T, H, K, V, seed=3, normalizer=200.0)[3].to(device)
    lib, p, scale, st = be.lib(), be.ptr, K ** -0.5, be.stream_of(q)
    sp, bufs = _split(q, B, T, H, V // 64, _delta(1, K) * delta, K * V, K * K if delta else K)
    assert sp.nseg > 1
    print("cut against uncut", op, K, V, dtype, sp.nseg, sp.sub_chunks, sp.ratio, flush=True)
    o, ht = [torch.empty_like(v) for _ in range(2)], [torch.empty_like(h0) for _ in range(2)]
    dims, chunks = (B, T, H, K, V, B), -(-T // 64) * B
    if delta:
        AT, gc = q.new_empty(chunks, H, 10, 16, 16), torch.empty_like(g)
        be.check(lib.fla_gdr_fwd_prep(p(k), p(beta), p(g), 0, p(gc), p(AT), None, None, None, None, 0, be.dt(q), *dims[:4], st), "prep")
        be.check(lib.fla_chunk_gated_delta_rule_fwd_scan(p(q), p(k), p(v), p(AT), p(gc), p(h0), p(o[0]), p(ht[0]), *[None] * 6,
                                                         be.dt(q), *dims, scale, st), "scan")
        be.check(lib.fla_chunk_gated_delta_rule_fwd_scan_split(p(q), p(k), p(v), p(AT), p(gc), None, p(h0), p(o[1]), p(ht[1]),
                                                               *[None] * 5, ctypes.byref(sp), be.dt(q), *dims, scale, 0.0, st),
                 "scan_split")
        call = lambda: chunk_gated_delta_rule(q, k, v, g, beta, initial_state=h0, output_final_state=True, head_first=False)
    else:
        ws = [torch.empty(chunks, H, dtype=torch.int32, device=device), q.new_empty(chunks, H, K * V)]
        be.check(lib.fla_chunk_gla_fwd_fused(*map(p, (q, k, v, g, h0, o[0], ht[0], *ws)), *[None] * 4, 0, be.dt(q), be.dt(g), *dims,
                                             scale, st), "fused")
        be.check(lib.fla_chunk_gla_fwd_fused_split(*map(p, (q, k, v, g, h0, o[1], ht[1], *ws)), *[None] * 8, ctypes.byref(sp), 0,
                                                   be.dt(q), be.dt(g), *dims, scale, 0, 1.0, 0, 0.0, st), "fused_split")
        call = lambda: chunk_gla(q, k, v, g, initial_state=h0, output_final_state=True, head_first=False)
    tol = 4 * 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    assert_close("o", o[0].cpu(), o[1].cpu(), tol)
    assert_close("ht", ht[0].cpu(), ht[1].cpu(), tol)
    first = 64 * sp.sub_chunks * sp.ratio
    assert torch.equal(o[0][:, :first], o[1][:, :first])
    assert not torch.equal(ht[0], ht[1])   # (so that the comparison below tells the two apart)
    with torch.no_grad():
        oo, hh = call()
    assert torch.equal(oo, o[1]) and torch.equal(hh, ht[1])


@pytest.mark.parametrize("bounds", [None, [0, 1790, 1854, 3200]])
def test_gdr_cut_forward_with_its_backward_under_capture(device, bounds):
    """The forward runs eagerly and leaves its transitions.  A backward that is captured finds no tables of its own for a
    packed batch and runs uncut; for one sequence it needs none."""
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule
    T, N = 3200, 1 if bounds is None else 3
    assert _cut(N, T, 1, 1, False, bounds, _delta(2, 64)) and _cut(N, T, 1, 1, True, bounds, _delta(2, 64))
    leaves = [x.to(device).requires_grad_() for x in gdr_inputs(1, T, 1, 64, 64, seed=2, normalizer=600.0, h0=False)[:5]]
    do = torch.randn(1, T, 1, 64, device=device).to(leaves[0].dtype)
    offs = None if bounds is None else torch.tensor(bounds, device=device)
    other = None if bounds is None else offs.clone()   # tables of its own
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())

    def forward(offs):
        return chunk_gated_delta_rule(*leaves, cu_seqlens=offs, head_first=False)[0]

    def backward(o):
        return torch.autograd.grad(o, leaves, do, retain_graph=True)

    with torch.cuda.stream(side):
        backward(forward(other))
        o = forward(offs)
    torch.cuda.synchronize()
    print("capture a backward", bounds, flush=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        grads = backward(o)
    with torch.cuda.stream(side):
        eager = backward(o)
    torch.cuda.synchronize()
    for _ in range(3):
        for x in grads:
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for name, r, d in zip(("dq", "dk", "dv", "dg", "dbeta"), eager, grads):
            assert_close(name, r.float().cpu(), d.float().cpu(), 2e-2)


@pytest.mark.parametrize("op", ["chunk_gla", "chunk_simple_gla", "chunk_gated_delta_rule"])
def test_cut_states_at_any_float_address(device, op):
    """An initial state and a gradient of the final one that begin four bytes behind a 16-byte boundary: the same bits."""
    from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule
    from fla_amd.ops.gla import chunk_gla
    from fla_amd.ops.simple_gla import chunk_simple_gla
    T, K = 2020, 64
    delta = op == "chunk_gated_delta_rule"
    assert _cut(1, T, 2, 1, False, None, _delta(2, K) * delta) and _cut(1, T, 2, 1, True, None, _delta(2, K) if delta else 4)
    q, k, v, g, beta, h0 = (x.to(device) for x in gdr_inputs(1, T, 2, K, K, seed=4, normalizer=200.0))
    do, dht = torch.randn(v.shape, device=device).to(v.dtype), torch.randn(h0.shape, device=device)

    def moved(x):
        y = torch.empty(x.numel() + 1, device=device)[1:].view(x.shape)
        assert y.data_ptr() % 16 == 4
        return y.copy_(x)

    def call(h0, dht):
        print("states at", h0.data_ptr() % 16, op, flush=True)
        leaves = [q.detach().requires_grad_(), h0.requires_grad_()]
        kw = dict(initial_state=h0, output_final_state=True, head_first=False)
        if delta:
            o, ht = chunk_gated_delta_rule(leaves[0], k, v, g, beta, **kw)
        elif op == "chunk_simple_gla":
            o, ht = chunk_simple_gla(leaves[0], k, v, g, **kw)
        else:
            o, ht = chunk_gla(leaves[0], k, v, g[..., None].expand(-1, -1, -1, K).contiguous(), **kw)
        return [o, ht, *torch.autograd.grad((o, ht), leaves, (do, dht))]

    for a, b in zip(call(h0.clone(), dht), call(moved(h0), moved(dht))):
        assert torch.equal(a, b)
