"""GPU kernels at the edges of their tiles and of their dispatch rules, against fp64 on the CPU."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _rand(*shape, dtype=torch.float32, seed=0, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype).cuda()


# One size per tile shape of the small- and medium-output kernel with remainders in M, N and K (32x64,
# 64x64, 64x128, 128x128, 256x128, the wide outputs of few rows), the smallest outputs, and K split
# over workgroups (M, N, K: K at least 8192, or 16384 for fewer than 256 rows).
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (136, 200, 72), (264, 3080, 136), (1000, 1992, 200), (1992, 2056, 72),
                                   (2056, 3080, 136), (24, 33000, 64), (136, 33032, 72), (264, 520, 8200),
                                   (104, 264, 16400)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, True), (True, False)])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                                             (torch.float32, torch.float32)])
def test_gemm_tile_choice_and_remainders(M, N, K, ta, tb, dtype, out_dtype):
    from qwen_triton.kernels.matmul import gemm

    if not ta and not tb:
        K += 8 if dtype != torch.float32 else 4  # another remainder of the last k-tile
    if ta:
        M = -(-M // 8) * 8  # a k-outer operand needs 16-byte aligned rows along M
    a = _rand(*((K, M) if ta else (M, K)), dtype=dtype, seed=1)
    b = _rand(*((K, N) if tb else (N, K)), dtype=dtype, seed=2, scale=0.1)
    bias = _rand(N, dtype=dtype, seed=3)
    # rows of C stand apart: nothing may be written between them
    out = torch.full((M, N + 8), 7.0, dtype=out_dtype, device="cuda")
    gemm(ta, tb, M, N, K, a, a.stride(0), b, b.stride(0), out, N + 8, bias)
    ad, bd = (t.cpu().double() for t in (a.T if ta else a, b if tb else b.T))
    ref = ad @ bd + bias.cpu().double()
    # fp32 sums of K exact products and the bias, then one rounding to the output type
    bound = (K + 1) * 2.0 ** -24 * (ad.abs() @ bd.abs() + bias.cpu().double().abs()) + EPS[out_dtype] * ref.abs()
    assert ((out[:, :N].cpu().double() - ref).abs() <= bound).all()
    assert (out[:, N:] == 7.0).all()


def test_gemm_asks_for_no_workspace_that_its_kernel_does_not_take():
    """Decode products (up to 128 rows, both operands k-contiguous) run in one launch whatever K is."""
    from qwen_triton import _native, kernels

    dt = torch.bfloat16
    x, w = _rand(64, 16384, dtype=dt, seed=1), _rand(512, 16384, dtype=dt, seed=2, scale=0.02)
    with torch.no_grad():
        kernels.triton_matmul(x, w)
        torch.cuda.synchronize()
        calls, used = _native.CALLS["qh_gemm_ws"], torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        out = kernels.triton_matmul(x, w)
    assert _native.CALLS["qh_gemm_ws"] == calls
    assert torch.cuda.max_memory_allocated() - used <= out.numel() * 2 + 512
    ref = x.cpu().double() @ w.cpu().double().T
    assert ((out.cpu().double() - ref).abs() <= 2 * EPS[dt] * ref.abs() + 1e-3).all()


def _delta_inputs(B, S, H, K, V, seed, initial):
    import torch.nn.functional as F

    g = torch.Generator().manual_seed(seed)
    q = F.normalize(torch.randn(B, S, H, K, generator=g), dim=-1).bfloat16()
    k = F.normalize(torch.randn(B, S, H, K, generator=g), dim=-1).bfloat16()
    v = torch.randn(B, S, H, V, generator=g).bfloat16()
    decay = -F.softplus(torch.randn(B, S, H, generator=g)) * 0.3
    beta = torch.sigmoid(torch.randn(B, S, H, generator=g))
    state = torch.randn(B, H, K, V, generator=g) * 0.2 if initial else None
    return q, k, v, decay, beta, state


def _delta_reference(q, k, v, decay, beta, state, dtype):
    """The recurrence token by token in ``dtype`` on the CPU (q scaled and rounded to its own type)."""
    B, S, H, K = q.shape
    q = (q * K ** -0.5).to(dtype)
    k, v, decay, beta = (t.to(dtype) for t in (k, v, decay, beta))
    st = torch.zeros(B, H, K, v.shape[-1], dtype=dtype) if state is None else state.to(dtype)
    outs = []
    for t in range(S):
        st = st * decay[:, t].exp()[..., None, None]
        d = (v[:, t] - (st * k[:, t, :, :, None]).sum(2)) * beta[:, t, :, None]
        st = st + k[:, t, :, :, None] * d[:, :, None, :]
        outs.append((st * q[:, t, :, :, None]).sum(2))
    return torch.stack(outs, 1), st


# From the shortest length that runs in chunks: last chunks of 1 to 64 tokens, around their 16-token
# blocks; both key sizes, value columns that end inside a workgroup's 64 and inside a wavefront's 16.
@pytest.mark.parametrize("S", [320, 321, 336, 337, 383, 384, 385])
@pytest.mark.parametrize("K,V,initial", [(128, 128, True), (64, 72, False), (128, 8, True)])
def test_delta_rule_chunks(S, K, V, initial):
    from qwen_triton.kernels import gated_delta_rule_sequence

    args = _delta_inputs(2, S, 3, K, V, 40 + S, initial)
    out, st = gated_delta_rule_sequence(*(None if t is None else t.cuda() for t in args[:5]),
                                        initial_state=None if args[5] is None else args[5].cuda())
    ro, rs = _delta_reference(*args, torch.float64)
    assert ((out.cpu().double() - ro).abs() <= EPS[torch.bfloat16] * ro.abs() + 2e-6).all()  # one rounding of fp32 sums
    # the state is as close to fp64 as the recurrence in fp32 is (a quarter for another order of the sums)
    err = lambda x: float((x.double() - rs).norm() / rs.norm())  # noqa: E731
    assert err(st.cpu()) <= 1.25 * err(_delta_reference(*args, torch.float32)[1])


# Keys with a common direction, of norm 1 (solved in chunks) and beyond (chunks whose update is no contraction
# run token by token), a call with both, and growing states (positive log-decays).
@pytest.mark.parametrize("K,V", [(128, 72), (64, 64)])
@pytest.mark.parametrize("norm,cosine,growth", [(1.0, 0.9, False), (1.4, 0.9, False), (1.6, 0.99, False),
                                                (2.0, 0.0, False), ("rising", 0.9, False), (1.0, 0.9, True)])
def test_delta_rule_chunks_of_related_keys(K, V, norm, cosine, growth):
    import torch.nn.functional as F

    from qwen_triton.kernels import gated_delta_rule_sequence

    q, k, v, decay, beta, state = _delta_inputs(1, 400, 3, K, V, 61, True)
    g = torch.Generator().manual_seed(62)
    common = F.normalize(torch.randn(1, 1, 3, K, generator=g), dim=-1)
    size = torch.linspace(1.0, 1.5, 400)[None, :, None, None] if norm == "rising" else norm
    k = (F.normalize(cosine ** 0.5 * common + (1 - cosine) ** 0.5 * k.float(), dim=-1) * size).bfloat16()
    beta = torch.sigmoid(2 + torch.randn(1, 400, 3, generator=g))
    decay = torch.full_like(decay, 0.01) if growth else decay * 0.3
    args = (q, k, v, decay, beta, state)
    out, st = gated_delta_rule_sequence(*(t.cuda() for t in args[:5]), initial_state=state.cuda())
    ro, rs = _delta_reference(*args, torch.float64)
    fo, fs = _delta_reference(*args, torch.float32)
    err = lambda x, r: float((x.double() - r).norm() / r.norm())  # noqa: E731
    # the state is as close to fp64 as the recurrence in fp32 (a quarter for another order of the sums);
    # solved chunks of related keys up to twice as far: their corrections are as large as the values
    solved = norm == 1.0 or norm == "rising"
    assert err(st.cpu(), rs) <= (2.0 if solved else 1.25) * err(fs, rs)
    assert err(out.cpu(), ro) <= EPS[torch.bfloat16] + 2 * err(fo, ro)


def test_delta_rule_split_at_a_chunk_boundary():
    """Two launches of at least 320 tokens, split at a multiple of 64: the bits of one launch."""
    from qwen_triton.kernels import gated_delta_rule_sequence as rule

    q, k, v, g, b, s0 = (t.cuda() for t in _delta_inputs(1, 750, 2, 128, 128, 5, True))
    out, st = rule(q, k, v, g, b, initial_state=s0)
    o1, s1 = rule(*(t[:, :384] for t in (q, k, v, g, b)), initial_state=s0)
    o2, s2 = rule(*(t[:, 384:] for t in (q, k, v, g, b)), initial_state=s1)
    assert torch.equal(torch.cat((o1, o2), 1), out) and torch.equal(s2, st)


@pytest.mark.parametrize("S,first", [(384, 320), (448, 64), (401, 400), (700, 350)])
def test_delta_rule_continued_by_a_call_of_another_kind(S, first):
    """A call of fewer than 320 tokens runs token by token, and a split off the 64-token grid moves the chunks:
    two calls through the state are then as close to 64 bits as one, not equal to it in every bit."""
    from qwen_triton.kernels import gated_delta_rule_sequence as rule

    args = _delta_inputs(1, S, 2, 128, 64, 9, True)
    q, k, v, g, b, s0 = (t.cuda() for t in args)
    o1, s1 = rule(*(t[:, :first] for t in (q, k, v, g, b)), initial_state=s0)
    o2, s2 = rule(*(t[:, first:] for t in (q, k, v, g, b)), initial_state=s1)
    ro, rs = _delta_reference(*args, torch.float64)
    err = lambda x: float((x.double() - rs).norm() / rs.norm())  # noqa: E731
    assert err(s2.cpu()) <= 1.25 * err(_delta_reference(*args, torch.float32)[1])
    out = torch.cat((o1, o2), 1).cpu().double()
    assert ((out - ro).abs() <= EPS[torch.bfloat16] * ro.abs() + 2e-6).all()


@pytest.mark.parametrize("case", ["nan_value", "inf_value", "nan_key", "reset", "reset_all"])
def test_delta_rule_chunks_not_finite(case):
    """A NaN or infinity reaches its own and later tokens only; a log-decay of -inf clears the state."""
    from qwen_triton.kernels import gated_delta_rule_sequence

    args = list(_delta_inputs(1, 400, 2, 128, 64, 77, True))
    if case == "nan_value":
        args[2][0, 75, 1, 5] = float("nan")
    elif case == "inf_value":
        args[2][0, 75, 1, 5] = float("inf")
    elif case == "nan_key":
        args[1][0, 75, 1, 5] = float("nan")
    elif case == "reset":
        args[3][0, 75, 1] = -float("inf")
    else:
        args[3][0, :, 1] = -float("inf")
    out, st = gated_delta_rule_sequence(*(t.cuda() for t in args[:5]), initial_state=args[5].cuda())
    ro, rs = _delta_reference(*args, torch.float64)
    out, st = out.cpu().double(), st.cpu().double()
    assert torch.equal(torch.isfinite(out), torch.isfinite(ro)) and torch.equal(torch.isfinite(st), torch.isfinite(rs))
    ok = torch.isfinite(ro)
    assert ((out - ro)[ok].abs() <= EPS[torch.bfloat16] * ro[ok].abs() + 2e-6).all()
    ok = torch.isfinite(rs)
    assert ((st - rs)[ok].abs() <= 1e-6 * (1 + rs[ok].abs())).all()


@pytest.mark.parametrize("Sk", [1, 31, 33, 128, 129, 257, 500])
def test_decode_attention_rotated_tiles(Sk):
    """One workgroup per (sequence, kv-head): every starting tile, partial last tiles, waves without
    a tile, per-sequence lengths."""
    from qwen_triton.kernels.flash_attention import flash_decode

    B, Hq, Hkv, D = 66, 16, 8, 128
    q = _rand(B, Hq, 1, D, dtype=torch.bfloat16, seed=1)
    k, v = (_rand(B, Hkv, Sk + 3, D, dtype=torch.bfloat16, seed=2 + i)[:, :, :Sk] for i in range(2))
    lens = torch.randint(1, Sk + 1, (B,), generator=torch.Generator().manual_seed(4))
    lens[0] = Sk
    out = flash_decode(q, k, v, D ** -0.5, Hq // Hkv, seqlens=lens.to(torch.int32).cuda()).cpu().double()
    qd, kd, vd = (t.cpu().double() for t in (q, k, v))
    kd, vd = (t.repeat_interleave(2, dim=1) for t in (kd, vd))
    s = torch.matmul(qd, kd.transpose(2, 3)) * D ** -0.5
    s = s.masked_fill(torch.arange(Sk)[None, None, None, :] >= lens[:, None, None, None], float("-inf"))
    p = torch.softmax(s, -1)
    ref = torch.matmul(p, vd)
    # probabilities and outputs are rounded to bf16 once each
    assert ((out - ref).abs() <= EPS[torch.bfloat16] * (torch.matmul(p, vd.abs()) + ref.abs()) + 1e-6).all()


# One workgroup up to 2048 assignments and 256 experts, the sort beyond; ids out of range sort last.
@pytest.mark.parametrize("T,k,E", [(1, 1, 1), (1, 8, 128), (64, 8, 128), (9, 7, 5), (256, 8, 256), (257, 8, 256),
                                   (100, 4, 257)])
def test_moe_dispatch_orders_like_a_stable_sort(T, k, E):
    from qwen_triton import _native

    g = torch.Generator().manual_seed(T + E)
    sel = torch.stack([torch.randperm(max(E, k), generator=g)[:k] for _ in range(T)])
    sel = torch.where(torch.rand(T, k, generator=g) < 0.05, torch.tensor(-1), sel)
    wt = torch.randn(T, k, generator=g).bfloat16()
    n, dev = T * k, "cuda"
    s, w = sel.cuda(), wt.cuda()
    ws = _native.workspace(_native.call("qh_moe_dispatch_workspace", T, k, E), s.device)
    rows, inv = (torch.full((n,), -7, dtype=torch.int32, device=dev) for _ in range(2))
    wsorted = torch.empty(n, dtype=torch.bfloat16, device=dev)
    seg, toff = (torch.full((E + 1,), -7, dtype=torch.int32, device=dev) for _ in range(2))
    _native.call("qh_moe_dispatch", s.data_ptr(), w.data_ptr(), T, k, E, 128, ws.data_ptr(), ws.numel(),
                 rows.data_ptr(), wsorted.data_ptr(), inv.data_ptr(), seg.data_ptr(), toff.data_ptr(),
                 _native.dtype_code(w.dtype), _native.stream(s.device))
    keys = torch.where((sel >= 0) & (sel < E), sel, torch.tensor(E)).flatten()
    order = torch.sort(keys, stable=True).indices
    counts = torch.bincount(keys, minlength=E + 1)[:E]
    assert torch.equal(rows.cpu().long(), order // k) and torch.equal(wsorted.cpu(), wt.flatten()[order])
    assert torch.equal(inv.cpu().long(), torch.sort(order).indices)
    zero = torch.zeros(1, dtype=torch.long)
    assert torch.equal(seg.cpu().long(), torch.cat((zero, counts.cumsum(0))))
    assert torch.equal(toff.cpu().long(), torch.cat((zero, ((counts + 127) // 128).cumsum(0))))


@pytest.mark.parametrize("T", [1, 33, 250])
@pytest.mark.parametrize("dtype,I", [(torch.bfloat16, 136), (torch.float16, 192)])
def test_moe_experts_few_rows(T, dtype, I):
    """The weight-streaming kernel: experts of no row, of one, of one to several 16-row blocks and (the
    fixed assignment) of more than 64 and more than 128 rows; output columns that end inside a
    workgroup's."""
    from qwen_triton.kernels.moe_experts import moe_experts_forward

    E, k, H = 24, 2, 192
    g = torch.Generator().manual_seed(T)
    sel = torch.stack([torch.randperm(E - 4, generator=g)[:k] for _ in range(T)])  # four experts see no token
    if T == 250:
        sel[:200, 0] = 3
        sel[:200, 1] = torch.where(torch.arange(200) < 70, 5, 7)
    x, rw = _rand(T, H, dtype=dtype, seed=1), _rand(T, k, dtype=dtype, seed=2, scale=0.5)
    gate, up = (_rand(E, I, H, dtype=dtype, seed=3 + i, scale=0.1) for i in range(2))
    down = _rand(E, H, I, dtype=dtype, seed=5, scale=0.1)
    gu = torch.tensor([t[e].data_ptr() for e in range(E) for t in (gate, up)], dtype=torch.int64, device="cuda")
    dn = torch.tensor([down[e].data_ptr() for e in range(E)], dtype=torch.int64, device="cuda")
    out = moe_experts_forward(x, rw, sel.cuda(), gu, dn, E, I, (H, I)).cpu().double()
    xd, rd, gd, ud, dd = (t.cpu().double() for t in (x, rw, gate, up, down))
    ref, mag = torch.zeros(T, H, dtype=torch.float64), torch.zeros(T, H, dtype=torch.float64)
    for t in range(T):
        for j in range(k):
            e = int(sel[t, j])
            a = gd[e] @ xd[t]
            h = a * torch.sigmoid(a) * (ud[e] @ xd[t])
            y = (dd[e] @ h) * rd[t, j]
            ref[t] += y
            mag[t] += (dd[e].abs() @ h.abs()) * rd[t, j].abs() + y.abs()
    # gate, up, their product, the expert output, its scaled copy and each of the k sums round once
    assert ((out - ref).abs() <= (6 + k) * EPS[dtype] * mag + 1e-4).all()


# 64x64, 64x128 and 128x128 tiles, remainders in M, N and K, uneven products with and without biases.
@pytest.mark.parametrize("M,ns,K", [(517, (256, 128, 200), 200), (517, (1024, 1024, 512), 264),
                                    (517, (2048, 1024, 1024), 72), (1000, (2048, 1024, 1024), 1024),
                                    (300, (1536, 1544), 136)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gemm_group_equals_the_separate_products(M, ns, K, dtype):
    from qwen_triton import kernels
    from qwen_triton.kernels.matmul import linear_group, linear_group_rows_ok

    x = _rand(M, K, dtype=dtype, seed=1)
    ws = [_rand(n, K, dtype=dtype, seed=2 + i, scale=0.1) for i, n in enumerate(ns)]
    bs = [None] + [_rand(n, dtype=dtype, seed=9 + i) for i, n in enumerate(ns[1:])]
    with torch.no_grad():
        served = linear_group_rows_ok(x, ws, bs)
        # a product small enough for the 32x64 tile, whose k is split otherwise, keeps its own launch
        assert served == all(-(-M // 32) * -(-n // 64) > 256 for n in ns)
        if served:
            for w, b, o in zip(ws, bs, linear_group(x, ws, bs)):
                assert torch.equal(o, kernels.triton_matmul(x, w, b))
        n = ns[0] // 64 * 64
        gu = [ws[0][:n], _rand(n, K, dtype=dtype, seed=20, scale=0.1)]
        # (517, 1024): 64x128 tiles; (517, 2048) and (1000, 2048): 128x128
        gated = linear_group_rows_ok(x, gu, gated=True)
        assert gated == (-(-M // 32) * (n // 64) > 256)
        if gated:
            want = kernels.silu_mul(kernels.triton_matmul(x, gu[0]), kernels.triton_matmul(x, gu[1]))
            got = linear_group(x, gu, gated=True)
            if dtype == torch.bfloat16:
                assert torch.equal(got, want)
            else:  # the compiler may fold the last product into its conversion to fp16: one unit
                assert ((got.double() - want.double()).abs() <= 2.0 ** -10 * want.double().abs() + 2.0 ** -24).all()


# Under vmap the projections have no memory to launch on: the modules are called, as for any other shape.
def test_grouped_rows_under_vmap(monkeypatch):
    from qwen_triton.kernels import matmul, swiglu
    from qwen_triton.modules import QwenMLP

    monkeypatch.delenv("QWEN_TRITON_STRICT", raising=False)
    dt = torch.bfloat16
    torch.manual_seed(0)
    mlp = QwenMLP(256, 2048).to("cuda", dt).eval()
    x = _rand(2, 300, 256, dtype=dt, seed=1)
    with torch.no_grad():
        assert matmul.linear_group_rows_ok(x[0], [mlp.gate_proj.weight, mlp.up_proj.weight], gated=True)
        want = torch.stack([mlp(t) for t in x]).double()
        try:
            with pytest.warns(RuntimeWarning):
                got = torch.vmap(mlp)(x).double()
        finally:
            matmul._GUARD.reset()
            swiglu._GUARD.reset()
    # three bf16 roundings of sums in another order
    assert (got - want).norm() <= 4 * EPS[dt] * want.norm()


# Rows that a product has to copy first are not copied to look at them.
@pytest.mark.parametrize("form", ["every_other", "overlapping", "expanded", "plain"])
def test_grouped_rows_are_not_copied_to_look_at_them(form):
    from qwen_triton import kernels
    from qwen_triton.kernels.matmul import linear_group, linear_group_rows_ok

    M, K, dt = 300, 256, torch.bfloat16
    base = _rand(M * 2 * K, dtype=dt, seed=1)
    x = dict(every_other=base.view(M, 2 * K)[:, ::2], overlapping=base.as_strided((M, K), (8, 1)),
             expanded=base[:K].expand(2, M // 2, K), plain=base.view(M, 2 * K)[:, :K])[form]
    ws = [_rand(n, K, dtype=dt, seed=2 + i, scale=0.1) for i, n in enumerate((2048, 2056))]
    with torch.no_grad():
        linear_group_rows_ok(x, ws)
        count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]  # noqa: E731
        before = count()
        assert linear_group_rows_ok(x, ws)
        assert count() == before
        for w, o in zip(ws, linear_group(x, ws)):
            assert torch.equal(o, kernels.triton_matmul(x, w))


# From K = 8192 on the separate products split K over workgroups: they keep their launches, and their bits.
@pytest.mark.parametrize("K", [8184, 8192])
def test_gemm_group_leaves_split_products_alone(K):
    from qwen_triton import kernels
    from qwen_triton.modules import QwenMLP

    dt = torch.bfloat16
    torch.manual_seed(0)
    mlp = QwenMLP(K, 1536).to("cuda", dt).eval()
    x = _rand(1, 517, K, dtype=dt, seed=1)
    seen = []
    mlp.down_proj.register_forward_pre_hook(lambda m, a: seen.append(a[0]))
    with torch.no_grad():
        mlp(x)
        want = kernels.silu_mul(mlp.gate_proj(x), mlp.up_proj(x))
    assert torch.equal(seen[0], want)


# A prompt past 128 rows calls a projection module that does more than its product (a forward hook, a
# replaced forward), and its result is used.
@pytest.mark.parametrize("how", ["hook", "pre_hook", "forward"])
def test_grouped_rows_leave_no_module_behaviour_out(how):
    from qwen_triton.modules import QwenMLP

    torch.manual_seed(0)
    mlp = QwenMLP(1024, 3072).to("cuda", torch.bfloat16).eval()
    x = _rand(1, 517, 1024, dtype=torch.bfloat16, seed=1)
    with torch.no_grad():
        plain = mlp(x)
        if how == "hook":
            mlp.gate_proj.register_forward_hook(lambda m, a, y: -y)
        elif how == "pre_hook":
            mlp.gate_proj.register_forward_pre_hook(lambda m, a: (-a[0],))
        else:
            own = mlp.gate_proj.forward
            mlp.gate_proj.forward = lambda t: -own(t)
        got = mlp(x)
        gate, up = x @ mlp.gate_proj.weight.T, x @ mlp.up_proj.weight.T
        want = torch.nn.functional.silu(-gate) * up @ mlp.down_proj.weight.T
    assert not torch.equal(got, plain)
    # three bf16 roundings (products, activation, output), each 2^-8 of values that add up in quadrature
    assert (got - want).double().norm() <= 4 * EPS[torch.bfloat16] * want.double().norm()


# Rows so far apart that a lane's 32-bit byte offset would not reach them (the vector-ALU kernel).
@pytest.mark.parametrize("dtype,stride", [(torch.bfloat16, 320_000_000), (torch.float32, 160_000_000)])
def test_gemm_rows_far_apart(dtype, stride):
    from qwen_triton.kernels.matmul import gemm

    M, N, K = 32, 64, 64
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 20 GB of device memory")
    a = torch.empty(stride * (M - 1) + K, dtype=dtype, device="cuda").as_strided((M, K), (stride, 1))
    a.copy_(_rand(M, K, dtype=dtype, seed=1))
    b = _rand(K, N, dtype=dtype, seed=2)
    out = torch.empty(M, N, dtype=dtype, device="cuda")
    gemm(False, True, M, N, K, a, stride, b, N, out, N)
    ad, bd = a.cpu().double(), b.cpu().double()
    bound = (K + 1) * 2.0 ** -24 * (ad.abs() @ bd.abs()) + EPS[dtype] * (ad @ bd).abs()
    assert ((out.cpu().double() - ad @ bd).abs() <= bound).all()
    del a
    torch.cuda.empty_cache()


# Up to 256 blocks of 64 queries: two groups of wavefronts take the key tiles in turn (one tile more for the
# first group, equally many, none for the second); the same sequences in a batch of more blocks: one group.
@pytest.mark.parametrize("Sq,Sk,off", [(65, 65, 0), (128, 128, 0), (129, 192, 63), (33, 1000, 967), (300, 300, 0),
                                       (20, 300, -5)])
@pytest.mark.parametrize("D,causal,masked", [(128, True, False), (64, False, False), (24, True, False),
                                             (128, True, True)])
def test_flash_forward_key_groups(Sq, Sk, off, D, causal, masked):
    from qwen_triton.kernels import flash_attention as FA

    Hq, Hkv, dt = 2, 1, torch.bfloat16
    q, k, v = (_rand(1, h, n, D, dtype=dt, seed=i) for i, (h, n) in enumerate([(Hq, Sq), (Hkv, Sk), (Hkv, Sk)]))
    see = torch.ones(Sq, Sk, dtype=torch.bool)
    if causal:
        see &= torch.arange(Sk)[None] <= torch.arange(Sq)[:, None] + off
    kw = {}
    if masked:  # a window, and padding whose last keys lie in the second tile
        pad, window = min(70, Sk - 1), 90
        ok = torch.arange(Sk) >= pad
        kw = dict(key_bits=FA.pack_key_bits(ok[None].cuda()), window=window)
        see &= ok[None] & (torch.arange(Sk)[None] > torch.arange(Sq)[:, None] + off - window)
    s = (q.cpu().double() @ k.cpu().double().transpose(-1, -2)) * D ** -0.5
    s = s.masked_fill(~see, float("-inf"))
    p = torch.softmax(s, -1).nan_to_num(0.0)
    want, lse_want = p @ v.cpu().double(), torch.logsumexp(s, -1)
    # probabilities rounded to bf16 (relative 2^-8 each) and the output's own rounding
    bound = EPS[dt] * (p @ v.cpu().double().abs() + want.abs()) + 1e-4
    for reps in (1, 129):
        if masked and reps > 1:
            kw["key_bits"] = kw["key_bits"].expand(reps, -1).contiguous()
        out, lse = FA.flash_forward(*(t.expand(reps, -1, -1, -1).contiguous() for t in (q, k, v)), D ** -0.5, causal,
                                    Hq // Hkv, off, **kw)
        for b in {0, reps - 1}:
            assert ((out[b:b + 1].cpu().double() - want).abs() <= bound).all()
            fin = torch.isfinite(lse_want[0])
            got = lse.view(reps, Hq, Sq)[b].cpu().double()
            assert (torch.isfinite(got) == fin).all()
            assert ((got - lse_want[0]).abs()[fin] <= 1e-4).all()


# Half a workgroup per CU up to one: the shortest and longest streams of the rule, a position in the
# first, a middle and the last tile, with and without non-temporal loads.
@pytest.mark.parametrize("B,Sk", [(16, 513), (16, 3072), (25, 700), (32, 1111)])
def test_decode_prepare_of_a_middling_batch(B, Sk):
    from qwen_triton import _native
    from qwen_triton.kernels.flash_attention import flash_decode

    Hq, Hkv, D, dt = 16, 8, 128, torch.bfloat16
    assert _native.call("qh_flash_decode_prepare_ok", B, Hq, Hkv, Sk, D)
    assert not _native.call("qh_flash_decode_prepare_ok", 16, Hq, Hkv, 3073, D)
    q2, k2, v2 = (_rand(B, h * D, dtype=dt, seed=i) for i, h in enumerate((Hq, Hkv, Hkv)))
    wq, wk = (_rand(D, dtype=dt, seed=5 + i) for i in range(2))
    ang = torch.arange(D // 2).float() * 0.1
    cos, sin = (torch.cat((f(ang), f(ang)))[None, None].to(dt).cuda() for f in (torch.cos, torch.sin))
    kv = _rand(B, Hkv, Sk, 2, D, dtype=dt, seed=9)
    for pos in (0, Sk // 2, Sk - 1):
        outs = []
        for fused in (True, False):
            base = kv.clone()
            kc, vc = base[:, :, :, 0], base[:, :, :, 1]
            p = torch.tensor([pos], device="cuda")
            common = (cos.data_ptr(), sin.data_ptr())
            code = _native.dtype_code(dt)
            if fused:
                out = torch.empty(B, Hq, D, dtype=dt, device="cuda")
                _native.call("qh_flash_decode_prepare", q2.data_ptr(), Hq * D, k2.data_ptr(), Hkv * D, v2.data_ptr(),
                             Hkv * D, wq.data_ptr(), wk.data_ptr(), 1e-6, 0, *common, cos.stride(0), 1, D,
                             kc.data_ptr(), *kc.stride()[:3], vc.data_ptr(), *vc.stride()[:3], Sk, p.data_ptr(),
                             out.data_ptr(), None, None, B, Hq, Hkv, Sk, D, D ** -0.5, code, code, code,
                             _native.stream(out.device))
            else:
                q = torch.empty(B, Hq, 1, D, dtype=dt, device="cuda")
                _native.call("qh_attn_prepare", q2.data_ptr(), Hq * D, k2.data_ptr(), Hkv * D, v2.data_ptr(), Hkv * D,
                             wq.data_ptr(), wk.data_ptr(), 1e-6, 0, *common, cos.stride(0), cos.stride(1), 1, D,
                             q.data_ptr(), kc.data_ptr(), *kc.stride()[:3], vc.data_ptr(), *vc.stride()[:3],
                             p.data_ptr(), B, 1, Hq, Hkv, D, Sk, code, code, code, _native.stream(q.device))
                out = flash_decode(q, kc, vc, D ** -0.5, Hq // Hkv)[:, :, 0]
            outs.append((out, base))
        assert torch.equal(outs[0][1], outs[1][1])  # the same rows written
        # probabilities round to bf16 in another order of the keys; then one rounding each
        err = (outs[0][0].double() - outs[1][0].double()).abs()
        assert (err <= 3 * EPS[dt] * (kv[:, :, :, 1].double().abs().mean() + outs[1][0].double().abs())).all()


# The same for the 256x256 tiles, whose loading waves reach rows 32 further on: the widest stride that they
# take and the first that they do not.
@pytest.mark.parametrize("stride", [(1 << 25) - 8, 1 << 25, 1 << 26])
def test_gemm_large_output_of_rows_far_apart(stride):
    from qwen_triton.kernels.matmul import gemm

    M, N, K, dt = 256, 32776, 64, torch.bfloat16
    if torch.cuda.mem_get_info()[0] < 50 << 30:
        pytest.skip("needs 35 GB of device memory")
    a = torch.empty(stride * (M - 1) + K, dtype=dt, device="cuda").as_strided((M, K), (stride, 1))
    a.copy_(_rand(M, K, dtype=dt, seed=1))
    b = _rand(N, K, dtype=dt, seed=2)
    out = torch.empty(M, N, dtype=dt, device="cuda")
    gemm(False, False, M, N, K, a, stride, b, K, out, N)
    ad, bd = a.cpu().double(), b.cpu().double()
    ref = ad @ bd.T
    bound = (K + 1) * 2.0 ** -24 * (ad.abs() @ bd.T.abs()) + EPS[dt] * ref.abs()
    assert ((out.cpu().double() - ref).abs() <= bound).all()
    del a
    torch.cuda.empty_cache()


# A prompt whose rows lie past the grouped launch's 32-bit lane offsets runs as separate products.
def test_grouped_rows_far_apart():
    from qwen_triton.kernels.matmul import linear_group_rows_ok
    from qwen_triton.modules import QwenMLP

    M, H, stride, dt = 161, 1024, 1 << 27, torch.bfloat16
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 44 GB of device memory")
    torch.manual_seed(0)
    mlp = QwenMLP(H, 3072).to("cuda", dt).eval()
    far = torch.empty(stride * (M - 1) + H, dtype=dt, device="cuda").as_strided((M, H), (stride, 1))
    far.copy_(_rand(M, H, dtype=dt, seed=1))
    near = far.contiguous()
    with torch.no_grad():
        weights = [mlp.gate_proj.weight, mlp.up_proj.weight]
        assert linear_group_rows_ok(near, weights, gated=True) and not linear_group_rows_ok(far, weights, gated=True)
        want, got = mlp(near).double(), mlp(far).double()
    # the same roundings of fp32 sums in another order: three bf16 roundings that may fall the other way
    assert (got - want).norm() <= 4 * EPS[dt] * want.norm()
    del far
    torch.cuda.empty_cache()


def _expert_gemm(mode, a, rows, table, ldb, n, wrow, seg, toff, E):
    from qwen_triton import _native

    R = rows.shape[0] if rows is not None else a.shape[0]
    out = torch.full((R, n), 7.0, dtype=a.dtype, device="cuda")
    _native.call("qh_moe_gemm", mode, a.data_ptr(), a.stride(0), None if rows is None else rows.data_ptr(),
                 table.data_ptr(), ldb, out.data_ptr(), n, None if wrow is None else wrow.data_ptr(), seg.data_ptr(),
                 toff.data_ptr(), R, E, n, a.shape[1], _native.dtype_code(a.dtype), _native.stream(a.device))
    return out


def _expert_segments(counts):
    c = torch.tensor(counts)
    zero = torch.zeros(1, dtype=torch.long)
    return tuple(torch.cat((zero, x.cumsum(0))).to(torch.int32).cuda() for x in (c, (c + 127) // 128))


# The scaled product's rows are contiguous whatever row list it is handed: few rows per expert (weights
# streamed) and many (128-row tiles).
@pytest.mark.parametrize("counts", [(5, 0, 40, 19), (200, 0, 150, 130)])
def test_moe_scaled_product_reads_contiguous_rows(counts):
    E, K, N, dt = len(counts), 128, 264, torch.bfloat16
    seg, toff = _expert_segments(counts)
    R = sum(counts)
    a, w, down = _rand(R, K, dtype=dt, seed=1), _rand(R, dtype=dt, seed=2), _rand(E, N, K, dtype=dt, seed=3)
    table = torch.tensor([down[e].data_ptr() for e in range(E)], dtype=torch.int64, device="cuda")
    rows = (torch.arange(R, device="cuda") // 2).to(torch.int32)
    want = _expert_gemm(1, a, None, table, K, N, w, seg, toff, E)
    assert torch.equal(_expert_gemm(1, a, rows, table, K, N, w, seg, toff, E), want)
    expert = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ref = torch.einsum("rk,rnk->rn", a.cpu().double(), down.cpu().double()[expert]) * w.cpu().double()[:, None]
    # the product and its scaled copy round once each
    assert ((want.cpu().double() - ref).abs() <= 2.1 * EPS[dt] * ref.abs() + 1e-3).all()


# A row list entry below 0 is a row of zeros, in the first, a middle and the last place of a segment.
@pytest.mark.parametrize("counts", [(5, 0, 40, 19), (200, 0, 150, 130)])
def test_moe_gated_product_of_missing_rows(counts):
    E, K, N, dt = len(counts), 128, 136, torch.bfloat16
    seg, toff = _expert_segments(counts)
    R, T = sum(counts), 30
    x, gu = _rand(T, K, dtype=dt, seed=1), _rand(2 * E, N, K, dtype=dt, seed=3, scale=0.2)
    table = torch.tensor([w.data_ptr() for w in gu], dtype=torch.int64, device="cuda")
    rows = torch.arange(R, device="cuda") % T
    want = _expert_gemm(0, x, rows.to(torch.int32), table, K, N, None, seg, toff, E)
    gone = torch.tensor([0, 2, 4, 5, 17, R - 1], device="cuda")
    rows[gone] = -1
    got = _expert_gemm(0, x, rows.to(torch.int32), table, K, N, None, seg, toff, E)
    want[gone] = 0
    assert torch.equal(got, want)


# However few rows the experts have on average, the tiles of one with more than 64 are 128-row tiles: the
# bits of a call whose average is high. One with 64 rows is streamed.
@pytest.mark.parametrize("mode,N", [(0, 136), (1, 264)])
@pytest.mark.parametrize("count", [64, 65, 128, 193, 130])
def test_moe_full_expert_among_empty_ones(mode, N, count):
    K, dt = 1216, torch.bfloat16
    x, w = _rand(count, K, dtype=dt, seed=1), _rand(count, dtype=dt, seed=2)
    mats = _rand(2, N, K, dtype=dt, seed=3, scale=0.1)
    rows = torch.arange(count, device="cuda").flip(0).to(torch.int32)
    outs = []
    for E in (1, 9):
        table = torch.tensor([m.data_ptr() for m in (mats if mode == 0 else mats[:1])] * E, dtype=torch.int64,
                             device="cuda")
        seg, toff = _expert_segments([0] * (E // 2) + [count] + [0] * (E // 2))
        outs.append(_expert_gemm(mode, x, rows if mode == 0 else None, table, K, N, w if mode else None, seg, toff, E))
    if count > 64:
        assert torch.equal(outs[0], outs[1])
    # fp32 sums of the same products in another order: a rounding or two of the result either way
    err = (outs[0].double() - outs[1].double()).abs()
    assert (err <= 4 * EPS[dt] * outs[0].double().abs() + 1e-3).all()


def test_moe_tokens_on_few_experts_are_not_streamed_twice():
    """4096 rows on 8 of 128 experts take about as long as on 8 of 8, where the average rows per expert alone
    choose the 128-row tiles (1.0 times; 1.7 when every tile was streamed, 64 rows a pass)."""
    K, N, n, dt = 2048, 768, 512, torch.bfloat16
    x, gu = _rand(n, K, dtype=dt, seed=1), _rand(16, N, K, dtype=dt, seed=2, scale=0.02)
    rows = (torch.arange(8 * n, device="cuda") % n).to(torch.int32)

    def best(E):
        table = torch.tensor([gu[i % 16].data_ptr() for i in range(2 * E)], dtype=torch.int64, device="cuda")
        seg, toff = _expert_segments([n] * 8 + [0] * (E - 8))
        times = []
        for _ in range(10):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                _expert_gemm(0, x, rows, table, K, N, None, seg, toff, E)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    assert best(128) <= 1.3 * best(8)


# One workgroup per (sequence, kv-head) starts long streams at different parts: a sequence's result may not
# depend on its place in the batch (equal sequences in slots of every starting part), and it is right where
# parts hold no tile, one or many; lengths on both sides of the 960 keys up to which a stream is not parted.
@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (16, 8), (32, 8), (64, 8)])
@pytest.mark.parametrize("Sk", [700, 961, 1111, 2050])
def test_decode_attention_does_not_depend_on_the_slot(Hq, Hkv, Sk):
    from qwen_triton.kernels.flash_attention import flash_decode

    n, reps, D, dt = 6, 11, 128, torch.bfloat16  # 6 sequences, each in 11 slots
    q, k, v = (_rand(n, h, s, D, dtype=dt, seed=i) for i, (h, s) in enumerate([(Hq, 1), (Hkv, Sk), (Hkv, Sk)]))
    lens = torch.tensor([Sk, 960, 961, Sk - 1, 33, (Sk + 961) // 2], dtype=torch.int32).clamp(max=Sk)
    slot = torch.arange(n * reps) % n
    i = slot.cuda()
    out = flash_decode(q[i], k[i].contiguous(), v[i].contiguous(), D ** -0.5, Hq // Hkv, seqlens=lens[slot].cuda())
    assert torch.equal(out, out[:n][i])
    qd, kd, vd = (t.cpu().double() for t in (q, k, v))
    kd, vd = (t.repeat_interleave(Hq // Hkv, dim=1) for t in (kd, vd))
    s = torch.matmul(qd, kd.transpose(2, 3)) * D ** -0.5
    s = s.masked_fill(torch.arange(Sk)[None, None, None, :] >= lens[:, None, None, None], float("-inf"))
    p = torch.softmax(s, -1)
    ref = torch.matmul(p, vd)
    # probabilities and outputs are rounded to bf16 once each
    bound = EPS[dt] * (torch.matmul(p, vd.abs()) + ref.abs()) + 1e-6
    assert ((out[:n].cpu().double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("Hq,Hkv", [(16, 8), (64, 8)])
@pytest.mark.parametrize("key", [5, 900, 1400, 2000])
def test_decode_attention_of_an_infinite_value(Hq, Hkv, key):
    """An infinity among the values reaches its own output dimension as an infinity, whatever part of the
    stream it lies in, and nothing else."""
    from qwen_triton.kernels.flash_attention import flash_decode

    B, Sk, D, dt = 66, 2050, 128, torch.bfloat16
    q, k, v = (_rand(B, h, s, D, dtype=dt, seed=i) for i, (h, s) in enumerate([(Hq, 1), (Hkv, Sk), (Hkv, Sk)]))
    v[:, 3, key, 17] = float("inf")
    out = flash_decode(q, k, v, D ** -0.5, Hq // Hkv).view(B, Hkv, Hq // Hkv, D)
    assert (out[:, 3, :, 17] == float("inf")).all()
    out[:, 3, :, 17] = 0
    assert torch.isfinite(out).all()


# The step that prepares its own rows: the same, for 8 wavefronts (32 sequences) and 4.
@pytest.mark.parametrize("B,Sk,pos", [(32, 1100, 1099), (32, 970, 100), (32, 600, 599), (72, 2050, 1300)])
def test_decode_step_does_not_depend_on_the_slot(B, Sk, pos):
    from qwen_triton import _native

    Hq, Hkv, D, dt, n = 16, 8, 128, torch.bfloat16, 4
    i = torch.arange(B, device="cuda") % n
    q2, k2, v2 = (_rand(n, h * D, dtype=dt, seed=j)[i] for j, h in enumerate((Hq, Hkv, Hkv)))
    wq, wk = (_rand(D, dtype=dt, seed=5 + j) for j in range(2))
    cos, sin = (torch.full((1, 1, D), c, dtype=dt, device="cuda") for c in (0.8, 0.6))
    kc, vc = (_rand(n, Hkv, Sk, D, dtype=dt, seed=9 + j)[i].contiguous() for j in range(2))
    out = torch.empty(B, Hq, D, dtype=dt, device="cuda")
    p, code = torch.tensor([pos], device="cuda"), _native.dtype_code(dt)
    _native.call("qh_flash_decode_prepare", q2.data_ptr(), Hq * D, k2.data_ptr(), Hkv * D, v2.data_ptr(), Hkv * D,
                 wq.data_ptr(), wk.data_ptr(), 1e-6, 0, cos.data_ptr(), sin.data_ptr(), D, 1, D, kc.data_ptr(),
                 *kc.stride()[:3], vc.data_ptr(), *vc.stride()[:3], Sk, p.data_ptr(), out.data_ptr(), None, None, B, Hq,
                 Hkv, Sk, D, D ** -0.5, code, code, code, _native.stream(out.device))
    assert torch.equal(out, out[:n][i]) and torch.equal(kc, kc[:n][i])
