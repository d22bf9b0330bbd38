"""The row-per-wave kernels of narrow rows against the float64 oracle, at the
row widths, source counts and row counts where they can go wrong: one chunk
less and more than a whole KiB, the narrowest row, waves without a row."""

import math

import numpy as np
import pytest
import torch

import kotodama_amd
from kotodama_amd import _capi, ops
from oracle import attnres_oracle as O

from .test_gpu_accumulate import _call, _case
from .test_gpu_backward import Norm, _bwd_kernel_name, bwd_queries_kernel, check_grad, make_case, np64, oracle_grads
from .test_gpu_parity import check_bf16, check_weights, merge_kernel, route_kernel

pytestmark = pytest.mark.gpu


def test_narrow_backward_policy(gpu):
    auto = _capi.POLICY_AUTO
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    assert _bwd_kernel_name(9, 4 * cus, 512, auto) == "attnres_route_bwd_rows_c1_s9"
    assert _bwd_kernel_name(5, 8192, 520, auto) == "attnres_route_bwd_rows_c2_s5"
    assert _bwd_kernel_name(5, 8192, 1536, auto) == "attnres_route_bwd_rows_c3_s5"
    assert _bwd_kernel_name(5, 4 * cus - 1, 512, auto) == "attnres_route_bwd_bf_gbf_s5_v1"
    assert _bwd_kernel_name(10, 8192, 512, auto) == "attnres_route_bwd_bf_gbf_s10_v1"
    assert _bwd_kernel_name(5, 8192, 1544, auto) == "attnres_route_bwd_bf_gbf_s5_v1"


CASES = [(8, 2, 3, None), (504, 9, 1030, None), (512, 9, 2049, None), (520, 1, 1025, None), (1000, 5, 1027, None),
         (1024, 8, 1500, None), (1032, 3, 1100, torch.float32), (1536, 9, 1026, None), (1536, 4, 1, None)]


@pytest.mark.parametrize("D,S,N,pd", CASES, ids=[f"D{c[0]}-S{c[1]}-N{c[2]}{'-pf32' if c[3] else ''}" for c in CASES])
def test_narrow_backward_matches_oracle(gpu, D, S, N, pd):
    print(f"narrow backward D={D} S={S} N={N} param={pd}", flush=True)
    assert _bwd_kernel_name(S, N, D, _capi.POLICY_STREAM) == f"attnres_route_bwd_rows_c{(D + 511) // 512}_s{S}"
    buf, query, gain, G = make_case(gpu, S, 0, 1, N, D, torch.bfloat16, seed=500 + S + D + N, param_dtype=pd)
    buf.requires_grad_(True)
    query.requires_grad_(True)
    norm = Norm(gain.clone(), 1e-5)
    mask = torch.ones(S, dtype=torch.bool, device=gpu)
    prev = _capi.set_kernel_policy(_capi.POLICY_STREAM)
    try:
        out = kotodama_amd.route_static(buf, query, norm, mask, S)
        (out.float() * G).sum().backward()
        torch.cuda.synchronize()
    finally:
        _capi.set_kernel_policy(prev)
    dx, dq, dg = oracle_grads(buf, S, query, norm.weight, G, 1e-5, pd or torch.bfloat16)
    check_grad(buf.grad.reshape(S, -1, D), dx, torch.bfloat16, "dsources")
    check_grad(query.grad, dq, query.dtype, "dquery")
    check_grad(norm.weight.grad, dg, query.dtype, "dgain")


@pytest.mark.parametrize("D,S,N", [(520, 9, 1030), (512, 1, 1025), (1536, 6, 1100)])
def test_narrow_backward_adds_in_place(gpu, D, S, N):
    # addend rows (here the gradient rows themselves) for every other source: those sources get
    # the plain gradient plus the addend within one rounding of it, the others its exact bits
    src, q, gain, gout, addend = _case(gpu, S, N, D, torch.bfloat16, 900 + S)
    prev = _capi.set_kernel_policy(_capi.POLICY_STREAM)
    try:
        plain = torch.full_like(src, 3.0)
        dq0, dg0 = _call(gpu, src, q, gain, gout, plain, None)
        grads = addend.clone()
        dq1, dg1 = _call(gpu, src, q, gain, gout, grads, [grads[s] if s % 2 == 0 else None for s in range(S)])
    finally:
        _capi.set_kernel_policy(prev)
    assert torch.equal(dq0, dq1) and torch.equal(dg0, dg1)
    for s in range(S):
        if s % 2:
            assert torch.equal(grads[s], plain[s])
        else:
            # plain is rounded to bf16 (2^-9 of it) and the sum once more (2^-9 of the sum)
            want = plain[s].double() + addend[s].double()
            bar = 2.0**-8 * (plain[s].double().abs() + want.abs()) + 1e-30
            assert ((grads[s].double() - want).abs() <= bar).all()


@pytest.mark.parametrize("D,S,lo,hi", [(1000, 4, 3000, 3300), (4096, 9, 300, 400)])
def test_cached_and_streamed_sources_agree(gpu, D, S, lo, hi):
    # the row-per-workgroup kernel reads up to 24 MiB of sources without the non-temporal hint:
    # the same rows in a call on either side of that line route to the same bits
    assert S * lo * D * 2 <= 24 << 20 < S * hi * D * 2
    g = torch.Generator(device=gpu).manual_seed(D)
    buf = torch.randn((S, hi, D), generator=g, device=gpu).to(torch.bfloat16)
    query = (torch.randn(D, generator=g, device=gpu) * 0.05).to(torch.bfloat16)
    norm = Norm(torch.ones(D, device=gpu, dtype=torch.bfloat16), 1e-5)
    mask = torch.ones(S, dtype=torch.bool, device=gpu)
    with torch.no_grad():
        small = kotodama_amd.route_static(buf[:, :lo].contiguous(), query, norm, mask, S)
        large = kotodama_amd.route_static(buf, query, norm, mask, S)
    assert torch.equal(small, large[:lo])


MERGE_CASES = [(8, 5, None), (504, 1100, None), (520, 2049, torch.float32), (1536, 1027, None), (2560, 1025, None),
               (3072, 3, None)]


@pytest.mark.parametrize("D,N,qd", MERGE_CASES, ids=[f"D{c[0]}-N{c[1]}{'-qf32' if c[2] else ''}" for c in MERGE_CASES])
def test_row_per_wave_merge_backward_matches_oracle(gpu, D, N, qd):
    print(f"row-per-wave merge backward D={D} N={N} query={qd}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(D + N)
    p, inter = ((torch.randn(1, N, D, generator=g) * s).to(torch.bfloat16).to(gpu).requires_grad_() for s in (2, 1))
    q = (torch.randn(D, generator=g) * 0.1).to(qd or torch.bfloat16).to(gpu).requires_grad_()
    lse = torch.randn(1, N, generator=g).to(gpu).requires_grad_()
    G = torch.randn(1, N, D, generator=g).to(torch.bfloat16).to(gpu)
    prev = _capi.set_kernel_policy(_capi.POLICY_STREAM)
    try:
        out = ops.merge_call(p, q, inter, lse, 1e-5)
        out.backward(G)
        torch.cuda.synchronize()
    finally:
        _capi.set_kernel_policy(prev)
    b = O.merge_backward(np64(p).reshape(N, D), np64(q), np64(inter).reshape(N, D), np64(lse).reshape(N), 1e-5,
                         np64(G).reshape(N, D))
    check_grad(p.grad.reshape(N, D), b["dpartial"], torch.bfloat16, "dpartial")
    check_grad(inter.grad.reshape(N, D), b["dinter"], torch.bfloat16, "dinter")
    check_grad(lse.grad.reshape(N), b["dlse"], torch.float32, "dlse")
    check_grad(q.grad, b["dq"], q.dtype, "dquery")


QUERY_CASES = [(8, 3, 5, 2), (504, 8, 1030, 8), (520, 5, 1027, 5), (1024, 3, 1025, 6), (1016, 1, 2, 8)]


@pytest.mark.parametrize("D,S,N,Q", QUERY_CASES, ids=[f"D{c[0]}-S{c[1]}-N{c[2]}-Q{c[3]}" for c in QUERY_CASES])
def test_row_per_wave_batched_backward_matches_oracle(gpu, D, S, N, Q):
    print(f"row-per-wave batched backward D={D} S={S} N={N} Q={Q}", flush=True)
    v = 1 if D <= 512 else 2
    assert bwd_queries_kernel(S, D, torch.bfloat16, Q) == f"attnres_route_bwd_mqg_rows_v{v}_s{S}_q{(Q + 3) // 4}"
    g = torch.Generator(device="cpu").manual_seed(D + S + N)
    buf = torch.randn(S, 1, N, D, generator=g).to(torch.bfloat16).to(gpu).requires_grad_()
    qs = (torch.randn(Q, D, generator=g) * 0.05).to(torch.bfloat16).to(gpu).requires_grad_()
    G = torch.randn(Q, 1, N, D, generator=g).to(torch.bfloat16).to(gpu)
    GL = torch.randn(Q, 1, N, generator=g).to(gpu)
    out, _, lse, _, _ = ops.route_call(buf, S, qs, None, 1e-5, torch.bfloat16, want_lse=True)
    torch.autograd.backward([out, lse], [G, GL])
    x, dx = np64(buf).reshape(S, N, D), 0
    for j in range(Q):
        b = O.route_backward(x, np64(qs[j]), 1e-5, np64(G[j]).reshape(N, D), np64(GL[j]).reshape(N))
        dx = dx + b["dx"]
        check_grad(qs.grad[j], b["dqw"], torch.bfloat16, f"dquery[{j}]")
    check_grad(buf.grad.reshape(S, N, D), dx, torch.bfloat16, "dsources")


# (hidden, sources, rows, queries, gain) of the grouped query-gradient pass: exactly 64 KiB of sums,
# two and three row groups that each walk several rows, a second pass over a ragged last query with
# the per-query reduction
GROUPED_CASES = [(2048, 4, 2051, 8, False), (1288, 3, 3001, 5, True), (1024, 3, 1030, 9, False),
                 (1024, 2, 700, 9, True)]


@pytest.mark.parametrize("D,S,N,Q,with_gain", GROUPED_CASES,
                         ids=[f"D{c[0]}-S{c[1]}-N{c[2]}-Q{c[3]}" for c in GROUPED_CASES])
def test_grouped_query_gradients_match_oracle(gpu, D, S, N, Q, with_gain):
    print(f"grouped query gradients D={D} S={S} N={N} Q={Q}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(D + S + N)
    bf = torch.bfloat16
    buf = torch.randn(S, 1, N, D, generator=g).to(bf).to(gpu)
    qs = (torch.randn(Q, D, generator=g) * 0.05).to(bf).to(gpu).requires_grad_()
    gain = (1 + 0.1 * torch.randn(D, generator=g)).to(bf).to(gpu).requires_grad_() if with_gain else None
    G = torch.randn(Q, 1, N, D, generator=g).to(bf).to(gpu)
    buf.requires_grad_()
    out = ops.route_call(buf, S, qs, gain, 1e-5, bf)[0]
    out.backward(G)
    x, dx, dgain = np64(buf).reshape(S, N, D), 0, 0
    for j in range(Q):
        b = O.route_backward(x, O.fold_query(np64(qs[j]), np64(gain) if with_gain else None, "bf16"), 1e-5,
                             np64(G[j]).reshape(N, D))
        dx = dx + b["dx"]
        dgain = dgain + b["dqw"] * np64(qs[j])
        check_grad(qs.grad[j], b["dqw"] * (np64(gain) if with_gain else 1.0), bf, f"dquery[{j}]")
    check_grad(buf.grad.reshape(S, N, D), dx, bf, "dsources")
    if with_gain:
        check_grad(gain.grad, dgain, bf, "dgain")


FORWARD_MERGE_CASES = [(8, 1024, None), (504, 1025, None), (520, 3001, torch.float32), (1536, 1030, None)]


@pytest.mark.parametrize("D,N,qd", FORWARD_MERGE_CASES,
                         ids=[f"D{c[0]}-N{c[1]}{'-qf32' if c[2] else ''}" for c in FORWARD_MERGE_CASES])
def test_narrow_merge_matches_oracle(gpu, D, N, qd):
    print(f"narrow merge D={D} N={N} query={qd}", flush=True)
    assert merge_kernel(N, D, qd or torch.bfloat16) == f"attnres_merge_rows_c{(D + 511) // 512}"
    g = torch.Generator(device="cpu").manual_seed(D + N)
    p = (torch.randn(N, D, generator=g) * 2).to(torch.bfloat16).to(gpu)
    inter = torch.randn(N, D, generator=g).to(torch.bfloat16).to(gpu)
    q = (torch.randn(D, generator=g) * 0.1).to(qd or torch.bfloat16).to(gpu)
    lse = torch.randn(N, generator=g).to(gpu)
    with torch.no_grad():
        out, logit, inv = ops.merge(p, q, inter, lse, 1e-5)
    ref = O.merge(np64(p), np64(q), np64(inter), np64(lse), 1e-5)
    check_bf16(out, ref["out"], f"narrow merge D={D} N={N}")
    np.testing.assert_allclose(np64(logit), ref["logit"], rtol=1e-4, atol=1e-4)
    np.testing.assert_allclose(np64(inv), ref["inv_rms"], rtol=1e-5)


def test_narrow_routing_policy(gpu):
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    assert route_kernel(2, 4 * cus, 1032, 1) == "attnres_route_rows_c3_s2"
    assert route_kernel(9, 8192, 1536, 1) == "attnres_route_rows_c3_s9"
    for s, n, d, q in ((2, 4 * cus - 1, 1536, 1), (1, 8192, 1536, 1), (10, 8192, 1536, 1), (5, 8192, 1024, 1),
                       (5, 8192, 1544, 1), (5, 8192, 1536, 2)):
        assert "_rows_" not in route_kernel(s, n, d, q), (s, n, d, q)
    prev = _capi.set_kernel_policy(_capi.POLICY_STREAM)
    try:
        assert "_rows_" not in route_kernel(5, 8192, 1536, 1)
    finally:
        _capi.set_kernel_policy(prev)


# (hidden, sources, rows, separate allocations, gain): the narrowest and the widest row, a third
# chunk of one lane, half and all lanes, the fewest rows, waves without a row, one and two
# workgroups per CU (from 64 rows per CU on one, with 5 sources and more)
ROUTE_CASES = [(1032, 2, 1024, False, True), (1032, 9, 16391, False, False), (1280, 5, 1027, True, True),
               (1536, 3, 2049, True, False), (1536, 4, 4097, False, True), (1528, 6, 1100, False, True),
               (1536, 7, 1025, True, True), (1272, 8, 1500, True, False), (1536, 9, 3001, False, True)]


@pytest.mark.parametrize("D,S,N,separate,with_gain", ROUTE_CASES, ids=[f"D{c[0]}-S{c[1]}-N{c[2]}" for c in ROUTE_CASES])
def test_narrow_routing_matches_oracle_and_workgroup_kernel(gpu, D, S, N, separate, with_gain):
    print(f"narrow routing D={D} S={S} N={N}", flush=True)
    assert route_kernel(S, N, D, 1) == f"attnres_route_rows_c3_s{S}"
    g = torch.Generator(device=gpu).manual_seed(D + S + N)
    bf, canary, pad_in, pad_out = torch.bfloat16, 7.0, 64, 32
    big = torch.full((S + 1, N, D + pad_in), canary, device=gpu, dtype=bf)
    rows = [big[s] for s in range(S)]
    if separate:  # not equally spaced
        rows = [big[s] for s in [S, *range(S - 1)]]
    for s, r in enumerate(rows):
        r[:, :D] = (torch.randn((N, D), generator=g, device=gpu) * (0.3 + 0.4 * s)).to(bf)
    query = (torch.randn(D, generator=g, device=gpu) * 0.05).to(bf)
    gain = (1 + 0.1 * torch.randn(D, generator=g, device=gpu)).to(bf) if with_gain else None

    def call():
        out = torch.full((N, D + pad_out), canary, device=gpu, dtype=bf)
        w, lse = torch.empty((S, N), device=gpu), torch.empty(N, device=gpu)
        inv, lg = torch.empty((N, S), device=gpu), torch.empty((N, S), device=gpu)
        _capi.route_fwd(_capi.pointer_array([r.data_ptr() for r in rows]), S, N, D, D + pad_in, _capi.DTYPE_BF16,
                        query.data_ptr(), None if gain is None else gain.data_ptr(), 1, _capi.DTYPE_BF16, 1e-5,
                        out.data_ptr(), _capi.DTYPE_BF16, D + pad_out, N * (D + pad_out), w.data_ptr(),
                        lse.data_ptr(), inv.data_ptr(), lg.data_ptr(), torch.cuda.current_stream(gpu).cuda_stream)
        torch.cuda.synchronize()
        assert (out[:, D:] == canary).all(), "output padding written"
        return out[:, :D], w, lse, inv, lg

    out, w, lse, inv, lg = call()
    pick = np.unique(np.concatenate([np.arange(0, 64), np.arange(N // 2, N // 2 + 64), np.arange(N - 64, N)]))
    qw = np64(query) if gain is None else np64(query * gain)  # rounded to bf16, as the kernels fold it
    ref = O.route(np.stack([np64(r[pick, :D]) for r in rows]), qw, 1e-5)
    check_bf16(out[pick], ref["out"][0], f"D={D} S={S}")
    check_weights(w[:, pick], ref["weights"][0], f"D={D} S={S}")
    np.testing.assert_allclose(np64(lse[pick]), ref["lse"][0], rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(np64(inv[pick]), ref["inv_rms"], rtol=1e-5)
    np.testing.assert_allclose(np64(lg[pick]), ref["logits"][0], rtol=1e-4, atol=1e-4)
    # every row against the workgroup kernel, with rows of zeros, an infinity, a NaN and the largest
    # value (whose squares overflow) among them
    for i, v in enumerate((0.0, math.inf, math.nan, torch.finfo(bf).max)):
        for r in rows[i % 2:]:
            r[5 * i, :D if v == 0 else 1] = v
    mine = call()
    prev = _capi.set_kernel_policy(_capi.POLICY_WORKGROUP)
    try:
        other = call()
    finally:
        _capi.set_kernel_policy(prev)
    for a, b, name in zip(mine, other, ("out", "weights", "lse", "inv_rms", "logits")):
        a, b = a.double(), b.double()
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()), name
        ok = a.isfinite()
        # bf16 rounding of two fp32 evaluations: one ulp (2^-7 relative) beside the fp32 difference
        rel, ab = (2.0**-7, 1e-4) if name == "out" else (1e-4, 1e-4)
        assert ((a - b).abs()[ok] <= rel * b.abs()[ok] + ab).all(), name


def _odd_rows(*bufs):
    """Rows of zeros, an infinity, a NaN and the largest value (whose squares overflow) into (n, D) rows."""
    for i, v in enumerate((0.0, math.inf, math.nan, torch.finfo(torch.bfloat16).max)):
        for r in bufs:
            r[5 * i, : r.shape[1] if v == 0 else 1] = v


def _agree(mine, other, rel, names):
    """Infinities and NaN in the same places, and every finite value within ``rel`` of the other's."""
    for a, b, r, name in zip(mine, other, rel, names):
        a, b = a.double(), b.double()
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()), name
        ok = b.isfinite()
        assert ((a - b).abs()[ok] <= r * b.abs()[ok] + 1e-4).all(), name


def _both_policies(call):
    res = []
    for policy in (_capi.POLICY_AUTO, _capi.POLICY_WORKGROUP):
        prev = _capi.set_kernel_policy(policy)
        try:
            res.append(call())
        finally:
            _capi.set_kernel_policy(prev)
    return res


# one bf16 ulp (2^-7 relative) between the roundings of two fp32 evaluations
ULP = 2.0**-7


@pytest.mark.parametrize("D,S,N", [(520, 5, 1030), (1024, 9, 1100), (1536, 3, 1026)])
@pytest.mark.parametrize("add", [False, True], ids=["plain", "add"])
def test_narrow_backward_of_odd_values_as_the_workgroup_kernel(gpu, D, S, N, add):
    print(f"narrow backward, odd values D={D} S={S} N={N} add={add}", flush=True)
    assert _bwd_kernel_name(S, N, D, _capi.POLICY_AUTO) == f"attnres_route_bwd_rows_c{(D + 511) // 512}_s{S}"
    src, q, gain, gout, addend = _case(gpu, S, N, D, torch.bfloat16, 40 + S)
    _odd_rows(*src[::2])
    gout[25, 0], gout[30, 0] = math.inf, math.nan

    def call():
        grads = torch.zeros_like(src)
        dq, dg = _call(gpu, src, q, gain, gout, grads, list(addend) if add else None)
        return grads, dq, dg

    mine, other = _both_policies(call)
    assert mine[0].isnan().any() and mine[0].isfinite().any()
    _agree(mine, other, [ULP] * 3, ["dsources", "dquery", "dgain"])


@pytest.mark.parametrize("D,N", [(520, 1030), (1536, 1026)])
def test_narrow_merge_of_odd_values_as_the_workgroup_kernel(gpu, D, N):
    print(f"narrow merge, odd values D={D} N={N}", flush=True)
    bf = torch.bfloat16
    assert merge_kernel(N, D, bf) == f"attnres_merge_rows_c{(D + 511) // 512}"
    g = torch.Generator(device=gpu).manual_seed(D)
    p, inter, G = (torch.randn((N, D), generator=g, device=gpu).to(bf) for _ in range(3))
    q, lse = (torch.randn(D, generator=g, device=gpu) * 0.1).to(bf), torch.randn(N, generator=g, device=gpu)
    _odd_rows(p)
    inter[25, 0], inter[30, 0], lse[35], lse[40], lse[45] = math.inf, math.nan, math.inf, -math.inf, math.nan
    G[50, 0], G[55, 0] = math.inf, math.nan

    def call():
        leaves = [t.clone().requires_grad_() for t in (p, q, inter, lse)]
        out = ops.merge_call(*leaves, 1e-5)
        return [out.detach(), *torch.autograd.grad(out, leaves, G)]

    mine, other = _both_policies(call)
    assert mine[0].isnan().any() and mine[0].isfinite().any()
    _agree(mine, other, [ULP] * 4 + [1e-4], ["out", "dpartial", "dquery", "dinter", "dlse"])
