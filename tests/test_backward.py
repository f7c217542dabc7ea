"""Backward (sas_bwd_v1): the fp64 autograd oracle pinned by the golden
forward, finite differences and the closed-form sink gradient; the GPU
kernel against the oracle."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from dsv4_amd import cases, paged
from oracle import backward_ref as BR
from oracle import golden_ref as O


def _tiny(dtype=torch.float64, seed=0, scenario=3):
    """2 batches (q_lens 3 and 1, kv_lens 40 and 23), H = 2, D = 576, block
    size 8, window 15, ratio 4, top-k 6: every kind of row in a few keys."""
    g = torch.Generator().manual_seed(seed)
    q_lens, kv_lens, bs, H, D, K, ratio = [3, 1], [40, 23], 8, 2, 576, 6, 4
    T = sum(q_lens)
    ori_bt, ori_nb = paged.random_block_table(kv_lens, bs, g, extra_blocks=2)
    cmp_lens = [k // ratio for k in kv_lens]
    cmp_bt, cmp_nb = paged.random_block_table(cmp_lens, bs, g, extra_blocks=1)
    kw = dict(
        ori_kv=torch.randn(ori_nb, bs, 1, D, generator=g).to(dtype), ori_block_table=ori_bt,
        cu_seqlens_q=torch.tensor([0] + np.cumsum(q_lens).tolist(), dtype=torch.int32),
        seqused_kv=torch.tensor(kv_lens, dtype=torch.int32), sinks=torch.randn(H, generator=g).double(),
        softmax_scale=1 / math.sqrt(D), ori_win_left=15, dv=512)
    if scenario >= 2:
        kw.update(cmp_kv=torch.randn(cmp_nb, bs, 1, D, generator=g).to(dtype), cmp_block_table=cmp_bt,
                  cmp_ratio=ratio)
    if scenario == 3:
        kw["cmp_sparse_indices"] = cases.topk_indices(q_lens, kv_lens, K, ratio, g)
    q = torch.randn(T, H, D, generator=g).to(dtype)
    dout = torch.randn(T, H, 512, generator=g).to(dtype)
    return q, dout, kw


def test_oracle_forward_is_golden():
    q, dout, kw = _tiny()
    r = BR.backward_paged(q, dout, **kw)
    g = dict(kw)
    g.pop("dv")
    out, lse = O.golden_paged(q, dv=512, exact=True, **g)
    torch.testing.assert_close(r["out"], out, atol=1e-10, rtol=1e-10)
    torch.testing.assert_close(r["lse"], lse, atol=1e-10, rtol=1e-10)


def test_oracle_planted_dropped_sink_fails():
    q, dout, kw = _tiny()
    r = BR.backward_paged(q, dout, drop_sink=True, **kw)
    g = dict(kw)
    g.pop("dv")
    out, _ = O.golden_paged(q, dv=512, exact=True, **g)
    assert not torch.allclose(r["out"], out, atol=1e-6, rtol=1e-6)


def test_oracle_sink_gradient_closed_form():
    """d(sink_h) = -sum_t exp(sink_h - lse_th) (dO_th . O_th): the sink's value
    row is zero, so only the softmax normaliser depends on it."""
    q, dout, kw = _tiny()
    r = BR.backward_paged(q, dout, **kw)
    delta = (dout.double() * r["out"]).sum(-1)                       # [T, H]
    ref = -(torch.exp(kw["sinks"].view(1, -1) - r["lse"]) * delta).sum(0)
    torch.testing.assert_close(r["d_sinks"], ref, atol=1e-12, rtol=1e-10)


@pytest.mark.parametrize("scenario", [1, 2, 3])
def test_oracle_given_forward_equals_autograd(scenario):
    """The explicit FlashAttention-2 formulas from the exact forward's out /
    lse give the autograd gradients (dq, touched cache rows, sinks); a
    planted sign error in dS does not."""
    q, dout, kw = _tiny(scenario=scenario, seed=10 + scenario)
    r = BR.backward_paged(q, dout, **kw)
    e = BR.backward_given_forward(q, dout, r["out"], r["lse"], **kw)
    torch.testing.assert_close(e["dq"], r["dq"], atol=1e-10, rtol=1e-9)
    torch.testing.assert_close(e["d_sinks"], r["d_sinks"], atol=1e-10, rtol=1e-9)
    for key in ("d_ori", "d_cmp") if scenario >= 2 else ("d_ori",):
        assert torch.equal(e[key][0], r[key][0])
        torch.testing.assert_close(e[key][1], r[key][1], atol=1e-10, rtol=1e-9)
    bad = BR.backward_given_forward(q, dout, r["out"], r["lse"], plant_sign=True, **kw)
    assert not torch.allclose(bad["dq"], r["dq"], atol=1e-6, rtol=1e-6)


@pytest.mark.parametrize("scenario", [1, 2, 3])
def test_oracle_finite_differences(scenario):
    """Central differences of sum(dO * out) in fp64 match the autograd
    gradients of q, of cache rows (a V channel and a rope channel) and of the
    sinks."""
    q, dout, kw = _tiny(scenario=scenario, seed=scenario)
    r = BR.backward_paged(q, dout, **kw)
    eps = 1e-6

    def loss(qq=q, sinks=kw["sinks"], ori=kw["ori_kv"], cmp_=kw.get("cmp_kv")):
        k2 = dict(kw, sinks=sinks, ori_kv=ori)
        if cmp_ is not None:
            k2["cmp_kv"] = cmp_
        return BR.loss_fp64(qq, dout, **{k: v for k, v in k2.items() if k not in ("sinks", "ori_kv", "cmp_kv")},
                            sinks=k2["sinks"], ori_kv=k2["ori_kv"], cmp_kv=k2.get("cmp_kv"))

    def fd(name, tensor, index):
        hi, lo = tensor.clone(), tensor.clone()
        hi[index] += eps
        lo[index] -= eps
        return (loss(**{name: hi}) - loss(**{name: lo})) / (2 * eps)

    for t, h, c in [(0, 0, 3), (2, 1, 511), (3, 0, 570)]:
        assert abs(fd("qq", q, (t, h, c)) - float(r["dq"][t, h, c])) < 1e-6
    rows, grads = r["d_ori"]
    D = q.shape[-1]
    for i in (0, len(rows) // 2, len(rows) - 1):
        row = int(rows[i])
        for c in (5, 530):
            ix = (row // kw["ori_kv"].shape[1], row % kw["ori_kv"].shape[1], 0, c)
            assert abs(fd("ori", kw["ori_kv"], ix) - float(grads[i, c])) < 1e-6
    if scenario >= 2:
        rows, grads = r["d_cmp"]
        row = int(rows[0])
        ix = (row // kw["cmp_kv"].shape[1], row % kw["cmp_kv"].shape[1], 0, 100)
        assert abs(fd("cmp_", kw["cmp_kv"], ix) - float(grads[0, 100])) < 1e-6
    for h in range(2):
        assert abs(fd("sinks", kw["sinks"], (h,)) - float(r["d_sinks"][h])) < 1e-6


# ---------------------------------------------------------------------------
# GPU: the kernel against the oracle
# ---------------------------------------------------------------------------

def _gpu_case(name):
    from tests.test_gpu_parity import _small
    if name == "C1":
        return cases.make_inputs(cases.CONFIGS["C1"], device="cpu")
    spec = {
        "scfa_prefill": dict(B=2, H=32, q_lens=[40, 3], kv_lens=[300, 90], K=64, bs=16),
        "swa": dict(B=3, H=16, q_lens=[1, 5, 2], kv_lens=[50, 700, 128], K=0, scenario=1),
        "cfa": dict(B=2, H=16, q_lens=[2, 1], kv_lens=[500, 333], K=0, scenario=2, ratio=8),
        "fp16_d512": dict(B=2, H=16, q_lens=[1, 2], kv_lens=[900, 400], K=64, D=512, dtype=torch.float16),
        "decode_h64": dict(B=8, H=64, q_lens=[1] * 8, kv_lens=[4000, 900, 129, 2500, 60, 3000, 1000, 2048], K=128),
        # kv shorter than the query: early tokens attend to no row (sink only)
        "short_kv": dict(B=4, H=32, q_lens=[1, 3, 2, 5], kv_lens=[1, 3, 60, 3], K=32),
        # 128 + 2048 dense compressed slots per token: beyond one workgroup's
        # 1280-slot range, so the planner splits the key range
        "cfa_2176_slots": dict(B=2, H=16, q_lens=[2, 1], kv_lens=[8192, 6000], K=0, scenario=2, ratio=4),
        # the same beyond-1280-slot split through the 64-head kernel
        # (sas_bwd64_kernel: H a multiple of 64), with 64 and 128 heads
        "cfa_2176_slots_h64": dict(B=2, H=64, q_lens=[2, 1], kv_lens=[8192, 6000], K=0, scenario=2, ratio=4),
        "cfa_2176_slots_h128": dict(B=2, H=128, q_lens=[1, 2], kv_lens=[7000, 8192], K=0, scenario=2, ratio=4),
    }[name]
    return _small(**spec)


def _rel_err(got, ref):
    ref = ref.double()
    return float((got.double() - ref).abs().max() / max(float(ref.abs().max()), 1e-30))


GRAD_TOL = 2e-2


def _check_elem(got, ref, what, tol=GRAD_TOL):
    """Element-wise: |got - ref| <= tol |ref| + tol max|ref over the element's
    row| (the last dimension: a (token, head)'s dq channels, a cache row's
    gradient channels, the H sink gradients), so a wrong small row fails even
    when the largest gradients are right. Returns the worst err / bound."""
    got, ref = got.double().reshape(-1, got.shape[-1]), ref.double().reshape(-1, ref.shape[-1])
    if ref.numel() == 0:
        return 0.0
    rowmax = ref.abs().amax(dim=1, keepdim=True)
    bound = tol * ref.abs() + tol * rowmax
    err = (got - ref).abs()
    ratio = err / bound.clamp_min(1e-300)
    bad = err > bound
    worst = float(ratio.max())
    assert bool(torch.isfinite(got).all()), f"{what}: {int((~torch.isfinite(got)).sum())} non-finite elements"
    assert not bool(bad.any()), (f"{what}: {int(bad.sum())} of {err.numel()} elements beyond "
                                 f"{tol}|ref| + {tol} rowmax|ref| (worst err/bound {worst:.3g})")
    return worst


def _check_against_oracle(name, inp, dq, d_ori, d_cmp, d_sinks, r):
    """dq, the touched cache rows (untouched rows exactly zero) and d_sinks
    element-wise against the fp64 oracle result ``r``."""
    c = inp.cfg
    D = inp.q.shape[-1]
    worst = {"dq": _check_elem(dq.cpu(), r["dq"], f"{name} dq")}
    rows, grads = r["d_ori"]
    flat = d_ori.cpu().reshape(-1, D)
    worst["d_ori"] = _check_elem(flat[rows], grads, f"{name} d_ori")
    untouched = torch.ones(flat.shape[0], dtype=torch.bool)
    untouched[rows] = False
    if untouched.any():
        assert float(flat[untouched].abs().max()) == 0.0, f"{name}: untouched ori rows changed"
    if c.scenario >= 2:
        rows, grads = r["d_cmp"]
        cflat = d_cmp.cpu().reshape(-1, D)
        if rows.numel():
            worst["d_cmp"] = _check_elem(cflat[rows], grads, f"{name} d_cmp")
        untouched = torch.ones(cflat.shape[0], dtype=torch.bool)
        untouched[rows] = False
        if untouched.any():
            assert float(cflat[untouched].abs().max()) == 0.0, f"{name}: untouched cmp rows changed"
    worst["d_sinks"] = _check_elem(d_sinks.cpu().reshape(1, -1), r["d_sinks"].reshape(1, -1), f"{name} d_sinks")
    print(f"[bwd] {name}: worst err / bound = {worst}", flush=True)


def _oracle_bwd(inp, dout, out, lse, tokens=None):
    """The fp64 backward from the GPU forward's own out / lse (the inputs
    sas_bwd_v1 takes; the formulas are pinned to autograd above): the GPU
    result may then differ only by its bf16 operand roundings and fp32
    accumulation, element by element."""
    c = inp.cfg
    return BR.backward_given_forward(
        inp.q, dout, out, lse, ori_kv=inp.ori_kv, ori_block_table=inp.ori_bt, cu_seqlens_q=inp.cu_seqlens_q,
        seqused_kv=inp.seqused_kv, sinks=inp.sinks, softmax_scale=c.scale,
        cmp_kv=inp.cmp_kv if c.scenario >= 2 else None, cmp_block_table=inp.cmp_bt if c.scenario >= 2 else None,
        cmp_sparse_indices=inp.cmp_idx if c.scenario == 3 else None, cmp_ratio=c.cmp_ratio,
        ori_win_left=c.win_left, tokens=tokens)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["C1", "scfa_prefill", "swa", "cfa", "fp16_d512", "decode_h64", "short_kv",
                                  "cfa_2176_slots", "cfa_2176_slots_h64", "cfa_2176_slots_h128"])
def test_gpu_backward_matches_oracle(name):
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    inp = _gpu_case(name)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(5)
    dout = torch.randn(out.shape, generator=g).to(inp.q.dtype)
    dq, d_ori, d_cmp, d_sinks = sparse_attn_sharedkv_backward(dout.cuda(), d.q, out, lse, **kw)
    torch.cuda.synchronize()
    # tolerance: bf16 / fp16 rounding of the forward output (used in Delta),
    # of the MFMA operands dS / P and of dq; fp32 accumulation elsewhere
    _check_against_oracle(name, inp, dq, d_ori, d_cmp, d_sinks, _oracle_bwd(inp, dout, out, lse))


@pytest.mark.gpu
@pytest.mark.parametrize("i", range(24))
def test_gpu_backward_random_configurations(i):
    """Seeded random configurations (scenario, H, D, dtype, window, block
    size, ratio, top-k, decode or short prefill batches), every gradient
    element against the oracle from the GPU forward's own out / lse."""
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    from tests.test_gpu_parity import _fuzz_case, _small
    kw, _ = _fuzz_case(500 + i)
    kw["fp8"] = False   # the backward takes caches in the query dtype
    print(f"[bwd fuzz {i}] {kw}", flush=True)
    inp = _small(**kw)
    d = inp.to("cuda")
    akw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **akw)
    g = torch.Generator().manual_seed(7 + i)
    dout = torch.randn(out.shape, generator=g).to(inp.q.dtype)
    dq, d_ori, d_cmp, d_sinks = sparse_attn_sharedkv_backward(dout.cuda(), d.q, out, lse, **akw)
    torch.cuda.synchronize()
    _check_against_oracle(f"bwd fuzz {i}", inp, dq, d_ori, d_cmp, d_sinks, _oracle_bwd(inp, dout, out, lse))


@pytest.mark.gpu
def test_gpu_backward_c2_decode_full():
    """The C2 workload the bench times (32 tokens, H = 64, top-k 512 +
    window 128 over 8K-32K contexts), every gradient against the oracle."""
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    inp = cases.make_inputs(cases.CONFIGS["C2"], device="cpu")
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(21)
    dout = torch.randn(out.shape, generator=g).to(inp.q.dtype)
    dq, d_ori, d_cmp, d_sinks = sparse_attn_sharedkv_backward(dout.cuda(), d.q, out, lse, **kw)
    torch.cuda.synchronize()
    _check_against_oracle("C2", inp, dq, d_ori, d_cmp, d_sinks, _oracle_bwd(inp, dout, out, lse))


@pytest.mark.gpu
def test_gpu_backward_c3_prefill_sampled():
    """The C3 4096-token prefill the bench times, with dout nonzero on 48
    sampled tokens only (first, last, window and block edges, random): the
    other tokens then contribute nothing to any gradient, so the oracle on
    the sampled tokens gives the exact expected dq, cache and sink
    gradients of the whole launch."""
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    inp = cases.make_inputs(cases.CONFIGS["C3"], device="cpu")
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(22)
    toks = sorted(set([0, 1, 127, 128, 129, 511, 512, 2047, 4094, 4095] +
                      torch.randint(0, 4096, (38,), generator=g).tolist()))
    dout = torch.zeros(out.shape, dtype=inp.q.dtype)
    dout[toks] = torch.randn((len(toks),) + tuple(out.shape[1:]), generator=g).to(inp.q.dtype)
    dq, d_ori, d_cmp, d_sinks = sparse_attn_sharedkv_backward(dout.cuda(), d.q, out, lse, **kw)
    torch.cuda.synchronize()
    r = _oracle_bwd(inp, dout, out, lse, tokens=toks)
    _check_against_oracle("C3 sampled", inp, dq, d_ori, d_cmp, d_sinks, r)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["prefill_2b", "prefill_bs16_h16", "swa", "short_kv", "decode_h64", "cfa",
                                  "fp16_d512", "prefill_wide_window", "prefill_swa_bs16"])
def test_gpu_backward_window_pass_both_ways(name):
    """Rows' gradients summed per (token, row) and key-major (forced both ways,
    whatever the library would choose: all rows by the prefill path where H is
    a multiple of 32, the window rows by the window pass elsewhere): each
    element-wise against the fp64 oracle, on prefills (several batches, pages
    of 16, a window wider than the 64-position tile) and on decode and
    short-KV batches (tokens with empty windows, rows past act_kv)."""
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    from tests.test_gpu_parity import _small
    extra = {
        "prefill_2b": dict(B=2, H=64, q_lens=[300, 170], kv_lens=[300, 420], K=64, bs=64),
        "prefill_bs16_h16": dict(B=3, H=16, q_lens=[90, 17, 64], kv_lens=[90, 200, 64], K=32, bs=16),
        "prefill_wide_window": dict(B=1, H=32, q_lens=[400], kv_lens=[400], K=48, win=300),
        "prefill_swa_bs16": dict(B=2, H=16, q_lens=[200, 70], kv_lens=[260, 70], K=0, scenario=1, bs=16),
    }
    inp = _small(**extra[name]) if name in extra else _gpu_case(name)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(31)
    dout = torch.randn(out.shape, generator=g).to(inp.q.dtype)
    r = _oracle_bwd(inp, dout, out, lse)
    for wp in (False, True):
        dq, d_ori, d_cmp, d_sinks = sparse_attn_sharedkv_backward(dout.cuda(), d.q, out, lse, window_pass=wp, **kw)
        torch.cuda.synchronize()
        _check_against_oracle(f"{name} window_pass={wp}", inp, dq, d_ori, d_cmp, d_sinks, r)


@pytest.mark.gpu
def test_gpu_backward_window_pass_bsnd():
    """The key-major passes with BSND queries (per-batch lengths, padded rows:
    the kernels read act_q instead of a prefix difference) give the TND
    per-token result up to summation order."""
    from tests.test_gpu_parity import _small
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    q_lens = [70, 30]
    inp = _small(B=2, H=64, q_lens=q_lens, kv_lens=[90, 30], K=16)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(33)
    dout = torch.randn(out.shape, generator=g).to(out.dtype).cuda()
    ref = sparse_attn_sharedkv_backward(dout, d.q, out, lse, window_pass=False, **kw)
    S = max(q_lens)
    q_b = torch.zeros(2, S, 64, 576, dtype=torch.bfloat16, device="cuda")
    idx_b = torch.full((2, S, 1, 16), -1, dtype=torch.int32, device="cuda")
    o_b = torch.zeros(2, S, 64, 512, dtype=torch.bfloat16, device="cuda")
    l_b = torch.zeros(2, S, 64, dtype=torch.float32, device="cuda")
    do_b = torch.zeros(2, S, 64, 512, dtype=torch.bfloat16, device="cuda")
    t_ = 0
    for b, n in enumerate(q_lens):
        q_b[b, :n], idx_b[b, :n], o_b[b, :n], l_b[b, :n], do_b[b, :n] = (
            d.q[t_:t_ + n], d.cmp_idx[t_:t_ + n], out[t_:t_ + n], lse[t_:t_ + n], dout[t_:t_ + n])
        t_ += n
    kwb = dict(kw, layout_q="BSND", cmp_sparse_indices=idx_b)
    dq_b, d_ori, d_cmp, d_snk = sparse_attn_sharedkv_backward(do_b, q_b, o_b, l_b, window_pass=True, **kwb)
    torch.cuda.synchronize()
    assert _rel_err(dq_b[0, :70].float().cpu(), ref[0][:70].float().cpu()) < 1e-2
    assert _rel_err(dq_b[1, :30].float().cpu(), ref[0][70:].float().cpu()) < 1e-2
    assert torch.count_nonzero(dq_b[1, 30:].cpu().float()) == 0
    assert _rel_err(d_ori.cpu(), ref[1].cpu()) < 1e-4 and _rel_err(d_cmp.cpu(), ref[2].cpu()) < 1e-4
    assert _rel_err(d_snk.cpu(), ref[3].cpu()) < 1e-4


@pytest.mark.gpu
def test_gpu_backward_captured_in_a_graph():
    """The prepared backward of a prefill captured in a HIP graph: with its fp32
    dq it gives way to per-token adds under capture (the default) or, when
    asked for, sums every row's gradient key-major on the captured stream.
    Every replay (with eager work between them) equals the eager run of the
    same mode up to fp32 summation order; the two modes differ from each
    other only by where the keys' products are rounded."""
    from dsv4_amd.api import prepare_sparse_attn_sharedkv_backward, sparse_attn_sharedkv
    from tests.test_gpu_parity import _small
    inp = _small(B=2, H=64, q_lens=[300, 170], kv_lens=[300, 420], K=64)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
        g = torch.Generator().manual_seed(35)
        dout = torch.randn(out.shape, generator=g).to(out.dtype).cuda()
        refs = {}
        for wp in (False, True):
            eager = prepare_sparse_attn_sharedkv_backward(dout, d.q, out, lse, window_pass=wp, **kw)
            eager.launch(side)
            torch.cuda.synchronize()
            refs[wp] = [t.clone() for t in (eager.dq, eager.d_ori_kv, eager.d_cmp_kv, eager.d_sinks)]
        for a, b in zip(refs[False], refs[True]):
            assert _rel_err(a.cpu(), b.cpu()) < 1e-4
        for wp, mode in ((None, False), (True, True)):
            pb = prepare_sparse_attn_sharedkv_backward(dout, d.q, out, lse, window_pass=wp, **kw)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                pb.zero_grads()
                pb.launch(side)
            grads = (pb.dq, pb.d_ori_kv, pb.d_cmp_kv, pb.d_sinks)
            for i in range(3):
                for t in grads:
                    t.fill_(float(i + 7))             # eager work between replays
                graph.replay()
                torch.cuda.synchronize()
                for name, got, want in zip(("dq", "d_ori", "d_cmp", "d_sinks"), grads, refs[mode]):
                    assert _rel_err(got.cpu(), want.cpu()) < 1e-5, f"window_pass={wp} replay {i} {name}"
            del graph, pb


@pytest.mark.gpu
def test_gpu_backward_split_count_invariance():
    """The key range split over 1, 3 or 7 workgroups per (token, head group)
    (dq then accumulated atomically) gives the same gradients up to fp32
    summation order."""
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    inp = _gpu_case("decode_h64")
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(6)
    dout = torch.randn(out.shape, generator=g).to(inp.q.dtype).cuda()
    res = [sparse_attn_sharedkv_backward(dout, d.q, out, lse, num_splits=ns, **kw) for ns in (1, 3, 7)]
    torch.cuda.synchronize()
    for other in res[1:]:
        for a_, b_ in zip(res[0], other):
            if a_ is not None:
                assert _rel_err(b_.float().cpu(), a_.float().cpu()) < 1e-2 if a_.dtype != torch.float32 \
                    else _rel_err(b_.cpu(), a_.cpu()) < 1e-5


@pytest.mark.gpu
def test_gpu_autograd_binding():
    """loss.backward() through sparse_attn_sharedkv_autograd gives the
    gradients of sparse_attn_sharedkv_backward."""
    from dsv4_amd.api import sparse_attn_sharedkv_autograd, sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    inp = _gpu_case("scfa_prefill")
    d = inp.to("cuda")
    kw = d.api_kwargs()
    q = d.q.clone().requires_grad_(True)
    ori = d.ori_kv.clone().requires_grad_(True)
    cmp_ = d.cmp_kv.clone().requires_grad_(True)
    snk = d.sinks.clone().requires_grad_(True)
    rest = {k: v for k, v in kw.items() if k not in ("ori_kv", "cmp_kv", "sinks")}
    out = sparse_attn_sharedkv_autograd(q, ori_kv=ori, cmp_kv=cmp_, sinks=snk, **rest)
    g = torch.Generator().manual_seed(8)
    dout = torch.randn(out.shape, generator=g).to(out.dtype).cuda()
    (out.float() * dout.float()).sum().backward()
    o2, lse2 = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    ref = sparse_attn_sharedkv_backward(dout, d.q, o2, lse2, **kw)
    torch.cuda.synchronize()
    assert torch.equal(out.detach().cpu(), o2.cpu())
    assert _rel_err(q.grad.float().cpu(), ref[0].float().cpu()) < 1e-2
    assert _rel_err(ori.grad.float().cpu(), ref[1].cpu()) < 1e-2
    assert _rel_err(cmp_.grad.float().cpu(), ref[2].cpu()) < 1e-2
    assert _rel_err(snk.grad.cpu(), ref[3].cpu()) < 1e-4


@pytest.mark.gpu
def test_gpu_backward_bsnd_padding_matches_tnd():
    """BSND q [B, S, N, D] with per-batch lengths: the valid rows' dq and the
    cache / sink gradients equal the TND backward of the same tokens up to
    summation order (the two layouts get different KV split counts, so bf16
    dq may differ by a rounding step), and the padded rows' dq is zero."""
    from tests.test_gpu_parity import _small
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    inp = _small(B=2, H=64, q_lens=[3, 1], kv_lens=[800, 400], K=64)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(9)
    dout = torch.randn(out.shape, generator=g).to(out.dtype).cuda()
    ref = sparse_attn_sharedkv_backward(dout, d.q, out, lse, **kw)
    slot = [(0, 0), (0, 1), (0, 2), (1, 0)]                       # (b, s) of the 4 packed tokens
    q_b = torch.zeros(2, 3, 64, 576, dtype=torch.bfloat16, device="cuda")
    idx_b = torch.full((2, 3, 1, 64), -1, dtype=torch.int32, device="cuda")
    o_b = torch.zeros(2, 3, 64, 512, dtype=torch.bfloat16, device="cuda")
    l_b = torch.zeros(2, 3, 64, dtype=torch.float32, device="cuda")
    do_b = torch.zeros(2, 3, 64, 512, dtype=torch.bfloat16, device="cuda")
    for t_, (b, s_) in enumerate(slot):
        q_b[b, s_], idx_b[b, s_], o_b[b, s_], l_b[b, s_], do_b[b, s_] = (
            d.q[t_], d.cmp_idx[t_], out[t_], lse[t_], dout[t_])
    kwb = dict(kw, layout_q="BSND", cmp_sparse_indices=idx_b)
    dq_b, d_ori, d_cmp, d_snk = sparse_attn_sharedkv_backward(do_b, q_b, o_b, l_b, **kwb)
    torch.cuda.synchronize()
    assert dq_b.shape == q_b.shape
    for t_, (b, s_) in enumerate(slot):
        assert _rel_err(dq_b[b, s_].float().cpu(), ref[0][t_].float().cpu()) < 1e-2
    assert torch.count_nonzero(dq_b[1, 1:].cpu().float()) == 0
    assert _rel_err(d_ori.cpu(), ref[1].cpu()) < 1e-4 and _rel_err(d_cmp.cpu(), ref[2].cpu()) < 1e-4
    assert _rel_err(d_snk.cpu(), ref[3].cpu()) < 1e-4


@pytest.mark.gpu
def test_gpu_backward_h48_d512_matches_oracle():
    """H = 48 (three 16-head workgroups per token) at D = 512."""
    from tests.test_gpu_parity import _small
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    inp = _small(B=2, H=48, q_lens=[3, 1], kv_lens=[2000, 700], K=100, D=512)
    c = inp.cfg
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(10)
    dout = torch.randn(out.shape, generator=g).to(out.dtype)
    dq, d_ori, d_cmp, d_snk = sparse_attn_sharedkv_backward(dout.cuda(), d.q, out, lse, **kw)
    torch.cuda.synchronize()
    _check_against_oracle("h48_d512", inp, dq, d_ori, d_cmp, d_snk, _oracle_bwd(inp, dout, out, lse))


@pytest.mark.gpu
@pytest.mark.parametrize("name,spec", [
    # tokens on both sides of the density rule (a few K rows): dense ones by the
    # key-major pass, the others by per-token adds; 64- and 32-head groups
    ("both_h64", dict(B=1, H=64, q_lens=[400], kv_lens=[400], K=8)),
    ("both_h32", dict(B=2, H=32, q_lens=[270, 90], kv_lens=[330, 500], K=8, D=512, bs=16)),
    ("per_token_only", dict(B=1, H=64, q_lens=[100], kv_lens=[900], K=8, dtype=torch.float16)),
    # a row listed twice counts twice
    ("listed_twice", dict(B=1, H=64, q_lens=[200], kv_lens=[400], K=16,
                          idx_fn=lambda i: torch.cat([i[..., :1], i[..., :-1]], -1))),
    # more key slots than one resolution pass holds, and lists past 2048 entries
    ("dense_passes", dict(B=1, H=64, q_lens=[70], kv_lens=[5200], K=0, scenario=2)),
    ("long_lists", dict(B=1, H=128, q_lens=[66], kv_lens=[8600], K=2100, D=512, win=1)),
    # segment and tile edges, windows off the tile grid; 96-token segments
    ("long_segments", dict(B=2, H=128, q_lens=[1100, 97], kv_lens=[1100, 500], K=24, win=90, D=512, dtype=torch.float16)),
    ("edges", dict(B=4, H=32, q_lens=[63, 64, 65, 129], kv_lens=[63, 191, 65, 400], K=40, win=66, bs=16)),
])
def test_gpu_backward_prefill_path(name, spec):
    """The prefill path's branches (dq in the query dtype from the call, fp32
    from the prepared one), every gradient element against the oracle."""
    from dsv4_amd.api import (prepare_sparse_attn_sharedkv_backward, sparse_attn_sharedkv,
                              sparse_attn_sharedkv_backward)
    from tests.test_gpu_parity import _small
    inp = _small(**spec)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(41)
    dout = torch.randn(out.shape, generator=g).to(inp.q.dtype)
    r = _oracle_bwd(inp, dout, out, lse)
    got = sparse_attn_sharedkv_backward(dout.cuda(), d.q, out, lse, **kw)
    pb = prepare_sparse_attn_sharedkv_backward(dout.cuda(), d.q, out, lse, **kw)
    assert pb.dq.dtype == torch.float32
    pb.launch()
    torch.cuda.synchronize()
    _check_against_oracle(name, inp, *got, r)
    _check_against_oracle(f"{name} prepared", inp, *pb.result(), r)
    assert torch.equal(pb.dq.to(got[0].dtype).cpu(), got[0].cpu())


@pytest.mark.gpu
@pytest.mark.parametrize("H,D,bs", [(64, 576, 64), (32, 512, 16)])
def test_gpu_backward_table_narrower_than_the_sequences(H, D, bs):
    """A compressed block table that ends before the causal thresholds: the
    entries past it are not attended, and every token's gradients are still
    written (a few times K rows lie between the table's end and the largest
    threshold, on both sides of the density rule)."""
    from dataclasses import replace
    from dsv4_amd.api import (prepare_sparse_attn_sharedkv_backward, sparse_attn_sharedkv,
                              sparse_attn_sharedkv_backward)
    from tests.test_gpu_parity import _small
    K, cap = 32, 64
    inp = _small(B=2, H=H, q_lens=[80, 70], kv_lens=[4000, 330], K=K, D=D, bs=bs)
    g = torch.Generator().manual_seed(43)
    idx = torch.full_like(inp.cmp_idx, -1)
    inside = torch.full_like(inp.cmp_idx, -1)
    for t in range(idx.shape[0]):
        thr = (4000 - 80 + t + 1) // 4 if t < 80 else (330 - 70 + t - 80 + 1) // 4
        n = min(K // 2, thr)
        head = torch.randperm(min(cap, thr), generator=g)[:n].to(torch.int32)
        inside[t, 0, :n] = head
        idx[t, 0, :n] = head
        if thr > cap:
            idx[t, 0, n:] = cap + torch.randperm(thr - cap, generator=g)[:K - n].to(torch.int32) \
                if thr - cap >= K - n else -1
    inp = replace(inp, cmp_idx=idx, cmp_bt=inp.cmp_bt[:, :cap // bs].contiguous())
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    dout = torch.randn(out.shape, generator=g).to(inp.q.dtype)
    r = _oracle_bwd(replace(inp, cmp_idx=inside), dout, out, lse)
    dout = dout.cuda()
    # fill the blocks that the call's own tensors are likely to get (one of
    # them may be left unwritten)
    torch.full(d.q.shape, float("nan"), dtype=d.q.dtype, device="cuda")
    torch.full(lse.shape, float("nan"), device="cuda")
    got = sparse_attn_sharedkv_backward(dout, d.q, out, lse, **kw)
    pb = prepare_sparse_attn_sharedkv_backward(dout, d.q, out, lse, **kw)
    pb.launch()
    torch.cuda.synchronize()
    assert all(torch.isfinite(x).all() for x in (*got, *pb.result()))
    _check_against_oracle(f"narrow table H{H}", inp, *got, r)
    _check_against_oracle(f"narrow table H{H} prepared", inp, *pb.result(), r)


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["q_nan", "q_inf_rope", "dout_inf", "dout_nan"])
@pytest.mark.parametrize("spec", [
    dict(H=64, q_lens=[200], kv_lens=[400], K=24),
    dict(H=32, q_lens=[130], kv_lens=[700], K=8, bs=16, dtype=torch.float16),
    dict(H=32, q_lens=[150], kv_lens=[300], K=0, scenario=2, win=40),
], ids=["topk", "both_passes", "dense"])
def test_gpu_backward_non_finite_token_stays_in_its_rows(spec, what):
    """A token with a NaN or Inf in one head's q or dout makes the gradients of
    the rows it attends non-finite, and no others: they, every other token's
    dq and every other head's sink gradient are those of the call without it."""
    from dsv4_amd.api import sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    from tests.test_gpu_parity import _small
    inp = _small(B=1, **spec)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    g = torch.Generator().manual_seed(47)
    D, T, H = inp.q.shape[-1], inp.q.shape[0], spec["H"]
    dout = torch.randn((T, H, 512), generator=g).to(inp.q.dtype).cuda()
    t, h = 77, 5
    clean_out, clean_lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    q, bad_dout = d.q.clone(), dout.clone()
    if what == "q_nan":
        q[t, h, 100] = float("nan")
    elif what == "q_inf_rope":
        q[t, h, D - 3] = float("inf")
    else:
        bad_dout[t, h, 300] = float("inf" if what == "dout_inf" else "nan")
    out, lse = sparse_attn_sharedkv(q, return_softmax_lse=True, **kw)
    got = sparse_attn_sharedkv_backward(bad_dout, q, out, lse, **kw)
    # the call without the token's contributions
    dout[t] = 0
    ref = sparse_attn_sharedkv_backward(dout, d.q, clean_out, clean_lse, **kw)
    torch.cuda.synchronize()
    others = [i for i in range(T) if i != t]
    assert torch.equal(got[0][others], ref[0][others])
    heads = [i for i in range(H) if i != h]
    sg = spec["kv_lens"][0] - T + t
    win = spec.get("win", 127)

    def rows(table, positions, bs):
        return torch.tensor([int(table[0, p // bs]) * bs + p % bs for p in positions])

    sets = [(got[1], ref[1], rows(inp.ori_bt, range(max(0, sg - win), sg + 1), inp.ori_kv.shape[1]))]
    if got[2] is not None:
        thr = (sg + 1) // 4
        pos = [int(x) for x in inp.cmp_idx[t, 0] if 0 <= int(x) < thr] if spec["K"] else range(thr)
        sets.append((got[2], ref[2], rows(inp.cmp_bt, pos, inp.cmp_kv.shape[1])))
    for name, (a, b, hit) in zip(("ori", "cmp"), sets):
        a, b = a.cpu().reshape(-1, D), b.cpu().reshape(-1, D)
        assert not torch.isfinite(a[hit]).all(dim=1).any(), f"{name}: an attended row stayed finite"
        free = torch.ones(a.shape[0], dtype=torch.bool)
        free[hit] = False
        assert torch.isfinite(a[free]).all(), f"{name}: {int((~torch.isfinite(a[free])).any(1).sum())} other rows hit"
        # fp32 sums over the tokens in another order
        assert float((a[free] - b[free]).abs().max()) <= 1e-5 * float(b[free].abs().max()), name
    snk = got[3][heads]
    assert torch.isfinite(snk).all()


@pytest.mark.gpu
def test_gpu_backward_output_gradient_at_any_alignment():
    """An output gradient that starts 8 bytes off a 16-byte boundary: the
    gradients of the aligned one, by the kernels that load it through
    registers."""
    from dsv4_amd import _lib
    from dsv4_amd.api import prepare_sparse_attn_sharedkv_backward, sparse_attn_sharedkv, sparse_attn_sharedkv_backward
    from tests.test_gpu_parity import _small
    inp = _small(B=1, H=64, q_lens=[130], kv_lens=[300], K=24)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(53)
    dout = torch.randn(out.shape, generator=g).to(out.dtype)
    buf = torch.zeros(dout.numel() + 4, dtype=dout.dtype, device="cuda")
    off = buf[4:].view(dout.shape)
    off.copy_(dout)
    assert off.data_ptr() % 16 == 8 and off.is_contiguous()
    r = _oracle_bwd(inp, dout, out, lse)
    pb = prepare_sparse_attn_sharedkv_backward(off, d.q, out, lse, **kw)
    assert not pb.args.fwd.flags & _lib.SAS_BWD_WORKSPACE
    got = sparse_attn_sharedkv_backward(off, d.q, out, lse, **kw)
    torch.cuda.synchronize()
    _check_against_oracle("dout off alignment", inp, *got, r)


# ---------------------------------------------------------------------------
# callers without a workspace: per-token kernels, the window pass beside them
# ---------------------------------------------------------------------------

def _without_workspace(pb):
    """A prepared backward as a C caller that gives no workspace calls it."""
    from dsv4_amd import _lib
    a = pb.args.fwd
    a.flags &= ~_lib.SAS_BWD_WORKSPACE
    a.workspace, a.workspace_bytes = None, 0
    return pb


@pytest.mark.gpu
@pytest.mark.parametrize("name,spec", [
    # the 64-head and the 32-head per-token kernel, prefills (the window pass
    # beside them on the library's side stream) and decode-like calls
    ("h64", dict(B=2, H=64, q_lens=[300, 170], kv_lens=[300, 420], K=64)),
    ("h128_d512_fp16", dict(B=1, H=128, q_lens=[140], kv_lens=[500], K=48, D=512, dtype=torch.float16)),
    ("h32_bs16", dict(B=3, H=32, q_lens=[90, 17, 130], kv_lens=[90, 200, 130], K=32, bs=16)),
    ("h32_wide_window", dict(B=1, H=32, q_lens=[200], kv_lens=[400], K=48, win=300)),
    ("h64_swa", dict(B=2, H=64, q_lens=[200, 70], kv_lens=[260, 70], K=0, scenario=1)),
    ("h64_cfa", dict(B=2, H=64, q_lens=[128, 40], kv_lens=[500, 40], K=0, scenario=2, ratio=8)),
    ("h64_short_kv", dict(B=2, H=64, q_lens=[150, 90], kv_lens=[40, 3], K=8)),
    ("h64_decode", dict(B=3, H=64, q_lens=[1, 2, 1], kv_lens=[700, 90, 300], K=64)),
])
def test_gpu_backward_without_workspace(name, spec):
    """Without a workspace: the library's choice, per-token adds for every row,
    and the window pass, each element-wise against the fp64 oracle."""
    from dsv4_amd.api import prepare_sparse_attn_sharedkv_backward, sparse_attn_sharedkv
    from tests.test_gpu_parity import _small
    inp = _small(**spec)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(59)
    dout = torch.randn(out.shape, generator=g).to(inp.q.dtype)
    r = _oracle_bwd(inp, dout, out, lse)
    dout = dout.cuda()
    for wp in (None, False, True):
        pb = _without_workspace(prepare_sparse_attn_sharedkv_backward(dout, d.q, out, lse, window_pass=wp, **kw))
        pb.launch()
        torch.cuda.synchronize()
        _check_against_oracle(f"{name} no workspace window_pass={wp}", inp, *pb.result(), r)


@pytest.mark.gpu
@pytest.mark.parametrize("H", [32, 64])
def test_gpu_backward_without_workspace_captured(H):
    """The same under capture: per-token adds (the default), or the window pass
    after the per-token kernel on the captured stream, on every replay."""
    from dsv4_amd.api import prepare_sparse_attn_sharedkv_backward, sparse_attn_sharedkv
    from tests.test_gpu_parity import _small
    inp = _small(B=2, H=H, q_lens=[200, 70], kv_lens=[200, 320], K=32)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
        g = torch.Generator().manual_seed(61)
        dout = torch.randn(out.shape, generator=g).to(inp.q.dtype)
        r = _oracle_bwd(inp, dout, out, lse)
        dout = dout.cuda()
        for wp in (None, True):
            pb = _without_workspace(prepare_sparse_attn_sharedkv_backward(dout, d.q, out, lse, window_pass=wp, **kw))
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                pb.zero_grads()
                pb.launch(side)
            for i in range(3):
                for t in (pb.dq, pb.d_ori_kv, pb.d_cmp_kv, pb.d_sinks):
                    t.fill_(float(i + 7))             # eager work between replays
                graph.replay()
                torch.cuda.synchronize()
                _check_against_oracle(f"captured H{H} window_pass={wp} replay {i}", inp, *pb.result(), r)
            del graph, pb


@pytest.mark.gpu
def test_gpu_backward_without_workspace_bsnd():
    """The window pass beside the per-token kernels with BSND queries (padded
    rows, lengths read from act_q): the TND gradients up to summation order."""
    from tests.test_gpu_parity import _small
    from dsv4_amd.api import prepare_sparse_attn_sharedkv_backward, sparse_attn_sharedkv
    q_lens, S = [130, 40], 130
    inp = _small(B=2, H=64, q_lens=q_lens, kv_lens=[200, 40], K=16)
    d = inp.to("cuda")
    kw = d.api_kwargs()
    out, lse = sparse_attn_sharedkv(d.q, return_softmax_lse=True, **kw)
    g = torch.Generator().manual_seed(67)
    dout = torch.randn(out.shape, generator=g).to(out.dtype).cuda()

    def padded(t, fill=0):
        p = torch.full((2, S) + tuple(t.shape[1:]), fill, dtype=t.dtype, device="cuda")
        p[0], p[1, :40] = t[:130], t[130:]
        return p

    kwb = dict(kw, layout_q="BSND", cmp_sparse_indices=padded(d.cmp_idx, -1))
    ref = prepare_sparse_attn_sharedkv_backward(dout, d.q, out, lse, window_pass=False, **kw)
    pb = _without_workspace(prepare_sparse_attn_sharedkv_backward(padded(dout), padded(d.q), padded(out), padded(lse), **kwb))
    ref.launch()
    pb.launch()
    torch.cuda.synchronize()
    (dq, *rows), (dq_ref, *rows_ref) = pb.result(), ref.result()
    assert _rel_err(dq[0].float().cpu(), dq_ref[:130].float().cpu()) < 1e-2
    assert _rel_err(dq[1, :40].float().cpu(), dq_ref[130:].float().cpu()) < 1e-2
    assert torch.count_nonzero(dq[1, 40:].cpu().float()) == 0
    for a, b in zip(rows, rows_ref):
        assert _rel_err(a.cpu(), b.cpu()) < 1e-4
