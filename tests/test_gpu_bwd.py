"""GPU parity of the backward pass (cfg 5 path) against autograd through the CPU oracle.

Tolerance (north star): gradients within max-abs <= 2e-2 and mean-abs <= 2e-3 of the fp32 oracle's
autograd, for inputs and upstream gradients of unit scale. Routing is not differentiated (as in the
reference), so the GPU and oracle runs must route identically — checked first where it matters."""
import pytest
import torch

from oracle import hsa as O
from worldattention_amd import hsa as W
from worldattention_amd import workloads
from worldattention_amd.hsa import attention as WA

pytestmark = pytest.mark.gpu
DEV = "cuda"


def assert_close(got, want, max_abs=2e-2, mean_abs=2e-3, what=""):
    assert got is not None and want is not None, f"{what}: missing (gpu {got is None}, oracle {want is None})"
    got, want = got.detach().float().cpu(), want.detach().float().cpu()
    assert torch.isfinite(got).all(), f"{what}: non-finite"
    diff = (got - want).abs()
    assert diff.max().item() <= max_abs, f"{what}: max-abs {diff.max().item():.3e} (ref max {want.abs().max():.2e})"
    assert diff.mean().item() <= mean_abs, f"{what}: mean-abs {diff.mean().item():.3e}"


@pytest.mark.parametrize("d,bs", [(64, 64), (128, 64), (64, 128), (128, 128)])
def test_sparse_backward_matches_oracle_autograd(d, bs):
    torch.manual_seed(d + bs)
    b, h, nq, nkv = 2, 3, 4, 7
    lkv = nkv * bs - bs // 4           # partial trailing key block
    q = torch.randn(b, h, nq * bs, d).bfloat16()
    k = torch.randn(b, h, nkv * bs, d).bfloat16()
    v = torch.randn(b, h, nkv * bs, d).bfloat16()
    k[:, :, lkv:] = 0
    v[:, :, lkv:] = 0
    index = torch.stack([torch.randperm(nkv) for _ in range(b * h * nq)]).view(b, h, nq, nkv).int()
    num = torch.randint(0, nkv + 1, (b, h, nq), dtype=torch.int32)
    num[0, 0, 0] = 0                   # empty row
    index[1, 2, 1, :3] = torch.tensor([4, 4, 2])  # a duplicated block counts twice
    num[1, 2, 1] = 3
    sizes = O.variable_block_sizes(lkv, nkv * bs, bs)
    do = torch.randn(b, h, nq * bs, d)

    qr, kr, vr = (t.double().requires_grad_() for t in (q, k, v))
    want = O.block_sparse_attention(qr, kr, vr, index, num, sizes, bs)
    want.backward(do.double())

    qg, kg, vg = (t.to(DEV).requires_grad_() for t in (q, k, v))
    got = W.block_sparse_attention_reference(qg, kg, vg, index.to(DEV), num.to(DEV), sizes.to(DEV), bs)
    got.float().backward(do.to(DEV))
    assert_close(got, want, what="out")
    for name, g, r in (("dq", qg.grad, qr.grad), ("dk", kg.grad, kr.grad), ("dv", vg.grad, vr.grad)):
        assert_close(g[:, :, :lkv] if name != "dq" else g, r[:, :, :lkv] if name != "dq" else r,
                     what=f"{name} d={d} bs={bs}")


@pytest.mark.parametrize("d,bs,tail", [(64, 64, 1), (128, 64, 20), (128, 64, 45), (64, 128, 70), (128, 128, 127)])
def test_sparse_backward_long_lists_in_block_order(d, bs, tail):
    """Lists of more than 32 blocks are walked in block order unless a block occurs twice; the last
    key block holds ``tail`` real keys (none of a wave's key half, or part of it)."""
    torch.manual_seed(d + bs + tail)
    b, h, nq, nkv = 1, 2, 3, 40
    lkv = (nkv - 1) * bs + tail
    q, k, v = (torch.randn(b, h, n * bs, d).bfloat16() for n in (nq, nkv, nkv))
    k[:, :, lkv:] = 0
    v[:, :, lkv:] = 0
    index = torch.stack([torch.randperm(nkv) for _ in range(b * h * nq)]).view(b, h, nq, nkv).int()
    num = torch.tensor([[33, 32, 40], [40, 37, 34]], dtype=torch.int32).view(b, h, nq)
    index[0, 1, 0, 3] = index[0, 1, 0, 30]  # a duplicate keeps the list's order
    index[0, 1, 1, 5] = nkv + 9             # clamped onto the last block
    sizes = O.variable_block_sizes(lkv, nkv * bs, bs)
    do = torch.randn(b, h, nq * bs, d)
    qr, kr, vr = (t.double().requires_grad_() for t in (q, k, v))
    O.block_sparse_attention(qr, kr, vr, index, num, sizes, bs).backward(do.double())
    qg, kg, vg = (t.to(DEV).requires_grad_() for t in (q, k, v))
    got = W.block_sparse_attention_reference(qg, kg, vg, index.to(DEV), num.to(DEV), sizes.to(DEV), bs)
    got.float().backward(do.to(DEV))
    for name, g, r in (("dq", qg.grad, qr.grad), ("dk", kg.grad, kr.grad), ("dv", vg.grad, vr.grad)):
        assert_close(g[:, :, :lkv] if name != "dq" else g, r[:, :, :lkv] if name != "dq" else r, what=name)


def test_sparse_backward_rectangular_lq_ne_lkv():
    """cfg-5-like rectangle (the Triton reference backward assumes Lq == Lkv)."""
    torch.manual_seed(5)
    b, h, d, bs = 1, 2, 128, 128
    nq, nkv = 3, 20
    q, k, v = torch.randn(b, h, nq * bs, d).bfloat16(), torch.randn(b, h, nkv * bs, d).bfloat16(), \
        torch.randn(b, h, nkv * bs, d).bfloat16()
    index = torch.stack([torch.randperm(nkv) for _ in range(b * h * nq)]).view(b, h, nq, nkv).int()
    num = torch.full((b, h, nq), 6, dtype=torch.int32)
    sizes = torch.full((nkv,), bs, dtype=torch.int32)
    do = torch.randn(b, h, nq * bs, d)
    qr, kr, vr = (t.double().requires_grad_() for t in (q, k, v))
    O.block_sparse_attention(qr, kr, vr, index, num, sizes, bs).backward(do.double())
    qg, kg, vg = (t.to(DEV).requires_grad_() for t in (q, k, v))
    W.block_sparse_attention_reference(qg, kg, vg, index.to(DEV), num.to(DEV), sizes.to(DEV), bs).float().backward(do.to(DEV))
    for name, g, r in (("dq", qg.grad, qr.grad), ("dk", kg.grad, kr.grad), ("dv", vg.grad, vr.grad)):
        assert_close(g, r, what=name)


@pytest.mark.parametrize("nq,nkv", [(65, 31), (130, 33), (256, 32)])
def test_sparse_backward_transposed_lists_by_counting(nq, nkv):
    """Transposed lists from the counting kernel at the edges of its 64-query and 32-key-block runs,
    with duplicates, empty rows and rows of up to all key blocks; gradients keep bf16 inputs' type."""
    torch.manual_seed(nq)
    b, h, d, bs = 1, 2, 64, 64
    q, k, v = (torch.randn(b, h, n * bs, d).bfloat16() for n in (nq, nkv, nkv))
    index = torch.stack([torch.randperm(nkv) for _ in range(b * h * nq)]).view(b, h, nq, nkv).int()
    num = torch.randint(0, 4, (b, h, nq), dtype=torch.int32)
    num[0, 0, nq - 1], num[0, 1, 0] = nkv, 0
    index[0, 1, 1, :2] = nkv - 1
    num[0, 1, 1] = 2
    sizes = torch.full((nkv,), bs, dtype=torch.int32)
    do = torch.randn(b, h, nq * bs, d)
    qr, kr, vr = (t.float().requires_grad_() for t in (q, k, v))
    O.block_sparse_attention_gather(qr, kr, vr, index, num, sizes, bs).backward(do)
    qg, kg, vg = (t.to(DEV).requires_grad_() for t in (q, k, v))
    got = W.block_sparse_attention_reference(qg, kg, vg, index.to(DEV), num.to(DEV), sizes.to(DEV), bs)
    got.backward(do.to(DEV).bfloat16())
    for name, g, r in (("dq", qg.grad, qr.grad), ("dk", kg.grad, kr.grad), ("dv", vg.grad, vr.grad)):
        # dO is rounded to bf16 on the GPU side (2^-9), gradients of up to ~|r| are stored in bf16
        assert g.dtype == torch.bfloat16
        scale = max(1.0, r.abs().max().item())
        assert_close(g, r, 2e-2 * scale, 2e-3 * scale, what=name)


@pytest.mark.parametrize("d,bs,lkv,sparse,acc,bf16", [
    (64, 64, 1, False, False, False), (128, 64, 525, False, True, False), (128, 128, 525, False, False, True),
    (64, 128, 130, True, False, True), (128, 64, 200, True, True, False), (128, 128, 257, True, False, False)])
def test_key_side_lists_cut_into_runs_match_the_oracle(d, bs, lkv, sparse, acc, bf16):
    """Few key blocks: every list is cut into runs that a second launch adds up. Dense lists, lists
    shorter than the number of runs, empty ones, partial last blocks, a heads subset, added-to fp32
    gradients and bf16 ones (rounded once: 2^-9 of the gradient on top of the fp32 bound)."""
    from worldattention_amd.hsa._bwd import bsa_backward
    from worldattention_amd.hsa.block_sparse import bsa_forward
    torch.manual_seed(lkv + d)
    b, h, lq = 1, 3, 2500
    nq, nkv = -(-lq // bs), -(-lkv // bs)
    q = torch.randn(b, h, lq, d).bfloat16()
    k, v = (torch.randn(b, h, lkv, d).bfloat16() for _ in range(2))
    do = torch.randn(b, h, lq, d).bfloat16() * 0.25
    index = num = None
    allow = torch.ones(h, lq, lkv, dtype=torch.bool)
    if sparse:
        index = torch.stack([torch.randperm(nkv) for _ in range(b * h * nq)]).view(b, h, nq, nkv).int()
        num = torch.randint(1, nkv + 1, (b, h, nq), dtype=torch.int32)
        num[0, 0] = (index[0, 0] == nkv - 1).int().argmax(-1).clamp(min=1)  # the last block: (nearly) never
        index[0, 2, 3:, 0], num[0, 2, 3:] = 0, 1             # blocks other than 0: at most three query blocks
        blocks = torch.zeros(h, nq, nkv, dtype=torch.bool)
        for i in range(h):
            for r in range(nq):
                blocks[i, r, index[0, i, r, :num[0, i, r]].long()] = True
        allow = blocks.repeat_interleave(bs, 1)[:, :lq].repeat_interleave(bs, 2)[:, :, :lkv]
    heads = torch.tensor([2, 0], dtype=torch.int32)
    dev = lambda t: None if t is None else t.to(DEV)
    qg, kg, vg = dev(q), dev(k), dev(v)
    out = torch.zeros(b, h, lq, d, device=DEV)
    _, lse = bsa_forward(qg, kg, vg, index=dev(index), num=dev(num), block_size=bs, heads=dev(heads), out=out,
                         want_lse=True)
    kw = dict(dtype=torch.bfloat16 if bf16 else torch.float32, device=DEV)
    dk, dv = (torch.full((b, h, lkv, d), 0.5, **kw) for _ in range(2))
    bsa_backward(qg, kg, vg, out, lse, dev(do), index=dev(index), num=dev(num), block_size=bs, heads=dev(heads),
                 dk=dk, dv=dv, kv_accumulate=acc)
    qr, kr, vr = (t[0].double().requires_grad_() for t in (q, k, v))
    p = (qr @ kr.transpose(1, 2) * d ** -0.5).masked_fill(~allow, float("-inf")).softmax(-1)
    (p @ vr).backward(do[0].double())
    for name, g, r in (("dk", dk, kr.grad), ("dv", dv, vr.grad)):
        for i in range(h):
            want = r[i] + (0.5 if acc else 0.0) if i in (0, 2) else torch.full_like(r[i], 0.5)
            scale = max(1.0, r[i].abs().max().item())
            assert_close(g[0, i], want, 2e-2 * scale, 2e-3 * scale, what=f"{name} head {i}")


@pytest.mark.parametrize("b,h,d,bs,lkv,seg,rank,bf16", [
    (1, 2, 128, 64, 700, 156, 3, True), (2, 1, 64, 128, 333, 100, 40, True), (1, 1, 128, 128, 1000, 1000, 128, False),
    (1, 2, 64, 64, 130, 10, 5, True), (1, 1, 128, 64, 6200, 1560, 25, True)])
def test_compressed_term_in_the_key_side_pass_equals_its_own_pass(b, h, d, bs, lkv, seg, rank, bf16):
    """E^T g of compressed keys and values added by the dK/dV pass against wa_compress_kv_bwd's dx
    (same products in the same order: equal): segments that end within a wave's 32 keys, several
    segments there, ranks past 32, a partial last block, unlisted key blocks, an infinite gradient."""
    from worldattention_amd.hsa._autograd import _compress_backward
    from worldattention_amd.hsa._bwd import bsa_backward
    from worldattention_amd.hsa.block_sparse import bsa_forward
    torch.manual_seed(lkv + seg)
    lq = 300
    nq, nkv = -(-lq // bs), -(-lkv // bs)
    q = torch.randn(b, lq, h, d, device=DEV).bfloat16()
    k, v = (torch.randn(b, lkv, h, d, device=DEV).bfloat16() for _ in range(2))
    do = torch.randn(b, lq, h, d, device=DEV)
    index = torch.randint(0, max(nkv - 1, 1), (b, h, nq, nkv), dtype=torch.int32, device=DEV)
    num = torch.randint(0, min(nkv, 4) + 1, (b, h, nq), dtype=torch.int32, device=DEV)
    rows = sum(min(rank, -(-min(seg, lkv - s) // bs)) for s in range(0, lkv, seg))
    gk, gv = (torch.randn(b, rows, h, d, device=DEV) for _ in range(2))
    gk[0, rows - 1, 0, 3] = float("inf")
    pk, pv = (torch.randn(rank, seg + 2, device=DEV).bfloat16() for _ in range(2))
    out = torch.zeros(b, lq, h, d, device=DEV)
    _, lse = bsa_forward(q, k, v, index=index, num=num, block_size=bs, layout="blhd", out=out, want_lse=True)
    kw = dict(index=index, num=num, block_size=bs, layout="blhd")
    dt = torch.bfloat16 if bf16 else torch.float32
    dk, dv = (torch.full((b, lkv, h, d), 7.0, dtype=dt, device=DEV) for _ in range(2))
    dq, _, _ = bsa_backward(q, k, v, out, lse, do, dk=dk, dv=dv, compressed=(gk, gv, pk, pv, seg, bs), **kw)
    dq_want, dk_want, dv_want = bsa_backward(q, k, v, out, lse, do, **kw)
    dk_want, _ = _compress_backward(gk, k, pk, seg, bs, dx=dk_want, out_dtype=dt)
    dv_want, _ = _compress_backward(gv, v, pv, seg, bs, dx=dv_want, out_dtype=dt)
    assert torch.equal(dq, dq_want)
    assert dk_want.isinf().any() and not dk_want[0, :seg].isinf().any() or lkv <= seg
    for name, got, want in (("dk", dk, dk_want), ("dv", dv, dv_want)):
        assert got.dtype == want.dtype
        torch.testing.assert_close(got, want, rtol=0, atol=0, equal_nan=True, msg=lambda m: f"{name}: {m}")
    assert _compress_backward(gk, k, pk, seg, bs, want_dx=False)[0] is None


def test_sparse_backward_many_query_blocks():
    """More than 256 query blocks: the transposed lists come from the scanning kernel instead of the
    counting one."""
    torch.manual_seed(9)
    b, h, d, bs = 1, 1, 64, 64
    nq, nkv = 260, 64                  # about 12 query blocks per key block: unit-scale gradients
    q = torch.randn(b, h, nq * bs, d).bfloat16()
    k, v = torch.randn(b, h, nkv * bs, d).bfloat16(), torch.randn(b, h, nkv * bs, d).bfloat16()
    index = torch.randint(0, nkv, (b, h, nq, 3), dtype=torch.int32)
    num = torch.randint(0, 4, (b, h, nq), dtype=torch.int32)
    sizes = torch.full((nkv,), bs, dtype=torch.int32)
    do = torch.randn(b, h, nq * bs, d)
    qr, kr, vr = (t.double().requires_grad_() for t in (q, k, v))
    O.block_sparse_attention(qr, kr, vr, index, num, sizes, bs).backward(do.double())
    qg, kg, vg = (t.to(DEV).requires_grad_() for t in (q, k, v))
    W.block_sparse_attention_reference(qg, kg, vg, index.to(DEV), num.to(DEV), sizes.to(DEV), bs).float().backward(do.to(DEV))
    for name, g, r in (("dq", qg.grad, qr.grad), ("dk", kg.grad, kr.grad), ("dv", vg.grad, vr.grad)):
        assert_close(g, r, what=name)


@pytest.mark.parametrize("d", [64, 128])
def test_elu1_backward_matches_oracle_autograd(d):
    from worldattention_amd.hsa._autograd import elu1_backward
    torch.manual_seed(d)
    b, lq, lkv, h = 1, 300, 2000, 3
    q, k, v = (torch.randn(b, n, h, d) for n in (lq, lkv, lkv))
    g = torch.randn(b, lq, h, d)
    qr, kr, vr = (t.double().requires_grad_() for t in (q, k, v))
    out = O.linear_branch_elu1(qr.transpose(1, 2), kr.transpose(1, 2), vr.transpose(1, 2), compute_dtype=torch.float64)
    out.transpose(1, 2).backward(g.double())
    heads = torch.tensor([0, 2], dtype=torch.int32, device=DEV)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    s, z = WA.elu1_state(kd, vd, heads)
    dq, dk, dv = (torch.zeros(t.shape, device=DEV) for t in (q, k, v))
    elu1_backward(qd, kd, vd, g.to(DEV), s, z, heads, dq, dk, dv)
    for hh in (0, 2):
        assert_close(dq[:, :, hh], qr.grad[:, :, hh], what=f"dq h{hh}")
        assert_close(dk[:, :, hh], kr.grad[:, :, hh], what=f"dk h{hh}")
        assert_close(dv[:, :, hh], vr.grad[:, :, hh], what=f"dv h{hh}")
    assert torch.count_nonzero(dq[:, :, 1]) == 0


def _grads_both(cfg, gate_w, gate_b, do, proj=None, keep_dtype=False):
    """(GPU grads, oracle grads, oracle parts) of hsa_attention for one config. The oracle runs fp32
    autograd on the same input values; the GPU gets fp32 copies, or (``keep_dtype``) the tensors
    themselves, e.g. bf16 as the benchmark feeds them, and then so does the oracle's forward."""
    q, k, v = cfg["q"], cfg["k"], cfg["v"]
    d = q.shape[-1]
    kw = dict(block_size=cfg["block_size"], routing=cfg["routing"], topk=cfg.get("topk"),
              head_modes=cfg.get("head_modes"), linear_mode=cfg["linear_mode"], proj_segment_len=cfg["proj_segment_len"])
    if proj is None:
        rank = -(-cfg["proj_segment_len"] // cfg["block_size"])
        proj = O.init_projection(rank, cfg["proj_segment_len"], cfg["block_size"])
    qr, kr, vr = (t.detach().float().clone().requires_grad_() for t in (q, k, v))
    wr, br = gate_w.clone().requires_grad_(), gate_b.clone().requires_grad_()
    # With keep_dtype the oracle's forward sees the inputs in their own dtype too (bf16 inputs make
    # the reference round the pooled block means to bf16, which decides the routing), while its
    # math runs in fp32 and the gradients reach the fp32 leaves through the casts.
    qi, ki, vi = (t.to(s.dtype) for t, s in zip((qr, kr, vr), (q, k, v))) if keep_dtype else (qr, kr, vr)
    out_r, parts = O.hsa_attention(qi, ki, vi, k_proj_mat=proj, v_proj_mat=proj, gate_weight=wr, gate_bias=br,
                                   return_parts=True, **kw)
    out_r.float().backward(do.float())
    lin = torch.nn.Linear(d, d).to(DEV)
    with torch.no_grad():
        lin.weight.copy_(gate_w)
        lin.bias.copy_(gate_b)
    qg, kg, vg = ((t.detach().to(DEV) if keep_dtype else t.detach().float().to(DEV)).requires_grad_()
                  for t in (q, k, v))
    out_g = W.hsa_attention(qg, kg, vg, k_proj_mat=proj.to(DEV), v_proj_mat=proj.to(DEV), gate_lin=lin, **kw)
    out_g.float().backward(do.to(DEV).float())
    return ((out_g, qg.grad, kg.grad, vg.grad, lin.weight.grad, lin.bias.grad),
            (out_r, qr.grad, kr.grad, vr.grad, wr.grad, br.grad), parts)


def test_hsa_split_heads_topk_elu1_gradients_match_oracle():
    torch.manual_seed(11)
    cfg = workloads.cfg1()
    cfg["q"], cfg["k"], cfg["v"] = (t * 8 for t in (cfg["q"], cfg["k"], cfg["v"]))  # unit-scale inputs
    d = cfg["q"].shape[-1]
    do = torch.randn(cfg["q"].shape)
    got, want, _ = _grads_both(cfg, torch.randn(d, d) * 0.1, torch.full((d,), 0.3), do)
    for name, g, r in zip(("out", "dq", "dk", "dv", "dW", "db"), got, want):
        tol = (0.1, 1e-2) if name in ("dW", "db") else (2e-2, 2e-3)   # parameter grads sum over tokens
        assert_close(g, r, *tol, what=name)


@pytest.mark.parametrize("b,length,h,d,seg,bs,rank,plen,xdt", [
    (2, 700, 3, 64, 256, 64, 4, 256, torch.bfloat16),     # three segments, the last of rank 3
    (1, 1000, 5, 128, 1000, 32, 20, 1000, torch.float32),  # one segment, rank 20, fp32 x
    (1, 300, 2, 32, 128, 64, 8, 200, torch.bfloat16),     # rows and columns of E no segment uses
])
def test_compress_backward_matches_oracle_autograd(b, length, h, d, seg, bs, rank, plen, xdt):
    """wa_compress_kv_bwd: dx and dE against autograd through the oracle's compress_kv in fp32 (the
    same fp32 arithmetic, so only the summation order differs: 1e-3 max-abs, 1e-4 mean-abs), dx
    added to an existing gradient, and two calls bit for bit equal (fixed-order dE sum)."""
    from worldattention_amd.hsa._autograd import _compress_backward
    torch.manual_seed(length + d)
    x = torch.randn(b, length, h, d).to(xdt)
    proj = (torch.randn(rank, plen) / 16).bfloat16()
    lc = O.compress_kv(x.permute(0, 2, 1, 3), x.permute(0, 2, 1, 3), segment_len=seg, k_proj_mat=proj,
                       v_proj_mat=proj, block_size=bs)[0].shape[2]
    g = torch.randn(b, lc, h, d)
    xr = x.float().permute(0, 2, 1, 3).clone().requires_grad_(True)
    pr = proj.float().clone().requires_grad_(True)
    out, _ = O.compress_kv(xr, xr.detach(), segment_len=seg, k_proj_mat=pr, v_proj_mat=pr.detach(), block_size=bs)
    (out * g.permute(0, 2, 1, 3)).sum().backward()
    want_dx, want_dp = xr.grad.permute(0, 2, 1, 3), pr.grad

    xg, pg, gg = x.to(DEV), proj.to(DEV), g.to(DEV)
    dx, dp = _compress_backward(gg, xg, pg, seg, bs)
    assert_close(dx, want_dx, 1e-3, 1e-4, what="dx")
    assert_close(dp, want_dp, 1e-3, 1e-4, what="dE")
    base = torch.randn(b, length, h, d, device=DEV)
    dx2, dp2 = _compress_backward(gg, xg, pg, seg, bs, dx=base.clone())
    assert torch.equal(dp2, dp), "dE differs between two calls"
    assert_close(dx2, base + dx, 1e-6, 1e-7, what="accumulated dx")


@pytest.mark.parametrize("b,length,h,d,seg,bs,rank,xdt,pdt", [
    (1, 133, 5, 64, 100, 64, 2, torch.bfloat16, torch.bfloat16),    # a last segment of rank 1; 10 columns of 32
    (2, 260, 1, 128, 130, 4, 33, torch.float32, torch.float32),     # one row in a second 32-row tile
    (1, 640, 3, 32, 320, 4, 80, torch.float32, torch.float32),      # rank over 64
    (1, 64, 2, 128, 64, 1, 64, torch.bfloat16, torch.float32),      # exactly one token tile and two row tiles
    (3, 65, 2, 64, 65, 1, 65, torch.float32, torch.bfloat16),       # one token and one row past the tiles
])
def test_compress_backward_split_products_match_fp64(b, length, h, d, seg, bs, rank, xdt, pdt):
    """dx and dE on the matrix cores from three-part splits of the fp32 operands, against fp64: a sum
    of n fp32 products in any order is within n 2^-24 of the sum of their magnitudes; the bf16 form
    of dx is the rounding of the fp32 one, and infinities and NaN in a gradient column stay in it."""
    from worldattention_amd.hsa._autograd import _compress_backward
    torch.manual_seed(length + rank)
    x = torch.randn(b, length, h, d, device=DEV).to(xdt)
    proj = (torch.randn(rank, seg, device=DEV) / 16).to(pdt)
    spans = [(s, min(seg, length - s)) for s in range(0, length, seg)]
    ranks = [min(rank, -(-n // bs)) for _, n in spans]
    g = torch.randn(b, sum(ranks), h, d, device=DEV) * torch.randn(b, sum(ranks), h, d, device=DEV).exp()
    base = torch.randn(b, length, h, d, device=DEV)
    dx, dp = _compress_backward(g, x, proj, seg, bs)
    added, _ = _compress_backward(g, x, proj, seg, bs, dx=base.clone())
    rounded, _ = _compress_backward(g, x, proj, seg, bs, dx=base, out_dtype=torch.bfloat16)
    assert torch.equal(added, base + dx) and torch.equal(rounded, added.bfloat16())
    want_p, row = torch.zeros(2, rank, seg, dtype=torch.float64, device=DEV), 0
    for (s, n), r in zip(spans, ranks):
        e, xs, gs = proj[:r, :n].double(), x[:, s:s + n].double(), g[:, row:row + r].double()
        want = torch.einsum("jt,bjhd->bthd", e, gs)
        bound = (r + 2) * 2.0 ** -24 * torch.einsum("jt,bjhd->bthd", e.abs(), gs.abs())
        assert ((dx[:, s:s + n].double() - want).abs() <= bound).all(), f"dx of segment {s}"
        want_p[0, :r, :n] += torch.einsum("bjhd,bthd->jt", gs, xs)
        want_p[1, :r, :n] += torch.einsum("bjhd,bthd->jt", gs.abs(), xs.abs())
        row += r
    assert ((dp.double() - want_p[0]).abs() <= (b * h * d + len(spans) + 8) * 2.0 ** -24 * want_p[1]).all()
    g[0, 0, 0, 0], g[0, 0, 0, 1], g[0, 0, 0, 2] = float("inf"), float("nan"), 3.3e38
    odd, _ = _compress_backward(g, x, proj, seg, bs)
    t0 = spans[0][1] // 2
    want = torch.einsum("jt,jd->td", proj[:ranks[0], t0:t0 + 1].double(), g[0, :ranks[0], 0, :4].double())
    assert torch.equal(odd[0, t0, 0, 0].double(), want[0, 0]) and odd[0, t0, 0, 1].isnan()
    assert (odd[0, t0, 0, 2].double() - want[0, 2]).abs() <= 1e-6 * want[0, 2].abs()


def test_hsa_reference_mode_gradients_match_oracle():
    """Reference semantics: every head runs both branches, Gini routing, low-rank softmax branch."""
    torch.manual_seed(3)
    b, lq, lkv, h, d = 1, 200, 640, 2, 64
    cfg = dict(q=torch.randn(b, lq, h, d), k=torch.randn(b, lkv, h, d), v=torch.randn(b, lkv, h, d), block_size=64,
               routing="gini", linear_mode="lowrank", proj_segment_len=128)
    proj = (torch.rand(2, 128) / 64).bfloat16()
    do = torch.randn(b, lq, h, d)
    got, want, parts = _grads_both(cfg, torch.randn(d, d) * 0.1, torch.zeros(d), do, proj=proj)
    for name, g, r in zip(("out", "dq", "dk", "dv", "dW", "db"), got, want):
        tol = (0.1, 1e-2) if name in ("dW", "db") else (2e-2, 2e-3)
        assert_close(g, r, *tol, what=name)


_LOWRANK_TRAINING = [  # dtype, d, head modes, lq, lkv, coarse caches given, runs of a key list > 1
    ("bfloat16", 128, "BBB", 200, 700, False, False),    # written bf16 dK / dV with the compression's term added
    ("bfloat16", 128, "BBB", 1100, 330, False, True),    # lists in runs: the term by its own pass, from fp32
    ("float32", 64, "BB", 1100, 330, False, True),
    ("float32", 128, "SBB", 200, 700, False, False),     # every head sparse, not every one linear
    ("bfloat16", 64, "BLB", 200, 330, False, False),     # every head linear, not every one sparse
    ("bfloat16", 128, "BSL", 300, 700, False, False),    # neither: everything accumulated
    ("bfloat16", 64, "SL", 1100, 330, False, True),
    ("bfloat16", 128, "BB", 200, 700, True, False),      # given coarse keys and values
    ("float32", 64, "SBL", 1100, 330, True, True),
]


@pytest.mark.parametrize("case", _LOWRANK_TRAINING, ids=lambda c: "-".join(str(x) for x in c))
def test_hsa_lowrank_gradients_match_oracle(case):
    """Training of the low-rank configuration in every form its backward distinguishes: outputs and
    gradients of q, k, v, the projections (or the coarse caches) and the gate against fp32 autograd
    through the oracle. bf16 operands, probabilities, their gradients and results carry up to 2^-9
    a rounding; five of them are within 1e-2 of a tensor's norm. Memory the backward allocates holds
    NaN, so that a gradient nobody wrote shows."""
    from worldattention_amd import _lib
    dtype, d, modes, lq, lkv, coarse, runs = case
    torch.manual_seed(lq + lkv + d)
    dt, h, bs, seg = getattr(torch, dtype), len(modes), 64, 156
    n_sparse = sum(m != "L" for m in modes)
    assert (_lib.lib().wa_bsa_bwd_key_runs(1, n_sparse, lq, lkv, bs) > 1) == runs
    leaves = {n: torch.randn(1, length, h, d).to(dt).float() for n, length in (("q", lq), ("k", lkv), ("v", lkv))}
    proj = {n: (torch.randn(3, seg) / 16).bfloat16().float() for n in ("pk", "pv")}
    if coarse:
        lc = sum(min(3, -(-min(seg, lkv - s) // bs)) for s in range(0, lkv, seg))
        leaves.update((n, torch.randn(1, lc, h, d).to(dt).float()) for n in ("kc", "vc"))
    else:
        leaves.update(proj)
    leaves.update(w=torch.randn(d, d) * 0.1, bias=torch.randn(d) * 0.1)
    do = torch.randn(1, lq, h, d).to(dt).float()
    kw = dict(block_size=bs, routing="gini", linear_mode="lowrank", proj_segment_len=seg,
              head_modes=[{"B": "both", "S": "sparse", "L": "linear"}[m] for m in modes])

    want = {n: t.clone().requires_grad_() for n, t in leaves.items()}
    ref = {n: want[n].to(dt) for n in ("q", "k", "v")}
    extra = {a: want[n].to(dt) for a, n in (("k_coarse", "kc"), ("v_coarse", "vc"))} if coarse else {}
    out_r = O.hsa_attention(*ref.values(), k_proj_mat=want.get("pk"), v_proj_mat=want.get("pv"), gate_weight=want["w"],
                            gate_bias=want["bias"], **extra, **kw)
    out_r.float().backward(do)

    lin = torch.nn.Linear(d, d).to(DEV)
    with torch.no_grad():
        lin.weight.copy_(leaves["w"])
        lin.bias.copy_(leaves["bias"])
    types = dict(pk=torch.bfloat16, pv=torch.bfloat16)
    got = {n: t.to(DEV, types.get(n, dt)).requires_grad_() for n, t in leaves.items() if n not in ("w", "bias")}
    extra = dict(k_coarse=got["kc"], v_coarse=got["vc"]) if coarse else {}
    pk, pv = (got[n] if n in got else proj[n].to(DEV, torch.bfloat16) for n in ("pk", "pv"))
    out_g = W.hsa_attention(got["q"], got["k"], got["v"], k_proj_mat=pk, v_proj_mat=pv, gate_lin=lin, **extra, **kw)
    for _ in range(2):  # every block the caching allocator hands to the backward held NaN
        junk = [torch.full((n,), float("nan"), device=DEV) for t in got.values() for n in (t.numel(), t.numel() // 2) * 4]
        del junk
    out_g.backward(do.to(DEV, out_g.dtype))
    grads = {n: t.grad for n, t in got.items()} | dict(w=lin.weight.grad, bias=lin.bias.grad)
    for name, g, r in [("out", out_g, out_r)] + [(n, grads[n], want[n].grad) for n in grads]:
        g, r = g.detach().double().cpu(), r.detach().double()
        assert torch.isfinite(g).all(), name
        rel = ((g - r).norm() / r.norm()).item()
        assert rel <= 1e-2, f"{name}: relative error {rel:.2e}"


@pytest.mark.parametrize("keep_dtype", [True, False], ids=["bf16", "fp32"])
def test_cfg5_wan_chunk_fwd_bwd_matches_oracle(keep_dtype):
    """cfg 5: Lq=4680, Lkv=32760, H=12, D=128, block 128, top-k 16 on 8 sparse heads + 4 elu1 heads;
    dO ~ N(0, 1); a gate with N(0, 0.02) weights. Compares the output and dQ, dK, dV of both
    branches with the oracle's fp32 autograd at max-abs 2e-2 / mean-abs 2e-3. ``bf16``: the bf16
    tensors go in as the benchmark feeds them (bf16 elu1 state and key-side kernels, dK / dV written
    once in bf16); ``fp32``: fp32 copies of the same values (the fp32 kernels)."""
    cfg = workloads.cfg5()
    d = cfg["q"].shape[-1]
    g = torch.Generator().manual_seed(5)
    gate_w = torch.randn(d, d, generator=g) * 0.02
    got, want, parts = _grads_both(cfg, gate_w, torch.zeros(d), cfg["do"], keep_dtype=keep_dtype)
    if keep_dtype:
        assert got[2].dtype == got[3].dtype == torch.bfloat16
    for name, gg, r in zip(("out", "dq", "dk", "dv"), got[:4], want[:4]):
        assert_close(gg, r, what=f"cfg5 {name}")


@pytest.mark.parametrize("d", [64, 128])
def test_bf16_dk_dv_are_the_fp32_gradients_rounded(d):
    """dkv_dtype = WA_BF16: the sparse and elu1 backward kernels write dK / dV once in bf16; the
    values are the fp32 path's, rounded to nearest even (bit-exact). At D = 64 this also pins the
    bf16 elu1 key side against the fp32 kernel on every token (the elu1 gradients are ~1e-3, below
    what the oracle tolerances resolve)."""
    from worldattention_amd.hsa._autograd import elu1_backward
    from worldattention_amd.hsa._bwd import bsa_backward
    from worldattention_amd.hsa.block_sparse import bsa_forward
    torch.manual_seed(21)
    b, h, bs, nq, nkv = 1, 2, 128, 3, 9
    lkv = nkv * bs - 40
    q = torch.randn(b, nq * bs, h, d, device=DEV).bfloat16()
    k = torch.randn(b, lkv, h, d, device=DEV).bfloat16()
    v = torch.randn(b, lkv, h, d, device=DEV).bfloat16()
    index = torch.stack([torch.randperm(nkv) for _ in range(b * h * nq)]).view(b, h, nq, nkv).int().to(DEV)
    num = torch.tensor([[[4, 9, 2], [0, 5, 7]]], dtype=torch.int32, device=DEV)
    out = torch.empty(b, nq * bs, h, d, device=DEV)
    _, lse = bsa_forward(q, k, v, index=index, num=num, block_size=bs, layout="blhd", out=out, lkv=lkv,
                           want_lse=True)
    do = torch.randn(out.shape, device=DEV)
    f32 = [torch.empty(t.shape, device=DEV) for t in (q, k, v)]
    bsa_backward(q, k, v, out, lse, do, index=index, num=num, block_size=bs, layout="blhd", lkv=lkv,
                 dq=f32[0], dk=f32[1], dv=f32[2])
    dk16, dv16 = (torch.empty(t.shape, device=DEV, dtype=torch.bfloat16) for t in (k, v))
    bsa_backward(q, k, v, out, lse, do, index=index, num=num, block_size=bs, layout="blhd", lkv=lkv,
                 dq=torch.empty(q.shape, device=DEV), dk=dk16, dv=dv16)
    assert torch.equal(dk16, f32[1].bfloat16()) and torch.equal(dv16, f32[2].bfloat16())

    heads = torch.tensor([1], dtype=torch.int32, device=DEV)
    s, z = WA.elu1_state(k, v, heads)
    g = torch.randn(b, nq * bs, h, d, device=DEV)
    grads = []
    for dt in (torch.float32, torch.bfloat16):
        dq = torch.zeros(q.shape, device=DEV)
        dk, dv = (torch.zeros(t.shape, device=DEV, dtype=dt) for t in (k, v))
        elu1_backward(q, k, v, g, s, z, heads, dq, dk, dv, kv_accumulate=False)
        grads.append((dk, dv))
    (dk32, dv32), (dk16, dv16) = grads
    assert torch.equal(dk16[:, :, 1], dk32[:, :, 1].bfloat16()) and torch.equal(dv16[:, :, 1], dv32[:, :, 1].bfloat16())
    with pytest.raises(Exception):
        bsa_backward(q, k, v, out, lse, do, index=index, num=num, block_size=bs, layout="blhd", lkv=lkv,
                     dq=torch.zeros(q.shape, device=DEV), dk=dk16, dv=dv16, accumulate=True)


@pytest.mark.parametrize("b,lkv,h,heads", [(1, 20, 2, [0]), (1, 64, 3, [0, 2]), (2, 777, 3, [1, 2]),
                                           (1, 4100, 2, [0, 1])])
def test_bf16_elu1_key_side_equals_the_fp32_path_rounded(b, lkv, h, heads):
    """The elu1 key side with bf16 K / V and bf16 dK / dV at D = 128 (the streamed kernel: runs of
    one, two and many 32-token tiles, a partial last tile, two batches, a subset of the heads) gives
    the fp32 key side's values rounded to bf16, bit for bit, and leaves the other heads untouched."""
    from worldattention_amd.hsa._autograd import elu1_backward
    torch.manual_seed(lkv)
    d, lq = 128, 300
    q = torch.randn(b, lq, h, d, device=DEV).bfloat16()
    k = torch.randn(b, lkv, h, d, device=DEV).bfloat16()
    v = torch.randn(b, lkv, h, d, device=DEV).bfloat16()
    heads_t = torch.tensor(heads, dtype=torch.int32, device=DEV)
    s, z = WA.elu1_state(k, v, heads_t)
    g = torch.randn(b, lq, h, d, device=DEV)
    grads = []
    for dt in (torch.float32, torch.bfloat16):
        dq = torch.zeros(q.shape, device=DEV)
        dk, dv = (torch.full(t.shape, 7.0, device=DEV, dtype=dt) for t in (k, v))
        elu1_backward(q, k, v, g, s, z, heads_t, dq, dk, dv, kv_accumulate=False)
        grads.append((dk, dv))
    (dk32, dv32), (dk16, dv16) = grads
    assert torch.equal(dk16[:, :, heads], dk32[:, :, heads].bfloat16())
    assert torch.equal(dv16[:, :, heads], dv32[:, :, heads].bfloat16())
    others = [x for x in range(h) if x not in heads]
    if others:
        assert bool((dk16[:, :, others] == 7.0).all()) and bool((dv16[:, :, others] == 7.0).all())
    assert torch.isfinite(dk16.float()).all() and float(dk16[:, :, heads].float().abs().max()) > 0


def test_hsa_bf16_inputs_get_bf16_gradients_within_tolerance():
    """Split heads with bf16 q / k / v: dK and dV come back bf16 straight from the kernels."""
    torch.manual_seed(12)
    cfg = workloads.cfg1()
    q, k, v = (t * 8 for t in (cfg["q"], cfg["k"], cfg["v"]))
    kw = dict(block_size=cfg["block_size"], routing=cfg["routing"], topk=cfg["topk"], head_modes=cfg["head_modes"],
              linear_mode=cfg["linear_mode"], proj_segment_len=cfg["proj_segment_len"])
    q16, k16, v16 = (t.bfloat16() for t in (q, k, v))
    do = torch.randn(q.shape)
    qr, kr, vr = (t.float().requires_grad_() for t in (q16, k16, v16))
    O.hsa_attention(qr.bfloat16(), kr.bfloat16(), vr.bfloat16(), **kw).float().backward(do)
    qg, kg, vg = (t.to(DEV).requires_grad_() for t in (q16, k16, v16))
    W.hsa_attention(qg, kg, vg, k_proj_mat=None, v_proj_mat=None, **kw).float().backward(do.to(DEV))
    assert kg.grad.dtype == vg.grad.dtype == torch.bfloat16
    for name, g, r in (("dq", qg.grad, qr.grad), ("dk", kg.grad, kr.grad), ("dv", vg.grad, vr.grad)):
        assert_close(g, r, what=f"bf16 {name}")


def test_training_step_graph_replays_equal_eager_steps():
    """Forward + backward at the cfg 5 shape captured in a HIP graph (as bench.py times the training
    step): every replay, with eager steps and synchronizations between replays, gives the eager
    step's gradients bit for bit."""
    cfg = workloads.cfg5(device=DEV, seed=4)
    d = cfg["q"].shape[-1]
    gate = torch.nn.Linear(d, d).to(DEV)
    with torch.no_grad():
        gate.weight.normal_(0, 0.02)
        gate.bias.normal_(0, 0.02)
    q, k, v = (cfg[n].detach().requires_grad_() for n in ("q", "k", "v"))
    kw = dict(k_proj_mat=None, v_proj_mat=None, gate_lin=gate, block_size=128, routing="topk", topk=cfg["topk"],
              head_modes=cfg["head_modes"], linear_mode="elu1", proj_segment_len=1560)
    params = (q, k, v, gate.weight, gate.bias)

    def step():
        for t in params:
            t.grad = None
        W.hsa_attention(q, k, v, **kw).backward(cfg["do"])

    step()
    want = [t.grad.clone() for t in params]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    got = [t.grad for t in params]
    for i in range(3):
        graph.replay()
        torch.cuda.synchronize()
        for name, g, w in zip(("dq", "dk", "dv", "dW", "db"), got, want):
            assert torch.equal(g, w), f"replay {i}: {name} differs from the eager step"
        step()                            # eager step between replays
        torch.cuda.synchronize()
        for name, t, w in zip(("dq", "dk", "dv", "dW", "db"), params, want):
            assert torch.equal(t.grad, w), f"eager step after replay {i}: {name} differs"


@pytest.mark.parametrize("which", ["cfg1", "cfg5"])
def test_one_call_backward_equals_the_composed_calls(which, monkeypatch):
    """Split top-k / elu1 heads with bf16 inputs train through wa_hsa_fwd (with its training
    outputs) and wa_hsa_bwd, two library calls with the linear heads on a side stream. With the
    one-call path switched off the same step runs the composed path (a dozen launches on one
    stream, dq in fp32 then rounded): output and dQ, dK, dV, dW, db must agree bit for bit."""
    cfg = workloads.cfg5(device=DEV, seed=6) if which == "cfg5" else workloads.cfg1(device=DEV)
    if which == "cfg1":
        cfg["q"], cfg["k"], cfg["v"] = (t * 8 for t in (cfg["q"], cfg["k"], cfg["v"]))
    q0, k0, v0 = (cfg[n].to(DEV, torch.bfloat16) for n in ("q", "k", "v"))
    d = q0.shape[-1]
    gate = torch.nn.Linear(d, d).to(DEV)
    with torch.no_grad():
        gate.weight.normal_(0, 0.05)
        gate.bias.normal_(0, 0.05)
    do = torch.randn(q0.shape, generator=torch.Generator().manual_seed(3)).to(DEV, torch.bfloat16)
    kw = dict(k_proj_mat=None, v_proj_mat=None, gate_lin=gate, block_size=cfg["block_size"], routing="topk",
              topk=cfg["topk"], head_modes=cfg["head_modes"], linear_mode="elu1",
              proj_segment_len=cfg["proj_segment_len"])
    results = []
    for one_call in (True, False):
        monkeypatch.setattr(WA, "ONE_CALL", one_call)
        q, k, v = (t.clone().requires_grad_() for t in (q0, k0, v0))
        gate.weight.grad = gate.bias.grad = None
        out = W.hsa_attention(q, k, v, **kw)
        out.backward(do)
        results.append((out.detach().clone(), q.grad, k.grad, v.grad, gate.weight.grad.clone(),
                        gate.bias.grad.clone()))
    torch.cuda.synchronize()
    one, composed = results
    assert one[1].dtype == one[2].dtype == one[3].dtype == torch.bfloat16
    for name, a, b in zip(("out", "dq", "dk", "dv", "dW", "db"), one, composed):
        assert a.dtype == b.dtype, name
        assert torch.equal(a, b), f"{which} {name}: one-call path differs from the composed calls"


def test_one_call_backward_with_and_without_the_dq_stream_is_identical(monkeypatch):
    """The one-call backward's sparse dQ pass on its own stream (the default) or on the caller's
    stream after the transposed lists: the same kernels on the same inputs, the same bits."""
    from worldattention_amd.hsa import _autograd as A
    cfg = workloads.cfg5(device=DEV, seed=8)
    d = cfg["q"].shape[-1]
    gate = torch.nn.Linear(d, d).to(DEV)
    kw = dict(k_proj_mat=None, v_proj_mat=None, gate_lin=gate, block_size=128, routing="topk", topk=cfg["topk"],
              head_modes=cfg["head_modes"], linear_mode="elu1", proj_segment_len=1560)
    grads = []
    for flag in (True, False):
        monkeypatch.setattr(A, "DQ_STREAM", flag)
        q, k, v = (cfg[n].detach().clone().requires_grad_() for n in ("q", "k", "v"))
        W.hsa_attention(q, k, v, **kw).backward(cfg["do"])
        torch.cuda.synchronize()
        grads.append((q.grad, k.grad, v.grad))
    for name, a, b in zip(("dq", "dk", "dv"), *grads):
        assert torch.equal(a, b), f"{name} differs with the dQ pass on the caller's stream"


@pytest.mark.parametrize("d,bs", [(64, 64), (128, 128)])
def test_one_call_path_batch_of_two_matches_composed_and_oracle(d, bs, monkeypatch):
    """Two samples, ragged lengths (Lq = 300, Lkv = 1000: partial last query and key blocks),
    top-k sparse heads and elu1 linear heads in bf16 through the one-call forward and backward:
    output and gradients equal the composed launches bit for bit and the oracle within the
    forward / backward tolerances."""
    g = torch.Generator().manual_seed(d + bs)
    h, lq, lkv = 4, 300, 1000
    q = (torch.randn(2, lq, h, d, generator=g)).bfloat16()
    k = (torch.randn(2, lkv, h, d, generator=g) + torch.randn(2, 1, h, d, generator=g)).bfloat16()
    v = torch.randn(2, lkv, h, d, generator=g).bfloat16()
    do = torch.randn(2, lq, h, d, generator=g)
    w, b = torch.randn(d, d, generator=g) * 0.05, torch.randn(d, generator=g) * 0.05
    kw = dict(block_size=bs, routing="topk", topk=[3, 0, 5, 0], head_modes=["sparse", "linear", "sparse", "linear"],
              linear_mode="elu1", proj_segment_len=lkv)
    gate = torch.nn.Linear(d, d).to(DEV)
    with torch.no_grad():
        gate.weight.copy_(w)
        gate.bias.copy_(b)
    results = []
    for one_call in (True, False):
        monkeypatch.setattr(WA, "ONE_CALL", one_call)
        qg, kg, vg = (t.to(DEV).requires_grad_() for t in (q, k, v))
        gate.weight.grad = gate.bias.grad = None
        out = W.hsa_attention(qg, kg, vg, k_proj_mat=None, v_proj_mat=None, gate_lin=gate, **kw)
        out.float().backward(do.to(DEV))
        results.append((out.detach(), qg.grad, kg.grad, vg.grad, gate.weight.grad.clone(), gate.bias.grad.clone()))
    torch.cuda.synchronize()
    for name, a, c in zip(("out", "dq", "dk", "dv", "dW", "db"), *results):
        assert torch.equal(a, c), f"B=2 {name}: one-call path differs from the composed calls"
    ref = [t.float().clone().requires_grad_() for t in (q, k, v)]
    wr, br = w.clone().requires_grad_(), b.clone().requires_grad_()
    out_r = O.hsa_attention(*(t.bfloat16() for t in ref), gate_weight=wr, gate_bias=br, **kw)
    out_r.float().backward(do)
    assert_close(results[0][0], out_r, what="B=2 out")
    for name, got, r in zip(("dq", "dk", "dv"), results[0][1:4], ref):
        assert_close(got, r.grad, what=f"B=2 {name}")
