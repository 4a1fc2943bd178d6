"""The AlphaFold2 triangle-attention block around attention(): the pure-PyTorch form of the block on
the CPU (structure, ending = starting on the transposed pair tensor, key mask), and on the GPU the
block with the HIP kernels against that form, outputs and every gradient."""
import math

import pytest
import torch

from triangle_attention import TriangleAttention


def _rel_l2(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


def test_block_reference_form_on_cpu():
    torch.manual_seed(0)
    start = TriangleAttention(16, 8, 2, starting=True)
    end = TriangleAttention(16, 8, 2, starting=False)
    end.load_state_dict(start.state_dict())
    z = torch.randn(2, 6, 6, 16)
    out = start.reference_forward(z)
    assert out.shape == z.shape and torch.isfinite(out).all()
    # Alg. 14 is Alg. 13 on the transposed pair representation
    assert torch.allclose(end.reference_forward(z), start.reference_forward(z.transpose(1, 2)).transpose(1, 2), atol=1e-6)
    # a masked key position influences nothing but its own row/column of the output
    km = torch.ones(2, 6)
    km[:, 4:] = 0
    z2 = z.clone()
    z2[:, :4, 4:] += 1.0  # pairs (i, k) with a masked key k, rows i that are kept
    a, b = start.reference_forward(z, km), start.reference_forward(z2, km)
    assert torch.allclose(a[:, :4, :4], b[:, :4, :4], atol=1e-5)


def test_block_needs_the_gpu_library():
    blk = TriangleAttention(32, 32, 2)
    with pytest.raises(ValueError, match="no CPU path"):
        blk(torch.randn(1, 128, 128, 32))


@pytest.mark.gpu
@pytest.mark.parametrize("starting", [True, False])
def test_block_matches_pure_torch_on_gpu(starting):
    torch.manual_seed(1)
    dev = "cuda:0"
    blk = TriangleAttention(64, 32, 4, starting=starting).to(dev)
    z = torch.randn(1, 128, 128, 64, device=dev)
    km = torch.ones(1, 128, device=dev)
    km[:, 120:] = 0
    dout = torch.randn_like(z)
    res = {}
    for name, fn in (("hip", blk.forward), ("ref", blk.reference_forward)):
        zz = z.clone().requires_grad_(True)
        blk.zero_grad(set_to_none=True)
        out = fn(zz, km)
        out.backward(dout)
        torch.cuda.synchronize()
        res[name] = {"out": out.detach(), "z": zz.grad.detach(), **{n: p.grad.detach().clone() for n, p in blk.named_parameters()}}
    assert (res["hip"]["out"] - res["ref"]["out"]).abs().max().item() <= 1e-2
    for n in res["ref"]:
        if n != "out":
            assert _rel_l2(res["hip"][n], res["ref"][n]) <= 1e-2, n


class _OracleAttention(torch.autograd.Function):
    """attention() restated with the oracle: forward = oracle_forward, backward = the closed forms of
    oracle_backward (fp32, L1-chunked).  Plugged into the block in place of the HIP op."""

    @staticmethod
    def forward(ctx, q, k, v, b, sm):
        from oracle import tt_attn_oracle as orc
        ctx.save_for_backward(q, k, v, b)
        ctx.sm = sm
        return orc.oracle_forward(q, k, v, b, sm, dtype=torch.float32, l1_chunk=64)[0].to(q.dtype)

    @staticmethod
    def backward(ctx, do):
        from oracle import tt_attn_oracle as orc
        q, k, v, b = ctx.saved_tensors
        g = orc.oracle_backward(q, k, v, b, ctx.sm, do, dtype=torch.float32, l1_chunk=64)
        return g["dq"].to(q.dtype), g["dk"].to(k.dtype), g["dv"].to(v.dtype), g["db"].to(b.dtype), None


@pytest.mark.gpu
@pytest.mark.parametrize("zdtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("starting", [True, False])
def test_block_at_the_crop_shape_against_the_oracle(starting, zdtype):
    """The block at the AlphaFold2 crop size (c_z 128, 4 heads of 32, L 384; fp32 and bf16 pair
    representation, both node types) against the same block with the attention op replaced by the oracle's
    forward and closed-form backward on the same 16-bit operands: output max-abs <= 1e-2 (bf16: 3e-2,
    half a unit in the last place of the block's bf16 output), gradients relative-L2 <= 1e-2 (bf16 2e-2)."""
    import math
    torch.manual_seed(2)
    dev = "cuda:0"
    blk = TriangleAttention(128, 32, 4, starting=starting).to(dev).to(zdtype)
    z = torch.randn(1, 384, 384, 128, device=dev).to(zdtype)
    dout = torch.randn_like(z)
    res = {}
    for name in ("hip", "oracle"):
        zz = z.clone().requires_grad_(True)
        blk.zero_grad(set_to_none=True)
        if name == "hip":
            out = blk(zz)
        else:
            q, k, v, bias, gate = blk._operands(zz, None)
            out = blk._finish(_OracleAttention.apply(q, k, v, bias, 1.0 / math.sqrt(blk.c_hidden)), gate, zz.dtype)
        out.backward(dout)
        torch.cuda.synchronize()
        res[name] = {"out": out.detach().float(), "z": zz.grad.detach().float(),
                     **{n: p.grad.detach().float().clone() for n, p in blk.named_parameters()}}
    o_tol, g_tol = (1e-2, 1e-2) if zdtype == torch.float32 else (3e-2, 2e-2)
    assert (res["hip"]["out"] - res["oracle"]["out"]).abs().max().item() <= o_tol
    for n in res["oracle"]:
        if n != "out":
            assert _rel_l2(res["hip"][n], res["oracle"][n]) <= g_tol, n


class _Unfused(TriangleAttention):
    """The block as separate torch operations around attention() (a subclass does not take the fused kernels)."""


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("C,H,D,B,L,starting,masked,dropout_p", [
    (128, 4, 32, 1, 1, True, False, 0.0),      # one pair
    (128, 4, 32, 2, 5, False, True, 0.0),      # 25 rows of a 32-row block, two batch entries
    (128, 4, 32, 1, 33, True, True, 0.0),      # 1089 rows: a last block of one row
    (128, 4, 32, 2, 64, False, False, 0.0),    # whole blocks
    (128, 4, 32, 1, 200, True, False, 0.2),    # enough rows for the weights in LDS, several chunks of the weight gradients
    (64, 2, 32, 1, 40, True, False, 0.0), (64, 4, 32, 1, 41, False, True, 0.0),
    (128, 1, 64, 1, 40, True, True, 0.0), (128, 2, 64, 1, 39, False, False, 0.0), (64, 1, 64, 1, 9, True, False, 0.0)])
def test_fused_block_kernels_against_separate_operations(C, H, D, B, L, starting, masked, dropout_p, dtype):
    torch.manual_seed(4)
    fused = TriangleAttention(C, D, H, starting=starting, dropout_p=dropout_p).to("cuda:0")
    with torch.no_grad():
        fused.layer_norm.weight.add_(0.3 * torch.randn(C, device="cuda:0"))
        fused.layer_norm.bias.add_(0.3 * torch.randn(C, device="cuda:0"))
    plain = _Unfused(C, D, H, starting=starting, dropout_p=dropout_p).to("cuda:0")
    plain.load_state_dict(fused.state_dict())
    z = torch.randn(B, L, L, C, device="cuda:0").to(dtype) + 0.5
    dout = torch.randn_like(z)
    km = None
    if masked:
        km = torch.ones(B, L, device="cuda:0")
        km[:, L - max(1, L // 8):] = 0
    res = []
    for blk in (fused.to(dtype), plain.to(dtype)):
        zz = z.clone().requires_grad_(True)
        out = blk(zz, km, 7)
        res.append({"out": out, "z": torch.autograd.grad(out, [zz, *blk.parameters()], dout)})
        torch.cuda.synchronize()
    assert fused._fused(z, km, 7) is not None and plain._fused(z, km, 7) is None
    tol = {torch.float16: 3e-3, torch.bfloat16: 2e-2, torch.float32: 1e-3}[dtype]
    names = ["z", *(n for n, _ in fused.named_parameters())]
    assert _rel_l2(res[0]["out"], res[1]["out"]) <= tol
    for n, a, b in zip(names, res[0]["z"], res[1]["z"]):
        # (one pair: every softmax is over one key, the gradients of q, k and the bias are zero up to rounding)
        assert _rel_l2(a, b) <= tol or (L == 1 and b.abs().max() < 1e-2), n


@pytest.mark.gpu
@pytest.mark.parametrize("L,dtype", [(192, torch.float32), (257, torch.float32), (363, torch.bfloat16)])
def test_row_blocks_beyond_a_round_of_the_waves(L, dtype):
    """The output and gate-gradient kernels deal row blocks of 32 pairs to the workgroups in turn.  2304 halves of row blocks, 2065 and 4118 whole
    ones for 2048, 2048 and 4096 waves: a second round that few of the waves have.  Same tolerance as above."""
    test_fused_block_kernels_against_separate_operations(128, 4, 32, 1, L, True, False, 0.0, dtype)


@pytest.mark.gpu
def test_block_dropout_draws_a_fresh_mask_per_call_and_replays_a_given_seed():
    torch.manual_seed(3)
    dev = "cuda:0"
    blk = TriangleAttention(64, 32, 2, dropout_p=0.25).to(dev)
    z = torch.randn(1, 128, 128, 64, device=dev)
    blk.train()
    a, b = blk(z), blk(z)
    assert not torch.equal(a, b)                      # two calls, two masks
    assert torch.equal(blk(z, seed=11), blk(z, seed=11))
    blk.eval()
    assert torch.equal(blk(z), blk(z))                # no dropout outside training


@pytest.mark.gpu
def test_example_script_runs_as_upstream_s_does():
    """example_usage.py (the call sequence of upstream's example: inputs, attention(), MSE loss, backward,
    print the gradients) runs as a program: k and v, which do not require gradients, print None."""
    import os
    import re
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "example_usage.py")], capture_output=True, text=True, timeout=600, cwd=root)
    assert r.returncode == 0, r.stderr[-2000:]
    lines = dict(l.split(" ", 1) for l in r.stdout.strip().splitlines())
    assert lines["k"] == "None" and lines["v"] == "None"
    for name, shape in (("q", "(4, 8, 128, 128, 32)"), ("bias", "(4, 8, 128, 128)")):
        m = re.match(r"\(\((.*)\), ([0-9.e+-]+)\)", lines[name])
        assert m and "(" + m.group(1) + ")" == shape and 0.0 < float(m.group(2)) < float("inf"), lines[name]


def test_block_imports_after_the_repo_root_alias_module():
    """`flash_tt_attn` at the repo root (the documented import path) and the block must load in one
    process, whichever of the two module files `flash_tt_attn` resolved to first."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = ("import sys; sys.path.insert(0, %r); import flash_tt_attn; "
            "assert flash_tt_attn.__file__ == %r, flash_tt_attn.__file__; "
            "sys.path.insert(1, %r); import triangle_attention; print(triangle_attention.TriangleAttention.__name__)"
            % (root, os.path.join(root, "flash_tt_attn.py"), os.path.join(root, "flash-triangle-attention_amd")))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300, cwd="/")
    assert r.returncode == 0 and "TriangleAttention" in r.stdout, r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,C,H,D", [
    (1, 1, 128, 4, 32),    # one row of a 32-row stage
    (1, 33, 128, 4, 32),   # 1089 rows: a last stage of one row
    (2, 40, 64, 2, 32), (1, 23, 64, 4, 32), (1, 41, 128, 1, 64), (1, 96, 128, 2, 64),
    (1, 160, 128, 4, 32)])  # several stages per workgroup, both workgroups of a row
def test_fp32_block_products_hold_fp32_precision(B, L, C, H, D):
    """Every product of an fp32 block, formed again in float64 from the operands that the kernels left in the forward
    state and the backward workspace.  Bound: an operand short of its third bf16 part is off by up to 2^-17 (typically
    3e-6 of the result), sums of up to 25600 rows in fp32 by chunks stay below 6e-7: 1e-6."""
    import ctypes

    import fta_lib
    lib = fta_lib.load()
    torch.manual_seed(5)
    HD, n, m = H * D, B * L * L * H * D, B * L * L * H
    rn = lambda *s: torch.randn(*s, device="cuda:0")
    z, dout = rn(B, L, L, C), rn(B, L, L, C)
    w = {"norm_weight": 1 + 0.1 * rn(C), "norm_bias": 0.1 * rn(C), "bg": 0.1 * rn(HD), "bo": 0.1 * rn(C), "wb": rn(H, C) / C ** 0.5,
         "wo": rn(C, HD) / HD ** 0.5, **{k: rn(HD, C) / C ** 0.5 for k in ("wq", "wk", "wv", "wg")}}
    st = (ctypes.c_int64 * 3)(L * L * C, L * C, C)
    blk = fta_lib.Block(B=B, L=L, C=C, H=H, D=D, dtype=fta_lib.DTYPE_F32, eps=1e-5, sm_scale=D ** -0.5, z=z.data_ptr(), z_stride=st)
    state = torch.empty(lib.fta_block_state_bytes(ctypes.byref(blk)), dtype=torch.uint8, device="cuda:0")
    ws = torch.empty(lib.fta_block_bwd_workspace_bytes(ctypes.byref(blk)), dtype=torch.uint8, device="cuda:0")
    out, dz, g = torch.empty_like(z), torch.empty_like(z), {k: torch.empty_like(t) for k, t in w.items()}
    grads = fta_lib.BlockGrads(z=dz.data_ptr(), z_stride=st)
    for k in w:
        setattr(blk, k, w[k].data_ptr())
        setattr(grads, k, g[k].data_ptr())
    fta_lib.check(lib.fta_block_fwd(ctypes.byref(blk), out.data_ptr(), st, state.data_ptr(), 0))
    fta_lib.check(lib.fta_block_bwd(ctypes.byref(blk), state.data_ptr(), dout.data_ptr(), st, ctypes.byref(grads), ws.data_ptr(), ws.numel(), 0))
    torch.cuda.synchronize()

    def parts(buf, sizes):  # regions at multiples of 256 bytes
        at, r = 0, []
        for by in sizes:
            r.append(buf[at:at + by])
            at += (by + 255) // 256 * 256
        return r
    rows = lambda t, dt, d: t.view(dt).view(B, H, L, L, d).permute(0, 2, 3, 1, 4).reshape(-1, H * d).double()
    q, k, v, o, bias, gate, _ = parts(state, [2 * n] * 4 + [2 * m, 4 * n, 4 * m])
    _, dgp, dq, dk, dv, db = parts(ws, [2 * n, 4 * n, 2 * n, 2 * n, 2 * n, 2 * m])
    o, gate, dgp = rows(o, torch.float16, D), rows(gate, torch.float32, D), rows(dgp, torch.float32, D)
    dq, dk, dv, db = (rows(t, torch.float16, d) for t, d in ((dq, D), (dk, D), (dv, D), (db, 1)))
    w = {k: t.double() for k, t in w.items()}
    z, dout, dz, out = (t.reshape(-1, C).double() for t in (z, dout, dz, out))
    mean, rstd = z.mean(-1, keepdim=True), (z.var(-1, unbiased=False, keepdim=True) + 1e-5).rsqrt()
    xh = (z - mean) * rstd
    x = xh * w["norm_weight"] + w["norm_bias"]
    dx = dq @ w["wq"] + dk @ w["wk"] + dv @ w["wv"] + dgp @ w["wg"] + db @ w["wb"]
    dxh = dx * w["norm_weight"]
    pairs = {"gate": (gate, torch.sigmoid(x @ w["wg"].T + w["bg"])), "out": (out, (gate * o) @ w["wo"].T + w["bo"]),
             "d gate": (dgp, (dout @ w["wo"]) * o * gate * (1 - gate)),
             "dz": (dz, rstd * (dxh - dxh.mean(-1, keepdim=True) - xh * (dxh * xh).mean(-1, keepdim=True))),
             "wq": (g["wq"], dq.T @ x), "wk": (g["wk"], dk.T @ x), "wv": (g["wv"], dv.T @ x), "wg": (g["wg"], dgp.T @ x),
             "wb": (g["wb"], db.T @ x), "wo": (g["wo"], dout.T @ (gate * o)), "bg": (g["bg"], dgp.sum(0)), "bo": (g["bo"], dout.sum(0)),
             "norm_weight": (g["norm_weight"], (dx * xh).sum(0)), "norm_bias": (g["norm_bias"], dx.sum(0))}
    for name, (a, b) in pairs.items():
        # (one pair: the softmax over one key passes nothing on to q, k and the bias)
        assert _rel_l2(a, b) <= 1e-6 or (L == 1 and name in ("wq", "wk", "wb") and (a.double() - b).abs().max() <= 1e-6), name
    # what proj rounds to the attention's type: half a unit of fp16
    for name, got in (("wq", q), ("wk", k), ("wv", v)):
        assert _rel_l2(rows(got, torch.float16, D), x @ w[name].T) <= 2 ** -11, name
    assert _rel_l2(rows(bias, torch.float16, 1), x @ w["wb"].T) <= 2 ** -11


def _same_values(a, b, tol, name):
    """NaN where NaN is, infinity of the same sign where infinity is, elsewhere the same values (relative L2)."""
    a, b = a.double(), b.double()
    assert torch.equal(a.isnan(), b.isnan()), f"{name}: {int(a.isnan().sum())} NaN for {int(b.isnan().sum())}"
    for sign in (1, -1):
        assert torch.equal(a == sign * float("inf"), b == sign * float("inf")), f"{name}: infinities"
    ok = b.isfinite()
    if bool(ok.any()):
        scale = b[ok].abs().max().clamp_min(1e-30)  # (squares of the largest values overflow)
        assert _rel_l2(a[ok] / scale, b[ok] / scale) <= tol, name


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,C,H,D", [(1, 33, 128, 4, 32), (2, 40, 64, 2, 32), (1, 41, 128, 1, 64), (1, 24, 64, 4, 32), (1, 160, 128, 4, 32)])
@pytest.mark.parametrize("where", ["gate weight", "output weight", "largest output weight", "gradient", "largest gradient", "key weight", "norm weight"])
def test_infinities_of_an_fp32_block_come_out_as_they_went_in(where, B, L, C, H, D):
    """An infinite weight or incoming gradient, and finite ones next to the type's largest value, against the block as
    separate fp32 layers around attention(): the same infinities, the same NaN, and the finite values as without them.  (The
    gradients of the projections are gamma * (d^T xhat) + beta * (sum of d), with infinite d not what d^T x is: not compared.)"""
    torch.manual_seed(6)
    fused, plain = TriangleAttention(C, D, H).to("cuda:0"), _Unfused(C, D, H).to("cuda:0")
    z = torch.randn(B, L, L, C, device="cuda:0")
    dout = torch.randn_like(z)
    inf, big = float("inf"), 3.4e38
    with torch.no_grad():
        if where == "gate weight":  # saturated gates: everything stays finite but the sums over this channel
            fused.linear_g.weight[5, 7] = inf
            fused.linear_g.weight[C // 2 - 1, 3] = -inf
        elif where == "output weight":
            fused.linear_o.weight[3, 9] = inf
        elif where == "largest output weight":
            fused.linear_o.weight[3, 9] = big
        elif where == "key weight":
            fused.linear_k.weight[1, 2] = -inf
        elif where == "norm weight":
            fused.layer_norm.weight[4] = inf
        elif where == "gradient":
            dout[0, L - 1, L - 2, 6] = -inf
            dout[0, 1, 2, 8] = inf
        else:
            dout[0, 1, 2, 8] = -big
    plain.load_state_dict(fused.state_dict())
    res = []
    for blk in (fused, plain):
        zz = z.clone().requires_grad_(True)
        out = blk(zz)
        res.append([out, *torch.autograd.grad(out, [zz, *blk.parameters()], dout)])
        torch.cuda.synchronize()
    assert fused._fused(z, None, None) is not None
    for name, a, b in zip(["out", "z", *(n for n, _ in fused.named_parameters())], *res):
        if where != "gradient" or name in ("out", "z", "linear_o.weight", "linear_o.bias"):
            _same_values(a, b, 1e-3, name)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,L,C,H,D", [(1, 33, 128, 4, 32), (2, 41, 64, 2, 32), (1, 35, 128, 2, 64), (1, 40, 128, 4, 32)])
def test_an_infinite_bias_gradient_of_the_last_pair_makes_infinite_weight_gradients(B, L, C, H, D, dtype):
    """The bias gradient, fp16, overflows at the last pair alone (every row adds to it, and its softmax weight, half, is that of all
    other keys together).  The bias weights' gradient is then infinite wherever norm weight * xhat and norm bias agree in sign, also where
    the pairs do not fill the last stage of 64 (32 in fp32) rows, which repeats the last pair."""
    torch.manual_seed(8)
    blk = TriangleAttention(C, D, H).to("cuda:0", dtype)
    z = 0.01 * torch.randn(B, L, L, C, device="cuda:0")
    z[:, :, L - 1, 1] = 6.0       # this key's value, the same in every row
    z[:, L - 1, L - 1, 0] = 6.0   # the last pair's bias
    with torch.no_grad():
        for lin in (blk.linear_q, blk.linear_k, blk.linear_v, blk.linear_b):
            lin.weight.zero_()
        x0 = torch.nn.functional.layer_norm(z[0, L - 1, L - 1].double(), (C,))[0].item()
        blk.linear_b.weight[:, 0] = math.log(L - 1.0) / (x0 + 1.0)  # (beside the other pairs' bias of about -1 times the same)
        blk.linear_v.weight[:, 1] = 1.0
        blk.layer_norm.bias.fill_(-1.0)
        blk.linear_g.weight.zero_()
        blk.linear_o.weight.copy_(torch.eye(C, H * D))
    zz = z.to(dtype).requires_grad_(True)
    out = blk(zz)
    dout = torch.zeros_like(out)
    dout[:, :, L - 1] = 300.0
    wb, wv = torch.autograd.grad(out, (blk.linear_b.weight, blk.linear_v.weight), dout)
    torch.cuda.synchronize()
    assert blk._fused(zz, None, None) is not None
    assert bool(wv.isfinite().all())
    live = (C + D - 1) // D  # heads that the output projection reads
    assert bool((wb[:live, 2:] == -float("inf")).all()), wb
    assert bool(wb[live:].isfinite().all())


@pytest.mark.gpu
def test_gate_of_an_fp32_block_is_the_sigmoid_to_fp32_precision():
    """With zero gate weights the logits are the bias, from saturated to subnormal gates.  Bound: exp, good to one unit in the
    last place, and three roundings; an absolute 2^-149 where the gate is subnormal."""
    import ctypes

    import fta_lib
    lib = fta_lib.load()
    L, C, H, D = 3, 128, 4, 32
    st = (ctypes.c_int64 * 3)(L * L * C, L * C, C)
    zero, one = torch.zeros(C, C, device="cuda:0"), torch.ones(C, device="cuda:0")
    z, out = torch.randn(1, L, L, C, device="cuda:0"), torch.empty(1, L, L, C, device="cuda:0")
    for lo, hi in ((-88.6, -86.0), (-86.0, -20.0), (-20.0, 20.0), (-1.0, 1.0), (-110.0, -89.0)):
        bg = torch.linspace(lo, hi, H * D, device="cuda:0")
        blk = fta_lib.Block(B=1, L=L, C=C, H=H, D=D, dtype=fta_lib.DTYPE_F32, eps=1e-5, sm_scale=1.0, z=z.data_ptr(), z_stride=st,
                            norm_weight=one.data_ptr(), norm_bias=one.data_ptr(), bg=bg.data_ptr(),
                            **{k: zero.data_ptr() for k in ("wq", "wk", "wv", "wb", "wg", "wo")})
        state = torch.empty(lib.fta_block_state_bytes(ctypes.byref(blk)), dtype=torch.uint8, device="cuda:0")
        fta_lib.check(lib.fta_block_fwd(ctypes.byref(blk), out.data_ptr(), st, state.data_ptr(), 0))
        torch.cuda.synchronize()
        n = L * L * H * D
        at = 4 * ((2 * n + 255) // 256 * 256) + (2 * L * L * H + 255) // 256 * 256
        gate = state[at:at + 4 * n].view(torch.float32).view(H, L, L, D).permute(1, 2, 0, 3).reshape(L * L, H * D).cpu().double()
        ref = torch.sigmoid(bg.cpu().double())
        # (exp(-x) overflows at 88.7: the gate is 0 from there)
        ref = torch.where(bg.cpu() < -88.72, torch.zeros_like(ref), ref)
        assert ((gate - ref).abs() <= 5 * 2.0 ** -24 * ref + 2.0 ** -149).all(), (lo, hi, ((gate - ref).abs() / ref.clamp_min(2.0 ** -149)).max())
