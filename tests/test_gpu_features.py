"""GPU parity of what upstream's README lists as future work (README.md:15-16) and this library has:
bf16 inputs and dropout on the attention weights, through the drop-in attention() and the C ABI,
against the same fp32 oracle (with the explicit keep mask for dropout)."""
import ctypes
import math

import numpy as np
import pytest
import torch

from oracle import dropout_mask as dm
from oracle import tt_attn_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# fp16 bars (north star): O max-abs <= 1e-2, gradients relative-L2 <= 1e-2.
# bf16 keeps 8 significant bits where fp16 keeps 11: every rounding (of the stored O and gradients, and
# of P and dS on their way into the matrix core -- upstream's kernels round them to the input type as
# well, flash_tt_attn.py:99, :356, :425) is 8 times coarser.  A stored O of magnitude 4..8 is off by up to
# half a unit in the last place = 1.6e-2 from the store alone, hence the absolute bar 3e-2 (two such
# units) for O; the gradients' relative-L2 averages the roundings and stays well under 8 x 1e-2: the bar
# is 2e-2 (measured 2e-3 to 5e-3; O 1.7e-2 at the benchmark shapes).
TOL = {torch.float16: (1e-2, 1e-2), torch.bfloat16: (3e-2, 2e-2)}


def _oracle(q, k, v, b, sm, do, **kw):
    B, H, L1, L2, D = q.shape
    chunk = max(1, min(L1, (1 << 27) // (L2 * L2 * B * H)))
    return orc.oracle_backward(q, k, v, b, sm, do, dtype=torch.float32, l1_chunk=chunk, **kw)


def _run(q, k, v, b, sm, do, *extra):
    import flash_tt_attn as fta
    qq, kk, vv, bb = (t.detach().requires_grad_(True) for t in (q, k, v, b))
    o = fta.attention(qq, kk, vv, bb, sm, *extra)
    dq, dk, dv, db = torch.autograd.grad(o, (qq, kk, vv, bb), do)
    torch.cuda.synchronize()
    return {"o": o, "dq": dq, "dk": dk, "dv": dv, "db": db}


def _compare(got, ref, dtype, tag):
    o_tol, g_tol = TOL[dtype]
    err = (got["o"].float() - ref["o"]).abs().max().item()
    errs = {n: orc.rel_l2(got[n], ref[n]) for n in ("dq", "dk", "dv", "db")}
    print(f"{tag}: O max-abs {err:.2e} " + " ".join(f"{n} {e:.2e}" for n, e in errs.items()), flush=True)
    assert got["o"].dtype == dtype and all(got[n].dtype == dtype for n in errs)
    assert err <= o_tol, f"{tag} O max-abs {err}"
    for n, e in errs.items():
        assert e <= g_tol, f"{tag} {n} rel-L2 {e}"


def _inputs(B, H, L1, L2, D, seed, dtype, bias_std=1.0):
    return orc.make_inputs(B, H, L1, L2, D, seed=seed, bias_std=bias_std, dtype=dtype, device=DEV)


# ---- bf16 ---------------------------------------------------------------------------------------------

@pytest.mark.parametrize("L", [128, 256, 512, 1024])
def test_bf16_benchmark_shapes_b4_h8_d32(L):
    # BASELINE configs[1] in bf16, sm_scale 1.3 as the upstream benchmark (:783)
    print(f"case bf16 bench L={L}", flush=True)
    q, k, v, b, do = _inputs(4, 8, L, L, 32, 20, torch.bfloat16)
    _compare(_run(q, k, v, b, 1.3, do), _oracle(q, k, v, b, 1.3, do), torch.bfloat16, f"bf16 L{L}")


def test_bf16_alphafold_crop_projected_inputs():
    # B=1,H=4,D=32,L=384, projections of a pair tensor, non-contiguous views
    H, D, L, C = 4, 32, 384, 128
    g = torch.Generator(device="cpu").manual_seed(7)
    z = torch.randn(1, L, L, C, generator=g)
    xavier = lambda i, o: (torch.rand(i, o, generator=g) * 2 - 1) * math.sqrt(6.0 / (i + o))
    proj = lambda w: (z @ w).view(1, L, L, H, D).permute(0, 3, 1, 2, 4).to(torch.bfloat16).to(DEV)
    q, k, v = proj(xavier(C, H * D)), proj(xavier(C, H * D)), proj(xavier(C, H * D))
    b = (z @ xavier(C, H)).permute(0, 3, 1, 2).to(torch.bfloat16).to(DEV)
    do = torch.randn(1, H, L, L, D, generator=g).to(torch.bfloat16).to(DEV)
    sm = 1.0 / math.sqrt(D)
    _compare(_run(q, k, v, b, sm, do), _oracle(q, k, v, b, sm, do), torch.bfloat16, "bf16 af2-crop")


@pytest.mark.parametrize("L", [1024, 1536])
def test_bf16_long_crop_peaked_softmax(L):
    # bias scaled by 3
    print(f"case bf16 long L={L}", flush=True)
    sm = 1.0 / math.sqrt(32)
    q, k, v, b, do = _inputs(1, 4, L, L, 32, 20, torch.bfloat16, bias_std=3.0)
    _compare(_run(q, k, v, b, sm, do), _oracle(q, k, v, b, sm, do), torch.bfloat16, f"bf16 long L{L}")


def test_bf16_ending_node_by_manual_permute_d64():
    # B=2,H=8,D=64,L=512, L1<->L2 transposed views
    sm = 1.0 / math.sqrt(64)
    q, k, v, b, do = _inputs(2, 8, 512, 512, 64, 5, torch.bfloat16)
    qt, kt, vt, dot = (t.transpose(2, 3) for t in (q, k, v, do))
    _compare(_run(qt, kt, vt, b, sm, dot), _oracle(qt, kt, vt, b, sm, dot), torch.bfloat16, "bf16 ending-node")


@pytest.mark.parametrize("B,H,L1,L2,D", [(1, 2, 9, 200, 32), (1, 1, 5, 900, 64), (2, 1, 3, 2560, 32), (1, 2, 7, 131, 32),
                                         (1, 1, 3, 1280, 64), (1, 1, 2, 1920, 32), (2, 2, 21, 384, 64), (1, 2, 8, 290, 64)])
def test_bf16_other_lengths_masks_and_determinism(B, H, L1, L2, D):
    print(f"case bf16 B={B} H={H} L1={L1} L2={L2} D={D}", flush=True)
    sm = 1.0 / math.sqrt(D)
    q, k, v, b, do = _inputs(B, H, L1, L2, D, 9, torch.bfloat16)
    b[..., L2 - 5:] = float("-inf")   # a key mask, as in the fp16 tests
    b[..., :3] = -1e9
    a = _run(q, k, v, b, sm, do)
    _compare(a, _oracle(q, k, v, b, sm, do), torch.bfloat16, f"bf16 L{L2} D{D}")
    c = _run(q, k, v, b, sm, do)
    for n in a:
        assert torch.isfinite(a[n].float()).all() and torch.equal(a[n], c[n]), n


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,L1,L2,D,lo,hi", [
    (1, 2, 5, 520, 64, 508, 520),    # every real key of the forward's last 128-key slab
    (1, 2, 5, 512, 32, 0, 256),      # the first four 64-key steps of a one-slab row
    (1, 2, 5, 1024, 32, 512, 1024),  # the whole second slab
    (1, 1, 4, 640, 64, 0, 130),      # the first slab and the start of the second
])
@pytest.mark.parametrize("mask", [float("-inf"), -1e9])
def test_masks_that_cover_all_keys_a_wave_has_seen(dtype, B, H, L1, L2, D, lo, hi, mask):
    """While every key a wave has seen is masked its running maximum is the floor that replaces the mask
    value, and the weights are exp2 of a difference of two products near that floor: it has to stay small
    enough for that difference to be harmless (a bf16 floor of -1e30 gave inf, then NaN, here)."""
    if mask == -1e9 and dtype == torch.float16:
        pytest.skip("-1e9 is not an fp16 value")
    print(f"case mask {dtype} B={B} H={H} L1={L1} L2={L2} D={D} keys {lo}..{hi} = {mask}", flush=True)
    sm = 1.0 / math.sqrt(D)
    q, k, v, b, do = _inputs(B, H, L1, L2, D, 13, dtype, bias_std=3.0)
    b[..., lo:hi] = mask
    got = _run(q, k, v, b, sm, do)
    for n in got:
        assert torch.isfinite(got[n].float()).all(), n
    _compare(got, _oracle(q, k, v, b, sm, do), dtype, f"mask {lo}..{hi} L{L2} D{D}")


_ALL_MASKED = [
    # one-kernel backward
    (64, 32, "plain"), (128, 32, "plain"), (128, 64, "plain"), (128, 32, "dropout"), (128, 64, "dropout"), (64, 32, "precise"), (128, 64, "precise"),
    (256, 32, "dropout"),
    # hand-scheduled backward (one and several key ranges; the precise instances in natural units)
    (256, 32, "plain"), (384, 32, "plain"), (512, 32, "plain"), (1024, 32, "plain"), (256, 64, "plain"), (384, 64, "plain"), (512, 64, "plain"),
    (256, 32, "precise"), (512, 32, "precise"),
    # general backward kernels
    (512, 32, "dropout"), (1024, 32, "dropout"), (256, 64, "dropout"), (512, 64, "precise"),
    # rows that end inside a tile: the keys beyond them weigh nothing beside masked ones either
    (3, 32, "plain"), (7, 64, "plain"), (9, 32, "dropout"), (33, 32, "plain"), (64, 64, "plain"), (64, 32, "dropout"), (97, 32, "precise"), (101, 64, "dropout"),
    (131, 32, "plain"), (200, 32, "plain"), (300, 32, "precise"), (457, 32, "plain"), (701, 32, "plain"), (1290, 32, "plain"), (1801, 32, "plain"),
    (200, 64, "plain"), (333, 64, "plain"), (514, 64, "plain"), (901, 64, "precise"),
    (131, 32, "dropout"), (300, 32, "dropout"), (514, 32, "dropout"), (202, 64, "dropout"), (514, 64, "dropout"),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("mask", ["-inf", "lowest"])
@pytest.mark.parametrize("L2,D,mode", _ALL_MASKED)
def test_queries_whose_keys_are_all_masked_attend_by_their_scores(L2, D, mode, mask, dtype):
    """With the same mask value on every key of a query (-inf, or the type's lowest) its softmax is that of the scores
    alone, in the output and in every gradient; other queries have the same value on some keys, which get weight 0.
    The weights of such a query are differences beside the floor that stands for the mask, where fp32 holds a
    score to 2^-9 and the logsumexp, a base-2 logarithm, to 2^-8: 5e-3 of a weight at most, half the tolerance."""
    import flash_tt_attn as fta
    if mode == "precise" and dtype == torch.bfloat16:
        pytest.skip("a mode of fp16")
    B, H, L1, sm = 1, 2, 3, 1.0 / math.sqrt(D)
    rows = sorted({0, 7 % L2, L2 - 1})
    q, k, v, b, do = _inputs(B, H, L1, L2, D, 3, dtype)
    low = float("-inf") if mask == "-inf" else torch.finfo(dtype).min
    b[..., L2 // 2:L2 // 2 + 5] = low
    ref_b = b.float()
    ref_b[..., L2 // 2:L2 // 2 + 5] = float("-inf")
    b[:, :, rows] = low
    ref_b[:, :, rows] = 0.0
    extra, kw, scale = (), {}, 1.0
    if mode == "dropout":
        keep, scale = dm.keep_mask(1234, 0.25, B, H, L1, L2)
        extra, kw = (0.25, 1234), dict(keep=torch.from_numpy(keep).to(DEV), keep_scale=scale)
    fta.PRECISE_BACKWARD = mode == "precise"
    try:
        got = _run(q, k, v, b, sm, do, *extra)
    finally:
        fta.PRECISE_BACKWARD = False
    ref = _oracle(q, k, v, ref_b, sm, do, **kw)
    got["o"], ref["o"] = (got["o"].detach().float() / scale).to(dtype), ref["o"] / scale  # (as the other dropout tests)
    _compare(got, ref, dtype, f"all masked L{L2} D{D} {mode}")
    for n in ("o", "dq", "db"):  # the masked queries by themselves
        e = orc.rel_l2(got[n][..., rows, :], ref[n][..., rows, :])
        assert e <= TOL[dtype][1], f"{n} of the masked queries: rel-L2 {e}"


@pytest.fixture
def general_kernels():
    """Selects the general backward kernels where the pipelined ones would run (library test hook)."""
    import fta_lib
    lib = fta_lib.load()
    old = lib.fta_debug_select_kernels(3)
    yield lib
    lib.fta_debug_select_kernels(old)


def test_bf16_feature_instances_where_the_pipelined_kernels_would_run(general_kernels):
    """bf16 at D=32, L2 a multiple of 128 and a moderate softmax scale runs the hand-scheduled backward
    kernels (scaled Q/K rounded to bf16, bias and row constants through fp16 MFMAs); with those switched
    off the vector-ALU instances run (as they do for D=64, tails, large scales and the precise mode).
    Both meet the same bars."""
    sm = 0.3
    q, k, v, b, do = _inputs(2, 2, 24, 512, 32, 31, torch.bfloat16)
    _compare(_run(q, k, v, b, sm, do), _oracle(q, k, v, b, sm, do), torch.bfloat16, "bf16 general L512")


def test_bf16_long_d64_rows_on_the_vector_alu_instances():
    """D=64 rows beyond 1024 keys run forward instances with 32-key stages; a bf16 call at a scale that
    selects the vector-ALU backward instances has to tile such a row from the full forward set."""
    q, k, v, b, do = _inputs(1, 1, 2, 1280, 64, 3, torch.bfloat16)
    _compare(_run(q, k, v, b, 0.9, do), _oracle(q, k, v, b, 0.9, do), torch.bfloat16, "bf16 D64 L1280 sm 0.9")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L1,L2,cut", [(5, 600, "64,10,"), (4, 800, "64,14,"), (3, 1100, "64,12,"), (3, 1500, "64,12,"), (2, 1700, "64,14,"),
                                       (2, 1280, "64,10,"), (2, 1900, "64,12,")])
def test_head_dim_64_rows_beyond_512_keys_in_wide_slabs(L1, L2, cut, dtype):
    """D=64 rows beyond 512 keys are cut into two to five slabs of 320, 384 or 448 keys (10, 12 or 14 tiles of
    bias per wave) where such a cut exists; here with a masked tail (the length is not a multiple of the
    slab), a key mask, both element types, forward and backward (whose tiles cover a length of their own)."""
    import fta_lib
    assert fta_lib.describe_plan(1, 2, L1, L2, 64)["fwd"]["kernel"].startswith(f"fta_fwd_kernel<{cut}")
    q, k, v, b, do = _inputs(1, 2, L1, L2, 64, 41, dtype)
    b[..., L2 // 2:L2 // 2 + 70] = float("-inf")
    _compare(_run(q, k, v, b, 0.125, do), _oracle(q, k, v, b, 0.125, do), dtype, f"D64 L{L2} {dtype}")


@pytest.mark.parametrize("sm", [0.34, 0.36])
def test_bf16_either_side_of_the_scale_that_selects_the_backward_kernels(sm):
    """sm_scale * log2(e) <= 0.5 runs the plain hand-scheduled backward for bf16; beyond it the rounding
    of the scaled Q/K to 8 bits would show, and D=32 runs the instances that keep the product as a
    (hi, lo) pair of bf16 values (D=64: the instances that apply the scale in fp32)."""
    q, k, v, b, do = _inputs(1, 2, 16, 384, 32, 35, torch.bfloat16)
    _compare(_run(q, k, v, b, sm, do), _oracle(q, k, v, b, sm, do), torch.bfloat16, f"bf16 L384 sm={sm}")


@pytest.mark.parametrize("L1,L2,D", [(12, 1152, 32), (5, 300, 32), (9, 256, 32), (6, 512, 64)])
def test_bf16_large_scale_keeps_the_accuracy_of_a_small_one(L1, L2, D):
    """sm_scale = 1.3 (upstream's benchmark scale, flash_tt_attn.py:783) against 1/sqrt(D) on the same
    inputs: the gradients of the large scale are no further from the oracle than 2x those of the small
    one (with the scaled operands rounded to 8 bits once, dQ and dK were 4x off).  1152 takes three ranges of
    384 in the (hi, lo) instances (their other range sizes: test_backward_tiles_in_steps_of_64), 300 a masked tail."""
    print(f"case bf16 scales L1={L1} L2={L2} D={D}", flush=True)
    q, k, v, b, do = _inputs(1, 2, L1, L2, D, 36, torch.bfloat16)
    errs = {}
    for sm in (1.0 / math.sqrt(D), 1.3):
        got, ref = _run(q, k, v, b, sm, do), _oracle(q, k, v, b, sm, do)
        _compare(got, ref, torch.bfloat16, f"bf16 L{L2} D{D} sm={sm:.3f}")
        errs[sm] = {n: orc.rel_l2(got[n], ref[n]) for n in ("dq", "dk", "dv", "db")}
        print("   ", {n: f"{e:.2e}" for n, e in errs[sm].items()}, flush=True)
    for n, e in errs[1.3].items():
        assert e <= 2.0 * errs[1.0 / math.sqrt(D)][n], f"{n}: {e:.2e} at 1.3"


def test_bf16_precise_mode_and_sum_over_key_ranges():
    """The precise switch routes bf16 to the vector-ALU instances; without it L2 = 1152 runs three ranges of 384 of the
    hand-scheduled kernels with the bf16 read-modify-write of dQ, dK, dV between launches (the other range sizes:
    test_backward_tiles_in_steps_of_64)."""
    import flash_tt_attn as fta
    sm = 1.0 / math.sqrt(32)
    q, k, v, b, do = _inputs(1, 2, 12, 1152, 32, 33, torch.bfloat16)
    ref = _oracle(q, k, v, b, sm, do)
    _compare(_run(q, k, v, b, sm, do), ref, torch.bfloat16, "bf16 L1152")
    fta.PRECISE_BACKWARD = True
    try:
        _compare(_run(q, k, v, b, sm, do), ref, torch.bfloat16, "bf16 L1152 precise")
    finally:
        fta.PRECISE_BACKWARD = False


def test_bf16_fp32_dbias_through_the_c_abi():
    """fta_bwd_ex with dbias_f32: the bias gradient comes out unrounded (fp32), the bf16 one is its
    rounding; everything else is unchanged."""
    import fta_lib
    lib = fta_lib.load()
    B, H, L1, L2, D, sm = 1, 2, 17, 256, 32, 0.25
    q, k, v, b, do = _inputs(B, H, L1, L2, D, 4, torch.bfloat16)
    t5 = lambda t: fta_lib.t5(t.data_ptr(), t.stride())
    t4 = lambda t: fta_lib.t4(t.data_ptr(), t.stride())
    o = torch.empty_like(q)
    lse = torch.empty(B, H, L1, L2, device=DEV, dtype=torch.float32)
    res = {}
    for f32 in (0, 1):
        opt = fta_lib.Options(fta_lib.DTYPE_BF16, f32, 0.0, 0)
        fta_lib.check(lib.fta_fwd_ex(t5(q), t5(k), t5(v), t4(b), t5(o), lse.data_ptr(), B, H, L1, L2, D, sm, ctypes.byref(opt), 0))
        dq, dk, dv = (torch.empty_like(t) for t in (q, k, v))
        db = torch.full((B, H, L2, L2), float("nan"), device=DEV, dtype=torch.float32 if f32 else torch.bfloat16)
        n = lib.fta_bwd_workspace_bytes_ex(B, H, L1, L2, D, ctypes.byref(opt))
        ws = torch.empty(n, dtype=torch.uint8, device=DEV)
        fta_lib.check(lib.fta_bwd_ex(t5(q), t5(k), t5(v), t4(b), t5(o), lse.data_ptr(), t5(do), t5(dq), t5(dk), t5(dv), t4(db),
                                     ws.data_ptr(), n, B, H, L1, L2, D, sm, ctypes.byref(opt), 0))
        torch.cuda.synchronize()
        res[f32] = (dq, dk, dv, db)
    for a, c in zip(res[0][:3], res[1][:3]):
        assert torch.equal(a, c)
    assert res[1][3].dtype == torch.float32 and torch.equal(res[1][3].to(torch.bfloat16), res[0][3])
    ref = _oracle(q, k, v, b, sm, do)
    assert orc.rel_l2(res[1][3], ref["db"]) < orc.rel_l2(res[0][3], ref["db"]) + 1e-6 <= 2e-2
    # option errors are argument errors
    bad = fta_lib.Options(7, 0, 0.0, 0)
    assert lib.fta_fwd_ex(t5(q), t5(k), t5(v), t4(b), t5(o), lse.data_ptr(), B, H, L1, L2, D, sm, ctypes.byref(bad), 0) == -11
    bad = fta_lib.Options(0, 0, 1.0, 0)
    assert lib.fta_fwd_ex(t5(q), t5(k), t5(v), t4(b), t5(o), lse.data_ptr(), B, H, L1, L2, D, sm, ctypes.byref(bad), 0) == -12


# ---- dropout --------------------------------------------------------------------------------------------

def _device_mask(p, seed, B, H, L1, L2):
    import fta_lib
    lib = fta_lib.load()
    opt = fta_lib.Options(0, 0, p, seed)
    m = torch.empty(B, H, L1, L2, L2, dtype=torch.uint8, device=DEV)
    fta_lib.check(lib.fta_dropout_mask(ctypes.byref(opt), B, H, L1, L2, m.data_ptr(), 0))
    torch.cuda.synchronize()
    return m


def test_dropout_mask_is_the_documented_function_of_seed_and_coordinates():
    for p, seed, shape in ((0.1, 1, (1, 2, 3, 64)), (0.5, 2**40 + 17, (2, 1, 5, 200)), (0.25, 0xFFFFFFFFFFFFFFFF, (1, 1, 2, 132)),
                           (0.3, 99, (1, 2, 3, 131)), (0.2, 5, (1, 1, 2, 1))):
        host, scale = dm.keep_mask(seed, p, *shape)
        dev = _device_mask(p, seed, *shape).cpu().numpy()
        assert np.array_equal(host, dev), (p, seed, shape)
        assert host.size < 10000 or abs(host.mean() - 1 / scale) < 0.02


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,L1,L2,D,p", [(1, 2, 9, 256, 32, 0.1), (1, 1, 5, 384, 64, 0.5), (1, 2, 7, 200, 32, 0.25),
                                           (2, 2, 4, 1024, 32, 0.15), (1, 1, 3, 900, 64, 0.3), (1, 2, 6, 201, 32, 0.2),
                                           (1, 1, 4, 387, 64, 0.1), (1, 1, 2, 1280, 64, 0.2), (1, 2, 2, 2048, 64, 0.1),
                                           (1, 1, 3, 1531, 64, 0.3)])
def test_dropout_against_the_oracle_with_the_same_mask(B, H, L1, L2, D, p, dtype):
    """attention(..., dropout_p, seed): forward and all four gradients against the oracle's masked
    closed forms, with the mask rebuilt on the host from (seed, coordinates) alone."""
    print(f"case dropout {dtype} B={B} H={H} L1={L1} L2={L2} D={D} p={p}", flush=True)
    sm, seed = 1.0 / math.sqrt(D), 1000 + L2
    q, k, v, b, do = _inputs(B, H, L1, L2, D, 21, dtype)
    keep, scale = dm.keep_mask(seed, p, B, H, L1, L2)
    keep = torch.from_numpy(keep).to(DEV)
    got = _run(q, k, v, b, sm, do, p, seed)
    _compare(got, _oracle(q, k, v, b, sm, do, keep=keep, keep_scale=scale), dtype, f"dropout L{L2} D{D} p{p}")
    again = _run(q, k, v, b, sm, do, p, seed)
    for n in got:
        assert torch.equal(got[n], again[n]), n
    other = _run(q, k, v, b, sm, do, p, seed + 1)
    assert not torch.equal(got["o"], other["o"])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L1,L2,p", [(4, 129, 0.1), (9, 192, 0.5), (5, 193, 0.75), (20, 300, 0.25), (3, 320, 0.9), (6, 321, 0.1), (5, 384, 0.6),
                                     (7, 385, 0.25), (3, 448, 0.5), (4, 449, 0.1), (2, 700, 0.25), (2, 768, 0.4)])
def test_dropout_at_the_tiled_lengths_of_head_dim_32(L1, L2, p, dtype):
    """The dropout instances at the edges of the lengths they tile a row as, at keep thresholds below 128 (of 256), at it
    and above, against the oracle with the mask rebuilt on the host."""
    B, H, sm = 1, 2, 0.6
    q, k, v, b, do = _inputs(B, H, L1, L2, 32, 31, dtype)
    keep, scale = dm.keep_mask(77 + L2, p, B, H, L1, L2)
    ref = _oracle(q, k, v, b, sm, do, keep=torch.from_numpy(keep).to(DEV), keep_scale=scale)
    got = _run(q, k, v, b, sm, do, p, 77 + L2)
    # (kept weights are 1/(1-p) times larger, and with them O and the rounding error of the weights (2^-10 of each in fp16,
    # 2^-9 in bf16) and of O: the absolute tolerance of O is for weights that sum to one, i.e. for (1-p) O)
    got["o"], ref["o"] = (got["o"].float() / scale).to(dtype), ref["o"] / scale
    _compare(got, ref, dtype, f"dropout {L1}x{L2} p{p}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L1,L2", [(61, 257), (8, 288), (33, 289), (17, 353), (64, 384), (9, 400), (40, 481), (7, 512)])
def test_dropout_backward_in_workgroups_of_four_waves(L1, L2, dtype):
    """257 to 512 keys: one query block (up to 384 keys; two in eight waves beyond) or two key blocks to a workgroup; groups that end in a block of one
    query, odd numbers of key blocks, chunks of one and of several rows (whose turns of priority are two rows long)."""
    import fta_lib
    B, H, p, sm = 2, 3, 0.15, 1.0 / math.sqrt(32)
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, p, 77, 0)
    plan = fta_lib.describe_plan(B, H, L1, L2, 32, sm, opt)
    assert plan["dkdv"]["block"] == 256 and plan["dq"]["block"] == (256 if L2 <= 384 else 512)
    print(f"case dropout four waves {L1}x{L2} {dtype}", flush=True)
    q, k, v, b, do = _inputs(B, H, L1, L2, 32, 53, dtype)
    keep, scale = dm.keep_mask(77, p, B, H, L1, L2)
    ref = _oracle(q, k, v, b, sm, do, keep=torch.from_numpy(keep).to(DEV), keep_scale=scale)
    _compare(_run(q, k, v, b, sm, do, p, 77), ref, dtype, f"dropout four waves {L1}x{L2}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L1,L2,launches,launches2", [(5, 513, 2, 2), (4, 640, 2, 2), (9, 768, 2, 1), (3, 801, 2, 2), (4, 1024, 2, 1), (3, 1100, 3, 3),
                                                      (3, 2011, 4, 2)])
def test_dropout_beyond_512_keys_in_ranges_of_their_own(L1, L2, launches, launches2, dtype):
    """Key and query ranges of 256, 384 and 512 in one row, each by eight waves, summed over their launches, or 768 and 1024
    queries to a launch where those are fewer; rows that end inside a range's last blocks."""
    import fta_lib
    B, H, p, sm = 1, 2, 0.2, 1.0 / math.sqrt(32)
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, p, 77, 0)
    plan = fta_lib.describe_plan(B, H, L1, L2, 32, sm, opt)
    assert plan["dq"]["launches"] == launches and plan["dkdv"]["launches"] == launches2
    assert plan["dq"]["block"] == plan["dkdv"]["block"] == 512
    print(f"case dropout ranges {L1}x{L2} {dtype}", flush=True)
    q, k, v, b, do = _inputs(B, H, L1, L2, 32, 47, dtype)
    keep, scale = dm.keep_mask(77, p, B, H, L1, L2)
    ref = _oracle(q, k, v, b, sm, do, keep=torch.from_numpy(keep).to(DEV), keep_scale=scale)
    _compare(_run(q, k, v, b, sm, do, p, 77), ref, dtype, f"dropout ranges {L1}x{L2}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("L1,L2,p", [(3, 2, 0.0), (5, 32, 0.0), (4, 33, 0.25), (6, 64, 0.1), (3, 65, 0.0), (7, 96, 0.25), (9, 97, 0.0), (40, 128, 0.1)])
def test_one_kernel_backward_of_short_rows(L1, L2, p, D, dtype):
    """Rows of up to 128 keys: all gradients in one kernel of one to four waves, with and without dropout, at the edges
    of its 32-key blocks."""
    import fta_lib
    assert fta_lib.describe_plan(1, 2, L1, L2, D)["dq"]["kernel"] == f"fta_bwd_short_kernel<{D},{(L2 + 31) // 32}>"
    B, H, sm = 1, 2, 1.0 / math.sqrt(D)
    q, k, v, b, do = _inputs(B, H, L1, L2, D, 29, dtype)
    extra, kw = (), {}
    if p:
        keep, scale = dm.keep_mask(1234, p, B, H, L1, L2)
        extra, kw = (p, 1234), dict(keep=torch.from_numpy(keep).to(DEV), keep_scale=scale)
    _compare(_run(q, k, v, b, sm, do, *extra), _oracle(q, k, v, b, sm, do, **kw), dtype, f"short {L1}x{L2}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L1,L2,p", [(1, 129, 0.0), (2, 160, 0.0), (5, 161, 0.0), (40, 192, 0.0), (300, 137, 0.0), (3, 150, 0.25), (7, 192, 0.1),
                                     (4, 193, 0.25), (33, 224, 0.1), (3, 225, 0.25), (70, 256, 0.1)])
def test_one_kernel_backward_of_rows_that_fill_a_compute_unit(L1, L2, p, dtype):
    """D = 32, 129 to 192 keys (with dropout 256): the one-kernel backward with five to eight waves, the bias packed in
    memory and the next row's tiles loaded ahead; at the edges of its 32-key blocks, with one and with several rows per
    workgroup, and with bias, q and dO as views of other strides.  Tolerances as for the shorter rows."""
    import fta_lib
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, p, 1234)
    assert fta_lib.describe_plan(1, 2, L1, L2, 32, 0.2, opt)["dq"]["kernel"] == f"fta_bwd_short_kernel<32,{(L2 + 31) // 32}>"
    B, H, sm = 1, 2, 0.2
    q, k, v, b, do = _inputs(B, H, L1, L2, 32, 31, dtype)
    extra, kw = (), {}
    if p:
        keep, scale = dm.keep_mask(1234, p, B, H, L1, L2)
        extra, kw = (p, 1234), dict(keep=torch.from_numpy(keep).to(DEV), keep_scale=scale)
    ref = _oracle(q, k, v, b, sm, do, **kw)
    _compare(_run(q, k, v, b, sm, do, *extra), ref, dtype, f"one kernel {L1}x{L2}")
    rows = lambda t: t.permute(0, 2, 3, 1, 4).contiguous().permute(0, 3, 1, 2, 4)  # (B, L1, L2, H, D) in memory
    wide = torch.zeros(B, H, L2, L2 + 3, device=DEV, dtype=dtype)[..., :L2].copy_(b)
    _compare(_run(rows(q), k, rows(v), wide, sm, rows(do), *extra), ref, dtype, f"one kernel {L1}x{L2}, strided")


def test_dropout_zero_is_the_plain_path_and_lse_ignores_the_mask():
    import fta_lib, flash_tt_attn as fta
    lib = fta_lib.load()
    B, H, L1, L2, D, sm = 1, 2, 8, 256, 32, 0.3
    q, k, v, b, do = _inputs(B, H, L1, L2, D, 8, torch.float16)
    plain = _run(q, k, v, b, sm, do)
    zero = _run(q, k, v, b, sm, do, 0.0, 99)
    for n in plain:
        assert torch.equal(plain[n], zero[n]), n
    # the saved logsumexp is that of the undropped softmax
    t5 = lambda t: fta_lib.t5(t.data_ptr(), t.stride())
    t4 = lambda t: fta_lib.t4(t.data_ptr(), t.stride())
    lse = [torch.empty(B, H, L1, L2, device=DEV, dtype=torch.float32) for _ in range(2)]
    o = torch.empty_like(q)
    for i, p in enumerate((0.0, 0.4)):
        opt = fta_lib.Options(0, 0, p, 5)
        fta_lib.check(lib.fta_fwd_ex(t5(q), t5(k), t5(v), t4(b), t5(o), lse[i].data_ptr(), B, H, L1, L2, D, sm, ctypes.byref(opt), 0))
    torch.cuda.synchronize()
    # (to the rounding of the row sum: without dropout it is taken over the weights as rounded toward
    # zero for the matrix core, 2^-12 low on average, with dropout over the unrounded ones)
    assert (lse[0] - lse[1]).abs().max().item() < 2e-3
    with pytest.raises(ValueError):
        fta.attention(q, k, v, b, sm, 1.0)


def test_dropout_without_a_seed_draws_one_and_lengths_beyond_what_is_built_raise_value_error():
    import flash_tt_attn as fta
    B, H, L1, L2, D, sm = 1, 2, 6, 256, 32, 0.3
    q, k, v, b, _ = _inputs(B, H, L1, L2, D, 9, torch.float16)
    # no seed: a fresh mask per call, reproducible through torch's generator
    torch.manual_seed(5)
    a1, a2 = fta.attention(q, k, v, b, sm, 0.3), fta.attention(q, k, v, b, sm, 0.3)
    torch.manual_seed(5)
    b1 = fta.attention(q, k, v, b, sm, 0.3)
    assert not torch.equal(a1, a2) and torch.equal(a1, b1)
    # and gradients flow with the drawn seed (the backward replays the same mask)
    qq = q.clone().requires_grad_(True)
    fta.attention(qq, k, v, b, sm, 0.3).float().sum().backward()
    assert bool(torch.isfinite(qq.grad.float()).all())
    # D = 64 rows end at 2048 keys, with dropout too: longer ones are refused before any launch, as a ValueError
    x = torch.zeros(1, 1, 1, 2052, 64, device=DEV, dtype=torch.float16)
    bias = torch.zeros(1, 1, 2052, 2052, device=DEV, dtype=torch.float16)
    with pytest.raises(ValueError, match="with these options"):
        fta.attention(x, x, x, bias, 0.1, 0.1, 3)


# ---- precise fp16 backward --------------------------------------------------------------------------------

@pytest.mark.parametrize("L1,L2,D", [(16, 512, 32), (7, 384, 32), (9, 256, 32), (5, 300, 32), (3, 1280, 32), (6, 203, 32),
                                     (6, 512, 64), (4, 128, 32)])
@pytest.mark.parametrize("bias_std,std,sm", [(30.0, 1.0, 1.0 / math.sqrt(32)), (1.0, 3.0, 1.3)])
def test_precise_backward_holds_the_tolerance_on_large_biases_and_scores(bias_std, std, sm, L1, L2, D):
    """Bias spread 30 or score spread ~60: the default backward kernels round log2(e)*bias and the
    scaled Q/K to fp16 on their way into the matrix core and leave the 1e-2 gradient bar there
    (documented); the precise mode does not and holds it: at D = 32 and rows beyond 192 keys through
    the hand-scheduled kernels' instances with the operand pair and the exponent in natural units (tails, one
    range and several), at 128 through the one-kernel backward (more of that one below), at D = 64 through the
    vector-ALU kernels."""
    import flash_tt_attn as fta
    B, H = 1, 2
    if D == 64:
        std, sm = (std, sm) if std == 1.0 else (2.5, 1.0)   # (the same score spread at the wider head)
    q, k, v, b, do = orc.make_inputs(B, H, L1, L2, D, seed=17, std=std, bias_std=bias_std, device=DEV)
    ref = _oracle(q, k, v, b, sm, do)
    default = _run(q, k, v, b, sm, do)
    fta.PRECISE_BACKWARD = True
    try:
        precise = _run(q, k, v, b, sm, do)
    finally:
        fta.PRECISE_BACKWARD = False
    e_def = {n: orc.rel_l2(default[n], ref[n]) for n in ("dq", "dk", "dv", "db")}
    e_pre = {n: orc.rel_l2(precise[n], ref[n]) for n in ("dq", "dk", "dv", "db")}
    print("default", e_def, "precise", e_pre, flush=True)
    assert torch.equal(default["o"], precise["o"])
    _compare(precise, ref, torch.float16, f"precise bias_std{bias_std} std{std}")
    assert max(e_pre.values()) < max(e_def.values())


@pytest.mark.parametrize("L1,L2", [(4, 97), (5, 131), (3, 160), (40, 192)])
def test_precise_instances_of_the_one_kernel_backward(L1, L2):
    """The one-kernel backward (here with four, five and six waves) keeps everything per score in fp32 either way; its
    precise instances round P and dS to nearest on their way into the matrix core instead of toward zero: dQ, dK and dV come
    closer, the bias gradient, summed unrounded, is the same."""
    import fta_lib
    import flash_tt_attn as fta
    B, H, sm = 1, 2, 1.0 / math.sqrt(32)
    opt = fta_lib.Options(fta_lib.DTYPE_F16, 0, 0.0, 0, 1)
    assert fta_lib.describe_plan(B, H, L1, L2, 32, sm, opt)["dq"]["kernel"] == f"fta_bwd_short_kernel<32,{(L2 + 31) // 32}>"
    q, k, v, b, do = orc.make_inputs(B, H, L1, L2, 32, seed=17, bias_std=30.0, device=DEV)
    ref, default = _oracle(q, k, v, b, sm, do), _run(q, k, v, b, sm, do)
    fta.PRECISE_BACKWARD = True
    try:
        precise = _run(q, k, v, b, sm, do)
    finally:
        fta.PRECISE_BACKWARD = False
    _compare(precise, ref, torch.float16, f"precise one kernel L{L2}")
    for n in ("dq", "dk", "dv"):
        assert orc.rel_l2(precise[n], ref[n]) < orc.rel_l2(default[n], ref[n]), n
    assert torch.equal(precise["db"], default["db"])


# ---- the hand-scheduled forward with an odd number of tiles per slab ----------------------------------------

@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L1,L2,tiled", [(9, 129, 160), (5, 160, 160), (40, 224, 224), (3, 257, 288), (6, 288, 288), (8, 351, 352), (3, 416, 416), (7, 457, 480),
                                         (3, 545, 576), (4, 576, 576), (5, 701, 704), (9, 704, 704), (3, 832, 832), (2, 950, 960),
                                         (3, 1100, 1152), (2, 1152, 1152), (2, 1408, 1408), (2, 1601, 1664)])
def test_forward_rows_of_an_odd_number_of_tiles(L1, L2, tiled, dtype):
    """Stages of one tile (two barriers in a row) and of three, one, two and four slabs, whole rows and rows that end inside
    a tile; the large scale takes the branch that raises a row's reference, in the tile that changes registers too."""
    import fta_lib
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, 0.0, 0, 0)
    plan = fta_lib.describe_plan(1, 2, L1, L2, 32, 1.0, opt)["fwd"]
    assert plan["kernel"].startswith("fta_fwd1_kernel") and plan["tiled_length"] == tiled
    for sm in (1.0 / math.sqrt(32), 1.3):
        print(f"case odd tiles {L1}x{L2} {dtype} sm={sm:.2f}", flush=True)
        q, k, v, b, do = _inputs(1, 2, L1, L2, 32, 43, dtype)
        _compare(_run(q, k, v, b, sm, do), _oracle(q, k, v, b, sm, do), dtype, f"odd tiles {L1}x{L2}")


# ---- the hand-scheduled backward at tiled lengths in steps of 64 -------------------------------------------

@pytest.mark.parametrize("mode", ["fp16", "bf16", "bf16 operand pair", "precise"])
@pytest.mark.parametrize("D,L2", [(32, L) for L in (193, 256, 257, 320, 385, 448, 449, 513, 640, 703, 896, 1024, 1088)]
                         + [(64, L) for L in (129, 192, 257, 320, 400, 576, 640, 701, 832)])
def test_backward_tiles_in_steps_of_64(D, L2, mode):
    """Every number of tiles per wave (key ranges of 256 to 512 keys in two slabs, first and later ones: 513, 640, 703, 896
    and 1024 have later ranges of 256, 320, 384 (1088), 448 and 512; of 256 in one; D = 64: 160 to 256 in one slab up to 384 keys, 256, 384 and 512 in
    two beyond; query ranges of 256 to 512, at D = 64 without 448), odd numbers of them (stages of unequal length), groups of 128 queries or keys
    that end beyond the tiled length, one to three ranges; rows that end inside a tile and whole ones."""
    import fta_lib
    import flash_tt_attn as fta
    if D == 64 and mode in ("bf16 operand pair", "precise"):
        pytest.skip("no such instances at head dim 64")
    dtype = torch.bfloat16 if mode.startswith("bf16") else torch.float16
    B, H, L1, sm = 1, 2, 5, 1.3 if mode == "bf16 operand pair" else 1.0 / math.sqrt(D)
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, 0.0, 0, 1 if mode == "precise" else 0)
    plan = fta_lib.describe_plan(B, H, L1, L2, D, sm, opt)
    assert "dq1" in plan["dq"]["kernel"] and "dkdv1" in plan["dkdv"]["kernel"]
    print(f"case {mode} D={D} L2={L2}", flush=True)
    q, k, v, b, do = _inputs(B, H, L1, L2, D, 41, dtype)
    fta.PRECISE_BACKWARD = mode == "precise"
    try:
        got = _run(q, k, v, b, sm, do)
    finally:
        fta.PRECISE_BACKWARD = False
    _compare(got, _oracle(q, k, v, b, sm, do), dtype, f"tiles of 64 {mode} D{D} L{L2}")


@pytest.mark.parametrize("mode", ["fp16", "bf16", "bf16 operand pair", "precise"])
@pytest.mark.parametrize("L1,L2,launches", [(41, 257, 1), (40, 384, 1), (20, 576, 2), (19, 640, 2), (21, 703, 2), (20, 768, 2)])
def test_dq_at_head_dim_32_in_two_slabs_over_several_rows_and_chunks(L1, L2, launches, mode):
    """dQ/dBias at D = 32 of four, five and six tiles a slab, where a wave reads its partner's share of a row behind the last barrier of the
    next one: first and later ranges, several chunks of several rows each.  Every run gives the same bits."""
    import fta_lib
    import flash_tt_attn as fta
    dtype = torch.bfloat16 if mode.startswith("bf16") else torch.float16
    B, H, sm = 1, 2, 1.3 if mode == "bf16 operand pair" else 1.0 / math.sqrt(32)
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, 0.0, 0, 1 if mode == "precise" else 0)
    plan = fta_lib.describe_plan(B, H, L1, L2, 32, sm, opt)["dq"]
    assert plan["kernel"].startswith("fta_bwd_dq1_kernel<32,2>") and plan["launches"] == launches
    assert plan["grid"] >= 2 * H * ((L2 + 63) // 64)   # (two chunks or more)
    print(f"case two slabs {mode} D=32 {L1}x{L2}", flush=True)
    q, k, v, b, do = _inputs(B, H, L1, L2, 32, 47, dtype)
    fta.PRECISE_BACKWARD = mode == "precise"
    try:
        got, again = _run(q, k, v, b, sm, do), _run(q, k, v, b, sm, do)
    finally:
        fta.PRECISE_BACKWARD = False
    _compare(got, _oracle(q, k, v, b, sm, do), dtype, f"two slabs {mode} D32 {L1}x{L2}")
    for n in got:
        assert torch.equal(got[n], again[n]), n


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L2", [160, 161, 255, 288, 289, 353, 384, 1153, 1281, 1408, 1700, 415, 449, 545, 641, 1025])
def test_dq_at_head_dim_64_tiles_to_the_next_32_keys(L2, dtype):
    """dQ/dBias at D = 64 in one slab ends its key tiles at the next multiple of 32, dK/dV at its own length: one tile more or less
    than a whole range, whole rows of an odd number of tiles, the two ranges of 160 below 288, uneven ranges (five to seven from 1153 keys
    on), and a last group of 128 queries that only dK/dV reads to its end.  In two slabs (385 to 1152 keys among these) the tiles end at the
    next multiple of 128.  Chunks of fewer rows than eight at L1 = 5."""
    import fta_lib
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, 0.0, 0, 0)
    kernel = fta_lib.describe_plan(1, 2, 5, L2, 64, 0.125, opt)["dq"]["kernel"]
    assert kernel.startswith("fta_bwd_dq1w_kernel" if 384 < L2 <= 1152 else "fta_bwd_dq1_kernel<64,1>")
    print(f"case dq tiles D=64 L2={L2} {dtype}", flush=True)
    q, k, v, b, do = _inputs(1, 2, 5, L2, 64, 44, dtype)
    _compare(_run(q, k, v, b, 0.125, do), _oracle(q, k, v, b, 0.125, do), dtype, f"dq tiles D64 L{L2}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout", ["contiguous", "projection", "ending"])
@pytest.mark.parametrize("L1,L2", [(20, 577), (17, 513), (19, 640), (20, 700)])
def test_dq_at_head_dim_64_later_ranges_over_several_rows_and_chunks(L1, L2, layout, dtype):
    """dQ/dBias at D = 64 of two ranges, 384 + 256 keys (four tiles a slab in the later one: a wave reads its partner's share of a row in the
    row's last iteration) and 384 + 384: three chunks of several rows each, in every layout that the projections leave; plain, and with the
    whole later range or its first slab masked.  Every run gives the same bits."""
    import fta_lib
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, 0.0, 0, 0)
    plan = fta_lib.describe_plan(1, 2, L1, L2, 64, 0.125, opt)["dq"]
    assert plan["kernel"].startswith("fta_bwd_dq1w_kernel") and plan["launches"] == 2
    assert plan["grid"] >= 2 * 2 * ((L2 + 63) // 64)   # (two chunks or more)
    order = {"contiguous": (0, 1, 2, 3, 4), "projection": (0, 2, 3, 1, 4), "ending": (0, 1, 3, 2, 4)}[layout]
    q, k, v, b, do = _inputs(1, 2, L1, L2, 64, 46, dtype)
    q, k, v, do = (t.permute(order).contiguous().permute([order.index(d) for d in range(5)]) for t in (q, k, v, do))
    assert layout == "contiguous" or not q.is_contiguous()
    for masked in ((0, 0), (384, L2), (384, 512)):
        print(f"case later ranges D=64 {L1}x{L2} {layout} {dtype} masked {masked}", flush=True)
        bm = b.clone()
        bm[..., masked[0]:masked[1]] = -math.inf
        got, again = _run(q, k, v, bm, 0.125, do), _run(q, k, v, bm, 0.125, do)
        _compare(got, _oracle(q, k, v, bm, 0.125, do), dtype, f"later ranges D64 {L1}x{L2} {layout} masked {masked}")
        for n in got:
            assert torch.equal(got[n], again[n]), n


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L1,L2", [(7, 129), (3, 160), (4, 161), (1, 191), (9, 192)])
def test_forward_at_head_dim_64_of_129_to_192_keys(L1, L2, dtype):
    """One slab of six tiles: two of the eight query blocks beyond the row, whole rows, one key more than a tile; one row,
    and chunks of unequal numbers of rows.  The keys of the first and of the last tile masked out by the bias."""
    import fta_lib
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, 0.0, 0, 0)
    plan = fta_lib.describe_plan(2, 2, L1, L2, 64, 0.125, opt)["fwd"]
    assert plan["kernel"].startswith("fta_fwd2_kernel") and plan["tiled_length"] == 192
    for masked in ((0, 0), (0, 32), (L2 - 32, L2)):
        print(f"case D=64 {L1}x{L2} {dtype} masked {masked}", flush=True)
        q, k, v, b, do = _inputs(2, 2, L1, L2, 64, 45, dtype)
        b[..., masked[0]:masked[1]] = -1e4
        _compare(_run(q, k, v, b, 0.125, do), _oracle(q, k, v, b, 0.125, do), dtype, f"D64 L{L2} masked {masked}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("L1,L2,tiled", [(3, 3, 64), (5, 7, 64), (2, 8, 64), (9, 33, 64), (5, 64, 64), (6, 65, 96), (1, 95, 96), (7, 96, 96),
                                         (3, 97, 128)])
def test_forward_at_head_dim_64_of_up_to_96_keys(L1, L2, tiled, dtype):
    """One slab of two or three tiles, a stage a row: rows shorter than a piece of the bias, ends inside a tile and on one,
    one row and odd numbers of rows (the buffers change places from row to row).  (Of a row of one key dQ, dK and dBias
    are 0 whatever the inputs, and a relative error has no meaning: three keys are the shortest here.)"""
    import fta_lib
    opt = fta_lib.Options(fta_lib.DTYPE_BF16 if dtype == torch.bfloat16 else fta_lib.DTYPE_F16, 0, 0.0, 0, 0)
    plan = fta_lib.describe_plan(2, 3, L1, L2, 64, 0.125, opt)["fwd"]
    assert plan["tiled_length"] == tiled
    print(f"case D=64 {L1}x{L2} {dtype}", flush=True)
    q, k, v, b, do = _inputs(2, 3, L1, L2, 64, 46, dtype)
    _compare(_run(q, k, v, b, 0.125, do), _oracle(q, k, v, b, 0.125, do), dtype, f"D64 L{L2} {dtype}")


# ---- magnitudes of bf16 gradients -------------------------------------------------------------------------

def _check_gradients_scale_with_dout(q, k, v, b, sm, do, *extra):
    """The gradients are linear in dO, and bf16 has the exponents of fp32: dO times a power of two scales every product and sum
    exactly, so the gradients are the same bits but for their exponent (a mean over a long pair tensor leaves some of 1e-8, and less).
    Weights near 2^-126 times a small dO vanish: less than 2^-126 of each of L2 products with factors of up to 2^6."""
    want = _run(q, k, v, b, sm, do, *extra)
    for e in (-40, -24, 20, 40):
        got = _run(q, k, v, b, sm, do * 2.0 ** e, *extra)
        for n in ("dq", "dk", "dv", "db"):
            off = (got[n].double() - want[n].double() * 2.0 ** e).abs().max().item()
            assert off <= k.shape[3] * 2.0 ** -120, f"{n} at 2^{e}: {orc.rel_l2(got[n].double() * 2.0 ** -e, want[n].double()):.2e}"


@pytest.mark.parametrize("D,L2,sm,p", [
    (32, 300, 0.17, 0.15), (32, 384, 0.17, 0.15), (32, 450, 1.3, 0.15), (32, 600, 0.17, 0.15), (32, 768, 0.17, 0.15), (32, 1000, 0.17, 0.15),
    (32, 1408, 0.17, 0.15), (64, 100, 0.17, 0.15), (64, 150, 0.17, 0.15), (64, 300, 0.17, 0.15), (64, 512, 0.17, 0.15), (64, 600, 0.17, 0.15),
    (64, 200, 1.3, 0.0), (64, 384, 1.3, 0.0), (64, 500, 1.3, 0.0), (64, 1024, 1.3, 0.0)])
def test_bf16_gradients_of_any_magnitude_from_the_general_kernels(D, L2, sm, p):
    """Shares of dQ, dK and dV that slabs hand to each other, in every number of slabs."""
    print(f"case magnitudes D={D} L2={L2} sm={sm} p={p}", flush=True)
    q, k, v, b, do = _inputs(1, 2, 3, L2, D, 61, torch.bfloat16)
    _check_gradients_scale_with_dout(q, k, v, b, sm, do, *((p, 7) if p else ()))


@pytest.mark.parametrize("D,L2", [(32, 384), (32, 512), (32, 640), (32, 1024), (64, 256), (64, 384), (64, 512)])
def test_bf16_gradients_of_any_magnitude_from_the_general_kernels_at_every_scale(D, L2):
    import fta_lib
    lib = fta_lib.load()
    print(f"case magnitudes D={D} L2={L2} general", flush=True)
    q, k, v, b, do = _inputs(1, 2, 3, L2, D, 62, torch.bfloat16)
    before = lib.fta_debug_select_kernels(3)
    try:
        _check_gradients_scale_with_dout(q, k, v, b, 0.17, do)
    finally:
        lib.fta_debug_select_kernels(before)


@pytest.mark.parametrize("D,L2,sm", [(32, 200, 0.17), (32, 256, 1.3), (32, 383, 0.17), (32, 512, 0.17), (32, 512, 1.3), (32, 700, 0.17), (32, 1100, 1.3),
                                     (64, 150, 0.17), (64, 256, 0.17), (64, 401, 0.17), (64, 1024, 0.17)])
def test_bf16_gradients_of_any_magnitude_from_the_hand_scheduled_kernels(D, L2, sm):
    """Delta, which the matrix core adds as a pair of 16-bit values."""
    import fta_lib
    assert "dq1" in fta_lib.describe_plan(1, 2, 3, L2, D, sm, fta_lib.Options(fta_lib.DTYPE_BF16, 0, 0.0, 0, 0))["dq"]["kernel"]
    print(f"case magnitudes D={D} L2={L2} sm={sm}", flush=True)
    q, k, v, b, do = _inputs(1, 2, 3, L2, D, 63, torch.bfloat16)
    _check_gradients_scale_with_dout(q, k, v, b, sm, do)


# ---- everything at once, drawn at random -------------------------------------------------------------------

def test_random_draws_over_types_masks_dropout_modes_and_layouts():
    """120 seeded draws over head dim, type, shape (ragged lengths included), softmax scale (both sides
    of the bf16 kernel choice), bias spread, key masks (-inf or -1e9; leading, trailing, inner, whole
    128-key slabs, scattered), dropout, the precise mode, permuted q/k/v/dO and a bias that is a window
    of a larger tensor.  At least eight keys stay unmasked: with one left the softmax is one-hot and
    every gradient but dV is zero, so a relative error says nothing."""
    import random
    import flash_tt_attn as fta
    rng = random.Random(2024)
    for it in range(120):
        D = rng.choice([32, 32, 64])
        dtype = rng.choice([torch.float16, torch.bfloat16])
        B, H, L1 = rng.choice([1, 2]), rng.choice([1, 2, 3]), rng.randint(1, 10)
        Lmax = 1300 if D == 32 else 1600
        L2 = rng.choice([rng.randint(3, Lmax // 4) * 4, rng.choice([128, 256, 384, 512, 640, 768, 896, 1024]), rng.randint(12, Lmax)])
        sm = rng.choice([1 / math.sqrt(D), rng.uniform(0.05, 0.6), rng.uniform(0.6, 1.3)])
        bias_std = rng.choice([0.5, 1.0, 3.0])
        drop = rng.choice([0, 0, 0, rng.uniform(0.05, 0.6)])
        precise = rng.random() < 0.2
        seed = rng.getrandbits(64)
        kind = rng.choice(["none", "tail", "head", "mid", "slab", "scatter"])
        value = float("-inf") if (dtype == torch.float16 or rng.random() < 0.5) else -1e9
        q, k, v, b, do = orc.make_inputs(B, H, L1, L2, D, seed=3000 + it, std=1.0 if sm < 0.6 else 0.5,
                                         bias_std=bias_std, dtype=dtype, device=DEV)
        masked = torch.zeros(L2, dtype=torch.bool)
        if kind == "tail":
            masked[L2 - rng.randint(1, min(L2 - 8, 140)):] = True
        elif kind == "head":
            masked[:rng.randint(1, min(L2 - 8, 300))] = True
        elif kind == "mid":
            lo = rng.randint(1, L2 - 9)
            masked[lo:rng.randint(lo + 1, L2 - 8)] = True
        elif kind == "slab" and L2 > 256:
            lo = rng.randint(0, L2 // 128 - 1) * 128
            masked[lo:lo + rng.choice([128, 256, 384])] = True
        elif kind == "scatter":
            masked = torch.rand(L2, generator=torch.Generator().manual_seed(it)) < 0.3
        if int((~masked).sum()) < 8:
            masked[:] = False
        b[..., masked.to(DEV)] = value
        if rng.random() < 0.5:   # (B, H, L2, L1, D) storage seen through a transpose
            q, k, v, do = (t.transpose(2, 3).contiguous().transpose(2, 3) for t in (q, k, v, do))
        if rng.random() < 0.5:   # a window of a larger bias tensor (row stride not L2, offset start)
            big = torch.zeros(B, H, L2 + 3, L2 + 8, dtype=dtype, device=DEV)
            big[:, :, 1:L2 + 1, 8:L2 + 8] = b
            b = big[:, :, 1:L2 + 1, 8:L2 + 8]
        tag = (f"draw {it}: D{D} {dtype} B{B} H{H} L1={L1} L2={L2} sm={sm:.3f} bias_std={bias_std} drop={drop:.2f} "
               f"precise={precise} mask={kind}:{int(masked.sum())}={value}")
        print(tag, flush=True)
        kw, keep_scale = {}, 1.0
        if drop:
            keep, keep_scale = dm.keep_mask(seed, drop, B, H, L1, L2)
            kw = dict(keep=torch.from_numpy(keep).to(DEV), keep_scale=keep_scale)
        fta.PRECISE_BACKWARD = precise
        try:
            got = _run(q, k, v, b, sm, do, *((drop, seed) if drop else ()))
        finally:
            fta.PRECISE_BACKWARD = False
        ref = _oracle(q, k, v, b, sm, do, **kw)
        # (dropout scales the kept weights, and with them O and its rounding to the stored type, by 1/(1-p))
        o_tol, g_tol = TOL[dtype]
        err = (got["o"].float() - ref["o"]).abs().max().item()
        assert err <= o_tol * keep_scale, f"{tag}: O max-abs {err}"
        for n in ("dq", "dk", "dv", "db"):
            assert torch.isfinite(got[n].float()).all(), f"{tag}: {n}"
            e = orc.rel_l2(got[n], ref[n])
            assert e <= g_tol, f"{tag}: {n} rel-L2 {e}"
