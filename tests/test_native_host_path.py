"""What the C++ host path has to leave to the Python path, and what attention() and the block then do there (also
where the module is missing or was built for another torch): a call whose
operations something watches (tracing, dispatch and function modes, functorch), tensors with a tangent,
tensor subclasses, sizes that are not built, submodules that are not as the block made them.  And what the
backward of both paths is handed: gradients and saved tensors in any layout, or as others than they were."""
import pytest
import torch
import torch.autograd.forward_ad as fwad

from oracle import tt_attn_oracle as orc

gpu = pytest.mark.gpu
DEV = "cuda:0"


def _operands(seed, L2=96):
    return orc.make_inputs(1, 2, 5, L2, 32, seed=seed, device=DEV)


def _block(C=64, D=32, H=2, **kw):
    from triangle_attention import TriangleAttention
    torch.manual_seed(1)
    return TriangleAttention(C, D, H, **kw).to(DEV)


def _separate(blk):
    """The same block as separate layers around attention(): a subclass does not take the fused kernels."""
    from triangle_attention import TriangleAttention
    return type("Separate", (TriangleAttention,), {})(blk.c_z, blk.c_hidden, blk.n_heads, blk.starting, blk.dropout_p).to(DEV)


def _pair(seed, L=48, C=64):
    return torch.randn(1, L, L, C, device=DEV, generator=torch.Generator(DEV).manual_seed(seed))


@gpu
@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
def test_a_traced_call_runs_the_kernels_on_replay():
    """The trace is replayed on other inputs than it was recorded on, twice, so that no buffer can hold the answer."""
    from flash_tt_attn import attention
    blk = _block().eval()
    with torch.no_grad():
        op = torch.jit.trace(lambda q, k, v, b: attention(q, k, v, b, 0.3), _operands(1)[:4], check_trace=False)
        mod = torch.jit.trace(blk, (_pair(1),), check_trace=False)
        for seed in (2, 3):
            x, z = _operands(seed)[:4], _pair(seed)
            assert torch.equal(op(*x), attention(*x, 0.3))
            # (the fused block against separate layers: fp32 with the attention in fp16, as in the block's own tests)
            assert orc.rel_l2(mod(z), blk(z)) <= 1e-3


@gpu
def test_a_dispatch_mode_sees_the_operations_of_the_block():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))
    blk, z, seen = _block(), _pair(1), []
    with Log(), torch.no_grad():
        blk(z)
    assert any("native_layer_norm" in str(f) for f in seen)


@gpu
def test_functorch_transforms_are_refused_also_where_they_only_enclose_the_call():
    from flash_tt_attn import attention
    x = _operands(1)[:4]
    with pytest.raises(RuntimeError, match="functorch"):
        torch.vmap(lambda t: t.sum() + attention(*x, 0.3).sum())(torch.ones(3, 2, device=DEV))


@gpu
@pytest.mark.parametrize("which", ["q", "k", "v", "bias", "z", "weight"])
@pytest.mark.parametrize("grad", [False, True])
def test_forward_mode_derivatives_are_refused_not_dropped(which, grad):
    from flash_tt_attn import attention
    dual = lambda t: fwad.make_dual(t.detach(), torch.ones_like(t))
    x, blk, z = list(_operands(1)[:4]), _block().requires_grad_(False), _pair(1)
    with fwad.dual_level(), torch.set_grad_enabled(grad), pytest.raises(NotImplementedError, match="jvp"):
        if which in ("z", "weight"):
            if which == "weight":
                blk.linear_v._parameters["weight"] = dual(blk.linear_v.weight)
            blk(dual(z) if which == "z" else z)
        else:
            n = ("q", "k", "v", "bias").index(which)
            x[n] = dual(x[n])
            if grad:
                x[n - 1].requires_grad_(True)
            attention(*x, 0.3)


@gpu
def test_tensor_subclasses_keep_their_type():
    from flash_tt_attn import attention

    class Sub(torch.Tensor):
        pass
    x, blk, z = list(_operands(1)[:4]), _block(), _pair(1)
    got, plain = attention(x[0].as_subclass(Sub), *x[1:], 0.3), attention(*x, 0.3)
    assert type(got) is Sub and type(plain) is torch.Tensor and torch.equal(got.as_subclass(torch.Tensor), plain)
    assert type(blk(z.as_subclass(Sub))) is Sub
    assert type(attention(torch.nn.Parameter(x[0]), *x[1:], 0.3)) is torch.Tensor


@gpu
@pytest.mark.parametrize("C,D,H", [(64, 16, 4), (64, 16, 8), (128, 128, 1)])
def test_a_refused_head_dim_leaves_other_calls_of_its_length_alone(C, D, H):
    z = _pair(1, 71 + H, C)  # (a length no other test asks for)
    with pytest.raises(ValueError, match="not built"):
        _block(C, D, H)(z)
    z = z[..., :64].contiguous()
    assert _block()._fused(z, None, None) is not None


def test_a_dropout_probability_that_rounds_to_one_is_refused_as_such():
    """(not as a length that is not built, which would be kept for the length)"""
    import flash_tt_attn as fta
    x = torch.zeros(1, 1, 1, 8, 32, dtype=torch.float16)
    for p in (1.0, 1.0 - 1e-9, float("nan"), -0.1):
        with pytest.raises(ValueError, match="dropout_p"):
            fta.attention(x, x, x, torch.zeros(1, 1, 8, 8, dtype=torch.float16), 0.1, p, 3)


@gpu
@pytest.mark.parametrize("autocast", [False, True])
def test_a_call_draws_one_dropout_seed_whichever_path_takes_it(autocast):
    """The generator ends where one draw leaves it, and the mask is that draw's, on the fused path and on the separate
    layers (which the fused path leaves an autocast call to)."""
    z, blk = _pair(1), _block(dropout_p=0.25)
    sep = _separate(blk)
    sep.load_state_dict(blk.state_dict())
    outs, states = [], []
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        for m in (blk, sep):
            torch.manual_seed(5)
            outs.append(m(z).float())
            states.append(torch.get_rng_state())
    torch.manual_seed(5)
    torch.randint(0, 2 ** 62, (1,))
    assert all(torch.equal(s, torch.get_rng_state()) for s in states)
    assert (blk._fused(z, None, 7) is not None) and orc.rel_l2(*outs) <= 1e-3


def _own_forward(blk):
    lin = blk.linear_v
    lin.forward = lambda x: 2.0 * torch.nn.functional.linear(x, lin.weight)


def _plain_bias(blk):
    for lin in (blk.linear_g, blk.linear_o):
        value = lin.bias.detach() + 1.0
        del lin.bias
        lin.bias = value


def _bias_of_a_projection(blk):
    lin = blk.linear_q
    del lin.bias
    lin.bias = torch.ones(lin.out_features, device=DEV)


def _plain_weight(blk):
    lin = blk.linear_b
    value = 2.0 * lin.weight.detach()
    del lin.weight
    lin.weight = value


def _buffer_bias(blk):
    value = blk.linear_g.bias.detach() + 1.0
    del blk.linear_g.bias
    blk.linear_g.register_buffer("bias", value)


@gpu
@pytest.mark.parametrize("change", [_own_forward, _plain_bias, _bias_of_a_projection, _plain_weight, _buffer_bias])
def test_changed_submodules_are_used_as_they_are(change):
    blk, z = _block(), _pair(1)
    sep = _separate(blk)
    sep.load_state_dict(blk.state_dict())
    with torch.no_grad():
        before = blk(z)
        change(blk)
        change(sep)
        assert torch.equal(blk(z), sep(z)) and orc.rel_l2(blk(z), before) > 1e-2


def _native_file(kind, tmp_path):
    import fta_lib
    path = tmp_path / "fta_native.so"
    if kind == "other torch":
        data = open(fta_lib.NATIVE_PATH, "rb").read()
        assert data.count(fta_lib._BUILT_FOR + torch.__version__.encode()) == 1
        path.write_bytes(data.replace(fta_lib._BUILT_FOR, fta_lib._BUILT_FOR + b"9."))
    elif kind == "not a library":
        path.write_bytes(fta_lib._BUILT_FOR + torch.__version__.encode() + b"\0")
    return str(path)


@pytest.fixture(params=["missing", "other torch", "not a library"])
def no_native(request, tmp_path, monkeypatch):
    import fta_lib
    import flash_tt_attn
    monkeypatch.setattr(fta_lib, "NATIVE_PATH", _native_file(request.param, tmp_path))
    monkeypatch.setattr(fta_lib, "_native", None)
    monkeypatch.setattr(flash_tt_attn, "_native", None)
    with pytest.warns(RuntimeWarning, match="Python path"):
        assert fta_lib.native() is None


def test_without_the_module_calls_take_the_python_path(no_native):
    import warnings
    import flash_tt_attn as fta
    x = torch.zeros(1, 1, 1, 8, 32, dtype=torch.float16)
    with warnings.catch_warnings():
        warnings.simplefilter("error")  # (said once)
        with pytest.raises(ValueError, match="no CPU path"):
            fta.attention(x, x, x, torch.zeros(1, 1, 8, 8, dtype=torch.float16), 0.1)


@gpu
def test_without_the_module_the_results_are_the_same(no_native, monkeypatch):
    import fta_lib
    import flash_tt_attn as fta
    x, dout, blk, z = _operands(1)[:4], _operands(1)[4], _block(), _pair(1)

    def results():
        q = x[0].clone().requires_grad_(True)
        o = fta.attention(q, *x[1:], 0.3)
        return o, *torch.autograd.grad(o, q, dout), blk(z)
    slow = results()
    monkeypatch.undo()
    assert fta_lib.native() is not None
    fast = results()
    assert all(torch.equal(a, b) for a, b in zip(slow[:2], fast[:2])) and orc.rel_l2(slow[2], fast[2]) <= 1e-3


def test_the_build_follows_the_torch_at_hand(monkeypatch):
    import importlib.util
    import os
    import fta_lib
    spec = importlib.util.spec_from_file_location("fta_build", os.path.join(fta_lib.HERE, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    assert fta_lib.native_torch_version(build.NATIVE) == torch.__version__
    before = build.needs_build()
    monkeypatch.setattr(build, "torch_version", lambda: "9.9")
    assert build.needs_build()  # the module there is for another one
    monkeypatch.setattr(build, "torch_version", lambda: None)
    assert build.native_commands("hipcc", "x.o") is None
    monkeypatch.setattr(build, "NATIVE", "/nowhere/fta_native.so")
    assert build.needs_build() <= before  # without torch its absence is no reason to build


@gpu
def test_the_backward_outlives_the_module_it_came_from():
    import gc
    import importlib.util
    import os
    import fta_lib
    import flash_tt_attn
    q, k, v, b, dout = _operands(1)
    q.requires_grad_(True)
    spec = importlib.util.spec_from_file_location("fta_module_to_drop", os.path.join(fta_lib.HERE, "flash_tt_attn.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    o = mod.attention(q, k, v, b, 0.3)
    del mod, spec
    gc.collect()
    got, = torch.autograd.grad(o, q, dout)
    assert torch.equal(got, torch.autograd.grad(flash_tt_attn.attention(q, k, v, b, 0.3), q, dout)[0])


@gpu
@pytest.mark.parametrize("grad", [False, True])
def test_arguments_the_library_refuses_raise_its_error_with_and_without_grad(grad):
    import fta_lib
    from flash_tt_attn import attention
    x = list(_operands(1)[:4])
    x[0].requires_grad_(grad)
    with pytest.raises(fta_lib.FtaError) as e:
        attention(*x, float("inf"))
    assert e.value.status == -8  # (the scale)


def test_a_subclass_of_the_function_runs_its_own_forward_and_backward():
    import flash_tt_attn as fta

    class Scaled(fta._attention):
        @staticmethod
        def forward(ctx, q, factor):
            ctx.factor = factor
            return q * factor

        @staticmethod
        def backward(ctx, do):
            return do * ctx.factor, None
    q = torch.ones(2, 3, requires_grad=True)
    out = Scaled.apply(q, 3.0)
    assert torch.equal(out, 3.0 * q) and torch.equal(torch.autograd.grad(out.sum(), q)[0], torch.full_like(q, 3.0))


@gpu
@pytest.mark.parametrize("which", ["attention", "python path", "block"])
def test_gradients_may_start_off_a_16_byte_boundary(which, monkeypatch):
    """(what the backward of a concatenation hands on, for instance)"""
    import flash_tt_attn as fta
    if which == "python path":
        monkeypatch.setattr(fta, "_native", lambda *a, **kw: None)
    *x, dout = _operands(1)
    run = lambda: fta.attention(*x, 0.3)
    if which == "block":
        blk, x, dout = _block(), [_pair(1)], _pair(2)
        run = lambda: blk(x[0])
    x[0].requires_grad_(True)
    off = torch.empty(dout.numel() + 3, dtype=dout.dtype, device=DEV)[3:].view(dout.shape).copy_(dout)
    assert off.data_ptr() % 16 != 0
    assert torch.equal(*(torch.autograd.grad(run(), x[0], g)[0] for g in (off, dout)))


def _transposing_hooks():
    """Saved tensors packed with their last two dimensions in the other order: the same values come back with other strides."""
    return torch.autograd.graph.saved_tensors_hooks(lambda t: t.mT.contiguous().mT if t.dim() > 1 else t, lambda t: t)


@gpu
@pytest.mark.parametrize("which", ["attention", "python path", "block"])
def test_tensors_saved_for_the_backward_may_come_back_in_another_layout(which, monkeypatch):
    import flash_tt_attn as fta
    if which == "python path":
        monkeypatch.setattr(fta, "_native", lambda *a, **kw: None)
    if which == "block":
        blk, z = _block(), _pair(1).requires_grad_(True)
        run, inputs, dout = lambda: blk(z, torch.ones(1, 48, device=DEV)), [z, *blk.parameters()], _pair(2)
    else:
        *x, dout = _operands(1)
        inputs = [t.requires_grad_(True) for t in x]
        run = lambda: fta.attention(*x, 0.3)
    want = torch.autograd.grad(run(), inputs, dout)
    with _transposing_hooks():
        got = torch.autograd.grad(run(), inputs, dout)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


_OTHER = {"type": lambda t: t.to(torch.float8_e5m2 if t.dtype != torch.uint8 else torch.int8), "device": lambda t: t.cpu(),
          "size": lambda t: t.flatten()[:1].clone()}


@gpu
@pytest.mark.parametrize("other", sorted(_OTHER))
@pytest.mark.parametrize("which,nth", [(w, n) for w, saved in (("attention", 6), ("python path", 6), ("block", 13)) for n in range(saved)])
def test_saved_tensors_that_come_back_as_others_are_refused(which, nth, other, monkeypatch):
    """One of them at a time, on the host: before anything is launched."""
    import flash_tt_attn as fta
    if which == "python path":
        monkeypatch.setattr(fta, "_native", lambda *a, **kw: None)
    blk, z, count = _block(), _pair(1), [0]
    *x, dout = _operands(1)
    x[0].requires_grad_(True)

    def pack(t):
        count[0] += 1
        return _OTHER[other](t.detach()) if count[0] == nth + 1 else t
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        out = blk(z, torch.ones(1, 48, device=DEV)) if which == "block" else fta.attention(*x, 0.3)
    assert count[0] == (13 if which == "block" else 6)
    with pytest.raises(RuntimeError, match="hook for saved tensors"):
        out.backward(torch.ones_like(out))


@gpu
def test_a_function_mode_sees_the_layers_of_the_block():
    from torch.overrides import TorchFunctionMode

    class Log(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))
    blk, z, seen = _block(), _pair(1), []
    with Log(), torch.no_grad():
        blk(z)
    assert torch.nn.functional.linear in seen
    with torch.device(DEV):  # (says where new tensors go: nothing the fused path hides from it)
        assert blk._fused(z, None, None) is not None


@gpu
def test_a_mask_of_a_subclass_goes_to_the_separate_layers():
    class Sub(torch.Tensor):
        pass
    blk, z, mask = _block(), _pair(1), torch.ones(1, 48, device=DEV)
    assert blk._fused(z, mask, None) is not None and type(blk(z, mask)) is torch.Tensor
    assert blk._fused(z, mask.as_subclass(Sub), None) is None


@gpu
def test_second_derivatives_of_the_block_are_refused_not_dropped():
    blk, z = _block(), _pair(1).requires_grad_(True)
    out = blk(z)
    dz, = torch.autograd.grad(out.square().sum(), z, create_graph=True)
    want, = torch.autograd.grad(blk(z).square().sum(), z)
    assert torch.equal(dz, want)
    with pytest.raises(RuntimeError, match="twice"):
        (out.sum() + dz.square().sum()).backward()


@gpu
@pytest.mark.parametrize("nth", [1, 2, 3])
@pytest.mark.parametrize("device", ["cpu", "meta"])
@pytest.mark.parametrize("grad", [False, True])
def test_operands_on_another_device_are_refused(nth, device, grad):
    from flash_tt_attn import attention
    x = list(_operands(1)[:4])
    x[nth] = x[nth].to(device)
    x[0].requires_grad_(grad)
    with pytest.raises(ValueError, match="same device"):
        attention(*x, 0.3)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["contiguous", "projection", "ending", "every other row", "one of two batches"])
def test_the_output_has_the_strides_that_empty_like_gives(layout):
    """The forward's output keeps a dense tensor's strides, whatever their order; of a tensor with gaps it takes the order."""
    import flash_tt_attn as fta
    q = {"contiguous": lambda: torch.randn(2, 4, 6, 40, 32), "projection": lambda: torch.randn(2, 6, 40, 4, 32).permute(0, 3, 1, 2, 4),
         "ending": lambda: torch.randn(2, 4, 40, 6, 32).transpose(2, 3), "every other row": lambda: torch.randn(2, 4, 12, 40, 32)[:, :, ::2],
         "one of two batches": lambda: torch.randn(4, 6, 4, 40, 32).permute(0, 2, 1, 3, 4)[::2]}[layout]()
    storage = torch.empty(q.untyped_storage().nbytes() // 4, dtype=torch.float16, device="cuda").normal_()
    q = storage.as_strided(q.shape, q.stride(), q.storage_offset())
    b = torch.randn(2, 4, 40, 40, device="cuda", dtype=torch.float16)
    for grad in (False, True):
        o = fta.attention(q.detach().requires_grad_(grad), q, q, b, 0.2)
        assert o.stride() == torch.empty_like(q).stride() and o.storage_offset() == 0
        ref = torch.nn.functional.scaled_dot_product_attention(q.float().cpu(), q.float().cpu(), q.float().cpu(), b.float().cpu()[:, :, None], scale=0.2)
        assert (o.detach().float().cpu() - ref).abs().max() <= 1e-2
