"""What the Python side of the blocks hands to the native library, recorded on the CPU: nothing is launched, so the calls
that must be refused ahead of a launch can be made here."""
import weakref

import pytest
import torch


class Calls(list):
    """The native calls made, as (name, arguments)."""

    def names(self):
        return [c[0] for c in self]


@pytest.fixture
def calls(pkg, monkeypatch):
    """CPU tensors pass for GPU tensors and native calls are recorded instead of made."""
    seen = Calls()
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(pkg._lib, "call", lambda name, *args: seen.append((name, args)))
    monkeypatch.setattr(pkg.ops, "_stream", lambda: 0)
    monkeypatch.setattr(pkg.ops, "workspaces", lambda device, *req: [torch.empty(s, dtype=t) for _, s, t in req])
    return seen


def layer_of(pkg, preset="ref", cls=None, **kw):
    torch.manual_seed(1)
    return (cls or pkg.SwinLayer)(None, 128, 2, 64, 256, (8, 8), (16, 32), False, 10_000, preset=preset, **kw).to(torch.bfloat16)


def inputs(pkg, n=512, b=1, dtype=torch.float32, rows=1):
    return torch.randn(b, n, 128).to(dtype), torch.randn(rows, 128)


def model_of(pkg, layers=2, **kw):
    return pkg.LocalAERIS(None, 2, 128, 64, 256, (8, 8), (16, 32), n_layers=layers + 2, model_in_channels=10, model_out_channels=4, **kw)


@pytest.mark.parametrize("preset", ["ref", "spec"])
@pytest.mark.parametrize("n", [64, 511, 513, 1024])
def test_another_token_count_than_the_grid_is_refused(pkg, calls, preset, n):
    layer = layer_of(pkg, preset)
    x, t = inputs(pkg, n)
    for run in (lambda: layer(x, t), lambda: layer.block_forward(0, x, t, (0, 0)), lambda: layer.block_forward(0, x, t, (0, 0), out=x.clone())):
        with pytest.raises(RuntimeError, match="tokens"):
            run()
    with pytest.raises(RuntimeError, match="tokens"):
        model_of(pkg)(torch.randn(1, n, 10), torch.zeros(1))
    assert "aeris_blocks_fwd" not in calls.names()
    layer(*inputs(pkg))
    assert calls.names()[-1] == "aeris_blocks_fwd"


def modulation_of(pkg, calls, make):
    """Address and row stride that the native call gets for a hooked modulation's result ``make(vectors)``, and that result."""
    layer, kept = layer_of(pkg), []

    def hook(module, args, out):
        kept.append(make(out))
        return kept[-1]
    layer.modulelist[0][4].register_forward_hook(hook)
    layer(*inputs(pkg, b=3, rows=3))
    record = pkg.ops.BLOCK_RECORD.unpack(calls[-1][1][1])
    return record[14:16], kept[0]


@pytest.mark.parametrize("name,make", [
    ("as_it_is", lambda m: m),
    ("one_row", lambda m: m[:1].clone()),
    ("row_expanded", lambda m: m[:1].expand(3, -1)),
    ("columns_of_a_wider_matrix", lambda m: torch.randn(3, 1000)[:, 100:868]),
    ("every_other_row", lambda m: torch.randn(6, 768)[::2]),
])
def test_modulation_is_read_with_its_own_rows(pkg, calls, name, make):
    got, m = modulation_of(pkg, calls, make)
    assert got == (m.data_ptr(), 0 if m.shape[0] == 1 else m.stride(0))


@pytest.mark.parametrize("name,make", [
    ("bf16", lambda m: m.to(torch.bfloat16)),
    ("f64", lambda m: m.double()),
    ("too_few_columns", lambda m: m[:, :640]),
    ("two_rows_of_three", lambda m: m[:2]),
    ("columns_strided", lambda m: torch.randn(3, 1536)[:, ::2]),
])
def test_modulation_of_another_form_is_refused(pkg, calls, name, make):
    with pytest.raises(RuntimeError, match="modulation"):
        modulation_of(pkg, calls, make)
    assert "aeris_blocks_fwd" not in calls.names()


@pytest.mark.parametrize("tokens", [0, 1, 511, 513])
def test_a_result_of_another_size_is_refused(pkg, calls, tokens):
    layer = layer_of(pkg)
    x, t = inputs(pkg)
    with pytest.raises(RuntimeError, match="out has the wrong size"):
        layer.block_forward(0, x, t, (0, 0), out=torch.empty(1, tokens, 128))
    assert "aeris_blocks_fwd" not in calls.names()


@pytest.mark.parametrize("window", [8, 16])  # the attention kernel's table; the one-kernel attention's
def test_a_bias_table_of_another_shape_is_refused(pkg, calls, window):
    torch.manual_seed(1)
    layer = pkg.SwinLayer(None, 256, 4, 64, 512, (window, window), (16, 32), False, 10_000, preset="spec", mod_ways=0).to(torch.bfloat16)
    x = torch.randn(1, 512, 256)
    layer(x)
    attn = layer.modulelist[0][1]
    good = attn.relative_position_bias_table
    for shape in (good.shape[::-1], (good.numel(), 1), (good.shape[0], 2), (good.shape[0] - 1, 4)):
        attn.relative_position_bias_table = torch.nn.Parameter(torch.zeros(shape, dtype=torch.bfloat16))
        del calls[:]
        with pytest.raises(RuntimeError, match="table"):
            layer(x)
        assert "aeris_blocks_fwd" not in calls.names()


def test_a_module_saved_whole_by_an_earlier_version_still_runs(pkg, calls):
    """A pickled module brings the attributes it was saved with: those of the attention module as it has always been made."""
    layer = layer_of(pkg, "spec", mod_ways=0)
    known = {"training", "heads", "head_dim", "window_size", "image_shape", "scale", "shift_mask", "fuse_qkv", "_b4cache"}
    for name in [k for k in vars(layer.modulelist[0][1]) if k not in known and not k.startswith(("_parameters", "_buffers", "_modules",
                 "_non_persistent", "_backward", "_is_full", "_forward", "_state_dict", "_load_state"))]:
        del layer.modulelist[0][1].__dict__[name]
    layer(inputs(pkg)[0])
    assert calls.names()[-1] == "aeris_blocks_fwd"


def core_users(pkg, seen):
    """Layers whose attention is computed by a ``core`` of the caller's: an attention module of a subclass, one with a ``core``
    of its own, one that is no ``Attention`` at all."""
    class Mine(pkg.Attention):
        def core(self, y, shift=(0, 0), out=None):
            seen.append(("subclass", shift))
            return super().core(y, shift, out=out)

    class Other(torch.nn.Module):
        def __init__(self, wo):
            super().__init__()
            self.wo = wo

        def core(self, y, shift, out=None):
            seen.append(("module", shift))
            return out.zero_()

    a, b, c = layer_of(pkg, sublayers=2), layer_of(pkg, sublayers=2), layer_of(pkg, sublayers=2)
    a.modulelist[1][1].__class__ = Mine
    attn = b.modulelist[1][1]
    attn.core = lambda y, shift, out=None: seen.append(("instance", shift)) or pkg.Attention.core(attn, y, shift, out=out)
    c.modulelist[1][1] = Other(c.modulelist[1][1].wo)
    return {"subclass": a, "instance": b, "module": c}


def test_an_attention_core_of_the_callers_is_called(pkg, calls):
    x, t = inputs(pkg)
    seen = []
    for name, layer in core_users(pkg, seen).items():
        del seen[:], calls[:]
        layer(x, t, shift=(4, 4))
        assert seen == [(name, (4, 4))]
        # the other block goes in one call; this one step by step, both norms, the two MLP projections and the output projection
        assert calls.names().count("aeris_blocks_fwd") == 1 and calls.names().count("aeris_norm_modulate_fwd") == 2
        assert calls.names().count("aeris_gemm_fwd") == 3
        model = model_of(pkg, layers=1)
        model.layers[0] = layer
        del seen[:]
        model(torch.randn(1, 512, 10), torch.zeros(1))
        assert seen == [(name, (0, 0))]


@pytest.mark.parametrize("current", [0, 1])
def test_sampler_update_stays_on_the_tensors_device(pkg, calls, monkeypatch, current):
    """The kernel goes to the current device's stream: a caller's own model on another device keeps the element-wise route."""
    x, f, t = torch.randn(1, 8, 4), torch.randn(1, 8, 4), torch.linspace(1, 0, 3)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: current)
    monkeypatch.setattr(torch.Tensor, "device", torch.device("cuda:1"))
    assert pkg.ops.heun_update_supported(x, f, None, t) == (current == 1)
    assert pkg.ops.heun_update_supported(x, f, f, t) == (current == 1)


@pytest.mark.parametrize("shape", [(0, 8, 4), (2, 0, 4)])
def test_sampler_update_of_nothing(pkg, calls, monkeypatch, shape):
    """No members, or no tokens: an empty result, and no launch (the native call refuses a size of 0)."""
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: None)
    s = pkg.TrigFlowSampler(lambda x, t, cond=None, x_div=1.0: torch.sin(x) * t, n_steps=2, device="cpu")
    del calls[:]
    assert s.sample(torch.zeros(shape), torch.zeros(shape)).shape == shape and not calls


@pytest.mark.parametrize("preset", ["ref", "spec"])
def test_a_tap_sees_the_intermediates_before_they_are_used(pkg, calls, preset):
    """``tap`` may change what it is shown: it is called between the operation that writes the tensor and the one that reads it."""
    layer = layer_of(pkg, preset)
    x, t = inputs(pkg)
    seen = []
    layer(x, t, tap=lambda name, tensor, block: seen.append((name, tensor, block, len(calls))))
    assert [s[0] for s in seen] == ["attn", "hidden"] and all(s[2] is layer.modulelist[0] for s in seen)
    (_, attn, _, at_attn), (_, hidden, _, at_hidden) = seen
    assert attn.shape == (512, 128) and hidden.shape == (1, 512, 256)
    wo, down = calls[at_attn], calls[at_hidden]
    assert (wo[0], wo[1][0]) == ("aeris_gemm_fwd", attn.data_ptr()) and calls[at_attn - 1][0] == "aeris_window_attention_heads_fwd"
    assert (down[0], down[1][0]) == ("aeris_gemm_fwd", hidden.data_ptr()) and at_hidden == len(calls) - 1


@pytest.mark.parametrize("x_dtype,out_dtype", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
def test_a_result_of_another_type_than_x(pkg, calls, x_dtype, out_dtype):
    x, t = inputs(pkg, dtype=x_dtype)
    out = torch.empty(1, 512, 128, dtype=out_dtype)
    assert layer_of(pkg).block_forward(0, x, t, (0, 0), out=out) is out
    code = pkg.ops._DT
    wo, down = [a for name, a in calls if name == "aeris_gemm_fwd" and a[2] == out.data_ptr()]
    assert (wo[5], wo[11], wo[12]) == (x.data_ptr(), code[x_dtype], code[out_dtype])  # residual, its type, the result's
    assert (down[5], down[11], down[12]) == (out.data_ptr(), code[out_dtype], code[out_dtype])


def test_a_block_hook_may_change_the_blocks_to_come(pkg, calls):
    """Weights brought in by the hook ahead of their block: the block runs with what its modules hold when its turn comes, and the
    stream after the block before it stays whole until the block after it has run."""
    model = model_of(pkg, layers=3)
    blocks = [layer.modulelist[0] for layer in model.layers]
    new = {}
    states = []

    def hook(k, hidden):
        states.append(hidden.data_ptr())
        if k in (1, 2):
            for linear in (blocks[k][1].wo, blocks[k][4].modulation[2]):
                linear.weight = torch.nn.Parameter(linear.weight.detach().clone())
            new[k] = (blocks[k][1].wo.weight.data_ptr(), blocks[k][4].modulation[2].weight.data_ptr())

    model(torch.randn(1, 512, 10), torch.zeros(1), block_hook=hook)
    records = [pkg.ops.BLOCK_RECORD.unpack(a[1]) for name, a in calls if name == "aeris_blocks_fwd"]
    read = [c for c in calls if c[0] in ("aeris_modulation_linear_fwd", "aeris_modulation_layers_fwd")]
    assert [r[6] for r in records[1:]] == [new[1][0], new[2][0]]
    for k in (1, 2):
        assert any(new[k][1] in a or new[k][1].to_bytes(8, "little") in (a[0] if isinstance(a[0], bytes) else b"") for _, a in read)
    assert len(states) == 4 and all(a != b for a, b in zip(states, states[1:]))


@pytest.mark.parametrize("whole_model", [False, True])
def test_a_hooked_modulation_is_called_when_its_block_is_due(pkg, calls, whole_model):
    """A hook on a block's modulation may bring in that block's weights: it runs after the blocks before it are launched, and
    its block's weights are read after it."""
    if whole_model:
        run = model_of(pkg, layers=3)
        blocks = [layer.modulelist[0] for layer in run.layers]
    else:
        run = layer_of(pkg, sublayers=3)
        blocks = list(run.modulelist)
    new = []

    def bring_in(module, args):
        assert calls.names().count("aeris_blocks_fwd") == 2
        linear = blocks[2][1].wo
        linear.weight = torch.nn.Parameter(linear.weight.detach().clone())
        new.append(linear.weight.data_ptr())
    blocks[2][4].register_forward_pre_hook(bring_in)
    if whole_model:
        run(torch.randn(1, 512, 10), torch.zeros(1))
    else:
        run(*inputs(pkg))
    records = [a[1] for name, a in calls if name == "aeris_blocks_fwd"]
    assert len(new) == 1 and pkg.ops.BLOCK_RECORD.unpack(records[2])[6] == new[0]


def test_a_modulation_mlp_with_more_in_its_sequence(pkg, calls):
    """The first and third module of a modulation's sequence are its Linears, whatever follows them."""
    model = model_of(pkg)
    model(torch.randn(1, 512, 10), torch.zeros(1))  # (packs the input stage's weight)
    del calls[:]
    model(torch.randn(1, 512, 10), torch.zeros(1))
    want = calls.names()
    del calls[:]
    for seq in (model.layers[0].modulelist[0][4].modulation, model.output_stage.modulation):
        seq.append(torch.nn.Identity())
    model(torch.randn(1, 512, 10), torch.zeros(1))
    assert calls.names() == want


@pytest.mark.parametrize("whole_model", [False, True])
def test_computed_weights_live_one_block_at_a_time(pkg, calls, monkeypatch, whole_model):
    """Weights that a parametrisation computes at the access exist for their own block only, not for all blocks of a call."""
    import torch.nn.utils.parametrize as parametrize
    made, most = [], []

    class Computed(torch.nn.Module):
        def forward(self, w):
            made.append(weakref.ref(w2 := w.clone()))
            return w2

    if whole_model:
        run = model_of(pkg, layers=3)
        blocks = [layer.modulelist[0] for layer in run.layers]
    else:
        run = layer_of(pkg, sublayers=3)
        blocks = list(run.modulelist)
    for b in blocks:
        for linear in (b[1].to_qkv, b[1].wo, b[3].w1, b[3].w2, b[4].modulation[0], b[4].modulation[2]):
            parametrize.register_parametrization(linear, "weight", Computed())
    del made[:]

    def call(name, *args):
        calls.append((name, args))
        most.append(sum(r() is not None for r in made))
    monkeypatch.setattr(pkg._lib, "call", call)
    if whole_model:
        run(torch.randn(1, 512, 10), torch.zeros(1))
    else:
        run(*inputs(pkg))
    assert len(made) == 18 and max(most) == 4, (len(made), most)


@pytest.mark.parametrize("cls,method", [("Attention", "core"), ("SwinLayer", "block_forward"), ("ModulationLinear", "forward"),
                                        ("OutputStage", "forward")])
def test_a_method_wrapped_on_the_class_is_called(pkg, calls, monkeypatch, cls, method):
    """A profiler's or a patch's wrapper around a class's own method counts like an override on a module."""
    cls, seen = getattr(pkg.model, cls), []
    plain = getattr(cls, method)
    monkeypatch.setattr(cls, method, lambda self, *args, **kw: seen.append(args) or plain(self, *args, **kw))
    model_of(pkg, layers=2)(torch.randn(1, 512, 10), torch.zeros(1))
    assert len(seen) == (1 if cls is pkg.model.OutputStage else 2)


def test_hooks_on_all_modules_see_the_modulation_modules(pkg, calls):
    """Hooks registered for every module (torch.nn.modules.module.register_module_forward_hook) see what they always saw: each
    block's modulation, and the output stage with the arguments that count."""
    model = model_of(pkg, layers=2)
    hooks, seen = torch.nn.modules.module, []
    with hooks.register_module_forward_hook(lambda module, args, out: seen.append((type(module).__name__, len(args)))):
        model(torch.randn(1, 512, 10), torch.zeros(1))
    assert [s for s in seen if s[0] == "ModulationLinear"] == [("ModulationLinear", 1)] * 2
    given = []
    with hooks.register_module_forward_pre_hook(lambda m, args: given.append(args) if isinstance(m, pkg.model.OutputStage) else None):
        model.forward(torch.randn(1, 512, 10), torch.zeros(1))
    with model.output_stage.register_forward_pre_hook(lambda m, args, kw: given.append(kw), with_kwargs=True):
        model.forward(torch.randn(1, 512, 10), torch.zeros(1))
    assert len(given) == 2 and len(given[0]) == 2 and given[1] == {}


@pytest.mark.parametrize("layers", [0, 1, 2])
def test_the_embedding_survives_a_model_of_one_block(pkg, calls, layers):
    """What the input stage returns is overwritten from the second block on, not by the first."""
    model, tok = model_of(pkg, layers=layers), []
    model.input_stage.register_forward_hook(lambda m, args, out: tok.append(out[0].data_ptr()))
    _, hidden = model(torch.randn(1, 512, 10), torch.zeros(1), return_hidden=True)
    assert (hidden.data_ptr() == tok[0]) == (layers != 1)


@pytest.mark.parametrize("how", ["vmap", "jvp", "dual", "jit_trace", "make_fx", "function_mode", "subclass", "negated_view"])
def test_sampler_update_under_transforms_and_tracing(pkg, calls, monkeypatch, how):
    """With a model of the caller's own the sampler is ordinary tensor code: what follows tensors through it (vmap, forward-mode
    derivatives, tracing, tensor subclasses) meets element-wise operations and no native call."""
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: None)
    s = pkg.TrigFlowSampler(lambda x, t, cond=None, x_div=1.0: torch.sin(x) * t + cond, n_steps=2, device="cpu")
    cond, lat, tangent = torch.randn(3, 5, 4), torch.randn(3, 5, 4), torch.randn(3, 5, 4)

    def chain(x):
        ts = s.t_steps
        f0 = torch.sin(x) * ts[0] + cond
        f1 = torch.sin(x + (ts[1] - ts[0]) * f0) * ts[1] + cond
        x = x + (0.5 * (ts[1] - ts[0])) * (f0 + f1)
        return x + (ts[2] - ts[1]) * (torch.sin(x) * ts[1] + cond)

    def run(x):
        return s.sample(cond, x)
    del calls[:]
    if how == "vmap":
        got, want = torch.vmap(s.sample)(cond, lat), chain(lat)
    elif how == "jvp":
        got, want = torch.func.jvp(run, (lat,), (tangent,))[1], torch.func.jvp(chain, (lat,), (tangent,))[1]
    elif how == "dual":
        import torch.autograd.forward_ad as fw
        with fw.dual_level():
            got, want = (fw.unpack_dual(f(fw.make_dual(lat, tangent))).tangent for f in (run, chain))
    elif how == "jit_trace":
        got, want = torch.jit.trace(run, (torch.zeros_like(lat),), check_trace=False)(lat), chain(lat)
    elif how == "make_fx":
        from torch.fx.experimental.proxy_tensor import make_fx
        got, want = make_fx(run)(torch.zeros_like(lat))(lat), chain(lat)
    elif how == "function_mode":
        class Counts(torch.overrides.TorchFunctionMode):
            updates = 0

            def __torch_function__(self, func, types, args=(), kwargs=None):
                self.updates += func in (torch.add, torch.Tensor.add)
                return func(*args, **(kwargs or {}))
        with Counts() as mode:
            got, want = run(lat), chain(lat)
        assert mode.updates == 2 * (3 + 1 + 3)  # the model's own, F_s + F_t, the updates
    elif how == "negated_view":
        plain = s.model
        s.model = lambda x, t, cond=None, x_div=1.0: torch._neg_view(-plain(x, t, cond))
        got, want = run(lat), chain(lat)
        s.model = plain
    else:
        class Mine(torch.Tensor):
            pass
        got = run(lat.as_subclass(Mine))
        assert type(got) is Mine
        want = chain(lat)
    assert torch.allclose(got.as_subclass(torch.Tensor), want, rtol=1e-5, atol=1e-5) and not calls
    run(lat)
    assert calls.names() == ["aeris_heun_update_fwd"] * 3


def test_a_weight_that_a_subclass_works_out(pkg, calls):
    """A Linear whose class answers ``weight`` with something else than the parameter it stores: that is what the block takes."""
    layer, made = layer_of(pkg), []

    class Doubled(torch.nn.Linear):
        @property
        def weight(self):
            made.append(2 * self._parameters["weight"])
            return made[-1]
    layer.modulelist[0][1].wo.__class__ = Doubled
    layer(*inputs(pkg))
    assert pkg.ops.BLOCK_RECORD.unpack(calls[-1][1][1])[6] == made[-1].data_ptr()
    mod = layer.modulelist[0][4].modulation[2]
    mod.__class__ = Doubled
    layer(*inputs(pkg))
    assert any(made_.data_ptr() in args for made_ in made for name, args in calls if name == "aeris_modulation_linear_fwd")


def test_an_mlp_that_passes_its_parts_through(pkg, calls):
    """A wrapper in the MLP's place whose w1 and w2 are attributes but not modules of its own."""
    class Around(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        w1 = property(lambda self: self.inner.w1)
        w2 = property(lambda self: self.inner.w2)
    layer = layer_of(pkg)
    ff = layer.modulelist[0][3]
    layer.modulelist[0][3] = Around(ff)
    layer(*inputs(pkg))
    assert pkg.ops.BLOCK_RECORD.unpack(calls[-1][1][1])[8:12:2] == (ff.w1.weight.data_ptr(), ff.w2.weight.data_ptr())


def test_a_swiglu_mlp_has_no_biases(pkg, calls):
    """FeedForward multiplies by its two weights: a bias that one of its Linears holds counts neither there nor in a block, and
    what stands in a Linear's place needs none."""
    layer = layer_of(pkg)
    ff = layer.modulelist[0][3]
    ff.w1.bias, ff.w2.bias = (torch.nn.Parameter(torch.ones(n, dtype=torch.bfloat16)) for n in (512, 128))
    layer(*inputs(pkg))
    assert pkg.ops.BLOCK_RECORD.unpack(calls[-1][1][1])[9:12:2] == (0, 0)
    layer(*inputs(pkg), tap=lambda *a: None)
    assert [args[3] for name, args in calls if name == "aeris_gemm_fwd"] == [None] * 3

    class Weight(torch.nn.Module):
        def __init__(self, weight):
            super().__init__()
            self.weight = weight
    ff.w1, ff.w2 = Weight(ff.w1.weight), Weight(ff.w2.weight)
    layer(*inputs(pkg))
    layer(*inputs(pkg), tap=lambda *a: None)


def draw_of(pkg, calls, monkeypatch, change=lambda sampler: None, steps=10, **kw):
    """The native calls of one draw, by name, with a model of two blocks."""
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: None)
    s = pkg.TrigFlowSampler(model_of(pkg, **kw), n_steps=steps, device="cpu")
    change(s)
    del calls[:]
    s.sample(torch.randn(1, 512, 6), torch.randn(1, 512, 4))
    return calls.names()


@pytest.mark.parametrize("kw", [dict(preset="ref"), dict(preset="spec", mod_ways=2)])
def test_a_draw_computes_the_modulation_of_several_levels_at_once(pkg, calls, monkeypatch, kw):
    """Ten levels: two passes over the modulation matrices for nineteen denoiser calls, each with its own level's vectors."""
    names = draw_of(pkg, calls, monkeypatch, **kw)
    assert names.count("aeris_blocks_fwd") == 19 and names.count("aeris_modulation_layers_fwd") == 4
    assert [c[1][2] for c in calls if c[0] == "aeris_modulation_layers_fwd"] == [8, 8, 2, 2]
    records = [c[1][1] for c in calls if c[0] == "aeris_blocks_fwd"]
    size = pkg.ops.BLOCK_RECORD.size
    vectors = [[pkg.ops.BLOCK_RECORD.unpack(r[k:k + size])[14] for k in (0, size)] for r in records]
    level = [0] + [k for i in range(1, 10) for k in (i, i)]
    for k in range(2):  # consecutive rows within a pass
        width = 4 * 128 * 2 * kw.get("mod_ways", 3)
        for a, b, va, vb in zip(level, level[1:], vectors, vectors[1:]):
            if a // 8 == b // 8:
                assert vb[k] - va[k] == (b - a) * width


@pytest.mark.parametrize("what", ["model_hook", "input_hook", "output_hook", "modulation_hook", "core", "model_class", "model_forward",
                                  "sampler_class", "sampler_method", "advance", "modulations", "block_calls", "_block_call", "layer_class",
                                  "model_compiled", "input_compiled"])
def test_a_draw_with_parts_of_the_callers_looks_at_every_call(pkg, calls, monkeypatch, what):
    seen = []

    def change(s):
        m = s.model
        if what == "model_hook":
            m.register_forward_hook(lambda *a: seen.append(1))
        elif what == "input_hook":
            m.input_stage.register_forward_hook(lambda *a: seen.append(1))
        elif what == "output_hook":
            m.output_stage.register_forward_pre_hook(lambda *a: seen.append(1))
        elif what == "modulation_hook":
            m.layers[0].modulelist[0][4].register_forward_hook(lambda *a: seen.append(1))
        elif what == "core":
            attn = m.layers[0].modulelist[0][1]
            attn.core = lambda y, shift, out=None: seen.append(1) or pkg.Attention.core(attn, y, shift, out=out)
        elif what == "model_class":
            m.__class__ = type("Mine", (pkg.LocalAERIS,), {"forward": lambda self, *a, **kw: seen.append(1) or pkg.LocalAERIS.forward(self, *a, **kw)})
        elif what == "model_forward":
            m.forward = lambda *a, **kw: seen.append(1) or pkg.LocalAERIS.forward(m, *a, **kw)
        elif what in ("model_compiled", "input_compiled"):  # (a compiler that calls what it is given)
            monkeypatch.setattr(torch, "compile", lambda f, *a, **kw: lambda *a, **kw: seen.append(1) or f(*a, **kw))
            (m if what == "model_compiled" else m.input_stage).compile()
        elif what in ("modulations", "block_calls", "_block_call"):
            layer, plain = m.layers[0], getattr(pkg.SwinLayer, what)
            setattr(layer, what, lambda *a: seen.append(1) or plain(layer, *a))
        elif what == "layer_class":
            plain = pkg.SwinLayer._block_call
            monkeypatch.setattr(pkg.SwinLayer, "_block_call", lambda self, *a: (self is m.layers[0] and seen.append(1)) or plain(self, *a))
        elif what == "sampler_class":
            s.__class__ = type("Mine", (pkg.TrigFlowSampler,), {"_denoise": lambda self, *a: seen.append(1) or pkg.TrigFlowSampler._denoise(self, *a)})
        elif what == "sampler_method":
            s._denoise = lambda *a: seen.append(1) or pkg.TrigFlowSampler._denoise(s, *a)
        else:
            s._advance = lambda *a: seen.append(1) or pkg.TrigFlowSampler._advance(s, *a)
    draw_of(pkg, calls, monkeypatch, change, steps=2)
    assert len(seen) == 3


def test_a_draw_with_computed_weights_makes_them_at_every_call(pkg, calls, monkeypatch):
    """... once per call, and holds one block's at a time: as the calls one by one do."""
    made, most = [], []

    class Made(torch.nn.Module):
        def forward(self, w):
            r = w.clone()
            made.append(weakref.ref(r))
            return r

    def change(s):
        for layer in s.model.layers:
            torch.nn.utils.parametrize.register_parametrization(layer.modulelist[0][1].wo, "weight", Made())
        record = pkg._lib.call

        def call(name, *args):
            record(name, *args)
            most.append(sum(r() is not None for r in made))
        monkeypatch.setattr(pkg._lib, "call", call)
        del made[:]
    names = draw_of(pkg, calls, monkeypatch, change, steps=2, layers=4)
    assert names.count("aeris_blocks_fwd") == 12 and len(made) == 12 and max(most) == 1, (len(made), most)


@pytest.mark.parametrize("part", ["to_qkv", "w2", "norm"])
def test_a_draw_asks_a_part_of_the_callers_at_every_call(pkg, calls, monkeypatch, part):
    """A replaced part whose weight is a property (weights that are swapped in, say) may return another one each time."""
    class Swapped(torch.nn.Module):
        def __init__(self, weight):
            super().__init__()
            self.a, self.b, self.asked = torch.nn.Parameter(weight.detach().clone()), torch.nn.Parameter(weight.detach().clone()), 0

        @property
        def weight(self):
            self.asked += 1
            return self.a if self.asked % 2 else self.b

    parts = []

    def change(s):
        n1, attn, _, ff = list(s.model.layers[1].modulelist[0])[:4]
        if part == "norm":
            parts.append(Swapped(n1.weight))
            s.model.layers[1].modulelist[0][0] = parts[0]
        else:
            owner = attn if part == "to_qkv" else ff
            parts.append(Swapped(getattr(owner, part).weight))
            setattr(owner, part, parts[0])
    names = draw_of(pkg, calls, monkeypatch, change, steps=2)
    size, at = pkg.ops.BLOCK_RECORD.size, {"norm": 0, "to_qkv": 4, "w2": 10}[part]
    given = [pkg.ops.BLOCK_RECORD.unpack(c[1][1][size:2 * size])[at] for c in calls if c[0] == "aeris_blocks_fwd"]
    a, b = parts[0].a.data_ptr(), parts[0].b.data_ptr()
    assert names.count("aeris_blocks_fwd") == 3 and parts[0].asked == 3 and given == [a, b, a]


@pytest.mark.parametrize("window", [8, 16])  # the attention kernel's table; the one-kernel attention's
@pytest.mark.parametrize("what", ["storage", "parameter", "table"])
def test_a_draw_sees_parameters_that_move(pkg, calls, monkeypatch, window, what):
    """Another thread may replace a parameter or its storage while a draw runs: the calls that follow take it where it is."""
    torch.manual_seed(1)
    model = pkg.LocalAERIS(None, 4, 256, 64, 512, (window, window), (16, 32), n_layers=4, model_in_channels=10, model_out_channels=4,
                           preset="spec", mod_ways=2)
    attn = model.layers[1].modulelist[0][1]
    given, record = [], pkg._lib.call

    def where():
        table = attn.relative_position_bias_table
        return attn.wo.weight.data_ptr(), table.data_ptr() if window == 8 else 0, attn._bias4().data_ptr() if window == 16 else 0

    def call(name, *args):
        record(name, *args)
        if name != "aeris_blocks_fwd":
            return
        r = pkg.ops.BLOCK_RECORD.unpack(args[1][-pkg.ops.BLOCK_RECORD.size:])
        given.append((r[6], r[12], r[13]) == where())
        if len(given) in (1, 3):  # between the calls of the draw
            if what == "table":
                with torch.no_grad():
                    attn.relative_position_bias_table = torch.nn.Parameter(attn.relative_position_bias_table + 1)
            elif what == "parameter":
                attn.wo.weight = torch.nn.Parameter(attn.wo.weight.detach().clone())
            else:
                attn.wo.weight.data = attn.wo.weight.detach().clone()
    monkeypatch.setattr(pkg._lib, "call", call)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: None)
    pkg.TrigFlowSampler(model, n_steps=3, device="cpu").sample(torch.randn(1, 512, 6), torch.randn(1, 512, 4))
    assert given == [True] * 5


def test_an_empty_model_draws(pkg, calls, monkeypatch):
    names = draw_of(pkg, calls, monkeypatch, steps=2, layers=0)
    assert names.count("aeris_output_stage_fwd") == 3 and "aeris_blocks_fwd" not in names
