"""The wrappers' native host side: what it takes gives what the wrappers' own way gives, bit for bit, and what it does not take it leaves alone."""
import pytest
import torch


@pytest.fixture
def both(monkeypatch):
    """run(f): f() with the native calls and without them."""
    from jacobiforcing_amd import layer_ops as LO

    class Nothing:
        def __getattr__(self, name):
            return lambda *a: NotImplemented

    def run(f):
        got = f()
        with monkeypatch.context() as m:
            m.setattr(LO, "_H", Nothing())
            return got, f()
    return run


def test_the_rules_of_linear():
    """The product that the native call takes is the one that the wrapper's rules name, at their lines and around them."""
    from jacobiforcing_amd import layer_ops as LO
    H = LO._host()
    for n in (1, 2, 16, 17, 63, 64, 65, 127, 191, 193, 512, 1021, 2553, 9000):
        for k in (4, 64, 512, 1020, 1024, 1028, 2048, 2052, 4096):
            for o in (1, 16, 96, 1024, 4096, 4097, 8192, 16384, 16385, 32000):
                for size in (2, 4):
                    small = n <= LO.LINEAR_SMALL_ROWS and LO.linear_small(n, k, o, size)
                    want = 1 if small else (2 if LO.linear_split(n, k, o) else 0) if size == 4 else 3 if LO.linear_mid(n, k, o, torch.bfloat16) else 0
                    assert H.linear_rule(n, k, o, size) == want, (n, k, o, size)


@pytest.mark.parametrize("n,k,o,own", [
    (2553, 1024, 1024, True), (2553, 1024, 3072, True), (4096, 4096, 4096, True), (2049, 1028, 1153, True), (1700, 1024, 1024, True), (128, 1024, 16384, True), (8192, 512, 1024, True), (640, 64, 2500, True),
    (96, 1024, 16384, False), (160, 1024, 8192, False), (65, 2048, 25000, False), (650, 1024, 3072, False), (513, 1024, 4096, False), (1290, 1024, 3072, False), (2060, 1024, 1024, False),
    (4100, 2048, 1024, False), (1536, 4096, 1024, False), (640, 512, 1024, False), (1, 1024, 100000, False), (0, 1024, 1024, False),
])
def test_linear_leaves_what_fills_tiles_badly_to_the_library(n, k, o, own):
    """Products that were measured faster one way or the other (jl_linear_split_ok)."""
    from jacobiforcing_amd import layer_ops as LO
    assert LO.linear_split(n, k, o) == own


def test_what_it_does_not_take():
    """Host tensors, other numbers of arguments, other kinds of values: handed back, nothing raised."""
    from jacobiforcing_amd import layer_ops as LO
    H, x = LO._host(), torch.randn(4, 64)
    assert H.linear(x, x, None, None) is NotImplemented and H.linear(x, x) is NotImplemented and H.linear(None, 1, "x", 2.0) is NotImplemented
    assert H.add_rmsnorm(x, None, None, None, "eps", None) is NotImplemented and H.sandwich_norm(x, None, None, 1e-5, None, torch.float16, None, None, False) is NotImplemented
    assert H.moe_experts(*[None] * 15) is NotImplemented and H.attention_args(*[7] * 30) is NotImplemented and H.linear_scan(*[x] * 19) is NotImplemented


@pytest.mark.parametrize("broken", ["no compiler", "not a library"])
def test_without_it(monkeypatch, tmp_path, broken):
    """Where the module can be neither built nor loaded the wrappers go their own way, with a warning; one built for another torch is not found."""
    from jacobiforcing_amd import _build, _native as N, layer_ops as LO
    assert torch.__version__ in _build.host_lib().name
    monkeypatch.setattr(torch, "__version__", "0.1")
    assert not _build.host_lib().exists()
    monkeypatch.setattr(_build, "LIB_DIR", tmp_path)
    if broken == "no compiler":
        monkeypatch.setenv("PATH", "/nowhere")
        monkeypatch.setattr(_build, "hipcc", lambda: "/nowhere/hipcc")
    else:
        _build.host_lib().write_text("")
    with pytest.warns(RuntimeWarning, match="more of the host"):
        H = N.host(LO.LINEAR_SMALL_ROWS, LO.LINEAR_ONE_TILE, LO.LINEAR_X_BYTES)
    x = torch.randn(4, 64)
    assert H.linear(x, x, None, None) is NotImplemented and H.moe_experts() is NotImplemented


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 5, 130])
def test_the_same_as_the_wrappers(both, dtype, n):
    from jacobiforcing_amd import _native as N, layer_ops as LO
    dev, W, H, D = "cuda", 64, 2, 32
    g = torch.Generator(device=dev).manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, y, y3, w, row, wide = rnd(n, W), rnd(n, W).to(dtype), rnd(n, 3, W), rnd(W), rnd(W), rnd(n, 6 * W).to(dtype)
    mat, bias = rnd(96, W).to(dtype), rnd(96).to(dtype)
    counts, starts = ([1] * n, [3] * n) if n < 100 else ([60, 70], [0, 9])
    batch = LO.RaggedBatch.build(counts, starts, list(range(len(counts))), [list(range(2 * b, 2 * b + 2)) for b in range(len(counts))], 64, dev)
    B, cos, sin = len(counts), rnd(200, 8), rnd(200, 8)
    pool, pool_v = (torch.zeros(B * 128, H * D, dtype=dtype, device=dev) for _ in range(2))
    calls = dict(
        linear=lambda s: [LO.linear(y, mat, b, f) for b in (None, bias) for f in (None, True, False)] + [LO.linear(wide[:, W:2 * W], mat)],
        add_rmsnorm=lambda s: [LO.add_rmsnorm(s["x"], v, u, k, 1e-5, t) for v, u, k, t in ((y, None, w.to(dtype), dtype), (y3, x, None, torch.float32), (None, None, None, None))] + [s["x"]],
        sandwich_norm=lambda s: [LO.sandwich_norm(s["x"], y, w, 1e-5, row, dtype), LO.sandwich_norm(s["x"], None, None, 1e-5, None, torch.float32, add_row=row, plain=True),
                                 LO.sandwich_norm(s["x"], y, w, 1e-5, w, None, out=s["wide"][:, W:2 * W]), s["x"], s["wide"]],
        output_norm=lambda s: [LO.output_norm(s["x"], [(y, None), (y3, row)], w, 1e-5, kind, 0.5, row, dtype) for kind in (LO.NORM_RMS, LO.NORM_LAYER)] + [LO.output_norm(s["x"], [], None, 1e-5, 0, out_dtype=dtype)],
        gated_norm=lambda s: [LO.gated_norm(x, wide[:, :W], w, 1e-5, N.JL_ACT_SILU, True, 2, 0.5), LO.gated_norm(x, wide[:, :W], w, 1e-5, N.JL_ACT_SIGMOID, False, out=s["wide"][:, 2 * W:3 * W]), s["wide"]],
        gated_act=lambda s: [LO.gated_act(wide, 0, W, W, LO.ACT_SILU), LO.gated_act(wide, W, -1, 2 * W, LO.ACT_GELU_ERF, row_gate=wide[:, 5])],
        heads_gate=lambda s: [LO.heads_gate(wide.view(H, n, 3 * W), None), LO.heads_gate(wide[:, :2 * W].contiguous().view(H, n, W), wide[:, 2 * W:4 * W])],
        embed_scale=lambda s: [v for v in LO.embed_scale(mat, torch.arange(n, device=dev) % 96, 1.5, True, copy_dtype=torch.bfloat16) + LO.embed_scale(mat, torch.arange(n, device=dev) % 96, 2.0, False, s["x"])],
        token_shift=lambda s: [LO.token_shift(x, w, batch, s["tail"], dtype), s["tail"]],
        short_conv=lambda s: [LO.short_conv(wide, W, W, rnd(W, 4).to(dtype).zero_() + 0.5, batch, s["tail3"], bias=mat[0], out_dtype=dtype), s["tail3"]],
        depth_mix_norm=lambda s: [v for v in LO.depth_mix_norm(x, [(y, row)], 0.7, s["streams"], 1, w, s["x"], w, 1e-5, dtype, True, (row, batch, s["tail"]) if n < 100 else None)] + [s["streams"][1], s["tail"]],
        linear_scan=lambda s: [LO.linear_scan(wide, (0, 64, 128), batch, H, H, 32, 32, s["state"], act=N.JL_ACT_SILU, decay=torch.full((H,), 0.9, device=dev), skip=row[:H].contiguous()), s["state"]],
        qk_norm_append=lambda s: [LO.qk_norm_append(wide, (0, 64, 128), H, H, D, D, w.to(dtype), row.to(dtype), 1e-5, s["k"], s["v"], batch.kv_slot, 16, batch=batch, cos=cos, sin=sin), s["k"], s["v"]],
        latent_prep=lambda s: [LO.latent_prep(wide, 0, 64, 64, 48, 16, 16, w.to(dtype), w[:48].to(dtype), 1e-5, batch, cos, sin, s["k"]), s["k"]],
        latent_q_pack=lambda s: [LO.latent_q_pack(wide.view(H, n, 3 * W)[:, :, :48].contiguous(), wide[:, :H * (D + 16)], H, D, 48, 16, 16, batch, cos, sin)],
        moe_experts=lambda s: [v for route, identity in (("sigmoid", 0), ("top_softmax", 2)) for kw in (dict(router_logits=rnd_logits[:, :4 + identity].contiguous(), router=None),
                               dict(router_logits=None, router=(x, rnd_w[:4 + identity].contiguous(), None)))
                               for r in [LO.moe_experts(y, kw["router_logits"], row[:4 + identity].contiguous(), 2, 0.5, up, down, route=route, gated=(LO.ACT_SILU, 0.0, 1.0, 0.0), identity=identity, router=kw["router"])]
                               for v in ((r,) if torch.is_tensor(r) else r[1:])],
        attention_args=lambda s: [LO.attn_window(wide[:, :H * D].contiguous(), wide[:, 64:128], pool + 0.5, pool_v + 0.25, batch, H, H, D, D, 0.2, 0, 0, None, None, None, sink=row[:H].contiguous()),
                             LO.attn_sweep(wide[:, :H * D].contiguous(), pool + 0.5, pool_v + 0.25, batch, H, H, D, D, 0.2, 16, gate=wide[:, :H], gate_per_head=True)],
    )
    rnd_logits, rnd_w, up, down = rnd(n, 6), rnd(6, W), rnd(4, 2 * 32, W).to(dtype), rnd(4, W, 32).to(dtype)
    slots = B
    fresh = lambda: dict(x=x.clone(), wide=wide.clone(), tail=torch.ones(slots, 1, W, device=dev), tail3=torch.ones(slots, 3, W, device=dev), streams=torch.ones(2, n, W, device=dev),
                         state=torch.ones(slots, H, 32, 32, device=dev), k=pool.clone(), v=pool_v.clone())
    taken = []
    from unittest import mock
    host = LO._host()

    class Watched:
        def __getattr__(self, name):
            def call(*a):
                r = getattr(host, name)(*a)
                if r is not NotImplemented:
                    taken.append(name)
                return r
            return call
    with mock.patch.object(LO, "_H", Watched()):
        for name, f in calls.items():
            got, want = both(lambda: f(fresh()))
            assert len(got) == len(want) and all((a is None) == (b is None) and (a is None or (a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b))) for a, b in zip(got, want)), name
    left = set(calls) - set(taken)
    assert left == (set() if n < 100 else {"linear_scan"} | ({"linear"} if dtype == torch.float32 else set())), left      # portions of 32 tokens and more go in pieces; 130 float rows to the library


@pytest.mark.gpu
def test_refused_as_before():
    """Wrong shapes, types, devices and streams' tensors raise what the wrappers raise; gradients go where they went."""
    from jacobiforcing_amd import _native as N, layer_ops as LO
    dev = "cuda"
    x, w = torch.randn(4, 64, device=dev), torch.randn(64, device=dev)
    for call in (lambda: LO.add_rmsnorm(x.bfloat16(), None, None, None, 1e-5, torch.float32), lambda: LO.add_rmsnorm(x, x[:3], None, None, 1e-5, torch.float32),
                 lambda: LO.sandwich_norm(x, None, None, 1e-5, None, torch.float32), lambda: LO.gated_act(x, 60, -1, 8, LO.ACT_SILU), lambda: LO.add_rmsnorm(x, None, None, w, 1e-5, torch.float16),
                 lambda: LO.output_norm(x, [(x, None)] * 4, w, 1e-5, 0), lambda: LO.output_norm(x, [(x, None)], w, 1e-5, 9), lambda: LO.heads_gate(x.view(2, 2, 64).half(), None)):
        with pytest.raises(ValueError):
            call()
    with pytest.raises(N.NativeLibraryError):
        LO.add_rmsnorm(x.cpu(), None, None, None, 1e-5, torch.float32)
    leaf = torch.randn(16, 64, device=dev, requires_grad=True)
    LO.linear(x, leaf).sum().backward()
    assert leaf.grad is not None
    with torch.no_grad():
        assert not LO.linear(x, leaf).requires_grad
    seen = []

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))
    with Mode():
        LO.add_rmsnorm(x.clone(), None, None, w, 1e-5, torch.float32)
    assert torch.empty in seen                                                               # a mode that watches calls still sees the wrapper's


@pytest.mark.parametrize("n", [4, 200, 640])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_of_tensors_without_memory(n, dtype):
    """Fake tensors are answered by their shape, whatever launch the sizes would go to."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from jacobiforcing_amd import layer_ops as LO
    with FakeTensorMode():
        x, w, b = (torch.empty(*s, dtype=dtype, device="cuda") for s in ((n, 64), (2500, 64), (2500,)))
        for bias in (None, b):
            for float_out in (None, True, False):
                if float_out and dtype != torch.float32:
                    continue                                                                  # torch's product with a type of its own for the result has no fake form on every version
                y = LO.linear(x, w, bias, float_out)
                assert y.shape == (n, 2500) and y.dtype == (dtype if float_out is None else torch.float32) and y.is_cuda


@pytest.mark.gpu
@pytest.mark.parametrize("n", [4, 640])
def test_linear_lets_transforms_and_modes_pass(n):
    """Forward-mode tangents, vmap, and modes and subclasses that see the library's call: as they were without launches; a default device changes nothing."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from jacobiforcing_amd import layer_ops as LO
    dev = "cuda"
    g = torch.Generator(device=dev).manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, w, b, t, u = rnd(n, 64), rnd(2500, 64), rnd(2500), rnd(n, 64), rnd(2500, 64)
    assert LO.linear_split(n, 64, 2500) == (n == 640) and LO.linear_small(n, 64, 2500, 4) == (n == 4)
    close = lambda a, c: torch.allclose(a, c, rtol=1e-4, atol=1e-4)
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        for args, want in (((torch.autograd.forward_ad.make_dual(x, t), w, b), t @ w.T), ((x, torch.autograd.forward_ad.make_dual(w, u), b), x @ u.T)):
            y, tangent = torch.autograd.forward_ad.unpack_dual(LO.linear(*args))
            assert tangent is not None and close(tangent, want) and close(y, x @ w.T + b)
    many = rnd(3, n, 64)
    assert close(torch.vmap(lambda r: LO.linear(r, w, b))(many), many @ w.T + b)
    seen = []

    class Functions(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Operations(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Kind(torch.Tensor):
        pass
    with Functions():
        LO.linear(x, w, b)
    assert torch.nn.functional.linear in seen
    seen.clear()
    with Operations():
        LO.linear(x, w, b)
    assert any("addmm" in str(f) or "linear" in str(f) for f in seen)
    assert type(LO.linear(x.as_subclass(Kind), w, b)) is Kind
    want = LO.linear(x, w, b)
    with torch.device(dev):
        assert torch.equal(LO.linear(x, w, b), want)                                          # the same launch
    calls = []
    with pytest.MonkeyPatch.context() as m:
        m.setattr(LO.F, "linear", lambda *a: calls.append(a))
        with torch.device(dev):
            LO.linear(x, w, b)
    assert not calls


@pytest.mark.gpu
@pytest.mark.parametrize("n", [4, 640])
def test_linear_is_traced_and_compiled(n):
    """A trace records the library's product, and so does a compiler, which finds no call that it cannot follow."""
    from jacobiforcing_amd import layer_ops as LO
    g = torch.Generator(device="cuda").manual_seed(n)
    x, y, w, b = (torch.randn(*s, generator=g, device="cuda") for s in ((n, 64), (n, 64), (2500, 64), (2500,)))
    call, want = lambda v: LO.linear(v, w, b), y @ w.T + b
    with torch.no_grad():
        traced = torch.jit.trace(call, (x,), check_trace=False)
        assert "linear" in str(traced.graph) and torch.allclose(traced(y), want, rtol=1e-4, atol=1e-4)
        compiled = torch.compile(call, backend="eager", fullgraph=True)
        assert torch.allclose(compiled(x), x @ w.T + b, rtol=1e-4, atol=1e-4) and torch.allclose(compiled(y), want, rtol=1e-4, atol=1e-4)


@pytest.mark.gpu
def test_linear_of_many_rows_under_autocast():
    """Float products of many rows are the library's to round there."""
    from jacobiforcing_amd import layer_ops as LO
    x, w = torch.randn(640, 64, device="cuda"), torch.randn(2500, 64, device="cuda")
    assert LO.linear_split(640, 64, 2500)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y, want = LO.linear(x, w), torch.nn.functional.linear(x, w)
    assert y.dtype == want.dtype == torch.bfloat16 and torch.equal(y, want) and LO.linear(x, w).dtype == torch.float32


@pytest.mark.gpu
def test_other_threads_run_beside_a_launch(tmp_path):
    """A launch that waits (for a full queue, here by sleeping) holds no lock that other threads of the program need."""
    import ctypes as C
    import importlib.machinery
    import importlib.util
    import shutil
    import subprocess
    import threading
    import time
    from jacobiforcing_amd import _build, _native as N, layer_ops as LO
    (tmp_path / "wait.c").write_text("#include <unistd.h>\nint wait_in_a_launch() { usleep(500000); return 0; }\n")
    subprocess.check_call([shutil.which("gcc") or "cc", "-shared", "-fPIC", "-O1", str(tmp_path / "wait.c"), "-o", str(tmp_path / "wait.so")])
    wait = C.CDLL(str(tmp_path / "wait.so"))
    own = shutil.copy(_build.host_lib(), tmp_path / "own.so")                                   # a module of its own: the package's keeps its launches
    loader = importlib.machinery.ExtensionFileLoader("_jl_host", str(own))
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_jl_host", loader))
    loader.exec_module(module)
    L, address = N.layers(), lambda f: C.cast(f, C.c_void_p).value
    symbols = {name: address(getattr(L, name)) for name in module.symbols()}
    symbols["jl_last_error"], symbols["jl_last_error of the recurrences"] = (address(L._library(name).jl_last_error) for name in ("jl_linear_small", "jl_linear_scan"))
    symbols["jl_linear_small"] = address(wait.wait_in_a_launch)
    module.bind(symbols, LO.LINEAR_SMALL_ROWS, LO.LINEAR_ONE_TILE, LO.LINEAR_X_BYTES)
    x, w = torch.zeros(4, 64, device="cuda"), torch.zeros(64, 64, device="cuda")
    taken = []
    thread = threading.Thread(target=lambda: taken.append(module.linear(x, w, None, None)))
    last, longest, alive = time.monotonic(), 0.0, True
    thread.start()
    while alive:
        alive, now = thread.is_alive(), time.monotonic()
        last, longest = now, max(longest, now - last)
    assert torch.is_tensor(taken[0]) and longest < 0.25, longest
