"""The GEMMs as PyTorch custom operators (`torch.ops.streamk.*`): the boundary the reference reaches with
`@jit(out_idx=[2])`, which wraps its kernel as `f(A, B) -> C` (autotune/streamk_fp16_autotune.py:93-94).

CPU part: the operators are registered with the schemas the wrappers rely on, and their fake
implementations give the result's shape and dtype without touching a device.  GPU part: the operator
returns the bits of a direct C-ABI call, traces under torch.compile without a graph break, and passes
torch.library.opcheck.
"""
import ctypes

import numpy as np
import pytest


@pytest.fixture(scope="module")
def sk():
    import streamk
    return streamk


def test_operators_are_registered_with_fake_implementations(sk):
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    ops = torch.ops.streamk
    for name in ("gemm_f16", "gemm_bf16", "gemm_f32", "gemm_q4", "gemm_f8", "gemm_i8", "dequant_q4"):
        schema = str(getattr(ops, name).default._schema)
        assert schema.endswith("-> Tensor"), schema
        out_schema = str(getattr(ops, name + "_out").default._schema)
        assert "Tensor(a!) out" in out_schema and out_schema.endswith("-> ()"), out_schema
    with FakeTensorMode():
        h = lambda *s: torch.empty(*s, dtype=torch.float16, device="cuda")  # noqa: E731
        C = ops.gemm_f16(h(5, 64), h(32, 64))
        assert C.shape == (5, 32) and C.dtype == torch.float16 and C.device.type == "cuda" and C.stride() == (32, 1)
        assert ops.gemm_f16(h(5, 64), h(64, 32), "nn").shape == (5, 32)
        assert ops.gemm_bf16(h(5, 64).bfloat16(), h(32, 64).bfloat16()).dtype == torch.bfloat16
        assert ops.gemm_f32(h(5, 64).float(), h(64, 32).float()).shape == (5, 32)
        Wq = torch.empty(48, 128, dtype=torch.uint8, device="cuda")
        C = ops.gemm_q4(h(3, 256), Wq, h(48, 2), None)
        assert C.shape == (3, 48) and C.dtype == torch.float16
        assert ops.dequant_q4(Wq, h(48, 2), None).shape == (48, 256)
        i8 = torch.empty(7, 64, dtype=torch.int8, device="cuda")
        assert ops.gemm_i8(i8, i8).dtype == torch.int32 and ops.gemm_i8(i8, i8).shape == (7, 7)
        f8 = torch.empty(7, 64, dtype=torch.uint8, device="cuda")
        assert ops.gemm_f8(f8, f8).dtype == torch.float16
        assert ops.gemm_f16_out(h(5, 64), h(32, 64), h(5, 32)) is None


def test_configuration_strings_round_trip(sk):
    import sys
    ops = sys.modules["streamk.ops"]
    text = ops._config_string(None, dict(bm=128, schedule="basic"), dict(grid=40, fixup=None))
    assert text == "bm=128;grid=40;schedule=basic"
    assert ops._parse_config(text) == dict(bm=128, grid=40, schedule="basic")
    assert ops._config_string(None, None, {}) == ""


def test_text_that_is_no_configuration_is_refused(sk):
    import sys
    ops = sys.modules["streamk.ops"]
    for text in ("long rows", "splitk", "bm"):
        for M in (1, 24, 200):
            with pytest.raises(ValueError):
                ops._plan_for(text, M, 2048, 2048, "float16", "nt")


@pytest.mark.gpu
def test_operator_equals_direct_c_abi_call(sk):
    """torch.ops.streamk.gemm_f16(A, B) against sk_gemm_f16 called by hand with the same plan, workspace
    rules and stream: the same bits (data-parallel, and the ordered reduce)."""
    import sys
    import torch
    L = sk.lib()
    rng = np.random.default_rng(5)
    M, N, K = 300, 520, 1024
    A = torch.from_numpy((rng.random((M, K), dtype=np.float32) * 2 - 1).astype(np.float16)).cuda()
    B = torch.from_numpy((rng.random((N, K), dtype=np.float32) * 2 - 1).astype(np.float16)).cuda()
    for cfg in (dict(bm=128, bn=128, bk=64, schedule="dp"), dict(bm=128, bn=128, bk=64, schedule="basic", fixup="reduce", grid=24)):
        plan = sk.make_plan(M, N, K, "float16", "nt", cfg)
        ws = torch.zeros(max(int(plan.workspace_bytes), 256), dtype=torch.uint8, device="cuda")
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert L.sk_workspace_init(ws.data_ptr(), ws.numel(), stream) == 0
        C0 = torch.empty(M, N, dtype=torch.float16, device="cuda")
        rc = L.sk_gemm_f16(A.data_ptr(), B.data_ptr(), C0.data_ptr(), M, N, K, K, K, N, ctypes.byref(plan),
                           ws.data_ptr(), ws.numel(), stream)
        assert rc == 0
        assert L.sk_workspace_release(ws.data_ptr()) == 0
        text = sys.modules["streamk.ops"]._config_string(None, cfg, {})
        C1 = torch.ops.streamk.gemm_f16(A, B, "nt", text)
        C2 = torch.empty_like(C0)
        assert torch.ops.streamk.gemm_f16_out(A, B, C2, "nt", text) is None
        C3 = sk.streamk_fp16(A, B, **cfg)
        torch.cuda.synchronize()
        assert torch.equal(C0, C1) and torch.equal(C0, C2) and torch.equal(C0, C3), cfg
    sk.workspace_status()


@pytest.mark.gpu
def test_empty_batch_returns_an_empty_result(sk):
    """No rows of A: the operators return an empty C without a launch (torch.nn.Linear does the same); a wrong
    `out` is still refused."""
    import torch
    A = torch.empty(0, 256, dtype=torch.float16, device="cuda")
    B = torch.randn(72, 256, device="cuda").half()
    C = torch.ops.streamk.gemm_f16(A, B)
    assert C.shape == (0, 72) and C.dtype == torch.float16
    assert sk.streamk_fp16(A, B).shape == (0, 72)
    lin = sk.StreamKLinear.from_linear(torch.nn.Linear(256, 72).cuda().half())
    assert lin(A).shape == (0, 72) and lin(A.reshape(0, 3, 256)).shape == (0, 3, 72)
    out = torch.empty(0, 72, dtype=torch.float16, device="cuda")
    assert torch.ops.streamk.gemm_f16_out(A, B, out) is None
    with pytest.raises(ValueError):
        torch.ops.streamk.gemm_f16_out(A, B, torch.empty(1, 72, dtype=torch.float16, device="cuda"))


@pytest.mark.gpu
def test_linear_module_compiles_without_a_graph_break(sk):
    import torch
    import torch._dynamo
    torch.manual_seed(3)
    K, H = 1024, 1536
    layers = torch.nn.Sequential(
        sk.StreamKLinear.from_linear(torch.nn.Linear(K, H, bias=True).cuda().half(), activation="silu"),
        sk.StreamKLinear.from_linear(torch.nn.Linear(H, K, bias=True).cuda().half(), weight_format="q4"),
        sk.StreamKLinear.from_linear(torch.nn.Linear(K, H, bias=False).cuda().half(), weight_format="q4_zp"))
    x = torch.randn(2, 3, K, device="cuda").half()
    want = layers(x)
    torch._dynamo.reset()
    explained = torch._dynamo.explain(layers)(x)
    assert explained.graph_break_count == 0, explained.break_reasons
    assert explained.graph_count == 1
    compiled = torch.compile(layers, fullgraph=True, backend="aot_eager")
    got = compiled(x)
    assert got.shape == (2, 3, H) and torch.equal(got, want)
    got2 = compiled(torch.randn(5, K, device="cuda").half())   # another M: a new trace, still one graph
    assert got2.shape == (5, H)
    torch.cuda.synchronize()
    sk.workspace_status()


@pytest.mark.gpu
def test_operators_pass_opcheck(sk):
    """torch.library.opcheck: schema (the functional forms mutate nothing, the _out forms only `out`), fake
    implementation against the real one (shape, dtype, strides, device), and tracing through AOT dispatch."""
    import torch
    from torch.library import opcheck
    rng = np.random.default_rng(9)
    h = lambda *s: torch.from_numpy((rng.random(s, dtype=np.float32) * 2 - 1).astype(np.float16)).cuda()  # noqa: E731
    ops = torch.ops.streamk
    A, B = h(40, 256), h(72, 256)
    tests = ("test_schema", "test_faketensor", "test_aot_dispatch_static", "test_aot_dispatch_dynamic")
    opcheck(ops.gemm_f16.default, (A, B), test_utils=tests)
    opcheck(ops.gemm_f16.default, (A, h(256, 72), "nn", "bm=128;bn=128;schedule=basic;grid=6", h(72), "relu"), test_utils=tests)
    opcheck(ops.gemm_f16_out.default, (A, B, torch.empty(40, 72, dtype=torch.float16, device="cuda")), test_utils=tests)
    opcheck(ops.gemm_bf16.default, (A.bfloat16(), B.bfloat16()), test_utils=tests)
    opcheck(ops.gemm_f32.default, (A.float(), h(256, 72).float()), test_utils=tests)
    Wq = torch.from_numpy(rng.integers(0, 256, (72, 128), dtype=np.uint8)).cuda()
    sc = torch.from_numpy(rng.uniform(0.005, 0.02, (72, 2)).astype(np.float16)).cuda()
    opcheck(ops.gemm_q4.default, (h(4, 256), Wq, sc, None), test_utils=tests)
    opcheck(ops.gemm_q4_out.default, (h(4, 256), Wq, sc, None, torch.empty(4, 72, dtype=torch.float16, device="cuda")),
            test_utils=tests)
    opcheck(ops.dequant_q4.default, (Wq, sc, None), test_utils=tests)
    i8 = torch.from_numpy(rng.integers(-128, 128, (40, 256), dtype=np.int8)).cuda()
    opcheck(ops.gemm_i8.default, (i8, i8), test_utils=tests)
    # (raw bytes: opcheck perturbs its inputs with arithmetic torch does not have for its float8 types)
    f8a, f8b = A.to(torch.float8_e4m3fn).view(torch.uint8), B.to(torch.float8_e4m3fn).view(torch.uint8)
    opcheck(ops.gemm_f8.default, (f8a, f8b, 0.5, "e4m3"), test_utils=tests)
    torch.cuda.synchronize()
    sk.workspace_status()


def _calls_of(fn):
    """The streamk operators a call goes through, and its result or the type of its exception."""
    import torch
    with torch.autograd.profiler.profile() as prof:
        try:
            out = fn()
        except Exception as e:  # noqa: BLE001
            out = type(e)
    return [e.name.split("::")[1] for e in prof.function_events if e.name.startswith("streamk::")], out


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["gemm_f16", "gemm_bf16", "gemm_f32", "gemm_f8", "gemm_i8", "gemm_q4"])
def test_native_operators_answer_like_the_general_ones(name):
    """Calls of every form, twice each: by the operator -- natively once its plan is known -- and by the Python
    implementation it stands in for.  Same bits, or the same exception; ordinary forms run natively from the second call
    on, the others never do."""
    import torch
    import streamk
    ops = torch.ops.streamk
    op, general = getattr(ops, name), getattr(ops, name + "_general")
    out_op, out_general = getattr(ops, name + "_out"), getattr(ops, name + "_out_general")
    torch.manual_seed(5)
    M, N, K = 5, 264, 384
    kind = {"gemm_f16": torch.float16, "gemm_bf16": torch.bfloat16, "gemm_f32": torch.float32, "gemm_f8": torch.float8_e4m3fn,
            "gemm_i8": torch.int8, "gemm_q4": torch.float16}[name]
    ctype = {"gemm_f8": torch.float16, "gemm_i8": torch.int32}.get(name, kind)

    def mat(rows, cols):
        if kind == torch.int8:
            return torch.randint(-9, 10, (rows, cols), device="cuda", dtype=kind)
        return torch.randint(-3, 4, (rows, cols), device="cuda").float().to(kind)

    A, big = mat(M, K), mat(M + 2, K + 64)
    q4 = name == "gemm_q4"
    Wq = torch.randint(0, 256, (N, K // 2), device="cuda", dtype=torch.uint8)
    sc, zp = torch.rand(N, K // 128, device="cuda").half(), torch.randint(0, 16, (N, K // 128), device="cuda").half()
    weights = (Wq, sc, None) if q4 else (mat(N, K),)
    bias = torch.randint(-5, 6, (N,), device="cuda").to(ctype)
    lead = {"gemm_f8": (0.5, ""), "gemm_q4": (8, 128, False)}.get(name, () if name == "gemm_i8" else ("nt",))
    epi = (bias, "relu") if name not in ("gemm_f32", "gemm_i8") else ()
    ordinary = [(A, *weights, *lead), (A[:1], *weights, *lead), (big[1:1 + M, 16:16 + K], *weights, *lead)]
    other = [(A[:0], *weights, *lead),                                              # no rows
             (A.cpu(), *weights, *lead), (A.double(), *weights, *lead), (A[:, :-128], *weights, *lead),   # refused
             (A.t(), *weights, *lead), (A[0], *weights, *lead), (A, *weights, *lead, "schedule=dp")]
    if epi:
        ordinary += [(A, *weights, *lead, "", *epi), (A, *weights, *lead, "", None, "silu")]
        other += [(A, *weights, *lead, "", bias[:-1], "none"), (A, *weights, *lead, "", None, "tanh"),
                  (A, *weights, *lead, "", bias.double(), "none")]
    if name in ("gemm_f16", "gemm_bf16", "gemm_f32"):
        ordinary += [(A, mat(K, N), "nn"), (A, mat(N, K + 8)[:, :K], "nt")]
        other += [(A, mat(N, K), "tn")]
    if kind in (torch.float16, torch.bfloat16):
        other += [(big[:M, 1:1 + K], *weights, *lead)]                              # copied before the launch
    if name == "gemm_f8":
        ordinary += [(A, *weights, 0.25, "e4m3")]
        other += [(A, *weights, 0.25, "e5m2"), (A.view(torch.uint8), weights[0].view(torch.uint8), 1.0, "e4m3"), (A, *weights, float("nan"), "")]
    if q4:
        ordinary += [(A, Wq, sc, zp), (A, Wq, sc, None, 3), (torch.randn(80, K, device="cuda").half(), Wq, sc, None),
                     (torch.randn(80, K, device="cuda").half(), Wq, sc, zp)]
        other += [(A, Wq, sc, zp.to(torch.uint8)), (A, Wq, sc, zp[:, :2]), (A, Wq, sc, None, 16), (A, Wq, sc, None, 8, 64),
                  (A, Wq.t().contiguous().t(), sc, None), (A, streamk.tile_q4(Wq), sc, None, 8, 128, True),
                  (torch.randn(1100, K, device="cuda").half(), Wq, sc, None)]

    def same(a, b):
        return a is b if isinstance(a, type) or isinstance(b, type) else (a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b))

    n_operands = 4 if q4 else 2
    for native, args in [(True, x) for x in ordinary] + [(False, x) for x in other]:
        if q4 and len(args) < 4:
            args = args + (None,)
        _, want = _calls_of(lambda: general(*args))
        _, first = _calls_of(lambda: op(*args))
        names, got = _calls_of(lambda: op(*args))
        text = [tuple(a.shape) if isinstance(a, torch.Tensor) else a for a in args]
        assert same(first, want) and same(got, want), (text, want, got)
        if isinstance(want, torch.Tensor) and native:
            assert names == [name], (text, names)
        elif not native:
            assert names[:1] == [name] and (name + "_general" in names or isinstance(want, type)), (text, names)
        if isinstance(want, torch.Tensor):   # into a caller's C, rows further apart than they are long
            C = torch.full((want.shape[0], want.shape[1] + 8), 7, device="cuda", dtype=ctype)
            out_op(*args[:n_operands], C[:, :-8], *args[n_operands:])
            assert torch.equal(C[:, :-8], want) and (C[:, -8:] == 7).all(), text
            bad = torch.empty(want.shape[0] + 1, want.shape[1], device="cuda", dtype=ctype)
            assert _calls_of(lambda: out_op(*args[:n_operands], bad, *args[n_operands:]))[1] is \
                _calls_of(lambda: out_general(*args[:n_operands], bad, *args[n_operands:]))[1]
    # workspaces taken back: the general implementation makes a new one where the plan needs it
    streamk.reset_workspaces()
    for args in ordinary:
        assert torch.equal(op(*args, *((None,) if q4 and len(args) < 4 else ())), general(*args, *((None,) if q4 and len(args) < 4 else ())))
    # another stream, a graph, and a tuned cache that changed
    args = ordinary[0]
    want = general(*args)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = op(*args)
    s.synchronize()
    assert torch.equal(got, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        got = op(*args)
    for _ in range(3):
        torch.cuda.synchronize()
        got.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    streamk.plan.invalidate_tuned_cache()
    names, got = _calls_of(lambda: op(*args))
    assert names == [name, name + "_general"] and torch.equal(got, want)
    if kind.is_floating_point and kind != torch.float8_e4m3fn:   # an input that requires a gradient: the result as it was
        x = args[0].clone().requires_grad_()
        assert op(x, *args[1:]).requires_grad == general(x, *args[1:]).requires_grad
    streamk.workspace_status()


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", ["float16", "bfloat16", "q4", "q4_zp"])
def test_a_layers_plan_is_what_its_call_runs(sk, fmt, monkeypatch):
    """StreamKLinear.plan_for against the plan that forward's operator call asks for, on either side of 16, 64, 128, 256 and 512
    rows; a plan of the layer's own type also where forward dequantises the weights first."""
    import sys
    import torch
    ops = sys.modules["streamk.ops"]
    layer = sk.StreamKLinear(1024, 3584, weight_format=fmt, device="cuda")
    sk.plan.invalidate_tuned_cache()   # (a call goes through Python until its plan is known)
    asked, plan_for = [], ops._plan_for

    def recorded(*args):
        asked.append(plan_for(*args))
        return asked[-1]
    for M in (1, 4, 17, 40, 64, 65, 128, 200, 257, 520, 1100):
        with monkeypatch.context() as m:
            m.setattr(ops, "_plan_for", recorded)
            layer(torch.zeros(M, 1024, dtype=layer.dtype, device="cuda"))
        plan, ran = layer.plan_for(M), asked[-1]
        if M == 1100 and fmt in ("q4", "q4_zp"):
            assert ran.dtype != plan.dtype and (plan.M, plan.N, plan.K) == (M, 3584, 1024)
        else:
            assert (plan.kernel_id, plan.grid, plan.dtype) == (ran.kernel_id, ran.grid, ran.dtype), (fmt, M)
    # the plan of a launch with zero points that the operator would not take leaves its way alone
    if fmt == "q4_zp":
        x = torch.randn(520, 1024, device="cuda").half()
        wide = sk.StreamKLinear(1024, 64 * 300, weight_format=fmt, device="cuda")
        wide.scales.fill_(1.0)
        first = wide(x)
        wide.plan_for(520)
        names, again = _calls_of(lambda: wide(x))
        assert "gemm_q4_general" in names and torch.equal(first, again)


def test_where_zero_points_are_dequantised_first(sk, monkeypatch):
    """Sizes on either side of each limit, as they measured."""
    import sys
    ops = sys.modules["streamk.ops"]
    monkeypatch.setattr(sk.plan, "num_cus", lambda: 256)
    first = lambda *size: ops._dequantises(*size, True)   # noqa: E731
    for size in ((512, 8192, 8192), (768, 4096, 11008), (517, 3072, 9472), (700, 2560, 14336), (849, 1832, 8320), (1025, 256, 128)):
        assert first(*size), size
    for size in ((512, 4096, 4096), (320, 8192, 8192), (500, 4096, 11008), (510, 6048, 7040), (656, 2560, 2304), (256, 28672, 8192)):
        assert not first(*size), size
    assert not ops._dequantises(1024, 28672, 8192, False) and ops._dequantises(1025, 256, 128, False)


def test_a_configuration_without_a_plan_is_asked_for_once(sk, monkeypatch):
    """Per-group zero points with more than 64 rows ask on every call whether one launch runs the configuration."""
    import sys
    ops = sys.modules["streamk.ops"]
    asked = []

    def make_plan(*args):
        asked.append(args)
        raise sk.StreamKError(-4, "no kernel")
    monkeypatch.setattr(ops, "make_plan", make_plan)
    monkeypatch.setattr(ops, "_without_plan", set())
    for _ in range(3):
        assert not ops._has_plan("schedule=dp", 100, 1024, 1024, "q4_zp", 2048, 512)
    assert len(asked) == 1
    assert not ops._has_plan("schedule=dp", 101, 1024, 1024, "q4_zp", 2048, 512) and len(asked) == 2


# (two shapes per operator whose plans split tiles: one that the smallest workspace serves, one that it does not)
_SPLIT_SHAPES = {"gemm_f16": ("float16", (64, 256, 4096), (100, 4096, 8192)), "gemm_bf16": ("bfloat16", (64, 256, 4096), (100, 4096, 8192)),
                 "gemm_f32": ("float32", (16, 256, 2048), (512, 1024, 4096)), "gemm_f8": ("float8_e4m3", (64, 256, 8192), (300, 1024, 16384)),
                 "gemm_i8": ("int8", (64, 256, 8192), (300, 1024, 16384)), "gemm_q4": ("q4", (64, 256, 4096), (300, 1024, 8192))}


def test_split_shapes_need_the_workspaces_they_stand_for(sk):
    for dtype, small, large in _SPLIT_SHAPES.values():
        sizes = [sk.make_plan(*shape, dtype, "nt", sk.plan.operator_config(*shape, dtype, "nt"), cus=256).workspace_bytes for shape in (small, large)]
        assert 0 < sizes[0] <= 1 << 20 < sizes[1], (dtype, sizes)


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(_SPLIT_SHAPES))
def test_native_operators_with_a_workspace(name):
    """Calls whose plans split tiles: natively from the second call on, on the workspace that the Python layer owns -- after
    it was taken back, after it grew and for the smaller plan on the grown one, on a stream of its own, replayed from a
    graph between eager calls, and with another thread's calls on the same stream.  Bits as the general implementation."""
    import sys
    import threading
    import torch
    import streamk
    dtype, *shapes = _SPLIT_SHAPES[name]
    op, general = getattr(torch.ops.streamk, name), getattr(torch.ops.streamk, name + "_general")
    torch.manual_seed(6)
    kind = {"q4": torch.float16, "float8_e4m3": torch.float8_e4m3fn}.get(dtype, getattr(torch, dtype, None))
    calls, wants = [], []
    for M, N, K in shapes:
        plan = sys.modules["streamk.ops"]._plan_for("", M, N, K, dtype, "nt")
        assert plan.workspace_bytes > (0 if not calls else 1 << 20)
        A = torch.randint(-3, 4, (M, K), device="cuda").float().to(kind)
        if name == "gemm_q4":
            args = (A, torch.randint(0, 256, (N, K // 2), device="cuda", dtype=torch.uint8), torch.rand(N, K // 128, device="cuda").half(), None)
        else:
            args = (A, torch.randint(-3, 4, (N, K), device="cuda").float().to(kind)) + (("nt",) if kind != torch.float8_e4m3fn and name != "gemm_i8" else ())
        calls.append(args)
    streamk.reset_workspaces()
    wants = [general(*args) for args in calls]

    def check(args, want, native):
        names, got = _calls_of(lambda: op(*args))
        assert names == ([name] if native else [name, name + "_general"]), names
        assert torch.equal(got, want)

    small, large = zip(calls, wants)
    for _ in range(2):
        streamk.reset_workspaces()
        check(*small, False)    # nothing to launch with: the general implementation makes a workspace
        check(*small, True)
        check(*large, False)    # too small: it makes a larger one
        check(*large, True)
        check(*small, True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        check(*large, False)
        check(*small, True)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        got = op(*small[0])
    for _ in range(3):
        got.zero_()
        check(*large, True)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, small[1])
    # two threads on one stream: both run natively on its workspace, one behind the other
    wrong = []

    def calls_of_a_thread(args, want):
        for _ in range(20):
            if not torch.equal(op(*args), want):
                wrong.append(args[0].shape)

    threads = [threading.Thread(target=calls_of_a_thread, args=pair) for pair in (small, large)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong
    streamk.workspace_status()


_WITHOUT_NATIVE = """
import ctypes, sys, warnings
import torch
load = ctypes.CDLL
def refuse(name, *args, **kwargs):
    if str(name).endswith("libstreamk_torch.so"):
        raise OSError("undefined symbol: of another libtorch")
    return load(name, *args, **kwargs)
ctypes.CDLL = refuse
with warnings.catch_warnings(record=True) as caught:
    warnings.simplefilter("always")
    sys.path.insert(0, sys.argv[1])
    import streamk
assert [w for w in caught if w.category is RuntimeWarning and "another libtorch" in str(w.message)], caught
for name in ("gemm_f16", "gemm_bf16", "gemm_f32", "gemm_f8", "gemm_i8", "gemm_q4"):
    for op in (name, name + "_out", name + "_general", name + "_out_general"):
        assert torch._C._dispatch_has_kernel_for_dispatch_key("streamk::" + op, "CUDA"), op
assert streamk.make_plan(100, 512, 8192, "float16", "nt", cus=256).workspace_bytes > 0
streamk.plan.invalidate_tuned_cache()
streamk.reset_workspaces()
if sys.argv[2:] == ["gpu"]:
    A = torch.randint(-3, 4, (100, 8192), device="cuda").half()
    B = torch.randint(-1, 2, (512, 8192), device="cuda").half()
    for _ in range(2):
        assert torch.equal(streamk.streamk_fp16(A, B), (A.float() @ B.float().T).half())
    streamk.reset_workspaces()
    assert torch.equal(streamk.streamk_fp16(A, B, out=torch.empty(100, 512, device="cuda").half()), (A.float() @ B.float().T).half())
print("answered")
"""


@pytest.mark.parametrize("where", ["host", pytest.param("gpu", marks=pytest.mark.gpu)])
def test_operators_without_their_native_library(where):
    """libstreamk_torch.so built against another libtorch: the package imports with a warning and the operators answer from
    their Python implementations, on the kernels as ever."""
    import os
    import subprocess
    import sys
    package = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stream-k.tvm_amd")
    done = subprocess.run([sys.executable, "-c", _WITHOUT_NATIVE, package] + (["gpu"] if where == "gpu" else []), capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and done.stdout.strip().endswith("answered"), done.stderr[-2000:]
