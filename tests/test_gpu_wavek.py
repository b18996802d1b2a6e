"""Tiles whose waves stream K on their own (tile_wavek.h, tile_wavek_q4.h): every tile of every type on operands whose sums are
exact in fp32, so that results are equal to the bit whatever the order of the sums; and the operators' choice of them against
the kernels that plans take."""
import numpy as np
import pytest

_TILES = [(32, 32), (32, 64), (64, 32), (64, 48), (64, 64), (64, 80), (64, 96), (64, 112), (64, 128), (96, 32), (96, 64), (128, 32),
          (128, 48), (128, 64)]
_TILES_NN = [(32, 32), (32, 64), (32, 128), (64, 32), (64, 64), (96, 64), (128, 32)]
_TILES_Q4 = [(32, 32), (32, 64), (64, 32), (64, 64), (64, 96), (128, 32)]


@pytest.fixture(scope="module")
def sk():
    import streamk
    return streamk


def _small(rng, shape, most=2):
    return rng.integers(-most, most + 1, shape).astype(np.float64)


def _operands(torch, dtype, rng, M, N, K, pad=0, layout="nt"):
    """A call on A (rows `pad` elements further apart, which hold what would show) and weights, and the exact product."""
    if dtype.startswith("q4"):
        A = _small(rng, (M, K))
        q = rng.integers(0, 16, (N, K))
        zeros = rng.integers(0, 16, (N, K // 128)) if dtype == "q4_zp" else np.full((N, K // 128), 8)
        scales = 2.0 ** rng.integers(-4, -1, (N, K // 128))
        W = (q - np.repeat(zeros, 128, 1)) * np.repeat(scales, 128, 1)
        Wq = torch.from_numpy((q[:, 0::2] | q[:, 1::2] << 4).astype(np.uint8)).cuda()
        ds, dz = torch.from_numpy(scales).half().cuda(), torch.from_numpy(zeros).half().cuda() if dtype == "q4_zp" else None
        kind, rest = torch.float16, (Wq, ds)
    else:
        A, W = _small(rng, (M, K)), _small(rng, (N, K))
        kind = {"float8_e4m3": torch.float8_e4m3fn, "float8_e5m2": torch.float8_e5m2}.get(dtype) or getattr(torch, dtype)
        rest = (torch.from_numpy(W if layout == "nt" else W.T.copy()).float().cuda().to(kind),)
    dA = torch.full((M, K + pad), float("nan"), device="cuda").to(kind) if kind != torch.int8 else torch.full((M, K + pad), 77, device="cuda", dtype=kind)
    dA[:, :K].copy_(torch.from_numpy(A).float().cuda().to(kind))
    import streamk
    f = {"float16": streamk.streamk_fp16, "bfloat16": streamk.streamk_bf16, "int8": streamk.streamk_int8}.get(dtype)
    if dtype in ("float16", "bfloat16"):
        call = lambda **kw: f(dA[:, :K], rest[0], layout=layout, **kw)   # noqa: E731
    elif dtype == "int8":
        call = lambda **kw: f(dA[:, :K], rest[0], **kw)   # noqa: E731
    elif dtype.startswith("float8"):
        call = lambda **kw: streamk.streamk_fp8(dA[:, :K], rest[0], **kw)   # noqa: E731
    else:
        call = lambda **kw: streamk.streamk_q4(dA[:, :K], rest[0], rest[1], zeros=dz, **kw)   # noqa: E731
    return call, A @ W.T


def _rounded(torch, exact, dtype):
    if dtype == "int8":
        return torch.from_numpy(exact).to(torch.int32)
    return torch.from_numpy(exact).float().to(torch.bfloat16 if dtype == "bfloat16" else torch.float16)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,layout", [("float16", "nt"), ("bfloat16", "nt"), ("float8_e4m3", "nt"), ("float8_e5m2", "nt"), ("int8", "nt"),
                                          ("q4", "nt"), ("q4_zp", "nt"), ("float16", "nn"), ("bfloat16", "nn")])
def test_every_tile_is_exact(sk, dtype, layout):
    import torch
    rng = np.random.default_rng(41)
    step = 128 if dtype.startswith("q4") else (16 if "8" in dtype and dtype != "bfloat16" and dtype != "float16" else 8)
    long = {128: 6528, 16: 5136, 8: 2568}[step]   # rings full, iterations that K does not fill, odd numbers of them
    for bm, bn in _TILES_Q4 if dtype.startswith("q4") else (_TILES if layout == "nt" else _TILES_NN):
        for M, N, K in ((bm + 1, 2 * bn + 8, long), (1, 1 if layout == "nt" else 8, step), (2 * bm - 3, bn + (5 if layout == "nt" else 8), 3 * step + (128 if step < 128 else 0)), (bm, 3 * bn, 2048)):
            call, exact = _operands(torch, dtype, rng, M, N, K, pad=8 if dtype in ("float16", "bfloat16") or step == 128 else 16, layout=layout)
            want = _rounded(torch, exact, dtype)
            for sched in (dict(schedule="dp"), dict(schedule="splitk", split=2, fixup="reduce"), dict(schedule="basic", grid=7, fixup="reduce"),
                          dict(schedule="basic", grid=5, fixup="atomic")):
                try:
                    plan = sk.make_plan(M, N, K, dtype, layout, dict(sched, bm=bm, bn=bn, variant=11))
                except sk.StreamKError:
                    assert sched["schedule"] == "splitk"   # (a split that does not divide the iterations)
                    continue
                assert sk.kernel_name(plan.kernel_id).startswith("wavek_")
                got = call(plan=plan).cpu()
                assert torch.equal(got, want), (dtype, bm, bn, M, N, K, sched, (got != want).sum().item())
            if dtype != "int8":
                kind = torch.bfloat16 if dtype == "bfloat16" else torch.float16
                bias = torch.from_numpy(rng.integers(-8, 9, N).astype(np.float32)).to(kind)
                plan = sk.make_plan(M, N, K, dtype, layout, dict(bm=bm, bn=bn, variant=11, schedule="dp"))
                got = call(plan=plan, bias=bias.cuda(), activation="relu").cpu()
                want = _rounded(torch, np.maximum(exact + bias.double().numpy(), 0), dtype)
                assert torch.equal(got, want), (dtype, bm, bn, M, N, K)
    sk.workspace_status()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float8_e4m3", "int8", "q4"])
def test_alignments_of_the_epilogue(sk, dtype):
    """C and the bias at every alignment that decides how they are accessed, by tiles with pieces of eight and of four columns,
    as whole tiles in one round and through the fix-up."""
    import torch
    rng = np.random.default_rng(43)
    for bm, bn in ((64, 64), (32, 32), (96, 64)) if dtype != "q4" else ((64, 64), (32, 32), (64, 96)):
        for N in (4 * bn, bn + 4, bn + 13):
            M, K = bm + 5, 2048
            call, exact = _operands(torch, dtype, rng, M, N, K)
            kind = torch.bfloat16 if dtype == "bfloat16" else torch.float16
            values = torch.from_numpy(rng.integers(-8, 9, N).astype(np.float32)).to(kind)
            for sched in (dict(schedule="dp"), dict(schedule="basic", grid=5, fixup="reduce")):
                plan = sk.make_plan(M, N, K, dtype, "nt", dict(sched, bm=bm, bn=bn, variant=11))
                for at, ldc in ((0, N), (0, (N + 7) // 8 * 8), (4, (N + 7) // 8 * 8 + 4), (1, N + 1), (8, (N + 7) // 8 * 8 + 1)):
                    for bias_at in (0, 4, 1) if dtype != "int8" else (None,):
                        bias = None
                        if bias_at is not None:
                            bias = torch.zeros(N + bias_at, dtype=kind, device="cuda")[bias_at:]
                            bias.copy_(values)
                        want = _rounded(torch, exact if bias is None else exact + values.double().numpy(), dtype)
                        buf = torch.zeros(at + M * ldc, dtype=want.dtype, device="cuda")
                        out = buf[at:].view(M, ldc)[:, :N]
                        call(plan=plan, out=out, **({} if bias is None else {"bias": bias}))
                        assert torch.equal(out.cpu(), want), (dtype, bm, bn, N, sched, at, ldc, bias_at)
                        assert not buf[:at].any() and not buf[at:].view(M, ldc)[:, N:].any(), (dtype, bm, bn, N, sched, at, ldc, bias_at)
    sk.workspace_status()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,layout", [("float16", "nt"), ("bfloat16", "nt"), ("float8_e4m3", "nt"), ("int8", "nt"), ("q4", "nt"), ("q4_zp", "nt"),
                                          ("float16", "nn"), ("bfloat16", "nn")])
def test_operator_calls_equal_the_plans_they_replace(sk, dtype, layout):
    """What an operator call takes by itself against the plan that make_plan gives (per-group zero points beyond 64 rows: the
    exact product alone), sizes around the limits of the rule, rows of A and C further apart than they are long, C at an odd
    element."""
    import torch
    rng = np.random.default_rng(42)
    step = 128 if dtype.startswith("q4") else (16 if dtype in ("float8_e4m3", "int8") else 8)
    seen = set()
    for M, N, K in ((1, 2048, 1024), (17, 768, 1536), (24, 1290, 1408), (31, 2056, 3200), (33, 770, 6144), (40, 2049, 2048), (64, 1000, 8192), (65, 775, 512), (100, 3001, 1664), (128, 768, 4096),
                    (129, 1031, 640), (257, 2050, 1152), (300, 769, 2304), (513, 801, 384)):
        K, N = K // step * step, N if layout == "nt" else N // 8 * 8
        call, exact = _operands(torch, dtype, rng, M, N, K, pad=8 * (2 if step == 16 else 1), layout=layout)
        want = _rounded(torch, exact, dtype)
        plan = sk.make_plan(M, N, K, dtype, layout, sk.plan.operator_config(M, N, K, dtype, layout))
        seen.add(sk.kernel_name(plan.kernel_id).split("_")[0])
        for _ in range(2):   # (the first call through Python, the second natively)
            assert torch.equal(call().cpu(), want), (dtype, M, N, K, sk.kernel_name(plan.kernel_id))
        if not (dtype == "q4_zp" and M > 64):
            assert torch.equal(call(plan=sk.make_plan(M, N, K, dtype, layout, use_tuned=False)).cpu(), want), (dtype, M, N, K)
        buf = torch.zeros(M * (N + 3) + 1, dtype=want.dtype, device="cuda")
        out = buf[1:].view(M, N + 3)[:, :N]
        call(out=out)
        assert torch.equal(out.cpu(), want) and not buf[1:].view(M, N + 3)[:, N:].any() and not buf[:1].any(), (dtype, M, N, K)
    assert "wavek" in seen, dtype
    sk.workspace_status()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,layout", [("float16", "nt"), ("bfloat16", "nt"), ("float8_e4m3", "nt"), ("q4", "nt"), ("q4_zp", "nt"), ("float16", "nn")])
def test_equal_rows_give_equal_bits(sk, dtype, layout):
    """Rows of A that repeat from one row of tiles to the next, on values whose sums round: every tile of a column adds up K in one
    order, also where a column straddles two XCDs, has more than eight tiles, or a launch several rounds or a fixed split."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(44)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")   # noqa: E731
    kind = {"float8_e4m3": torch.float8_e4m3fn}.get(dtype) or getattr(torch, dtype, torch.float16)
    for bm, bn in ((32, 64), (64, 64), (128, 32)):
        for rows, N, K, split in ((2, 115 * bn, 2048, 1), (3, 41 * bn, 4096, 2), (5, 61 * bn - 8, 1536, 1), (11, 21 * bn, 1024, 1), (7, 90 * bn, 1024, 1)):
            A = normal(bm, K).to(torch.float16).to(kind).repeat(rows, 1) if kind != torch.float8_e4m3fn else normal(bm, K).repeat(rows, 1).to(kind)
            plan = sk.make_plan(rows * bm, N, K, dtype, layout, dict(bm=bm, bn=bn, variant=11, schedule="splitk" if split > 1 else "dp", split=split))
            if dtype.startswith("q4"):
                Wq = torch.randint(0, 256, (N, K // 2), generator=gen, device="cuda", dtype=torch.uint8)
                zeros = torch.randint(0, 16, (N, K // 128), generator=gen, device="cuda").half() if dtype == "q4_zp" else None
                C = sk.streamk_q4(A, Wq, normal(N, K // 128).half(), zeros=zeros, plan=plan)
            elif kind == torch.float8_e4m3fn:
                C = sk.streamk_fp8(A, normal(N, K).to(kind), plan=plan, alpha=0.01)
            else:
                f = sk.streamk_fp16 if kind == torch.float16 else sk.streamk_bf16
                C = f(A, normal(*((N, K) if layout == "nt" else (K, N))).to(kind), layout=layout, plan=plan)
            C = C.view(rows, bm, N)
            assert (C == C[:1]).all(), (dtype, layout, bm, bn, rows, N, K, split, [(C[r] != C[0]).any(0).sum().item() for r in range(rows)])
    sk.workspace_status()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,layout", [("float16", "nt"), ("bfloat16", "nt"), ("float8_e4m3", "nt"), ("float8_e5m2", "nt"), ("q4", "nt"), ("q4_zp", "nt"),
                                          ("float16", "nn"), ("bfloat16", "nn")])
def test_infinities_and_nan_reach_their_own_sums(sk, dtype, layout):
    """Infinities and NaN in A, the weights (Q4: the scales) and between A's rows, on tiles that M, N and K do not fill: the result has
    them where the product has, through whole tiles, fixed splits and both fix-ups."""
    import torch
    rng = np.random.default_rng(47)
    q4 = dtype.startswith("q4")
    kind = {"float8_e4m3": torch.float8_e4m3fn, "float8_e5m2": torch.float8_e5m2}.get(dtype) or getattr(torch, dtype, torch.float16)
    odd = (np.nan,) if dtype == "float8_e4m3" else (np.inf, -np.inf, np.nan)   # (e4m3 has no infinities)
    plain = lambda t: t.float().nan_to_num(1e9, 2e9, 3e9)   # noqa: E731
    for bm, bn in _TILES_Q4 if q4 else (_TILES if layout == "nt" else _TILES_NN):
        M, N, K = bm + 3, 2 * bn + (5 if layout == "nt" else 8), 2176 if q4 else (1088 if kind.itemsize == 2 else 2192)
        A = _small(rng, (M, K))
        for i, (m, k) in enumerate(((0, 0), (M - 1, K - 1), (bm - 1, K // 2))):
            A[m, k] = odd[i % len(odd)]
        dA = torch.full((M, K + 16), float("nan"), device="cuda").to(kind)
        dA[:, :K].copy_(torch.from_numpy(A).float().cuda().to(kind))
        if q4:
            q = rng.integers(0, 16, (N, K))
            zeros = rng.integers(0, 16, (N, K // 128)) if dtype == "q4_zp" else np.full((N, K // 128), 8)
            scales = 2.0 ** rng.integers(-4, -1, (N, K // 128))
            scales[1, 0], scales[N - 1, K // 128 - 1], scales[bn, 2] = odd
            with np.errstate(invalid="ignore"):
                W = (q - np.repeat(zeros, 128, 1)) * np.repeat(scales, 128, 1)
            Wq = torch.from_numpy((q[:, 0::2] | q[:, 1::2] << 4).astype(np.uint8)).cuda()
            kw = dict(zeros=torch.from_numpy(zeros).half().cuda()) if dtype == "q4_zp" else {}
            call = lambda **c: sk.streamk_q4(dA[:, :K], Wq, torch.from_numpy(scales).half().cuda(), **kw, **c)   # noqa: E731
        else:
            W = _small(rng, (N, K))
            for i, (n, k) in enumerate(((1, 0), (N - 1, K - 1), (bn, K // 3))):
                W[n, k] = odd[(i + 1) % len(odd)]
            dB = torch.from_numpy(W if layout == "nt" else W.T.copy()).float().cuda().to(kind)
            f = {torch.float16: sk.streamk_fp16, torch.bfloat16: sk.streamk_bf16}.get(kind)
            call = (lambda **c: f(dA[:, :K], dB, layout=layout, **c)) if f else (lambda **c: sk.streamk_fp8(dA[:, :K], dB, **c))   # noqa: E731
        with np.errstate(invalid="ignore"):
            want = _rounded(torch, A @ W.T, dtype)
        assert want.isnan().any() and want.isfinite().any()
        for sched in (dict(schedule="dp"), dict(schedule="basic", grid=5, fixup="reduce"), dict(schedule="basic", grid=7, fixup="atomic")):
            got = call(plan=sk.make_plan(M, N, K, dtype, layout, dict(sched, bm=bm, bn=bn, variant=11))).cpu()
            assert torch.equal(plain(got), plain(want)), (dtype, layout, bm, bn, sched)
            sk.workspace_status()
            # (the accumulating fix-up leaves its buffers at zero: the next call must not see what this one had)
    call, exact = _operands(torch, dtype, rng, 40, 200, 2048, layout=layout)
    plan = sk.make_plan(40, 200, 2048, dtype, layout, dict(schedule="basic", grid=7, fixup="atomic", bm=32, bn=32, variant=11))
    assert torch.equal(call(plan=plan).cpu(), _rounded(torch, exact, dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn", _TILES_NN)
def test_short_k_over_rows_far_apart(sk, bm, bn):
    """[K, N] weights with fewer K than a chunk has rows and rows so far apart that 32 of them span 4 GiB: what lies past K is not
    read, so infinities of the weights reach only the sums that they belong to."""
    import torch
    rng = np.random.default_rng(45)
    ldb, N = 1 << 26, 2 * bn + 8
    base = torch.zeros(7 * ldb + N, dtype=torch.float16, device="cuda")
    K = 8
    B = base.as_strided((K, N), (ldb, 1))
    values = _small(rng, (K, N))
    values[0, 3], values[2, bn + 1], values[7, N - 1] = np.inf, -np.inf, np.nan
    B.copy_(torch.from_numpy(values).half())
    A = np.abs(_small(rng, (bm + 1, K))) + 1
    want = torch.from_numpy(A @ values).half()
    for sched in (dict(schedule="dp"), dict(schedule="dp", grid=2)):
        plan = sk.make_plan(bm + 1, N, K, "float16", "nn", dict(sched, bm=bm, bn=bn, variant=11))
        got = sk.streamk_fp16(torch.from_numpy(A).half().cuda(), B, layout="nn", plan=plan).cpu()
        assert torch.equal(got.nan_to_num(99.0, 98.0, 97.0), want.nan_to_num(99.0, 98.0, 97.0)), (bm, bn, sched)


def test_the_operators_rule(sk):
    """Plans keep the kernels they had; an operator call takes these where the models say so, never for fix-ups that they do not
    have."""
    wavek = lambda *a, **k: sk.kernel_name(sk.make_plan(*a, cus=256, use_tuned=False, **k).kernel_id).startswith("wavek_")   # noqa: E731
    for dtype in ("float16", "bfloat16", "float8_e4m3", "float8_e5m2", "int8", "q4", "q4_zp"):
        for M, N, K in ((100, 4096, 4096), (256, 4096, 4096), (128, 2048, 2048)):
            assert wavek(M, N, K, dtype, "nt", variant=12), (dtype, M, N, K)
            if dtype == "q4_zp":   # (a plain plan of them has 64 rows at most)
                with pytest.raises(sk.StreamKError):
                    sk.make_plan(M, N, K, dtype, "nt", cus=256, use_tuned=False)
            else:
                assert not wavek(M, N, K, dtype, "nt"), (dtype, M, N, K)
        assert not wavek(16, 4096, 4096, dtype, "nt", variant=12)
        assert wavek(100, 760, 4096, dtype, "nt", variant=12) and wavek(100, 256, 4096, dtype, "nt", variant=12)   # few columns too
        assert wavek(4096, 8192, 8192, dtype, "nt", variant=12) == (dtype == "q4_zp")
    # 17 to 64 rows: few columns, or more than one round of 64-wide tiles where wider ones need one; no depth of K between others is
    # an exception
    for dtype in ("float8_e4m3", "int8", "float16"):
        assert wavek(48, 2048, 5120, dtype, "nt", variant=12) and wavek(24, 20480, 3072, dtype, "nt", variant=12)
        assert wavek(24, 2048, 2048, dtype, "nt", variant=12) and not wavek(24, 11008, 2048, dtype, "nt", variant=12)
        assert wavek(24, 1024, 1024, dtype, "nt", variant=12) == (dtype != "float16")
        assert all(wavek(48, 4096, K, dtype, "nt", variant=12) for K in (4080, 4096, 4352, 4592, 4608))
    # K unsplit on few CUs and rows that are no multiple of 128 bytes: 1.3 to 2.3 times as long as on the streaming kernels
    for dtype in ("float16", "bfloat16"):
        for shape in ((63, 1408, 15096), (44, 1248, 15056), (50, 1152, 6816), (26, 2056, 3752), (19, 1280, 8448), (45, 2128, 8904), (93, 6448, 4600)):
            assert not wavek(*shape, dtype, "nt", variant=12), (dtype, shape)
        # 65 to 96 rows over the width of the 96 x 32 streaming kernel: 80 x 8192 x 8192 38 us on it, 37 on 96 x 32 wave-K tiles, 33 on these
        assert sk.make_plan(80, 8192, 8192, dtype, "nt", cus=256, use_tuned=False, variant=12).bn == 64
    for dtype in ("float16", "bfloat16"):
        for layout in ("nt", "nn"):
            assert not wavek(100, 4096, 4096, dtype, layout, variant=12, fixup="atomic_c")
        assert wavek(1, 4096, 4096, dtype, "nn", variant=12) and wavek(100, 4096, 4096, dtype, "nn", variant=12)
        assert not wavek(1, 4096, 4096, dtype, "nn") and wavek(64, 8192, 8192, dtype, "nn", variant=12)
        assert not wavek(64, 28672, 8192, dtype, "nn", variant=12)
        # weights from HBM: a wide margin while one row of the others' tiles holds them
        assert wavek(320, 4096, 11008, dtype, "nt", variant=12) and not wavek(100, 4096, 11008, dtype, "nt", variant=12)
        assert wavek(80, 5120, 5120, dtype, "nn", variant=12) and not wavek(128, 5120, 5120, dtype, "nn", variant=12)
    assert sk.make_plan(40, 4096, 4096, "q4_zp", "nt", cus=256, use_tuned=False).kernel_id < 400
    # zero points with a long K, and large products that the two models put close to each other: 1.13 to 1.4 times as long
    for shape, dtype in (((23, 10144, 14720), "q4_zp"), ((22, 9360, 12288), "q4_zp"), ((534, 24608, 9056), "int8"), ((307, 10656, 11072), "int8"), ((906, 2912, 8432), "float16")):
        assert not wavek(*shape, dtype, "nt", variant=12), (dtype, shape)
    assert wavek(48, 4096, 11008, "q4_zp", "nt", variant=12) and wavek(209, 5696, 15376, "float8_e4m3", "nt", variant=12)


def test_tiled_weights_take_the_plan_of_row_major_ones(sk):
    """An operator's plan for the tiled layout of Q4 weights, wherever one for the row-major layout is of these tiles: the same tile,
    schedule and grid."""
    rng, seen = np.random.default_rng(48), 0
    for dtype in ("q4", "q4_zp"):
        for _ in range(200):
            M, N, K = int(rng.integers(17, 257)), int(rng.integers(1, 12000)), 128 * int(rng.integers(1, 90))
            rows = sk.make_plan(M, N, K, dtype, "nt", cus=256, use_tuned=False, variant=12)
            if sk.kernel_name(rows.kernel_id).startswith("wavek_"):
                tiled = sk.make_plan(M, N, K, dtype + "_tiled", "nt", cus=256, use_tuned=False, variant=12)
                fields = ("bm", "bn", "bk", "schedule", "grid", "fixup", "raster", "streamk_tiles", "iters_per_tile", "workspace_bytes")
                assert tiled.kernel_id == rows.kernel_id + 40 and all(getattr(tiled, f) == getattr(rows, f) for f in fields), (dtype, M, N, K)
                seen += 1
    assert seen > 200
    with pytest.raises(sk.StreamKError):   # (what names no kernel for many rows has 64 of them at most)
        sk.make_plan(65, 1024, 1024, "q4_tiled", "nt", cus=256, use_tuned=False)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["q4", "q4_zp"])
def test_tiled_weights_give_the_bits_of_row_major_ones(sk, dtype):
    """The same call on both layouts, on values whose sums round and rows that 16 does not divide: operator calls of 17 to 256 rows
    and every tile through whole tiles, fixed splits and both fix-ups (the accumulating one on exact sums)."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(49)
    zp = dtype == "q4_zp"

    def operands(M, N, K, exact=False):
        A = torch.randint(-2, 3, (M, K), generator=gen, device="cuda").half() if exact else torch.randn(M, K, generator=gen, device="cuda").half()
        Wq = torch.randint(0, 256, (N, K // 2), generator=gen, device="cuda", dtype=torch.uint8)
        scales = torch.full((N, K // 128), 0.125, device="cuda").half() if exact else torch.rand(N, K // 128, generator=gen, device="cuda").half()
        zeros = dict(zeros=torch.randint(0, 16, (N, K // 128), generator=gen, device="cuda").half()) if zp else {}
        return (lambda **kw: sk.streamk_q4(A, Wq, scales, **zeros, **kw)), (lambda **kw: sk.streamk_q4(A, sk.tile_q4(Wq), scales, **zeros, tiled=True, **kw))
    for M, N, K in ((17, 200, 640), (33, 3001, 1152), (64, 768, 4096), (64, 11008, 1024), (65, 775, 512), (130, 1000, 2048), (200, 260, 4096), (256, 4097, 1280)):
        rows, tiled = operands(M, N, K)
        name = sk.kernel_name(sk.make_plan(M, N, K, dtype, "nt", sk.plan.operator_config(M, N, K, dtype, "nt")).kernel_id)
        if name.startswith("wavek_"):
            assert torch.equal(rows(), tiled()), (dtype, M, N, K)
        else:   # (the plans they take otherwise are of other kernels)
            assert ((rows() - tiled()).float().norm() / rows().float().norm()).item() < 2e-3, (dtype, M, N, K)
    for bm, bn in _TILES_Q4:
        M, N, K = bm + 3, 2 * bn + 5, 2176
        for exact, sched in ((False, dict(schedule="dp")), (False, dict(schedule="basic", grid=5, fixup="reduce")), (True, dict(schedule="basic", grid=7, fixup="atomic")), (False, dict(schedule="dp", grid=3))):
            rows, tiled = operands(M, N, K, exact)
            pr, pt = (sk.make_plan(M, N, K, dtype + layout, "nt", dict(sched, bm=bm, bn=bn, variant=11)) for layout in ("", "_tiled"))
            assert torch.equal(rows(plan=pr), tiled(plan=pt)), (dtype, bm, bn, sched)
    rows, tiled = operands(300, 256, 256)
    with pytest.raises(ValueError):
        tiled()
    sk.workspace_status()


def test_whole_tiles_get_a_cta_each(sk):
    """Fewer tiles than CUs and nothing split: as many CTAs as tiles, for few tiles too."""
    for dtype, step in (("float16", 8), ("float8_e4m3", 16), ("int8", 16), ("q4", 128)):
        for M, bm, bn in ((18, 32, 32), (40, 32, 32), (40, 64, 32), (100, 64, 64), (100, 128, 32)):
            for tiles in range(1, 65):
                for K in (step * (512 // step), 2304, 2560, 3072, 4096, 16384):
                    plan = sk.make_plan(M, tiles * bn - 5, K, dtype, "nt", dict(bm=bm, bn=bn, variant=11, schedule="dp"), cus=256)
                    assert plan.grid == min(plan.total_tiles, 256), (dtype, M, bm, bn, tiles, K, plan.grid)
    for shape in ((18, 264, 3072), (21, 312, 2560), (35, 272, 2304)):
        plan = sk.make_plan(*shape, "float8_e4m3", "nt", cus=256, use_tuned=False, variant=12)
        assert plan.grid >= plan.total_tiles, shape


def test_groups_of_rows_are_alike(sk):
    """More than eight rows of tiles stand in groups of eight at most that differ by less than one row a group; other kernels and
    rasters of the caller's as they were."""
    for bm in (32, 64, 128):
        for rows in range(1, 60):
            plan = sk.make_plan(rows * bm, 512, 2048, "float16", "nt", dict(bm=bm, bn=32, variant=11, schedule="dp"), cus=256)
            groups = -(-rows // 8)
            if rows <= 8:
                assert plan.raster == (8 if rows > 1 else 0)
            else:
                tail = rows - (groups - 1) * plan.raster
                assert plan.raster <= 8 and plan.raster - groups < tail <= plan.raster, (bm, rows, plan.raster)
            assert sk.make_plan(rows * bm, 512, 2048, "float16", "nt", dict(bm=bm, bn=32, variant=11, schedule="dp", raster=3), cus=256).raster == 3
            if rows * bm > 64:
                assert sk.make_plan(rows * bm, 512, 2048, "float16", "nt", dict(bm=64, bn=128, schedule="dp"), cus=256).raster in (0, 8)
    # a call whose rows were eight and one
    assert sk.make_plan(277, 1792, 15616, "bfloat16", "nt", cus=256, use_tuned=False, variant=12).raster == 5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float16", "float8_e4m3", "int8"])
def test_rows_far_apart(sk, dtype):
    """Rows of A up to 2 GiB of them to a tile run on the plan of the call's shape, natively from the second call on -- one row
    whatever its stride -- and rows further apart on the kernel that the call takes otherwise, whose tile has fewer of them."""
    import sys
    import torch
    from test_torch_ops import _calls_of
    rng = np.random.default_rng(46)
    plan_for = sys.modules["streamk.ops"]._plan_for
    kind = {"float8_e4m3": torch.float8_e4m3fn}.get(dtype) or getattr(torch, dtype)
    size, op = torch.empty(0, dtype=kind).element_size(), getattr(torch.ops.streamk, {"float16": "gemm_f16", "int8": "gemm_i8"}.get(dtype, "gemm_f8"))
    for M, N, K in ((1, 1024, 1024), (24, 20480, 3072)):
        A, B = _small(rng, (M, K)), _small(rng, (N, K))
        want, dB = _rounded(torch, A @ B.T, dtype), torch.from_numpy(B).float().cuda().to(kind)
        usual = plan_for("", M, N, K, dtype, "nt")
        most = (1 << 31) // (usual.bm * size)
        for lda, native in ((most - 16, True), (most, M == 1)):
            lda -= 16 if M == 1 else 0   # (the library looks at the stride of a single row too)
            dA = torch.empty((M - 1) * lda + K, dtype=torch.uint8 if size == 1 else kind, device="cuda").view(kind).as_strided((M, K), (lda, 1))
            dA.copy_(torch.from_numpy(A).float().cuda().to(kind))
            args = (dA, dB) + (("nt",) if dtype == "float16" else ())
            assert torch.equal(op(*args).cpu(), want), (dtype, M, lda)
            names, got = _calls_of(lambda: op(*args))
            assert torch.equal(got.cpu(), want) and (len(names) == 1) == native, (dtype, M, lda, names)
            plan = plan_for("", M, N, K, dtype, "nt", lda * size, K * size)
            other = sk.make_plan(M, N, K, dtype, "nt", None if dtype == "float16" else {"variant": 9})
            assert plan.kernel_id == (usual if native else other).kernel_id, (dtype, M, lda)
            del dA, args, got
