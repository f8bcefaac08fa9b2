"""The torch-level calls (gg_call / gg_call_device_lens): one call in memory from torch's allocator gives
the bits of a plan over the same buffers, for every pass, type and kind of sizes; the workspace
protocol; calls from several threads and streams."""
import ctypes
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _stream():
    return torch.cuda.current_stream(DEV).cuda_stream


# (pass, type, group rows, N, K): few-row, 128 x 128, short, split-K, tail and persistent plans, more than
# 64 groups, no rows at all, an empty contraction
CASES = [
    ("fwd", "bf16", [5, 0, 33], 264, 520), ("fwd", "fp16", [512], 2880, 2880), ("fwd", "bf16", [520] * 32, 2880, 256),
    ("fwd", "e4m3", [300, 0, 77], 264, 1040), ("fwd", "bf16", [7] * 70, 128, 72), ("fwd", "bf16", [0, 0], 64, 64),
    ("fwd", "bf16", [17, 5], 64, 0), ("dgrad", "bf16", [300, 0, 200], 2056, 520), ("dgrad", "e4m3", [64, 1], 1040, 272),
    ("dgrad", "bf16", [1000, 2000, 1100], 1024, 2048), ("wgrad", "bf16", [300, 0, 17], 272, 528),
    ("wgrad", "fp16", [600, 1000, 513], 1024, 2304), ("wgrad", "e4m3", [9] * 70, 64, 144), ("wgrad", "bf16", [0], 64, 64),
]


def _inputs(op, t, gm, n, k, seed=0):
    gen = torch.Generator().manual_seed(seed)
    td = {"bf16": torch.bfloat16, "fp16": torch.float16, "e4m3": torch.float8_e4m3fn}[t]
    rows, b = sum(gm), len(gm)

    def rand(shape):
        return torch.randn(shape, generator=gen).to(td).to(DEV)

    a = rand((rows, k if op == "fwd" else n))
    other = rand((rows, k) if op == "wgrad" else (b, n, k))
    return a, other, torch.tensor([0.5], device=DEV), torch.linspace(0.25, 1.0, b, device=DEV)


def _call(pkg, op, t, a, other, sizes, sa, sb, out=None, stream=None):
    if t == "e4m3":
        f = {"fwd": pkg.grouped_gemm_fp8, "dgrad": pkg.grouped_gemm_dgrad_fp8, "wgrad": pkg.grouped_gemm_wgrad_fp8}[op]
        return f(a, other, sizes, sa, sb, out=out, stream=stream)
    f = {"fwd": pkg.grouped_gemm, "dgrad": pkg.grouped_gemm_dgrad, "wgrad": pkg.grouped_gemm_wgrad}[op]
    return f(a, other, sizes, out=out, stream=stream)


@pytest.mark.parametrize("small", ["0", None])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_calls_give_the_bits_of_plans(pkg, monkeypatch, case, small):
    """An explicit stream takes the plan route, none the one-call route."""
    if small is None:
        monkeypatch.delenv("GG_SMALL", raising=False)
    op, t, gm, n, k = CASES[case]
    a, other, sa, sb = _inputs(op, t, gm, n, k, seed=case)
    for sizes in (gm, torch.tensor(gm, dtype=torch.int64, device=DEV)):
        if t == "e4m3" and op == "fwd" and sizes is not gm:
            continue  # the fp8 forward function takes host sizes
        print(f"[call] {op} {t} {gm[:4]} N={n} K={k} device={sizes is not gm}", flush=True)
        shape = {"fwd": (sum(gm), n), "dgrad": (sum(gm), k), "wgrad": (len(gm), n, k)}[op]
        odt = torch.bfloat16 if t == "e4m3" else a.dtype
        one, plan = (torch.full(shape, float("nan"), dtype=odt, device=DEV) for _ in range(2))
        assert _call(pkg, op, t, a, other, sizes, sa, sb, one) is one
        _call(pkg, op, t, a, other, sizes, sa, sb, plan, _stream())
        torch.cuda.synchronize(DEV)
        assert not torch.isnan(one.float()).any()
        assert torch.equal(one.view(torch.int16), plan.view(torch.int16))


# more groups than fill one launch of the table upload (3584 bytes of kernel arguments) and its limit of 32
# KB, with and without tile descriptors in the call's plan (from 128 groups on, up to 4 tiles per group)
MANY = [
    ("fwd", "bf16", 127, 40, 24), ("fwd", "bf16", 300, 512, 64), ("fwd", "fp16", 300, 1032, 64), ("fwd", "bf16", 2100, 24, 40),
    ("fwd", "bf16", 9000, 16, 16), ("fwd", "e4m3", 300, 520, 48), ("dgrad", "bf16", 300, 40, 512), ("dgrad", "bf16", 2100, 40, 16),
    ("wgrad", "bf16", 300, 24, 40), ("wgrad", "fp16", 2100, 16, 24),
]


@pytest.mark.parametrize("small", ["0", None])
@pytest.mark.parametrize("case", range(len(MANY)))
def test_many_groups(pkg, monkeypatch, case, small):
    """Rows are ragged, some groups empty; the plan route gives the same bits."""
    if small is None:
        monkeypatch.delenv("GG_SMALL", raising=False)
    op, t, b, n, k = MANY[case]
    gm = [(7 * g * g + g // 64) % 5 for g in range(b - 1)] + [300]
    a, other, sa, sb = _inputs(op, t, gm, n, k, seed=case)
    print(f"[call] {op} {t} {b} groups N={n} K={k}", flush=True)
    one = _call(pkg, op, t, a, other, gm, sa, sb)
    plan = _call(pkg, op, t, a, other, gm, sa, sb, stream=_stream())
    torch.cuda.synchronize(DEV)
    assert not torch.isnan(one.float()).any() and one.float().abs().max() > 1
    assert torch.equal(one.view(torch.int16), plan.view(torch.int16))


@pytest.mark.parametrize("b", [40, 300, 3000])
def test_call_replays_in_a_graph(pkg, monkeypatch, b):
    """gg_call captured with tables of one launch, of several and past the size that is copied outside a
    capture: nothing is waited for, and every replay, with eager work between, writes the tables again and
    gives the plan's bits."""
    monkeypatch.delenv("GG_SMALL", raising=False)
    gm = [(7 * g * g) % 5 for g in range(b - 1)] + [300]
    a, w, _, _ = _inputs("fwd", "bf16", gm, 72, 40, seed=b)
    want = pkg.grouped_gemm(a, w, gm, stream=_stream())
    lib, need, out = pkg.load_library(), ctypes.c_size_t(0), torch.empty_like(want)
    sizes, ws = (ctypes.c_int64 * b)(*gm), torch.empty(1 << 20, dtype=torch.uint8, device=DEV)

    def call():
        st = lib.gg_call(pkg.OP_FORWARD, 0, 0, b, 72, 40, sizes, a.data_ptr(), w.data_ptr(), 0, 0, out.data_ptr(),
                         ws.data_ptr(), ws.numel(), ctypes.byref(need), torch.cuda.current_stream(DEV).cuda_stream)
        assert st == pkg.GG_OK, pkg.last_error()

    call()
    torch.cuda.synchronize(DEV)
    assert torch.equal(out, want) and (need.value > 32768) == (b == 3000)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for replay in range(3):
        out.fill_(float("nan"))
        ws.zero_()
        pkg.grouped_gemm(a, w, gm)
        graph.replay()
        torch.cuda.synchronize(DEV)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), replay


def test_workspace_protocol(pkg, monkeypatch):
    """Too little workspace enqueues nothing and says how much is needed; that much is enough."""
    monkeypatch.setenv("GG_SPLIT_K", "3")
    a, w, _, _ = _inputs("fwd", "bf16", [256], 256, 1024)
    out = torch.full((256, 256), float("nan"), dtype=torch.bfloat16, device=DEV)
    lib, gm, need = pkg.load_library(), (ctypes.c_int64 * 1)(256), ctypes.c_size_t(0)

    def call(ws, nbytes):
        return lib.gg_call(pkg.OP_FORWARD, 0, 0, 1, 256, 1024, gm, a.data_ptr(), w.data_ptr(), 0, 0, out.data_ptr(), ws, nbytes,
                           ctypes.byref(need), _stream())

    small = torch.empty(512, dtype=torch.uint8, device=DEV)
    assert call(small.data_ptr(), 512) == pkg.GG_ERR_WORKSPACE
    assert need.value == 256 + 3 * 262144  # one group's table, three ranges of one tile
    torch.cuda.synchronize(DEV)
    assert torch.isnan(out.float()).all()
    ws = torch.empty(need.value + 16, dtype=torch.uint8, device=DEV)
    assert call(ws.data_ptr() + 16, need.value) == pkg.GG_ERR_INVALID  # not 256-byte aligned
    assert call(ws.data_ptr(), need.value) == pkg.GG_OK
    torch.cuda.synchronize(DEV)
    ref = a.float() @ w[0].float().t().contiguous()
    assert torch.allclose(out.float(), ref, rtol=1e-2, atol=1e-2)


def test_bad_device_sizes_raise(pkg):
    for b in (3, 70):  # the GEMM builds the table; the table kernel does
        a, w, _, _ = _inputs("fwd", "bf16", [8] * b, 64, 72)
        lens = torch.tensor([8] * b, dtype=torch.int64, device=DEV)
        lens[b - 2] = -1
        with pytest.raises(pkg.GGError, match=f"group {b - 2} "):
            pkg.grouped_gemm(a, w, lens)


def test_default_device_is_the_gpu(pkg):
    """A program may make the GPU torch's default device; the status of a device-size call stays host memory."""
    a, w, _, _ = _inputs("fwd", "bf16", [5, 3], 64, 72)
    want = pkg.grouped_gemm(a, w, [5, 3])
    with torch.device(DEV):
        for sizes in ([5, 3], torch.tensor([5, 3], dtype=torch.int64, device=DEV)):
            assert torch.equal(pkg.grouped_gemm(a, w, sizes), want)


def test_threads_and_streams(pkg, monkeypatch):
    """Four threads, each on a stream of its own with sizes of its own, 30 calls each."""
    monkeypatch.delenv("GG_SMALL", raising=False)
    failures = []

    def work(i):
        try:
            gm = [(7 * i + 5 * g) % 40 for g in range(6 + 30 * (i % 2))]
            with torch.cuda.stream(torch.cuda.Stream(DEV)):
                a, w, _, _ = _inputs("fwd", "bf16", gm, 256, 320, seed=i)
                lens = torch.tensor(gm, dtype=torch.int64, device=DEV)
                first = [pkg.grouped_gemm(a, w, sizes) for sizes in (gm, lens)]  # (may sum in another order)
                for _ in range(30):
                    for sizes, want in zip((gm, lens), first):
                        if not torch.equal(pkg.grouped_gemm(a, w, sizes), want):
                            failures.append(i)
                ref = torch.cat([a[sum(gm[:g]):sum(gm[:g + 1])].float() @ w[g].float().t().contiguous() for g in range(len(gm))])
                if not all(torch.allclose(f.float(), ref, rtol=1e-2, atol=1e-2) for f in first):
                    failures.append(("ref", i))
        except Exception as e:  # noqa: BLE001 (a thread's failure is the test's)
            failures.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
