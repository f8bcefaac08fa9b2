"""The 128 x 128 wgrad kernel for groups with few rows (gg_wfew.hip), through the C ABI.

Every output of forced plans (GG_WFEW=1) against a torch fp32 product, in every operand format and
over host and device sizes: rows at the edges of a chunk (32; fp8: 128), empty groups, widths that
end inside a tile. An output may be off by its own rounding (2^-8 relative in bf16, 2^-11 in fp16)
and by fp32 sums of the group's rows in another order (rows 2^-23 sum |a b|, twice: the reference is
rounded too); the fp8 MFMA aligns its 128 products to the largest before it adds them, which costs
up to 2^-13.9 sum |a b| against float64 on such inputs (16-700 rows, the three format pairs; the
persistent kernel gives the same bits): 2^-13 is allowed for it.
"""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
TDT = {"bf16": torch.bfloat16, "fp16": torch.float16, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}


def _stream():
    return torch.cuda.current_stream(DEV).cuda_stream


def _gdt(pkg, t):
    return {"bf16": pkg.DType.BF16, "fp16": pkg.DType.FP16, "e4m3": pkg.DType.FP8_E4M3, "e5m2": pkg.DType.FP8_E5M2}[t]


class Case:
    def __init__(self, pkg, ta, tb, gm, n, k, device, ints=False, seed=0):
        gen = torch.Generator().manual_seed(seed)

        def rand(shape):
            return torch.randint(-1, 2, shape, generator=gen).float() if ints else torch.randn(shape, generator=gen)

        self.gm, self.f8, rows, b = gm, ta in ("e4m3", "e5m2"), sum(gm), len(gm)
        self.go, self.x = rand((rows, n)).to(TDT[ta]).to(DEV), rand((rows, k)).to(TDT[tb]).to(DEV)
        self.odt = torch.bfloat16 if self.f8 else TDT[ta]
        self.out = torch.full((b, n, k), float("nan"), dtype=self.odt, device=DEV)
        self.sa = torch.tensor([0.5], device=DEV)
        self.sb = torch.tensor([0.25 * (1 + g % 3) for g in range(b)], device=DEV)
        p = [t.data_ptr() for t in (self.go, self.x, self.out)]
        sp = [self.sa.data_ptr(), self.sb.data_ptr()] if self.f8 else [0, 0]
        self.lens = torch.tensor(gm, dtype=torch.int64, device=DEV)
        if device:
            self.plan = pkg.DeviceLensPlan(pkg.OP_WGRAD, _gdt(pkg, ta), _gdt(pkg, tb), b, rows, n, k, self.lens.data_ptr(), 0,
                                           *p, _stream(), *sp)
        else:
            self.plan = pkg.BackwardPlan("wgrad", _gdt(pkg, ta), n, k, gm, *p, _stream(), other_dtype=_gdt(pkg, tb),
                                         grad_scale=sp[0], other_scale=sp[1])

    def run(self):
        self.plan.run(_stream())
        torch.cuda.synchronize(DEV)
        return self

    def check(self):
        half, r0 = 2.0 ** -11 if self.odt == torch.float16 else 2.0 ** -8, 0
        for g, m in enumerate(self.gm):
            a, b = self.go[r0:r0 + m].float().t().contiguous(), self.x[r0:r0 + m].float()
            scale = float(self.sa[0] * self.sb[g]) if self.f8 else 1.0
            ref, mag = (a @ b) * scale, (a.abs() @ b.abs()) * scale
            sums = 2 * max(m, 1) * 2.0 ** -23 + (2.0 ** -13 if self.f8 else 0.0)
            got = self.out[g].float()
            assert not torch.isnan(got).any(), f"group {g}: unwritten outputs ({self.plan.detail()})"
            off = int(((got - ref).abs() > half * ref.abs() * (1 + 2.0 ** -8) + sums * mag + 1e-7).sum())
            assert off == 0, f"group {g}: {off} outputs off ({self.plan.detail()})"
            if m == 0:
                assert torch.count_nonzero(got) == 0
            r0 += m

    def close(self):
        self.plan.release()


FORMATS = [("bf16", "bf16"), ("fp16", "fp16"), ("e4m3", "e4m3"), ("e5m2", "e5m2"), ("e5m2", "e4m3")]
SHAPES = [
    ([31, 0, 32, 33, 1, 129], 144, 272),
    ([127, 128, 257], 128, 16),
    ([3, 0] * 35, 32, 144),  # 70 groups (device sizes: the table kernel)
    ([700, 5], 1040, 656),   # partial tiles in both widths
    ([9, 0, 40, 33] * 5, 1040, 1040),  # 1620 tiles: a whole round of 1024 in the XCD remap and a partial one
]


@pytest.mark.parametrize("fmt", range(len(FORMATS)))
@pytest.mark.parametrize("device", [False, True])
def test_wgrad_few_vs_torch_fp32(pkg, monkeypatch, fmt, device):
    monkeypatch.delenv("GG_SMALL", raising=False)
    monkeypatch.setenv("GG_WFEW", "1")
    ta, tb = FORMATS[fmt]
    for i, (gm, n, k) in enumerate(SHAPES):
        if ta in ("bf16", "fp16"):
            n, k = n - 8, k - 8
        print(f"[wgrad few] {ta} x {tb} shape {i} N={n} K={k} device={device}", flush=True)
        c = Case(pkg, ta, tb, gm, n, k, device, seed=i)
        assert "few-row 128x128" in c.plan.detail(), c.plan.detail()
        c.run().check()
        if device:
            st, tiles, msg = c.plan.status(_stream())
            assert st == pkg.GG_OK and tiles == len(gm) * -(-n // 256) * -(-k // 256), (msg, tiles)
        c.close()


def test_wgrad_few_same_outputs_as_the_persistent_kernel(pkg, monkeypatch):
    """Inputs in {-1, 0, 1}: exact sums, so both kernels give the same bits, host and device sizes."""
    gm, n, k, outs = [70, 0, 31, 1, 300], 136, 200, []
    for few in (False, True):
        monkeypatch.setenv("GG_SMALL", "0")
        if few:
            monkeypatch.delenv("GG_SMALL")
            monkeypatch.setenv("GG_WFEW", "1")
        for device in (False, True):
            c = Case(pkg, "bf16", "bf16", gm, n, k, device, ints=True).run()
            assert ("few-row" in c.plan.detail()) == few
            outs.append(c.out.clone())
            c.close()
    for o in outs[1:]:
        assert torch.equal(o.view(torch.int16), outs[0].view(torch.int16))


def test_wgrad_few_bad_group_and_planner_choice(pkg, monkeypatch):
    monkeypatch.delenv("GG_SMALL", raising=False)
    c = Case(pkg, "bf16", "bf16", [16] * 8, 512, 1024, True)
    assert "few-row 128x128" in c.plan.detail(), c.plan.detail()
    c.lens[3] = -5
    c.run()
    st, _, msg = c.plan.status(_stream())
    assert st == pkg.GG_ERR_INVALID and "group 3" in msg, msg
    assert torch.count_nonzero(c.out[3].float()) == 0 and not torch.isnan(c.out.float()).any()
    c.close()
    for device in (False, True):
        c = Case(pkg, "bf16", "bf16", [2600] * 4, 2816, 2048, device, ints=True)
        assert "persistent" in c.plan.detail(), c.plan.detail()
        c.close()


@pytest.mark.parametrize("few", [False, True])
@pytest.mark.parametrize("device", [False, True])
def test_fp8_gradients_of_no_rows_need_no_scales(pkg, monkeypatch, few, device):
    """No group has a row, so nothing is read and the scales may be null: the gradients are zeros, from
    either kernel, as a plan, as one call and (device sizes) without allocations."""
    if few:
        monkeypatch.delenv("GG_SMALL", raising=False)
        monkeypatch.setenv("GG_WFEW", "1")
    b, n, k = 3, 272, 144
    e5, e4 = _gdt(pkg, "e5m2"), _gdt(pkg, "e4m3")
    out = torch.empty((b, n, k), dtype=torch.bfloat16, device=DEV)
    lens = torch.zeros(b, dtype=torch.int64, device=DEV)
    lib, sizes, need = pkg.load_library(), (ctypes.c_int64 * b)(), ctypes.c_size_t(0)
    ws = torch.empty(4096, dtype=torch.uint8, device=DEV)
    status = torch.empty(4, dtype=torch.int32, device="cpu", pin_memory=True)

    def zeros(run):
        out.fill_(float("nan"))
        run()
        torch.cuda.synchronize(DEV)
        assert torch.count_nonzero(out.float()) == 0

    if device:
        plan = pkg.DeviceLensPlan(pkg.OP_WGRAD, e5, e4, b, 0, n, k, lens.data_ptr(), 0, 0, 0, out.data_ptr(), _stream())
        zeros(lambda: pkg.run_device_lens_noalloc(pkg.OP_WGRAD, e5, e4, b, 0, n, k, lens.data_ptr(), 0, 0, 0, out.data_ptr(),
                                                  _stream()))
        zeros(lambda: lib.gg_call_device_lens(pkg.OP_WGRAD, int(e5), int(e4), b, 0, n, k, lens.data_ptr(), 0, 0, 0, 0, 0,
                                              out.data_ptr(), ws.data_ptr(), 4096, status.data_ptr(), _stream()))
        assert lib.gg_check_status(status.data_ptr()) == pkg.GG_OK
    else:
        plan = pkg.BackwardPlan("wgrad", e5, n, k, [0] * b, 0, 0, out.data_ptr(), _stream(), other_dtype=e4)
        zeros(lambda: lib.gg_call(pkg.OP_WGRAD, int(e5), int(e4), b, n, k, sizes, 0, 0, 0, 0, out.data_ptr(), ws.data_ptr(), 4096,
                                  ctypes.byref(need), _stream()))
    assert ("few-row" in plan.detail()) == few, plan.detail()
    zeros(lambda: plan.run(_stream()))
    plan.release()


def test_more_tiles_than_one_launch_takes(pkg, monkeypatch):
    """2^24 groups of one tile each: a launch of one workgroup per tile would pass HIP's 2^32 threads, so the
    persistent kernel runs, also where the 128 x 128 one is asked for."""
    monkeypatch.delenv("GG_SMALL", raising=False)
    monkeypatch.setenv("GG_WFEW", "1")
    lib, b, plan = pkg.load_library(), 1 << 24, ctypes.c_void_p()
    out = torch.ones((b, 8, 8), dtype=torch.bfloat16, device=DEV)
    st = lib.gg_prepare_wgrad(int(pkg.DType.BF16), b, 8, 8, (ctypes.c_int64 * b)(), 0, 0, out.data_ptr(), _stream(),
                              ctypes.byref(plan))
    assert st == pkg.GG_OK, pkg.last_error()
    assert "persistent" in lib.gg_plan_detail(plan).decode()
    assert lib.gg_run(plan, _stream()) == pkg.GG_OK, pkg.last_error()
    torch.cuda.synchronize(DEV)
    lib.gg_release(plan)
    assert torch.count_nonzero(out) == 0


# past 300 rows per group the share it must promise is smaller in less than two rounds of workgroups:
# (group rows, N, K, few-row tiles expected)
PAST_300 = [
    ([1193] * 5, 6432, 512, False),    # 1.0 rounds, predicted at 0.79 of the persistent plan
    ([316] * 11, 5376, 3344, True),    # 12 rounds, 0.89
    ([320] * 4, 512, 512, True),       # 0.06 rounds, far below it
]


@pytest.mark.parametrize("case", range(len(PAST_300)))
def test_planner_choice_past_300_rows(pkg, monkeypatch, case):
    monkeypatch.delenv("GG_SMALL", raising=False)
    gm, n, k, few = PAST_300[case]
    p, e4 = torch.empty(16, dtype=torch.uint8, device=DEV).data_ptr(), _gdt(pkg, "e4m3")  # plans read no operand
    plan = pkg.BackwardPlan("wgrad", e4, n, k, gm, p, p, p, _stream(), other_dtype=e4, grad_scale=p, other_scale=p)
    assert ("few-row" in plan.detail()) == few, plan.detail()
    plan.release()
