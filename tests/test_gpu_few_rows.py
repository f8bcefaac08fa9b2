"""The few-row kernel (gg_few.hip): forward and dgrad of groups with few rows, through the C ABI.

Every instance is forced (GG_FEW) on shapes at the edges of its tiles and K split, host- and
device-size, in every operand format, against a torch fp32 product of the same inputs. An output
may be off by its own 16-bit rounding (half a unit in the last of 8 significant bits: 2^-8 relative
in bf16; 11 bits, 2^-11, in fp16) and by fp32 sums of K products in another order (at most
K 2^-23 sum |a b|, which the product of the absolute values gives). The fp8 MFMA aligns its 128
products to the largest before it adds them, which costs up to 2^-13.9 sum |a b| against float64 on
such inputs (contractions of 16-700; the persistent kernel gives the same bits): 2^-13 is allowed.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
INSTANCES = 5
TDT = {"bf16": torch.bfloat16, "fp16": torch.float16, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}


def _stream():
    return torch.cuda.current_stream(DEV).cuda_stream


def _gdt(pkg, t):
    return {"bf16": pkg.DType.BF16, "fp16": pkg.DType.FP16, "e4m3": pkg.DType.FP8_E4M3, "e5m2": pkg.DType.FP8_E5M2}[t]


class Case:
    """One plan over random inputs; a and b in fp32 are what the reference multiplies."""

    def __init__(self, pkg, op, ta, tb, gm, n, k, device, ints=False, offs=None, rows=None, seed=0):
        gen = torch.Generator().manual_seed(seed)
        self.op, self.gm, self.f8 = op, gm, ta in ("e4m3", "e5m2")
        rows = sum(gm) if rows is None else rows
        ka, ko = (k, n) if op == "fwd" else (n, k)  # contraction, output columns

        def rand(shape):
            return torch.randint(-1, 2, shape, generator=gen).float() if ints else torch.randn(shape, generator=gen)

        self.a = rand((rows, ka)).to(TDT[ta]).to(DEV)
        self.b = rand((len(gm), n, k)).to(TDT[tb]).to(DEV)
        self.odt = torch.bfloat16 if self.f8 else TDT[ta]
        self.out = torch.full((rows, ko), float("nan"), dtype=self.odt, device=DEV)
        self.sa = torch.tensor([0.5], device=DEV)
        self.sb = torch.tensor([0.25 * (1 + g % 3) for g in range(len(gm))], device=DEV)
        p = [t.data_ptr() for t in (self.a, self.b, self.out)]
        sp = [self.sa.data_ptr(), self.sb.data_ptr()] if self.f8 else [0, 0]
        self.lens = torch.tensor(gm, dtype=torch.int64, device=DEV)
        self.offs = None if offs is None else torch.tensor(offs, dtype=torch.int64, device=DEV)
        if device:
            code = pkg.OP_FORWARD if op == "fwd" else pkg.OP_DGRAD
            self.plan = pkg.DeviceLensPlan(code, _gdt(pkg, ta), _gdt(pkg, tb), len(gm), rows, n, k, self.lens.data_ptr(),
                                           0 if offs is None else self.offs.data_ptr(), *p, _stream(), *sp)
        elif op == "dgrad":
            self.plan = pkg.BackwardPlan("dgrad", _gdt(pkg, ta), n, k, gm, *p, _stream(), other_dtype=_gdt(pkg, tb),
                                         grad_scale=sp[0], other_scale=sp[1])
        elif self.f8:
            self.plan = pkg.Fp8Plan(_gdt(pkg, ta), n, k, gm, p[0], p[1], sp[0], sp[1], p[2], _stream())
        else:
            self.plan = pkg.make_mi355x_backend()
            assert self.plan.prepare(pkg.GroupedGemmProblem(_gdt(pkg, ta), len(gm), n, k, gm, *p), _stream()) == ""

    def run(self):
        self.plan.run(_stream())
        torch.cuda.synchronize(DEV)
        return self

    def close(self):
        self.plan.release()

    def product(self, g, r0, m, f=lambda t: t):
        a, b = f(self.a[r0:r0 + m].float()), f(self.b[g].float())
        scale = float(self.sa[0] * self.sb[g]) if self.f8 else 1.0
        return (a @ (b.t().contiguous() if self.op == "fwd" else b)) * scale

    def check(self):
        half = 2.0 ** -11 if self.odt == torch.float16 else 2.0 ** -8
        k = self.a.shape[1]
        r0 = 0
        for g, m in enumerate(self.gm):
            got, ref = self.out[r0:r0 + m].float(), self.product(g, r0, m)
            # the reference is rounded too: twice the sums' bound; 1e-7: fp16 below its normal range
            sums = 2 * k * 2.0 ** -23 + (2.0 ** -13 if self.f8 else 0.0)
            tol = half * ref.abs() * (1 + 2.0 ** -8) + sums * self.product(g, r0, m, torch.abs) + 1e-7
            assert not torch.isnan(got).any(), f"group {g}: unwritten outputs ({self.plan.detail()})"
            off = int(((got - ref).abs() > tol).sum())
            assert off == 0, f"group {g}: {off} outputs off ({self.plan.detail()})"
            r0 += m


FORMATS = [("fwd", "bf16", "bf16"), ("fwd", "fp16", "fp16"), ("fwd", "e4m3", "e4m3"), ("fwd", "e5m2", "e5m2"),
           ("dgrad", "bf16", "bf16"), ("dgrad", "fp16", "fp16"), ("dgrad", "e4m3", "e4m3"), ("dgrad", "e5m2", "e5m2"),
           ("dgrad", "e5m2", "e4m3")]
# (group rows, N, K): rows at the edges of 16-, 32- and 64-row tiles with empty groups; widths that
# end inside a 16- and a 64-column tile; contractions of one piece, of one chunk short of and past
# what 4 and 8 waves share, and of several chunks per wave
SHAPES = [
    ([1, 0, 16, 17, 33, 64, 65, 0, 129], 144, 80),
    ([3, 5], 16, 16),
    ([40, 0, 7], 272, 560),
    ([9], 1040, 4112),
    ([2, 1] * 33, 64, 320),  # 66 groups: the table is read in two parts (device sizes: table kernel)
]


@pytest.mark.parametrize("instance", range(INSTANCES))
@pytest.mark.parametrize("fmt", range(len(FORMATS)))
def test_instances_vs_torch_fp32(pkg, monkeypatch, instance, fmt):
    monkeypatch.delenv("GG_SMALL", raising=False)
    monkeypatch.setenv("GG_FEW", str(instance))
    op, ta, tb = FORMATS[fmt]
    for i, (gm, n, k) in enumerate(SHAPES):
        if ta in ("bf16", "fp16"):
            n, k = n - 8, k - 8  # 16-bit rows may end in half an fp8 piece
        for device in (False, True):
            print(f"[few] instance {instance} {op} {ta} x {tb} shape {i} N={n} K={k} device={device}", flush=True)
            c = Case(pkg, op, ta, tb, gm, n, k, device, seed=i)
            assert "few-row" in c.plan.detail(), c.plan.detail()
            c.run().check()
            c.close()


@pytest.mark.parametrize("op", ["fwd", "dgrad"])
def test_same_outputs_as_the_persistent_kernel(pkg, monkeypatch, op):
    """Inputs in {-1, 0, 1}: every partial sum is exact in fp32, so the persistent kernel and every
    instance, over host and device sizes, give the same bits."""
    gm, n, k = [70, 0, 31, 1], 136, 200
    outs = []
    for few in [None] + list(range(INSTANCES)):
        monkeypatch.setenv("GG_SMALL", "0")
        if few is not None:
            monkeypatch.delenv("GG_SMALL")
            monkeypatch.setenv("GG_FEW", str(few))
        for device in (False, True):
            c = Case(pkg, op, "bf16", "bf16", gm, n, k, device, ints=True).run()
            assert ("few-row" in c.plan.detail()) == (few is not None)
            outs.append(c.out.clone())
            c.close()
    for o in outs[1:]:
        assert torch.equal(o.view(torch.int16), outs[0].view(torch.int16))


@pytest.mark.parametrize("b", [64, 65, 128, 129, 4096, 4097, 9000])
@pytest.mark.parametrize("instance", [1, 3])
def test_group_search(pkg, monkeypatch, b, instance):
    """Tables of one, two and three levels of 64, whole and ragged, with empty groups at the start, at the end
    and between: every row is multiplied with its own expert (integers: exact)."""
    monkeypatch.delenv("GG_SMALL", raising=False)
    monkeypatch.setenv("GG_FEW", str(instance))
    gm = [0, 0] + [(7 * g * g + g // 64) % 5 for g in range(b - 5)] + [40, 0, 0]
    rows = torch.repeat_interleave(torch.arange(b, device=DEV), torch.tensor(gm, device=DEV))
    for device in (False, True):
        print(f"[few search] {b} groups device={device}", flush=True)
        c = Case(pkg, "fwd", "bf16", "bf16", gm, 24, 16, device, ints=True, seed=b).run()
        assert "few-row" in c.plan.detail(), c.plan.detail()
        ref = (c.a.float()[:, None, :] * c.b.float()[rows]).sum(-1)
        assert torch.equal(c.out.float(), ref)
        c.close()


@pytest.mark.parametrize("b", [3, 70])
def test_device_sizes_gaps_and_bad_groups(pkg, monkeypatch, b):
    """Rows outside every group stay as they were; a group whose rows do not fit is named and left
    out; the status counts 256 x 256 tiles as every plan's does."""
    monkeypatch.delenv("GG_SMALL", raising=False)
    monkeypatch.setenv("GG_FEW", "0")
    gm = [20] * b
    offs = [30 * g + 5 for g in range(b)] + [0]
    c = Case(pkg, "fwd", "bf16", "bf16", gm, 264, 72, True, offs=offs, rows=30 * b + 5).run()
    st, tiles, msg = c.plan.status(_stream())
    assert st == pkg.GG_OK and tiles == 2 * b, (msg, tiles)
    inside = torch.zeros(30 * b + 5, dtype=torch.bool, device=DEV)
    for g in range(b):
        r0 = offs[g]
        inside[r0:r0 + 20] = True
        assert torch.allclose(c.out[r0:r0 + 20].float(), c.product(g, r0, 20), rtol=2.0 ** -8, atol=1e-3)
    assert torch.isnan(c.out[~inside].float()).all() and not torch.isnan(c.out[inside].float()).any()
    c.lens[b - 1] = 400
    c.out.fill_(float("nan"))
    c.run()
    st, _, msg = c.plan.status(_stream())
    assert st == pkg.GG_ERR_INVALID and f"group {b - 1}" in msg, msg
    assert torch.isnan(c.out[offs[b - 1]:].float()).all() and not torch.isnan(c.out[offs[0]:offs[0] + 20].float()).any()
    c.close()


def test_more_tiles_than_the_launch_was_sized_for(pkg, monkeypatch):
    """Groups that all own the same rows make more tiles than their rows alone would: the workgroups
    go on to further tiles. All experts are equal, so every group writes the same values."""
    monkeypatch.delenv("GG_SMALL", raising=False)
    monkeypatch.setenv("GG_FEW", "0")
    b, m = 40, 100
    c = Case(pkg, "fwd", "bf16", "bf16", [m] * b, 136, 72, True, ints=True, offs=[0] * (b + 1), rows=m)
    c.b.copy_(c.b[:1].expand_as(c.b))
    c.run()
    assert torch.equal(c.out.float(), c.product(0, 0, m).to(torch.bfloat16).float())
    c.close()


def test_allocation_free_call_replays_in_a_graph(pkg, monkeypatch):
    """gg_run_device_lens_noalloc captured with the few-row kernel (with and without the table kernel):
    each replay, with eager work between, gives the plan's bits."""
    monkeypatch.delenv("GG_SMALL", raising=False)
    for b in (5, 70):
        c = Case(pkg, "fwd", "bf16", "bf16", [4] * b, 264, 520, True, seed=b)
        assert "few-row" in c.plan.detail(), c.plan.detail()
        c.run()
        want, out = c.out.clone(), torch.empty_like(c.out)
        args = (pkg.OP_FORWARD, pkg.DType.BF16, pkg.DType.BF16, b, 4 * b, 264, 520, c.lens.data_ptr(), 0, c.a.data_ptr(),
                c.b.data_ptr(), out.data_ptr())
        pkg.run_device_lens_noalloc(*args, _stream())
        torch.cuda.synchronize(DEV)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            pkg.run_device_lens_noalloc(*args, torch.cuda.current_stream(DEV).cuda_stream)
        for replay in range(3):
            out.fill_(float("nan"))
            c.run()
            graph.replay()
            torch.cuda.synchronize(DEV)
            assert torch.equal(out.view(torch.int16), want.view(torch.int16)), replay
        c.close()


# (op, formats, group rows, N, K, few-row tiles expected)
AUTO = [
    ("fwd", "bf16", [256] * 4, 512, 1024, True),
    ("fwd", "bf16", [16] * 36, 2048, 1024, True),
    ("dgrad", "e4m3", [10] * 16, 2048, 1024, True),
    ("fwd", "bf16", [128] * 8, 4096, 7168, False),    # 128 x 128 tiles: half the staged bytes
    ("dgrad", "bf16", [4096] * 8, 1024, 2048, False),
]


@pytest.mark.parametrize("case", range(len(AUTO)))
def test_planner_choice(pkg, monkeypatch, case):
    monkeypatch.delenv("GG_SMALL", raising=False)
    op, t, gm, n, k, few = AUTO[case]
    for device in (False, True):
        c = Case(pkg, op, t, t, gm, n, k, device, ints=True)
        assert ("few-row" in c.plan.detail()) == few, c.plan.detail()
        c.close()


# long contractions (rows of 8 KB and more) in less than 1.4 rounds of workgroups promise less than the model
# says: (op, group rows, N, K, few-row tiles expected)
LONG = [
    ("dgrad", [26] * 3, 13888, 1024, False),   # 0.19 rounds, predicted at 0.73 of the persistent plan
    ("fwd", [16] * 2, 512, 12288, True),       # 0.03 rounds, far below it
    ("fwd", [12] * 12, 4096, 4160, True),      # 1.5 rounds: the usual share
]


@pytest.mark.parametrize("case", range(len(LONG)))
def test_planner_choice_for_long_contractions(pkg, monkeypatch, case):
    monkeypatch.delenv("GG_SMALL", raising=False)
    op, gm, n, k, few = LONG[case]
    p = torch.empty(16, dtype=torch.uint8, device=DEV).data_ptr()  # plans read no operand
    if op == "dgrad":
        plan = pkg.BackwardPlan("dgrad", pkg.DType.BF16, n, k, gm, p, p, p, _stream())
    else:
        plan = pkg.make_mi355x_backend()
        assert plan.prepare(pkg.GroupedGemmProblem(pkg.DType.BF16, len(gm), n, k, gm, p, p, p), _stream()) == ""
    assert ("few-row" in plan.detail()) == few, plan.detail()
    plan.release()
