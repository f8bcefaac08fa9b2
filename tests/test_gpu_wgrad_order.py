"""The persistent wgrad kernel's walk of ragged groups by descending K steps, through the C ABI.

A tile's sums do not depend on when its workgroup runs it: device-size plans (the order found in the
kernel) and host-size plans (in the tile descriptors) give the bits of a host-size plan that walks the
group table in the groups' own order, and every output is within the bound of a torch fp32 product
that the 128 x 128 kernel's test derives. Fewer tiles than CUs, whole rounds and partial ones, empty
and equal groups, all 64 lanes of the in-kernel table and a 65th group past it.
"""
import pytest
import torch

from test_gpu_wgrad_few import Case

pytestmark = pytest.mark.gpu

SHAPES = [
    ([5, 700, 0, 64, 300, 300], 272, 528),               # 36 tiles, one partial round
    ([900, 0, 130, 1500], 2064, 2032),                   # 288 tiles: a whole round and a partial one
    ([40, 600, 333, 1, 257, 0, 512, 511], 2048, 2048),   # 512: two whole rounds
    ([0, 300, 100, 999, 20, 64, 65, 640], 2064, 2320),   # 720: two and a partial one
    ([(37 * g) % 300 for g in range(64)], 528, 1040),    # 960: every lane of the table
    ([(37 * g) % 300 for g in range(65)], 272, 272),     # no in-kernel table
]


@pytest.mark.parametrize("ta,tb", [("bf16", "bf16"), ("fp16", "fp16"), ("e5m2", "e4m3")])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_wgrad_walk_order(pkg, monkeypatch, shape, ta, tb):
    monkeypatch.delenv("GG_SMALL", raising=False)
    monkeypatch.setenv("GG_WFEW", "0")
    gm, n, k = SHAPES[shape]
    outs = {}
    for walk in ("table", "descriptors", "device"):
        monkeypatch.setenv("GG_TILE_DESC", "0" if walk == "table" else "1")
        print(f"[wgrad order] {ta} x {tb} shape {shape} {walk}", flush=True)
        c = Case(pkg, ta, tb, gm, n, k, walk == "device", seed=shape).run()
        assert "persistent" in c.plan.detail(), c.plan.detail()
        if walk == "device":
            assert ("in-kernel table" in c.plan.detail()) == (len(gm) <= 64)
        c.check()
        outs[walk] = c.out.clone()
        c.close()
    for walk in ("descriptors", "device"):
        assert torch.equal(outs[walk].view(torch.int16), outs["table"].view(torch.int16)), walk
