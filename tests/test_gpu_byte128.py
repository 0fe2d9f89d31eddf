"""The K = V = 128 byte-page kernel against the general one (MI355X): the same
operations in the same order, so outputs and pages agree bit for bit, and the
fused step with the split one.
"""
import numpy as np
import pytest
import torch

from stepquant_amd import _native as N
from tests.helpers import dev, device_plan, make_plan

pytestmark = pytest.mark.gpu


def _bits(arch, H, rng):
    if arch == "gdn":
        return np.repeat(np.array([6, 4, 8, 16, 2])[:H, None], 128, 1)
    bits = np.where(rng.random((H, 128)) < .04, 16, rng.choice([2, 4, 6, 8], (H, 128)))
    bits[1] = 16                     # a head of pivot rows only
    bits[2, [0, 15, 16, 63, 64, 127]] = 16  # pivots at the edges of the row groups
    bits[3, bits[3] == 16] = 6       # a head without
    return bits


@pytest.mark.parametrize("arch,group,dtype,gate,scale", [
    ("gdn", 32, torch.bfloat16, torch.float32, .05), ("gdn", 64, torch.float32, torch.bfloat16, .05),
    ("gdn", 128, torch.float16, torch.float32, 3.),
    ("gdn", 128, torch.float32, torch.float32, 1e12), ("kda", 32, torch.bfloat16, torch.float32, .05),
    ("kda", 32, torch.float32, torch.float16, 1e-6)])
def test_byte_kernel_matches_the_general_one(arch, group, dtype, gate, scale):
    from stepquant_amd.kernels.pool import PackedStatePool
    print(f"case {arch} group={group} {dtype} scale={scale}", flush=True)
    rng = np.random.default_rng(2)
    H, K, V, B = 5, 128, 128, 3
    HK = 5 if arch == "kda" else 1
    bits = _bits(arch, H, rng)
    if scale > 1e4:  # past the fp16 range: saturated row and column scales, no pivots
        bits[bits == 16] = 8
    oplan = make_plan(arch, bits, group=group, seed=4)
    pools = [PackedStatePool(device_plan(oplan), B + 2, V, writeback_stream=torch.cuda.Stream(), storage="byte")
             for _ in range(3)]
    assert all(p._desc.flags == N.POOL_FAST_BYTE128 for p in pools)
    pools[1]._desc.flags = 0  # the general kernel
    g = torch.Generator().manual_seed(3)
    r = torch.exp(torch.randn(B, H, K, 1, generator=g) * .5)
    c = torch.exp(torch.randn(B, H, 1, V, generator=g) * .5)
    slots = torch.tensor([4, 0, 2], device=dev())
    pools[0].encode((r * torch.randn(B, H, K, V, generator=g) * c * scale).to(dev()), slots)
    torch.cuda.synchronize()
    for p in pools[1:]:
        p.data.copy_(pools[0].data)
    if arch == "kda":
        # carriers of pivot rows are no one's: they stay as they are
        for p in pools:
            base = int(p.offsets[H * K + 2])
            p.data[:, base + 15:base + K * V:K] = 77
    mixed = torch.randn(B, 2 * HK * K + H * V, generator=g).to(dev(), dtype)
    q, k, v = mixed.split([HK * K, HK * K, H * V], -1)
    gv = torch.randn((B, H, K) if arch == "kda" else (B, H), generator=g).to(dev(), gate)
    beta = torch.randn(B, H, generator=g).to(dev(), gate)
    a_log, dt_bias = (torch.randn(n, generator=g).mul(.3).to(dev(), gate) for n in (H, H * K if arch == "kda" else H))
    torch.cuda.synchronize()
    outs = []
    for p in pools[:2]:
        outs.append(p.step(q, k, v, gv, beta, slots, normalize=True, scale=K ** -.5, a_log=a_log, dt_bias=dt_bias))
        p.wait()
    fused = pools[2]
    out = torch.empty_like(outs[0])
    args, keep = fused._step_args(q.reshape(B, HK, K), k.reshape(B, HK, K), v.reshape(B, H, V), gv, beta, slots, out,
                                  True, K ** -.5, a_log, dt_bias, B, HK)
    N.check(N.lib().sq_decode_step(fused._desc, args, N.stream_handle()), "fused byte step")
    torch.cuda.synchronize()
    assert torch.equal(out, outs[0]) and torch.equal(fused.data, pools[0].data)
    assert torch.equal(outs[0], outs[1]), "outputs differ from the general kernel's"
    assert not outs[0][1].any()
    assert torch.equal(pools[0].data, pools[1].data), "pages differ from the general kernel's"


def test_infinite_pivots_stay_out_of_the_column_scales():
    """A pivot value past the fp16 range comes back as infinity.  The pages stay
    the general kernel's: its column's integer rows saturate, and no scale
    turns NaN."""
    from stepquant_amd.kernels.pool import PackedStatePool
    rng = np.random.default_rng(6)
    H, K, V, B = 2, 128, 128, 2
    bits = rng.choice([4, 6, 8], (H, K))
    bits[0, [3, 70]] = 16
    oplan = make_plan("kda", bits, seed=4)
    pools = [PackedStatePool(device_plan(oplan), B + 1, V, writeback_stream=torch.cuda.Stream(), storage="byte")
             for _ in range(2)]
    assert pools[0]._desc.flags == N.POOL_FAST_BYTE128
    pools[1]._desc.flags = 0  # the general kernel
    g = torch.Generator().manual_seed(8)
    slots = torch.tensor([2, 1], device=dev())
    x = torch.randn(B, H, K, V, generator=g) * .05
    for p in pools:
        p.encode(x.to(dev()), slots)
        p.wait()
    torch.cuda.synchronize()
    at = [int(pools[0].offsets[row]) + 2 * j for row, j in ((3, 0), (3, 65), (70, 66), (70, 127))]
    for p in pools:
        for e in at:
            p.data[:, e + 1] = 0x7c  # the halves' high bytes: infinity
            p.data[:, e] = 0
    q, k, v = (torch.randn(B, H * K, generator=g).to(dev()) for _ in range(3))
    gate = -torch.rand(B, H, K, generator=g).to(dev())
    beta = torch.rand(B, H, generator=g).to(dev())
    torch.cuda.synchronize()
    pages = []
    for p in pools:
        p.step(q, k, v, gate, beta, slots, normalize=True, scale=K ** -.5)
        p.wait()
        torch.cuda.synchronize()
        for e in at:  # infinity less infinity: NaN, of either payload
            half = p.data[slots, e:e + 2].contiguous().view(torch.float16)
            assert torch.isnan(half).all()
            p.data[:, e:e + 2] = 0
        pages.append(p.data[slots])
    column = int(pools[0].columns[0])
    scales = [d[:, column:column + 2 * V].contiguous().view(torch.float16) for d in pages]
    assert torch.isfinite(scales[1]).all() and torch.equal(scales[0], scales[1])
    assert torch.equal(pages[0], pages[1])
