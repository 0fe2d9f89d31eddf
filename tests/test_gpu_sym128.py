"""Symmetric, dual-axis and fp32 format steps at K = V = 128: the width-compiled kernel against the
general one (MI355X), the same operations in the same order, so outputs and
pages agree bit for bit; zeros, infinities and NaN, scales at both ends of
fp16, and pages on odd offsets among them."""
import pytest
import torch

from tests.helpers import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,arch,dtype,gate,pad", [
    (4, "gdn", torch.bfloat16, torch.float32, 0), (6, "gdn", torch.float32, torch.bfloat16, 0),
    (8, "kda", torch.float16, torch.float32, 0), (6, "kda", torch.bfloat16, torch.float16, 4),
    (32, "gdn", torch.bfloat16, torch.float32, 0), (32, "kda", torch.float32, torch.bfloat16, 4),
    ("dsq4", "gdn", torch.bfloat16, torch.float32, 0), ("dsq6", "kda", torch.float32, torch.bfloat16, 0),
    ("dsq6", "gdn", torch.float16, torch.float32, 4), ("dsq8", "gdn", torch.bfloat16, torch.float32, 2),
    (4, "gdn", torch.bfloat16, torch.float32, 2), (8, "gdn", torch.float32, torch.float32, 6)])
def test_sym_kernel_matches_the_general_one(bits, arch, dtype, gate, pad):
    """FP32 pages among them (32 bits).  ``pad`` bytes before the first code row move every region off its alignment."""
    from stepquant_amd.formats import FormatPlan, StateFormat, get_format
    from stepquant_amd.kernels.format_pool import FormatStatePool, format_layout
    print(f"case {bits} {arch} {dtype} pad={pad}", flush=True)
    H, K, V, B = 3, 128, 128, 4
    HK = 3 if arch == "kda" else 1
    name, bits = str(bits), int(str(bits)[-2:].strip("q"))
    if "dsq" in name:
        spec = StateFormat(f"dsq_int{bits}", "dsq", bits, 128, "k")
    else:
        spec = get_format(f"sym_int{bits}_g128" if bits < 32 else "fp32")
    plan = FormatPlan(arch, torch.full((H, K), bits).to(dev()), torch.ones(H, K, device=dev()))
    offsets, rows, columns, size = format_layout(plan, V, spec)
    if pad:
        offsets, rows, size = [o + pad for o in offsets], [r + 4 * pad for r in rows], size + 8 * pad
        columns = [c + 8 * pad for c in columns]
    pools = [FormatStatePool(plan, B + 1, V, spec, layout=(offsets, rows, columns, size)) for _ in range(2)]
    assert pools[0]._fdesc.flags
    pools[1]._fdesc.flags = 0  # rows read from the page by the general kernel
    g = torch.Generator().manual_seed(bits)
    slots = torch.tensor([3, 1, 0, 4], device=dev())
    x = torch.randn(B, H, K, V, generator=g)
    x[0, 0] *= torch.exp(torch.randn(K, 1, generator=g) * 6)
    x[1, 0, :8] = 0.
    x[1, 1] *= 1e30
    x[1, 2] *= 1e-30
    x[3, 0, 5] = float("inf")
    x[3, 1, 7, 9] = float("nan")
    for p in pools:
        p.encode(x.to(dev()), slots)
    mixed = torch.randn(B, 2 * HK * K + H * V, generator=g).to(dev(), dtype)
    q, k, v = mixed.split([HK * K, HK * K, H * V], -1)
    k[0, :4] = 0.
    gv = torch.randn((B, H, K) if arch == "kda" else (B, H), generator=g).to(dev(), gate)
    beta = torch.randn(B, H, generator=g).to(dev(), gate)
    a_log, dt_bias = (torch.randn(n, generator=g).mul(.3).to(dev(), gate) for n in (H, H * K if arch == "kda" else H))
    for raw in (True, False):
        outs = [p.step(q, k, v, gv if raw else -gv.abs(), beta, slots, normalize=raw, scale=K ** -.5,
                       a_log=a_log if raw else None, dt_bias=dt_bias if raw else None) for p in pools]
        torch.cuda.synchronize()
        a, b = (o.view(torch.int32 if o.dtype == torch.float32 else torch.int16) for o in outs)
        nan = torch.isnan(outs[1])
        assert torch.equal(a[~nan], b[~nan]) and torch.equal(torch.isnan(outs[0]), nan)
        a, b = pools[0].data, pools[1].data
        if bits == 32:  # values: bit for bit but for the payload of a NaN, which the operand order chooses
            a, b = (d.contiguous().view(torch.float32) for d in (a, b))
            assert torch.equal(torch.isnan(a), torch.isnan(b))
            a, b = (torch.where(torch.isnan(d), torch.zeros_like(d), d).view(torch.int32) for d in (a, b))
        assert torch.equal(a, b), "pages differ"
        assert not outs[0][2].any()
