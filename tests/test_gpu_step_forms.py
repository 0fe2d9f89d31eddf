"""Forms of a decode step's arguments (MI355X): the packed argument block that
the usual call takes against the views and conversions of every other one.
All forms of one step give the same bits; what is refused is refused by both."""
import numpy as np
import pytest
import torch

from tests.helpers import dev, device_plan, make_plan

pytestmark = pytest.mark.gpu


def _forms(q, k, v, g, beta, slots, B, HK, H, K):
    wide = torch.cat([q, k, v], 1)
    a, b, c = wide.split([HK * K, HK * K, v.shape[1]], -1)
    yield "rows", (q, k, v, g, beta, slots)
    yield "views of one row", (a, b, c, g, beta, slots)
    yield "heads apart", (q.view(B, HK, K), k.view(B, HK, K), v.view(B, H, -1), g, beta, slots)
    yield "a leading axis", (q[None], k[None], v[None], g[None], beta[None], slots)
    yield "strided heads", (torch.stack([q.view(B, HK, K)] * 2, 2)[:, :, 0], k, v, g, beta, slots)
    yield "int32 slots", (q, k, v, g, beta, slots.int())
    yield "host slots", (q, k, v, g, beta, slots.cpu())
    yield "a slot column", (q, k, v, g, beta, slots[:, None])
    yield "strided slots", (q, k, v, g, beta, torch.stack([slots, slots], 1)[:, 0])
    yield "transposed gates", (q, k, v, g, beta.t().contiguous().t(), slots)
    yield "host gates", (q, k, v, g.cpu(), beta.cpu(), slots)
    yield "float64 gates", (q, k, v, g.double(), beta.double(), slots)
    yield "mixed types", (q.float(), k, v, g, beta, slots)


@pytest.mark.parametrize("arch,kind", [("gdn", "fused"), ("kda", "fused"), ("gdn", "split"), ("gdn", "sym")])
@pytest.mark.parametrize("raw", [True, False])
def test_every_form_of_a_step_gives_the_same_bits(arch, kind, raw):
    from stepquant_amd.formats import FormatPlan, get_format
    from stepquant_amd.kernels.format_pool import FormatStatePool
    from stepquant_amd.kernels.pool import PackedStatePool
    print(f"case {arch} {kind} raw={raw}", flush=True)
    H, K, V, B = 4, 128, 128, 3
    HK = 4 if arch == "kda" else 2
    if kind == "sym":
        plan = FormatPlan(arch, torch.full((H, K), 6).to(dev()), torch.ones(H, K, device=dev()))
        pool = FormatStatePool(plan, B + 1, V, get_format("sym_int6_g128"))
    else:
        pool = PackedStatePool(device_plan(make_plan(arch, np.full((H, K), 6), seed=1)), B + 1, V,
                               writeback_stream=torch.cuda.Stream() if kind == "split" else None)
    g = torch.Generator().manual_seed(5)
    slots = torch.tensor([2, 3, 1], device=dev())
    pool.encode((torch.randn(B, H, K, V, generator=g) * .1).to(dev()), slots)
    torch.cuda.synchronize()
    pages = pool.data.clone()
    q, k = (torch.randn(B, HK * K, generator=g).to(dev(), torch.bfloat16) for _ in range(2))
    v = torch.randn(B, H * V, generator=g).to(dev(), torch.bfloat16)
    gate = -torch.rand((B, H, K) if arch == "kda" else (B, H), generator=g).to(dev())
    beta = torch.rand(B, H, generator=g).to(dev())
    al, db = ((torch.randn(n, generator=g) * .3).to(dev()) for n in (H, H * K if arch == "kda" else H))
    kw = dict(normalize=True, scale=K ** -.5, a_log=al if raw else None, dt_bias=db if raw else None)
    ref = None
    for name, args in _forms(q, k, v, gate, beta, slots, B, HK, H, K):
        pool.wait()
        pool.data.copy_(pages)
        out = pool.step(*args, **kw)
        pool.wait()
        torch.cuda.synchronize()
        got = (out.to(torch.bfloat16).reshape(B, H, V), pool.data.clone())
        ref = ref or got
        assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1]), name
    for bad in (dict(kw, a_log=None, dt_bias=db), dict(kw, a_log=al[:2], dt_bias=db), dict(kw, a_log=al, dt_bias=db[:2])):
        with pytest.raises(ValueError):
            pool.step(q, k, v, gate, beta, slots, **bad)
    for args in ((q, k, v, gate[:2], beta, slots), (q, k, v, gate, beta[:, :2], slots), (q, k[:, :K], v, gate, beta, slots)):
        with pytest.raises((ValueError, RuntimeError)):
            pool.step(*args, **kw)
