"""sq_prefill_plan on the host: which calls are cut into segments, and how."""
import numpy as np
import pytest
import torch

from stepquant_amd import _native as N

CUS = 256


def _plan(lens, heads=32, arch="gdn"):
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    return N.prefill_plan(N.Pool(heads=heads, keys=128, values=128, kda=int(arch == "kda")), cu, CUS)


@pytest.mark.parametrize("lens,heads", [([2048] * 8, 32), ([333] * 24, 32), ([64], 32), ([4096] * 4, 32), ([], 32),
                                        ([0, 0], 8), ([8192], 300)])
def test_whole_sequences(lens, heads):
    """Calls that fill the device, short ones and empty ones stay whole."""
    plan = _plan(lens, heads)
    assert (plan.tokens, plan.count, plan.workspace_bytes) == (0, 0, 0)


@pytest.mark.parametrize("arch", ["gdn", "kda"])
@pytest.mark.parametrize("lens,heads", [([8192], 32), ([8192], 8), ([8192], 4), ([3000, 17, 0, 900], 16), ([6972, 6972], 16),
                                        ([4096, 1], 32), ([65536], 1)])
def test_segments_cover_the_sequences_and_fit_the_device(lens, heads, arch):
    plan = _plan(lens, heads, arch)
    n = [-(-t // plan.tokens) for t in lens]
    assert plan.tokens % (64 if arch == "gdn" else 32) == 0 and plan.count == max(n) >= 2
    assert sum(n) * heads <= CUS and sum(max(0, x - 1) for x in n) * heads <= CUS
    # every segment's workspace slot, t0 / tokens + b + s, is its own and inside the workspace
    starts = np.concatenate([[0], np.cumsum(lens)])[:-1]
    slots = [t0 // plan.tokens + b + s for b, (t0, x) in enumerate(zip(starts, n)) for s in range(x)]
    assert len(set(slots)) == len(slots)
    assert (max(slots) + 1) * heads * 2 * 65536 <= plan.workspace_bytes


def test_split_arguments_are_checked():
    """Segments that are not whole chunks, or without their workspace, are refused before any launch."""
    L = N.lib()
    pool = N.Pool(data=1, page_bytes=64, num_slots=1, bits=1, offsets=1, rows=1, columns=1, impact=1, head_meta=1,
                  heads=2, keys=128, values=128, group=32, flags=N.POOL_FAST_GDN128)
    args = N.PrefillArgs(q=16, k=16, v=16, g=16, beta=16, out=16, cu_seqlens=16, init_slots=16, batch=1, key_heads=2,
                         qkv_dtype=N.BF16, gate_dtype=N.F32, out_dtype=N.BF16, slots_dtype=N.I64)
    state = 2 * 2 * 65536
    for segments in (N.PrefillSegments(60, 2, state, 16), N.PrefillSegments(64, 1, state, 16),
                     N.PrefillSegments(64, 2, state, None), N.PrefillSegments(64, 2, state // 2, 16),
                     N.PrefillSegments(64, 2, state + 16, 16), N.PrefillSegments(64, 2, state, 8)):
        assert L.sq_prefill_split(pool, args, segments, None) == -22
    with pytest.raises(ValueError):
        N.check(L.sq_prefill_plan(pool, None, 1, CUS, N.PrefillSegments()), "plan")


@pytest.mark.parametrize("tokens,split", [(256, False), (640, True)])
@pytest.mark.parametrize("batch,heads", [(2, 32), (1, 64), (3, 16), (7, 8)])
def test_short_kda_sequences_stay_whole(tokens, split, batch, heads):
    """256 tokens in segments of 64 measured slower than whole, 640 tokens faster cut."""
    assert bool(_plan([tokens] * batch, heads, "kda").tokens) is split
