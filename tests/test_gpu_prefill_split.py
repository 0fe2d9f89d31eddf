"""Prefill with sequences cut into segments (sq_prefill_plan / sq_prefill_split, MI355X).

Gates that forget slowly (down to 1e-3 a token) carry the state across
segments, so an error in a segment's transition or start state shows.  Bars
as for whole sequences: states rtol 1e-3 / atol 1e-4 of the float64
recurrence, outputs rtol 2^-8 / atol 1e-4; the segments' states are chained
in fp32, which adds about 2^-24 relative a segment.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import check_prefill, check_states, dev, device_plan, make_plan

pytestmark = pytest.mark.gpu


def _case(arch, lens, ck, tokens, monkeypatch, storage="packed", cu_on_device=False):
    from stepquant_amd import _native as N
    from stepquant_amd.kernels.pool import PackedStatePool
    H, HK, K, V = 4, 4 if arch == "kda" else 2, 128, 128
    B, NC = np.shape(ck)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    T = int(cu[-1])
    rng = np.random.default_rng(3)
    bits = np.repeat(np.array([6, 8, 4, 6])[:, None], K, 1) if arch == "gdn" else rng.choice([4, 6, 8, 16], (H, K))
    stream = torch.cuda.Stream() if storage == "byte" else None
    pool = PackedStatePool(device_plan(make_plan(arch, bits, seed=3)), B * (NC + 1) + 1, V, storage=storage,
                           writeback_stream=stream)
    g = torch.Generator().manual_seed(11)
    q, k = (torch.randn(T, HK, K, generator=g).to(torch.bfloat16) for _ in range(2))
    v = torch.randn(T, H, V, generator=g).to(torch.bfloat16)
    shape = (T, H, K) if arch == "kda" else (T, H)
    rate = torch.tensor([1e-3, 5e-3, 5e-2, .5]).reshape(1, H, *([1] * (len(shape) - 2)))
    gate = -rate * torch.rand(shape, generator=g) * 2
    beta = torch.rand(T, H, generator=g)
    init = torch.arange(B)  # slot 0: the first sequence starts from zero
    pool.encode((torch.randn(B, H, K, V, generator=g) * .5).to(dev()), init.to(dev()))
    pool.wait()
    torch.cuda.synchronize()
    lay = O.layout(make_plan(arch, bits, seed=3), V, storage)
    S0 = O.decode_page(pool.data.cpu().numpy(), init.numpy(), make_plan(arch, bits, seed=3), lay, V,
                       storage).astype(np.float64)
    seen = []
    if tokens:
        def plan(desc, offsets, cus=0):
            slots = int(offsets[-1]) // tokens + B
            seen.append(N.PrefillSegments(tokens, -(-max(lens) // tokens), 2 * slots * H * K * V * 4, None))
            return seen[-1]
    else:
        whole = N.prefill_plan

        def plan(desc, offsets, cus=0):
            seen.append(whole(desc, offsets, cus))
            return seen[-1]
    monkeypatch.setattr(N, "prefill_plan", plan)
    pool.keep_prefill_states = True
    offsets = torch.from_numpy(cu)
    out = pool.extend(q.to(dev()), k.to(dev()), v.to(dev()), gate.to(dev()), beta.to(dev()), init,
                      offsets.to(dev()) if cu_on_device else offsets, checkpoints=torch.tensor(ck),
                      checkpoint_slots=torch.arange(B, B + B * NC).reshape(B, NC), init_slots=init, normalize=True,
                      scale=K ** -.5)
    torch.cuda.synchronize()
    assert seen[0].tokens and seen[0].count >= 2
    ref_out, ref_states, _ = O.prefill(q.float().numpy(), k.float().numpy(), v.float().numpy(), gate.numpy(),
                                       beta.numpy(), S0, cu, ck, normalize=True, scale=K ** -.5)
    states = pool.last_prefill[-1].cpu().numpy().reshape(B, NC, H, K, V)
    check_prefill(out, ref_out, f"{arch} {storage} tokens={tokens}")
    for b in range(B):
        for c in range(NC):
            if 0 < ck[b][c] <= lens[b]:
                check_states(states[b, c], ref_states[b, c], f"state b={b} c={c}")


# lengths: below, at and past a segment, empty, one token, many segments;
# checkpoints inside, at and just past a segment's end
LENS = [640, 0, 128, 129, 1, 333]
MARKS = [[128, 640], [0, 0], [64, 128], [128, 129], [1, 0], [130, 333]]


@pytest.mark.parametrize("arch,tokens", [("gdn", 64), ("gdn", 128), ("gdn", 320), ("kda", 32), ("kda", 96),
                                         ("kda", 320)])
def test_segments_against_the_recurrence(arch, tokens, monkeypatch):
    print(f"case {arch} tokens={tokens}", flush=True)
    _case(arch, LENS, MARKS, tokens, monkeypatch)


@pytest.mark.parametrize("arch,storage", [("gdn", "packed"), ("gdn", "byte"), ("kda", "packed"),
                                          ("kda", "byte")])
def test_planned_segments_against_the_recurrence(arch, storage, monkeypatch):
    """The plan's own choice, offsets on the device, byte pages (dense
    initial states) and packed ones."""
    print(f"case {arch} {storage} planned", flush=True)
    _case(arch, [1500, 70], [[700, 1500], [64, 70]], 0, monkeypatch, storage, cu_on_device=True)


def _split(arch, lens, tokens, rate, beta, monkeypatch, repeats=1, planned=None):
    """Final states and outputs of ``repeats`` calls in segments of ``tokens``
    (0: whole sequences) planned for the lengths ``planned`` (default: the
    call's own) with log decays of -rate (times 0 to 2) and the write strengths
    ``beta`` [T], and the float64 recurrence's."""
    from stepquant_amd import _native as N
    from stepquant_amd.kernels.pool import PackedStatePool
    H, HK, K, V = 4, 4 if arch == "kda" else 2, 128, 128
    B, T = len(lens), sum(lens)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    bits = np.full((H, K), 8)
    pool = PackedStatePool(device_plan(make_plan(arch, bits, seed=5)), 2 * B + 1, V)
    g = torch.Generator().manual_seed(17)
    q, k = (torch.randn(T, HK, K, generator=g).to(torch.bfloat16) for _ in range(2))
    v = torch.randn(T, H, V, generator=g).to(torch.bfloat16)
    gate = -rate * 2 * torch.rand((T, H, K) if arch == "kda" else (T, H), generator=g)
    beta = torch.as_tensor(beta, dtype=torch.float32).reshape(T, 1) * (.9 + .1 * torch.rand(T, H, generator=g))
    init = torch.arange(1, B + 1)
    pool.encode((torch.randn(B, H, K, V, generator=g) * .5).to(dev()), init.to(dev()))
    torch.cuda.synchronize()
    plan, lay = make_plan(arch, bits, seed=5), O.layout(make_plan(arch, bits, seed=5), V)
    S0 = O.decode_page(pool.data.cpu().numpy(), init.numpy(), plan, lay, V).astype(np.float64)
    planned = lens if planned is None else planned
    segments = N.PrefillSegments(tokens, -(-max(planned) // tokens),
                                 2 * (sum(planned) // tokens + B) * H * K * V * 4, None) if tokens else \
        N.PrefillSegments()
    monkeypatch.setattr(N, "prefill_plan", lambda desc, offsets, cus=0: segments)
    pool.keep_prefill_states = True
    ck = np.asarray(lens).reshape(B, 1)
    inputs = [t.to(dev()) for t in (q, k, v, gate, beta)]
    got = []
    for _ in range(repeats):
        out = pool.extend(*inputs, init, torch.from_numpy(cu), checkpoints=torch.tensor(ck),
                          checkpoint_slots=torch.arange(B + 1, 2 * B + 1).reshape(B, 1), init_slots=init,
                          normalize=True, scale=K ** -.5)
        torch.cuda.synchronize()
        got.append((out.cpu(), pool.last_prefill[-1].cpu().reshape(B, H, K, V)))
    ref_out, _, ref_states = O.prefill(q.float().numpy(), k.float().numpy(), v.float().numpy(), gate.numpy(),
                                       beta.numpy(), S0, cu, ck, normalize=True, scale=K ** -.5)
    return got, ref_out, ref_states


@pytest.mark.parametrize("arch,tokens", [("gdn", 64), ("gdn", 192), ("kda", 32), ("kda", 96), ("kda", 224)])
def test_segments_with_write_strengths_that_change_by_chunk(arch, tokens, monkeypatch):
    """Write strengths of .98 and .02 in turn from chunk to chunk: a wave that
    scales a chunk's rows with the next chunk's strengths is far off.  Equal
    calls give equal bits."""
    print(f"case {arch} tokens={tokens}", flush=True)
    lens = [960, 417]
    chunk = 64 if arch == "gdn" else 32
    beta = np.concatenate([np.where(np.arange(t) // chunk % 2, .98, .02) for t in lens])
    got, ref_out, ref_states = _split(arch, lens, tokens, 1e-3, beta, monkeypatch, repeats=6)
    for out, states in got:
        assert torch.equal(out, got[0][0]) and torch.equal(states, got[0][1])
    check_prefill(got[0][0], ref_out, f"{arch} tokens={tokens}")
    check_states(got[0][1].numpy(), ref_states)


@pytest.mark.parametrize("arch,tokens,lens,planned", [
    ("gdn", 64, [960, 417], [65, 1]),      # the first in two segments, the second without a slot of its own
    ("gdn", 128, [100, 961], [961, 100]),  # slots for both, the long one elsewhere
    ("gdn", 64, [1, 700], [700, 1]),
    ("kda", 32, [960, 417], [65, 1]),
    ("kda", 96, [417, 960, 5], [961, 1, 1])])
def test_segments_planned_for_other_lengths(arch, tokens, lens, planned, monkeypatch):
    """A plan that belongs to other offsets leaves no token out."""
    print(f"case {arch} tokens={tokens} {lens} planned for {planned}", flush=True)
    beta = np.full(sum(lens), .5)
    got, ref_out, ref_states = _split(arch, lens, tokens, 1e-3, beta, monkeypatch, planned=planned)
    check_prefill(got[0][0], ref_out, f"{arch} tokens={tokens}")
    check_states(got[0][1].numpy(), ref_states)


@pytest.mark.parametrize("arch", ["gdn", "kda"])
@pytest.mark.parametrize("rate,strength", [(1e-5, .01), (1e-4, .1), (1e-3, .5)])
def test_segments_carry_the_state_as_whole_sequences_do(arch, rate, strength, monkeypatch):
    """States that forget little, through 32 segments: as near to float64 as
    the uncut sequence's, plus one fp32 rounding (2^-24) of the state a
    segment.  (Operands of 16 bits in the chain would add 2^-18 a segment.)"""
    lens, beta = [2048], np.full(2048, strength)

    def error(tokens):
        got, _, ref = _split(arch, lens, tokens, rate, beta, monkeypatch)
        return np.linalg.norm(got[0][1].double().numpy() - ref) / np.linalg.norm(ref)

    whole = error(0)
    for tokens in (64, 320):
        split, bound = error(tokens), 1.25 * whole + -(-2048 // tokens) * 2 ** -24
        print(f"case {arch} rate={rate} tokens={tokens}: {split:.2e}, whole {whole:.2e}", flush=True)
        assert split <= bound
