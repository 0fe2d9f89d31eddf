"""Page copies against a gather followed by a scatter on the host (MI355X)."""
import numpy as np
import pytest
import torch

from stepquant_amd import _native as N
from tests.helpers import dev

pytestmark = pytest.mark.gpu


# page bytes: multiples of 16 around a workgroup's range, sizes that put every
# page on another even byte, one shorter than a window; counts around the
# change of the lanes per row and past the direct kernel
@pytest.mark.parametrize("page_bytes,n,dtype", [
    (1024, 1, torch.int64), (1040, 64, torch.int32), (400 * 16, 65, torch.int64), (16, 256, torch.int64),
    (1008, 129, torch.int64), (2, 3, torch.int64), (14, 64, torch.int32), (1006, 63, torch.int64),
    (1010, 65, torch.int64), (4098, 128, torch.int64), (722, 256, torch.int32), (1040, 257, torch.int64),
    (722, 257, torch.int64)])
def test_copy_is_gather_then_scatter(page_bytes, n, dtype):
    print(f"case {page_bytes} B, {n} pages", flush=True)
    slots = n + 9
    rng = np.random.default_rng(page_bytes + n)
    pages = rng.integers(0, 256, slots * page_bytes + 64, dtype=np.uint8)
    # overlapping lists: destinations that are sources of other pairs, wrapped
    # and out-of-pool indices among them
    src = rng.permutation(slots)[:n].astype(np.int64)
    dst = rng.permutation(slots)[:n].astype(np.int64)
    if n > 3:
        src[0] -= slots
        dst[1] -= slots
        src[2] = slots
        dst[3] = -slots - 1
    data = torch.from_numpy(pages.copy()).to(dev())
    pool = N.Pool(data=data.data_ptr(), page_bytes=page_bytes, num_slots=slots)
    s, d = (torch.from_numpy(x).to(dev(), dtype) for x in (src, dst))
    temp = torch.empty(n * page_bytes, dtype=torch.uint8, device=dev())
    code = N.dtype_code(s)
    if n <= N.COPY_DIRECT_PAGES:
        N.check(N.lib().sq_copy_slots_direct(pool, N.ptr(s), N.ptr(d), code, n, N.stream_handle()), "copy")
    else:
        assert N.lib().sq_copy_slots_direct(pool, N.ptr(s), N.ptr(d), code, n, N.stream_handle()) == -22
        N.check(N.lib().sq_copy_slots(pool, N.ptr(s), N.ptr(d), code, n, N.ptr(temp), N.stream_handle()), "copy")
    torch.cuda.synchronize()
    ref = pages.copy()
    body = ref[:slots * page_bytes].reshape(slots, page_bytes)
    old = body.copy()
    for a, b in zip(src, dst):
        a, b = (x + slots if x < 0 else x for x in (a, b))
        if 0 <= a < slots and 0 <= b < slots:
            body[b] = old[a]
    assert np.array_equal(data.cpu().numpy(), ref)
