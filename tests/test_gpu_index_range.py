"""The index check of the batch calls: the exact smallest and largest values at
the edges of its workgroups (integers: equality), and the refusals built on it."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no HIP device", allow_module_level=True)

from frealign_amd import _native as N  # noqa: E402
from frealign_amd import api  # noqa: E402


@pytest.mark.parametrize("n", [1, 63, 64, 255, 257, 4096, 4097, 64 * 4096, 1_000_003])
def test_range(n):
    ctx = api.Context(0)
    rng = np.random.default_rng(n)
    for at_lo, at_hi in ((0, n - 1), (n - 1, 0), (n // 2, n // 3)):
        v = rng.integers(-5, 1000, n).astype(np.int32)
        v[at_hi] = 2**31 - 1 if n > 1 else 7
        v[at_lo] = -(2**31) if n > 1 else 7
        d = torch.from_numpy(v).cuda()
        lo, hi = C.c_int(), C.c_int()
        N.check(N.lib().fr_index_range(ctx.h, n, C.c_void_p(d.data_ptr()), C.byref(lo),
                                       C.byref(hi)), "fr_index_range")
        assert (lo.value, hi.value) == (v.min(), v.max())
    top = torch.arange(n, dtype=torch.int32, device="cuda")
    assert ctx._inside(top, n) and not ctx._inside(top, n - 1)
    assert not ctx._inside(top - 1, n)
    ctx.close()


def test_refusals():
    """A class label or particle index out of range on either side is refused."""
    ctx = api.Context(0)
    shape = (16, 4, 1, 3)
    count = api.cnn_param_count(*shape)
    wq, grad = (torch.zeros(count, device="cuda") for _ in range(2))
    img = torch.zeros((2, 16, 16), device="cuda")
    for bad in ([0, 3], [-1, 2]):
        with pytest.raises(ValueError):
            ctx.cnn_gradients(shape, wq, img, torch.tensor(bad, dtype=torch.int32, device="cuda"),
                              grad)
    ns, jc = 64, 33
    vol = torch.zeros((ns, ns, jc), dtype=torch.complex64, device="cuda")
    ctff = torch.zeros((2, 2, ns, jc), dtype=torch.complex64, device="cuda")
    dm = torch.eye(3, device="cuda").repeat(2, 1, 1).contiguous()
    for bad in ([0, 2], [-1, 1]):
        with pytest.raises(ValueError):
            ctx.pextract(ns, vol, dm, ctff, torch.tensor(bad, dtype=torch.int32, device="cuda"))
    ctx.close()
