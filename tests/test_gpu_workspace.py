"""Memory that the operators keep between calls: a call with a temporary too large to keep leaves the
rest of its blocks (and those of other calls) for the next one, and a destroyed context gives all of
it back."""
import ctypes

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import Simulation, _lib  # noqa: E402
from pic_amd._lib import check, lib  # noqa: E402

DEV = "cuda:0"
MIB = 1 << 20


def dptr(t):
    return ctypes.c_void_p(t.data_ptr())


def give_back():
    """Frees what the operators keep."""
    with Simulation(_lib.default_config(nx=16, ny=16, capacity=64)):
        pass


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info(0)[0]


def test_large_temporary_leaves_the_rest():
    """Deposit of 33.6 M positions on 2048^2: 269 MB of moved positions (freed at the end) beside the
    32 MiB of sums and the counts (kept)."""
    n, side = 33_600_000, 2048
    x, y = (torch.rand(n, device=DEV) for _ in range(2))
    rho = torch.empty(side * side, dtype=torch.float64, device=DEV)
    g = _lib.pic_grid(side, side, 1.0, 1.0)
    give_back()
    before = free_bytes()
    for _ in range(2):
        check(lib.pic_op_deposit(dptr(x), dptr(y), n, _lib.PIC_FP32, ctypes.byref(g), 1.0, dptr(rho),
                                 None))
        kept = before - free_bytes()
        assert 32 * MIB <= kept <= 256 * MIB, kept
    give_back()
    assert before - free_bytes() < 8 * MIB


def test_large_temporaries_of_one_call():
    """Sort of 50 M keys: three temporaries of 200 MB, of which one is kept, and small ones."""
    n, cells = 50_000_000, 1 << 16
    keys = torch.randint(0, cells, (n,), dtype=torch.int32, device=DEV)
    perm = torch.empty(n, dtype=torch.int32, device=DEV)
    counts = torch.empty(cells, dtype=torch.int32, device=DEV)
    offsets = torch.empty(cells + 1, dtype=torch.int32, device=DEV)
    give_back()
    before = free_bytes()
    for _ in range(2):
        check(lib.pic_op_sort(dptr(keys), n, cells, dptr(perm), dptr(counts), dptr(offsets), None))
        kept = before - free_bytes()
        assert 190 * MIB <= kept <= 256 * MIB, kept
    give_back()
    assert before - free_bytes() < 8 * MIB
