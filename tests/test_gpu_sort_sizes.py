"""pic_op_sort at the sizes where its radix passes can go wrong: one item, tiles of 1024 and
4096 items and one off, more tiles than one scan round, digit counts at powers of two, keys
all alike, and the refusal of keys outside the cells (outputs untouched)."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from pic_amd import _lib  # noqa: E402
from pic_amd._lib import check, lib  # noqa: E402

DEV = "cuda:0"


def dptr(t):
    return ctypes.c_void_p(t.data_ptr())


def sort(keys, ncells):
    n = keys.size
    tk = torch.from_numpy(keys).to(DEV)
    perm = torch.full((n,), -1, dtype=torch.int32, device=DEV)
    cnt = torch.full((ncells,), -1, dtype=torch.int32, device=DEV)
    off = torch.full((ncells + 1,), -1, dtype=torch.int32, device=DEV)
    rc = lib.pic_op_sort(dptr(tk), n, ncells, dptr(perm), dptr(cnt), dptr(off), None)
    torch.cuda.synchronize()
    return rc, perm.cpu().numpy(), cnt.cpu().numpy(), off.cpu().numpy()


@pytest.mark.parametrize("n,ncells,same", [
    (1, 1, False), (63, 2, False), (1023, 256, False), (1024, 257, False), (1025, 3, True),
    (100_003, 2, False), (50_000, 65_537, False), (1 << 20, 65_536, False),
    ((1 << 20) + 1, 65_536, False), (1_200_000, 300_000, True), (4_300_000, 70_000, False),
    (2_000, 20_000_000, False)])
def test_sort_matches_stable_argsort(n, ncells, same):
    print(f"sort n={n} ncells={ncells}", flush=True)
    rng = np.random.default_rng(n + ncells)
    keys = np.full(n, ncells - 1, np.int32) if same else rng.integers(0, ncells, n).astype(np.int32)
    rc, perm, cnt, off = sort(keys, ncells)
    check(rc)
    assert np.array_equal(perm, np.argsort(keys, kind="stable"))
    counts = np.bincount(keys, minlength=ncells)
    assert np.array_equal(cnt, counts)
    assert np.array_equal(off, np.concatenate([[0], np.cumsum(counts)]))


@pytest.mark.parametrize("bad", [-1, 70_000])
def test_refused_keys_leave_the_outputs(bad):
    keys = np.zeros(5000, np.int32)
    keys[4321] = bad
    rc, perm, cnt, off = sort(keys, 70_000)
    assert rc == _lib.PIC_ERR_ARG
    assert (perm == -1).all() and (cnt == -1).all() and (off == -1).all()
