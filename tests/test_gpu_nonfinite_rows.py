"""A coordinate that is no finite number, in the allocation-free pair call.
Where the atom's cell holds few atoms the row of the atom itself is the only
one that meets it: the filter must keep a row whose distance to the cell's box
is no number (infinity is, in the box that it widens itself), so that the
call's status flags it."""
import numpy as np
import pytest
import torch

from omegagene_amd.celeste import ZeroDipole, pairwise_ljzd_noalloc

pytestmark = pytest.mark.gpu

FLAG_NAN = 8
SELF = sum(((0xff << a) & 0xff) << (8 * a) for a in range(8))   # bit a2 * 8 + a1 set for a1 >= a2: skipped


def _two_atoms(n_cells, second):
    """Cell 0 holds an atom in slot 0, `second` in slot 1 and dummies after them, and is paired with itself;
    the other cells hold dummies and no pairs."""
    x = np.zeros((8 * n_cells, 4), np.float32)
    x[:, :3] = 20.0
    x[0] = [10.0, 10.0, 10.0, 0.5]
    x[1, :3], x[1, 3] = second, -0.5
    x[2:8, :3] = second
    mask = SELF
    for a2 in range(8):
        mask |= 0xfc << (8 * a2)        # cell1's dummies
        if a2 > 1:
            mask |= 0xff << (8 * a2)    # cell2's dummies
    head = np.ones(n_cells + 1, np.int32)
    head[0] = 0
    dev = torch.device("cuda:0")
    put = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    d = [put(x), torch.zeros(8 * n_cells, dtype=torch.int32, device=dev),
         put(np.array([[[600.0, 6e5]]], np.float32)), put(head), put(np.zeros(1, np.int32)),
         put(np.array([mask], np.uint64).view(np.int64))]
    work = torch.zeros((8 * n_cells, 3), dtype=torch.float64, device=dev)
    energy = torch.zeros(2, dtype=torch.float64, device=dev)
    flags = torch.zeros(1, dtype=torch.int32, device=dev)
    pairwise_ljzd_noalloc(d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), 1, d[3].data_ptr(), d[4].data_ptr(),
                          d[5].data_ptr(), n_cells, np.full(3, 40.0, np.float32), 12.0, ZeroDipole(12.0),
                          work.data_ptr(), energy.data_ptr(), flags.data_ptr(),
                          torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return work.cpu().numpy(), int(flags.cpu()[0])


@pytest.mark.parametrize("n_cells", [4, 904])   # four waves on a cell; a wave per cell
def test_row_without_a_number_is_flagged(n_cells):
    print("[gpu-test] non-finite row,", n_cells, "cells", flush=True)
    w, f = _two_atoms(n_cells, [13.0, 10.0, 10.0])
    assert f == 0 and w[0, 0] < 0.0 < w[1, 0]
    for k in range(3):
        for x in (np.nan, np.inf, -np.inf):
            at = [13.0, 10.0, 10.0]
            at[k] = x
            assert _two_atoms(n_cells, at)[1] & FLAG_NAN, (k, x)
    w, f = _two_atoms(n_cells, [13.0, 10.0, 10.0])
    assert f == 0 and w[0, 0] < 0.0 < w[1, 0]
