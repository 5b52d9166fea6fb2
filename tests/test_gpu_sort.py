"""The forms of the radix sort at their edges (rows of one work-group, tile sizes, digit widths, key widths, the inverse
in a pass of its own) against a stable host sort, and ptv3_serialize against its two parts."""
import numpy as np
import pytest
import torch

from oracle import serialization as OS
from gpu_util import DEV, to_dev, unique_voxels

pytestmark = pytest.mark.gpu


# 8-bit digits: 24, 32, 40; 9-bit: 25, 36, 41 (wide), 33 (cut to 32 bits after the first pass); 1: a single pass
@pytest.mark.parametrize("bits", [1, 24, 25, 32, 33, 36, 41, 63])
@pytest.mark.parametrize("n,k", [(1, 2), (2047, 3), (2049, 1), (4096, 2), (4097, 2), (2048 * 9 + 1, 4), (4096 * 70 - 1, 3),
                                 (6144 * 40 + 5, 10)])
def test_argsort_forms(n, k, bits):
    from pointtransformerv3_amd import ops
    rng = np.random.default_rng(n + bits)
    code = rng.integers(0, 1 << bits, size=(k, n), dtype=np.int64)
    code[0] >>= bits // 2          # ties, and digits that are equal in a whole wave
    want = np.argsort(code, axis=1, kind="stable")
    order, inverse = ops.argsort_rows(to_dev(code), bits)
    assert np.array_equal(order.cpu().numpy(), want)
    assert torch.equal(inverse.gather(1, order), torch.arange(n, device=DEV).expand(k, n))


@pytest.mark.parametrize("limit", [-1, 0, 3])
@pytest.mark.parametrize("n,k,bits", [(4097, 2, 24), (2048 * 9 + 1, 4, 32), (2048 * 66 + 5, 2, 33), (4096 * 20 - 1, 3, 41), (6144 * 20 + 5, 4, 25)])
def test_tiles_that_do_not_wait_count_the_keys_in_front_of_them(n, k, bits, limit):
    """The way out of a wait that lasts too long, forced from the host: the same order, whoever does the counting."""
    from pointtransformerv3_amd import _lib
    lib = _lib.load()
    code = np.random.default_rng(n).integers(0, 1 << bits, size=(k, n), dtype=np.int64)
    code[0] >>= bits // 2
    dev = to_dev(code)
    order, inverse = torch.full((2, k, n), -1, dtype=torch.int64, device=DEV)
    nbytes = lib.ptv3_argsort_workspace_bytes(n, k)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    assert lib.ptv3_argsort_impatient(dev.data_ptr(), n, k, bits, limit, order.data_ptr(), inverse.data_ptr(), ws.data_ptr(), nbytes,
                                      torch.cuda.current_stream().cuda_stream) == 0
    assert np.array_equal(order.cpu().numpy(), np.argsort(code, axis=1, kind="stable"))
    assert torch.equal(inverse.gather(1, order), torch.arange(n, device=DEV).expand(k, n))


def test_argsort_of_a_row_with_its_own_inverse_pass():
    from pointtransformerv3_amd import ops
    n = (1 << 20) + 77
    g = torch.Generator(device=DEV).manual_seed(0)
    code = torch.randint(0, 1 << 31, (2, n), generator=g, device=DEV)
    order, inverse = ops.argsort_rows(code, 33)
    assert torch.equal(order, torch.sort(code, dim=1, stable=True)[1])
    assert torch.equal(inverse.gather(1, order), torch.arange(n, device=DEV).expand(2, n))


@pytest.mark.parametrize("n,extent,nb", [(1, 4, 1), (2048, 32, 2), (4096, 32, 5), (5000, 600, 1), (70_000, 1500, 3)])
def test_serialize_is_encode_and_argsort(n, extent, nb):
    from pointtransformerv3_amd import ops
    g, batch, _ = unique_voxels(np.random.default_rng(n), n, extent, nb)
    depth, code, order, inverse = OS.serialize(g, batch)
    bits = 3 * depth + max(1, (nb - 1).bit_length())
    got = ops.serialize(to_dev(g), to_dev(batch), depth, OS.ORDERS, bits)
    for a, b in zip(got, (code, order, inverse)):
        assert np.array_equal(a.cpu().numpy(), b)


@pytest.mark.parametrize("n", [1, 255, 400_001])
def test_scene_facts(n):
    from pointtransformerv3_amd.levels import SceneFacts
    rng = np.random.default_rng(n)
    grid = rng.integers(-3, 5000, size=(n, 3)).astype(np.int32)
    ends = np.sort(rng.integers(0, n + 1, size=300))
    ends[-1] = n
    top, got = SceneFacts(to_dev(grid), to_dev(ends.astype(np.int64))).get()
    assert top == grid.max(0).tolist() and got == ends.tolist()
