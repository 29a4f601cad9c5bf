"""The octree built from sorted keys against the oracle's, array by array: key counts around the bucket size and the
blocks of the build, clusters down to the deepest level, equal keys, and removed particles (keys past the curve)."""
import numpy as np
import pytest

from sphexa_amd import abi

from test_gpu_tree_update import assert_same_tree, gpu_tree

pytestmark = pytest.mark.gpu

END = 1 << 63


def keys_of(kind, n, rng):
    k = rng.integers(0, END, n, dtype=np.uint64)
    if kind == "cluster":  # every scale down to the deepest level
        k = (rng.integers(0, END, n, dtype=np.uint64) >> rng.integers(0, 63, n).astype(np.uint64)) ^ np.uint64(0x2AAAAAAAAAAAAAAA)
    elif kind == "equal":
        k[: n // 2] = 0
        k[n // 2:] = END - 1
    elif kind == "one":
        k[:] = 12345678901234567
    elif kind == "removed":
        k[-(n // 3):] = END
    elif kind == "all_removed":
        k[:] = END
    return np.sort(k)


@pytest.mark.parametrize("bucket", [1, 8, 64])
@pytest.mark.parametrize("kind", ["uniform", "cluster", "equal", "one", "removed", "all_removed"])
def test_tree_equals_the_oracles(orc, kind, bucket):
    import torch

    from oracle import oracle as O
    from sphexa_amd.lib import Workspace

    ws = Workspace(0)
    rng = np.random.default_rng(bucket)
    box = abi.Box.make((-1.0, 0.0, 2.0), (1.0, 3.0, 2.5), (0, 1, 0))
    for n in (0, 1, 2, bucket, bucket + 1, 63, 65, 511, 513, 2047, 2048, 2049, 4097, 50021):
        keys = keys_of(kind, n, rng)
        if n < 3 and "removed" in kind:
            continue
        d = torch.from_numpy(keys.view(np.int64)).cuda()
        ws.build_tree(d, box, bucket)
        # a removed particle counts in the curve's last cell
        want = O.Tree(orc, np.minimum(keys, np.uint64(END - 1)), box, bucket)
        assert_same_tree(gpu_tree(ws), want, f"{kind} n={n} bucket={bucket}")
