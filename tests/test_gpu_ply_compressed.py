"""Compressed PLY at the edges of the decode's groups of 128 splats and of the
chunks of 256, for every SH count, bit for bit against the restatement."""
import numpy as np
import pytest

from tests import ply_files as F
from tests.test_gpu_ply import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rest", [0, 9, 24, 45, 72])
@pytest.mark.parametrize("n,sub", [(1, None), (127, None), (128, None), (129, None), (257, None), (385, 3), (512, 4)])
def test_group_edges(gpu, n, sub, rest):
    print(f"[case] compressed ply n={n} sub={sub} rest={rest}", flush=True)
    rng = np.random.default_rng(n * 100 + rest)
    cm, vert, sh, _ = F.compressed_elements(rng, n, rest, True)
    els = [("chunk", cm), ("vertex", vert)] + ([("sh", sh)] if sh is not None else [])
    compare(F.write_ply("binary_little_endian", els), sub)
