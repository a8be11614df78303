"""The FP32 kernel's four-token tiles at their edges: rows that end inside a tile or a ring of tiles, partitions that
start inside a tile (split_tokens not a multiple of 4), partly filled head groups, private and shared pages, against the
FP64 oracle at the bound of the other FP32 tests. Every cache slot that holds no live token is NaN, so a row read past
an end would show."""
import numpy as np
import pytest

from gpu_util import announce, assert_parity, require_gpu

require_gpu()

import torch  # noqa: E402

from oracle.fp64 import dense_attention  # noqa: E402
from paged_decode.layout import Layout  # noqa: E402
from paged_decode.runtime import DecodePlan  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads", [(2, 2), (4, 2), (6, 2), (8, 2), (5, 1), (16, 2), (36, 3)])
@pytest.mark.parametrize("dim,page", [(64, 32), (128, 16)])
@pytest.mark.parametrize("split,shared", [(256, 0), (102, 0), (37, 2)])
def test_fp32_tile_edges_match_oracle(heads, kv_heads, dim, page, split, shared):
    announce(f"fp32 tiles {heads}/{kv_heads} D{dim} T{page} split {split} shared {shared}")
    lengths = np.array([1184, 1, 3, 4, 5, 7, 9, 31, 33, 257, 799, 1101, 0], dtype=np.int32)
    width = 1184 // page
    layout = Layout(len(lengths), heads, kv_heads, dim, page, len(lengths) * width)
    rng = np.random.default_rng(split + dim)
    table = rng.permutation(layout.physical_pages).reshape(len(lengths), width).astype(np.int32)
    table[:, :shared] = table[0, :shared]
    shape = (layout.physical_pages, page, kv_heads, dim)
    q = torch.from_numpy(rng.standard_normal((len(lengths), heads, dim), dtype=np.float32))
    k, v = (torch.from_numpy(rng.standard_normal(shape, dtype=np.float32)) for _ in range(2))
    dead = torch.ones(shape[:2], dtype=torch.bool)
    for b, n in enumerate(lengths):
        pos = np.arange(n)
        dead[table[b, pos // page], pos % page] = False
    exact = [t.double().numpy() for t in (q, k, v)]
    k[dead] = v[dead] = float("nan")
    plan = DecodePlan(layout, table, lengths, split_tokens=split)
    out = plan.run(q.cuda(), k.cuda(), v.cuda()).cpu().numpy()
    assert_parity(out, dense_attention(*exact, table, lengths), torch.float32)
    np.testing.assert_array_equal(out[lengths == 0], 0.0)
