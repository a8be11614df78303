"""The matrix-core kernel's tile pairs at their edges: waves of one tile, an odd number of tiles, rows that end inside
a tile, and partitions that start inside one (split_tokens not a multiple of 16), against the FP64 oracle. Every cache
slot that holds no live token is NaN, so a row read past an end would show."""
import numpy as np
import pytest

from gpu_util import announce, assert_parity, require_gpu

require_gpu()

import torch  # noqa: E402

from oracle.fp64 import dense_attention  # noqa: E402
from paged_decode.layout import Layout  # noqa: E402
from paged_decode.runtime import DecodePlan  # noqa: E402

pytestmark = pytest.mark.gpu

FORMATS = [(torch.float16, None), (torch.bfloat16, None), (torch.float16, torch.float8_e4m3fn),
           (torch.bfloat16, torch.float8_e5m2)]


@pytest.mark.parametrize("q_dtype,kv_dtype", FORMATS)
@pytest.mark.parametrize("heads,kv_heads,dim,page", [(8, 2, 128, 16), (16, 1, 64, 32), (20, 5, 128, 32)])
@pytest.mark.parametrize("split", [256, 100, 1200])
def test_tile_edges_match_oracle(q_dtype, kv_dtype, heads, kv_heads, dim, page, split):
    announce(f"tile pairs q={q_dtype} kv={kv_dtype} {heads}/{kv_heads} D{dim} T{page} split {split}")
    lengths = np.array([1184, 1, 15, 16, 17, 31, 33, 47, 257, 799, 1100, 0], dtype=np.int32)
    width = 1184 // page
    layout = Layout(len(lengths), heads, kv_heads, dim, page, len(lengths) * width)
    rng = np.random.default_rng(split + dim)
    table = rng.permutation(layout.physical_pages).reshape(len(lengths), width).astype(np.int32)
    shape = (layout.physical_pages, page, kv_heads, dim)
    store = kv_dtype or q_dtype
    q = torch.from_numpy(rng.standard_normal((len(lengths), heads, dim), dtype=np.float32)).to(q_dtype)
    k, v = (torch.from_numpy(rng.standard_normal(shape, dtype=np.float32)).to(store) for _ in range(2))
    exact = [t.double().numpy() for t in (q, k, v)]
    dead = torch.ones(shape[:2], dtype=torch.bool)
    for b, n in enumerate(lengths):
        pos = np.arange(n)
        dead[table[b, pos // page], pos % page] = False
    for t in (k, v):
        poisoned = t.float()
        poisoned[dead] = float("nan")
        t.copy_(poisoned.to(store))
    plan = DecodePlan(layout, table, lengths, split_tokens=split)
    out = plan.run(q.cuda(), k.cuda(), v.cuda()).cpu().numpy()
    assert_parity(out, dense_attention(*exact, table, lengths), torch.float16)
    np.testing.assert_array_equal(out[lengths == 0], 0.0)
