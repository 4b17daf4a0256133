"""Row argmax over segments (few rows): the first index of the maximum, ties
across a segment's edge, NaN, rows off 16-byte alignment, against torch."""
import pytest
import torch

from cast_amd import _lib, greedy_accept

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,V,pad", [(1, 151936, 0), (3, 40001, 3), (70, 32000, 0), (128, 32000, 0),
                                        (129, 128256, 8), (300, 33000, 0), (301, 4096, 0), (5, 100, 0)])
def test_segmented_argmax_matches_torch(gpu, rows, V, pad, dtype):
    dt = {torch.bfloat16: _lib.BF16, torch.float16: _lib.FP16, torch.float32: _lib.FP32}[dtype]
    need = _lib.load().cast_greedy_accept_workspace_size(rows, V, dt)
    print(f"case accept-segments rows={rows} V={V} pad={pad} {dtype}: workspace {need}", flush=True)
    f32 = dt == _lib.FP32
    assert (need > 0) == (rows <= (300 if f32 else 128) and V * (4 if f32 else 2) >= 2 * 16384)
    g = torch.Generator(gpu).manual_seed(rows + V)
    x = torch.randn(rows, V + pad, generator=g, device=gpu).to(dtype)[:, :V]
    per = need // (8 * rows)                       # segments of a row
    edge = (V // per) if per > 1 else V // 2
    for r in range(rows):
        kind = r % 6
        if kind == 1:                              # the maximum twice, once in an earlier segment
            x[r, V - 1] = x[r, min(edge, V - 2)] = 50.0
        elif kind == 2:
            x[r, edge - 1] = x[r, edge] = 50.0     # on both sides of an edge (or beside it)
        elif kind == 3:
            x[r] = -torch.inf
        elif kind == 4:
            x[r, V // 3] = x[r, V - 2] = torch.nan
            x[r, 1] = torch.inf
        elif kind == 5:
            x[r] = -x[r].abs() - 1
            x[r, V // 2], x[r, V - 1] = -0.0, 0.0
    cu = [min(i * 100, rows) for i in range((rows + 99) // 100 + 1)]
    parent = torch.cat([torch.tensor([-1] + [0] * (b - a - 1)) for a, b in zip(cu, cu[1:])]).to(torch.int32).to(gpu)
    token = torch.zeros(rows, dtype=torch.int64, device=gpu)
    want = torch.stack([row.float().cpu().argmax() for row in x]).to(torch.int32)
    token[:] = -1
    child = [a + 1 for a, b in zip(cu, cu[1:]) if b > a + 1]
    for c in child:                                # the first child of every root is accepted
        token[c] = int(want[c - 1])
    path, plen, bonus, am = greedy_accept(x, torch.tensor(cu, dtype=torch.int32, device=gpu), parent, token, check=True)
    assert torch.equal(am.cpu(), want)
    for b, (lo, hi) in enumerate(zip(cu, cu[1:])):
        one = hi > lo + 1
        assert int(plen[b]) == int(one) and int(bonus[b]) == int(want[lo + 1] if one else want[lo])
        assert path[b, :2].tolist() == ([0, -1] if one else [-1, -1])
