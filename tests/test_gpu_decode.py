"""The bf16 and code decode at the sizes where their launches differ: fewer
and more tiles than one round of waves, one and two workgroups a CU, tile
heights odd and even, below and above the size from which rows are stored in
pairs, a partial last block of column steps, and an output that is only 2-byte
aligned."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,R,C,S", [
    (2050, 256, 1, 64, 1),      # 8200 tiles: two workgroups a CU, single rows
    (9001, 256, 1, 64, 1),      # 36004: five rounds of them, the last one partial
    (4100, 2048, 2, 256, 1),    # 16400 tiles
    (4098, 2112, 3, 192, 1),    # odd tile height, three column steps per tile
    (8960, 960, 35, 192, 1),    # one round, odd tile height
    (4112, 2048, 16, 512, 2),   # two states per lane
    (2048, 4224, 8, 1408, 1),   # 22 column steps: five blocks and a partial one
    (4096, 2048, 4, 512, 4),    # four states per lane
    (32775, 2112, 3, 704, 1),   # 69M weights, odd tile height
    (24, 160, 8, 192, 1),       # one wave, appended columns
])
def test_decode_launches(rans, lib, rows, cols, R, C, S):
    print(f"case decode {rows}x{cols} R={R} C={C} S={S}", flush=True)
    rng = np.random.default_rng(rows + cols)
    few = min(rows, 3 * R + 1)  # rows of codes, repeated over the height
    codes = np.rint(rng.laplace(size=(few, cols)) * 2).astype(np.int32)
    hit = rng.random(codes.shape) < 0.003
    codes[hit] = rng.integers(-900, 900, int(hit.sum()))
    codes = np.resize(codes, (rows, cols))
    step = (rng.random(cols) + 0.25).astype(np.float32)
    m = rans.RansMatrix(rans.encode(codes, R, C, S), torch.from_numpy(step), lib)
    want = (torch.from_numpy(codes).float() * torch.from_numpy(step)).bfloat16().cuda()
    n = rows * cols
    for shift in (0, 1, 2, 3):  # of the output, in elements
        buf = torch.full((n + 8,), 7.0, device="cuda", dtype=torch.bfloat16)
        out = m.decode(buf[shift:shift + n].view(rows, cols))
        assert torch.equal(out, want), shift
        rest = torch.cat([buf[:shift], buf[shift + n:]])
        assert bool((rest == 7.0).all()), "stored outside the output"
    np.testing.assert_array_equal(m.decode_codes().cpu().numpy(), codes)


@pytest.mark.parametrize("rows,cols,R,C,S,scale", [
    (27650, 4096, 2, 2048, 1, 2), (53700, 2112, 3, 704, 1, 2), (13828, 8192, 4, 1024, 2, 2),
    (18440, 6144, 8, 1536, 4, 2), (27664, 4096, 16, 512, 2, 2), (22120, 5120, 20, 640, 1, 2),
    (49175, 2304, 35, 576, 1, 2),      # odd tile height
    (22128, 5120, 16, 2560, 2, 0.45),  # 2766 tiles: one round, no wave takes a second
    (1769500, 64, 1, 64, 1, 2)])       # single rows: nothing to pair
def test_paired_rows(rans, lib, rows, cols, R, C, S, scale):
    """Outputs of 108M weights and more, whose rows are stored in pairs, over
    tile heights, states per lane and both launches: every value, escapes in
    either row of a pair, in both, and in the row that an odd height leaves
    over; at a 4-byte boundary and 2 bytes past one, where rows go out singly."""
    print(f"case paired decode {rows}x{cols} R={R} C={C} S={S}", flush=True)
    assert rows * cols >= 108 << 20
    rng = np.random.default_rng(rows + cols)
    few = 2 * R  # rows of codes, repeated over the height
    codes = np.rint(rng.laplace(size=(few, cols)) * scale).astype(np.int32)
    hit = rng.random(codes.shape) < 0.003
    codes[hit] = rng.integers(128, 900, int(hit.sum()))
    codes[0, ::31] = -300                # the first row of a pair,
    codes[min(1, few - 1), ::17] = 301   # the second, and both
    codes[R - 1, -3:] = 302              # the last row of a tile, the last columns
    codes = np.resize(codes, (rows, cols))
    step = (rng.random(cols) + 0.25).astype(np.float32)
    m = rans.RansMatrix(rans.encode(codes, R, C, S), torch.from_numpy(step), lib)
    dev = torch.from_numpy(codes).cuda()
    want = (dev.float() * torch.from_numpy(step).cuda()).bfloat16()
    n = rows * cols
    for shift in (0, 1):  # of the output, in elements
        buf = torch.full((n + 8,), 7.0, device="cuda", dtype=torch.bfloat16)
        assert torch.equal(m.decode(buf[shift:shift + n].view(rows, cols)), want), shift
        rest = torch.cat([buf[:shift], buf[shift + n:]])
        assert bool((rest == 7.0).all()), "stored outside the output"
    assert torch.equal(m.decode_codes(), dev)
