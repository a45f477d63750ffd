"""rans_w64_matmul, the product fused with the decode: exact sums (small whole
x, steps that are powers of two) against the decoded matrix in 64 bits, over
the tile heights, one and several tile rows to a wave, ragged ends of both, and
the calls that RansLinear keeps on the dense product."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _matrix(rans, lib, rows, cols, R, C, esc, seed):
    rng = np.random.default_rng(seed)
    codes = np.round(rng.laplace(0, 3.0, (rows, cols))).clip(-127, 127).astype(np.int32)
    if esc:
        at = rng.random((rows, cols)) < esc
        codes[at] = rng.integers(128, 600, at.sum())
        codes[0, :70] = -300  # more in 64 columns than a wave holds at once
        codes[-1, -1] = 599
    step = np.exp2(rng.integers(-7, -4, cols)).astype(np.float32)
    return rans.RansMatrix(rans.encode(codes, R, C, 1), torch.from_numpy(step), lib)


# the wide ones read 136 MB or more of x at 64 rows, an odd number of tile
# rows most of them
WIDE = [(513, 6528, 3, 1088), (516, 8704, 4, 1088), (1032, 8704, 8, 1088), (4368, 4096, 16, 512),
        (2064, 8704, 16, 1088)]  # of the last, two tile rows to a wave do not fit the LDS


@pytest.mark.parametrize("rows,cols,R,C", WIDE + [
    (3, 64, 3, 64), (12, 2048, 4, 128), (1000, 1568, 8, 320), (48, 1024, 16, 256),
    (60, 640, 20, 128), (70, 1536, 35, 192)])
@pytest.mark.parametrize("esc", [0.0, 0.02])
def test_exact_sums(rans, lib, rows, cols, R, C, esc):
    m = _matrix(rans, lib, rows, cols, R, C, esc, rows + cols)
    w = m.decode().double()
    g = torch.Generator(device="cuda").manual_seed(rows)
    bias = torch.randn(rows, device="cuda", generator=g)
    for nb in (1, 16, 17, 47, 64):
        print(f"case matmul {rows}x{cols} R={R} C={C} esc={esc} rows of x {nb}", flush=True)
        x = torch.randint(-4, 5, (nb, cols), device="cuda", generator=g).bfloat16()
        want = (x.double() @ w.t()).float()
        assert torch.equal(m.matmul(x), want), nb
        assert torch.equal(m.matmul(x.float(), bias, torch.bfloat16), (want + bias).bfloat16()), nb
        assert torch.equal(m.matmul(x, bias, torch.float16), (want + bias).half()), nb


# many short tiles: several tile rows to a wave from these rows of x on,
# an odd number of tile rows, which 2 and 4 leave over
@pytest.mark.parametrize("rows,cols,R,C,tiles", [
    (2895, 256, 3, 64, 4), (3876, 320, 4, 64, 4), (8968, 192, 8, 64, 2), (5672, 768, 8, 192, 2),
    (8976, 1024, 16, 256, 2)])
@pytest.mark.parametrize("esc", [0.0, 0.02])
def test_several_tile_rows(rans, lib, rows, cols, R, C, tiles, esc):
    m = _matrix(rans, lib, rows, cols, R, C, esc, rows + cols)
    w = m.decode().double()
    g = torch.Generator(device="cuda").manual_seed(rows)
    bias = torch.randn(rows, device="cuda", generator=g)
    taken = []
    for nb in (1, 17, 33, 48, 64):
        taken.append(lib.rans_matmul_tiles(ctypes.byref(m._desc), nb))
        print(f"case matmul {rows}x{cols} R={R} C={C} esc={esc} rows of x {nb} T={taken[-1]}",
              flush=True)
        x = torch.randint(-4, 5, (nb, cols), device="cuda", generator=g).bfloat16()
        want = (x.double() @ w.t()).float()
        assert torch.equal(m.matmul(x), want), nb
        assert torch.equal(m.matmul(x, bias, torch.bfloat16), (want + bias).bfloat16()), nb
    assert taken[0] == 1 and taken[-1] == tiles


def test_refuses(rans, lib):
    m = _matrix(rans, lib, 48, 1024, 16, 256, 0.0, 1)
    with pytest.raises(AssertionError):
        m.matmul(torch.zeros(65, 1024, device="cuda"))


def test_bias(rans, lib):
    """A bias in another type or stride counts as its f32 values; one of
    another length or on the host is refused before any launch."""
    m = _matrix(rans, lib, 48, 1024, 16, 256, 0.0, 1)
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randint(-4, 5, (20, 1024), device="cuda", generator=g).bfloat16()
    b = torch.randint(-8, 9, (48, 2), device="cuda", generator=g).float()
    want = m.matmul(x) + b[:, 0]
    for bias in (b[:, 0], b[:, 0].bfloat16(), b[:, 0].contiguous().half(), b[:, 0].double()):
        assert torch.equal(m.matmul(x, bias), want)
    for bias in (b[:47, 0], b[:1, 0], b[:, 0].cpu(), b[:, :1], torch.zeros(64, device="cuda")):
        with pytest.raises(ValueError):
            m.matmul(x, bias)


def test_linear_route(rans, lib):
    """Misaligned rows, f16 and f32 inputs and leading dimensions on the fused
    product; a watched x on the dense one, with its gradient."""
    import rans_linear as L
    g = torch.Generator().manual_seed(3)
    codes, step = L.quantize_uniform(torch.randn(256, 1024, generator=g), 3.5)
    lin = L.RansLinear.from_codes(codes, step, torch.randn(256, generator=g), lib, tune=False)
    w = lin.matrix.decode().double()
    assert lin.matrix.matmul_rows == 64
    for dt in (torch.bfloat16, torch.float32, torch.float16):
        flat = torch.randn(24 * 1024 + 1, generator=g).cuda().to(dt)
        for x in (flat[1:].view(24, 1024), flat[:-1].view(2, 12, 1024)):
            y = lin(x)
            assert y.dtype is dt and y.shape == (*x.shape[:-1], 256)
            want = x.bfloat16().double() @ w.t() + lin.bias.double()
            # f32 sums of 1024 exact products, then one rounding to dt
            u = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11, torch.float32: 0}[dt]
            tol = 1100 * 2 ** -24 * (x.bfloat16().double().abs() @ w.abs().t()) + u * want.abs() + 1e-6
            assert ((y.double() - want).abs() <= tol).all()
    x = torch.randn(24, 1024, generator=g).cuda().requires_grad_()
    lin(x).sum().backward()
    assert torch.allclose(x.grad.double(), w.sum(0).expand(24, -1), rtol=1e-2, atol=1e-2)
