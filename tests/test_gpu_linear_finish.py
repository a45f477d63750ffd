"""rans_linear_finish, the last pass of RansLinear: bitwise the three torch
operations (to f32, add the bias, to the output type) it stands for, and out
of the way where something watches the tensors."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,extra", [(1, 1, 0), (3, 7, 0), (9, 8, 8), (5, 2048, 0),
                                             (17, 2050, 6), (512, 264, 24), (40000, 16, 0)])
@pytest.mark.parametrize("bias", [False, True])
def test_finish_matches_torch(rans, lib, rows, cols, extra, bias):
    import rans_linear as L
    print(f"case finish {rows}x{cols} of {cols + extra}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows * 7 + cols)
    wide = torch.randn(rows, cols + extra, device="cuda", generator=g)
    wide[0, 0], wide[-1, cols - 1] = float("inf"), -1e30
    b = torch.randn(cols, device="cuda", generator=g) if bias else None
    for first in {0, extra // 2, extra}:
        for dt in (torch.float32, torch.bfloat16):
            y = wide.to(dt)[:, first:first + cols]
            for out in (torch.float32, torch.bfloat16, torch.float16):
                want = y.float() if b is None else y.float() + b
                assert torch.equal(L._finish(lib, y, b, out), want.to(out)), (first, dt, out)


def test_prefill_still_differentiates_and_maps(rans, lib):
    """The prefill path is torch's own product: gradients with respect to x,
    forward-mode tangents and vmap go through it, with and without bias."""
    import rans_linear as L
    from torch.autograd import forward_ad
    g = torch.Generator().manual_seed(2)
    codes, step = L.quantize_uniform(torch.randn(64, 128, generator=g), 4.0)
    for bias in (None, torch.randn(64, generator=g)):
        lin = L.RansLinear.from_codes(codes, step, bias, lib, tune=False)
        w = lin.matrix.decode().float()
        x = torch.randn(32, 128, generator=g).cuda().requires_grad_()
        lin(x).sum().backward()
        assert torch.allclose(x.grad, w.sum(0).expand(32, -1), rtol=1e-2, atol=1e-2)
        t = torch.randn(32, 128, generator=g).cuda()
        with forward_ad.dual_level():
            y = lin(forward_ad.make_dual(x.detach(), t))
            tangent = forward_ad.unpack_dual(y).tangent
        assert torch.allclose(tangent, t @ w.t(), rtol=2e-2, atol=0.3)
        xs = torch.randn(3, 32, 128, generator=g).cuda()
        got = torch.func.vmap(lin)(xs)
        assert torch.allclose(got, torch.stack([lin(v) for v in xs]), rtol=2e-2, atol=0.1)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bias", [False, True])
def test_autocast(rans, lib, dtype, bias):
    """Under autocast the dense product comes in autocast's type, f16 by
    default; alone and in a group, with more rows than the GEMV takes and than
    the fused product does.  Bitwise the torch operations on that product."""
    import rans_linear as L
    print(f"case autocast {dtype} bias {bias}", flush=True)
    g = torch.Generator().manual_seed(11)
    tiling = rans.pick_group_tiling([256, 128], 512)
    mods = []
    for rows in (256, 128):
        codes, step = L.quantize_uniform(torch.randn(rows, 512, generator=g) * 0.05, 3.5)
        b = torch.randn(rows, generator=g) if bias else None
        mods.append(L.RansLinear.from_codes(codes, step, b, lib, tiling=(*tiling, 1), tune=False))
    assert all(m.matrix.fused_rows_limit < 20 <= m.matrix.matmul_rows < 100 for m in mods)
    ws = [m.matrix.decode() for m in mods]
    for grouped in (False, True):
        group = L.LinearGroup(mods) if grouped else None
        for m in mods:
            m.group = group
        for rows in (20, 100):
            for xt in (torch.float32, torch.bfloat16, torch.float16):
                x = torch.randn(rows, 512, generator=g).cuda().to(xt)
                with torch.no_grad(), torch.autocast("cuda", dtype=dtype):
                    got = [m(x) for m in mods]
                    if grouped:
                        y = torch.nn.functional.linear(x.bfloat16(), torch.cat(ws))
                        ys = y.split([256, 128], dim=1)
                    else:
                        ys = [torch.nn.functional.linear(x.bfloat16(), w) for w in ws]
                for m, y, out in zip(mods, ys, got):
                    assert y.dtype is dtype and out.dtype is xt
                    want = y.float() if m.bias is None else y.float() + m.bias
                    assert torch.equal(out, want.to(xt)), (grouped, rows, xt)
