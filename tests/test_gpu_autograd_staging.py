"""The torch gradient's host path: staged in pieces or whole, with arrays kept or
freed between calls, for float32, float64 and strided tensors, sizes changing
from call to call, it gives what the C ABI gives on uploaded arrays."""
import ctypes as C

import numpy as np
import pytest
import torch

from masterthesis_amd import autograd, capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stage", [8, 1000, 1 << 20])
@pytest.mark.parametrize("keep", [0, 1 << 20])
@pytest.mark.parametrize("dtype", ["f32_kahan", "f64"])
def test_kappa_host_path(hip, monkeypatch, stage, keep, dtype):
    if stage == 8 and keep == 0:
        pytest.skip("the smallest pieces once")
    monkeypatch.setattr(autograd, "_STAGE", stage)
    monkeypatch.setattr(autograd, "_KEEP", keep)
    n, steps = (9, 8, 7), 5
    shape = tuple(m + 2 for m in reversed(n))
    tau = 0.9 / sum(2 * 1.5 * (m - 1.0) ** 2 for m in n)
    npt = np.float64 if dtype == "f64" else np.float32
    mode = capi.HEATVAR_F64 if dtype == "f64" else capi.HEATVAR_F32_KAHAN
    with capi.Context(0) as ctx:
        fn = autograd.KappaMisfit(ctx, n, tau, steps, snapshots=3, dtype=dtype)
        for seed, kind in enumerate((torch.float64, torch.float32, torch.float64)):
            g = torch.Generator().manual_seed(seed)
            u0, kap, tgt = (torch.rand(shape, generator=g, dtype=torch.float64).to(kind) for _ in range(3))
            if seed == 2:  # the same values through other strides
                u0, kap, tgt = (v.permute(2, 1, 0).contiguous().permute(2, 1, 0) for v in (u0, kap, tgt))
            kap = (1.0 + 0.4 * kap).requires_grad_(True)
            J = fn(kap, u0, tgt)
            grad, = torch.autograd.grad(J, kap)
            bufs = [ctx.upload(v.detach().numpy().astype(npt)) for v in (u0, kap, tgt)]
            out, want = ctx.alloc(u0.numel()), C.c_double(0)
            gm = capi.geom(n)
            capi.check(ctx.L.scafes_heat7var_gradient(ctx.h, C.byref(gm), 1, mode, bufs[0].ptr, bufs[1].ptr,
                                                      bufs[2].ptr, tau, capi.BORDER_KEEP, 0.0, steps, 3, out.ptr,
                                                      C.byref(want), None))
            assert J.item() == want.value
            assert torch.equal(grad, torch.from_numpy(out.read(shape)).to(kind))
            assert bool(fn.fields.arrays) == (keep > 0)
            for b in bufs + [out]:
                b.free()
        del fn
