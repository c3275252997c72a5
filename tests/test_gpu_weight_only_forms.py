"""Every tile form of the weight-only GEMM at the edges of its range: remainders of rows, channels and k-tiles, groups of
wavefronts that share k out and get no tile at all, and the first sizes past a form's last full round."""
import pytest
import torch

from tests.helpers import TORCH_DT

pytestmark = pytest.mark.gpu

# (m, n, k): 32x32 with eight and with four k-groups, 64x64, 128x128, 128x256 and 256x256 tiles
SIZES = [(1, 32, 64), (33, 96, 192), (3, 8192, 128), (33, 8192, 640), (65, 8192, 192), (129, 8192, 576), (385, 2080, 128),
         (300, 9248, 192), (700, 9248, 128), (1300, 9248, 192)]


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("kind,group,zeros", [("int8", 0, False), ("int4", 0, False), ("int8", 64, True), ("int4", 64, False), ("int4", 64, True)])
def test_forms_against_float64(dev, dt, kind, group, zeros):
    from lyradiff_amd import ops

    t = TORCH_DT[dt]
    for m, n, k in SIZES:
        g = torch.Generator(device=dev).manual_seed(m * n + k)
        rand = lambda *s: torch.rand(s, generator=g, device=dev)
        half = 128 if kind == "int8" else 8
        q = torch.randint(-half, half, (k, n), generator=g, device=dev, dtype=torch.int8)
        w = ops.repack_weight_only(q if kind == "int8" else ((q[:, 0::2] & 15) | (q[:, 1::2] << 4)).contiguous(), kind)
        x = (rand(m, k) * 2 - 1).to(t)
        bias = rand(n).to(t)
        if group:
            s = (0.002 + 0.02 * rand(k // group, n)).to(t)
            z = (rand(k // group, n) - 0.5).to(t) if zeros else None
            wide = lambda v: v.double().repeat_interleave(group, 0)
            dq = (q.double() * wide(s)).to(t).double()  # q * s is exact before that rounding
            if zeros:
                dq = (dq + wide(z)).to(t).double() if dt == "f16" else (q.double() * wide(s) + wide(z)).float().to(t).double()
            y = ops.weight_only_linear_grouped(x, w, s, z, bias, kind, group)
            ref = x.double() @ dq + bias.double()
            terms = x.double().abs() @ dq.abs()
        else:
            s = (0.002 + 0.02 * rand(n)).to(t)
            y = ops.weight_only_linear(x, w, s, bias, kind)
            ref = (x.double() @ q.double()) * s.double() + bias.double()
            terms = (x.double().abs() @ q.double().abs()) * s.double()
        # half an ulp of the result, fp32 sums of at most k terms, and where a weight falls on a rounding midpoint its last bit
        ulp = 2.0 ** -11 if dt == "f16" else 2.0 ** -8
        bound = 1.01 * ulp * ref.abs() + (k + 4) * 2.0 ** -24 * (terms + bias.double().abs()) + (2 * ulp * 2e-3 * terms if zeros else 0.0) + 1e-7
        err = (y.double() - ref).abs()
        assert bool((err <= bound).all()), (m, n, k, float((err / bound).max()))
