"""The gated unit norm over parts of up to 256 values, four a lane: parts that fill their lanes and parts that do not, the last
block's idle lanes, added slices and divisors, a gain a part long and a row long, against 64-bit results; and the other kernel's
cases beside them (sizes that are no multiple of four, longer parts, rows that are not aligned)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("size,parts", [(4, 3), (8, 1), (12, 7), (64, 32), (100, 3), (128, 16), (252, 1), (256, 5), (257, 2), (260, 3), (30, 4)])
@pytest.mark.parametrize("T", [1, 5, 67])
@pytest.mark.parametrize("slices,offset", [(1, 0), (3, 4), (1, 1)])
def test_parts_against_64_bit(size, parts, T, slices, offset):
    from ullm_amd.kernels import ops
    g = torch.Generator().manual_seed(size * parts + T)
    width = size * parts
    o = torch.randn(slices, T, width, generator=g)
    wide = torch.randn(T, width + 8 + offset % 4, generator=g)
    for gain_len in {size, width}:
        gain = torch.randn(gain_len, generator=g)
        for kind in (ops.GATE_SILU, ops.GATE_SIGMOID):
            for divided in (False, True):
                den = torch.randn(T, parts, generator=g) if divided else None
                least = torch.rand(T, parts, generator=g) if divided else None
                z = wide[:, offset:offset + width]
                v = torch.stack([o.double().sum(0), o.double().abs().sum(0)]).view(2, T, parts, size)       # and what its roundings scale with
                if divided:
                    v = v / (torch.maximum(den.double().abs(), least.double()) + 1e-6)[..., None]
                v = v * torch.rsqrt(v[0].pow(2).mean(-1, keepdim=True) + 1e-5)
                s = torch.sigmoid(z.double())
                want, scale = v.reshape(2, T, width) * gain.double().repeat(width // gain_len) * (s if kind == ops.GATE_SIGMOID else z.double() * s)
                dev = wide.to(DEV)
                got = ops.gated_unit_norm((o if slices > 1 else o[0]).to(DEV), dev[:, offset:offset + width], gain.to(DEV), 1e-5, parts, kind,
                                          torch.float32, den=None if den is None else den.to(DEV), least=None if least is None else least.to(DEV))
                assert ((got.double().cpu() - want).abs() <= 2.0 ** -20 * scale.abs()).all()                # some ten roundings a value
                half = ops.gated_unit_norm((o if slices > 1 else o[0]).to(DEV), dev[:, offset:offset + width], gain.to(DEV), 1e-5, parts, kind,
                                           torch.bfloat16, den=None if den is None else den.to(DEV), least=None if least is None else least.to(DEV))
                assert torch.equal(half, got.bfloat16())
