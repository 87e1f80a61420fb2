"""The step of several streams with a row in registers: row lengths at the edges of a block's width and of the longest row its threads
hold, rows picked and all, one branch and two, both norms; against the same in 64 bits, and bit for bit against the kernel that takes
the rows it does not."""
import pytest
import torch

from ullm_amd.kernels import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [2, 3, 4, 5])
@pytest.mark.parametrize("H", [4, 252, 1024, 1028, 2048])
@pytest.mark.parametrize("kind", ["rms", "layer"])
@pytest.mark.parametrize("two,picked", [(False, False), (True, False), (True, True)])
def test_step_of_many_tokens(S, H, kind, two, picked):
    g = torch.Generator().manual_seed(S * H)
    T = 300
    x = torch.randn(S, T, H, generator=g)
    ya, yb = torch.randn(T, H, generator=g).bfloat16(), torch.randn(T, H, generator=g).bfloat16()
    mix, out_w, in_w, gain = torch.randn(S, S, generator=g), torch.randn(S, generator=g), torch.randn(S, generator=g), torch.randn(H, generator=g)
    rows = torch.randperm(T, generator=g)[:260].int() if picked else None
    dev = {n: t.cuda() for n, t in dict(x=x.clone(), ya=ya, yb=yb, mix=mix, out_w=out_w, in_w=in_w, gain=gain).items()}
    got = ops.streams_step(dev["x"], dev["ya"], dev["mix"], dev["out_w"], 0.5, dev["in_w"], dev["gain"], 1e-5,
                           ops.NORM_RMS if kind == "rms" else ops.NORM_LAYER, torch.float32, None if rows is None else rows.cuda(),
                           dev["yb"] if two else None, 0.5, 0.75)
    y = 0.5 * ya.double() + (0.75 * yb.double() if two else 0)
    new = torch.einsum("sto,sd->dto", x.double(), mix.double()) + out_w.double()[:, None, None] * (0.5 * y)
    u = torch.einsum("sto,s->to", new, in_w.double())
    d = u - u.mean(-1, keepdim=True) if kind == "layer" else u
    expect = d * torch.rsqrt(d.square().mean(-1, keepdim=True) + 1e-5) * gain.double()
    if rows is not None:
        expect = expect[rows.long()]
    # a value of u is a sum of at most S (S + 2) rounded products, each off by 2^-24 of it at most, and the norm divides by its spread
    terms = torch.einsum("sto,sd->dto", x.double().abs(), mix.double().abs()) + (out_w.double().abs()[:, None, None] * (0.5 * y).abs())
    size = torch.einsum("sto,s->to", terms, in_w.double().abs()).amax(-1)
    spread = (d.square().mean(-1) + 1e-5).sqrt()
    bound = (S * (S + 2) + 16) * 2.0 ** -24 * size / spread * float(gain.abs().max()) * 4
    bound = bound + 1e-6 * expect.abs().amax() if rows is None else bound[rows.long()] + 1e-6 * expect.abs().amax()
    assert ((got.cpu().double() - expect).abs().amax(-1) <= bound).all()
    if not picked:
        assert ((dev["x"].cpu().double() - new).abs() <= (S + 8) * 2.0 ** -24 * terms).all()
    else:
        assert torch.equal(dev["x"].cpu(), x)            # picked rows: nothing is written back


@pytest.mark.parametrize("S,H", [(2, 4), (2, 252), (2, 1028), (2, 2048), (3, 1024), (3, 2052), (4, 1020), (4, 2048), (2, 16384), (4, 16384),
                                 (2, 16388)])
@pytest.mark.parametrize("kind", ["rms", "layer"])
@pytest.mark.parametrize("two,picked", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("y_type,out_type", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32), (torch.bfloat16, torch.float32)])
def test_bits_of_the_kernel_without_the_row(S, H, kind, two, picked, y_type, out_type):
    """Gains at an address that is no multiple of 16 are all that keeps the row out of registers: threads and pieces stay the same."""
    g = torch.Generator(device="cuda").manual_seed(S * H)
    T = 300
    normal = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    x, ya, yb = normal(S, T, H), normal(T, H).to(y_type), normal(T, H).to(y_type)
    mix, out_w, in_w, gain = normal(S, S), normal(S), normal(S), normal(H)
    aside = torch.empty(H + 1, device="cuda")[1:].copy_(gain)
    assert gain.data_ptr() % 16 == 0 and aside.data_ptr() % 16 == 4
    rows = torch.arange(T, device="cuda").flip(0)[:260].int() if picked else None
    got = []
    for weight in (gain, aside):
        streams = x.clone()
        normed = ops.streams_step(streams, ya, mix, out_w, 0.5, in_w, weight, 1e-5, ops.NORM_RMS if kind == "rms" else ops.NORM_LAYER,
                                  out_type, rows, yb if two else None, 0.5, 0.75)
        got.append((streams, normed))
    assert torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][0], got[1][0])
