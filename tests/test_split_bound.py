"""The error bound of the fp32 split mode (torch's 'high' float32 matmul precision), which the
GPU parity band uses: with hi = bf16(x) and lo = bf16(x - hi) (round to nearest even, as
v_cvt_pk_bf16_f32 and torch's bfloat16 cast do), x - hi is exact in fp32,
|x - hi - lo| <= 2^-16 |x|, and a product taken as hi_a hi_b + hi_a lo_b + lo_a hi_b is within
3 * 2^-16 |a b| of the exact one. Checked in float64 on random values over a wide exponent
range, with a planted mistake (the hi_a lo_b term dropped) that the bound must reject. And the
split of larger fp32 batches, three bf16 parts and six products: exact, and within 2^-22.9."""
import torch

from _parity import SPLIT_REL


def split(x):
    hi = x.to(torch.bfloat16).to(torch.float32)
    r = x - hi  # exact in fp32
    lo = r.to(torch.bfloat16).to(torch.float32)
    return hi, lo, r


def sample(n, seed):
    g = torch.Generator().manual_seed(seed)
    mant = torch.rand(n, generator=g, dtype=torch.float64) + 1.0
    expo = torch.randint(-60, 60, (n,), generator=g).to(torch.float64)
    sign = torch.where(torch.rand(n, generator=g) < 0.5, -1.0, 1.0).to(torch.float64)
    return (sign * mant * torch.pow(2.0, expo)).to(torch.float32)


def test_remainder_is_exact_and_within_2_pow_minus_16():
    x = sample(200000, 1)
    hi, lo, r = split(x)
    xd, hid, lod = x.double(), hi.double(), lo.double()
    assert torch.equal(r.double(), xd - hid)  # x - hi needs no rounding
    assert bool(((xd - hid - lod).abs() <= 2.0 ** -16 * xd.abs()).all())
    assert bool(((xd - hid).abs() <= 2.0 ** -8 * xd.abs()).all())


def test_split_product_within_split_rel():
    a, b = sample(200000, 2), sample(200000, 3)
    ha, la, _ = split(a)
    hb, lb, _ = split(b)
    exact = a.double() * b.double()
    got = ha.double() * hb.double() + ha.double() * lb.double() + la.double() * hb.double()
    assert SPLIT_REL == 3 * 2.0 ** -16
    err = (got - exact).abs()
    assert bool((err <= SPLIT_REL * exact.abs()).all()), float((err / exact.abs()).max())
    # the bound is not loose by orders of magnitude: the worst case reaches a good part of it
    assert float((err / exact.abs()).max()) > 2.0 ** -17
    # a dropped cross term breaks it
    bad = ha.double() * hb.double() + la.double() * hb.double()
    assert not bool(((bad - exact).abs() <= SPLIT_REL * exact.abs()).all())


def parts(x):
    out = []
    for _ in range(3):
        p = x.to(torch.bfloat16).to(torch.float32)
        out.append(p)
        x = x - p
    return out


def test_three_parts_hold_every_bit():
    """Over the magnitudes that the kernel takes parts of, [2^-50, 2^48): the parts add up to the
    value, and each is 0 or a normal bf16. Two fp16 parts of scaled rows, 11 bits and a sign
    each, leave a quarter of the values one unit off."""
    g = torch.Generator().manual_seed(4)
    n = 400000
    x = (torch.rand(n, generator=g, dtype=torch.float64) + 1.0) * torch.pow(
        2.0, torch.randint(-50, 48, (n,), generator=g).double())
    x = torch.cat([x, -x, torch.tensor([2.0 ** -50, 2.0 ** 48 * (1 - 2.0 ** -24), 0.0, 1 + 2.0 ** -23])]).float()
    p = parts(x)
    assert torch.equal(sum(q.double() for q in p), x.double())
    for k, q in enumerate(p):
        assert bool(((q == 0) | (q.abs() >= 2.0 ** -126)).all())
        assert bool((q.abs().double() <= 2.0 ** (-8 * k) * (1 + 2.0 ** -8) * x.abs().double()).all())
    y = (x[:n].double() / torch.pow(2.0, x[:n].double().log2().floor()) * 2.0 ** 14).float()
    hi = y.half()
    lo = (y - hi.float()).half()
    assert 0.2 < float((hi.double() + lo.double() != y.double()).double().mean()) < 0.3


def test_six_products_of_parts():
    a, b = sample(200000, 5), sample(200000, 6)
    a, b = a.clamp(-2.0 ** 47, 2.0 ** 47), b.clamp(-2.0 ** 47, 2.0 ** 47)
    p, q = ([t.double() for t in parts(x)] for x in (a, b))
    pairs = [(2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)]
    got = sum(p[i] * q[j] for i, j in pairs)
    exact = a.double() * b.double()
    bound = 2.0 ** -22.9
    assert bool(((got - exact).abs() <= bound * exact.abs()).all())
    bad = sum(p[i] * q[j] for i, j in pairs if (i, j) != (1, 1))
    assert not bool(((bad - exact).abs() <= bound * exact.abs()).all())
