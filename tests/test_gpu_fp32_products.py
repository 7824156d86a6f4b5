"""fp32 layers in full precision whose results are one product each: rounded once, as by fp32 arithmetic, on every route, also where
a factor is far below the ordinary range (down to subnormal numbers) and the other as far above it."""
import pytest
import torch

from tests.test_gpu_fp32_special import CASES, Layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("small", ["none", "rows", "weights", "gradients"])
@pytest.mark.parametrize("n,shape,cloud", CASES)
def test_single_products(n, shape, cloud, small):
    layer = Layer(n, shape, cloud)
    x, w, g = layer.values
    k = int(torch.bincount(layer.offset[layer.offset != 13], minlength=27).argmax())
    pair = layer.offset == k
    row = int(layer.om[pair][n // 50])

    if small != "none":
        down, up = 2.0 ** -125, 2.0 ** 58
        tiny = torch.tensor([0, n // 3, row, int(layer.im[pair][n // 50]), layer.n - 1], device="cuda")
        x, w, g = (t * up for t in (x, w, g))
        for t, name in ((x, "rows"), (g, "gradients")):
            if small == name:
                t[tiny] = t[tiny] / up * down
        if small == "weights":
            w[k, 5:] = w[k, 5:] / up * down

    # one weight to a column and to a row, at one offset; one row of output gradients
    c = min(shape)
    at = torch.arange(c, device="cuda"), (7 * torch.arange(c, device="cuda") + 5) % c
    one_w, one_g = torch.zeros_like(w), torch.zeros_like(g)
    one_w[k][at] = w[k][at]
    one_g[row] = g[row]
    results = {what: (got, i) for what, got, i in layer.run(x, one_w, g)}
    results.update({what: (got, i) for what, got, i in layer.run(x, w, one_g) if i == 2})
    want = layer.exact(x, one_w, g)[:2] + layer.exact(x, w, one_g)[2:]
    for what, (got, i) in results.items():
        assert (want[i] != 0).any(), what
        # The result is rounded once; seven partial products of three parts each are less than 2^-6 of it, and each rounds their sum.
        bound = (1 + 7 * 2.0 ** -6) * 2.0 ** -24 * want[i].abs() + 2.0 ** -149
        assert ((got.double() - want[i]).abs() <= bound).all(), (what, ((got.double() - want[i]).abs() / bound).max())
