"""Residual codes against the canonical distances, where the screening by groups of four can go wrong.

The canonical distance is fl32(fl32(L - 2 X) + R) with L, X and R summed in float64 (quantization.py:206-252);
the lower index wins a tie.  Codes are whole numbers: they have to be the same.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

# rows: one and four sets a wave, partly filled blocks, both sides of the row limit of small codebooks
ROWS = [1, 65, 4097, 40001, 65536, 65537, 70003]


def _codes(rows, books):
    """First least canonical distance of each stage."""
    run, out = rows.float(), []
    index = torch.arange(books.shape[1], device=rows.device)
    for cb in books:
        c = cb.double()
        R = (c * c).sum(1).float()
        stage = []
        for part in run.split(8192):
            x = part.double()
            d = (x * x).sum(1).float()[:, None] - 2 * (x @ c.T).float() + R
            low = d.min(1, keepdim=True).values
            stage.append(torch.where(d == low, index, books.shape[1]).min(1).values)
        stage = torch.cat(stage)
        run = run - cb.float()[stage]
        out.append(stage)
    return torch.stack(out, 1)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("C", [3, 61, 512, 513, 1030])
def test_codes_are_the_first_least(D, C):
    from apple_amd import kernels as K

    g = torch.Generator(device="cuda").manual_seed(D + C)
    books = (torch.randn(2, C, D, generator=g, device="cuda") * (2 / D) ** 0.5).half()
    if C > 61:
        books[0, 40:60] = books[0, 7]   # more equal centroids than the rescoring takes
        books[1, C - 1] = books[1, 1]   # the last row ties an early one
        books[1, C - 2] = books[1, C - 3]
    for n in ROWS:
        x = (torch.randn(n, D, generator=g, device="cuda") * 0.6).half()
        if C > 61 and n > 60:
            x[::7] = books[0, 7]        # rows at the equal centroids
            x[3::11] = 0.5 * (books[0, 1] + books[0, 2])  # rows nearly between two
        codes = K.rvq_encode_full(x, books, 0.0)[0]
        want = _codes(x, books)
        assert torch.equal(codes.long().reshape(want.shape), want), (D, C, n)
