"""The one-launch warm encode picks its waves per block from the vector count: the codes of a vector do not
depend on it.  The sizes take each choice, with planted near-ties in every part (whole-codebook searches)."""

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,Mr,k", [(8, 8, 4), (16, 16, 4), (16, 0, 4), (8, 8, 0)])
def test_codes_do_not_depend_on_the_split(device, M, Mr, k):
    import torch
    from apple_amd import kernels as K

    g = torch.Generator().manual_seed(M + Mr)
    n, C = 70_001, 256
    x = (torch.randn(n, 64, generator=g) * 1.3).half()
    pq = (torch.randn(M, C, 64 // M, generator=g) * 1.3).half()
    rvq = (torch.randn(Mr, C, 64 // Mr, generator=g) * 0.5).half() if Mr else None
    pq[:, 9] = pq[:, 5] = pq[:, 2]                                  # a triple: three exact ties
    x[::997] = torch.cat([pq[m, 2] for m in range(M)])
    x, pq, rvq = x.to(device), pq.to(device), None if rvq is None else rvq.to(device)
    fmt = K.WarmFormat(64, M, C, Mr, C if Mr else 0, k)
    whole = K.warm_encode(x, fmt, pq, rvq)                          # rounds of 8-wave blocks
    assert bool((whole["pq"][::997] == 2).all())                    # the lowest index of the triple
    for size in (60_000, 30_000, 16_384, 1_001, 1):                 # 16, 8 and 4 waves, a partial block, one vector
        for a in (0, n - size):
            part = K.warm_encode(x[a:a + size], fmt, pq, rvq)
            for name, t in part.items():
                assert torch.equal(t.view(torch.uint8), whole[name][a:a + size].contiguous().view(torch.uint8)), (name, size)
    parts = K.warm_encode_batch([(x[:20_000], pq, rvq), (x[20_000:20_000], pq, rvq), (x[20_000:], pq, rvq)], fmt)
    for name, t in whole.items():
        assert torch.equal(torch.cat([p[name] for p in parts]).view(torch.uint8), t.view(torch.uint8))
