"""Which hybrid-attention calls decode their window once (kernels.decode_first)."""

import pytest

from apple_amd.kernels import decode_first
from apple_amd.storage import RFSNConfig


def test_decode_first_lines():
    assert not decode_first(1, 32, 32, 128, 24576, True)        # decode steps keep the score tables
    assert not decode_first(3, 32, 32, 128, 100_000, False)     # and the in-register kernel
    assert decode_first(128, 32, 32, 128, 4096, False)
    assert decode_first(8, 32, 32, 128, 4096, True) and not decode_first(8, 32, 32, 128, 20_000, True)
    assert not decode_first(64, 8, 8, 64, 64, False)            # launch-bound either way
    # query heads that share KV heads share their decode: 44 us in registers, 61 decoded first (32 / 32 heads: 80, 61)
    assert not decode_first(8, 32, 8, 128, 1000, False) and decode_first(8, 32, 32, 128, 1000, False)
    assert not decode_first(32, 32, 8, 128, 256, False) and not decode_first(4, 32, 8, 64, 4096, False)
    # four queries' tables over 8,192 tokens: 69 us, 99 decoded first; eight queries': 107 and 100
    assert not decode_first(4, 32, 32, 128, 8192, True) and decode_first(8, 32, 32, 128, 8192, True)
    assert not decode_first(4, 8, 8, 128, 4096, True) and decode_first(16, 8, 8, 128, 4096, True)
    assert not decode_first(128, 32, 32, 256, 4096, False)      # no matrix-core kernel of that head_dim
    assert not decode_first(128, 24, 8, 128, 4096, False)       # nor of three query heads per KV head
    assert not decode_first(128, 32, 32, 128, 70_000, False)    # a decoded window over 1 GiB
    assert not decode_first(128, 32, 32, 128, 4096, False, (1 << 26) - 1)  # or over the caller's limit: 64 MiB
    assert decode_first(128, 32, 32, 128, 4096, False, 1 << 26)
    assert not decode_first(128, 32, 32, 128, 4096, False, 0)
    with pytest.raises(ValueError):
        RFSNConfig(hybrid_window_bytes=-1)
