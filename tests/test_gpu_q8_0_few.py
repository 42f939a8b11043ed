"""GPU parity of the order-S products of few activation rows (q8_0_s.hip) with the C oracle
at the edges of their tiles: rows and tokens that end inside a tile, K that ends inside a
chunk, one chunk only, operands at any address.  Bar: bit-exact."""
import pytest

from bpd_substrate_amd import gpu, synth
from helpers import assert_bits_equal, to_np
from oracle import oracle as O
from test_gpu_q8_0 import _d, _q8_full_range, _q8_nan_heavy

pytestmark = pytest.mark.gpu

CASES = [(70, 1, 256, 0, 0),        # the kernel for any number of tokens still
         (70, 1, 480, 0, 0),        # 4 tokens per workgroup, a chunk that ends early
         (130, 3, 512, 0, 1),       # ... one whole chunk, X at an odd address
         (4099, 18, 768, 0, 2),     # 8 tokens, a ragged last tile of rows and of tokens
         (4100, 50, 1280, 0, 0),    # ... with several workgroups per CU
         (8201, 9, 256, 0, 0),      # 16 tokens x 64 rows, half a chunk, a ragged last tile of rows and of tokens
         (4100, 64, 1440, 2, 1),    # 16 tokens x 128 rows, 45 blocks, W off the 4-byte grid, X at an odd address
         (14340, 17, 1024, 0, 2),   # 16 tokens x 128 rows
         (66, 5, 14336, 0, 0),      # a long K: more than 64 KiB of LDS
         (130, 9, 28672, 0, 0),     # ... that only 4 tokens fit
         (18, 2, 32, 0, 0),         # one block
         (70, 5, 1440, 2, 0),       # 45 blocks: a last chunk of 13, W off the 4-byte grid
         (700, 3, 544, 1, 3)]       # 17 blocks: a last chunk of one, both at odd addresses


@pytest.mark.parametrize("mw,mt,K,wo,xo", CASES)
@pytest.mark.parametrize("kind", ["plain", "nan", "int8"])
def test_tokens_scalar_order(dev, mw, mt, K, wo, xo, kind):
    import torch

    nb = K // 32
    make = {"plain": lambda r, k: synth.q8_0(r, K, k), "nan": lambda r, k: _q8_nan_heavy(r, nb, k),
            "int8": lambda r, k: _q8_full_range(r, nb, k)}[kind]
    W, X = make(mw, synth.key(73, mw)), make(mt, synth.key(74, mt))
    wb, xb = (torch.zeros(a.size + 16, dtype=torch.uint8, device=dev) for a in (W, X))
    wb[wo:wo + W.size] = _d(W, dev)
    xb[xo:xo + X.size] = _d(X, dev)
    got = to_np(gpu.qmatmul_q8_0_dispatch_s(wb[wo:wo + W.size], xb[xo:xo + X.size], mw, mt, K))
    assert_bits_equal(got, O.dispatch_q8_0(W, X, mw, mt, K, "S", nthreads=8), f"{kind} {mw}x{mt}x{K} +{wo} +{xo}")
