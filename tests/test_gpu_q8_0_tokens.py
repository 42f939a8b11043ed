"""GPU parity of the order-T products of several activation rows (q8_0_t.hip) with the C
oracle at the edges of their tiles: rows and tokens that end inside a tile, K that ends
inside a chunk, operands that miss the alignment of the wide loads.  Bar: bit-exact."""
import numpy as np
import pytest

from bpd_substrate_amd import gpu, synth
from helpers import assert_bits_equal, to_np
from oracle import oracle as O
from test_gpu_q8_0 import _d, _q8_full_range, _q8_nan_heavy

pytestmark = pytest.mark.gpu

CASES = [(4099, 4, 256, 0),      # 4 tokens per wave, a half chunk
         (2050, 9, 768, 0),      # 4 tokens per wave, a whole and a half chunk, 3 token groups
         (4100, 13, 1280, 0),    # 8 tokens per wave
         (703, 65, 224, 0),      # 8 tokens per wave, an odd number of blocks
         (4100, 14, 544, 0),     # 8 tokens per wave, a last chunk of one block
         (8200, 2, 32, 2),       # the per-token GEMVs, W off the 4-byte grid
         (703, 65, 960, 1),      # 30 blocks, W at an odd address
         (1030, 290, 512, 0),    # 32 x 64 tiles
         (1030, 290, 192, 0),    # ... K % 256 != 0
         (1030, 290, 224, 0),    # ... an odd number of blocks
         (1030, 290, 256, 2),    # ... W off the 4-byte grid
         (1030, 290, 256, 1),    # ... W at an odd address
         (4100, 300, 128, 0),    # 64 x 64 tiles
         (4100, 300, 96, 0),
         (2000, 16, 480, 0),     # 4 tokens per wave, one chunk that ends early
         (1100, 20, 544, 1),     # ... a last chunk of one block, W at an odd address
         (33000, 3, 768, 0),     # ... several workgroups per CU, a ragged last one
         (703, 256, 32, 2)]      # 32 x 64 tiles, one block


@pytest.mark.parametrize("mw,mt,K,off", CASES)
@pytest.mark.parametrize("kind", ["plain", "nan", "int8"])
def test_tokens_tile_order(dev, mw, mt, K, off, kind):
    import torch

    nb = K // 32
    make = {"plain": lambda r, k: synth.q8_0(r, K, k), "nan": lambda r, k: _q8_nan_heavy(r, nb, k),
            "int8": lambda r, k: _q8_full_range(r, nb, k)}[kind]
    W, X = make(mw, synth.key(71, mw)), make(mt, synth.key(72, mt))
    buf = torch.zeros(W.size + 16, dtype=torch.uint8, device=dev)
    buf[off:off + W.size] = _d(W, dev)
    got = to_np(gpu.qmatmul_q8_0_dispatch(buf[off:off + W.size], _d(X, dev), mw, mt, K))
    assert_bits_equal(got, O.dispatch_q8_0(W, X, mw, mt, K, "T", nthreads=8), f"{kind} {mw}x{mt}x{K} +{off}")
