"""Which kernel the launchers choose, against the times measured for each form.

`launches` records what an entry point launches; the tables hold the microseconds per call of
every form on MI355X (graphs of back-to-back launches, weights beyond the MALL).  No GPU.
"""
import ctypes

import pytest
import torch

from bpd_substrate_amd import llama
from launches import Recorder

W, X, OUT = 0x100000, 0x200000, 0x300000  # never read: aligned as a torch tensor is


@pytest.fixture(scope="module")
def launched(tmp_path_factory):
    return Recorder(str(tmp_path_factory.mktemp("launches")))


def one_of(shapes, forms):
    """The time of the form that a launch belongs to (None: not measured at this shape)."""
    def f(launch):
        for form, t in zip(forms, shapes):
            if form(launch):
                return t
        raise AssertionError(f"{launch} is none of the forms")
    return f


# ---------------------------------------------------------------- Q8_0, order T, several rows of X

T_FORMS = [lambda l: l.kernel == "k_q8_0_gemm_TQ" and l.args[0] == 1,
           lambda l: l.kernel == "k_q8_0_gemm_TQ" and l.args[0] == 2,
           lambda l: l.kernel == "k_q8_0_gemm_TM" and l.args[0] == 2,
           lambda l: l.kernel == "k_q8_0_gemm_TM" and l.args[0] == 4,
           lambda l: l.kernel.startswith("k_q8_0_gemv_")]
# M, tokens, K, then us of TQ with 4 and 8 tokens, TM with 32 and 64 rows, the per-token GEMVs
T_US = [
    (2048, 16, 64, 4.3, 4.5, 4.1, 4.7, 6.1), (8192, 8, 32, 5.4, 4.8, 4.1, 5.2, 8.6),
    (8192, 8, 64, 5.0, 4.6, 4.1, 4.7, 8.8), (32000, 4, 64, 7.2, 8.5, 8.1, 8.2, 13.8),
    (32000, 2, 256, 8.3, 10.4, 14.3, 14.4, 13.4), (512, 200, 32, 7.5, 5.9, 4.5, 5.8, 11.8),
    (32000, 8, 512, 12.9, 11.8, 21.9, 21.3, 29.1),
    (1024, 16, 4096, 14.0, 17.7, None, None, 12.5), (1024, 16, 14336, 39.8, 51.7, None, None, 33.9),
    (2048, 8, 1024, 6.4, 7.4, None, None, 5.8), (2048, 8, 4096, 14.1, 17.7, None, None, 13.0),
    (2048, 8, 14336, 40.2, 52.1, None, None, 37.7), (2048, 33, 4096, None, 25.9, 44.8, 57.5, 38.6),
    (3000, 8, 1024, 6.7, 7.5, None, None, 8.3), (4096, 4, 1024, 6.4, 7.3, None, None, 5.9),
    (4096, 4, 4096, 14.5, 17.9, None, None, 14.1), (4096, 4, 14336, 40.6, 53.2, None, None, 40.4),
    (4096, 5, 4096, 14.6, 18.0, None, None, 16.2), (4096, 16, 4096, 19.5, 18.5, None, None, 39.8),
    (4096, 33, 4096, None, 44.4, 54.3, 60.9, 76.8), (4096, 65, 4096, None, 58.9, 47.6, 60.0, None),
    (5632, 3, 4096, 14.8, 18.2, None, None, 14.7), (5632, 3, 14336, 40.6, 53.3, None, None, 44.6),
    (5632, 12, 4096, 23.6, 26.2, None, None, 42.7), (8192, 2, 1024, 7.0, 7.8, None, None, 6.2),
    (8192, 2, 4096, 15.2, 18.7, None, None, 14.8), (8192, 2, 14336, 43.6, 57.0, None, None, 41.9),
    (8192, 3, 4096, 15.3, 19.0, None, None, 19.4), (8192, 8, 4096, 20.0, 19.7, None, None, 43.4),
    (8192, 33, 8032, None, 118.6, 97.7, 167.9, 399.2), (11008, 2, 1024, 9.0, 10.2, None, None, 7.2),
    (11008, 2, 4096, 20.6, 26.6, None, None, 18.7), (11008, 2, 14336, 60.7, 82.2, None, None, 54.8),
    (11008, 3, 4096, 20.8, 26.6, None, None, 25.5), (11008, 5, 4096, 25.8, 27.6, None, None, 39.3),
    (11008, 24, 14336, None, 266.0, 256.3, 215.4, 603.0), (14336, 2, 4096, 20.6, 26.9, None, None, 22.3),
    (14336, 4, 4096, 20.7, 27.0, None, None, 39.5), (14336, 8, 4096, 34.3, 30.2, None, None, 73.8),
    (14336, 9, 4096, 46.9, 53.5, None, None, 82.5), (14336, 16, 4096, 66.2, 55.6, None, None, 143.7),
    (14336, 33, 4096, None, 119.0, 86.3, 69.8, 285.6), (14336, 65, 4128, None, 189.2, 140.5, 171.9, None),
    (20000, 65, 1440, None, 109.5, 67.2, 88.6, None), (20000, 96, 1440, None, 146.5, 68.2, 89.5, None),
    (32000, 2, 1024, 14.6, 18.4, None, None, 16.1), (32000, 2, 4096, 37.2, 54.6, None, None, 44.0),
    (32000, 4, 14336, 119.4, 179.7, None, None, 290.9), (32000, 9, 4096, 84.6, 97.1, None, None, 183.6),
    (32000, 17, 4096, None, 169.0, 166.2, 140.9, 349.0), (32000, 64, 1440, None, 156.6, 59.0, 70.4, None),
    (65536, 2, 1440, 33.7, 45.5, None, None, 53.4), (65536, 4, 4096, 67.3, 104.5, None, None, 170.4),
    (65536, 5, 8032, 236.8, 195.8, None, None, 664.4), (128256, 2, 1024, 39.6, 61.2, None, None, 54.1),
    (128256, 2, 4096, 132.0, 224.2, None, None, 174.7), (128256, 4, 4096, 133.4, 211.0, None, None, 336.1),
    (128256, 5, 4096, 267.3, 200.9, None, None, 424.0), (128256, 17, 1440, None, 236.1, 214.2, 262.4, 703.9),
    (128256, 9, 1024, 107.9, 127.2, None, None, 247.7),
]


@pytest.mark.parametrize("M,T,K,tq1,tq2,tm32,tm64,gemv", T_US)
def test_order_t_takes_a_measured_fast_form(launched, M, T, K, tq1, tq2, tm32, tm64, gemv):
    """Within a sixth of the best form measured, and never slower than the per-token GEMVs
    that take every shape."""
    l, = launched("bpd_qmatmul_q8_0_dispatch_gpu", W, X, OUT, M, T, K)
    times = (tq1, tq2, tm32, tm64, gemv)
    t = one_of(times, T_FORMS)(l)
    assert t is not None, f"{l}: a form so far off that it was not measured"
    assert t <= 1.17 * min(x for x in times if x is not None), l
    assert gemv is None or t <= 1.02 * gemv, l


# ---------------------------------------------------------------- Q8_0, order S, few rows of X

def _sq(tokens, waves):
    return lambda l: l.kernel == "k_q8_0_gemm_SQ" and l.args == [tokens, waves]


S_FORMS = [_sq(4, 4), _sq(8, 4), _sq(16, 4), _sq(16, 8), lambda l: l.kernel in ("k_q8_0_gemm_SH", "k_q8_0_gemm_S")]
# M, tokens, K, then us of SQ with 4, 8 and 16 tokens x 64 rows and 16 x 128 (None: does not fit in
# LDS), of the kernels for any number of tokens
S_US = [
    (32000, 1, 32, 7.8, 7.8, 8.1, 7.8, 6.3), (8192, 200, 64, 44.7, 25.3, 16.5, 19.3, 12.6),
    (2048, 200, 64, 14.8, 9.3, 6.0, 6.1, 11.9), (70, 1, 256, 4.7, 4.8, 4.9, 5.9, 4.9),
    (2048, 4, 512, 5.7, 5.6, 5.9, 7.8, 7.8), (512, 16, 1024, 6.8, 6.6, 7.4, 10.5, 12.1),
    (8192, 17, 1024, 13.1, 9.8, 8.0, 10.6, 12.7), (14336, 24, 1024, 20.6, 14.1, 11.7, 11.4, 14.5),
    (32000, 8, 1024, 20.8, 13.4, 14.8, 15.0, 19.6), (32000, 17, 1024, 39.3, 28.2, 22.2, 25.7, 19.9),
    (32000, 32, 1024, 59.2, 35.1, 23.4, 26.2, 21.0), (128256, 16, 1024, 108.2, 64.4, 41.3, 52.4, 63.7),
    (20000, 32, 1024, 40.5, 25.5, 17.9, 22.8, 19.6), (20000, 128, 1440, 209.5, 116.9, 76.3, 79.7, 64.8),
    (14336, 64, 1440, 73.8, 42.7, 32.3, 31.6, 57.0), (32000, 64, 1440, 170.0, 96.2, 64.2, 66.9, 62.2),
    (65536, 48, 1440, 252.1, 143.0, 93.1, 97.8, 85.2), (128256, 32, 1440, 337.6, 194.3, 129.3, 138.5, 153.4),
    (4096, 200, 1440, 68.3, 41.8, 31.6, 31.0, 62.6), (2932, 197, 1248, 46.6, 28.9, 23.0, 28.1, 52.8),
    (10304, 152, 1600, 119.1, 69.5, 52.5, 64.3, 67.6), (32000, 16, 2048, 53.7, 33.2, 24.5, 23.8, 36.0),
    (32000, 24, 2048, 75.5, 46.0, 39.1, 39.7, 36.4), (32000, 32, 2048, 94.9, 58.0, 40.8, 41.0, 37.0),
    (25856, 96, 2336, 274.0, 163.4, 109.3, 109.4, 95.4), (4096, 1, 4096, 13.6, 14.7, 17.6, 26.4, 40.5),
    (4096, 64, 4096, 39.6, 26.8, 22.2, 30.3, 42.6), (14336, 1, 4096, 16.8, 17.7, 19.5, 27.3, 46.5),
    (14336, 16, 4096, 39.7, 27.2, 23.3, 31.5, 47.0), (14336, 48, 4096, 95.0, 64.8, 59.9, 60.0, 48.5),
    (8192, 96, 4096, 100.1, 62.9, 58.1, 57.1, 45.3), (32000, 17, 4096, 110.1, 76.7, 76.5, 63.4, 66.1),
    (128256, 1, 4096, 102.8, 108.3, 139.6, 123.5, 229.8), (13928, 25, 7296, 117.1, 95.2, 63.0, None, 85.3),
    (4096, 96, 8192, 97.9, 74.1, None, None, 84.7), (8192, 48, 8192, 101.0, 77.1, None, None, 79.9),
    (8192, 64, 8192, 130.2, 100.2, None, None, 83.2), (14336, 32, 8192, 115.0, 100.8, None, None, 89.6),
    (20000, 32, 8192, 199.9, 142.9, None, None, 123.5), (28672, 24, 8192, 175.8, 150.2, None, None, 123.1),
    (32000, 16, 8192, 169.1, 122.9, None, None, 126.0), (32000, 17, 8192, 206.7, 167.1, None, None, 128.1),
    (65536, 9, 8192, 200.3, 203.5, None, None, 226.1), (4096, 48, 14336, 106.9, 85.7, None, None, 135.4),
    (11584, 9, 16256, 125.9, None, None, None, 176.9), (2048, 16, 28672, 67.9, None, None, None, 261.0),
    (8192, 9, 28672, 127.8, None, None, None, 262.3),
]


@pytest.mark.parametrize("M,T,K,c4,c8,c16,c16w8,any_", S_US)
def test_order_s_takes_a_measured_fast_form(launched, M, T, K, c4, c8, c16, c16w8, any_):
    l, = launched("bpd_qmatmul_q8_0_dispatch_s_gpu", W, X, OUT, M, T, K)
    times = (c4, c8, c16, c16w8, any_)
    t = one_of(times, S_FORMS)(l)
    assert t is not None, l
    assert t <= 1.14 * min(x for x in times if x is not None), l
    assert t <= 1.05 * any_, l


# ---------------------------------------------------------------- gate and up of a layer, order S

# ffn_dim, tokens, embed_dim, then us of the products with SwiGLU in the epilogue, and of two
# products and k_swiglu
GLU_US = [
    (1408, 16, 1024, 22.4, 9.8), (2816, 200, 1024, 24.4, 20.9), (8192, 32, 1024, 23.4, 15.5),
    (14336, 17, 1024, 25.3, 22.6), (14336, 64, 1024, 25.9, 27.2), (28672, 16, 1024, 37.2, 27.7),
    (28672, 32, 1024, 38.5, 41.2), (4096, 8, 2048, 37.6, 12.6), (14336, 32, 2048, 41.8, 38.5),
    (28672, 32, 2048, 63.3, 66.6), (15488, 90, 2048, 47.5, 50.9), (4096, 1, 4096, 72.8, 17.3),
    (4096, 64, 4096, 74.6, 35.8), (14336, 8, 4096, 75.2, 34.4), (14336, 32, 4096, 76.4, 64.6),
    (14336, 96, 4096, 78.5, 81.3), (11008, 128, 4096, 77.0, 84.9), (28672, 16, 4096, 116.2, 72.8),
    (28672, 24, 4096, 114.9, 122.3), (28672, 32, 4096, 116.1, 123.5), (28672, 24, 5120, 141.7, 148.3),
    (4096, 48, 8192, 139.5, 82.4), (14336, 16, 8192, 141.6, 105.1), (28672, 24, 8192, 216.8, 226.7),
]


@pytest.mark.parametrize("F,T,E,joint,apart", GLU_US)
def test_block_takes_the_faster_gate_and_up(launched, F, T, E, joint, apart):
    import numpy as np

    cfg = llama.BpdLlamaConfig(1, E // 64, 1, 64, E, F, 1000, T, 1e-5, 1e4, 64, 0)
    lw = llama.BpdLlamaLayerWeights(*[ctypes.cast(W, t) for _, t in llama.BpdLlamaLayerWeights._fields_])
    pos = np.arange(T, dtype=np.int32)
    ls = launched("bpd_llama_block_s_gpu", X, ctypes.addressof(lw), ctypes.addressof(cfg), pos.ctypes.data, T, 0,
                  *[0x400000 + 0x100000 * i for i in range(5)], None)
    t = apart if any(l.kernel == "k_swiglu" for l in ls) else joint
    assert t <= 1.06 * min(joint, apart), ls


# ---------------------------------------------------------------- the padded layout

def test_one_padded_matrix_is_not_read_from_an_argument_block(launched):
    """The kernel for up to 3 matrices costs one matrix 0.4 us (1024x4096: 6.4 against 6.0)."""
    l, = launched("bpd_qmatmul_q8_pad64_gpu", W, X, OUT, 1024, 1, 4096)
    assert (l.kernel, l.args, l.grid) == ("k_q8_0_gemv_TP", [1], (128, 1, 1))


PAD_FORMS = [lambda l: l.kernel == "k_q8_0_gemv_TP" and l.args == [1],
             lambda l: l.kernel == "k_pad_gemv" and l.args[0] == 1,
             lambda l: l.kernel == "k_pad_gemv" and l.args[0] == 4 and not l.args[3]]
# M, tokens, K, then us of the producer/consumer kernel (None: its ring does not fit in LDS), of
# 16 and of 64 rows per workgroup, and of the kernel that took the shape before k_pad_gemv was there
PAD_US = [
    (1024, 1, 128, 3.8, 3.2, 3.1, 3.8), (5120, 1, 128, 6.3, 4.1, 3.7, 6.3), (2048, 1, 512, 4.0, 4.3, 4.1, 4.0),
    (4096, 1, 512, 4.6, 4.4, 4.2, 4.6), (1024, 2, 1024, 4.1, 4.9, 4.9, 4.1), (3072, 1, 1024, 4.7, 5.0, 5.0, 4.7),
    (4096, 1, 1024, 4.8, 5.0, 5.0, 4.8), (5120, 1, 1024, 7.0, 5.7, 5.2, 7.0), (2048, 2, 2048, 5.5, 6.3, 6.6, 5.5),
    (4096, 1, 2048, 6.2, 6.6, 7.0, 6.2), (6144, 1, 2048, 10.1, 8.0, 9.6, 10.1),
    (28672, 1, 2048, 38.9, 21.8, 21.4, 24.0), (1024, 4, 4096, 7.3, 9.0, 9.6, 7.3),
    (2048, 2, 4096, 7.8, 9.3, 10.0, 7.8), (3072, 1, 4096, 9.0, 9.7, 14.3, 9.0),
    (4096, 1, 4096, 10.2, 9.9, 14.3, 10.2), (3072, 2, 4096, 13.8, 10.7, 14.0, 13.8),
    (8192, 1, 4096, 22.4, 13.8, 16.0, 16.8), (16384, 1, 4096, 36.9, 23.6, 22.9, 25.1),
    (28672, 1, 4096, 58.8, 41.0, 40.2, 46.9), (2048, 2, 8192, 13.4, 15.2, 23.7, 13.4),
    (6144, 1, 8192, 23.2, 18.9, 26.6, 23.2), (1024, 4, 14336, 17.8, 23.4, 35.8, 17.8),
    (3072, 1, 14336, 22.6, 24.1, 38.9, 22.6), (4096, 1, 14336, 26.1, 24.7, 40.0, 26.1),
    (3072, 3, 28672, 87.9, 86.1, 74.0, 85.4), (2048, 2, 36864, 41.4, 55.7, 95.1, 41.4),
    (3072, 1, 36864, 47.2, 57.5, 100.1, 47.2), (3584, 3, 36864, 143.9, 115.4, 97.6, 110.6),
    (3072, 2, 40960, 84.8, 119.5, 107.7, 84.8), (2048, 4, 40960, 108.3, 118.8, 103.9, 110.6),
    (3072, 3, 45056, None, 194.9, 117.0, 132.8), (2048, 8, 45056, None, 257.1, 111.3, 136.8),
    (2048, 4, 57344, None, 166.1, 144.0, 152.8), (1024, 8, 65536, None, 188.4, 147.0, 843.4),
    (2800, 4, 22784, 94.1, 75.3, 57.9, 69.9), (5757, 3, 2336, 25.4, 12.6, 16.7, 15.5),
    (7296, 4, 1856, 33.2, 13.3, 18.0, 16.1), (9689, 2, 2880, 33.4, 23.2, 14.0, 26.1),
]


@pytest.mark.parametrize("M,T,K,tp,rows16,rows64,before", PAD_US)
def test_padded_product_takes_a_measured_fast_form(launched, M, T, K, tp, rows16, rows64, before):
    l, = launched("bpd_qmatmul_q8_pad64_gpu", W, X, OUT, M, T, K)
    times = (tp, rows16, rows64)
    t = one_of(times, PAD_FORMS)(l)
    assert t is not None, l
    assert t <= 1.17 * min(x for x in times if x is not None), l
    assert t <= 1.04 * before, l


# ff_dim, n_embd, then us of gate, up and SwiGLU in one launch, and of the two products in one launch
# and k_swiglu
PAD_GLU_US = [
    (1024, 1024, 5.7, 7.1), (1024, 2048, 7.3, 7.8), (4096, 2048, 12.0, 11.2), (1024, 4096, 10.7, 10.1),
    (2816, 4096, 17.4, 14.2), (4096, 4096, 17.0, 16.3), (5632, 4096, 19.6, 20.4), (14336, 4096, 42.2, 42.1),
    (1024, 8192, 25.4, 14.3), (4096, 8192, 27.3, 26.7), (5632, 8192, 31.7, 34.2), (512, 14336, 38.4, 17.4),
    (2048, 14336, 40.9, 26.9), (4096, 14336, 46.2, 42.5),
]


@pytest.mark.parametrize("F,E,joint,apart", PAD_GLU_US)
def test_padded_step_takes_the_faster_gate_and_up(launched, F, E, joint, apart):
    w = torch.zeros(64, dtype=torch.uint8)  # its address is all that is used
    cfg = dict(n_layers=1, n_embd=E, n_head=E // 64, n_head_kv=1, head_dim=64, ff_dim=F, vocab_size=1000, max_seq=64,
               eps=1e-5, rope_theta=1e4)
    m = llama.DecodeModel(cfg, [{k: w for k in llama.MATRICES + ("attn_norm", "ffn_norm")}], w, lm_head=w)
    ls = launched("bpd_llama_step_gpu", llama.W_Q8_PAD64, *m._args(w, 0))
    t = apart if any(l.kernel == "k_swiglu" for l in ls) else joint
    assert t <= 1.1 * min(joint, apart), ls


# ---------------------------------------------------------------- Q4_K spans

# M, K, then us with one and with two rows per wave (cold weights), and of the kernel without spans
SPAN_US = [
    (33, 1024, 1.9, None, 2.13), (700, 512, 1.98, None, 2.35), (1001, 1024, 2.1, None, 2.39),
    (2048, 2048, 2.38, None, 2.49), (3000, 256, 2.59, 3.2, 2.89), (3000, 1024, 2.76, 3.34, 2.98),
    (3000, 2048, 2.87, 3.47, 3.08), (3000, 3072, 2.91, 3.7, 3.2), (4096, 512, 2.92, 3.16, 2.96),
    (4096, 2048, 3.16, 3.59, 3.22), (4096, 3072, 3.32, 3.85, 3.38), (6144, 1024, 3.6, 3.82, 3.63),
    (6144, 2048, 3.9, 3.97, 3.84), (6144, 3072, 4.05, 4.3, 4.06),
]


@pytest.mark.parametrize("M,K,one,two,before", SPAN_US)
def test_short_span_rows_per_wave(launched, M, K, one, two, before):
    for name in ("bpd_qmatmul_q4k_q8k_gpu", "bpd_qmatmul_q4k_q8k_gguf_gpu"):
        l, = launched(name, W, X, OUT, M, K)
        assert l.kernel == "k_q4k_q8k_gemv_span" and not l.args[3]
        t = {1: one, 2: two}[l.args[2]]
        assert t <= 1.05 * before, l
        assert l.args[2] == 2 or l.grid[0] % 8 == 0, l  # else a line of outputs is written from 8 XCDs


# M, K, then us of the spans and of the general kernel, each quantizing x, and of the kernel that took
# the shape before there were spans of any length
FUSED_LONG_US = [
    (33, 4352, 3.79, 4.54, 4.56), (2048, 4352, 4.43, 5.47, 5.9), (5120, 4352, 7.12, 8.73, 8.72),
    (28672, 4352, 21.14, 24.27, 24.34), (512, 6144, 4.34, 5.35, 5.45), (3072, 6144, 5.88, 5.84, 6.15),
    (8192, 6144, 9.09, 9.25, 9.34), (2048, 8192, 4.73, 5.54, 5.83), (4096, 8192, 6.91, 6.88, 6.84),
    (7168, 8192, 9.98, 9.69, 9.96), (512, 8448, 5.53, 6.32, 6.52), (2048, 8448, 5.77, 6.51, 6.98),
    (3072, 8448, 8.36, 7.4, 7.41), (4096, 8448, 8.49, 8.06, 8.08), (5120, 8448, 10.39, 11.21, 11.17),
    (7168, 8448, 12.4, 11.37, 11.66), (11008, 8448, 16.61, 15.5, 15.57), (16384, 8448, 21.28, 20.12, 20.14),
    (28672, 8448, 36.64, 33.09, 33.16), (4096, 9216, 8.65, 8.3, 8.31), (9216, 9216, 14.79, 15.47, 15.37),
    (2048, 11008, 6.22, 7.39, 7.34), (4096, 11008, 8.93, 8.57, 8.55), (8192, 11008, 13.97, 13.05, 13.04),
    (11008, 11008, 18.27, 17.47, 17.46), (5120, 13824, 13.17, 14.4, 14.36), (8192, 13824, 16.49, 15.38, 15.72),
    (16384, 13824, 27.72, 27.64, 27.83), (2048, 14080, 7.28, 8.66, 8.59), (4096, 14080, 10.42, 9.92, 10.07),
    (512, 14336, 5.89, 7.96, 5.89), (2048, 14336, 6.66, 8.38, 6.66), (2560, 14336, 9.64, 8.68, 9.64),
    (3072, 14336, 9.63, 9.03, 9.63), (4096, 14336, 9.83, 10.06, 9.83), (7168, 14336, 15.49, 14.86, 15.49),
    (5120, 14336, 12.6, 14.37, 12.6), (8192, 14336, 15.85, 15.54, 15.85), (28672, 14336, 45.71, 46.08, 45.71),
]


@pytest.mark.parametrize("M,K,span,general,before", FUSED_LONG_US)
def test_long_fused_rows_take_a_measured_fast_form(launched, M, K, span, general, before):
    l, = launched("bpd_qmatmul_q4k_q8k_fused_gpu", W, X, OUT, M, K)
    t = {"k_q4k_fused_span": span, "k_q4k_fused_gemv": general}[l.kernel]
    assert t <= 1.04 * min(span, general), l
    assert t <= 1.04 * before, l
