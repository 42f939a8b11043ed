"""Products that share their activation rows in one launch: Q, K and V, gate and up of a
multi-token layer (bpd_llama_block_gpu, both orders) and of a padded-Q8 decode step, at row
counts that end inside a tile, and the binary16 cache values of the attention.

The expected layer is put together from the C oracle's own parts (norm, quantizer, single-
matrix products, rope, attention, SwiGLU), so nothing here needs the reference's C.  Bar:
bit-exact.
"""
import ctypes

import numpy as np
import pytest

import llama_model as LM
from bpd_substrate_amd import gpu, llama, synth
from helpers import assert_bits_equal, to_np
from launches import Recorder
from oracle import oracle as O
from test_gpu_forward import LAYER, config, make_layer

# order, embed_dim, heads, kv heads, ffn_dim, tokens, and the kernels of Q/K/V and of gate/up
TQ, TM, SQ, SH = "k_q8_0_gemm_TQ", "k_q8_0_gemm_TM", "k_q8_0_gemm_SQ", "k_q8_0_gemm_SH"
BLOCKS = [("T", 1056, 33, 33, 2784, 6, (TQ, 1), (TQ, 2)),
          ("T", 256, 8, 2, 2080, 300, (TQ, 2), (TM, 2)),
          ("T", 160, 5, 1, 544, 70, None, (TM, 2)),        # an odd number of blocks: no 4-byte alignment
          ("T", 512, 16, 16, 2080, 130, (TM, 2), (TM, 4)),
          ("T", 1024, 32, 32, 1056, 130, (TM, 4), (TM, 2)),
          ("S", 1024, 8, 8, 4128, 9, (SQ, 4), (SQ, 16)),
          ("S", 1024, 32, 8, 1120, 130, (SQ, 16), (SQ, 16)),
          ("S", 512, 16, 16, 8224, 20, (SQ, 4), (SH, 2)),
          ("S", 256, 8, 8, 4160, 130, (SH, 1), (SH, 4))]   # SwiGLU in the epilogue


def _block_cfg(E, H, HKV, F, T):
    return config(L=1, E=E, H=H, HKV=HKV, D=E // H, F=F, S=T + 3, f16=0)


def _call_block(call, order, cfg, layer, x, pos, T, kc, vc, scratch):
    c = llama.BpdLlamaConfig(*(cfg[n] for n, _ in llama.BpdLlamaConfig._fields_))
    return call("bpd_llama_block_s_gpu" if order == "S" else "bpd_llama_block_gpu", x, ctypes.addressof(layer),
                ctypes.addressof(c), pos.ctypes.data, T, 0, kc, vc, *scratch, None)


@pytest.mark.parametrize("order,E,H,HKV,F,T,qkv,gate_up", BLOCKS)
def test_blocks_take_the_kernels_they_are_for(tmp_path, order, E, H, HKV, F, T, qkv, gate_up):
    p = 0x100000
    layer = llama.BpdLlamaLayerWeights(*[ctypes.cast(p, t) for _, t in llama.BpdLlamaLayerWeights._fields_])
    pos = np.arange(T, dtype=np.int32)
    ls = _call_block(Recorder(str(tmp_path)), order, _block_cfg(E, H, HKV, F, T), layer, p, pos, T, p, p, [p, p, p])
    gemms = [(l.kernel, l.args[0]) for l in ls if "q8_0_gem" in l.kernel]
    o = 1 if qkv is not None else 3        # where Q, K and V are launches of their own
    assert len(gemms) == o + 3, gemms      # ..., O, gate and up, down
    assert qkv is None or gemms[0] == qkv
    assert gemms[o + 1] == gate_up


def _oracle_block(order, cfg, lw, x, pos):
    E, H, HKV, D, F = (cfg[n] for n in ("embed_dim", "n_heads", "n_kv_heads", "head_dim", "ffn_dim"))
    T, S = pos.size, cfg["max_seq_len"]
    rows = lambda a: np.concatenate([O.quant_q8_0(r) for r in a])
    norm = lambda a, w: np.stack([O.rmsnorm(r, w, cfg["rms_eps"]) for r in a])

    def mul(name, a, n, k):
        return O.dispatch_q8_0(lw[name], rows(a), n, T, k, order, nthreads=8).reshape(T, n)

    h = norm(x, lw["attn_norm_w"])
    q, k, v = mul("w_q", h, H * D, E), mul("w_k", h, HKV * D, E), mul("w_v", h, HKV * D, E)
    kc, vc = np.zeros((S, HKV * D), np.float32), np.zeros((S, HKV * D), np.float32)
    a = np.empty((T, H * D), np.float32)
    for t in range(T):
        q[t] = O.rope_norm(q[t], H, D, int(pos[t]), cfg["rope_base"])
        kc[t] = O.rope_norm(k[t], HKV, D, int(pos[t]), cfg["rope_base"])
        vc[t] = v[t]
        a[t] = O.gqa_attn(q[t], kc, vc, S, t, H, HKV, D, np.float32(1.0) / np.sqrt(np.float32(D)))
    x = x + mul("w_o", a, E, H * D)
    h = norm(x, lw["ffn_norm_w"])
    y = O.swiglu(mul("w_gate", h, F, E).reshape(-1), mul("w_up", h, F, E).reshape(-1)).reshape(T, F)
    return x + mul("w_down", y, E, F), kc, vc


@pytest.mark.gpu
@pytest.mark.parametrize("order,E,H,HKV,F,T,qkv,gate_up", BLOCKS)
def test_block_equals_single_products(dev, order, E, H, HKV, F, T, qkv, gate_up):
    import torch

    cfg = _block_cfg(E, H, HKV, F, T)
    lw = make_layer(cfg, 900 + E + F)
    x = synth.normal_f32(T * E, synth.key(91, F)).reshape(T, E)
    pos = np.arange(T, dtype=np.int32)
    want, kw, vw = _oracle_block(order, cfg, lw, x, pos)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    dl = {n: d(lw[n]) for n in LAYER}
    xd, kd, vd = d(x.reshape(-1)), d(np.zeros_like(kw).reshape(-1)), d(np.zeros_like(vw).reshape(-1))
    scratch = [torch.empty(T * max(E, F), device=dev) for _ in range(3)]
    print(f"block {order} {E}x{F} {T} tokens", flush=True)
    gpu._use_torch_stream()
    _call_block(gpu.call, order, cfg, llama.layer_struct(dl), xd, pos, T, kd, vd, scratch)
    torch.cuda.synchronize()
    assert_bits_equal(to_np(kd), kw.reshape(-1), "K cache")
    assert_bits_equal(to_np(vd), vw.reshape(-1), "V cache")
    assert_bits_equal(to_np(xd), want.reshape(-1), "x after the block")


# n_embd = 65 * 32: a last group of one block; Q, K and V together (6,240 rows) take k_pad_gemv's 16-row
# form with three matrices, gate and up its SwiGLU form; n_embd = 4,160: the 64-row form (12,480 rows), and
# gate and up two matrices of k_pad_gemv, as K >= 4096 and F <= 4096
@pytest.mark.gpu
@pytest.mark.parametrize("E,F", [(2080, 96), (2080, 1056), (4160, 160)])
@pytest.mark.parametrize("data", ["plain", "m128", "nan"])
def test_padded_step_equals_restatement(dev, E, F, data):
    """m128: -128 quants in every matrix, which a Q8_0 quantizer does not write; nan: a NaN scale in
    a block of a gate row and one of an up row, so y has NaNs and the down product's input with it."""
    import torch

    cfg = LM.config(E=E, H=E // 32, HKV=E // 32, D=32, F=F, L=1, vocab=200, max_seq=8)
    layers, head = LM.make(cfg, 0, seed=E + F)
    if data == "m128":
        for m in LM.MATS:
            b = layers[0][m].reshape(-1, 34)
            b[::7, 2 + 5] = 0x80
    if data == "nan":
        for m, row in (("gate", F // 2), ("up", F - 1)):
            layers[0][m].reshape(F, E // 32, 34)[row, 3, 0:2] = np.array([0x00, 0x7E], np.uint8)
    dl, on, lm, lmf = LM.to_device(cfg, layers, head, llama.W_Q8_PAD64, dev)
    m = llama.DecodeModel(cfg, dl, on, lm_head=lm, lm_f32=lmf, fmt=llama.W_Q8_PAD64, device=dev)
    ko, vo = LM.caches(cfg)
    for pos, e in enumerate(LM.embeddings(cfg, 2, seed=F)):
        print(f"padded step {E}x{F} {data} position {pos}", flush=True)
        tok, x, h, logits = O.llama_step(llama.W_Q8_PAD64, layers, cfg, ko, vo, pos, e, head["out_norm"], head["lm"],
                                         head["lm_f32"], cfg["vocab_size"])
        got = m.step(torch.from_numpy(e).to(dev), pos)
        assert got == tok
        nan = data == "nan"
        if nan:
            y = to_np(m.buf_t["gate"])
            assert np.flatnonzero(np.isnan(y)).tolist() == [F // 2, F - 1]
        assert_bits_equal(to_np(m.buf_t["x"]), x, "x", nan_equal=nan)
        assert_bits_equal(to_np(m.buf_t["logits"]), logits, "logits", nan_equal=nan)
        assert_bits_equal(to_np(m.k_cache[0]), ko[0], "K cache", nan_equal=nan)
        assert_bits_equal(to_np(m.v_cache[0]), vo[0], "V cache", nan_equal=nan)
        if nan:
            break  # the next position would start from NaNs only


@pytest.mark.gpu
@pytest.mark.parametrize("pos", [3, 1100])  # the short-context kernel, and the one that streams V
def test_every_binary16_cache_value(dev, pos):
    """All 65,536 binary16 values of a V cache in attention: row 0 holds them, every other row and the
    step's own v are zero, so column d gives value * p0, with p0 from a column that holds 1.0.  A NaN's
    sign and payload come back, quieted, as x86's conversion and product give them."""
    import torch

    H, D, S = 16, 128, 2048
    cfg = LM.config(E=H * D, H=H, HKV=H, D=D, F=64, L=1, vocab=64, max_seq=S)
    layers, head = LM.make(cfg, 0, seed=5)
    layers[0]["v"].reshape(-1, 34)[:, 2:] = 0
    dl, on, lm, lmf = LM.to_device(cfg, layers, head, llama.W_Q8_PAD64, dev)
    m = llama.DecodeModel(cfg, dl, on, lm_head=lm, lm_f32=lmf, fmt=llama.W_Q8_PAD64, device=dev, kv_cache_f16=True)
    e = torch.from_numpy(LM.embeddings(cfg, 1, seed=3)[0]).to(dev)
    per = H * (D - 1)
    for first in range(0, 65536, per):
        bits = np.arange(first, first + per, dtype=np.uint32) & 0xFFFF
        row = np.full((H, D), 0x3C00, np.uint16)
        row[:, 1:] = bits.astype(np.uint16).reshape(H, D - 1)
        m.k_cache[0].zero_()
        m.v_cache[0].zero_()
        m.v_cache[0][:H * D] = torch.from_numpy(row.view(np.int16).reshape(-1)).to(dev)
        m.step(e, pos)
        out = to_np(m.buf_t["attn_out"]).reshape(H, D)
        p0 = out[:, :1]
        assert (p0 > 0).all() and (p0 <= 1).all()
        with np.errstate(invalid="ignore"):
            want = row[:, 1:].view(np.float16).astype(np.float32) * p0 + np.float32(0.0)
        nan = (0x7FC00000 | ((bits & 0x8000) << 16) | ((bits & 0x3FF) << 13)).reshape(H, D - 1).view(np.float32)
        want = np.where(np.isnan(want), nan, want)
        assert_bits_equal(out[:, 1:].reshape(-1), want.reshape(-1), f"values from {first:#x}")
