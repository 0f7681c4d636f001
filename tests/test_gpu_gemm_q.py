"""The Q8_0 and Q6_K GEMMs of wide passes (k_gemm_q80, k_gemm_q6k) against the GEMVs of narrow ones: an
MoE layer over T rows gives the same bits as the same rows in calls of at most 16 (which take the
GEMVs; so do the shorter of the others, where the GEMMs do not pay), at token tiles of every height and their remainders, at rows and K that do not fill the blocks,
and with activations whose block scales are f16 subnormals or large. A prompt prefilled in one pass
(dense projections and dense FFN as GEMMs) gives the bits of 16-row passes. The GEMVs are held to the
oracle elsewhere; one layer here is too."""
import dataclasses

import numpy as np
import pytest

import oracle_py as O
from helpers import assert_close
from zonos2_amd import configs, synth
from zonos2_amd.z2h import Context, Model

pytestmark = pytest.mark.gpu

Q8, Q6 = configs.Q8_0, configs.Q6_K


def _cfg(bulk, E, k, ff, d=512, dense=0):
    return configs.ModelConfig(f"gq-{bulk}-{E}-{k}-{ff}", n_layer=1 + dense, n_embd=d, n_head=8, n_head_kv=2, head_dim=64, n_expert=E,
                               top_k=k, n_ff=ff, bulk=bulk, audio_vocab=33, expert_used=[0] * dense + [k], router_mlp_std=0.1, router_out_std=0.2)


@pytest.mark.parametrize("scale", [1.0, 1e-5, 1e5], ids=["x1", "x1e-5", "x1e5"])
@pytest.mark.parametrize("bulk,E,k,ff,T", [(Q8, 8, 2, 288, 67), (Q8, 4, 2, 288, 17), (Q8, 4, 1, 256, 300), (Q8, 2, 2, 800, 1501),
                                           (Q6, 8, 2, 256, 67), (Q6, 4, 2, 512, 17), (Q6, 4, 1, 256, 300), (Q6, 2, 2, 768, 1501),
                                           (Q8, 8, 2, 288, 325), (Q8, 64, 1, 288, 650), (Q8, 3, 1, 544, 647), (Q6, 8, 2, 256, 170), (Q6, 64, 1, 256, 650), (Q6, 3, 1, 512, 331)])
def test_moe_gemm_equals_gemv(bulk, E, k, ff, T, scale):
    cfg = _cfg(bulk, E, k, ff)
    m = Model(cfg.hparams(), synth.generate_model(cfg, 5 + T))
    ctx = Context(None, 1, 256, model=m, max_rows=T)
    x = (scale * np.random.default_rng(T).standard_normal((T, cfg.n_embd))).astype(np.float32)
    x[T // 2] = 0.0                                                  # an all-zero row: zero block scales
    print(f"{cfg.name} T={T} scale={scale}", flush=True)
    got = ctx.moe_forward(0, x)
    want = np.concatenate([ctx.moe_forward(0, x[i:i + 16]) for i in range(0, T, 16)])
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"max |d| {np.abs(got - want).max():.3e}"
    ctx.close(); m.close()


@pytest.mark.parametrize("bulk,offset,f16", [(Q8, 0, 0x7e01), (Q8, 0, 0x7c00), (Q6, 208, 0x7c00)], ids=["q8_0-nan", "q8_0-inf", "q6_k-inf"])
def test_non_finite_scales_stay_in_their_block(bulk, offset, f16):
    """a weight block's scale or a token's scale that is infinite or NaN gives what the GEMV gives: the other
    rows, and the sums of the other blocks, are untouched"""
    cfg = _cfg(bulk, 2, 2, 512)
    model = synth.generate_model(cfg, 21)
    t = model["blk.0.ffn_down_exps.weight"]
    raw = np.frombuffer(bytes(t.data), np.uint8).copy()
    rb = configs.row_bytes(bulk, cfg.n_ff)
    bb = configs.BLOCK[bulk][1]
    for row, blk in ((5, 1), (37, 0), (cfg.n_embd + 100, 1)):            # experts 0, 0 and 1
        raw[row * rb + blk * bb + offset:][:2] = np.frombuffer(np.uint16(f16).tobytes(), np.uint8)
    model["blk.0.ffn_down_exps.weight"] = dataclasses.replace(t, data=raw)
    m = Model(cfg.hparams(), model)
    T = 331
    ctx = Context(None, 1, 256, model=m, max_rows=T)
    x = np.random.default_rng(2).standard_normal((T, cfg.n_embd)).astype(np.float32)
    x[3] *= 1e9                                                          # its block scales are infinite in f16
    print(f"{cfg.name} non-finite scales", flush=True)
    got = ctx.moe_forward(0, x)
    want = np.concatenate([ctx.moe_forward(0, x[i:i + 16]) for i in range(0, T, 16)])
    rest = np.delete(np.arange(cfg.n_embd), [5, 37, 100])
    assert np.isfinite(want[4:][:, rest]).all() and not np.isfinite(want[:, [5, 37, 100]]).any()
    if f16 == 0x7c00:
        assert np.isinf(want[4:][:, [5, 37, 100]]).any()
    np.testing.assert_array_equal(got, want)                             # (NaN equals NaN)
    ctx.close(); m.close()


@pytest.mark.parametrize("bulk", [Q8, Q6], ids=["q8_0", "q6_k"])
def test_moe_gemm_vs_oracle(bulk):
    cfg = _cfg(bulk, 4, 2, 256)
    model = synth.generate_model(cfg, 9)
    ctx = Context(cfg.hparams(), 1, 256, max_rows=131)
    ctx.upload(model)
    om = O.OracleModel(cfg.hparams(), model)
    x = np.random.default_rng(3).standard_normal((131, cfg.n_embd)).astype(np.float32)
    print(f"{cfg.name} vs oracle", flush=True)
    got = ctx.moe_forward(0, x)
    ref = O.router(om, 0, x, None)
    _, want = O.experts(om, 0, x, ref["sel"], ref["w"])
    assert_close(cfg.name, got, want)
    ctx.close()


@pytest.mark.parametrize("bulk", [Q8, Q6], ids=["q8_0", "q6_k"])
def test_moe_gemm_of_many_rows_vs_oracle(bulk):
    """(331 rows: above the line from which layers of this size take the GEMMs)"""
    cfg = _cfg(bulk, 4, 2, 256)
    model = synth.generate_model(cfg, 9)
    ctx = Context(None, 1, 256, model=Model(cfg.hparams(), model), max_rows=331)
    om = O.OracleModel(cfg.hparams(), model)
    x = np.random.default_rng(3).standard_normal((331, cfg.n_embd)).astype(np.float32)
    print(f"{cfg.name}, {len(x)} rows vs oracle", flush=True)
    got = ctx.moe_forward(0, x)
    ref = O.router(om, 0, x, None)
    _, want = O.experts(om, 0, x, ref["sel"], ref["w"])
    assert_close(cfg.name, got, want)
    ctx.close()


@pytest.mark.parametrize("T", [150, 197, 705])
@pytest.mark.parametrize("bulk", [Q8, Q6], ids=["q8_0", "q6_k"])
def test_prefill_gemm_equals_narrow_passes(bulk, T):
    cfg = _cfg(bulk, 4, 2, 768, d=1024, dense=1)
    m = Model(cfg.hparams(), synth.generate_model(cfg, 7))
    rng = np.random.default_rng(T)
    ids = np.concatenate([rng.integers(0, cfg.audio_vocab, (T, cfg.n_codebooks)),
                          rng.integers(0, cfg.text_vocab + 1, (T, 1))], axis=1).astype(np.int32)
    outs, kvs = [], []
    for chunk in (T, 16):
        ctx = Context(None, 2, T, model=m, max_rows=T)
        ctx.set_prefill_chunk(chunk)
        print(f"{cfg.name}: {T} rows in passes of {chunk}", flush=True)
        outs.append(ctx.prefill(1, ids))
        kvs.append([ctx.kv_read(L, 1, 0, T) for L in range(cfg.n_layer)])
        ctx.close()
    np.testing.assert_array_equal(outs[0], outs[1])
    for a, b in zip(*kvs):
        np.testing.assert_array_equal(a[0], b[0])
        np.testing.assert_array_equal(a[1], b[1])
    m.close()


@pytest.mark.parametrize("T", [1037, 1080])
@pytest.mark.parametrize("bulk", [Q8, Q6], ids=["q8_0", "q6_k"])
def test_tall_tiles_equal_narrow_passes(bulk, T):
    """matrices of 2048 rows, where a pass of this length takes the tallest token tiles (32 rows for Q8_0, 64 for Q6_K) in
    W_o, the dense SwiGLU and down matmuls, and the experts'; the last tile is partly empty"""
    cfg = configs.ModelConfig(f"tall-{bulk}", n_layer=3, n_embd=2048, n_head=8, n_head_kv=2, head_dim=64, n_expert=2, top_k=2, n_ff=2048,
                              bulk=bulk, audio_vocab=33, expert_used=[0, 2, 0], router_mlp_std=0.1, router_out_std=0.2)
    m = Model(cfg.hparams(), synth.generate_model(cfg, 8))
    rng = np.random.default_rng(T)
    ids = np.concatenate([rng.integers(0, cfg.audio_vocab, (T, cfg.n_codebooks)),
                          rng.integers(0, cfg.text_vocab + 1, (T, 1))], axis=1).astype(np.int32)
    outs, kvs = [], []
    for chunk in (T, 16):
        ctx = Context(None, 1, T, model=m, max_rows=T)
        ctx.set_prefill_chunk(chunk)
        print(f"{cfg.name}: {T} rows in passes of {chunk}", flush=True)
        outs.append(ctx.prefill(0, ids))
        kvs.append([ctx.kv_read(L, 0, 0, T) for L in range(cfg.n_layer)])
        ctx.close()
    for a, b in zip(*kvs):
        np.testing.assert_array_equal(a[0], b[0])
        np.testing.assert_array_equal(a[1], b[1])
    np.testing.assert_array_equal(outs[0], outs[1])
    m.close()
