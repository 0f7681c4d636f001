"""Dense F16 matmuls of few rows (k_gemm_f16_few, 16 or 32 weight rows per block, or the narrow k_gemm_f16 where K is short) against the
wide GEMM: the columns
of a step of T requests (projections and head of T token rows: one wave's remainder, several waves, all
64) get the bits of the same columns in steps of at most 16 and in one of 70 (k_gemm_f16). Row lengths of one
superblock, of part of a phase and of more than two phases; head rows that leave remainders, below and above the
count from which a block takes 32."""
import numpy as np
import pytest

from zonos2_amd import configs, synth
from zonos2_amd.z2h import Context, Model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,vocab", [(256, 33), (512, 33), (512, 1026), (768, 1026), (2304, 1026)])
def test_few_rows_equal_wide_and_narrow(d, vocab):
    cfg = configs.ModelConfig(f"few-{d}-{vocab}", n_layer=1, n_embd=d, n_head=4, n_head_kv=2, head_dim=64, n_expert=0, top_k=0,
                              n_ff=256, bulk=configs.F16, audio_vocab=vocab, expert_used=[0])
    m = Model(cfg.hparams(), synth.generate_model(cfg, d))
    n = 70
    ctx = Context(None, n, 64, model=m)
    rng = np.random.default_rng(d)
    ids = np.concatenate([rng.integers(0, cfg.audio_vocab, (n, cfg.n_codebooks)),
                          rng.integers(0, cfg.text_vocab + 1, (n, 1))], axis=1).astype(np.int32)
    slots, past = np.arange(n, dtype=np.int32), np.zeros(n, np.int32)

    def step(i, j):
        print(f"{cfg.name} columns {i}..{j - 1}", flush=True)
        return ctx.step(slots[i:j], past[i:j], ids=ids[i:j]).view(np.uint32)

    wide = step(0, n)
    for T in (1, 16, 17, 33, 64):
        assert np.array_equal(step(0, T), wide[:T]), f"{T} columns"
    assert np.array_equal(step(53, 70), wide[53:])
    ctx.close()
    m.close()
