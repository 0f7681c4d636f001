"""The integer inputs of a pass share one staging block: steps keep theirs at fixed places, prompt chunks and mixed
passes pack theirs by their own row count. A sequence of all of them, of different widths after one another, gives the
same bits in a context of many rows as in one of few, and the fed tables of a resident step survive a refused call."""
import numpy as np
import pytest

from zonos2_amd import configs, synth
from zonos2_amd.z2h import Context, Model, Z2HError

pytestmark = pytest.mark.gpu


def _passes(cfg, model, max_rows):
    n_slots, cap, W = 6, 160, cfg.n_codebooks + 1
    ctx = Context(None, n_slots, cap, model=model, max_rows=max_rows)
    rng = np.random.default_rng(11)
    out = []

    def ids(n):
        return np.concatenate([rng.integers(0, cfg.audio_vocab, (n, cfg.n_codebooks)),
                               rng.integers(0, cfg.text_vocab + 1, (n, 1))], axis=1).astype(np.int32)

    def say(what):
        print(f"max_rows {max_rows}: {what}", flush=True)

    ctx.set_prefill_chunk(40)
    for slot, n in ((0, 97), (1, 5), (2, 41)):
        say(f"prefill {n}")
        out.append(ctx.prefill(slot, ids(n), spk=rng.standard_normal(cfg.spk_dim).astype(np.float32), spk_pos=n // 2))
    say("step of 3")
    out.append(ctx.step([0, 1, 2], [97, 5, 41], ids=ids(3)))
    say("mixed pass of 64 rows, no map")
    i64 = ids(64)
    out.append(ctx.step_mixed([3] * 61 + [0, 1, 2], list(range(61)) + [98, 6, 42], i64, [60, 61, 62, 63]))
    say("mixed pass of 2 rows with a map, rows asked for repeatedly")
    emb = rng.standard_normal((1, cfg.n_embd)).astype(np.float32)
    i2 = ids(2)
    i2[1] = -7                                                        # (not read: the row takes its embedding)
    out.append(ctx.step_mixed([4, 5], [0, 0], i2, [1, 0, 1, 1, 0], emb_map=[-1, 0], emb=emb))
    say("mixed pass without outputs")
    out.append(ctx.step_mixed([4, 5], [1, 1], ids(2), []))
    say("step of 5, fed")
    out.append(ctx.step([4, 0, 1, 2, 5], [2, 99, 7, 43, 2], ids=ids(5)))
    sp = [dict(temperature=0.8, top_k=20, top_p=0.9, min_p=0.0, rep_penalty=1.0, rep_codebooks=0, greedy=0)] * 5
    for _ in range(3):
        out.append(ctx.sample_feed(sp, rng.random((5, cfg.n_codebooks))))
        with pytest.raises(Z2HError):
            ctx.step([0, 0], [100, 101], ids=ids(2))                  # refused before anything is sent
        ctx.step_resident(5)
    out.append(ctx.sample(sp, rng.random((5, cfg.n_codebooks))))
    for L in range(cfg.n_layer):
        for slot, n in ((0, 103), (1, 11), (2, 47), (3, 61), (4, 6), (5, 6)):
            out += list(ctx.kv_read(L, slot, 0, n))
    ctx.close()
    return out


def test_pass_inputs_do_not_depend_on_the_capacity():
    cfg = configs.ModelConfig("inputs", n_layer=2, n_embd=256, n_head=8, n_head_kv=2, head_dim=32, n_expert=4, top_k=2, n_ff=256,
                              bulk=configs.Q8_0, audio_vocab=65, expert_used=[0, 2])
    model = Model(cfg.hparams(), synth.generate_model(cfg, 4))
    small, large = _passes(cfg, model, 64), _passes(cfg, model, 4099)
    assert len(small) == len(large)
    for a, b in zip(small, large):
        np.testing.assert_array_equal(a, b)
    model.close()
