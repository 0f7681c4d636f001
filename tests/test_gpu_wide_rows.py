"""Wide MoE layer calls (more than 64 rows: k_router_down_t, k_gemm_q4k for Q4_K experts, k_gemm_f16's
64- and 128-row tiles for F16 ones, the latter gate/up at 256 x 2048 and down at 256 x 4096) against calls
of at most 16 rows of the same layer: same bits. Model widths that fill and do not fill the router's 64
chains per step, and more than 2048 columns (two halves), on both sides of the line from which a call takes
k_router_down_t; rows that leave remainders in its 4-token tiles and its grid, and in the GEMMs' tiles."""
import numpy as np
import pytest

from zonos2_amd import configs, synth
from zonos2_amd.z2h import Context, Model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bulk,d,E,k,ff,T", [
    (configs.Q8_0, 320, 4, 2, 256, 65), (configs.Q8_0, 320, 4, 2, 256, 421), (configs.Q8_0, 2080, 4, 1, 256, 67), (configs.Q8_0, 2080, 4, 1, 256, 131), (configs.Q8_0, 4096, 2, 1, 256, 70),
    (configs.F16, 2048, 4, 2, 256, 2051), (configs.F16, 512, 4, 2, 256, 190), (configs.F16, 768, 4, 2, 512, 300), (configs.Q4_K, 256, 2, 1, 256, 65), (configs.Q4_K, 512, 4, 2, 768, 129),
    (configs.Q4_K, 1024, 2, 2, 1536, 97), (configs.Q4_K, 768, 3, 1, 256, 1300),
    (configs.F16, 256, 2, 2, 2048, 1101), (configs.F16, 256, 2, 2, 2048, 1072), (configs.F16, 4096, 2, 2, 256, 1101)],
    ids=lambda v: str(v))
def test_wide_rows_equal_narrow(bulk, d, E, k, ff, T):
    cfg = configs.ModelConfig(f"wr-{bulk}-{d}-{E}-{k}-{ff}", n_layer=2, n_embd=d, n_head=8, n_head_kv=2, head_dim=32, n_expert=E,
                              top_k=k, n_ff=ff, bulk=bulk, audio_vocab=33, expert_used=[k, k], router_mlp_std=0.1, router_out_std=0.2)
    m = Model(cfg.hparams(), synth.generate_model(cfg, 3 + T))
    ctx = Context(None, 1, 256, model=m, max_rows=T)
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, d)).astype(np.float32)
    state = rng.standard_normal((T, cfg.router_dim)).astype(np.float32)
    print(f"{cfg.name} T={T}", flush=True)
    got = ctx.moe_forward(1, x, state)
    want = np.concatenate([ctx.moe_forward(1, x[i:i + 16], state[i:i + 16]) for i in range(0, T, 16)])
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), f"max |d| {np.abs(got - want).max():.3e}"
    ctx.close(); m.close()
