"""The host rules that choose between two shapes of one kernel (csrc/z2h_rules.h), on the CPU: the choices at sizes
where both sides were measured on 256 compute units."""
import subprocess

import pytest

N_CU = 256


@pytest.fixture(scope="module")
def ask(root, tmp_path_factory):
    exe = tmp_path_factory.mktemp("rules") / "rules_kat"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", str(root / "tests" / "native" / "rules_kat.cpp"), "-o", str(exe)], check=True)

    def run(queries):
        text = "\n".join(" ".join(map(str, (*q, 0, 0, 0, 0)[:6])) for q in queries)
        out = subprocess.run([str(exe)], input=text, check=True, capture_output=True, text=True).stdout.split()
        assert len(out) == len(queries)
        return [x == "1" for x in out]
    return run


# (experts, routes per expert, FFN width, model width) -> 128-row tiles: gate/up, down
TALL = [
    # too few blocks for the chip: 64-row tiles measured 1.2 to 1.8 times as fast
    ((16, 93, 1536, 2048), (False, False)), ((16, 128, 1536, 2048), (False, False)), ((8, 128, 1536, 2048), (False, False)),
    ((4, 512, 1536, 2048), (False, False)), ((8, 260, 256, 512), (False, False)), ((8, 150, 4096, 2048), (True, False)),
    # a round of tall tiles more than the 64-row ones' rounds are worth
    ((32, 128, 1536, 2048), (False, True)), ((32, 210, 1536, 2048), (False, False)), ((16, 300, 1536, 2048), (False, True)),
    # uneven loads: no tall tiles at few routes per expert
    ((32, 75, 1536, 2048), (False, False)),
    # rounds saved
    ((16, 192, 1536, 2048), (True, False)), ((32, 260, 1536, 2048), (True, False)), ((32, 450, 1536, 2048), (True, False)),
    ((128, 512, 2048, 1024), (True, True)),
]


def test_f16_tall_tiles(ask):
    q, want = [], []
    for (E, per, ff, d), w in TALL:
        q += [("tall", -(-ff // 128), per * E, E, N_CU), ("tall", -(-d // 256), per * E, E, N_CU)]
        want += w
    assert ask(q) == want


def test_f16_tall_tiles_never_without_a_full_chip(ask):
    """no tall tiles where the 64-row ones fit one round, whatever the loads"""
    q = [("tall", rb, items, E, N_CU) for rb in (1, 3, 8, 16, 32) for E in (1, 2, 8, 32, 128) for items in (64, 500, 2047, 9001, 40000)
         if rb * (items / 64 + E) <= 2 * N_CU]
    assert q and not any(ask(q))


# (K, rows, tokens) -> k_gemm_f16_few: where the two differed by more than 5%
FEW = [
    ((256, 9234, 16), False), ((256, 9234, 64), False), ((256, 18468, 1), False),
    ((512, 512, 16), True), ((512, 512, 64), False), ((512, 3078, 16), True), ((512, 4104, 64), False), ((512, 9234, 16), False),
    ((768, 297, 64), True), ((768, 4104, 64), True), ((768, 9234, 1), True), ((768, 18468, 16), False),
    ((1024, 1028, 64), True), ((1024, 9234, 16), True), ((1024, 18468, 16), False),
    ((1536, 18468, 1), True), ((2048, 9225, 1), True), ((2048, 3088, 64), True), ((2048, 18468, 33), True), ((2048, 36864, 16), False),
]


def test_f16_few_rows(ask):
    assert ask([("few", rows, K // 256, T, 0) for (K, rows, T), _ in FEW]) == [w for _, w in FEW]


# (rows, model width) -> k_router_down_t in an MoE layer call
RDOWN = [((65, 768), False), ((200, 768), True), ((65, 1024), False), ((160, 1024), True), ((65, 1280), False), ((112, 1280), True),
         ((64, 2048), False), ((65, 2048), True), ((65, 2304), False), ((72, 3072), False), ((96, 3072), True), ((65, 4096), True),
         ((64, 512), False), ((65, 512), True), ((256, 256), True)]


def test_router_down_reuse(ask):
    full = lambda d: d % 64 == 0 and d // 64 & (d // 64 - 1) == 0
    assert ask([("rdown", T, d, int(full(d)), 0) for (T, d), _ in RDOWN]) == [w for _, w in RDOWN]


# (Q6_K, routes, experts, model width, FFN width) -> the GEMMs
QEXP = [((0, 72, 8, 512, 256), False), ((0, 384, 8, 512, 256), False), ((0, 800, 8, 512, 256), True), ((0, 192, 16, 1024, 768), False),
        ((0, 512, 8, 1024, 768), True), ((0, 256, 32, 2048, 1536), True), ((0, 255, 32, 2048, 1536), False), ((0, 64, 4, 2048, 1536), False),
        ((0, 256, 4, 2048, 1536), True), ((0, 1025, 128, 512, 256), True), ((0, 1025, 129, 512, 256), False),
        ((1, 72, 8, 512, 256), False), ((1, 384, 8, 512, 256), True), ((1, 72, 8, 1024, 768), False), ((1, 160, 8, 1024, 768), True),
        ((1, 72, 4, 2048, 1536), True), ((1, 255, 32, 2048, 1536), False)]


def test_quant_gemm_experts(ask):
    assert ask([("qexp", q6, r, E, d * ff, 1024) for (q6, r, E, d, ff), _ in QEXP]) == [w for _, w in QEXP]
