"""How the GEMMs of more than 16 rows split K: host arithmetic, no device
(parity unpinned: the reference has no counterpart)."""
import random
import subprocess
import sys

import pytest

import vlrf_amd as V
from conftest import ROOT, gemm_plan


@pytest.mark.parametrize("dtype", [V.DT_Q8_0, V.DT_Q4_0, V.DT_F32])
def test_plan_of_refused_k_leaves_it_whole(dtype):
    """K below a step of 64 or off it, and f32 weights: the calls size their
    scratch before they refuse these.  In a process of its own: a division by
    zero steps would end it."""
    code = ("import sys; sys.path[:0] = [%r, %r]\n"
            "from conftest import gemm_plan\n"
            "for M in (17, 100, 129, 2048):\n"
            "    for K in (32, 96, 160, 4128) + ((1, 63, 64, 4096) if %d == 0 else ()):\n"
            "        for sw in (0, 1):\n"
            "            assert gemm_plan(%d, M, 300, K, sw) == (1, K, False, 0), (M, K, sw)\n"
            "print('ok')" % (ROOT, ROOT + "/tests", dtype, dtype))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stderr[-800:])


def test_slices_cover_k_and_their_bytes():
    """Any accepted shape: whole steps, no empty slice, a bounded count, the bytes of the partial sums."""
    rng = random.Random(3)
    for _ in range(4000):
        M, N = int(2 ** rng.uniform(4.1, 11.2)), int(2 ** rng.uniform(0, 14))
        K, sw = 64 * int(2 ** rng.uniform(0, 8)), rng.random() < 0.3
        S, kl, few, part = gemm_plan(rng.choice([V.DT_Q8_0, V.DT_Q4_0]), M, N, K, sw)
        assert kl % 64 == 0 and (S - 1) * kl < K <= S * kl and 1 <= S <= K // 64, (M, N, K, sw)
        assert part == (S * M * N * (2 if sw else 1) * 4 if S > 1 else 0)
