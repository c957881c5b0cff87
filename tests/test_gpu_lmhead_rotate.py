"""The planar lm_head of one hidden state rotates a Hadamard-folded weight's
input inside the GEMV (tern_gemv.h): the same logits, bit for bit, as the
plain weight gives on the oracle's rotated input, from one 512-wide rotation
to the longest K, a ragged last round of blocks, with and without signs."""
import numpy as np
import pytest

from oracle import pyoracle as o
from tests.test_gpu_lmhead import PLANAR, run_gemv_ex
from tests.test_oracle_lmhead import random_blocks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", list(PLANAR))
@pytest.mark.parametrize("with_signs", [False, True])
@pytest.mark.parametrize("K,N", [(512, 1), (1536, 17), (2560, 4099), (4096, 300)])
def test_rotated_in_the_gemv(sampler, fmt, K, N, with_signs):
    rng = np.random.default_rng(K + N)
    w = random_blocks(PLANAR[fmt], N, K, rng)
    x = rng.standard_normal((1, K)).astype(np.float32)
    signs = rng.choice(np.float32([-1, 1]), K) if with_signs else None
    y = run_gemv_ex(sampler, PLANAR[fmt], x, w, N, hadamard=True, signs=signs, ldx=K + 1)
    want = run_gemv_ex(sampler, PLANAR[fmt], o.hadamard512(x, signs), w, N)
    assert np.array_equal(y.view(np.uint32), want.view(np.uint32))
    x[0, K // 2] = np.inf   # and an input the integer limbs cannot hold
    assert np.isnan(run_gemv_ex(sampler, PLANAR[fmt], x, w, N, hadamard=True, signs=signs)).all()
