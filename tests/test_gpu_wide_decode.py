"""The stand-alone RMSNorm with its rows in registers: every width at which the registers change."""
import pytest

from mortar_amd import ops, synth
from oracle import mortar_oracle as O
from util import assert_close_bf16, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,d", [(1, 8), (5, 1016), (3, 1024), (1025, 1032), (2, 2056), (1, 4096), (3, 4104), (2, 8192), (2, 8200)])
def test_rmsnorm_widths(dev, M, d):
    x = O.bf16_round(synth.synth_x(M, d, 90) * 3)
    w = O.bf16_round(1.0 + 0.1 * synth.synth_x(1, d, 91)[0])
    assert_close_bf16(to_np(ops.rmsnorm(to_dev(x, dev), to_dev(w, dev))), O.rmsnorm(x, w), "rmsnorm", ulps=2)
