"""hi/lo attention in four key groups (450 tokens and more in about a workgroup a CU) on both sides of its rule, from fp32 rows and, inside the fp32-class block
stack, from the planes the projection leaves.  References and tolerances as in test_gpu_flash_forms and test_gpu_vit_blocks."""
import pytest

from tests import test_gpu_flash_forms as F
from tests import test_gpu_vit_blocks as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("T,nh", [(449, 2), (450, 2), (512, 3), (577, 1), (1024, 16), (1030, 2), (450, 32), (450, 33), (450, 40), (450, 41)])
def test_rows(T, nh, causal):
    F.test_hd64(1, T, nh, causal, True)


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("B,T,D", [(1, 1, 64), (1, 64, 64), (2, 65, 128), (1, 449, 128), (1, 450, 64), (1, 1025, 192), (3, 500, 64), (5, 130, 512), (12, 300, 256)])
def test_planes(B, T, D, causal):
    V.test_stack(B, T, D, 1, 128, 1, causal, 1)
