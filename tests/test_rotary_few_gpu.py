"""Head norms and rotation in steps of few tokens: heads on both sides of a wave's 64, 128 and 256 channels, norms over a projection on
both sides of the 512 columns a wave asks for at once, angles beyond a wave's, and a last work-group that is not full."""
import pytest

from test_rotary_rows_gpu import test_rotation_of_many_tokens as rotation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,rot,norm,neighbours,same", [
    (1, 1, 64, 64, 64, "head", False, False), (2, 1, 65, 63, 64, "whole", True, False), (3, 1, 63, 65, 2, None, False, False),
    (4, 2, 128, 128, 128, "whole", False, True), (3, 3, 129, 1, 128, "whole", True, False), (1, 1, 256, 255, 256, "head", False, False),
    (2, 2, 256, 256, 0, "whole", False, False), (9, 3, 57, 256, 56, "whole", False, False)])
def test_rotation_of_few_tokens(dtype, heads, kv_heads, dim, vdim, rot, norm, neighbours, same):
    rotation(dtype, 5, heads, kv_heads, dim, vdim, rot, norm, neighbours, same)
