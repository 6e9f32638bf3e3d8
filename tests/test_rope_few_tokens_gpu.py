"""The rotated q / k / v group of up to 16 tokens (k_nf4_skinny) and just past them: the bits of the
unrotated group followed by the rotation launch, as at many tokens."""

import pytest

from tests.test_rope_fold_gpu import \
    test_folded_rope_equals_the_rotation_of_the_projection as check_fold

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,cos_batch,lora", [
    (1, 1, 1, 16), (1, 1, 1, 0), (1, 16, 1, 32), (16, 1, 16, 16), (2, 8, 2, 16), (3, 5, 1, 64),
    (1, 17, 1, 16)])
def test_rotated_group_equals_group_then_rotation(cuda, B, T, cos_batch, lora):
    check_fold(cuda, B, T, cos_batch, lora)
