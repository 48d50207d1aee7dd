"""GPU tests of the tree build at the sizes where its passes change."""
import pytest

import test_gpu_paths as paths

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["scattered", "coincident", "line"])
@pytest.mark.parametrize("n", [1151, 1152, 1153, 1343, 1344, 1345, 1536, 1537, 2047, 2048, 2049, 6143, 6144, 6145])
def test_exported_tree_is_whole_at_the_block_boundaries(ctx, n, layout):
    """A windowed pass takes 192 clusters per block (multiples of it, and one
    to each side), until 1024 are left."""
    paths.test_exported_tree_is_whole_at_the_pass_boundaries(ctx, n, layout)
