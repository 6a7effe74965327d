"""The training kernel's chunks: exactly one, one more sample, a partial chunk in several
workgroups, and more chunks than workgroups (each then takes several)."""
import pytest

from test_gpu_mlp import test_gradient_matches_oracle as gradient_matches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 65, 16384, 16385, 40000])
def test_gradient_at_chunk_edges(exe, n):
    gradient_matches(exe, n)
