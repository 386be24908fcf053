"""``eos.source_buffer``: the rows outside the species are zero on both sides of
the size from which only they are filled, and the buffer is the state's."""

import pytest

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("nodes", [0, 1, (1 << 17) - 1, 1 << 17])
def test_zero_rows(dim, nodes):
    from mirgecom_amd.eos import source_buffer
    q = torch.ones((9 + dim, nodes, 1), dtype=torch.float64)
    out = source_buffer(q, dim)
    assert out.shape == q.shape and out.dtype == q.dtype and out.is_contiguous()
    assert not out[:2 + dim].any() and out.data_ptr() != q.data_ptr() or nodes == 0
