"""Properties of the compiled kernels that the launches rely on (no GPU needed)."""
import pytest

import codeobj


@pytest.mark.parametrize("kernel", ["gdn_chunk_prep_kernel", "gdn_chunk_kernel"])
def test_gdn_chunk_buffer_offsets_are_bounds_checked(kernel):
    """Reads and writes past a chunk's last row count on the bounds check of the buffer descriptor, which is specified
    for the vector offset and not for the scalar one: that one is 0 in every buffer access."""
    bad = [i for i in codeobj.instructions(kernel)
           if i.startswith("buffer_") and i.replace(",", " ").split()[4] != "0"]
    assert not bad, bad
