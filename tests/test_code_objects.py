"""Properties of the compiled kernels that the launches rely on (no GPU needed)."""
import codeobj


def test_gdn_chunk_buffer_offsets_are_bounds_checked():
    """Reads and writes past a chunk's last row count on the bounds check of the buffer descriptor, which is specified
    for the vector offset and not for the scalar one: that one is 0 in every buffer access (of the instance without
    64-bit row offsets)."""
    access = [i for i in codeobj.instructions("gdn_chunk_kernelILb0E") if i.startswith("buffer_")]
    assert access
    bad = [i for i in access if i.replace(",", " ").split()[4] != "0"]
    assert not bad, bad


def test_kernels_use_no_scratch():
    """No kernel keeps registers in scratch memory, but the four-column IQ2_S GEMV over f32 activations, which is faster
    with one spilled register than with the registers it asks for."""
    known = {"qgemv_one_kernelILi22ELi4ELb1EE": 8}
    for name, k in codeobj.kernels().items():
        allowed = max((v for n, v in known.items() if n in name), default=0)
        assert k["private_segment_fixed_size"] <= allowed, (name, k)
