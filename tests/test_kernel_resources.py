"""What the compiler made of the kernels, from the metadata in the built library."""

import msgpack

import anetransformers_amd as mia


def _kernels():
    """The code objects' kernel descriptions (AMDGPU metadata notes, a msgpack map each)."""
    data = open(mia.LIB_PATH, "rb").read()
    at = data.find(b"amdhsa.kernels")
    while at >= 0:
        # the note's map starts one string header (1 or 2 bytes) and a map header before this key
        for start in (at - 2, at - 3):
            try:
                u = msgpack.Unpacker(raw=False, strict_map_key=False, max_buffer_size=len(data))
                u.feed(data[start:start + (4 << 20)])
                m = u.unpack()
            except Exception:
                continue
            if isinstance(m, dict) and "amdhsa.kernels" in m:
                yield from m["amdhsa.kernels"]
                break
        at = data.find(b"amdhsa.kernels", at + 1)


def test_the_attention_and_gemm_loops_spill_nothing():
    # A vector register spilled in their tile loops is reloaded behind the loop's
    # own loads in flight: every step then waits for all of them.
    hot = {k[".name"]: k for k in _kernels() if "flash_kernel" in k[".name"] or "gemm_kernel" in k[".name"]}
    assert sum("flash_kernel" in n for n in hot) >= 6 and sum("gemm_kernel" in n for n in hot) >= 20
    spilled = {n: k[".vgpr_spill_count"] for n, k in hot.items() if k[".vgpr_spill_count"]}
    assert not spilled
