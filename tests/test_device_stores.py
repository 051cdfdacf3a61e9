"""No-GPU check of the code that the compiler makes of a store written with a builtin (csrc/device_utils.hpp)."""
import re
import subprocess

from minml_amd.build import COMMON, CSRC, hipcc

KERNEL = """
#include "device_utils.hpp"
__global__ void four_stores(uint8_t *out, const mlhip::uint4_t *in, uint32_t step)
{
	const __amdgpu_buffer_rsrc_t buffer = mlhip::buffer_of(out);
	mlhip::uint4_t v = in[threadIdx.x];
	for (int i = 0; i < 4; i++)
	{
		mlhip::store_through_l2(buffer, i * 4096 + threadIdx.x * 16, v);
		v += step; /* in the registers that the store still reads */
	}
}
"""


def test_data_registers_of_a_store_through_the_l2_are_left_alone_for_two_wait_states(tmp_path):
    """A store of more than 8 bytes reads its data after it is issued: no vector instruction may write them within two wait states (one per
    instruction, n + 1 of s_nop n)."""
    source, asm = tmp_path / "k.hip", tmp_path / "k.s"
    source.write_text(KERNEL)
    subprocess.run([hipcc()] + COMMON + ["--cuda-device-only", "-S", "-I" + CSRC, str(source), "-o", str(asm)], check=True, capture_output=True)
    code = [l.split(";")[0].strip() for l in asm.read_text().splitlines() if l.startswith("\t") and not l.startswith("\t.")]
    code = [l for l in code if l]
    stores = [i for i, l in enumerate(code) if re.search(r"store_dwordx4.* sc1", l)]
    assert len(stores) == 4
    overwritten = 0
    for i in stores:
        first, last = (int(n) for n in re.search(r"store_dwordx4 (?:v\[\d+:\d+\], )?v\[(\d+):(\d+)\], (?:off|v\d)", code[i]).groups())
        waited = 0
        for line in code[i + 1:i + 6]:
            to = re.match(r"v_\w+ v(?:(\d+)|\[(\d+):(\d+)\])", line)
            if to and int(to.group(1) or to.group(2)) <= last and int(to.group(1) or to.group(3)) >= first:
                overwritten += 1
                assert waited >= 2, (code[i], line)
                break
            nop = re.match(r"s_nop (\d+)", line)
            waited += int(nop.group(1)) + 1 if nop else 1
    assert overwritten >= 2  # the test's own point: the registers are written again soon
