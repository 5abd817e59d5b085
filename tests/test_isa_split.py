"""The checks of test_isa.py on the split-plane kernels' assembly (no GPU needed)."""

import shutil
import os
import tempfile

import pytest

from tests.test_isa import (device_asm, test_no_vmem_reads_a_valu_written_sgpr_within_five_wait_states,  # noqa: F401
                            test_sgpr_based_lds_dma_reads_an_salu_copy)  # noqa: F401


@pytest.fixture(scope="module")
def asm_texts():
    if shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"):
        pytest.skip("hipcc is not available")
    with tempfile.TemporaryDirectory() as d:
        p, out = device_asm("pe_split.hip", d)
        _, err = p.communicate(timeout=600)
        assert p.returncode == 0, err[-2000:]
        return {"pe_split.hip": open(out).read()}
