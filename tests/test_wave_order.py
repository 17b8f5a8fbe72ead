"""The multi-row product's wavefronts pass activations between their lanes
through LDS without a barrier.  The hardware keeps a wavefront's LDS accesses
in order; the compiler keeps it only where it is told to, so in the assembly
it writes (csrc/qrows.hip, compiled here without a GPU) a wave barrier must
stand between the staging stores and the reads of another lane's values, and
between those reads and the next block's stores."""

import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "llm-inference-cpp_amd")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Every multi-row kernel's assembly, in program order, as the list of its
    LDS accesses and of what orders them."""
    obj = tmp_path_factory.mktemp("asm") / "qrows.s"
    line = subprocess.run(["make", "-C", PKG, "-n", "-B", "_build/qrows.o"], check=True, capture_output=True, text=True)
    cmd = next(ln for ln in line.stdout.splitlines() if "-c -o" in ln).replace("-c -o _build/qrows.o", f"-S --cuda-device-only -o {obj}")
    subprocess.run(cmd, shell=True, check=True, capture_output=True, cwd=PKG)
    out, cur = {}, None
    for ln in obj.read_text().splitlines():
        m = re.match(r"(_ZN\S*qgemm_rows\w*):", ln)
        if m:
            cur = out.setdefault(m.group(1), [])
        elif ln.startswith(".Lfunc_end"):
            cur = None
        elif cur is not None:
            m = re.match(r"\s+(ds_read\w*|ds_write\w*|s_barrier)\b", ln)
            if m:
                cur.append(m.group(1))
            elif "; wave barrier" in ln:
                cur.append("wave_barrier")
    return out


def test_lds_staging_is_ordered(kernels):
    """The operands are the kernels' only 16-byte LDS reads: never after a
    store with nothing between, and two wave barriers for each group of them,
    one on either side (the later one may stand before the next stores)."""
    assert len(kernels) >= 8
    for name, ops in kernels.items():
        stored = reading = False  # a store since the last barrier; within a group of reads
        groups = 0
        for i, op in enumerate(ops):
            if op == "ds_read_b128":
                assert not stored, (name, ops[max(0, i - 12) : i + 1])
                groups += not reading
                reading = True
            else:
                reading = False
                if op in ("wave_barrier", "s_barrier"):
                    stored = False
                elif op.startswith("ds_write"):
                    stored = True
        assert groups > 0 and ops.count("wave_barrier") >= 2 * groups, (name, groups, ops.count("wave_barrier"))
