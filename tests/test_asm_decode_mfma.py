"""M0 in the compiled matrix-core decode (CPU only): its LDS copies are inline assembly that
sets M0, a reserved register, so M0 may be written by those sequences alone and read by
nothing else."""
import os
import re
import subprocess

import pytest

import test_asm_invariants as inv


def test_m0_belongs_to_the_lds_copies(tmp_path):
    b = inv._build_module()
    if not os.path.exists(b.HIPCC):
        pytest.skip("hipcc is not installed")
    out = tmp_path / "decode_mfma.s"
    flags = [f for f in b.CFLAGS if f != "-fPIC"]
    r = subprocess.run([b.HIPCC, *flags, "-I", b.CSRC, "--cuda-device-only", "-S",
                        os.path.join(b.CSRC, "decode_mfma.hip"), "-o", str(out)], capture_output=True, text=True,
                       timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    asm = [l.split(";")[0].strip() for l in out.read_text().splitlines()]
    asm = [l for l in asm if l and not l.startswith(".")]
    uses = [i for i, l in enumerate(asm) if re.search(r"\bm0\b", l)]
    assert uses
    for i in uses:
        assert re.match(r"s_mov_b32 m0, (s\d+|vcc_lo|vcc_hi|ttmp\d+)$", asm[i]), asm[i]
        assert asm[i + 1] == "s_nop 0", asm[i + 1]
        assert asm[i + 2].startswith("global_load_lds_dword"), asm[i + 2]
    assert len(uses) == len([l for l in asm if l.startswith("global_load_lds")])
    inv.test_no_instruction_reads_m0_implicitly(asm)
