"""Which layer calls hand their GEMM the codes of the tokens stage by stage, run on the host."""
import os
import subprocess

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "c_host", "staged_rows_check.cpp")
NONE, DECODE, SKINNY, TILE, WHOLE = range(5)   # MG_KERNEL_*


def test_codes_go_stage_by_stage_where_a_step_fits_32_bits(tmp_path):
    """A stage of E4M3 codes is 128 bytes per row, and the GEMMs step from one to the next by 32 bits: on either side of 2^32 bytes, far beyond
    (where the step of a narrower format or of a multiple of 2^32 would wrap, too), and ordinary calls."""
    exe = str(tmp_path / "staged_rows_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", SRC, "-o", exe])
    most = (1 << 25) - 256
    want = {}
    for rows in (256, 512, 4096, 1 << 20, most):
        want.update({(k, t, rows): rows if k == WHOLE or (k == TILE and t) else 0 for k in range(5) for t in (0, 1)})
    for rows in (1 << 25, (1 << 25) + 256, 44739072, 44739328, 1 << 26, (1 << 26) + 256, 1 << 30, (1 << 31) - 256):
        want.update({(k, t, rows): 0 for k in range(5) for t in (0, 1)})
    text = "".join(f"{k} {t} {r}\n" for k, t, r in want)
    out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in out] == list(want.values())
