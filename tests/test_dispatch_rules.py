"""Host rules of the kernels' dispatch, compiled on the CPU: static_asserts over the
headers that hold them."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "go-darwinml_amd", "csrc")


def _check(tmp_path, header, asserts):
    src = tmp_path / "rules.cpp"
    src.write_text(f'#include "{header}"\nusing namespace ghip;\n' +
                   "".join(f'static_assert({a}, "");\n' for a in asserts))
    r = subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I", CSRC, str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def test_row_blocks(tmp_path):
    """Blocks of 16 bytes a row touches: 1024 threads hold 16 of them each in fp32 (8 in 16
    bits), so an aligned row of 65536 elements fits, and no row that touches more."""
    _check(tmp_path, "rows_dispatch.h", [
        "row_blocks(65536, 4, 0) == 16384", "row_blocks(65536, 8, 0) == 8192",
        "row_blocks(65536, 4, 3) == 16385", "row_blocks(65533, 4, 0) == 16384", "row_blocks(65534, 4, 0) == 16385",
        "row_blocks(1, 4, 3) == 1", "row_blocks(2, 4, 3) == 2", "row_blocks(4, 4, 1) == 2", "row_blocks(9, 8, 0) == 2"])


def test_staged_tiles(tmp_path):
    """Batches of small ragged products take tiles of their size, not 128 x 128 ones."""
    _check(tmp_path, "gemm_rules.h", [
        "gemm_staged_tile(512, 33, 33, 33, 2) == 64", "gemm_staged_tile(512, 63, 63, 1001, 2) == 64",
        "gemm_staged_tile(4096, 5, 5, 7, 2) == 16", "gemm_staged_tile(65536, 5, 5, 7, 2) == 64",
        "gemm_staged_tile(4096, 17, 17, 1001, 4) == 32", "gemm_staged_tile(4096, 33, 33, 65, 4) == 64",
        "gemm_staged_tile(512, 100, 100, 65, 2) == 128", "gemm_staged_tile(1, 1999, 1999, 1001, 2) == 128",
        "gemm_staged_tile(1, 1000, 776, 1531, 2) == 64", "gemm_staged_tile(1, 256, 10, 512, 4) == 32",
        "gemm_staged_tile(200, 5, 5, 300, 2) == 64"])


def test_half_tiles(tmp_path):
    """The shapes that test the 256 x 128 core run on it: whole tiles in any layout, ragged
    ones with a K-contiguous A alone."""
    whole = [(1, 2048, 4096, 2048), (1, 256, 32768, 2048)]
    ragged = [(1, 2056, 2184, 4104), (1, 4096, 1288, 4160), (2, 2048, 1152, 4232)]
    tiles = "gemm_half_tiles({}, {}, {}, {}, {})".format
    _check(tmp_path, "gemm_rules.h", [tiles(*s, a) for s in whole for a in ("true", "false")] +
           [tiles(*s, "true") for s in ragged] + ["!" + tiles(*s, "false") for s in ragged])
