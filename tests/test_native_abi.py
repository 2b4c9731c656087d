"""The HIP library loads (no GPU needed) and exports every entry point that
include/m2r.h declares; the Python binding knows each of them."""
import ctypes
import re
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def declared_symbols():
    text = (ROOT / "include" / "m2r.h").read_text()
    return sorted(set(re.findall(r"^\s*(?:const\s+)?\w+\*?\s+(m2r_\w+)\s*\(", text, re.M)))


def test_header_declares_entry_points():
    names = declared_symbols()
    assert "m2r_state_step_ridge" in names and "m2r_fp4_decode_g16" in names
    assert len(names) >= 13


def test_library_exports_every_declared_symbol():
    from mamba2_recall import _native
    lib = ctypes.CDLL(str(_native.LIB_PATH))
    missing = [n for n in declared_symbols() if not hasattr(lib, n)]
    assert not missing, missing


def test_binding_covers_header():
    from mamba2_recall import _native
    assert set(declared_symbols()) <= set(_native._SIGNATURES)


def test_error_reporting_without_device():
    """Rejected geometry returns nonzero with a message, before any launch."""
    from mamba2_recall import _native
    lib = _native.lib()
    rc = lib.m2r_fp4_decode_g16(None, None, None, None, 0, 16, None, None)
    assert rc != 0
    assert b"non-positive" in lib.m2r_last_error()


def test_step_shape_hook_accepts_documented_shapes_only():
    """m2r_set_step_shape takes the documented shapes, including (4, 0) (two
    waves per head slot) and (4, -4) (four), rejects the others with a message, and (0, 0)
    restores the automatic choice (no launch, no device)."""
    from mamba2_recall import _native
    lib = _native.lib()
    try:
        for shape in [(1, 1), (4, 1), (4, 2), (4, 4), (8, 2), (4, 0), (4, -2), (4, -4), (0, 0)]:
            assert lib.m2r_set_step_shape(*shape) == 0, shape
        for shape in [(8, 0), (2, 2), (8, 4), (1, 0), (16, 1), (4, -3), (8, -4), (4, -1)]:
            assert lib.m2r_set_step_shape(*shape) != 0, shape
            assert b"step shape" in lib.m2r_last_error()
    finally:
        lib.m2r_set_step_shape(0, 0)


LEGACY, TIER, RIDGE, DENSE3 = range(4)


def test_scan_lanes_leave_no_wave_without_rows():
    """The multi-token scan's lanes per row: 8, 4, 2 and 1 (4 for wide rows)
    with the slots of the 128-head model, and 0, the one-lane kernels, where a
    workgroup's four waves would not all have rows (3 or 6 heads per group
    with blocks of one or two waves), where a last round of waves is mostly
    empty, for few tokens and for ragged heads."""
    from mamba2_recall import _native
    lanes = _native.lib().m2r_scan_lanes
    model = (128, 64, 8)
    for codec, n8, n4 in ((RIDGE, 24, 44), (TIER, 32, 32)):
        assert [lanes(codec, n8, n4, b, 64, *model) for b in (1, 3, 4, 6, 7, 8, 12, 13, 16, 32, 64)] == [
            8, 8, 4, 4, 2, 2, 4, 1, 1, 1, 1]
        for batch, H, P, G in ((250, 8, 64, 8), (250, 8, 16, 8), (112, 8, 64, 8), (222, 9, 48, 3), (333, 6, 64, 3),
                               (139, 9, 80, 3), (1, 65540, 48, 4)):
            assert lanes(codec, n8, n4, batch, 64, H, P, G) == 0, (codec, batch, H, P, G)
        assert lanes(codec, n8, n4, 300, 64, 4, 64, 1) == 4 and lanes(codec, n8, n4, 450, 64, 4, 64, 1) == 1
        assert lanes(codec, n8, n4, 40, 64, 6, 64, 3) == 8 and lanes(codec, n8, n4, 1, 64, 8, 16, 8) == 8
    assert [lanes(TIER, 8, 80, b, 64, *model) for b in (1, 8, 16, 64)] == [8, 2, 4, 4]
    assert [lanes(TIER, 32, 32, b, 64, *model) for b in (17, 20, 24, 25)] == [0, 0, 0, 1]
    assert [lanes(TIER, 32, 32, b, 24, *model) for b in (16, 28, 32, 33)] == [1, 0, 1, 1]
    assert lanes(TIER, 44, 8, 20, 24, *model) == 1
    assert [lanes(RIDGE, 8, 76, 345, L, 16, 16, 8) for L in (63, 64, 105)] == [0, 4, 4]
    assert [lanes(RIDGE, 24, 44, b, 32, 8, 64, 8) for b in (16, 100, 138, 175)] == [8, 0, 0, 0]
    assert lanes(RIDGE, 24, 44, 138, 64, 8, 64, 8) == 4 and lanes(RIDGE, 8, 76, 122, 64, 9, 64, 3) == 4
    assert [lanes(DENSE3, 0, 0, b, 16, *model) for b in (1, 4, 8, 64)] == [8, 4, 2, 4]
    assert [lanes(LEGACY, 16, 64, 1, L, *model) for L in (1, 2, 7, 8, 512)] == [0, 0, 0, 8, 8]
    assert lanes(TIER, 32, 32, 1, 64, 8, 12, 8) == 0 and lanes(RIDGE, 24, 44, 1, 64, 9, 64, 2) == 0


def test_ridge_workspace_is_bounded():
    """1 KiB per batch row, token and group up to 256 MiB, then the records of
    a piece of the tokens, at least 64: no more than about the packed state of
    8 heads of 128 rows per group."""
    from mamba2_recall import _native
    need = _native.lib().m2r_ridge_records_bytes
    assert need(1, 512, 8) == 512 * 8 << 10 and need(3, 19, 8) == 3 * 19 * 8 << 10
    assert need(64, 512, 8) == need(64, 100000, 8) == 256 << 20
    assert need(60, 100000, 8) == 60 * 512 * 8 << 10
    assert need(4096, 64, 8) == need(4096, 1000, 8) == 4096 * 64 * 8 << 10
    assert need(0, 5, 8) == 0
