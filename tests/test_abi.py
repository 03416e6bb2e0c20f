"""CPU checks of the C-ABI library: it loads and exports every declared symbol.

No compute call is made (no GPU here)."""
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def declared_symbols():
    text = (ROOT / "include" / "pdscope_moe.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(pdscope_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_api():
    syms = declared_symbols()
    for name in ("pdscope_route_topk", "pdscope_route_hist", "pdscope_pack", "pdscope_swiglu_grouped",
                 "pdscope_swiglu_decode", "pdscope_merge", "pdscope_stage_expert", "pdscope_stage_merge",
                 "pdscope_last_error"):
        assert name in syms


def test_library_exports_every_declared_symbol():
    from pdscope_amd import _lib
    if not _lib.LIB_PATH.exists():
        pytest.fail("libpdscope_moe.so is not built (run python -m pdscope_amd.build)")
    lib = _lib.load()
    missing = [s for s in declared_symbols() if not hasattr(lib, s)]
    assert not missing, missing
    assert set(_lib.SIGNATURES) == set(declared_symbols())
    assert lib.pdscope_version().decode().startswith("pdscope_moe gfx950")
    assert lib.pdscope_route_workspace_bytes() >= 4
    assert [lib.pdscope_grouped_block_m(r) for r in (8, 32, 80, 128, 256, 600)] == [32, 64, 128, 256, 384, 256]


def test_invalid_arguments_raise_before_any_launch():
    """Argument validation happens on the host and maps to ValueError."""
    from pdscope_amd import _lib
    with pytest.raises(ValueError):
        _lib.call("pdscope_pack", None, 1, 1, 1, None, None, None, None, None, None, None)
    with pytest.raises(ValueError):
        _lib.call("pdscope_route_topk", None, None, None, 1, 2048, 128, 8, 1, None, None, None, None, None, None)
    with pytest.raises(ValueError):
        _lib.call("pdscope_schedule", None, 128, None, 0, 48, None, None)
    msg = _lib.load().pdscope_last_error().decode()
    assert "schedule" in msg
    # the bound decode layer checks its out-pointer, read-back words and
    # binding before touching the device
    import ctypes
    handle = ctypes.c_void_p()
    with pytest.raises(ValueError, match="null binding out-pointer"):
        _lib.call("pdscope_decode_bind", None, None, 2048, 128, 8, 1, 1, None, 768, None, None, None, None, None,
                  None, None, None, None)
    with pytest.raises(ValueError, match="null read-back pointer"):
        _lib.call("pdscope_decode_bind", None, None, 2048, 128, 8, 1, 1, None, 768, None, None, None, None, None,
                  None, None, None, ctypes.byref(handle))
    assert handle.value is None
    with pytest.raises(ValueError, match="null binding"):
        _lib.call("pdscope_decode_run", None, None, None, None, None, None, 1, None)
    _lib.load().pdscope_decode_unbind(None)   # freeing no binding is a no-op


@pytest.mark.parametrize("rows,nsel,I,want", [
    (0, 96, 384, 32), (1, 96, 384, 32), (2, 96, 384, 64), (16, 96, 384, 64), (17, 96, 384, 64), (50, 96, 384, 128),
    (12, 128, 768, 32), (2, 64, 384, 32), (2, 85, 384, 32), (2, 86, 384, 64), (2, 128, 384, 64), (2, 129, 384, 32),
])
def test_row_tile_of_thin_experts(rows, nsel, I, want):
    """Thin experts take the 64-row tile where one tile per expert ends in a
    sparse round; a mean of one row leaves a third of the experts without rows,
    so the launch has fewer tiles than that and keeps the 32-row tile."""
    from pdscope_amd import _lib
    assert _lib.load().pdscope_grouped_block_m_shape(rows, nsel, I) == want


GROUPED_CALLS = {
    # entry -> arguments from (nsel, bm, bm of the down half, H, I, shared I)
    "pdscope_swiglu_grouped": lambda p, n, bm, bd, H, I, Is: [p, p, p, p, n, p, 4, bm, p, H, I, p, p, None],
    "pdscope_swiglu_grouped_gateup": lambda p, n, bm, bd, H, I, Is: [p, p, p, p, n, p, 4, bm, p, H, I, p, None],
    "pdscope_swiglu_grouped_down": lambda p, n, bm, bd, H, I, Is: [p, p, p, n, p, 4, bd, p, H, I, p, None],
    "pdscope_swiglu_grouped_layer": lambda p, n, bm, bd, H, I, Is: [p, p, p, p, n, p, 4, bm, p, 4, bd, p, H, I, p, p, 3,
                                                                    p if Is else None, Is, p, p, None],
}


@pytest.mark.parametrize("entry,n,bm,bd,H,I,Is", [
    # I off the 256-column tiles' multiple, whatever the number of experts makes
    # of the width of the 64-row tiles (300 and 700: sparse last rounds)
    ("pdscope_swiglu_grouped", 8, 64, 64, 1536, 192, 0),
    ("pdscope_swiglu_grouped", 300, 64, 64, 1536, 192, 0),
    ("pdscope_swiglu_grouped", 300, 64, 64, 32768, 192, 0),
    ("pdscope_swiglu_grouped_gateup", 300, 64, 64, 1536, 192, 0),
    ("pdscope_swiglu_grouped_down", 700, 64, 64, 256, 192, 0),
    ("pdscope_swiglu_grouped_down", 8, 32, 32, 512, 192, 0),
    ("pdscope_swiglu_grouped_down", 8, 32, 32, 640, 256, 0),
    # 384 rows (128 columns)
    ("pdscope_swiglu_grouped", 8, 384, 384, 192, 128, 0),
    ("pdscope_swiglu_grouped", 8, 384, 384, 256, 96, 0),
    # a row tile that does not exist
    ("pdscope_swiglu_grouped", 8, 48, 48, 512, 256, 0),
    # the down half of a pair of launches: refused before the gate/up launch
    ("pdscope_swiglu_grouped_layer", 8, 32, 48, 512, 256, 0),
    ("pdscope_swiglu_grouped_layer", 8, 384, 64, 640, 256, 0),
    ("pdscope_swiglu_grouped_layer", 300, 64, 64, 1536, 192, 0),
    # shared experts off the tile
    ("pdscope_swiglu_grouped_layer", 300, 64, 64, 1536, 128, 192),
    ("pdscope_swiglu_grouped_layer", 8, 384, 384, 256, 128, 96),
    ("pdscope_swiglu_grouped_layer", 8, 384, 256, 256, 128, 192),
])
def test_grouped_shapes_are_refused_before_any_launch(entry, n, bm, bd, H, I, Is):
    """A shape outside the row tile's columns is an invalid argument in every
    grouped entry point (a launch would be a HIP error here, without a device)."""
    import ctypes

    from pdscope_amd import _lib
    memory = ctypes.create_string_buffer(64)   # non-null; refused before it is read
    with pytest.raises(ValueError, match="grouped"):
        _lib.call(entry, *GROUPED_CALLS[entry](ctypes.addressof(memory), n, bm, bd, H, I, Is))


def test_wide_stores_in_asm_carry_their_wait_states():
    """gfx950 reads the data registers of a vector store of more than 8 bytes
    after the store has issued: a VALU write to them needs two wait states in
    between.  The compiler keeps them for stores of its own and cannot see one
    inside an asm string, so the string has to end with them."""
    found = 0
    for path in sorted((ROOT / "pdscope_amd" / "csrc").iterdir()):
        for text in re.findall(r'asm\s+(?:volatile)?\s*\(\s*((?:"[^"]*"\s*)+)', path.read_text()):
            if re.search(r"_store_(dwordx[34]|b96|b128)", text):
                found += 1
                assert re.search(r"_store_\w+[^;]*\\n\\ts_nop 1\"\s*$", text), (path.name, text)
    assert found >= 1
