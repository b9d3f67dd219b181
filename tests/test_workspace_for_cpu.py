"""Bytes of a layer's workspace on given keys: the images of a large layer only where its kernel runs."""
import pytest


@pytest.mark.parametrize("Q, d, R, layout, core, images", [
    (512, 2048, 8192, "INT8", "AUTO", False), (4096, 4096, 16384, "INT8", "AUTO", True), (4096, 4096, 16384, "INT8_TILED", "AUTO", False),
    (4096, 4096, 16384, "INT8", "MFMA", False), (4096, 4096, 16384, "TILED16", "AUTO", False), (4096, 4096, 512, "INT8", "AUTO", False),
    (2048, 8192, 8192, "INT8", "AUTO", True), (511, 4096, 16384, "INT8", "AUTO", False), (4096, 4096, 0, "INT8", "AUTO", False)])
def test_images_only_where_they_are_read(Q, d, R, layout, core, images):
    from bsipytorch_amd import _lib

    layout, core = getattr(_lib, "LAYOUT_" + layout), getattr(_lib, "CORE_" + core)
    got = _lib.lib.bsi_hip_linear_workspace_bytes_for(Q, d, 7, layout, 6, R, core)
    most = _lib.lib.bsi_hip_linear_workspace_bytes(Q, d, 7)
    plain = Q * (7 * ((d + 63) // 64) * 8 + (d + 255) // 256 * (256 + 8))  # planes, image, shifts and scales
    assert got == most if images else plain <= got < plain + 4096


def test_the_tile_that_is_asked_for_counts():
    from bsipytorch_amd import _lib

    def bytes_of():
        return _lib.lib.bsi_hip_linear_workspace_bytes_for(512, 2048, 7, _lib.LAYOUT_INT8, 6, 8192, _lib.CORE_AUTO)

    least = bytes_of()
    try:
        _lib.check(_lib.lib.bsi_hip_set_option(_lib.OPT_I8_TILE, 256), "tile")
        assert bytes_of() == _lib.lib.bsi_hip_linear_workspace_bytes(512, 2048, 7) > least
    finally:
        _lib.check(_lib.lib.bsi_hip_set_option(_lib.OPT_I8_TILE, 0), "tile")
    assert bytes_of() == least
