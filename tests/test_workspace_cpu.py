"""Bytes of a layer's workspace: what the largest layers' images in units add, and where they end."""


def test_images_in_units_are_bounded():
    from bsipytorch_amd import _lib

    bytes_of = _lib.lib.bsi_hip_linear_workspace_bytes
    plain = lambda Q, d: Q * (7 * ((d + 63) // 64) * 8 + (d + 255) // 256 * (256 + 8))  # noqa: E731  planes, image, shifts and scales
    for Q, d, units in ((511, 4096, False), (512, 4096, True), (512, 16384, True), (512, 16385, False), (1 << 20, 1024, True),
                        ((1 << 20) + 1, 1024, False), (1 << 16, 16384, True), ((1 << 16) + 1, 16384, False)):
        extra = bytes_of(Q, d, 7) - plain(Q, d)
        image = Q * ((d + 255) // 256) * 256
        assert (extra >= 2 * image) == units and extra < (2.2 * image if units else 4096), (Q, d, extra)
