"""What a layer's call refuses, whichever kernel it would take: nothing is launched here."""
import pytest

AT = 1 << 20  # an address that is looked at, and never read


def call(warm, warm_bytes, Q, R_total=None, B=AT, R=16384, d=4096):
    from bsipytorch_amd import _lib

    L = _lib.lib
    rc = L.bsi_hip_linear_out(AT, _lib.DTYPE_F32, Q, d, 2, 7, 0, AT, 1 << 40, B, _lib.LAYOUT_INT8, AT, 6, R, 1e-4,
                              R if R_total is None else R_total, None, AT, _lib.DTYPE_F32, _lib.CORE_AUTO, warm, warm_bytes, None)
    return rc, L.bsi_hip_last_error()


@pytest.mark.parametrize("Q", [64, 512, 4096])  # 4096: a large layer
def test_null_warm_region_with_a_length(Q):
    rc, message = call(None, 128, Q)
    assert rc == 1 and b"null warm-up region" in message


@pytest.mark.parametrize("what, said", [({"R_total": 16383}, b"R_total must be >= R"), ({"B": None}, b"null pointer"),
                                        ({"B": AT + 8}, b"16-byte aligned"), ({"Q": 65535 * 32 + 1, "d": 256}, b"split the batch"),
                                        ({"R": (1 << 25) + 1}, b"2^25 key rows")])
def test_limits_of_a_large_layer(what, said):
    from bsipytorch_amd import _lib

    _lib.check(_lib.lib.bsi_hip_set_option(_lib.OPT_I8_TILE, 256), "tile")  # any layer of 512 rows is a large one
    try:
        rc, message = call(None, 0, **{"Q": 4096, **what})
    finally:
        _lib.check(_lib.lib.bsi_hip_set_option(_lib.OPT_I8_TILE, 0), "tile")
    assert rc == 1 and said in message
