"""The register-resident builders at the edges of their ranges, against the oracle: rows that end inside a quad, a chunk
or a tile, one row more or less than a tile of 16, the ends of what is kept in registers (8 and 16 chunks), magnitudes
around the limits of the float32 route, and the build without planes."""
import numpy as np
import pytest
import torch

from test_gpu_parity import dev, hip, host_u64, ops, st  # noqa: F401  (fixtures and helpers)

pytestmark = pytest.mark.gpu

LARGEST = {"small": 0.02, "held": 255.99, "reread": 256.0, "float": 65535.9, "wide": 65536.0, "huge": 3.0e9}


def _rows(rows, d, kind, dtype, seed):
    rng = np.random.default_rng(seed)
    x = torch.from_numpy((rng.standard_normal((rows, d)) * (0.02 if kind == "small" else 3.0)).astype(np.float32))
    x[::2, d // 2] = LARGEST[kind]
    x[0, 0] = -0.5 / 100.0  # a tie
    if kind == "huge" and d > 2:
        x[-1, 0], x[-1, 1], x[-1, 2] = float("nan"), float("inf"), -0.0
    return x.to(dtype)


@pytest.mark.parametrize("kind", sorted(LARGEST))
@pytest.mark.parametrize("rows,d,dtype", [(1, 1, torch.float32), (15, 64, torch.bfloat16), (16, 255, torch.float16),
                                          (17, 258, torch.float32), (33, 2048, torch.float32), (18, 2304, torch.bfloat16),
                                          (16, 4096, torch.float16), (31, 4100, torch.float32)])
def test_key_build_in_one_launch(hip, ops, oracle, rows, d, dtype, kind):
    x = _rows(rows, d, kind, dtype, rows + d)
    want = oracle.build_keys(x.to(torch.float32).numpy())
    keys, nbytes, *_ = ops.build_bsi_keys_cuda(x.cuda(), 2, 0.5)
    W = (d + 63) // 64
    assert nbytes == rows * 6 * W * 8
    np.testing.assert_array_equal(host_u64(ops.canonical_key_planes(keys)), want["words"])
    np.testing.assert_array_equal(keys.slice_weights[:, 0].cpu().numpy(), want["scales"])
    np.testing.assert_array_equal(keys.slice_weights[:, 5].cpu().numpy(), -32 * want["scales"])
    np.testing.assert_array_equal(np.exp2(keys.shifts.cpu().numpy().astype(np.float32)), want["scales"])
    planes, tiled, image = dev(want["words"]), torch.zeros_like(keys.words), torch.zeros_like(keys.ints8)
    hip.check(hip.lib.bsi_hip_tile_key_planes(planes.data_ptr(), rows, 6, W, tiled.data_ptr(), st()), "tile")
    hip.check(hip.lib.bsi_hip_planes_to_int8(planes.data_ptr(), rows, 6, W, image.data_ptr(), st()), "image")
    assert torch.equal(keys.words, tiled) and torch.equal(keys.ints8, image)


@pytest.mark.parametrize("kind", sorted(LARGEST))
@pytest.mark.parametrize("rows,d,dtype", [(3, 254, torch.float32), (5, 510, torch.float16), (9, 2048, torch.bfloat16),
                                          (2, 70, torch.bfloat16), (7, 1601, torch.float32), (4, 4164, torch.float16)])
def test_query_build_with_and_without_planes(hip, oracle, rows, d, dtype, kind):
    x = _rows(rows, d, kind, dtype, 3 * rows + d)
    W, chunks = (d + 63) // 64, (d + 255) // 256
    chunk = W % 4 == 0
    ints, shifts, scales = oracle.quantize_fixed(x.to(torch.float32).numpy(), 2, 7, chunk)
    want = oracle.pack(ints, 7)
    xd, code = x.cuda(), {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype]
    images = []
    for planes in (True, False):
        words = torch.zeros((rows, 7, W), dtype=torch.int64, device="cuda")
        sh = torch.full(shifts.shape, -1, dtype=torch.int32, device="cuda")
        sc = torch.full(scales.shape, -1.0, device="cuda")
        image = torch.full((rows, chunks * 256), 77, dtype=torch.int8, device="cuda")
        hip.check(hip.lib.bsi_hip_build_fixed(xd.data_ptr(), code, rows, d, 2, 7, int(chunk), 0.0, words.data_ptr() if planes else None,
                                              sh.data_ptr(), sc.data_ptr(), image.data_ptr(), st()), "build")
        np.testing.assert_array_equal(sh.cpu().numpy(), shifts)
        np.testing.assert_array_equal(sc.cpu().numpy(), scales)
        if planes:
            np.testing.assert_array_equal(host_u64(words), want)
        images.append(image)
    from_planes = torch.zeros_like(images[0])
    planes_dev = dev(want)
    hip.check(hip.lib.bsi_hip_planes_to_int8(planes_dev.data_ptr(), rows, 7, W, from_planes.data_ptr(), st()), "image")
    assert torch.equal(images[0], from_planes) and torch.equal(images[1], from_planes)


@pytest.mark.parametrize("bits", [2, 6, 8])
@pytest.mark.parametrize("largest", [1.2749, 1.275, 0.3149])
@pytest.mark.parametrize("rows,d,dtype", [(17, 2049, torch.float32), (16, 2304, torch.float16), (3, 4352, torch.bfloat16),
                                          (33, 8192, torch.float32), (5, 8450, torch.float16)])
def test_key_build_from_bytes(hip, oracle, rows, d, dtype, largest, bits):
    """Rows at the end of what is held as bytes, and past it; widths around the groups that are held."""
    rng = np.random.default_rng(rows + d + bits)
    x = torch.from_numpy(rng.uniform(-0.99 * largest, 0.99 * largest, (rows, d)).astype(np.float32))
    x[:, d - 1], x[::2, d // 2] = 0.005, -largest
    x = x.to(dtype)
    ints, shifts, scales = oracle.quantize_fixed(x.to(torch.float32).numpy(), 2, bits, False)
    planes, W, chunks = dev(oracle.pack(ints, bits)), (d + 63) // 64, (d + 255) // 256
    want = [torch.zeros(((rows + 15) // 16, chunks, bits, 64), dtype=torch.int64, device="cuda"),
            torch.zeros((rows, chunks * 256), dtype=torch.int8, device="cuda")]
    hip.check(hip.lib.bsi_hip_tile_key_planes(planes.data_ptr(), rows, bits, W, want[0].data_ptr(), st()), "tile")
    hip.check(hip.lib.bsi_hip_planes_to_int8(planes.data_ptr(), rows, bits, W, want[1].data_ptr(), st()), "image")
    tiled, image = torch.full_like(want[0], 77), torch.full_like(want[1], 77)
    sh, w = torch.full((rows,), -1, dtype=torch.int32, device="cuda"), torch.zeros((rows, bits), device="cuda")
    xd, code = x.cuda(), {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype]
    hip.check(hip.lib.bsi_hip_build_fixed_keys(xd.data_ptr(), code, rows, d, 2, bits, tiled.data_ptr(), image.data_ptr(),
                                               sh.data_ptr(), w.data_ptr(), st()), "keys")
    np.testing.assert_array_equal(sh.cpu().numpy(), shifts.reshape(-1))
    np.testing.assert_array_equal(w[:, 0].cpu().numpy(), scales.reshape(-1))
    assert torch.equal(tiled, want[0]) and torch.equal(image, want[1])
