"""No-GPU checks of the rules that choose a kernel for a product (csrc/gemm_tiles.hpp, csrc/gemm_direct.hpp): compiled for the host alone and asked
for the sides of their lines that measurements stand beside."""
import os
import subprocess

import pytest

from minml_amd.build import CSRC, hipcc

HERE = os.path.dirname(os.path.abspath(__file__))
SIZE = {"float16": 2, "float32": 4, "int8": 1}


@pytest.fixture(scope="module")
def decide(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("routes") / "product_routes")
    subprocess.run([hipcc(), "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-O0", "-I" + CSRC, "-x", "hip", os.path.join(HERE, "product_routes.cpp"),
                    "-o", exe], check=True, capture_output=True)

    def ask(kind, dtype, matrices, rows, columns, K):
        line = "%s %d %d %d %d %d\n" % (kind, SIZE[dtype], matrices, rows, columns, K * SIZE[dtype])
        return subprocess.run([exe], input=line, check=True, capture_output=True, text=True).stdout.split()

    return ask


@pytest.mark.parametrize("dtype,matrices,rows,columns,K,by_rows", [
    # the 36 products between two transforms, which divide the images in the same way
    ("float16", 36, 192, 256, 256, True), ("float16", 36, 1024, 64, 64, True), ("float32", 36, 512, 128, 128, True), ("float16", 36, 640, 384, 384, True),
    ("float16", 36, 191, 256, 256, False), ("float16", 36, 2304, 384, 384, False),
    # any other batch has no such neighbours, and more columns than rows make every XCD fetch more of B than it saves of A and C
    ("float16", 16, 512, 2048, 64, False), ("float16", 64, 192, 1024, 64, False), ("float16", 64, 192, 1024, 128, False), ("float16", 8, 1024, 1024, 256, False),
    ("float16", 36, 192, 1024, 192, False), ("float32", 16, 1024, 256, 64, False)])
def test_order_of_batched_products(decide, dtype, matrices, rows, columns, K, by_rows):
    assert decide("plain", dtype, matrices, rows, columns, K)[1] == str(int(by_rows))


def test_direct_kernel_takes_more_tiles_only_in_the_order_by_rows(decide):
    assert decide("plain", "float16", 36, 2048, 64, 64)[2] == "1"
    assert decide("plain", "float16", 16, 512, 2048, 64)[2] == "0"
    assert decide("plain", "float16", 64, 192, 256, 64)[2] == "1"


@pytest.mark.parametrize("kind,matrices,rows,columns,K,tile", [
    ("plain", 64, 64, 1024, 192, "64x64"), ("plain", 48, 22, 2000, 192, "64x64"), ("plain", 32, 190, 2048, 128, "64x64"), ("dense", 1, 40, 60000, 192, "64x64"),
    ("dense", 64, 40, 1024, 512, "64x64"), ("plain", 64, 70, 1024, 192, "128x64"), ("plain", 64, 70, 1024, 256, "128x128"), ("plain", 64, 300, 384, 384, "128x192"),
    ("plain", 36, 2304, 256, 256, "128x128"), ("plain", 36, 500, 256, 256, "128x64"), ("dense", 1, 14400, 256, 256, "128x128"), ("dense", 1, 57600, 192, 192, "128x64")])
def test_tiles_of_128_rows_where_the_matrix_fills_them(decide, kind, matrices, rows, columns, K, tile):
    taken, _, _, chosen = decide(kind, "float16", matrices, rows, columns, K)
    assert (taken, chosen) == ("1", tile)


@pytest.mark.parametrize("dtype,matrices,rows,columns,K,taken", [
    # fp32, long K rows: the small tiles of conv_tiles.hpp up to two 32x32 tiles per compute unit
    ("float32", 36, 16, 256, 256, False), ("float32", 8, 64, 512, 2048, False), ("float32", 8, 128, 512, 4096, False), ("float32", 9, 776, 56, 512, False),
    ("float32", 36, 64, 256, 256, True), ("float32", 8, 256, 512, 1024, True), ("float32", 36, 4096, 256, 256, True),
    # up to one per unit below that
    ("float32", 8, 512, 64, 160, False), ("float32", 8, 600, 64, 160, True), ("float32", 8, 512, 64, 192, False), ("float32", 8, 128, 256, 224, False), ("float32", 8, 150, 256, 224, True),
    ("float32", 8, 512, 64, 144, True), ("float32", 8, 512, 64, 128, True),
    # fp32, 128-byte K rows (32 planes): to 50 MB of A and C, 63 with one column tile
    ("float32", 36, 4096, 64, 32, True), ("float32", 36, 8000, 64, 32, False),
    ("float32", 36, 1616, 128, 32, True), ("float32", 36, 4096, 128, 32, False), ("float32", 36, 1616, 256, 32, False), ("float32", 36, 1024, 256, 32, True),
    # wide columns that fill the streaming kernel's slices: 768-byte fp16 rows of a network's batch to 168 or 105 MB, 256-byte fp32 rows to 268 MB; other widths further
    ("float16", 64, 1024, 1024, 384, False), ("float16", 64, 800, 1024, 384, False), ("float16", 64, 450, 1024, 384, True), ("float16", 36, 2400, 512, 384, True), ("float16", 36, 4300, 384, 384, True), ("float16", 36, 3300, 640, 384, True),
    ("float16", 36, 4300, 256, 384, False), ("float32", 64, 1024, 1024, 64, False), ("float32", 36, 16384, 64, 64, True), ("float32", 36, 9000, 192, 64, True),
    # fp16 rows of one to three pieces and a half: to 252 MB, with one or three column tiles at any size; other lengths at any size
    ("float16", 36, 7891, 256, 96, True), ("float16", 36, 11837, 256, 96, False), ("float16", 36, 10016, 256, 160, False), ("float16", 64, 11505, 256, 160, False),
    ("float16", 36, 8491, 512, 224, False), ("float16", 36, 43402, 64, 160, True), ("float16", 36, 17871, 384, 160, True), ("float16", 36, 21701, 256, 192, True),
    ("float16", 36, 17871, 256, 288, True), ("float32", 16, 20000, 256, 80, True),
    # few tiles: the direct kernel further in batches that are not between transforms
    ("float16", 36, 128, 256, 256, True), ("float16", 8, 400, 400, 256, False), ("float16", 24, 512, 256, 256, True), ("float16", 36, 64, 384, 384, True),
    ("float16", 16, 192, 256, 384, False), ("float16", 64, 128, 128, 384, True),
    # and the streaming kernel earlier, whose lead is larger with the operands from memory
    ("float16", 36, 2300, 256, 128, True), ("float16", 16, 2500, 256, 128, True), ("float16", 16, 3417, 256, 128, False), ("float16", 36, 2400, 256, 256, True),
    ("float16", 16, 4028, 256, 256, True), ("float16", 16, 5615, 256, 256, False), ("float16", 64, 442, 1024, 256, False), ("float16", 16, 3208, 512, 384, True),
    ("float16", 64, 1400, 512, 384, False), ("float16", 16, 2041, 1024, 384, False), ("float16", 16, 8138, 384, 384, True), ("float16", 16, 10172, 384, 384, False)])
def test_plain_batches_on_the_tiles(decide, dtype, matrices, rows, columns, K, taken):
    assert decide("plain", dtype, matrices, rows, columns, K)[0] == str(int(taken))


@pytest.mark.parametrize("dtype,matrices,rows,columns,K,taken", [
    # few columns: half of a tile would be padding
    ("float16", 1, 28800, 32, 256, False), ("float16", 1, 57600, 32, 256, True), ("float16", 1, 114119, 32, 192, False), ("float16", 1, 57600, 40, 192, False),
    ("float16", 1, 114119, 64, 192, True), ("float16", 1, 28800, 32, 96, True), ("float16", 1, 28800, 40, 256, True),
    # 1024-byte K rows: from where the 32x32 tiles of conv_tiles.hpp end, two per compute unit
    ("float16", 1, 2048, 256, 512, False), ("float16", 1, 2300, 256, 512, True), ("float16", 8, 228, 256, 512, False), ("float16", 8, 300, 256, 512, True),
    ("float16", 1, 2048, 256, 480, True),
    # longer ones: to four 64x64 tiles and 8192 bytes of K rows per unit
    ("float16", 8, 912, 256, 576, True), ("float16", 8, 1824, 256, 768, True), ("float16", 8, 1824, 256, 1024, True), ("float16", 8, 2100, 256, 1024, False),
    ("float16", 8, 1200, 256, 1536, True), ("float16", 8, 1824, 256, 1536, False), ("float16", 8, 912, 256, 2048, True), ("float16", 8, 1200, 256, 2048, False),
    ("float16", 8, 912, 256, 2080, False), ("float16", 8, 228, 256, 1024, False), ("float16", 8, 3072, 128, 1024, True), ("float16", 8, 3584, 128, 1024, False), ("float16", 8, 3584, 128, 768, True), ("float16", 1, 28672, 128, 1024, True),
    # short K rows from memory: the streaming kernel from 34, 46 and 67 MB of A and C on, with at most 128 columns later
    ("float16", 1, 41666, 256, 128, True), ("float16", 1, 52083, 256, 128, False), ("float16", 1, 128906, 128, 128, False), ("float16", 16, 1007, 2048, 128, False),
    ("float16", 1, 39062, 256, 256, True), ("float16", 1, 50781, 256, 256, False), ("float16", 4, 8140, 512, 256, False), ("float16", 1, 169270, 128, 256, True),
    ("float16", 1, 50000, 256, 384, True), ("float16", 1, 74218, 256, 384, False), ("float16", 1, 126953, 128, 384, True)])
def test_dense_layers_on_the_tiles(decide, dtype, matrices, rows, columns, K, taken):
    assert decide("dense", dtype, matrices, rows, columns, K)[0] == str(int(taken))


@pytest.mark.parametrize("kind,matrices,rows,columns,K,taken", [
    # fp32 experts of 256 and 512-byte K rows: the 32x32 tiles of conv_tiles.hpp up to two per compute unit; a single layer has no such kernel
    ("experts", 8, 64, 64, 128, False), ("experts", 8, 800, 64, 128, False), ("experts", 8, 1100, 64, 128, True), ("experts", 36, 85, 64, 64, False),
    ("experts", 8, 200, 256, 64, False), ("experts", 1, 225, 128, 128, False), ("experts", 4, 818, 256, 128, True), ("dense", 1, 225, 128, 128, True),
    ("experts", 4, 700, 256, 96, True), ("experts", 8, 640, 64, 192, False)])
def test_fp32_experts_on_the_tiles(decide, kind, matrices, rows, columns, K, taken):
    assert decide(kind, "float32", matrices, rows, columns, K)[0] == str(int(taken))


@pytest.mark.parametrize("rows,columns,K,taken", [
    # with a residual, which the streaming kernel does not hide: to 101 MB
    (74218, 256, 128, True), (80000, 256, 128, False), (61848, 256, 256, True), (53011, 256, 384, True), (27797, 384, 384, True), (169270, 128, 128, False), (126953, 128, 256, True)])
def test_dense_layers_with_residual_on_the_tiles(decide, rows, columns, K, taken):
    assert decide("residual", "float16", 1, rows, columns, K)[0] == str(int(taken))


@pytest.mark.parametrize("dtype,channels,kernel,pixels,columns,staged", [
    # 16-byte pixels of int8, more than one column tile and 8 tiles of 128x64 per compute unit; and beyond 2^32 threads of those
    ("int8", 16, 3, 230400, 256, True), ("int8", 16, 3, 79875, 256, True), ("int8", 16, 3, 39825, 256, False), ("int8", 16, 3, 460800, 64, False),
    ("int8", 16, 5, 230400, 256, True), ("int8", 32, 3, 230400, 256, False), ("int8", 48, 3, 460800, 128, False), ("float16", 8, 3, 460800, 256, False),
    ("float16", 16, 3, 115200, 128, False), ("float32", 4, 3, 460800, 256, False), ("float32", 12, 3, 230400, 64, False), ("float16", 8, 3, 1074790400, 65, True)])
def test_convolutions_with_straddling_pieces(decide, dtype, channels, kernel, pixels, columns, staged):
    assert decide("straddling", dtype, channels * SIZE[dtype], pixels, columns, kernel * kernel * channels) == [str(int(staged))]


@pytest.mark.parametrize("dtype,matrices,rows,columns,K,through", [
    # the products between transforms; rows that end inside a line of 128 bytes to 8 MB, tiles of 128x128 and large weights by rows never
    ("float16", 36, 192, 256, 256, True), ("float16", 36, 1616, 256, 256, False), ("float16", 36, 256, 384, 384, False), ("float16", 36, 2304, 384, 384, True),
    ("float16", 36, 1024, 96, 96, True), ("float16", 36, 1600, 96, 96, False), ("float32", 36, 4096, 256, 256, True), ("float16", 16, 192, 256, 256, False),
    # what a buffer's 32-bit offsets reach of 128 rows
    ("float32", 36, 1, (1 << 22) - 32, 8, True), ("float32", 36, 1, 1 << 22, 8, False)])
def test_products_that_write_through(decide, dtype, matrices, rows, columns, K, through):
    assert decide("through", dtype, matrices, rows, columns, K) == [str(int(through))]
