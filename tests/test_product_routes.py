"""Which products of many bfloat16 rows go to the tiles and which to the library: a rule on sizes alone (no GPU)."""
import pytest
import torch

from llmserve.parts.linear import TILES_WORK, tiles_pay

# kind, rows, weight [n, k], microseconds of the tiles and of the library with the kernel behind it, as they were when the lines were drawn (the
# tiles' gated products take 5 to 20 % less since)
MEASURED = [
    ("gated", 333, 11264, 2048, 34, 36), ("gated", 512, 11264, 2048, 36, 38), ("gated", 768, 11264, 2048, 45, 48),
    ("gated", 1300, 11264, 2048, 66, 75), ("gated", 1536, 11264, 2048, 68, 81),  # (as they are now; 86 and 73, 88 and 80 then)
    ("gated", 1258, 11264, 2048, 57, 62), ("gated", 1560, 11264, 2048, 77, 95), ("gated", 1300, 17920, 1536, 71, 83),
    ("gated", 1200, 17920, 1536, 70, 80), ("gated", 1300, 16384, 2048, 85, 94), ("gated", 700, 14336, 3072, 67, 72),
    ("gated", 400, 22016, 4096, 103, 85), ("gated", 512, 22016, 4096, 107, 88), ("gated", 896, 22016, 4096, 160, 153),
    ("gated", 1024, 22016, 4096, 188, 162), ("gated", 1100, 22016, 4096, 212, 179), ("gated", 1536, 22016, 4096, 253, 312),
    ("gated", 2048, 22016, 4096, 314, 424), ("gated", 400, 57344, 8192, 424, 360), ("gated", 512, 57344, 8192, 430, 376),
    ("gated", 1300, 57344, 8192, 1249, 1009), ("gated", 2048, 57344, 8192, 1415, 1299), ("gated", 640, 28672, 4096, 171, 140),
    ("gated", 2048, 28672, 4096, 428, 355), ("gated", 544, 16384, 3072, 91, 62), ("gated", 256, 8192, 1536, 13, 21),
    ("rotary", 512, 2560, 2048, 12, 20), ("rotary", 2048, 2560, 2048, 28, 33), ("rotary", 512, 12288, 4096, 57, 62),
    ("rotary", 1024, 12288, 4096, 106, 90), ("rotary", 2048, 12288, 4096, 185, 172), ("rotary", 256, 10240, 8192, 67, 95),
    ("rotary", 1024, 10240, 8192, 157, 142), ("rotary", 2048, 10240, 8192, 320, 275),
    ("plain", 333, 6144, 2048, 16, 20), ("plain", 2048, 6144, 2048, 57, 46), ("plain", 333, 4608, 2048, 12, 16),
    ("plain", 2048, 4608, 2048, 44, 40), ("plain", 1024, 12288, 4096, 101, 81), ("plain", 2048, 5120, 5120, 119, 103),
    ("plain", 128, 2048, 5632, 28, 16), ("plain", 228, 2048, 5632, 25, 21), ("plain", 613, 2048, 5632, 28, 33),
    ("plain", 128, 2048, 8192, 36, 22), ("plain", 96, 1024, 4096, 13, 9), ("plain", 560, 1024, 4096, 14, 18),
    ("plain", 512, 2048, 4096, 15, 20), ("plain", 228, 2048, 2048, 9, 10),
    ("parts", 512, 4096, 11008, 57, 78), ("parts", 200, 8192, 28672, 159, 313), ("parts", 1024, 8192, 28672, 479, 375),
    ("parts", 1100, 8192, 8192, 182, 137), ("parts", 128, 2048, 5632, 13, 17),
]


@pytest.mark.parametrize("kind,m,n,k,tiles,library", MEASURED)
def test_the_faster_way_is_taken(kind, m, n, k, tiles, library):
    assert tiles_pay(kind, m, n, k) == (tiles < library)


@pytest.mark.parametrize("kind,m,n,k,tiles,library", [
    ("plain", 2048, 4096, 11008, 145, 164), ("plain", 1629, 2048, 5632, 46, 51), ("plain", 768, 8192, 8192, 96, 103),
    ("gated", 330, 22016, 4096, 64, 78), ("gated", 610, 12288, 4096, 60, 67),
    ("plain", 2048, 2048, 16384, 151, 141), ("plain", 2500, 6144, 2048, 53, 48), ("plain", 1600, 6144, 2048, 41, 36)])
def test_large_products_of_one_round(kind, m, n, k, tiles, library):
    """One round of tiles, of up to 12,288 columns and not of 256 x 256; longer rows, those tiles and more rounds stay as they were."""
    assert tiles_pay(kind, m, n, k) == (tiles < library)


def test_what_the_tiles_leave_behind_is_the_librarys():
    """A gated product, a rotation or parts of K that the tiles decline become a plain product and a kernel: the plain product must
    then not be theirs either, as it was the library's product that was the faster one."""
    for kind in TILES_WORK:
        for m in (65, 200, 512, 700, 1100, 2048, 8192):
            for n, k in ((2560, 2048), (11264, 2048), (22016, 4096), (4096, 11008), (57344, 8192)):
                assert tiles_pay(kind, m, n, k) or not tiles_pay("plain", m, n, k)


@pytest.mark.parametrize("m,n,k,micros", [
    # microseconds of 32 x 32 and 32 x 64 with two buffers, 32 x 64, 64 x 64 and 128 x 128 with one
    (512, 11264, 64, (22.5, 22.0, 13.3, 14.1, 16.1)), (100, 2560, 64, (4.05, 4.32, 3.34, 4.08, 8.17)),
    (1900, 2560, 64, (20.1, 20.3, 11.9, 12.8, 16.1)), (65, 11264, 64, (7.15, 7.44, 5.12, 6.25, 8.36)),
    (200, 11264, 128, (12.3, 13.0, 10.5, 11.5, 14.6)), (512, 2560, 128, (7.77, 7.84, 7.19, 8.57, 13.7)),
    (64, 512, 128, (3.29, 4.16, 3.96, 5.28, 11.9)), (512, 11264, 256, (36.2, 35.4, 32.4, 33.1, 39.8)),
    (65, 256, 1024, (8.57, 13.7, 15.9, 24.3, 72.6)), (1900, 11264, 1024, (446, 415, 391, 371, 385)),
    (65, 512, 11008, (66.9, 120, 151, 237, 762)), (1900, 11264, 5632, (2405, 2178, 2119, 1977, 2019)),
])
def test_the_tile_of_a_32_bit_product_by_all_its_sizes(m, n, k, micros):
    """The number of columns counts too: what two buffers gain they gain from the steps of K."""
    from llmserve.ops import library

    tile = library.load("gemm32").llms_gemm32_tile(m, n, k, 256)
    assert micros[tile] <= 1.1 * min(micros)


def test_which_compute_units_bring_a_weight_nearer():
    """Those without a tile, where they are enough for the whole weight and memory has time for it (1.1B shape: q, k, v bring o_proj's,
    gate and up down_proj's); none where every compute unit has a tile."""
    from llmserve.ops import library

    def workers(m, n, rows, k=2048):
        return library.gemm_tiles_workers(library.gemm_tiles_plan(m, n, k)[0], m, n, k, 1, rows * k * 2)

    for m in (65, 130, 256, 320, 512, 560, 700, 1300, 2048):
        assert workers(m, 2560, 2048) > 0
    for m in (512, 560, 700, 1300):
        assert workers(m, 11264, 5632) > 0
    for m in (65, 130, 333):  # (the tiles wait for memory themselves)
        assert workers(m, 11264, 5632) == 0
    for m, n in ((1024, 2048), (2048, 4096), (4096, 8192)):
        bm, bn, held = library.GEMM_TILES[library.gemm_tiles_plan(m, n, 2048)[0]][:3]
        assert -(-m // bm) * -(-n // bn) % (256 * held) == 0 and workers(m, n, 1) == 0


@pytest.mark.parametrize("n,k", [(262144, 4096), (262208, 5376)])
def test_weights_of_2_gb_and_more_do_not_go_to_the_decode_kernel(n, k):
    """Its offsets are 32-bit (the launcher refuses 2^30 elements): such a weight goes to the streaming kernel, the tiles or the
    library, whatever the rows.  Shapes alone, on the meta device."""
    from llmserve.ops import library
    from llmserve.parts import linear

    def bf16(*shape):
        return torch.empty(shape, dtype=torch.bfloat16, device="meta")

    for m in (1, 8, 9, 16, 17, 64):
        fits = library.gemm_decode_fits(m, k)
        assert not linear.decode_product(bf16(m, k), bf16(n, k))
        assert linear.decode_product(bf16(m, k), bf16((1 << 30) // k - 1, k)) == fits
    assert linear.few_rows(16, bf16(n, k))
    assert not library.gemm_decode_reaches(bf16(40, 2048), bf16(1 << 19, 2048)) and library.gemm_decode_reaches(bf16(40, 2048), bf16((1 << 19) - 1, 2048))
    assert not library.gemm_decode_supported(bf16(4, 1 << 28)[:, :4096], bf16(64, 4096))


@pytest.mark.parametrize("m,n,k,decode,stream", [  # microseconds
    (1, 32000, 2048, 22.1, 24.2), (8, 32000, 2048, 22.5, 26.2), (1, 32000, 4096, 41.4, 43.4), (4, 128256, 2048, 79.7, 84.1),
    (1, 32064, 3072, 31.0, 31.9), (8, 100352, 6144, 190, 206), (8, 51200, 2560, 42.5, 46.0), (8, 256000, 2304, 185, 197),
    (8, 262144, 1152, 101, 105), (8, 151936, 896, 44.8, 45.5), (1, 50304, 1024, 19.8, 18.2), (4, 50264, 1600, 28.7, 27.2),
    (1, 262144, 1152, 94, 85), (1, 151936, 896, 42.1, 40.1), (1, 64000, 2560, 50.4, 49.1), (1, 256000, 2304, 171, 167),
    (1, 65024, 4096, 94, 83), (8, 65024, 4096, 97, 88), (1, 32512, 4096, 51, 44.5), (8, 32512, 2048, 31, 26.7), (1, 66048, 2048, 51, 48),
    (1, 65536, 4096, 79.7, 80.8), (1, 64768, 4096, 80.5, 83.3)])
def test_the_vocabularys_product_of_few_rows(m, n, k, decode, stream):
    """One stretch of the weight for each compute unit, or small workgroups: the faster one."""
    from llmserve.parts.linear import streams_large

    assert streams_large(m, n, k) == (stream < decode)


def test_smaller_weights_and_more_rows_do_not_go_to_the_streaming_kernel():
    from llmserve.parts.linear import streams_large

    assert not streams_large(9, 65024, 4096) and not streams_large(1, 8128, 4096) and not streams_large(1, 11264, 2048)
    assert not streams_large(1, 49152, 576)  # 57 MB


@pytest.mark.parametrize("m,n,k,micros", [  # microseconds by tile (those of the best third)
    (4096, 3072, 1024, {5: 34.5, 7: 37.5, 8: 37.4, 10: 37.0, 11: 30.1, 16: 34.8}), (4096, 3072, 2048, {5: 69.5, 7: 76.0, 11: 60.5, 16: 67.1}),
    (4096, 14336, 3072, {5: 347, 7: 341, 8: 315, 10: 338, 11: 319}), (3000, 9728, 896, {5: 67.2, 7: 64.1, 8: 66.2, 11: 59.6}),
    (2500, 5120, 3072, {5: 100, 8: 99, 11: 82.5}), (2500, 3072, 2048, {5: 37.7, 7: 45.1, 8: 39.3, 10: 41.5})])
def test_the_tile_beyond_2048_rows(m, n, k, micros):
    """Rows of x do not stay in L2 from one round of tiles to the next: tiles of few weight rows read them more often."""
    from llmserve.ops.library import gemm_tiles_plan

    assert micros[gemm_tiles_plan(m, n, k)[0]] <= 1.05 * min(micros.values())


def test_what_a_product_is_told_of_a_weight_brought_nearer(monkeypatch):
    """What `brings_near` says is what ops.gemm_tiles does: nothing is brought that starts between two words."""
    from llmserve.ops import library
    from llmserve.parts.linear import brings_near

    monkeypatch.setattr(library, "compute_units", lambda dev: 256)
    x, weight, near = torch.empty(512, 2048), torch.empty(11264, 2048, device="meta"), torch.empty(2048 * 5632 + 1, dtype=torch.bfloat16)
    assert brings_near(x, weight, near[:-1])[0] > 0 and brings_near(x, weight, near[1:])[0] == 0
    assert brings_near(torch.empty(2048, 2048), torch.empty(8192, 2048, device="meta"), near[:-1])[0] == 0


@pytest.mark.parametrize("n,long", [(1, True), (256, True), (1024, True), (4096, True), (4097, False), (5120, False), (5376, False), (5632, True), (6656, True),
                                    (8192, True), (8193, True), (12288, True)])
def test_long_rows_are_added_where_their_tiles_are_filled(n, long):
    """Rows of x that do not stay in a compute unit are taken in again for every tile of 16 weight rows: shares of 17 to 21 rows stay with the
    streaming kernel.  Rows that stay, and more than 16 of them, go where they went."""
    from llmserve.parts import linear

    def bf16(*shape):
        return torch.empty(shape, dtype=torch.bfloat16, device="meta")

    assert linear.adds_long_rows(n) == long
    assert linear.ops.gemm_decode_adds(16, 11008) and not linear.ops.gemm_decode_adds(17, 11008)
    assert not linear.adds_residual_in_epilogue(bf16(17, 11008), bf16(n, 11008))
    assert linear.adds_residual_in_epilogue(bf16(16, 6144), bf16(n, 6144))


@pytest.mark.parametrize("m,n,k,gated,micros,apart", [
    (1, 2304, 2304, False, 6.50, 7.26), (4, 2304, 2304, False, 6.70, 7.45), (5, 2304, 2304, False, 7.88, 7.60), (8, 2304, 2304, False, 7.97, 7.61),
    (8, 2048, 2304, False, 7.11, 7.47), (6, 2048, 2560, False, 7.18, 7.24), (8, 2560, 2560, False, 8.48, 8.15), (5, 3840, 2560, False, 9.05, 8.63),
    (8, 5120, 2560, False, 9.74, 10.21), (8, 12800, 2560, True, 15.43, 16.20), (8, 4096, 2560, True, 9.50, 8.98), (4, 4096, 2560, True, 8.17, 8.76),
    (8, 6144, 2560, True, 9.75, 10.78), (8, 10240, 3072, True, 14.96, 15.47), (5, 3072, 3072, False, 9.42, 8.67), (8, 3072, 3072, False, 9.15, 8.78),
    (8, 6144, 3072, False, 11.19, 11.49), (8, 15360, 3072, True, 18.81, 19.46), (8, 4096, 3072, True, 10.31, 9.69), (8, 1024, 4096, False, 9.07, 8.25),
    (4, 1024, 4096, False, 6.68, 7.75), (8, 4096, 4096, False, 11.80, 11.09), (5, 6144, 4096, False, 13.58, 13.04), (8, 20480, 4096, True, 31.27, 30.17),
    (2, 20480, 4096, True, 28.94, 29.54), (8, 2048, 2048, False, 5.93, 6.92), (8, 1536, 1536, False, 5.45, 6.28), (8, 10240, 2048, True, 10.37, 11.83)])
def test_an_open_sum_is_closed_the_faster_way(m, n, k, gated, micros, apart):
    """Microseconds of the product that closes its rows' sum on the way in, and of the kernel for it and the product."""
    from llmserve.parts.linear import joins_pay

    assert joins_pay(m, n, k, gated) == (micros < apart)


def test_rows_that_are_not_closed_on_the_way_in_stay_open(monkeypatch):
    from llmserve.parts import linear
    from llmserve.parts.registry import JoinedRows, NormedSum

    called = []
    monkeypatch.setattr(linear.ops, "compute_units", lambda dev: 256)
    monkeypatch.setattr(linear.ops, "gemm_decode_stream", lambda *a, **kw: called.append(a))
    monkeypatch.setattr(linear.ops, "gemm_decode_stream_supported", lambda x, w: True)
    for m, k, n, taken in ((8, 2048, 2048, True), (8, 4096, 4096, False), (4, 4096, 4096, True), (8, 2560, 2560, False), (8, 2560, 4608, True)):
        stream, weight = torch.empty(m, k, device="meta"), torch.empty(n, k, dtype=torch.bfloat16, device="meta")
        x = JoinedRows(stream, NormedSum(stream, torch.empty(k, device="meta"), 1e-5), torch.bfloat16, None)
        called.clear()
        assert linear.joined_product(x, weight, torch.empty(m, n, device="meta")) == taken
        assert x.resolved == taken and len(called) == taken
