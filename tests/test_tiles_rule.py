"""Which products of many rows go to the tiles: around the sizes at which both sides were measured inside prompt steps (the figures stand at the rules)."""
import pytest


@pytest.mark.parametrize("n,N,K,tiles", [
    (13550, 4096, 4096, True), (13550, 6144, 4096, True), (13550, 4096, 12288, True), (12285, 6144, 2048, True), (3000, 24576, 4096, True),      # passes that are not full
    (2000, 4096, 256, True), (9100, 1024, 256, True), (2000, 3072, 384, True), (767, 12288, 256, False),                                        # short reductions
    (1300, 4096, 2048, False), (1300, 4096, 4096, False), (1300, 4096, 12288, False), (2000, 4096, 3072, False), (3000, 2048, 6144, False),      # up to half a pass
    (900, 6144, 1536, False), (8190, 1024, 2048, False), (2000, 4096, 1024, True), (8190, 1024, 1024, True),
    (1300, 24576, 4096, False), (1300, 12288, 2048, False), (900, 16384, 4096, True), (3000, 6144, 2048, True),                                  # rows that end early in a tile
    (6600, 1040, 2048, False), (8190, 1040, 2048, True), (3000, 1824, 4096, False), (6600, 1824, 4096, True), (13550, 656, 1024, True),          # features that are no multiple of 128
    (12285, 640, 1024, False), (13550, 640, 1024, True), (12285, 640, 4096, False), (13550, 640, 4096, False),                                   # ... of 256
    (16384, 4096, 4096, True), (16384, 24576, 4096, True), (8192, 4096, 4096, True), (4096, 4096, 4096, True)])                                  # whole passes
def test_products_go_where_they_are_faster(n, N, K, tiles):
    from nano_vllm_amd import ops_seq
    assert ops_seq.tiles_rule(n, N, K) == tiles


@pytest.mark.parametrize("n,ff,K,tm", [
    (14600, 3072, 1024, 256), (2000, 3072, 1024, 256), (9000, 8192, 3072, 256), (1000, 12288, 4096, 256), (1300, 12288, 4096, 256),
    (1300, 3072, 4096, 0), (2700, 1536, 4096, 0), (2700, 1536, 3072, 0), (9100, 512, 2560, 0), (1300, 3072, 2560, 256), (1700, 3072, 4096, 0), (2000, 3072, 4096, 256), (1300, 3072, 2048, 256),    # a pass that is half to three quarters full
    (600, 6144, 1536, 0), (500, 6144, 1536, 256), (300, 12288, 1536, 0), (400, 12288, 1536, 256),                                                 # ... with rows that end early
    (600, 3072, 512, 64), (768, 3072, 512, 256), (1300, 1536, 512, 64), (300, 6144, 512, 64), (400, 6144, 512, 256), (600, 3072, 1024, 256),      # 64 rows: one pass
    (600, 12288, 512, 64), (600, 12288, 1024, 64), (1300, 6144, 512, 64), (3000, 3072, 1024, 256)])
def test_gated_products_take_the_tiles_that_are_faster(n, ff, K, tm):
    from nano_vllm_amd import ops_seq
    assert ops_seq.silu_linear_rows(n, ff, K) == tm
