"""The verify's tile choice (`verify_tile`, csrc/verify.hip) restated, so that a
test can name the tile its case takes; test_verify_tile_rule.py compares the two."""


def verify_tile(rows, value_heads, K, V, f32, qm, deferred):
    def waves(tile):
        return rows * value_heads * -(-V // tile)

    if deferred:
        if waves(16) <= (1280 if qm == 8 else 3072) or V <= 16:
            return 16
        if waves(32) <= 3072 or (V - 1) % 64 < 32:
            return 32
        if not f32 or qm == 8 or waves(64) <= 3072:
            return 64
        return 64 if qm == 4 and 64 < K <= 128 and waves(32) > 16384 else 32
    if waves(16) <= (1536 if qm < 8 and K <= 64 else 1280) or V <= 32:
        return 16
    if f32 and K > 64 and qm == 1 and waves(16) <= (4096 if K > 128 else 12288):
        return 16
    if f32 and 64 < K <= 128 and qm == 2 and 4096 <= waves(16) <= 8192:
        return 16
    if (V - 1) % 128 < 64:
        return 64
    return 64 if waves(64) <= (1024 if qm == 8 else 2560) else 128


def window_capacity(Q):
    return 1 if Q <= 1 else 2 if Q <= 2 else 4 if Q <= 4 else 8
