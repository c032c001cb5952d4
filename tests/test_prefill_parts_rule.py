"""Which prefill launches behind a cached prefix have their keys cut into parts, as the host decides
it (256 CUs where no device can be asked)."""
import pytest


def _bytes(tokens, batch, heads, kv_heads, positions, max_keys=0, page=32):
    from nanovllm_jax_amd import _lib
    return _lib.load().nvj_paged_prefill_split_workspace_bytes(tokens, batch, heads, kv_heads, page,
                                                               -(-positions // page), max_keys)


@pytest.mark.parametrize("tokens,batch,heads,kv_heads,positions", [
    (29, 21, 8, 1, 768), (229, 49, 4, 4, 1024), (78, 78, 8, 1, 1024), (24, 8, 32, 32, 1024),
    (115, 32, 28, 4, 2048), (243, 27, 28, 4, 2048), (634, 90, 8, 1, 1536), (24, 6, 32, 32, 2048),
    (260, 20, 28, 4, 4096), (8, 8, 32, 32, 4096),
    (100, 53, 4, 4, 6912), (20, 8, 32, 32, 4608), (1568, 168, 8, 1, 4832), (1100, 100, 4, 4, 8192),
    (110, 55, 16, 8, 8192), (157, 14, 32, 32, 8192), (84, 7, 32, 32, 8192), (54, 45, 32, 8, 8192),
])
def test_keys_stay_whole_where_parts_are_slower(tokens, batch, heads, kv_heads, positions):
    """Launches that took 1.05 .. 1.4 times as long in parts: sequences of a few tokens that give the
    CUs enough to do by themselves."""
    assert _bytes(tokens, batch, heads, kv_heads, positions) == 0


@pytest.mark.parametrize("tokens,batch,heads,kv_heads,positions", [
    (31, 1, 28, 4, 1024), (3, 1, 16, 16, 1024), (139, 1, 32, 8, 1536), (375, 5, 16, 16, 2048),
    (116, 3, 64, 8, 4096), (277, 2, 32, 8, 3904), (266, 4, 32, 8, 4096), (45, 11, 28, 4, 8192),
    (61, 17, 32, 8, 8192), (344, 11, 16, 8, 7936), (393, 2, 32, 8, 6144), (1805, 3, 8, 1, 8192),
    (277, 2, 64, 8, 8192), (500, 1, 32, 8, 5120), (30, 1, 32, 8, 5120),
])
def test_keys_are_cut_where_parts_are_faster(tokens, batch, heads, kv_heads, positions):
    """Launches that take 0.4 .. 0.85 of the time in parts; and the bound decides, not the table."""
    assert _bytes(tokens, batch, heads, kv_heads, positions) > 0
    assert _bytes(tokens, batch, heads, kv_heads, 4 * positions, positions) > 0
    assert _bytes(tokens, batch, heads, kv_heads, 4 * positions, 512) == 0


@pytest.mark.parametrize("tokens,batch,heads,kv_heads,positions,cut", [
    # workgroups at and past the line: up to 1024 positions 72
    (72, 5, 32, 8, 1024, True), (80, 6, 32, 8, 1024, False), (9, 9, 16, 8, 1024, True),
    # up to 2048 half the CUs (128), more where few sequences and KV heads share them
    (370, 1, 32, 8, 2048, True), (400, 1, 32, 8, 2048, False), (64, 17, 32, 8, 2048, False),
    (330, 1, 28, 4, 2048, True), (360, 1, 28, 4, 2048, False), (160, 16, 28, 4, 2048, False),
    # up to 4096
    (16, 16, 64, 8, 4096, True), (17, 17, 64, 8, 4096, False), (30, 30, 32, 8, 4096, False),
    (850, 2, 16, 1, 4096, True), (960, 3, 16, 1, 4096, False), (411, 94, 6, 2, 2688, False),
    (48, 48, 16, 1, 4096, True), (66, 66, 16, 1, 4096, False), (40, 40, 16, 1, 4096, True),
    # larger workgroups in parts, up to one a CU, 13 / 16 of that where the XCDs are not filled evenly
    (990, 1, 32, 8, 8192, True), (1050, 1, 32, 8, 8192, False), (390, 2, 64, 4, 8192, True),
    (410, 2, 64, 4, 8192, False),
])
def test_lines_of_the_cut(tokens, batch, heads, kv_heads, positions, cut):
    assert (_bytes(tokens, batch, heads, kv_heads, positions) > 0) == cut


def test_partials_have_a_bound():
    """No launch asks for more than 65 MiB of partials, half-empty batches included."""
    most = 0
    for heads, kv_heads in [(8, 1), (16, 1), (6, 2), (28, 4), (4, 4), (16, 8), (32, 8), (64, 8),
                            (128, 8), (16, 16), (32, 32), (64, 64), (12, 3)]:
        for batch in [*range(1, 33), 89, *range(36, 257, 4)]:
            for per in (0.5, 1, 2, 7, 15, 16, 17, 33, 100, 250, 700, 2000):
                for positions in (640, 1024, 2048, 4096, 4128, 8192, 32768):
                    tokens = max(1, int(per * batch))
                    most = max(most, _bytes(tokens, batch, heads, kv_heads, positions))
    assert 16 << 20 < most <= 65 << 20
