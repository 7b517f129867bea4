"""The numbering of the POTRF items of a tile (item_potrf in tasktorrent_amd/csrc/tile_ops.hpp): row r of 64x64 blocks
has r items (row 0 one), the blocks (r, 0 .. r-2) and then the tail item with (r, r-1) and (r, r). An executor that
claims items in order runs them without deadlock if every flag an item waits for is set by a lower-numbered one."""
import pytest


@pytest.mark.parametrize("nb", [1, 2, 3, 4, 8, 16, 64])
def test_items_wait_on_lower_numbers_only(nb):
    items = []
    for it in range(1 + nb * (nb - 1) // 2):
        r, rem = 0, it
        while rem >= max(1, r):
            rem -= max(1, r)
            r += 1
        items.append((r, rem, rem == max(1, r) - 1))
    setter = {}
    for it, (r, rem, tail) in enumerate(items):
        blocks = [(r, r - 1), (r, r)] if tail and r else [(r, r)] if tail else [(r, rem)]
        for b in blocks:
            assert b not in setter
            setter[b] = it
    assert set(setter) == {(r, q) for r in range(nb) for q in range(r + 1)}
    for it, (r, rem, tail) in enumerate(items):
        q = r - 1 if tail else rem
        waits = [(r, j) for j in range(q)] + [(q, j) for j in range(q)] + ([(q, q)] if r else [])
        assert all(setter[w] < it for w in waits)
