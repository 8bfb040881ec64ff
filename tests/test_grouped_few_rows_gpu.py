"""Grouped W4A16 calls of 16 to 47 rows per group on average, which take the
persistent tile launch where they bring its workspace and the groups hold
enough columns: both sides of the row and column lines, ragged tables, and the
calls that stay on the 16-row kernel (no workspace, one too small or not
16-byte aligned).  Tolerances: those of the persistent launch's own tests."""
import pytest

from tests.test_grouped_persistent_gpu import SLOT, Case, _workers, _workspace

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(lib):
    from longhornai_amd import ops as _ops
    return _ops


@pytest.mark.parametrize("rows,K,N,G,swiglu,tiles", [
    ([16] * 16, 512, 6144, 128, False, True),            # 384 column tiles, exactly 16 rows
    ([15] * 15 + [30], 512, 6144, 128, False, False),    # 15.9
    ([16] * 16, 512, 4096, 128, False, False),           # 256 column tiles
    ([0, 1, 97, 16, 3, 65, 5, 12] * 2, 256, 6200, 256, False, True),
    ([18] * 16, 1792, 5120, 128, False, True),           # 320
    ([17] * 16, 1792, 5120, 128, False, False),
    ([35] * 16, 512, 4096, 128, False, False),           # 256, and the row line that takes them
    ([36] * 16, 512, 4096, 128, False, True),
    ([40] * 15, 512, 4096, 128, False, False),           # 240 column tiles, short K
    ([17, 40] * 4, 12288, 4096, 128, False, True),       # 128, long K
    ([33] * 8, 512, 6144, 128, True, True),              # gate and up: 384
    ([20, 40, 10], 384, 1000, 128, True, False),
])
def test_both_sides(oracle, ops, rows, K, N, G, swiglu, tiles):
    c = Case(oracle, ops, rows, K, N, G, seed=len(rows) + K, swiglu=swiglu)
    need = c.workspace_bytes(ops)
    if _workers() == 512:
        assert (need > 0) == tiles
    c.check(oracle, c.run(ops, _workspace(ops, need, fill=0x7F), need))
    c.check(oracle, c.run(ops))


def test_workspaces_it_does_not_use(oracle, ops):
    c = Case(oracle, ops, [20] * 16, 256, 6144, 128, seed=4)
    need = c.workspace_bytes(ops)
    assert need > 0
    plain = c.run(ops)
    c.check(oracle, plain)
    assert (c.run(ops, _workspace(ops, need), SLOT - 16) == plain).all()
    assert (c.run(ops, _workspace(ops, need + 16)[4:], need) == plain).all()
