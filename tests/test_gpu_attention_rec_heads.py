"""The record attention's work split by KV head and key range, at the sizes where its indexing can go wrong.

One workgroup takes one (KV head, split): the grid is padded to whole groups of 8 splits, a split's pages run through a
3-slot ring (1 to 4 pages a split), a record's last piece ends with the record (the pool's last record ends the pool), the
block table of a split is read by one load per thread and a loop beyond 128 pages, and 1 to 4 row blocks of 16 rows run
in 2 to 4 waves. Against the oracle's fp64 attention over the same records, tolerance as in test_gpu_attention_rec.py.
"""
import pytest

from conftest import load_host
from test_gpu_attention_rec import dev, run_case  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 12, 16])
@pytest.mark.parametrize("pages,splits", [(1, 1), (2, 1), (3, 1), (4, 1), (9, 9), (17, 8), (24, 8), (35, 9)])
def test_pages_and_splits(dev, orc, M, pages, splits):  # noqa: F811
    """The last page is full: its last record is the pool's last."""
    run_case(dev, orc, load_host(), M, 32 * pages - M, splits=splits, paged=pages % 2 == 0, seed=1300 + M)


@pytest.mark.parametrize("M,pages", [(4, 129), (9, 193), (16, 300)])
def test_long_splits(dev, orc, M, pages):  # noqa: F811
    """More pages in a split than its workgroup has threads, through a permuted table."""
    run_case(dev, orc, load_host(), M, 32 * pages - M - 5, splits=1, paged=True, seed=1400 + M)


@pytest.mark.parametrize("M", [4, 8, 16])
@pytest.mark.parametrize("pages", [64, 65, 193, 321, 513])
def test_planned_splits(dev, orc, M, pages):  # noqa: F811
    """The library's own split counts on both sides of their rule's corners."""
    run_case(dev, orc, load_host(), M, 32 * pages - M, seed=1500 + M)
