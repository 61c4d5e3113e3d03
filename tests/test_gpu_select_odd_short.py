"""Odd rows at the edges of the row kernel's forms: a page per thread up to 1024
pages, 4 or 8 past it (the sums change hands through LDS), every group width; and
rows with more candidates than the finisher's registers hold."""
import pytest

from tests import test_gpu_select_odd as odd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("MP,G,b,combine", [
    (1, 16, 1, "nrm"), (2, 1, 1, "nrm"), (63, 16, 126, "nrm"), (65, 4, 9, "max"), (255, 8, 100, "nrm"), (1021, 1, 64, "nrm"),
    (1023, 16, 126, "nrm"), (1025, 16, 126, "nrm"), (1026, 4, 1000, "max"), (4095, 16, 410, "nrm"), (4093, 5, 126, "nrm"),
    (4097, 1, 4000, "nrm"), (8190, 4, 819, "nrm"), (8189, 7, 126, "max"),
    (40001, 4, 17000, "max"), (40003, 2, 17001, "nrm")])     # over 16384 candidates: finish_row
def test_short_and_long_odd_rows(MP, G, b, combine):
    odd.test_odd_rows(MP, G, b, combine)
