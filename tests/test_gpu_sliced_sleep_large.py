"""Worlds whose step tiles may sleep, beyond 2048 squares of 64 cells (by 2x2 and by 4x2
words), through everything that must wake a region or end the record."""
import pytest

from tests import test_gpu_sliced_sleep as Z

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(2945, 2881), (5903, 6101)], ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("name", list(Z.SIZES))
def test_sleeping_equals_plain_and_dense(name, size, monkeypatch):
    monkeypatch.setitem(Z.SIZES, name, size)
    Z.test_sleeping_equals_plain_and_dense(name)


def test_kernels_whose_tiles_sleep_are_named():
    print("\n[gpu] sleeping step kernels by name", flush=True)
    Z.rs("twelve_materials")
    for size, sleeping, dense in (((2049, 2048), 3, 3), ((2945, 2881), 4, 2), ((5903, 6101), 5, 3)):
        w = Z.S.World(Z._ctx, Z.rs("twelve_materials"), *size)
        assert w.variant_info(4, 24)[:2] == (1, sleeping)
        w.set_sleep(False)
        assert w.variant_info(4, 24)[:2] == (1, dense)
        w.close()


@pytest.mark.parametrize("name", ["four_materials", "features"])
@pytest.mark.parametrize("size", [(2049, 4097), (32801, 257)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_modifications_of_the_first_step(name, size):
    """Lists that go into the packed grid."""
    Z.test_modifications_of_the_first_step(name, size)
