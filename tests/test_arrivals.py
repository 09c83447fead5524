"""Arrivals at a counter that launches share, driven on the host: of each launch exactly one workgroup is the last one, and it is the one
that arrives last, whatever launches that overlapped or were abandoned have left behind."""
import ctypes
import random

import pytest

from host_arithmetic import load

PERIOD = (1 << 19) - 1


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return load(tmp_path_factory.mktemp("host"))


class Counters:
    def __init__(self, lib):
        self.lib, self.tagged = lib, lib.layout(1)
        self.words = (ctypes.c_int * (4 * lib.layout(0)))()

    def arrive(self, splits, epoch, count=None, tile=5):
        """Whether each of the arrivals was the last one."""
        return [bool(self.lib.arrive(self.words, tile, splits, epoch)) for _ in range(splits if count is None else count)]

    def clean(self, tile=5):
        return self.words[2 * tile] == self.words[2 * tile + 1] == 0


def once(splits):
    return [False] * (splits - 1) + [True]


@pytest.mark.parametrize("splits", [2, 4, 8, 100, 400])
def test_arrivals_of_one_launch_after_another(lib, splits):
    c = Counters(lib)
    for epoch in (1, 2, 3, 12345, PERIOD, 1):
        assert c.arrive(splits, epoch) == once(splits) and c.clean()
    for _ in range(3):
        assert c.arrive(splits, 0) == once(splits) and c.clean()      # a handle's counters


# A launch leaves fewer than its splits.  1 << 18, 1 << 13 and the like: where d times one tag and d times another agree in 20 bits.
@pytest.mark.parametrize("splits", [2, 4, 8, 128])
@pytest.mark.parametrize("apart", [1, 2, 1 << 11, 1 << 13, 1 << 16, 1 << 17, 1 << 18, PERIOD - 2])
def test_what_one_launch_left_is_no_later_ones_count(lib, splits, apart):
    for left in {1, 2, 3, 4, 7, 8, 64, splits - 1, splits + 1}:
        for epoch in (1, 77, PERIOD - 1 - apart):
            if epoch < 1 or epoch + apart > PERIOD:
                continue
            for first, second in ((epoch, epoch + apart), (epoch + apart, epoch)):    # (tags come round; streams may swap two launches)
                c = Counters(lib)
                c.arrive(1 << 11, first, left)
                assert c.arrive(splits, second) == once(splits), (left, first, second)
                assert c.clean() and c.arrive(splits, second % PERIOD + 1) == once(splits)


def test_what_several_launches_left_is_no_later_ones_count(lib):
    rng = random.Random(3)
    for _ in range(20000):
        c, splits = Counters(lib), rng.choice((2, 4, 8, 16))
        last = rng.randrange(40, PERIOD - 10)
        tags = [last - rng.choice((0, 1, 2, 3, rng.randrange(40))) for _ in range(rng.randrange(2, 8))]
        for tag in tags:
            c.arrive(splits, tag, 1)
        c.words[c.tagged + 5] = rng.choice((0, 3, -1, (min(tags) - 1) << lib.layout(2) | 1))
        epoch = max(tags) + rng.choice((1, 2, 3, rng.randrange(1, PERIOD - max(tags) + 1)))
        assert c.arrive(splits, epoch) == once(splits), (tags, epoch)
        assert c.clean()


def test_anything_in_the_words(lib):
    rng = random.Random(4)
    for _ in range(20000):
        c, splits, epoch = Counters(lib), rng.choice((2, 4, 8)), rng.randrange(1, PERIOD + 1)
        word = lambda: rng.choice((rng.randrange(9), rng.randrange(-2 ** 31, 2 ** 31), -1, 2 ** 31 - 1))
        c.words[10], c.words[11], c.words[c.tagged + 5] = count, tags, tagged = word(), word(), word()
        if tags % 2 ** 32 == count * epoch or tagged >> lib.layout(2) == epoch:
            continue        # (this launch's own)
        assert c.arrive(splits, epoch) == once(splits), (count, tags, tagged, epoch)
