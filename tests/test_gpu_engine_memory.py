"""The level-wise engine's device memory: what its rounds need is taken when it
is created (or tuned), so that a round allocates nothing."""
import numpy as np
import pytest
import torch

from tests.conftest import print_case
from warpgbm_amd import _lib
from warpgbm_amd import device as D

pytestmark = pytest.mark.gpu
dev = torch.device("cuda:0")


class Rounds:
    """An engine on random codes in eras of equal length, and its first round."""

    def __init__(self, N, F, B, E, depth, classes=0, level_bytes=0, tuning=()):
        g = torch.Generator(device=dev)
        g.manual_seed(N + F)
        x8 = torch.randint(0, B, (N, F), generator=g, device=dev, dtype=torch.int8)
        self.codes = D.codes_from_int8(x8, True, B)[0]
        _, _, order, start = D.era_layout((np.arange(N) * E // N).astype(np.int32))
        T, H = max(1, classes), (1 << (depth + 1)) - 1
        signal = x8[:, 0].float() / B + 0.3 * torch.randn(N, generator=g, device=dev)
        if classes:
            cuts = torch.quantile(signal, torch.linspace(0, 1, classes + 1, device=dev)[1:-1])
            self.target = torch.bucketize(signal, cuts).to(torch.int32)
            self.start = torch.full((classes, N), -1.0, device=dev)
        else:
            self.target, self.start = signal, torch.zeros(N, device=dev)
        self.sel = torch.arange(F, device=dev, dtype=torch.int32)
        self.rec = dict(feat=torch.zeros((T, H), dtype=torch.int32, device=dev),
                        bin=torch.zeros((T, H), dtype=torch.int32, device=dev),
                        leaf=torch.zeros((T, H), device=dev),
                        count=torch.zeros((T, H), dtype=torch.int64, device=dev),
                        gain=torch.zeros((T, H, E), device=dev))
        self.pred = self.start.clone()
        order, start = torch.from_numpy(order).to(dev), torch.from_numpy(start).to(dev)
        self.args = (self.codes, order, start, B, E, depth, T, 1 if classes else 0, 20.0, 0.0,
                     1e-6, 0.1)
        self.create(level_bytes)
        for key, value in tuning:
            self.eng.set_tuning(key, value)

    def create(self, level_bytes):
        self.eng = D.Engine(*self.args, level_bytes)

    def round(self):
        """A round from the start, and the device memory that it took."""
        self.pred.copy_(self.start)
        before = free_bytes()
        self.eng.round(self.target, self.pred, self.sel, self.rec)
        return before - free_bytes()

    def out(self):
        return [self.pred.clone()] + [self.rec[k].clone() for k in sorted(self.rec)]


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info(dev)[0]


def fill_memory():
    """All device memory but about 300 MB (what was freed before comes back late,
    and the largest piece that can be had may be less than what is free)."""
    hog, most = [], 1 << 62
    while (left := free_bytes() - 300_000_000) > 50_000_000:
        try:
            hog.append(torch.empty(min(left, most), dtype=torch.uint8, device=dev))
        except torch.OutOfMemoryError:
            most = min(left, most) // 2
            if most < 50_000_000:
                break
    return hog


# rows, features, bins, eras, depth, classes, level bytes, tuning
ERA_ENGINES = [
    # 12 nodes of three class trees in chunks of 8 and 4
    (80_000, 600, 127, 2, 3, 3, 150_000_000, ()),
    (80_000, 600, 127, 2, 4, 0, 0, ()),
    # smaller tiles, and int8 codes at few bins (tiled from shorter segments on)
    (180_000, 300, 127, 3, 3, 0, 0, ((1, 256),)),
    (190_000, 2000, 7, 3, 5, 0, 0, ((2, 0), (1, 256))),
]


@pytest.mark.parametrize("case", ERA_ENGINES, ids=[str(c) for c in ERA_ENGINES])
def test_era_rounds_allocate_nothing(gpu, case):
    """Direct era path with tiled levels, also in chunks that do not divide a
    level and with tile sizes set after the engine was created: the first round
    of an engine takes no device memory."""
    print_case("engine memory", "era rounds", *case)
    first = Rounds(*case)
    first.round()  # (kernels are loaded by now)
    r = Rounds(*case)
    assert r.round() <= 0  # (memory freed earlier may come back meanwhile)
    assert all(torch.equal(a, b) for a, b in zip(r.out(), first.out()))
    assert int((r.rec["feat"] >= 0).sum()) > 0


def test_era_tiles_within_the_level_budget(gpu):
    """The tiles' partials of a level are at most the level budget: with 100 MB the
    engine takes less than twice that besides its per-row arrays (a level of 40 (node,
    era)s and 342 row tiles would take 397 MB more), and grows the same trees."""
    case = (350_000, 1000, 127, 10, 6)
    print_case("engine memory", "era tiles within the budget", *case)
    big = Rounds(*case)
    big.round()
    budget = 100_000_000
    r = Rounds(*case, 0, budget)
    torch.cuda.empty_cache()
    r.eng.close()
    before = free_bytes()
    r.create(budget)
    taken = before - free_bytes()
    assert taken < 2 * budget + 150 * 350_000 + (64 << 20)
    r.round()
    assert all(torch.equal(a, b) for a, b in zip(r.out(), big.out()))
    assert int((r.rec["feat"] >= 0).sum()) > 20


def test_era_tiles_without_room(gpu):
    """A tile size whose buffers find no memory: the era levels go without tiles,
    and grow the same trees."""
    case = (400_000, 1000, 127, 7, 3)
    print_case("engine memory", "era tiles without room", *case)
    want = Rounds(*case)
    want.round()
    want = want.out()
    r = Rounds(*case)
    torch.cuda.empty_cache()
    hog = fill_memory()
    r.eng.set_tuning(1, 256)
    r.round()
    del hog
    torch.cuda.empty_cache()
    assert all(torch.equal(a, b) for a, b in zip(r.out(), want))
    assert int((r.rec["feat"] >= 0).sum()) > 0


def test_round_after_failed_growth(gpu):
    """One-era levels in chunks grow the tile buffers level by level.  A growth
    that finds no memory fails its round, and the next one (which starts without
    the buffers that were given back for it) fails or succeeds by what is free
    then, with the trees of an engine that never failed."""
    case = (1_000_000, 1000, 127, 1, 6, 0, 7_000_000)
    print_case("engine memory", "failed growth", *case)
    want = Rounds(*case)
    want.round()
    want = want.out()
    r = Rounds(*case)
    torch.cuda.empty_cache()
    hog = fill_memory()
    for _ in range(2):
        with pytest.raises(_lib.WgbmError, match="hipMalloc"):
            r.round()
    del hog
    torch.cuda.empty_cache()
    r.round()
    assert all(torch.equal(a, b) for a, b in zip(r.out(), want))
    assert int((r.rec["feat"] >= 0).sum()) > 0
