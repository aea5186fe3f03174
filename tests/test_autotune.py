"""The launch tuner on made-up solvers whose step times are known (no GPU)."""
import pytest

from seismod_amd import autotune


class Ctx:
    def sync(self):
        pass


class Timed:
    """Counts steps and the time that `step` gives for each of them."""

    def __init__(self):
        self.ms = self.n = 0

    def reset(self):
        pass

    def set_timing(self, on):
        if on:
            self.ms = self.n = 0

    def timing(self):
        return self.ms, self.n

    def tick(self, ms, n):
        self.ms, self.n = self.ms + ms * n, self.n + n


class E2d(Timed):
    """A multistep solver: rows per chunk matter for runs of one step only."""

    class cfg:
        nx, nz, npml = 200, 300, 20

    def __init__(self, best):
        super().__init__()
        self.best, self.shape = best, (5, 32)

    def launch(self):
        return self.shape

    def set_launch(self, rows, graph_steps=32):
        self.shape = (rows, graph_steps)

    def run(self, n):
        # (several steps a launch look best at the first candidate)
        self.tick(0.5 if n > 1 else 1.0 + abs(self.shape[0] - self.best), n)


class E2dBatch(Timed):
    def __init__(self, ctx, graph_steps=32):
        super().__init__()

    def set_variant(self, variant):
        self.variant = variant

    def set_group_bytes(self, nbytes):
        self.group = nbytes

    def run(self, sims, steps):
        assert len(steps) == len(sims)
        self.asked = list(steps)
        fast = self.variant == "staged" and all(s.shape[0] == s.best for s in sims)
        self.tick(0.5 if max(steps) > 1 else 1.0 if fast else 2.0, max(steps))

    def close(self):
        pass


@pytest.fixture(autouse=True)
def no_cache():
    autotune.clear_cache()
    yield
    autotune.clear_cache()


def test_e2d_tunes_the_one_step_launch():
    s = E2d(best=6)
    assert autotune.tune_e2d(s, Ctx()) == (6, 32) and s.shape == (6, 32)


def test_e2d_batch_tunes_the_one_step_launch(monkeypatch):
    from seismod_amd import solver
    monkeypatch.setattr(solver, "E2dBatch", E2dBatch)
    sims = [E2d(best=3) for _ in range(4)]
    assert autotune.tune_e2d_batch(sims, Ctx()) == (3, "staged")
    assert all(s.shape == (3, 32) for s in sims)


def test_e2d_groups_run_the_steps_asked_for():
    sims = [E2d(best=3) for _ in range(3)]
    b = E2dBatch(None)
    b.set_variant("rows")
    autotune.tune_e2d_groups(b, sims, candidates_mb=(0, 256))
    assert b.asked == [16, 16, 16]
    autotune.tune_e2d_groups(b, sims, steps=[10, 20, 30], candidates_mb=(0,))
    assert b.asked == [10, 20, 30] and b.group == 0


class A3d(Timed):
    """A flat grid: 15 tiles at 4 rows, 1024 slots, so many chunks are best."""

    class cfg:
        nx, ny, nz, np, storage = 320, 20, 20, 20, "f32"

    def __init__(self):
        super().__init__()
        self.v, self.shape = "cell", (4, 60)

    def variant(self):
        return self.v

    def set_variant(self, v):
        if v != self.v:
            self.v, self.shape = v, (4, 60)

    def launch(self):
        return self.shape

    def set_launch(self, rows, chunks):
        length = -(-360 // chunks)
        if (chunks - 1) * length >= 360:
            raise ValueError("empty chunk")
        self.shape = (rows, chunks)

    def run(self, n):
        rows, chunks = self.shape
        items = chunks * (60 // rows)
        self.tick((1.0 if self.v == "tile" else 1.2) * max(1.0, 1024 / items) * (1.1 if rows != 8 else 1.0), n)


def test_a3d_tunes_no_worse_than_its_own_launch():
    s = A3d()
    for v in ("cell", "tile"):
        s.set_variant(v)
        s.reset()
        s.run(1)
    own = autotune._time(s, Ctx(), 1)
    assert autotune.tune_a3d(s, Ctx()) == ("tile",) + s.launch()
    assert autotune._time(s, Ctx(), 1) <= own
    # the chunks of 4 rows at 8 rows, as many items: 120 wanted, 60 the most of 6 planes
    assert s.launch() == (4, 60)


def test_a3d_candidates_given_are_the_only_ones():
    s = A3d()
    assert autotune.tune_a3d(s, Ctx(), candidates=[(2, 8), (4, 8)], variants=("cell",))[0] == "cell"
    assert s.launch() in ((2, 8), (4, 8))
