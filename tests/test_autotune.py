"""What the tuning calls time and choose, on a context that answers from a table: one timing stands
for the ids that run the same walk, and a t-SNE descent is never given a split on the strength of
the walk that bh_forces takes at split 1."""
import pytest

from masterthesislucas_amd import autotune


class Context:
    """ms[split] (3 to 8: four waves) of the walk that bh_forces runs"""

    def __init__(self, kernel, n, ms):
        self.kernel, self.tree_mode, self.n, self.ms = kernel, "quadtree", n, ms
        self.variant, self.split, self.priority, self.walks, self.timed = 4, 1, True, 0, 0

    def variant_count(self):
        return 36

    def set_variant(self, v):
        self.variant = v

    def set_split(self, s):
        self.split = s

    def set_priority(self, on):
        self.priority = on

    def profile_enable(self, on=True):
        pass

    def forces_device_only(self, theta):
        self.walks += 1
        self.timed += 1

    def profile_read(self, reset=True):
        n, self.timed = self.timed, 0
        ms = self.ms[self.split if self.split < 3 else 4] + 1e-6 * ((self.walks * 7919) % 31)
        return {"traversal": (n * ms, n)}


def test_tune_times_one_walk(tmp_path):
    c = Context("gravity", 1000, {1: 0.1})
    c.set_variant(9)
    c.set_priority(False)
    best, times = autotune.tune(c, 0.5, save=True, path=str(tmp_path / "t.json"))
    assert best == 9 and list(times) == [9] and c.variant == 9 and c.priority is False
    assert c.walks <= 4
    assert autotune.lookup(c, 0.5, str(tmp_path / "t.json"))["variant"] == 9


@pytest.mark.parametrize("kernel,n,ms,want,walks", [
    ("gravity", 1000, {1: 0.3, 2: 0.2, 4: 0.1}, 4, 12),
    ("gravity", 200000, {1: 0.1, 2: 0.2, 4: 0.3}, 1, 12),
    # the walk of bh_forces at split 1 is not the descent's, whatever its time
    ("tsne", 70000, {1: 0.05, 2: 0.2, 4: 0.1}, 4, 8),
    ("tsne", 131072, {1: 0.05, 2: 0.1, 4: 0.2}, 2, 8),
    ("tsne", 131073, {1: 0.05, 2: 0.1, 4: 0.2}, 1, 12)])
def test_tune_split(kernel, n, ms, want, walks):
    c = Context(kernel, n, ms)
    (variant, split), times = autotune.tune_split(c, 0.5)
    assert (variant, split) == (4, want) and (c.variant, c.split) == (4, want)
    assert c.walks == walks and f"4/{want}" in times


def test_tune_split_of_one_setting():
    c = Context("tsne", 1000, {1: 0.1})
    assert autotune.tune_split(c, 0.5, splits=(1,), variants=(2,))[0] == (2, 1)
