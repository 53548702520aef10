"""tune_listfac's choice, on a stand-in for the handle and the clock: ms per
step by step number as measured on 1,024 replicas of a 500 eV impact, where
the longest lists are the fastest before the cascade and the slowest in it."""
import pytest

from fib_md_amd import autotune

# listfac: ms per step at steps 0, 100, 200, ..., 900 (1.25 with its lists
# grown at step 300), linear between
MEASURED = {
    1.10: (1.13, 1.44, 1.52, 1.57, 1.64, 1.72, 1.75, 1.74, 1.74, 1.75),
    1.15: (1.07, 1.31, 1.39, 1.43, 1.50, 1.59, 1.63, 1.63, 1.65, 1.66),
    1.20: (1.07, 1.37, 1.44, 1.48, 1.55, 1.65, 1.69, 1.69, 1.71, 1.73),
    1.25: (1.05, 1.33, 1.43, 1.94, 1.56, 1.67, 1.99, 1.75, 1.77, 1.79),
}
WHOLE = {1.10: 1.65, 1.15: 1.55, 1.20: 1.63, 1.25: 2.04}  # all 2,000 steps


class _Handle:
    def __init__(self, clock, listfac):
        self.clock, self.ms, self.step = clock, MEASURED[round(listfac, 2)], 0

    def md_run(self, n):
        for _ in range(n):
            k, f = divmod(self.step, 100)
            a, b = self.ms[min(k, 9)], self.ms[min(k + 1, 9)]
            self.clock[0] += (a + (b - a) * f / 100.0) * 1e-3
            self.step += 1

    def close(self):
        pass


def test_choice_holds_over_the_whole_run(monkeypatch):
    clock = [0.0]
    monkeypatch.setattr(autotune, "md_handle",
                        lambda inst, prec, params=None, use_graph=True: _Handle(clock, params.listfac))
    monkeypatch.setattr(autotune.time, "perf_counter", lambda: clock[0])
    best, table = autotune.tune_listfac([], candidates=tuple(MEASURED))
    assert best == min(WHOLE, key=WHOLE.get)
    assert [t[0] for t in table] == list(MEASURED) and all(t[1] > 0 and t[2] == "" for t in table)
    # the first steps alone would choose another
    best, _ = autotune.tune_listfac([], candidates=tuple(MEASURED), cascade=0, warmup=0, steps=40)
    assert best == pytest.approx(1.25)
