"""How bench.py prices the step's launches (no device)."""
import bench


class _Dev:
    def __init__(self, launches, pairs):
        self.n = launches, pairs

    def timed_launches(self):
        return self.n


def test_launches_of_one_and_two_steps():
    """9 launches of two steps and 2 of one: 20 steps of 1.5 ms in 11 launches."""
    k = bench.kernel_launches(_Dev(11, 9), 1.5)
    assert k["kernel_launches_timed"] == 11 and k["kernel_pairs_timed"] == 9
    assert abs(k["kernel_ms_avg"] * 11 - 30.0) < 1e-9
    assert k["steps_per_launch"] == round(20 / 11, 3)
    assert "9 launches" in bench.kernel_name(11, 9) and bench.kernel_name(5, 0).startswith("tlm::k_step ")


def test_traffic_is_of_the_kernel_that_ran(monkeypatch, tmp_path):
    (tmp_path / "profiles").mkdir()
    for name, kernel in (("one", "k_step"), ("two", "k_step2")):
        (tmp_path / "profiles" / f"pmc_k_step_{name}.md").write_text(
            f"`tlm::{kernel}<true, false>`\n\ntraffic_bytes_per_launch: 1.5e9\n")
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.read_traffic("one", False) == bench.read_traffic("two", True) == 1.5e9
    assert bench.read_traffic("one", True) is None and bench.read_traffic("two", False) is None
    assert bench.read_traffic("none", False) is None
