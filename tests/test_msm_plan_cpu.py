"""MSM configuration planners on the CPU.

* reference_choice reproduces every row the reference's cost model wrote
  (tests/golden/msm_cost_model_rows.json, made by make_msm_config_rows.py from
  core/src/msm/tuning/cost_model.py): alpha, s, c, w, h per (k, n, mem), and
  no choice where the script found no candidate under the memory limit.
* plan_msm keeps every choice within the memory limit as the library's own
  sizing call counts it, trades parts / batch_per_run / precomputation for
  memory as the limit tightens, and gives up only when nothing fits.
* A call's workspace is no larger than it was, nor than a longer call's.
"""
import json
import os

import pytest

from zkpoly_amd.msm import MSM, MsmConfig, workspace_least, workspace_size
from zkpoly_amd.msm_plan import Choice, model_time_us, plan_msm, reference_choice
from zkpoly_amd.runtime import Libs

ROWS = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "msm_cost_model_rows.json")))["rows"]


@pytest.mark.parametrize("row", ROWS, ids=lambda r: f"k{r['k']}-n{r['n']}-mem{r['mem'] >> 30}G")
def test_reference_choice_matches_cost_model_rows(row):
    got = reference_choice(row["k"], row["n"], 254, 254, row["mem"])
    if "error" in row:
        assert got is None
    else:
        assert got == Choice(row["alpha"], row["s"], row["c"], row["w"], row["h"])


def test_choice_maps_to_msm_config_like_get_best_config():
    # core/src/msm.rs:77-97: (precompute, window, _, parts, batch_per_run); stages 1 or 2
    cfg = Choice(alpha=17, s=15, c=1 << 18, w=4, h=2).to_config()
    assert (cfg.window_size, cfg.target_window, cfg.parts, cfg.batch_per_run) == (15, 17, 4, 2)
    assert (cfg.stage_scalars, cfg.stage_points) == (2, 2)
    one = Choice(alpha=16, s=16, c=1 << 20, w=1, h=1).to_config()
    assert (one.stage_scalars, one.stage_points) == (1, 1)


@pytest.fixture(scope="module")
def libs():
    return Libs()


def sizing(libs):
    def memory(cfg, n):
        return MSM(libs, cfg).get_buffer_size(n)[0]

    return memory


@pytest.mark.parametrize("length,batches", [(1 << 20, 1), (1 << 20, 4), (1 << 16, 3), (3 << 18, 2)])
def test_plan_fits_memory_and_tightens(libs, length, batches):
    mem = sizing(libs)
    loose = plan_msm(length, batches, 288 << 30, libs=libs)
    assert loose is not None and mem(loose, length) <= 288 << 30
    need = mem(loose, length)
    tight_limit = need // 3
    tight = plan_msm(length, batches, tight_limit, libs=libs)
    if tight is not None:
        assert mem(tight, length) <= tight_limit
        assert model_time_us(tight, length, batches) >= model_time_us(loose, length, batches)
    assert plan_msm(length, batches, 1 << 20, libs=libs) is None  # 1 MiB: nothing fits


def test_plan_prefers_parts_under_a_tight_limit(libs):
    """2^22 points in 96 MiB: the points alone of one part holding all of them
    (256 MiB) do not fit, so the plan streams parts."""
    cfg = plan_msm(1 << 22, 1, 96 << 20, libs=libs)
    assert cfg is not None and cfg.parts > 1
    assert (cfg.stage_points, cfg.stage_scalars) == (2, 2)


def test_model_counts_resident_points_across_runs():
    """With one part the points cross the link once per call whatever the
    runs; four runs of one batch differ from one run of four only by the
    three scalar copies that a shared run hides behind the accumulation."""
    one = MsmConfig(window_size=16, target_window=16, batch_per_run=1)
    four = MsmConfig(window_size=16, target_window=16, batch_per_run=4)
    scalars_copy_us = (1 << 20) * 32 / (55.0 * 1e3)
    assert model_time_us(one, 1 << 20, 4) - model_time_us(four, 1 << 20, 4) == pytest.approx(3 * scalars_copy_us)


# (points, window, target windows, bytes): workspaces that programs were told to keep before
KEPT_WORKSPACES = [
    (1, 8, 32, 581120), (256, 8, 32, 794624), (512, 5, 51, 835584), (953, 6, 43, 1334528), (1024, 6, 43, 1413376),
    (2048, 8, 32, 2332160), (4096, 8, 32, 4089344), (4096, 8, 8, 3610112), (5000, 12, 11, 10302720),
    (1 << 14, 10, 26, 15796224), (1 << 16, 12, 22, 53083392), (65537, 13, 10, 48094464), (1 << 16, 21, 13, 4486785792),
    (1 << 18, 14, 19, 171980032), (1 << 18, 16, 4, 144057344), (1 << 19, 18, 15, 835734272), (1 << 20, 12, 22, 456903168),
    (1 << 20, 16, 16, 511852032), (1 << 22, 16, 16, 1396862464)]


@pytest.mark.parametrize("n,window,target,kept", KEPT_WORKSPACES)
def test_kept_workspace_still_does(n, window, target, kept):
    assert workspace_least(Libs(), n, window, target) <= kept


@pytest.mark.parametrize("window,target", [(6, 43), (8, 32), (12, 11), (13, 20), (16, 16), (21, 13)])
def test_workspace_does_for_a_shorter_call(window, target):
    libs = Libs()
    lens = sorted({1, 2, 3, 7, 13, 30, 100, 300, 762, 763, 953, 1280, 1281, 2048, 2400, 2475, 2476, 18604, 18605, 30000,
                   50000, 100000, 104858, 131073, 139265, 262144, 262145, 300000, 1 << 19, 524289, 1 << 20, 1100000})
    for query in (workspace_least, workspace_size):
        sizes = [query(libs, n, window, target) for n in lens]
        assert sizes == sorted(sizes)


@pytest.mark.parametrize("window,target,kept", [(8, 32, 4250112), (13, 20, 49658112), (16, 16, 307735296)])
def test_kept_host_buffer_still_does(window, target, kept):
    """The drop-in call's buffer (its size does not come with the call): 5000 points, two batches a run."""
    cfg = MsmConfig(window, target, batch_per_run=2, parts=2, stage_scalars=2, stage_points=2)
    assert MSM(Libs(), cfg).get_buffer_size(5000)[0] <= kept
