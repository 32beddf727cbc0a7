"""HSMAC sweeps on the velocity itself (time blocking without overlap,
red-black, no time blocking): what the tests of batches and tile shapes show
with the default options, which sweep in divergence form, is shown here for the
in-place sweeps, whose tiles, persistent grids and chunks those tests name."""
import dataclasses

import pytest

import test_gpu_autotune as TA
import test_gpu_batch as TB

pytestmark = pytest.mark.gpu

FORMS = [(True, False, "red-black-fast"), (True, True, "red-black"), (False, True, "red-black-fast")]
forms = pytest.mark.parametrize("form", FORMS, ids=["blocked", "blocked-overlap-rb", "naive-overlap"])


@pytest.fixture
def in_place(form, monkeypatch):
    """The configurations of the reused tests, with HSMAC of the given form."""
    from lcs_mi355x import config as C
    hs = C.HSMAC(*form, 1.7, 1e-3, 6, 300)
    mixed, c1 = TB.mixed_configs, TA.c1_config

    def c1_config(*a, **k):
        c = c1(*a, **k)
        return dataclasses.replace(c, flow=dataclasses.replace(c.flow, couple=hs))

    monkeypatch.setattr(TB, "mixed_configs", lambda dtype="f64", rcf=True: mixed(dtype, hs, rcf))
    monkeypatch.setattr(TA, "c1_config", c1_config)


@forms
def test_batched_boxes_follow_the_oracle(in_place, form):
    TB.test_batched_boxes_follow_the_oracle()


@forms
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_box_result_does_not_depend_on_the_mix(in_place, form, dtype):
    TB.test_box_result_does_not_depend_on_the_mix(dtype)


@forms
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_persistent_sweeps_change_no_result(in_place, form, dtype):
    TB.test_persistent_sweeps_change_no_result(dtype)


@forms
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_batch_tiling_changes_no_result(in_place, form, dtype):
    TB.test_batch_tiling_changes_no_result(dtype)


@forms
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_every_shape_gives_the_same_box(in_place, form, dtype):
    TA.test_every_shape_gives_the_same_box(dtype)
