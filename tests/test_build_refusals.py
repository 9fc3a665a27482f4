"""CPU checks that every cache kind refuses inputs its kernels would read past, before any launch: plans whose pages
or index vectors do not fit the sequence, and values on the host or of a type that is no 16-bit row."""
import dataclasses

import pytest
import torch

from r2omni_amd import _lib, build_three_precision_cache
from r2omni_amd.policy import PageClass, plan_from_pages

KINDS = {"tiered": {}, "bf16 keys": dict(cache_variant="v_fourq_k_bf16"), "matched": dict(matched_fp=True)}
CLASSES = [int(PageClass.FP_PAGE), int(PageClass.INT4_PAGE)]


@pytest.fixture
def host_only(monkeypatch):
    """Host tensors marked ``on_device`` pass for device ones; a launch is an error of the test."""
    def call(name, *args):
        raise AssertionError(f"{name} was launched")

    real = _lib.require_device
    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(_lib, "require_device", lambda t, what: None if getattr(t, "on_device", False) else real(t, what))
    monkeypatch.setattr(_lib, "stream_of", lambda device: 0)


def _rows(dtype=torch.bfloat16, on_device=True):
    t = torch.zeros(2, 64, 128, dtype=dtype)
    t.on_device = on_device
    t.contiguous = lambda: t
    return t


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("host_table", [True, False])
def test_pages_outside_the_sequence_are_refused(host_only, kind, host_table):
    plan = plan_from_pages([0, 40], [32, 32], CLASSES)
    if not host_table:
        plan = dataclasses.replace(plan, host_page_table=None)
    with pytest.raises(ValueError, match="inside the K/V sequence"):
        build_three_precision_cache(_rows(), _rows(), plan, **KINDS[kind])


@pytest.mark.parametrize("kind", KINDS)
def test_short_index_vectors_are_refused(host_only, kind):
    plan = dataclasses.replace(plan_from_pages([0, 32], [32, 32], CLASSES), global_token_indices=torch.arange(63))
    with pytest.raises(ValueError, match="cover the K/V sequence"):
        build_three_precision_cache(_rows(), _rows(), plan, **KINDS[kind])


@pytest.mark.parametrize("kind", KINDS)
def test_values_off_the_device_or_of_another_type_are_refused(host_only, kind):
    plan = plan_from_pages([0, 32], [32, 32], CLASSES)
    with pytest.raises(RuntimeError, match="value must live on the GPU"):
        build_three_precision_cache(_rows(), _rows(on_device=False), plan, **KINDS[kind])
    with pytest.raises(ValueError, match="bfloat16 or float16"):
        build_three_precision_cache(_rows(), _rows(torch.float32), plan, **KINDS[kind])
