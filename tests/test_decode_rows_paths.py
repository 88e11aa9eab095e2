"""Which launches a decode step of a Llama model takes."""
from types import SimpleNamespace

import pytest


@pytest.mark.parametrize("splits", [True, False])
def test_no_split_sums_where_they_are_off(monkeypatch, splits):
    """TGIS_DEFER_REDUCE=0: dense steps keep off the launches that may split a residual product's sums, those of up to four rows stay."""
    from tgis_amd.models.custom_modeling import flash_llama_modeling as modeling

    monkeypatch.setattr(modeling, "DEFER_REDUCE", splits)
    lm = object.__new__(modeling.FlashLlamaForCausalLM)
    lm._rows16_path, lm._rows_path = {n: True for n in range(3, 65)}, {n: n <= 4 for n in range(65)}
    assert [lm.rows16_path(n) for n in (3, 5, 64)] == [splits] * 3
    assert lm.rows_path(4) and not lm.rows_path(5)


@pytest.mark.parametrize("width,served", [(512, True), (4096, True), (4608, False), (5120, False), (6144, True), (8192, True)])
def test_int4_widths(width, served):
    """Widths whose residual units are a little more than the chip has places stay with the other launches."""
    from tgis_amd.models.custom_modeling import flash_llama_modeling as modeling

    model = object.__new__(modeling.FlashLlamaModel)
    model.config, model.layers, model.int4_norms, model._int4_rows = SimpleNamespace(hidden_size=width), [], ([], []), {}
    assert model.serves_int4_rows(1) == served and not model.serves_int4_rows(33)
