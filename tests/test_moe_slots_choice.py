"""Which passes of the experts read their activations from slots: the choice by sizes, on stand-ins for the kernels."""
import pytest
import torch


@pytest.fixture
def passes(monkeypatch):
    """expert_mlp's passes in order, by the layout of their activations, for R sorted rows over E experts of F2 x D and D x F2 / 2."""
    from mxfp4_int8_m5_amd import sc_kernels as S
    from mxfp4_int8_m5_amd import sc_moe as M
    log = []

    def note(name, result):
        def stub(*a, **k):
            log.append(name)
            return result
        return stub

    monkeypatch.setattr(M, "moe_mm", note("rows", None))
    monkeypatch.setattr(M, "moe_mm_blocked", note("slots", None))
    monkeypatch.setattr(M, "gather_blocked", note("gather", (None, None)))
    monkeypatch.setattr(M, "act_quant_sorted", note("sort", (None, None)))
    monkeypatch.setattr(S, "act_quant", note("quant", (None, None)))
    monkeypatch.setattr(M, "takes_slots", lambda R, E, K, tm, fmt: tm == 256)

    def run(E, D, F2, R, tm=256):
        log.clear()
        M.expert_mlp(None, None, R, (None, None, torch.empty(E, F2)), (None, None, torch.empty(E, D)), None, None, None, 0, tm, None)
        return list(log)

    return run


GATE = {True: ["gather", "slots"], False: ["rows"]}
DOWN = {True: ["sort", "slots"], False: ["quant", "rows"]}


# both sides of each line: few tiles, where the rows' launch spreads over more CUs; rows an expert; narrow layers; reductions
@pytest.mark.parametrize("E,D,F2,rows,gate,down", [
    (8, 2048, 2048, 110, False, False), (8, 2048, 2048, 180, False, True), (4, 2048, 4096, 180, False, False),
    (4, 2048, 4096, 300, False, True), (8, 768, 2048, 180, False, False), (6, 640, 2560, 1053, False, False),
    (16, 1024, 2048, 110, False, False), (16, 1024, 2048, 300, False, True), (32, 2048, 2048, 110, False, True),
    (32, 2048, 2048, 220, False, True), (32, 2048, 2048, 300, True, True), (32, 512, 2048, 300, False, True),
    (48, 1536, 2048, 110, True, True), (64, 1024, 2048, 110, False, True), (64, 1024, 2048, 150, True, True),
    (64, 2048, 2048, 110, True, True), (16, 4096, 8192, 110, False, True), (16, 4096, 8192, 150, True, True),
    (128, 2048, 1536, 400, False, True)])
def test_layout_by_size(passes, E, D, F2, rows, gate, down):
    assert passes(E, D, F2, E * rows) == GATE[gate] + DOWN[down]


def test_other_row_tiles_stay_by_rows(passes):
    assert passes(64, 2048, 2048, 64 * 400, tm=64) == GATE[False] + DOWN[False]
