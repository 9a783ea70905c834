"""The kernels the batch attention chooses (host-only): each attention test on
the GPU runs the ones it says, and together they run every one there is."""
import pytest

import willamette_hip as wh
from test_gpu_batch import ATTENTION_CASES


def plan_of(case):
    head_dim, group, n_kv, ctx_len, n_new = case[:5]
    return tuple(wh.debug_batch_plan([ctx_len], [n_new], n_kv, group, head_dim).values())


@pytest.mark.parametrize("case", ATTENTION_CASES, ids=str)
def test_attention_case_runs_what_it_says(case):
    assert plan_of(case) == case[6]


def test_attention_cases_reach_every_kernel():
    # softmax: waves per row, float4s per lane
    assert {c[6][1:3] for c in ATTENTION_CASES} == {(1, 1), (1, 2), (1, 4), (1, 8), (1, 16), (4, 2), (4, 4)}
    # V: head dim, query heads per wave
    assert {(c[0], c[6][3]) for c in ATTENTION_CASES} == {(d, h) for d in (64, 128) for h in (1, 2, 4)}
    # scores: every group size, with more than one step of four rows per item
    assert {c[1] for c in ATTENTION_CASES if c[6][0] * c[1] > 4} == {1, 2, 4, 8}
    # dense softmaxes at each of the softmax's sizes above 1024 positions
    assert {c[6][1:3] for c in ATTENTION_CASES if c[5] and c[3] + c[4] > 1024} >= {(1, 8), (1, 16), (4, 2), (4, 4)}


def test_plan_of_several_sequences():
    assert wh.debug_batch_plan([0] * 16, [1] * 16, 5, 4, 128) == dict(
        scores_tokens=1, softmax_waves=1, softmax_slots=1, v_heads=1)
    # one long row sets the softmax's size for all
    assert wh.debug_batch_plan([4000] + [0] * 15, [1] * 16, 5, 4, 128)["softmax_waves"] == 4
    assert wh.debug_batch_plan([4000] + [0] * 15, [32] * 16, 5, 4, 128)["softmax_slots"] == 16


@pytest.mark.parametrize("contexts,n_new,n_kv,group,head_dim", [
    ([], [], 5, 4, 128), ([1], [0], 5, 4, 128), ([4090], [7], 5, 4, 128), ([0], [16385], 5, 4, 128),
    ([0xFFFFFFFF], [1], 5, 4, 128), ([1], [1], 0, 4, 128), ([1], [1], 5, 3, 128), ([1], [1], 5, 4, 96),
    ([1], [1], 0x80000000, 4, 128), ([1], [1], 17, 4, 128)])
def test_plan_rejects(contexts, n_new, n_kv, group, head_dim):
    with pytest.raises(wh.WillametteError):
        wh.debug_batch_plan(contexts, n_new, n_kv, group, head_dim)
