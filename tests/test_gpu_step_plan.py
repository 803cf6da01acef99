"""The chunk step's plan, built from chunks of 512, 1024 or 2048 routes by
token count, at the edges of its chunks and of the rule that picks them: the
plan arrays in the step's workspace must be those of a stable sort of the
step's expert ids (and so those of the staged plan, which always takes 2048)."""
import numpy as np
import pytest

from helpers import Layer, synth_hidden, synth_logits, torch
from test_gpu_wide import expected_plan, prefill_wide

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layer(q38m, orc):
    return Layer(q38m, orc, 23, 0, ("fmt", 4, 32, 0.02), ("fmt", 8, 0, 0.002), with_host=False)


def grab(ws, address, count, dtype):
    offset = address - ws.buffer.data_ptr()
    raw = ws.buffer[offset:offset + count * np.dtype(dtype).itemsize]
    return raw.cpu().numpy().view(dtype)


# one partial chunk; either side of one chunk of 512 routes; 64 chunks of 512
# and the first count past them; the same for 1024
@pytest.mark.parametrize("tokens,invalid", [(1, False), (51, False), (52, False), (1000, True),
                                            (3276, False), (3277, False), (6553, True),
                                            (6554, False)])
def test_step_plan_is_the_stable_sort(q38m, layer, tokens, invalid):
    t = torch()
    ws = q38m.WideWorkspace_(tokens)
    ws.buffer.fill_(0x5A)
    hidden = synth_hidden(q38m, 23, 3, tokens)
    logits = synth_logits(q38m, 23, 4, tokens)
    routes = tokens * 10
    plan = ws.ws.plan
    if invalid:  # given ids, one of them out of range: the plan fails closed
        ids = np.stack([np.random.default_rng(k).choice(512, 10, replace=False)
                        for k in range(tokens)]).astype(np.int32)
        ids.flat[routes // 2] = 512
        at = ws.ws.expert_ids - ws.buffer.data_ptr()
        ws.buffer[at:at + 4 * routes] = t.from_numpy(ids.ravel().view(np.uint8)).cuda()
        at = ws.ws.expert_weights - ws.buffer.data_ptr()
        ws.buffer[at:at + 4 * routes] = 0
        logits = None
    prefill_wide(q38m, layer, hidden, logits, ws)
    t.cuda.synchronize()
    ids = grab(ws, ws.ws.expert_ids, routes, np.int32)
    order, counts, offsets, task_offsets, tasks = expected_plan(ids, tokens)
    header = grab(ws, plan.header, 16, np.uint32)
    inverse = np.arange(routes)
    inverse[order] = np.arange(len(order))
    packed = np.concatenate([order, np.arange(len(order), routes)])
    assert header[5] == len(tasks) and header[6] == (1 if invalid else 0)
    assert np.array_equal(grab(ws, plan.expert_counts, 512, np.uint16), counts)
    assert np.array_equal(grab(ws, plan.expert_offsets, 513, np.uint32), offsets)
    assert np.array_equal(grab(ws, plan.expert_task_offsets, 513, np.uint32), task_offsets)
    assert np.array_equal(grab(ws, plan.packed_assignment, routes, np.uint32), packed)
    assert np.array_equal(grab(ws, plan.assignment_to_packed, routes, np.uint32), inverse)
    assert np.array_equal(grab(ws, plan.tasks, 2 * len(tasks), np.uint32).reshape(-1, 2), tasks)
