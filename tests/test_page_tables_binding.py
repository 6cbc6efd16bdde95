"""Block tables through the executors' binding: which arguments are taken and
which are refused does not depend on how the ids are held."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def executor(tmc):
    host = tmc.host()
    rt = host.HipRuntime()
    plan, att = host.DecoderLLMPlan(), host.KVCachePlan()
    att.heads, att.head_dimension, att.capacity = 2, 64, 64
    att.dtype = host.DType.Float16
    plan.attention = att
    plan.layer_count, plan.intermediate_size, plan.vocabulary_size = 2, 256, 512
    plan.rms_norm_epsilon, plan.key_value_heads = 1e-5, 2
    model = host.create_synthetic_model_resources(rt, plan, 3)
    pools = [host.create_kv_page_pool(rt, plan.kv_plan(), 16, 8) for _ in range(2)]
    states = [host.create_kv_cache_state(rt, plan.kv_plan(), p, False) for p in pools]
    for s in states:
        assert s.stage_length(rt, 1) == ""
        s.commit_length(1)
    ex = host.create_batched_decode_executor(rt, model, pools, 2)
    yield ex, [s.page_table() + [-1] * (ex.max_pages() - len(s.page_table())) for s in states]
    del ex, states, pools, model


def _forms(tables):
    return {
        "tuples": tuple(tuple(t) for t in tables),
        "array rows": [np.asarray(t, np.int32) for t in tables],
        "mixed": [list(tables[0]), tuple(tables[1])],
        "numpy ids": [[np.int32(v) for v in t] for t in tables],
    }


@pytest.mark.parametrize("form", ["tuples", "array rows", "mixed", "numpy ids"])
def test_forms_give_the_same_step(executor, form):
    ex, tables = executor
    want = ex.run([5], [1], tables, True, False)
    got = ex.run([5], [1], _forms(tables)[form], True, False)
    assert want["passed"] and got["passed"], (want["error"], got["error"])
    np.testing.assert_array_equal(got["logits"], want["logits"])


@pytest.mark.parametrize("bad", [1 << 31, -(1 << 31) - 1, 1 << 70, 0.5, "0", None])
def test_ids_out_of_type_are_refused(executor, bad):
    ex, tables = executor
    wrong = [list(t) for t in tables]
    wrong[-1][-1] = bad
    with pytest.raises(TypeError):
        ex.run([5], [1], wrong, False, False)


def test_ids_at_the_ends_of_their_type_reach_the_page_check(executor):
    ex, tables = executor
    wrong = [list(t) for t in tables]
    wrong[0][0] = (1 << 31) - 1
    assert "not allocated" in ex.run([5], [1], wrong, False, False)["error"]
    wrong[0][0] = -(1 << 31)
    assert "not allocated" in ex.run([5], [1], wrong, False, False)["error"]
    assert "shape" in ex.run([5], [1], [], False, False)["error"]
