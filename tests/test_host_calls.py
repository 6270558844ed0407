"""The host layer's calls into the device functions: their order on streams, and how it waits."""
import pytest

import recorded_calls


@pytest.mark.parametrize("prompt", [1, 3])
def test_a_batch_step_comes_behind_the_prompts_of_its_sequences(prompt):
    """A prompt runs on its sequence's stream, the step that reads its keys and values on the batch's: the former is waited for in between."""
    calls = recorded_calls.run(f"""
batch = P.BatchContext(tiny_model(), 2, context_len=64)
calls()
result = []
for b in range(2):
    batch.next_token(b, [1] * {prompt})
    result += calls()
batch.next_tokens([1, 2])
result += [("step", None)] + calls()
""")
    at = calls.index(["step", None])
    step, before = {s for name, s in calls[at + 1:] if name == "lcu_softmax_argmax_rows"}, calls[:at]
    prompts = {s for name, s in before if name == "lcu_softmax_argmax_status"}
    assert len(step) == 1 and len(prompts) == 2 and not step & prompts
    for stream in prompts:
        last = max(i for i, (name, s) in enumerate(before) if s == stream and name != "lcu_sync")
        assert ["lcu_sync", stream] in before[last:]


STEP = {"context": "context.next_token([1])", "batch": "batch.next_tokens([1, 2])[0]"}
CONTEXTS = """
model = tiny_model()
context, batch = P.Context(model, context_len=64), P.BatchContext(model, 2, context_len=64)
def names():
    return [name for name, _ in calls()]
"""


def test_a_prompt_waits_for_its_stream():
    """A call of several tokens has nothing to gain by looking for its token: it takes no processor time while it waits, however long."""
    tokens, seconds, seen = recorded_calls.run(CONTEXTS + """
stand_in.recorded_lateness(30000)
tokens, began = [], time.thread_time()
for _ in range(8):
    tokens.append(context.next_token([1, 2, 3]))
result = tokens, time.thread_time() - began, names()
""")
    assert tokens == [7] * 8 and seconds < 0.03 and seen[-1] == "lcu_sync"  # of 0.24 s in all


@pytest.mark.parametrize("kind", STEP)
def test_a_step_that_outlasts_the_watch_is_waited_for(kind):
    """The token of a quick step is taken as it comes, that of a slow one behind a wait for its stream."""
    tokens, quick, late, again = recorded_calls.run(CONTEXTS + f"""
step = lambda: {STEP[kind]}
tokens = [step() for _ in range(3)]
names(); tokens.append(step())
quick = names()
stand_in.recorded_lateness(1000)
tokens += [step(), step()]
late = names()
stand_in.recorded_lateness(-1)
tokens.append(step())
result = tokens, quick, late, names()
""")
    assert tokens == [7] * 7 and late == 2 * ["lcu_graph_launch", "lcu_sync"]
    assert quick == again == ["lcu_graph_launch"]


def test_contexts_say_what_their_models_hold():
    """Every stream of a context or a batch knows the bytes of the matrices that a call goes through, before its first launch."""
    weights = recorded_calls.run("""
model = tiny_model()
context, batch = P.Context(model, context_len=64), P.BatchContext(model, 2, context_len=64)
calls()
context.next_token([1, 2]); batch.next_token(0, [1, 2]); batch.next_token(1, [1, 2]); batch.next_tokens([1, 2])
of_llama = sorted({s for name, s in calls() if name.startswith("lcu_softmax")})
layered = P.Model(config={"architecture": "Logivik", "vocab": 301, "width": 64, "embedding": {"scale": 8.0}, "norm": {"eps": 1e-5}, "layers": [
    {"type": "latent_attention_2", "mlp": {"kind": "dense", "ff": 128},
     "mixer": {"heads": 2, "dim": 32, "vdim": 32, "kv_rank": 32, "q_rank": 32, "scale": 0.2, "mask": {"size": 64}}}]}, seed=4)
other = P.Context(layered, context_len=96)
result = [stand_in.recorded_weights(s) for s in of_llama], stand_in.recorded_weights(P.lib().lcu_context_stream(other.h))
""")
    dim, ffn = 256, 768
    assert weights[0] == 4 * [2 * (2 * (4 * dim * dim + 3 * dim * ffn) + 512 * dim)]
    assert weights[1] > 2 * (301 * 64 + 3 * 64 * 128)
