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
