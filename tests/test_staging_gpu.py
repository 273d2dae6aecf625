"""Steps launched one after another without a wait between them."""
import pytest
import torch

from helpers import make_model_folder, random_tokens

pytestmark = pytest.mark.gpu


def test_steps_one_after_another_without_a_wait(tmp_path):
    """The host fills the next steps' metadata while earlier steps are still running: the logits are those of steps
    with a wait after each, for single tokens (captured steps) and portions of prompts."""
    from lmsf_amd.engine import StepEntry, load_engine_core
    folder, cfg = make_model_folder(tmp_path, "W", dtype="bfloat16")
    prompts = [random_tokens(n, cfg.vocab_size, n) for n in (25, 70, 33)]
    steps = [[("r%d" % i, p[:3]) for i, p in enumerate(prompts)]]
    for at in range(3, 25):
        steps.append([("r%d" % i, p[at:at + 1]) for i, p in enumerate(prompts)])
    for at in range(25, 30):                      # portions beside single tokens
        steps.append([("r1", prompts[1][25 + 5 * (at - 25):30 + 5 * (at - 25)]), ("r2", prompts[2][at:at + 1])])

    def run(wait):
        core = load_engine_core(folder, dtype="bfloat16", num_pages=64, max_num_seqs=4)
        out = []
        busy = torch.ones(4096, 4096, device="cuda:0")
        for step in steps:
            if not wait:
                busy = busy @ busy * 2.0 ** -12       # the GPU falls behind the host
            out.append(core.executor.step([StepEntry(r, t, [len(t) - 1]) for r, t in step]))
            if wait:
                torch.cuda.synchronize()
        return torch.cat(out).cpu()
    assert torch.equal(run(True), run(False))
