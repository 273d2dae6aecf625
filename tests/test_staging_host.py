"""How often a step's metadata asks for host memory to travel through."""
import torch

from helpers import make_model_folder, random_tokens
from torch_ops import TorchOps

from lmsf_amd.engine import StepEntry, load_engine_core


def test_the_first_steps_share_one_allocation_and_longer_ones_are_seldom(tmp_path, monkeypatch):
    folder, cfg = make_model_folder(tmp_path, "B")
    core = load_engine_core(folder, dtype="float32", block_size=4, num_pages=4000, device="cpu", ops=TorchOps(), max_num_seqs=16)
    taken, empty = [], torch.empty

    def counting(*args, **kw):
        if "pin_memory" in kw:
            taken.append(args)
        return empty(*args, **kw)
    monkeypatch.setattr(torch, "empty", counting)
    tokens = random_tokens(60, cfg.vocab_size, 1)
    for at in range(0, 60, 10):
        core.executor.step([StepEntry("r", tokens[at:at + 10], [9])])
    assert len(taken) == 1
    core.executor.release("r")
    for n in range(50, 74, 4):                  # every step needs a little more than the one before
        entries = [StepEntry("s%d" % i, random_tokens(n, cfg.vocab_size, n + i), []) for i in range(16)]
        core.executor.step(entries)
        for e in entries:
            core.executor.release(e.request_id)
    assert len(taken) == 2
