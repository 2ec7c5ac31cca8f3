"""What the Qwen-Image loop hands the model as its timestep: the bits of the expression of one step, however the steps are given."""

import pytest
import torch

from vllm_omni_amd import denoise


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form", ["tensor", "list", "float64", "integers"])
@pytest.mark.parametrize("entries", [1, 2])
def test_every_step_gets_its_timestep(dtype, form, entries):
    seen = []

    class Pipe(denoise.QwenImageCFGParallelMixin):
        def predict_noise(self, **kw):
            seen.append(kw["timestep"].clone())
            return torch.zeros_like(kw["hidden_states"])

    class Scheduler:
        def set_begin_index(self, i):
            pass

        def step(self, noise, t, latents, return_dict=False):
            return (latents,)

    pipe = Pipe()
    pipe.transformer, pipe.scheduler = torch.nn.Identity(), Scheduler()
    steps = torch.tensor([1000.0, 937.31, 500.123, 3.7, 0.0])
    steps = {"tensor": steps, "list": list(steps), "float64": steps.double(), "integers": steps.long()}[form]
    latents = torch.zeros(entries, 4, 2, dtype=dtype)
    pipe.diffuse(torch.zeros(entries, 3, 2), None, None, None, latents, [], [3], None, steps, False, None, 1.0)
    assert len(seen) == 5
    for t, got in zip(steps, seen):
        want = t.expand(entries).to(dtype=dtype) / 1000
        assert got.shape == (entries,) and got.dtype == dtype and torch.equal(got, want)
