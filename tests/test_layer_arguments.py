"""A layer hands every argument of a call to the method that it was made with or given (CPU)."""

import pytest

from vllm_omni_amd import kernels
from vllm_omni_amd.layers.adalayernorm import AdaLayerNorm
from vllm_omni_amd.layers.rmsnorm import RMSNorm
from vllm_omni_amd.layers.rope import RotaryEmbedding


@pytest.mark.parametrize("kind,made_with", [(RMSNorm, (64,)), (RotaryEmbedding, ()), (AdaLayerNorm, (64,))])
def test_further_arguments(kind, made_with):
    kernels.native()

    class Mine(kind):
        def forward_hip(self, *args, **kwargs):
            return args, kwargs
    given = kind(*made_with)
    given._forward_method = lambda *args, **kwargs: (args, kwargs)
    for layer in (Mine(*made_with), given):
        for args, kwargs in (((), {}), ((1,), {}), ((1, 2, 3, 4), {}), ((1,), {"residual": 2}), ((), {"x": 1}), ((1, 2, 3, None), {"out": 5})):
            assert layer(*args, **kwargs) == (args, kwargs)
    with pytest.raises(TypeError):
        kind(*made_with)()
