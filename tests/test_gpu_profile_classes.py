"""tg_profile_step books what a step launches under what it is for: where the norm's ranges are a launch of their own, that launch
is the optimizer's, not the weight gradients' (whose work bench.py divides by their time)."""
import numpy as np
import pytest

from turbogpt_amd.bridge import ModelConfig, Native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("context,batch,optimizer", [(256, 1, 2),    # small tiles: the ranges are in their launch; AdamW, transposes
                                                     (1024, 8, 3)])  # 256 x 256 tiles: the ranges, then those two
def test_launches_by_class(context, batch, optimizer):
    with Native(ModelConfig(d_model=256, depth=2, ffn=1024, context=context, batch=batch, clip=1.0)) as engine:
        engine.set_weights((np.random.default_rng(1).standard_normal(engine.count) * 0.02).astype(np.float32))
        engine.set_data(np.arange(4096, dtype=np.uint32).astype(np.uint8))
        launches = {name: count for name, (_, count) in engine.profile_step().items()}
    assert launches["gemm_wgrad"] == 1 and launches["optimizer"] == optimizer
