"""tgk_w16_forward and tgk_w16_backward on teams and on lone waves, on either side of the line between them (1024 teams on 256
compute units): a sequence's logits do not depend on which, nor on whether a gradient is wanted, bit for bit.  Values and gradients
of both against the oracle: test_gpu_width16_blocks."""
import numpy as np
import pytest
import torch

from gpu_util import check, library, stream, sync
from test_gpu_width16 import reference_style_weights
from test_gpu_width16_shapes import run

pytestmark = pytest.mark.gpu


def forward(depth, context, batch, flat, x, y):
    lib = library()
    bits = torch.from_numpy(flat.view(np.int32))
    hi, lo = (half.to(torch.int16).cuda() for half in (bits >> 16, bits & 0xffff))
    tokens, targets = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    workspace = torch.full((lib.tgk_w16_workspace(depth, batch, context),), 255, dtype=torch.uint8, device="cuda")
    losses, logits = torch.empty(batch * context, device="cuda"), torch.empty(batch * context, 256, device="cuda")
    check(lib.tgk_w16_forward(stream(), depth, batch, context, hi.data_ptr(), lo.data_ptr(), tokens.data_ptr(),
                              targets.data_ptr(), workspace.data_ptr(), losses.data_ptr(), logits.data_ptr(), 0))
    sync()
    return logits.cpu().numpy().reshape(batch, context, 256), losses.cpu().numpy()


@pytest.mark.parametrize("depth,context,batch", [(2, 8, 2048), (2, 8, 2049),  # the last on teams, the first on lone waves
                                                 (8, 4, 4097), (3, 5, 3073),  # lone waves with sixteen and fifteen tokens
                                                 (1, 8, 5121),                # ten a unit: blocks of six, with gradient of four
                                                 (1, 8, 8197)])               # sixteen and one: three blocks of six a unit
def test_passes(depth, context, batch):
    flat = reference_style_weights(depth)
    rng = np.random.default_rng(batch)
    x, y = (rng.integers(0, 256, (batch, context), dtype=np.uint8) for _ in range(2))
    logits, losses, gradient = run(depth, context, batch, flat, x, y)
    for got, want in zip(forward(depth, context, batch, flat, x, y), (logits, losses)):
        np.testing.assert_array_equal(got, want)
    for got, want in zip(run(depth, context, batch, flat, x, y, 4), (logits, losses, gradient)):  # weights on an 8-byte boundary
        np.testing.assert_array_equal(got, want)
    few = slice(batch - 40, batch)
    np.testing.assert_array_equal(run(depth, context, 40, flat, x[few], y[few])[0], logits[few])
