"""The pose network over batches that leave every kind of remainder in its GEMM
tiles, split sums, operand staging and im2col vectors, against the FP64 oracle
on the same bf16-rounded operands (tolerances: tests/test_gpu_posenet.py)."""
import numpy as np
import pytest

from test_gpu_posenet import FWD_TOL, GRAD_TOL, random_pairs, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 2, 3, 13, 33])
def test_forward_and_gradients_over_batches(torch_gpu, batch):
    from kinectfusion_amd import posenet as PN
    from oracle import posenet_oracle as P

    net = PN.PoseNet(PN.PoseNetConfig(batch_capacity=batch, seed=batch))
    raw, dev, targets, tdev = random_pairs(torch_gpu, batch, seed=batch)
    params, inputs = net.parameters().astype(np.float64), P.inputs_from_pairs(raw)
    ref, _ = P.forward(params, inputs, emulate_bf16=True)
    assert rel(net.forward(dev).cpu().numpy(), ref * P.OUT_SCALE) < FWD_TOL
    loss, grads = net.gradients(dev, tdev)
    ref_loss, ref_grads = P.loss_and_grad(params, inputs, targets, emulate_bf16=True)
    assert abs(loss - ref_loss) <= 1e-3 * ref_loss
    off = 0
    for _, cin, cout, hin, win, hout, wout, fan in P.layer_shapes():
        for n in (cout * fan, cout):
            assert rel(grads[off: off + n], ref_grads[off: off + n]) < GRAD_TOL
            off += n
    net.close()
