"""Per-channel arguments of the fused epilogue are held against the layer before any kernel reads them
(host only)."""
import pytest
import torch

from sparsetriton_amd.nn.functional.conv.funcs.implicit_precomputed_gemm import conv_forward_epilogue

C = 8


def _bn(**kw):
    d = {"weight": torch.ones(C), "bias": torch.zeros(C), "mean": torch.zeros(C), "var": torch.ones(C), "eps": 1e-5}
    d.update(kw)
    return tuple(d.values())


@pytest.mark.parametrize("bias,scale,shift,bn,match", [
    (None, None, None, _bn(weight=torch.ones(C - 1)), "bn weight"),
    (None, None, None, _bn(bias=torch.ones(1)), "bn bias"),
    (None, None, None, _bn(mean=torch.ones(2 * C)), "running_mean"),
    (None, None, None, _bn(var=torch.ones(0)), "running_var"),
    (None, None, None, _bn(var=torch.ones(C, device="meta")), "running_var"),
    (None, None, None, _bn(mean=None), "needs running_mean"),
    (None, None, None, _bn(var=None), "needs running_mean"),
    (None, torch.ones(C), None, _bn(), "either bn or scale"),
    (None, None, torch.ones(C), _bn(), "either bn or scale"),
    (None, torch.ones(C - 1), None, None, "scale"),
    (None, torch.ones(C), torch.ones(1), None, "shift"),
    (torch.ones(C - 1), None, None, None, "bias"),
    (torch.ones(C, device="meta"), None, None, None, "bias"),
])
def test_wrong_channel_terms_are_refused(bias, scale, shift, bn, match):
    with pytest.raises(ValueError, match=match):
        conv_forward_epilogue(torch.zeros(3, 4), torch.zeros(27, 4, C), None, bias, scale, shift, None, False, bn=bn)


@pytest.mark.parametrize("bn", [_bn(), _bn(weight=None, bias=None), None])
def test_right_channel_terms_reach_the_device_check(bn):
    scale = None if bn is not None else torch.ones(C)
    with pytest.raises(RuntimeError, match="must live on the GPU"):
        conv_forward_epilogue(torch.zeros(3, 4), torch.zeros(27, 4, C), None, torch.zeros(C), scale, None, None, True, bn=bn)
