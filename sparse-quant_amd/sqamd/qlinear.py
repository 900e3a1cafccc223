"""WALinear: the quantized linear module the model files instantiate.

Mirror of the reference's module (test/muxi/module/qlinear/qlinear.py:8-106 and
test/nvidia/module/qlinear/qlinear.py:10-92): same constructor arguments, the same
buffer names, shapes and dtypes (so a state_dict saved by the reference loads
unchanged), the same forward contract `gemm_awq_ut(x, weight, zeros_scales, ...) +
bias` (the bias add is folded into the kernel; `forward` also takes an optional
residual and activation for the decoder layer's fused tails).  `layout` selects which of the reference's two buffer conventions is used:

    "l1" (default)  weight uint8 [N, K*w_bit/8], zeros_scales fp16 [N, 2K/g], g default 64
    "l2"            weight int32 [K, N*w_bit/32], zeros_scales fp16 [K/g, 2N], g default 128
"""
import torch
from torch import nn

import quant
from . import quant_funcs


class WALinear(nn.Module):
    def __init__(self, in_features, out_features, w_config=None, a_config=None, w_bit=4, a_bit=16,
                 group_size=None, bias=True, quantize_output=False, dev="cuda", dtype=None, layout="l1"):
        super().__init__()
        self._describe(in_features, out_features, w_config, a_config, w_bit, a_bit, group_size, quantize_output, layout)
        g = self.group_size
        if layout == "l1":
            self.register_buffer("zeros_scales", torch.zeros(out_features, in_features * 2 // g,
                                                             dtype=torch.float16, device=dev))
            self.register_buffer("weight", torch.zeros(out_features, in_features * w_bit // 8,
                                                       dtype=dtype or torch.uint8, device=dev))
        else:
            self.register_buffer("zeros_scales", torch.zeros(in_features // g, out_features * 2,
                                                             dtype=torch.float16, device=dev))
            self.register_buffer("weight", torch.zeros(in_features, out_features * w_bit // 32,
                                                       dtype=dtype or torch.int32, device=dev))
        if bias:
            self.register_buffer("bias", torch.zeros((1, out_features), dtype=torch.float16, device=dev))
        else:
            self.register_buffer("bias", None)

    def _describe(self, in_features, out_features, w_config, a_config, w_bit, a_bit, group_size, quantize_output, layout):
        if layout not in ("l1", "l2"):
            raise ValueError("layout must be 'l1' or 'l2'")
        # (plain values: nn.Module's attribute hook has nothing to sort them into and costs a microsecond each)
        self.__dict__.update(in_features=in_features, out_features=out_features, w_config=w_config, a_config=a_config,
                             w_bit=w_bit, a_bit=a_bit, layout=layout, quantize_output=quantize_output,
                             group_size=group_size if group_size is not None else (64 if layout == "l1" else 128))

    def forward(self, x, residual=None, act="none", pre_ln=None):
        """y = act(x W_hat^T + bias) + residual.  With the defaults this is the reference's
        forward (gemm_awq_ut, then + bias); bias, activation and residual all ride in the
        kernel's store instead of separate element-wise launches.  pre_ln: an nn.LayerNorm (or
        any object with weight, bias, eps) applied to x first, inside the same kernel where the
        shape allows (up to 8 tokens, group size 128, 2048 < K <= 4096)."""
        buffers = self._buffers  # (a look-up through the module costs four times as much, three times a call)
        weight = buffers.get("weight")
        zeros_scales = buffers.get("zeros_scales")
        if weight is None or zeros_scales is None:
            weight, zeros_scales = self.weight, self.zeros_scales
        bias = buffers["bias"] if "bias" in buffers else self.bias
        if self.w_bit == 2:
            # uint8 [N, K/4] or int32 [K, N/16] -> the 4-bit words of the same layout, as the
            # reference's forward does on every call (test/muxi/module/qlinear/qlinear.py:61-62,
            # test/nvidia/module/qlinear/qlinear.py:58-61).
            # The int32 expansion is kept while the stored words do not change, so that the
            # one-time conversion of that layout behind gemm_awq_ut is not repeated per call.
            if self.layout == "l1":
                weight = quant.convert_2bit_to_4bit(weight)
            else:
                key = (weight.data_ptr(), weight._version)
                if getattr(self, "_expanded_key", None) != key:
                    self._expanded = quant.convert_2bit_to_4bit(weight)
                    self._expanded_key = key
                weight = self._expanded
        if pre_ln is None:
            return quant.walinear_forward(x, weight, zeros_scales, bias, residual, act, self.out_features,
                                          self.group_size, False, None, None, 0.0)
        if self.layout != "l1":
            raise NotImplementedError("pre_ln is supported in layout 'l1' only")
        return quant.walinear_forward(x, weight, zeros_scales, bias, residual, act, self.out_features, self.group_size,
                                      True, pre_ln.weight, pre_ln.bias, pre_ln.eps)

    @staticmethod
    def from_float(module, w_config, a_config=None, quantize_output=False, layout="l1"):
        assert isinstance(module, nn.Linear)
        n_bit, g = w_config["n_bit"], w_config["group_size"]
        # The buffers are registered as they will be, not as the constructor's zeros: those, on the meta device, and
        # replacing them took most of the call's host time (1280 x 1472: 46 -> 16 us a call with the packer in the extension).
        new = WALinear.__new__(WALinear)
        nn.Module.__init__(new)
        new._describe(module.in_features, module.out_features, w_config, a_config, n_bit, 16, g, quantize_output, layout)
        if layout == "l1":
            weight, zeros_scales = quant_funcs.quant_muxi(module.weight.data, module.in_features, module.out_features,
                                                          n_bit=n_bit, group_size=g)
        else:
            weight, zeros_scales, _ = quant_funcs._lmdeploy(module.weight.data, module.in_features, module.out_features, g,
                                                            n_bit, want_fake=False)
        new.register_buffer("zeros_scales", zeros_scales)
        new.register_buffer("weight", weight)
        new.register_buffer("bias", None if module.bias is None else module.bias.data.half().unsqueeze(0))
        return new

    def __repr__(self):
        return "W{}A{}Linear({}, {})".format(self.w_bit, self.a_bit, self.in_features, self.out_features)
