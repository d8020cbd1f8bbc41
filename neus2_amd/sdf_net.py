"""The SDF network with its eikonal second-order path, composed from the encoding and the MLP the way
NerfNetwork does it (nerf_network.h:184-234 forward and normals, :402-429 first-order backward, :534-571
second-order backward), without the colour branch:

    input  = [x - 0.5 | grid(x) | 0]                (48 rows)
    sdf    = MLP(input)[0],   normal = d sdf / d x = dy_dx^T g[3:35] + g[0:3],  g = d sdf / d input
    loss   = mean |sdf| + w_ek * mean (|normal| - 1)^2

``loss_backward`` leaves d loss / d parameters (times loss_scale) in the gradient buffers of the two objects.
Every arithmetic step runs in the library; torch only owns the buffers,
which are allocated once per batch size.
"""
import ctypes as C

import torch

from . import capi
from .capi import check, ptr
from .tcnn_api import GRAD_OVERWRITE, FullyFusedMLP, GridEncoding, _stream, _stream_address


class SdfNet:
    def __init__(self, n_levels=16, log2_hashmap_size=19, base_resolution=16, per_level_scale=1.447, max_batch=1 << 18):
        self.grid = GridEncoding(n_levels, 2, log2_hashmap_size, base_resolution, per_level_scale)
        self.enc_w = 2 * n_levels
        self.in_w = (3 + self.enc_w + 15) // 16 * 16
        self.mlp = FullyFusedMLP(self.in_w, 1)
        self.grid.reserve_scatter_workspace(max_batch)
        self._n = 0

    def set_params(self, grid_params, grid_grads, mlp_params, mlp_grads):
        self.grid.set_params(grid_params, grid_grads)
        self.mlp.set_params(mlp_params, mlp_grads)

    def _buffers(self, n, device):
        if n != self._n:
            h = lambda rows: torch.empty((rows, n), dtype=torch.float16, device=device)
            f = lambda rows: torch.empty((rows, n), dtype=torch.float32, device=device)
            nb = int(capi.lib().n2_sdf_step_workspace_bytes(C.c_uint32(n)))
            b = dict(input=h(self.in_w), dy_dx=torch.empty((self.enc_w, n, 3), dtype=torch.float32, device=device), output=h(16), dsdf_dinput=h(self.in_w), normal=f(3),
                     dL_doutput=h(16), dL_dnormal=f(3), second_order_input=h(self.in_w), dL_dinput=h(self.in_w),
                     loss=torch.empty(1, dtype=torch.float32, device=device), workspace=torch.empty(nb, dtype=torch.uint8, device=device))
            self._b = (capi.SdfBuffers(workspace_bytes=nb, **{k: t.data_ptr() for k, t in b.items()}), b)
            self._n, self._cleared = n, False
        if not self._cleared:
            check(capi.lib().n2_sdf_clear_padding(_stream(), C.c_uint32(n), C.c_uint32(self.enc_w), C.c_uint32(self.in_w), C.byref(self._b[0])), "n2_sdf_clear_padding")
            # (under capture the clearing has only become part of the graph: a call outside it may come before the first replay)
            self._cleared = not torch.cuda.is_current_stream_capturing()
        return self._b

    def forward(self, x, ek_weight=0.1, loss_scale=128.0):
        """x fp32 [3, N].  Returns a context dict with sdf (fp16 [N]), normal (fp32 [3, N]), the loss (one-element device
        tensor) and what backward needs.  The tensors are the net's own buffers: they are overwritten by the next
        forward of the same batch size."""
        n = x.shape[1]
        own, b = buffers = self._buffers(n, x.device)
        check(capi.lib().n2_sdf_forward_and_loss(self.grid._h, self.mlp._h, _stream_address(), x.data_ptr(), 1, n, n, ek_weight, loss_scale, C.byref(own)), "n2_sdf_forward_and_loss")
        return dict(x=x, inp=b["input"], dy_dx=b["dy_dx"], y=b["output"], g=b["dsdf_dinput"], sdf=b["output"][0], normal=b["normal"], loss=b["loss"],
                    weights=(ek_weight, loss_scale), buffers=buffers)

    def _eikonal(self, ctx, ek_weight, loss_scale):
        """The loss and what backward takes with other weights."""
        n, b = ctx["x"].shape[1], ctx["buffers"][1]
        # normals: encoding backward of d sdf / d encoding without parameter gradients, J^T g (nerf_network.h:230-234)
        check(capi.lib().n2_sdf_normals_and_eikonal_loss(_stream(), C.c_uint32(n), C.c_uint32(self.enc_w), C.c_uint32(self.in_w), ptr(b["output"]),
                                                         ptr(b["dsdf_dinput"]), ptr(b["dy_dx"]), ptr(b["normal"]), C.c_float(ek_weight),
                                                         C.c_float(loss_scale), ptr(b["dL_doutput"]), ptr(b["dL_dnormal"]), ptr(b["second_order_input"]),
                                                         ptr(b["loss"]), ptr(b["workspace"]), C.c_uint64(b["workspace"].numel())),
              "n2_sdf_normals_and_eikonal_loss")
        ctx["weights"] = (ek_weight, loss_scale)

    def loss_backward(self, ctx, ek_weight=0.1, loss_scale=128.0):
        """Returns the loss as a one-element device tensor (no host synchronisation)."""
        x, n = ctx["x"], ctx["x"].shape[1]
        if ctx["weights"] != (ek_weight, loss_scale):
            self._eikonal(ctx, ek_weight, loss_scale)
        # both orders through the MLP in one pass (the second's first-order output gradient was e_0), then both through the grid;
        # the grid's dL_ddLdoutput (rows 3.. of the MLP's second-order input) was already formed from the saved Jacobian with
        # the loss
        check(capi.lib().n2_sdf_loss_backward(self.grid._h, self.mlp._h, _stream_address(), x.data_ptr(), 1, n, n, C.byref(ctx["buffers"][0]),
                                              GRAD_OVERWRITE), "n2_sdf_loss_backward")
        return ctx["loss"]
