"""A per-layer input of the token: the stream gates a slice of a second embedding of the token, and the projected result
is normed and added to the stream."""
import torch
from torch import nn

from .. import _lib
from .decoder_ops import ADD_NORMED, linear, residual_norm, token_gate


class TokenSideInput(nn.Module):

    ONE_LAUNCH_ROWS = 2     # in widths: fewer rows do not fill the chip with the one-launch kernel's workgroups

    def __init__(self, width: int, dim: int, column0: int, dtype):
        super().__init__()
        self.column0 = column0
        self.gate = nn.Parameter(torch.zeros(dim, width, dtype=dtype), requires_grad=False)
        self.proj = nn.Parameter(torch.zeros(width, dim, dtype=dtype), requires_grad=False)
        self.norm = nn.Parameter(torch.ones(width, dtype=torch.float32), requires_grad=False)
        for name in ("gate_packed", "proj_packed"):      # in operand order; they move with the module and are not saved
            self.register_buffer(name, None, persistent=False)

    def finish_loading(self) -> None:
        """Forms of the weights that the one-launch kernel reads: pieces of 16 rows x 32 columns, each as an MFMA takes it, so
        that a wave loads 1 KB that lies whole."""
        dim, W = self.gate.shape
        if self.gate.dtype == torch.bfloat16 and _lib.load_decoder().ed_token_side_packable(W, dim):
            pieces = lambda w: w.data.view(w.shape[0] // 16, 16, w.shape[1] // 32, 4, 8).permute(0, 2, 3, 1, 4)
            self.gate_packed, self.proj_packed = pieces(self.gate).transpose(0, 1).contiguous(), pieces(self.proj).contiguous()

    def forward(self, x: torch.Tensor, tokens: torch.Tensor, table: torch.Tensor) -> torch.Tensor:
        """x [T, width] (the stream in the compute type) -> what is to be normed with ``norm`` and added."""
        return linear(token_gate(x, self.gate, tokens, table, self.column0), self.proj)

    def close_layer(self, x: torch.Tensor, y: torch.Tensor, post_w: torch.Tensor, tokens: torch.Tensor, table: torch.Tensor,
                    eps: float, out: torch.Tensor, next_w) -> None:
        """Everything from the feed-forward's result ``y`` to the next layer's input: the stream ``x`` takes the normed y,
        then the token's input; ``out`` (rows may be strided) = x / rms(x) * next_w, or x.  One launch for a bfloat16
        prompt of a width its kernel takes; a few rows are better spread over the chip in four."""
        T, W = x.shape
        lib, dim = _lib.load_decoder(), self.gate.shape[0]
        if T >= self.ONE_LAUNCH_ROWS * W and y.dim() == 2 and y.dtype == torch.bfloat16 and out.stride(0) % 4 == 0 and lib.ed_token_side_supported(W, dim) == 1:
            packed = self.gate_packed is not None
            gate, proj = (self.gate_packed, self.proj_packed) if packed else (self.gate, self.proj)
            run = lib.ed_token_side_packed if packed else lib.ed_token_side
            code = run(x.data_ptr(), y.data_ptr(), post_w.data_ptr(), gate.data_ptr(), proj.data_ptr(), tokens.data_ptr(),
                       table.data_ptr(), table.stride(0), self.column0, self.norm.data_ptr(), None if next_w is None else next_w.data_ptr(),
                       out.data_ptr(), out.stride(0), T, W, dim, float(eps), _lib.current_stream(x.device))
            _lib.check_decoder(code, "token_side")
            return
        rows = torch.empty(T, W, dtype=out.dtype, device=x.device)
        residual_norm(ADD_NORMED, x, y, post_w, eps, rows)
        residual_norm(ADD_NORMED, x, self(rows, tokens, table), self.norm, eps, out, next_w)
