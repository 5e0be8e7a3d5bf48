// MI355X (gfx950) kernels and C ABI of the workspace transformer branch around the LTHC interface: RMSNorm +
// modulate with its gated forms, the q/k norm + RoPE, the attention and the SwiGLU gate.  Declarations are in
// include/lthc.h; the interface itself is lthc_kernels.hip.

#include "common.inc"

// RMSNorm + modulate (the decoder's input and the branch's pre-norms) with its gated forms.
#include "norm_modulate.inc"
#include "branch_ops.inc"
// Backward of the elementwise ops.
#include "branch_backward.inc"
// Fused q/k RMSNorm + RoPE and attention of the branch (matrix cores).
#include "attention.inc"
// The attention's backward.
#include "attention_backward.inc"
// Weight and bias gradients of the linear layers over many rows.
#include "linear_weight_grad.inc"
