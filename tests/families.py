"""Which family of kernels a problem runs on (s2attn_attention_family), for tests that mean to reach a certain one."""

import ctypes

import torch


def families(dtype, batch, num_heads, ck, cv, in_shape, out_shape, col_idx, row_off, alignment=16):
    """Names of the families of the forward, the dq and the dk/dv pass."""
    from torch_harmonics_amd import _lib
    from torch_harmonics_amd.plan import build_host_blob

    plan = build_host_blob(col_idx, row_off, *in_shape, *out_shape)
    code = {torch.float32: _lib.S2ATTN_F32, torch.bfloat16: _lib.S2ATTN_BF16, torch.float16: _lib.S2ATTN_F16}[dtype]
    shape = _lib.ShapeStruct(batch, num_heads, *in_shape, *out_shape, ck, cv, code)
    lib = _lib.load()
    return tuple(_lib.FAMILIES[_lib.check(lib.s2attn_attention_family(i, ctypes.byref(plan.struct), ctypes.byref(shape), alignment), "family")] for i in range(3))
