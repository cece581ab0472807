"""Decode GEMV call surface (the reference's e2e/sc_decode.py) on torch tensors over libscmx.so.

`gemv` keeps the reference's signature; `rows` / `vpl` / `nsg` / `splitk` are accepted as hints (the kernel picks its
own launch shape and the result never depends on it).  New here: a 2-D `xq` [B, K] without `eidx` runs B input rows
against one pass over the weights (up to 8 rows) and returns [B, N]."""
import torch

from . import _lib
from . import sc_format as F
from . import sc_kernels as S

GEMV_TILE = (4, 16, 2)
GEMV_TILES = {}


def gemv(xq, codes, bcodes, xscale, wscale, N, epi, dtype=torch.bfloat16, res=None, nsg=None, eidx=None, xstride=0,
         pro=0, nw=None, eps=None, rows=None, vpl=None, shared=None, splitk=None, fmt=None):
    """W4A8 GEMV.  pro=0: xq int8 [K] (or rows) with xscale; pro=1: xq is a bf16 row quantized in the kernel;
    pro=2: RMSNorm(nw, eps) + INT8 in the kernel.  Output EPI 1: [N]; 2: [N] = res + y; 3: [N/2].
    xq [B, K] with B = 2 ... 8 rows shares one pass over the weights (more than 8 rows take one pass per eight -- from a few
    dozen rows on the dense GEMM is the faster path).
    MoE (eidx int32 [S]): codes [E, ..], wscale [E, N]; slot j uses expert eidx[j] and input row j if xstride=1;
    shared=e adds one slot for expert e -> [S(+1), N or N/2]."""
    if dtype is not torch.bfloat16:
        S._check_dtype(dtype)
    fmt = fmt or F.DEFAULT
    # one native call where every operand is a plain tensor; None: what follows converts or refuses what is not
    out = _lib.native().gemv(fmt.c, xq, xscale, codes, bcodes, wscale, N, epi, res, eidx, xstride, shared, pro, nw, eps)
    if out is not None:
        return out
    K = xq.shape[-1]
    no = N // 2 if epi == 3 else N
    batch, nslot = 1, 0
    if eidx is not None:
        nslot = eidx.numel()
        slots = nslot + (shared is not None)
        eidx = eidx if eidx.dtype == torch.int32 else eidx.view(torch.int32) if eidx.element_size() == 4 else eidx.to(torch.int32)
        out = _lib.native().empty_bf16(xq, slots, no)
    elif xq.dim() == 2 and xq.shape[0] > 8:   # more rows than one pass takes: eight at a time
        cut = lambda t, i: None if t is None else t[i:i + 8]   # noqa: E731
        return torch.cat([gemv(xq[i:i + 8], codes, bcodes, cut(xscale, i), wscale, N, epi, dtype, cut(res, i), nsg, None,
                               xstride, pro, nw, eps, rows, vpl, shared, splitk, fmt).reshape(-1, no)
                          for i in range(0, xq.shape[0], 8)])
    elif xq.dim() == 2 and xq.shape[0] > 1:
        batch = xq.shape[0]
        out = _lib.native().empty_bf16(xq, batch, no)
    else:
        out = _lib.native().empty_bf16(xq, no)
    assert (pro == 0 and xq.dtype == torch.int8) or (pro in (1, 2) and xq.dtype == torch.bfloat16)
    nat = _lib.native()
    xscale = xscale if pro == 0 else None
    res = res if epi == 2 else None
    if batch in (3, 5, 6, 7):   # counts between the kernels' sizes come from any layout
        xq, xscale, res = (None if t is None else t.contiguous() for t in (xq, xscale, res))
    nw, eps = (nw, S._eps(eps)) if pro == 2 else (None, 0.0)
    if eidx is None:
        need = nat.scmx_gemv_rows_workspace(fmt.c, pro, batch, N, K) if batch > 1 else 0
        nat.scmx_gemv_rows(fmt.c, xq, xscale, codes, bcodes, wscale, res, out, epi, pro, nw, eps, batch, N, K,
                           nat.empty_u8(xq, need) if need else None, need)
    else:
        nat.scmx_gemv(fmt.c, xq, xscale, codes, bcodes, wscale, res, out, epi, pro, nw, eps, batch, N, K, eidx, nslot, xstride,
                      -1 if shared is None else int(shared))
    return out
