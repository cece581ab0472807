"""Dense prefill call surface: the function names, argument order and defaults of the reference's e2e/sc_kernels.py,
on torch (ROCm) tensors, backed by the HIP kernels of libscmx.so through its C ABI.

Conventions kept from the reference (e2e/sc_kernels.py:15-17): kernels take M rows and write Mp >= M rows, rows >= M
are zero; `deps` is accepted and ignored (it only ordered MLX's lazy graph — HIP streams are already ordered);
`tile` / `nt` are accepted as hints and never change a result.  `eps` may be a float or a 1-element tensor.

Difference by design: `unpack_i8` may return a `PackedWq` handle instead of an INT8 tensor (FUSE_UNPACK, default on).
`mm_epi` / `mm_i8_i32` given that handle run the GEMM whose workgroups unpack their weight tile in LDS, so the INT8
weights are never written to memory; `handle.materialize()` (or lazy=False) gives the reference's INT8 tensor.
"""
import numpy as np
import torch

from . import _lib
from . import sc_format as F

TM, TN, NSG, GROUP_M = 128, 64, 4, 8     # the reference's default tile (kept for pad_rows and as accepted hints)
FUSE_UNPACK = True


def set_format(fmt):
    """Switch the default weight format of every wrapper (the C ABI itself takes the format per call)."""
    F.DEFAULT = fmt


def pad_rows(M):
    return -(-M // TM) * TM


def _eps(eps):
    return float(eps) if not torch.is_tensor(eps) else float(eps.reshape(-1)[0].item())


def _check_dtype(dtype):
    if dtype not in (torch.bfloat16, None):
        raise ValueError("the kernels emit bfloat16 (the reference's model dtype)")


class PackedWq:
    """Packed weights standing in for the INT8 tensor unpack_i8 would produce."""

    def __init__(self, codes, bcodes, N, K, fmt, wscale=None):
        self.codes, self.bcodes, self.N, self.K, self.fmt = codes, bcodes, N, K, fmt
        self.wscale = wscale   # a standard MXFP4 tensor read in place decodes with its row scales (F.MXFP4)
        self.shape, self.dtype, self.device = (N, K), torch.int8, codes.device

    def materialize(self):
        return unpack_i8(self.codes, self.bcodes, self.N, self.K, lazy=False, fmt=self.fmt)

    def __getitem__(self, idx):          # row selection / permutation, as callers do on the INT8 tensor
        return self.materialize()[idx]

    def cpu(self):
        return self.materialize().cpu()


def unpack_i8(codes, bcodes, N, K, deps=(), lazy=None, fmt=None, wscale=None):
    """Packed codes (flat, 4-byte ints) + block codes uint8 [N, ..] -> INT8 [N, K].  fmt=F.MXFP4 (E8M0 bytes as block
    codes) exists as the lazy handle only and takes the row scales along (F.mxfp4_row_scales)."""
    fmt = fmt or F.DEFAULT
    if fmt.e8m0 and wscale is None:
        raise ValueError("the MXFP4 form decodes with its row scales: pass wscale=sc_format.mxfp4_row_scales(e8m0)")
    if FUSE_UNPACK if lazy is None else lazy:
        return PackedWq(codes, bcodes, N, K, fmt, wscale)
    assert codes.numel() * codes.element_size() == N * K // 2, "codes must hold N*K/2 bytes"
    wq = _lib.native().empty_i8(codes, N, K)
    _lib.native().scmx_unpack_i8(fmt.c, codes, bcodes, wq, N, K)
    return wq


def act_quant(x, Mp=None, nt=256, deps=()):
    """Per-token symmetric INT8: x bf16 [M, K] -> (xq int8 [Mp, K], xscale f32 [Mp]); rows >= M zero."""
    M, K = x.shape
    Mp = Mp or pad_rows(M)
    assert x.dtype == torch.bfloat16
    xq = _lib.native().empty_i8(x, Mp, K)
    xs = _lib.native().empty_f32(x, Mp)
    _lib.native().scmx_act_quant(x, xq, xs, M, Mp, K)
    return xq, xs


def rot_signs(K):
    """The sign vector of the block rotation for input width K (one per width, so q/k/v and gate/up share a rotated
    input); e2e/sc_kernels.py:566-569."""
    return torch.from_numpy(np.random.default_rng(0).choice([-1.0, 1.0], size=K).astype(np.float32)).cuda()


def rot_quant(x, signs, Mp=None, nt=512, deps=()):
    """x bf16 [M, K] -> (xq int8 [Mp, K], xscale f32 [Mp]): randomized Hadamard rotation of each 32-wide block, then
    per-token INT8 (e2e/sc_kernels.py:571-582)."""
    M, K = x.shape
    Mp = Mp or pad_rows(M)
    assert x.dtype == torch.bfloat16 and signs.dtype == torch.float32 and signs.numel() == K
    xq = _lib.native().empty_i8(x, Mp, K)
    xs = _lib.native().empty_f32(x, Mp)
    _lib.native().scmx_rot_quant(x, signs, xq, xs, M, Mp, K)
    return xq, xs


def _gemm(xq, wq, xscale, wscale, epi, res):
    (M, K), N = xq.shape, wq.shape[0]
    assert xq.dtype == torch.int8 and wq.shape[1] == K
    blocked = isinstance(xq, BlockedXq)
    like = xq.data if blocked else xq
    if epi == 0:
        out = _lib.native().empty_i32(like, M, N)
    else:
        out = _lib.native().empty_bf16(like, M, N // 2 if epi == 3 else N)
    if epi == 2:
        assert res is not None and tuple(res.shape) == (M, N) and res.dtype == torch.bfloat16
    r = res if epi == 2 else None
    if blocked:
        if not isinstance(wq, PackedWq):
            raise ValueError("blocked activations multiply packed weights (unpack_i8's lazy handle)")
        _lib.native().scmx_mm_w4a8_blocked(wq.fmt.c, xq.data, xscale, wq.codes, wq.bcodes,
                                           wscale if wscale is not None else wq.wscale, r, out, epi, M, N, K)
    elif isinstance(wq, PackedWq):
        _lib.native().scmx_mm_w4a8(wq.fmt.c, xq, xscale, wq.codes, wq.bcodes, wscale if wscale is not None else wq.wscale, r,
                                   out, epi, M, N, K)
    else:
        assert wq.dtype == torch.int8
        _lib.native().scmx_mm_epi(xq, wq, xscale, wscale, r, out, epi, M, N, K)
    return out


def mm_i8_i32(xq, wq, deps=(), tile=None):
    """INT8 [M, K] x INT8 [N, K]^T -> INT32 [M, N] (wq: INT8 tensor or PackedWq)."""
    return _gemm(xq, wq, None, None, 0, None)


def mm_epi(xq, wq, xscale, wscale, epi, dtype=torch.bfloat16, res=None, deps=(), tile=None):
    """INT8 GEMM + in-register epilogue (EPI 1: scaled bf16, 2: + residual, 3: swiglu of interleaved gate/up)."""
    _check_dtype(dtype)
    assert epi in (1, 2, 3)
    return _gemm(xq, wq, xscale, wscale, epi, res)


class BlockedXq:
    """INT8 activations in the blocked layout (act_quant_blocked): what mm_epi / mm_i8_i32 take in place of the [Mp, K]
    tensor when the weights are packed (PackedWq)."""

    def __init__(self, data, M, K):
        self.data, self.shape, self.dtype, self.device = data, (M, K), torch.int8, data.device

    def rows(self):
        """The [Mp, K] tensor act_quant returns (a copy)."""
        Mp, K = self.data.numel() // self.shape[1], self.shape[1]
        return self.data.view(Mp // 32, K // 32, 2, 32, 16).permute(0, 3, 1, 2, 4).reshape(Mp, K)


def act_quant_blocked(x, Mp=None):
    """act_quant for prefill-sized GEMMs on packed weights: the same codes and scales with xq in 32 x 32 blocks in the
    order the MFMA takes them, so that the large GEMM tiles load activation fragments straight from memory
    (scmx_act_quant_blocked / scmx_mm_w4a8_blocked).  -> (BlockedXq, xscale f32 [Mp]), Mp a multiple of 32."""
    M, K = x.shape
    Mp = Mp or pad_rows(M)
    assert x.dtype == torch.bfloat16 and Mp % 32 == 0
    xq = _lib.native().empty_i8(x, Mp * K)
    xs = _lib.native().empty_f32(x, Mp)
    _lib.native().scmx_act_quant_blocked(x, xq, xs, M, Mp, K)
    return BlockedXq(xq, Mp, K), xs   # Mp rows like act_quant's tensor: the padding rows are zeros


def linear_w4a8_workspace(M, K):
    """Bytes of workspace linear_w4a8 needs for M rows of K (the INT8 activations, then their scales)."""
    return int(_lib.load().scmx_linear_w4a8_workspace(M, K))


def linear_w4a8(x, codes, bcodes, wscale, N, epi=1, res=None, fmt=None, workspace=None):
    """One call for a whole W4A8 linear on bf16 activations [M, K]: the activation-quantization prologue and the
    fused-unpack GEMM are enqueued by a single C entry point (scmx_linear_w4a8).  Returns bf16 [M, N or N/2]."""
    fmt = fmt or F.DEFAULT
    M, K = x.shape
    assert x.dtype == torch.bfloat16 and epi in (1, 2, 3)
    need = _lib.native().scmx_linear_w4a8_workspace(M, K)
    if workspace is None or workspace.numel() * workspace.element_size() < need:
        workspace = _lib.native().empty_u8(x, need)
    out = _lib.native().empty_bf16(x, M, N // 2 if epi == 3 else N)
    _lib.native().scmx_linear_w4a8(fmt.c, x, codes, bcodes, wscale, res if epi == 2 else None, out, epi, M, N, K, workspace,
                                   workspace.numel() * workspace.element_size())
    return out


def interleave_gate_up(F_):
    """Row permutation of [gate (F rows); up (F rows)] into groups g_2p, g_2p+1, u_2p, u_2p+1 for EPI 3."""
    p = np.arange(F_ // 2)
    return np.stack([2 * p, 2 * p + 1, F_ + 2 * p, F_ + 2 * p + 1], 1).reshape(-1)


def _rms(x, w, eps, Mp, want_xn, blocked=False):
    M, K = x.shape
    Mp = Mp or pad_rows(M)
    assert x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
    blocked = blocked and Mp % 32 == 0 and K % 512 == 0 and K <= 4096
    xq = _lib.native().empty_i8(x, Mp, K)
    xs = _lib.native().empty_f32(x, Mp)
    xn = _lib.native().empty_bf16(x, Mp, K) if want_xn else None
    quantize = _lib.native().scmx_rmsnorm_quant_blocked if blocked else _lib.native().scmx_rmsnorm_quant
    quantize(x, w, _eps(eps), xq, xs, xn, M, Mp, K)
    if blocked:
        xq = BlockedXq(xq.reshape(-1), Mp, K)   # Mp rows like the tensor it stands for: the padding rows are zeros
    return (xq, xs, xn) if want_xn else (xq, xs)


def rmsnorm_quant(x, w, eps, Mp=None, deps=(), blocked=False):
    """x [M, K] -> (xq int8 [Mp, K], xscale f32 [Mp]) of rms_norm(x, w, eps).  blocked: xq as a BlockedXq (the layout of
    act_quant_blocked) where the shape allows it (Mp % 32 == 0, K % 512 == 0, K <= 4096), by rows otherwise."""
    return _rms(x, w, eps, Mp, False, blocked)


def rmsnorm_quant_n(x, w, eps, Mp=None, deps=(), blocked=False):
    """rmsnorm_quant that also returns the normalized bf16 rows: (xq, xscale, xn [Mp, K])."""
    return _rms(x, w, eps, Mp, True, blocked)


def rmsnorm(x, w, eps):
    """RMSNorm of bf16 rows x [M, K] -> bf16 [M, K] (K % 4 == 0, K <= 16384).  Other shapes, types and layouts, tensors off
    the current device, and callers that differentiate, trace or cast the norm get the array op."""
    if (_plain(x, w) and x.dim() == 2 and w.shape == x.shape[1:] and x.numel() and x.shape[1] % 4 == 0 and x.shape[1] <= 16384
            and not (x.data_ptr() | w.data_ptr()) % 8):
        out = _lib.native().empty_bf16(x, *x.shape)
        _lib.native().scmx_rmsnorm(x, w, _eps(eps), out, *x.shape)
        return out
    return rms_norm(x, w, eps)


def rms_norm(x, w, eps):
    """RMSNorm as array ops, whatever the shape and type."""
    v = x.float()
    return (v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + eps)).to(x.dtype) * w


def linear_bf16(x, w):
    """x w^T of bf16 rows x [M, K] and a bf16 matrix w [N, K] (output head, router) -> bf16 [M, N], sums in float32.  Up to
    16 rows the library's kernel, which reads w once at 5.2-5.8 TB/s, beyond K = 2048 (where the rows' fragments no longer stay
    in registers) for two rows.  The array op's time jumps with the shape.  One row, weights from HBM, calls in a row, us
    kernel / array op: 151936 x 2048 108 / 201, x 2560 141 / 239; 50304 x 2048 38 / 48 (sixteen rows 42 / 48); 32000 x 4096 47 / 55;
    128256 x 4096 174 / 183; a router of 64 x 2048 4.5 / 18.7.  Where it loses: 50304 x 2304 48 / 42, 65536 x 5120 123 / 111, 128256
    x 5120 242 / 223, sixteen rows of 65536 x 1920 48 / 45; a single call waited for costs the array op 14 us more on top.
    Sixteen rows beyond K = 2048: 32000 x 4096 66 / 56, 128256 x 4096 250 / 186.
    More rows, other types and layouts, tensors off the current device, and callers that differentiate, trace or cast the
    product get the array op."""
    if (_plain(x, w) and x.dim() == 2 and w.dim() == 2 and 0 < x.shape[0] <= 16 and w.shape[0]
            and x.shape[1] == w.shape[1] and x.shape[1] and x.shape[1] % 64 == 0
            and (x.shape[1] <= 2048 or x.shape[0] <= 2) and not (x.data_ptr() | w.data_ptr()) % 16):
        out = _lib.native().empty_bf16(x, x.shape[0], w.shape[0])
        _lib.native().scmx_linear_bf16(x, w, out, x.shape[0], w.shape[0], x.shape[1])
        return out
    return x @ w.T


def _plain(x, w):
    """Whether a kernel may stand in for an array op on x and w: contiguous bf16 tensors on the current device (where the
    binding launches) with which torch would do no more than run the op -- no subclass, autograd (reverse or forward),
    functorch, autocast, dispatch or function mode, tracing or compilation."""
    return (type(x) is type(w) is torch.Tensor and x.is_cuda and w.is_cuda
            and x.get_device() == w.get_device() == torch._C._cuda_getDevice() and x.dtype == w.dtype == torch.bfloat16
            and x.is_contiguous() and w.is_contiguous()
            and not (torch.is_autocast_enabled("cuda") or torch.compiler.is_compiling() or torch.jit.is_tracing()
                     or torch._C._functorch.maybe_current_level() is not None
                     or torch.autograd.forward_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack() > 0
                     or torch._C._len_torch_function_stack() > 0 or x.requires_grad or w.requires_grad))


def prefers_blocked(M, N, K):
    """Whether a dense [M, K] x [N, K]^T problem on packed weights runs faster from blocked activations."""
    return bool(_lib.native().scmx_mm_w4a8_prefers_blocked(M, N, K))


def res_norm_quant(acc, xscale, wscale, res, w, eps, deps=()):
    """h = res + bf16(acc * xscale * wscale); returns (h [Mp, K], xq, xscale') of rms_norm(h)."""
    Mp, K = acc.shape
    assert tuple(res.shape) == (Mp, K) and acc.dtype == torch.int32
    h = torch.empty_like(res)
    xq = _lib.native().empty_i8(acc, Mp, K)
    xs = _lib.native().empty_f32(acc, Mp)
    _lib.native().scmx_res_norm_quant(acc, xscale, wscale, res, w, _eps(eps), h, xq, xs, Mp, K)
    return h, xq, xs


def res_epilogue(acc, xscale, wscale, res, deps=()):
    """h = res + bf16(acc * xscale * wscale)."""
    Mp, N = acc.shape
    h = torch.empty_like(res)
    _lib.native().scmx_res_norm_quant(acc, xscale, wscale, res, None, 0.0, h, None, None, Mp, N)
    return h


def swiglu_quant(acc, xscale, wscale, dtype=torch.bfloat16, nt=512, deps=()):
    """acc [Mp, 2F] (gate | up) -> (xq int8 [Mp, F], xscale f32 [Mp]) of swiglu(bf16 gate, bf16 up)."""
    _check_dtype(dtype)
    Mp, F2 = acc.shape
    Fh = F2 // 2
    xq = _lib.native().empty_i8(acc, Mp, Fh)
    xs = _lib.native().empty_f32(acc, Mp)
    _lib.native().scmx_swiglu_quant(acc, xscale, wscale, xq, xs, Mp, Fh)
    return xq, xs


def _headnorm(acc, xscale, wscale, y, qn, kn, eps, L, hq, hk, d):
    like = y if y is not None else acc
    q = _lib.native().empty_bf16(like, hq, L, d)
    k = _lib.native().empty_bf16(like, hk, L, d)
    v = _lib.native().empty_bf16(like, hk, L, d)
    _lib.native().scmx_qkv_headnorm(acc, xscale, wscale, y, qn, kn, _eps(eps), q, k, v, L, hq, hk, d)
    return q, k, v


def qkv_epilogue_headnorm(acc, xscale, wscale, qn, kn, eps, L, hq, hk, d, dtype=torch.bfloat16, deps=()):
    """Qwen3: acc [Mp, (hq + 2 hk) d] -> q [hq, L, d], k [hk, L, d], v [hk, L, d] (q/k per-head RMSNorm)."""
    _check_dtype(dtype)
    return _headnorm(acc, xscale, wscale, None, qn, kn, eps, L, hq, hk, d)


def qkv_headnorm_y(y, qn, kn, eps, L, hq, hk, d, deps=()):
    """Qwen3: bf16 y [Mp, (hq + 2 hk) d] -> q, k, v head-major with per-head RMSNorm of q and k."""
    return _headnorm(None, None, None, y, qn, kn, eps, L, hq, hk, d)


def qkv_headnorm_rope(y, qn, kn, eps, L, hq, hk, d, kcache, vcache, pos, inv_freq, acc=None, xscale=None, wscale=None,
                      token_major=False):
    """qkv_headnorm_y (or, with acc / xscale / wscale, qkv_epilogue_headnorm) fused with the rotary embedding of q
    and k and the KV-cache append: returns q [hq, L, d]; k and v go to rows pos..pos+L-1 of kcache / vcache
    [hk, rows, d].  pos: int, or an int64 device tensor (for graph replay).  token_major=True stores q as [L, hq, d]
    and returns the [hq, L, d] view of it: an attention output that inherits this layout is [L, hq * d] without a
    transposing copy."""
    src = y if y is not None else acc
    q = _lib.native().empty_bf16(src, *((L, hq, d) if token_major else (hq, L, d)))
    assert kcache.shape == vcache.shape and kcache.shape[0] == hk and kcache.shape[2] == d
    assert kcache.dtype == torch.bfloat16 and inv_freq.dtype == torch.float32 and inv_freq.numel() == d // 2
    dev_pos = pos if torch.is_tensor(pos) else None
    assert dev_pos is None or dev_pos.dtype == torch.int64
    _lib.native().scmx_qkv_headnorm_rope(acc, xscale, wscale, y, qn, kn, _eps(eps), q, kcache, vcache, L, hq, hk, d,
                                         inv_freq, dev_pos, 0 if dev_pos is not None else int(pos), kcache.shape[1],
                                         int(token_major))
    return q.transpose(0, 1) if token_major else q


def attn_splits(rows):
    """Row ranges for the decode attention over up to `rows` cache rows and many heads (more than 32): one workgroup per head
    reads a short context fastest, longer ones are cut into 8 ranges, beyond 8192 rows into 16.  A split launch still serves
    contexts of up to 128 rows with one workgroup per head (decided on the device)."""
    return 1 if rows <= 1024 else 8 if rows <= 8192 else 16


def _decode_ranges(rows, hq, hk):
    """The same for any number of heads.  16 heads of 128 over 8 KV heads, attention and merge in a graph, one cache again and again, us
    with 1 / 8 / 16 ranges: 300 rows 6.2 / 6.8 / 6.2, 500 7.6 / 6.6 / 6.3, 1000 11.6 / 7.0 / 6.5, 3000 27 / 9.4 / 7.9; up to 512 rows the
    second launch costs a host-bound loop more than it gives.  32 ranges let the kernel serve two query heads of a KV head from one
    reading of the cache, which it does beyond 3072 rows (up to there it cuts them into 16).  24 caches in turn, as the layers of a
    model read theirs, 16 / 32 ranges: 3200 rows 10.6 / 9.8, 6000 14.5 / 11.6, 12000 21.7 / 15.8; 32 heads 14.0 / 12.6, 19.5 / 15.4, 33.7 /
    20.7; 8 heads 8.8 / 8.7, 11.3 / 10.6, 16.4 / 13.3; 16 heads of 64 8.3 / 8.3, 9.8 / 9.4, 14.1 / 11.6, of 256 15.8 / 12.7, 22.6 /
    16.6, 36.4 / 25.1; groups of four and eight like those of two.  16 ranges stay better up to 5000 rows for 8 heads of 64 (3200 7.5 /
    8.3) and to 8000 where 16 heads share a KV head (32 over 2: 10.9 / 12.4, 13.9 / 15.0, 21.9 / 20.4); with the one cache of a loop in
    the L2 also 16 heads of 128 to 3500 rows, 8 of 128 and 16 of 64 to 6000.
    With the position on the device `rows` is the cache's, and a short context in a longer cache pays for a merge that finds little
    or nothing to do, with 1 / 16 / 32 ranges: 30 rows 4.1 / 5.5 / 5.8, 128 4.7 / 6.2 / 6.1, 300 6.2 / 6.3 / 6.7 (32 heads of 256 - / 7.8 /
    8.7); from about 300 rows on the ranges win."""
    if hq > 32:
        return attn_splits(rows)
    return 1 if rows <= 512 else 16 if rows <= 3072 or hq // hk % 2 else 32


def _split_workspace(splits, hq, d, like):
    return _lib.native().empty_f32(like, splits * hq * (d + 2)) if splits > 1 else None


def attn_decode(q, kcache, vcache, n, scale=None, splits=None):
    """Single-token attention: q bf16 [hq, 1, d] (or [hq, d]) against caches [hk, rows, d] whose first n rows are valid
    (n: int, or an int64 device tensor holding the position n - 1, for graph replay) -> bf16 [1, hq * d].
    splits: row ranges per head (default: by n, or by the cache size when n lives on the device)."""
    hq, d = q.shape[0], q.shape[-1]
    hk, rows, _ = kcache.shape
    out = _lib.native().empty_bf16(q, 1, hq * d)
    dev_pos = n if torch.is_tensor(n) else None
    if splits is None:
        splits = _decode_ranges(rows if dev_pos is not None else int(n), hq, hk)
    work = _split_workspace(splits, hq, d, q)
    _lib.native().scmx_attn_decode(q, kcache, vcache, dev_pos, 0 if dev_pos is not None else int(n), out, hq, hk, d, rows,
                                   float(scale if scale is not None else d ** -0.5), work, splits)
    return out


def attn_prefill_splits(L, off, hq):
    """Key ranges for the attention of L new tokens behind `off` cached ones.  Unsplit, a workgroup per head and 128 queries
    walks all keys, 128 in 2 us.  Ranges help while all workgroups run at once (one a CU) and down to a range of 256 keys
    (128 in short contexts); joining them costs a launch and the ranges' traffic, which grows with L hq.  Measured, us
    whole / split, 16 heads, L behind off: 32 behind 300 11.4 / 10.6; 8 behind 500 13.2 / 10.8; 30 behind 2000 36 / 16; 100
    behind 4000 73 / 23; 300 behind 3000 61 / 29; 600 behind 4000 82 / 43; 1000 behind 1000 41 / 33; and where the line is:
    128 behind 256 (two steps of 128 keys fewer) 13.8 / 14.0; 300 behind 300 17.6 / 18.3 (three fewer); 300 behind 500
    20.0 / 19.4 (five); 1000 alone 23.6 / 23.5 (four); 1500 behind 1500, which fills more than half the CUs, 55 / 62."""
    tiles, pairs = -(-L // 128) * hq, -(-(off + L) // 128)
    if not 0 < tiles <= 128:
        return 1
    splits = min(64, 256 // tiles, pairs if pairs <= 4 else max(4, pairs // 2))
    saved = pairs - -(-pairs // splits)
    return splits if saved >= (2 if L * hq <= 1024 else 3 if L <= 128 else 5) else 1


def attn_prefill(q, kcache, vcache, off, scale=None, splits=None):
    """Causal attention of L new tokens: q bf16 [hq, L, d], best as the view of [L, hq, d] storage that
    qkv_headnorm_rope returns with token_major=True (any other layout is copied into that one), caches [hk, rows, d]
    whose rows off .. off+L-1 hold the new tokens' keys and values -> bf16 [L, hq * d].  Head dim 128.
    splits: ranges the keys are cut into (default: by the sizes)."""
    q = q.transpose(0, 1).contiguous()   # [L, hq, d] storage; no copy when q already is a view of it
    L, hq, d = q.shape
    hk, rows, _ = kcache.shape
    assert q.dtype == torch.bfloat16 and kcache.dtype == torch.bfloat16 and kcache.shape == vcache.shape
    out = _lib.native().empty_bf16(q, L, hq * d)
    if splits is None:
        splits = attn_prefill_splits(L, int(off), hq)
    work = _split_workspace(splits, L * hq, d, q)
    _lib.native().scmx_attn_prefill_split(q, kcache, vcache, out, L, int(off), hq, hk, d, rows,
                                          float(scale if scale is not None else d ** -0.5), work, splits)
    return out


def attn_decode_qkv(y, qn, kn, eps, hq, hk, d, kcache, vcache, pos, inv_freq, scale=None, splits=None):
    """qkv_headnorm_rope at L = 1 followed by attn_decode, in one launch and with the same bits: y bf16
    [1, (hq + 2 hk) d] -> bf16 [1, hq * d]; the token's k and v land in row pos of the caches.  pos: int, or an int64
    device tensor (for graph replay)."""
    assert kcache.shape == vcache.shape and kcache.shape[0] == hk and kcache.shape[2] == d
    assert y.dtype == torch.bfloat16 and y.numel() == (hq + 2 * hk) * d and kcache.dtype == torch.bfloat16
    assert inv_freq.dtype == torch.float32 and inv_freq.numel() == d // 2
    out = _lib.native().empty_bf16(y, 1, hq * d)
    dev_pos = pos if torch.is_tensor(pos) else None
    assert dev_pos is None or dev_pos.dtype == torch.int64
    if splits is None:
        splits = _decode_ranges(kcache.shape[1] if dev_pos is not None else int(pos) + 1, hq, hk)
    work = _split_workspace(splits, hq, d, y)
    _lib.native().scmx_attn_decode_qkv(y, qn, kn, _eps(eps), inv_freq, dev_pos, 0 if dev_pos is not None else int(pos),
                                       kcache, vcache, out, hq, hk, d, kcache.shape[1],
                                       float(scale if scale is not None else d ** -0.5), work, splits)
    return out


def qkv_fullnorm_y(y, qn, kn, eps, L, h, d, deps=()):
    """OLMoE: bf16 y [Mp, 3 h d] -> q, k, v [h, L, d] with RMSNorm over the full h*d-wide q and k."""
    q, k, v = (_lib.native().empty_bf16(y, h, L, d) for _ in range(3))
    _lib.native().scmx_qkv_fullnorm(y, qn, kn, _eps(eps), q, k, v, L, h, d)
    return q, k, v


def qkv_fullnorm_rope(y, qn, kn, eps, L, h, d, kcache, vcache, pos, inv_freq):
    """qkv_fullnorm_y fused with the rotary embedding of q and k and the KV-cache append: k and v go to rows
    pos..pos+L-1 of kcache / vcache [h, rows, d]; returns the [h, L, d] view of q stored as [L, h, d].  pos: int, or an
    int64 device tensor."""
    q = _lib.native().empty_bf16(y, L, h, d)
    assert kcache.shape == vcache.shape and kcache.shape[0] == h and kcache.shape[2] == d
    assert y.dtype == torch.bfloat16 and kcache.dtype == torch.bfloat16
    assert inv_freq.dtype == torch.float32 and inv_freq.numel() == d // 2
    dev_pos = pos if torch.is_tensor(pos) else None
    assert dev_pos is None or dev_pos.dtype == torch.int64
    _lib.native().scmx_qkv_fullnorm_rope(y, qn, kn, _eps(eps), q, kcache, vcache, L, h, d, inv_freq, dev_pos,
                                         0 if dev_pos is not None else int(pos), kcache.shape[1], 1)
    return q.transpose(0, 1)
