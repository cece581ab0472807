"""Grouped expert GEMM call surface (the reference's e2e/sc_moe.py) on torch tensors over libscmx.so.

Token-expert assignments are sorted by expert (`route_sort`), expert e owns rows [off[e], off[e+1]) of the sorted
activations, and one launch of the grouped INT8-MFMA GEMM covers all experts, each workgroup unpacking its expert's
weight tile in LDS.  Unlike the reference, `moe_mm` needs no padding rows after the R sorted rows (row indices are
clamped inside the kernel) and can gather the activation rows itself: pass the UNSORTED `xq`/`xscale` with
`gather=tok` to skip the xq[tok] copy.
"""
import torch

from . import _lib
from . import sc_format as F
from . import sc_kernels as S


def route(logits, k, renorm=True, shared_logit=None):
    """Router on bf16 logits [M, E]: (inds int32 [M, k], scores bf16 [M, k]) = the k experts of largest softmax
    probability (float32 softmax rounded to bf16) and their probabilities, divided by their sum when `renorm`
    (e2e/fused_olmoe.py:183-192).  shared_logit bf16 [M]: a last slot with expert index E and score
    sigmoid(shared_logit), outputs [M, k + 1] (e2e/fused_qwen35.py:171-180).  Slots are listed by falling probability."""
    M, E = logits.shape
    assert logits.dtype == torch.bfloat16 and (shared_logit is None or shared_logit.dtype == torch.bfloat16)
    logits = logits.contiguous()
    if shared_logit is not None:
        shared_logit = shared_logit.reshape(M).contiguous()
    width = k + (shared_logit is not None)
    inds = _lib.native().empty_i32(logits, M, width)
    scores = _lib.native().empty_bf16(logits, M, width)
    _lib.native().scmx_route_topk(logits, shared_logit, M, E, k, int(bool(renorm)), inds, scores)
    return inds, scores


def norm_route(x, w, eps, gate, k, renorm=True):
    """rmsnorm_quant_n, linear_bf16 and route of one row, the first two in one launch: x bf16 [1, D], norm weight w [D], router gate
    [E, D] -> (xq, xscale, xn, inds, scores) with the same bits.  None where that kernel does not take the shapes (D of 512 ... 2048) or
    tensors that linear_bf16 would leave to the array op."""
    D, E = x.shape[1], gate.shape[0]
    if not (x.shape[0] == 1 and D % 512 == 0 and 512 <= D <= 2048 and 0 < k <= E <= 1024 and gate.shape[1] == D and tuple(w.shape) == (D,)
            and S._plain(x, gate) and S._plain(x, w) and not (x.data_ptr() | w.data_ptr() | gate.data_ptr()) % 16):
        return None
    n = _lib.native()
    xq, xs, xn, logits = n.empty_i8(x, 1, D), n.empty_f32(x, 1), n.empty_bf16(x, 1, D), n.empty_bf16(x, 1, E)
    n.scmx_norm_linear(x, w, S._eps(eps), gate, D, E, xq, xs, xn, logits)
    return xq, xs, xn, *route(logits, k, renorm)


def route_sort(inds, n_experts, tm):
    """inds int [M, topk] -> (pos [R], tok [R + tm], e_sorted [R], off [E+1], tstart [E+1], max M-tiles)."""
    M, k = inds.shape
    R = M * k
    inds = inds.to(torch.int32).contiguous()
    pos = _lib.native().empty_i32(inds, R)
    tok = _lib.native().empty_i32(inds, R + tm)
    es = _lib.native().empty_i32(inds, R)
    off = _lib.native().empty_i32(inds, n_experts + 1)
    ts = _lib.native().empty_i32(inds, n_experts + 1)
    _lib.native().scmx_route_sort(inds, M, k, n_experts, tm, pos, tok, es, off, ts)
    return pos, tok, es, off, ts, -(-R // tm) + n_experts


def row_tile(R, n_experts):
    """Row tile of the grouped GEMM for R assignments over n_experts: 256-row tiles (the fewest LDS bytes per MFMA) from
    about 96 rows per expert on, below that 64-row tiles (less padding, packed weights in LDS).  Measured on 64 experts
    of 2048 x 2048 / 2048 x 1024 with top-8 routing: 512 tokens 149 us with 64-row tiles against 169 with 256-row ones,
    1024 tokens 205 against 180.  (With the 256-row tiles reading slots, below, the line is nearer 80 rows: 5600 over 64
    experts 115 us either way.)"""
    return 256 if R >= 96 * n_experts else 64


def segments(expert_sorted, n_experts, tm):
    """Sorted expert id per row -> (off int32 [E+1], tstart int32 [E+1], max number of M-tiles)."""
    R = expert_sorted.shape[0]
    counts = torch.bincount(expert_sorted.to(torch.int64), minlength=n_experts).to(torch.int32)
    zero = torch.zeros(1, dtype=torch.int32, device=counts.device)
    off = torch.cat([zero, torch.cumsum(counts, 0).to(torch.int32)])
    tstart = torch.cat([zero, torch.cumsum((counts + tm - 1) // tm, 0).to(torch.int32)])
    return off, tstart, -(-R // tm) + n_experts


def _out(R, N, epi, like):
    if epi == 0:
        return _lib.native().empty_i32(like, R, N)
    return _lib.native().empty_bf16(like, R, N // 2 if epi == 3 else N)


def moe_mm(xq, R, codes, bcodes, wscale, off, tstart, max_tiles, N, epi, xscale=None, dtype=torch.bfloat16,
           tile=(64, 64, 4), bk=128, gather=None, fmt=None):
    """Grouped W4A8 GEMM.  xq int8 [>= R, K] sorted by expert (or unsorted with gather=tok); packed expert weights
    codes [E, N*K/8], bcodes [E, N, ..], wscale f32 [E, N] -> INT32 [R, N] (EPI 0), bf16 [R, N] (1) or
    bf16 [R, N/2] (3, interleaved gate/up).  tile[0] is the row tile the segments were built for (64, 128 or 256)."""
    fmt = fmt or F.DEFAULT
    K = xq.shape[1]
    E = wscale.shape[0]
    assert xq.dtype == torch.int8 and (gather is not None or xq.shape[0] >= R)
    out = _out(R, N, epi, xq)
    _lib.native().scmx_moe_mm(fmt.c, xq, xscale, gather, R, codes, bcodes, wscale, off, tstart, E, tile[0], N, K, epi, out)
    return out


def gather_blocked(xq, xscale, tok, R, off, tstart):
    """The sorted rows xq[tok] (and their scales) in the 256-row slots of moe_mm_blocked -> (slots, xscale f32 [R])."""
    K, E = xq.shape[1], off.shape[0] - 1
    out, xs = _lib.native().empty_i8(xq, (-(-R // 256) + E) * 256 * K), _lib.native().empty_f32(xq, R)
    _lib.native().scmx_moe_gather_blocked(xq, xscale, tok, off, tstart, E, R, K, out, xs)
    return out, xs


def act_quant_sorted(x, R, off, tstart):
    """act_quant of sorted rows x bf16 [R, K] into the same slots -> (slots, xscale f32 [R])."""
    K, E = x.shape[1], off.shape[0] - 1
    assert x.dtype == torch.bfloat16
    xq, xs = _lib.native().empty_i8(x, (-(-R // 256) + E) * 256 * K), _lib.native().empty_f32(x, R)
    _lib.native().scmx_act_quant_sorted(x, off, tstart, E, R, K, xq, xs)
    return xq, xs


def moe_mm_blocked(slots, xscale, R, K, codes, bcodes, wscale, off, tstart, N, epi, fmt=None):
    """moe_mm on rows in slots (gather_blocked, act_quant_sorted; off / tstart of 256-row tiles)."""
    fmt = fmt or F.DEFAULT
    out = _out(R, N, epi, slots)
    _lib.native().scmx_moe_mm_blocked(fmt.c, slots, xscale, R, codes, bcodes, wscale, off, tstart, wscale.shape[0], N, K, epi, out)
    return out


def takes_slots(R, n_experts, K, tm, fmt):
    """Whether a grouped GEMM with reduction K and row tile tm can read its activations from slots."""
    return tm == 256 and bool(_lib.native().scmx_moe_mm_takes_slots(fmt.c, R, n_experts, K))


def slots_pay(R, n_experts, N, K, gathered):
    """Whether a grouped GEMM on N columns and 256-row tiles is faster from slots than by rows, what fills them included: the copy of
    `gathered` rows (6 - 10 us and R * K bytes), or the quantization, which writes either layout.  Slots always take one tile of 256 rows
    and 128 columns; by rows the launch chooses, and cuts a few tiles into pairs of 128 rows that reach more CUs.  Lines for 256 CUs, in
    256 x 256 tiles of the experts if none had more rows than that; 795 problems (4 ... 257 experts, 512 ... 4352 columns and reductions,
    96 ... 1500 rows an expert, four formats, skewed routing, 206 of them with weights from HBM): 1.7 per cent over the faster form on
    average for gate|up, 0.4 for down, where slots from 2048 columns on cost 4.5 and slots for all 3.7, and up to 2.05 and 1.8 times
    the rows' time.  us by rows / from slots:
    - quantized rows: 8 experts of 2048 x 1024, 100 rows 15.3 / 19.4, 150 rows 21.5 / 20.2; 16 of 768 x 768, 110 rows 0.8 times as
      fast, 300 rows 1.23; 64 of 2048 x 1024, 400 rows 106 / 99.  Columns that the 256x256 tile does not take (not a multiple of 256,
      under 1024) are 256x128 by rows as well: 6 of 640 x 1280, 1053 rows 0.86 times as fast.
    - gathered rows: 8 of 2048 x 2048, 100 rows 16.4 / 29.4, 400 rows 38.3 / 35.8; 16 of 4096 x 2048, 110 / 180 / 300 rows 0.91 ... 1.16 /
      0.96 ... 1.01 / 1.05 ... 1.11 times as fast; 32 of 2048 x 2048, 220 / 300 / 400 rows 0.96 / 1.04 / 1.01; 64 of 2048 x 2048, 100 ...
      400 rows 82 / 77, 98 / 88, 119 / 102, 172 / 169; under 128 rows 64 of 2048 x 1024 0.93 ... 1.03 and 16 of 8192 x 4096, whose code
      lines are read twice, 0.90 ... 1.0.  Less than 2048 columns do not earn the copy: 128 of 1536 x 2048, 100 ... 400 rows 0.98, 1.0,
      0.98, 0.91."""
    rows, tiles, cus = R / n_experts, n_experts * -(-N // 256), 256
    if not gathered:
        wide = N % 256 == 0 or N >= 1024
        return tiles > cus // 4 or (wide and (rows >= 256 or tiles * rows > 43 * cus))
    if N < 2048:
        return False
    if rows < 128:
        return tiles > cus and 1536 <= K < 4096
    return tiles > cus or (rows >= 256 and tiles > cus // 2 and K >= 1024)


def expert_mlp(xq, xs, R, gate_up, down, tok, off, tstart, max_tiles, tm, fmt):
    """Gate|up with SwiGLU, INT8, down of the routed experts on packed weights: xq int8 [M, D] with the token of each sorted row in tok,
    gate_up / down = (codes, bcodes, wscale) stacked over the experts -> bf16 [R, D] by sorted row.  With 256-row tiles the activations
    go through slots in the blocked layout where that pays.  Both GEMMs, quantization and copy, us without / with slots, 64 experts of
    2048 x 2048 and 2048 x 1024, skewed routing: 8000 rows 126 / 117, 12000 169 / 149, 24000 260 / 236, 48000 425 / 416, 24000 in
    e2m1/B16/M1..10 261 / 247; 16 of 4096 x 4096 264 / 225; 257 of 1024 x 2048, 54000 rows: down 145 / 136.  Working memory beyond the
    outputs: (ceil(R / 256) + E) * 256 * K bytes of slots for each of the two, one after the other (24000 rows over 64 experts:
    83 MB at K = 2048), where rows take R * K for down and gate|up nothing."""
    (cg, bg, sg), (cd, bd, sd) = gate_up, down
    E, F2 = sg.shape
    D, K2, tile = sd.shape[1], F2 // 2, (tm, 64, 4)
    if slots_pay(R, E, F2, D, True) and takes_slots(R, E, D, tm, fmt):
        slots, xs = gather_blocked(xq, xs, tok, R, off, tstart)
        act = moe_mm_blocked(slots, xs, R, D, cg, bg, sg, off, tstart, F2, 3, fmt)
    else:
        act = moe_mm(xq, R, cg, bg, sg, off, tstart, max_tiles, F2, 3, xs, tile=tile, gather=tok, fmt=fmt)
    if slots_pay(R, E, D, K2, False) and takes_slots(R, E, K2, tm, fmt):
        slots, xs = act_quant_sorted(act, R, off, tstart)
        return moe_mm_blocked(slots, xs, R, K2, cd, bd, sd, off, tstart, D, 1, fmt)
    xq, xs = S.act_quant(act, R)
    return moe_mm(xq, R, cd, bd, sd, off, tstart, max_tiles, D, 1, xs, tile=tile, fmt=fmt)


def moe_mm_i8(xq, R, wq, wscale, off, tstart, max_tiles, N, epi, xscale=None, dtype=torch.bfloat16, tile=(64, 64, 4),
              gather=None):
    """Two-pass variant: wq int8 [E * N, K] already unpacked (unpack_experts)."""
    K = xq.shape[1]
    E = wscale.shape[0]
    if isinstance(wq, S.PackedWq):
        wq = wq.materialize()
    assert tuple(wq.shape) == (E * N, K)
    out = _out(R, N, epi, xq)
    _lib.native().scmx_moe_mm_i8(xq, xscale, gather, R, wq, wscale, off, tstart, E, tile[0], N, K, epi, out)
    return out


def unpack_experts(codes, bcodes, N, K):
    """All experts' packed weights -> INT8 [E * N, K] (one unpack launch)."""
    E = codes.shape[0]
    return S.unpack_i8(codes.reshape(-1), bcodes.reshape(E * N, -1), E * N, K, lazy=False)


def moe_combine(y, pos, scores, res, w, eps, M, quant=True, blocked=False):
    """y bf16 [R, K] (sorted assignments), pos int32 [M*topk], scores bf16 [M, topk], res [Mp, K] ->
    (h [Mp, K], xq int8 [Mp, K], xscale [Mp]) with xq = INT8(rms_norm(h, w)); quant=False returns xq = xs = None.
    blocked: xq as a BlockedXq (the layout of act_quant_blocked) where the shape allows it (Mp % 32 == 0, K % 512 == 0, K <= 2048) and
    the rows are as many as the kernel that writes it is made for (1024), by rows otherwise.
    (The reference keeps this in e2e/fused_olmoe.py:87-97.)"""
    return _combine(y, pos, scores, None, res, w, eps, M, quant, blocked)


def moe_combine_split(y, pos, scores, sscore, res, w, eps, M):
    """moe_combine (no quantization) whose last slot's score is given separately (e2e/fused_olmoe.py:74-84)."""
    return _combine(y, pos, scores, sscore, res, w, eps, M, False)


def _combine(y, pos, scores, sscore, res, w, eps, M, quant, blocked=False):
    Mp, K = res.shape
    topk = scores.shape[1] + (1 if sscore is not None else 0)
    h = torch.empty_like(res)
    xq = _lib.native().empty_i8(res, Mp, K) if quant else None
    xs = _lib.native().empty_f32(res, Mp) if quant else None
    blocked = (blocked and quant and Mp % 32 == 0 and Mp >= 1024 and K % 512 == 0 and K <= 2048
               and not (y.data_ptr() | res.data_ptr() | w.data_ptr()) % 16)
    combine = _lib.native().scmx_moe_combine_blocked if blocked else _lib.native().scmx_moe_combine
    combine(y, pos, scores, sscore, res, w if quant else None, S._eps(eps) if quant else 0.0, h, xq, xs, M, Mp, K, topk)
    return h, S.BlockedXq(xq.reshape(-1), Mp, K) if blocked else xq, xs
