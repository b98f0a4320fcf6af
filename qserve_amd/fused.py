"""Pair fusions for the decode loop (extensions; NOT part of the reference's `qserve_backend` surface).

Each function is bit-identical to the two reference ops it replaces (tests/test_fused_gpu.py checks that on the GPU);
they exist because at decode batch sizes each row kernel is a fixed ~5 us latency chain, so a pair costs one.

    add_residual_rms_norm_general(_fuse_sum)  ==  hidden += delta ; layernorm_ops.rms_norm_general(_fuse_sum)(hidden)
    silu_and_mul_quant(_fuse_sum)             ==  activation_ops.silu_and_mul ; fused_kernels.invoke_quant(_fuse_sum)
    single_query_attention_quant(_fuse_sum)   ==  fused_attention.single_query_attention ; fused_kernels.invoke_quant(_fuse_sum)
    gemm_silu_and_mul_per_chn / _per_group    ==  qgemm_w4a8_per_*.gemm_forward_cuda(gate_up) ; activation_ops.silu_and_mul

"""
import torch

from .backend._util import check, expect, guard, lib, ptr, stream, widened_scratch


def add_residual_rms_norm_general(out, hidden, delta, weight, scaling, epsilon, input_sum=None):
    """hidden (fp16 [T, hid], updated in place) += delta; then out/scaling(/input_sum) = rms_norm_general(hidden)."""
    expect(out, torch.int8, "out")
    expect(hidden, torch.float16, "hidden")
    expect(delta, torch.float16, "delta")
    expect(weight, torch.float16, "weight")
    expect(scaling, torch.float16, "scaling")
    if input_sum is not None:
        expect(input_sum, torch.float16, "input_sum")
    if hidden.shape != delta.shape:
        raise RuntimeError(f"add_residual_rms_norm_general: hidden {tuple(hidden.shape)} vs delta {tuple(delta.shape)}")
    hid = hidden.size(-1)
    with guard(out):
        check(lib.qs_add_residual_rms_norm_general(ptr(out), ptr(hidden), ptr(delta), ptr(weight),
                                                   ptr(input_sum) if input_sum is not None else 0, ptr(scaling),
                                                   float(epsilon), hidden.numel() // hid, hid, stream()),
              "fused.add_residual_rms_norm_general")


def silu_and_mul_quant(out, input, scale, input_sum=None):
    """out int8 [T, d], scale(/input_sum) fp16 [T] = invoke_quant(silu_and_mul(input fp16 [T, 2d]))."""
    expect(out, torch.int8, "out")
    expect(input, torch.float16, "input")
    expect(scale, torch.float16, "scale")
    if input_sum is not None:
        expect(input_sum, torch.float16, "input_sum")
    d = input.size(-1) // 2
    if out.size(-1) != d:
        raise RuntimeError(f"silu_and_mul_quant: out width {out.size(-1)} != {d}")
    with guard(out):
        check(lib.qs_silu_and_mul_quant(ptr(out), ptr(input), ptr(input_sum) if input_sum is not None else 0, ptr(scale),
                                        input.numel() // (2 * d), d, stream()), "fused.silu_and_mul_quant")


def gemm_silu_and_mul_per_chn(in_feats, kernel, wscales, ascales, w_szs, a_ssums, out_act, tmp=None):
    """out_act fp16 [M, N/2] = silu_and_mul(per-channel W4A8 GEMM of the stacked gate_up weight `kernel` [N, K/2]) - one
    launch where the GEMM kernel has the activation epilogue, two through `tmp` (fp16 [M, N]) otherwise; bit-identical."""
    _gemm_silu(False, in_feats, kernel, (wscales, ascales, w_szs, a_ssums), out_act, tmp)


def gemm_silu_and_mul_per_group(in_feats, kernel, zeros, scales_i8, wscales, ascales, out_act, tmp=None):
    """Per-group (g128) form of `gemm_silu_and_mul_per_chn`."""
    _gemm_silu(True, in_feats, kernel, (zeros, scales_i8, wscales, ascales), out_act, tmp)


def _gemm_silu(per_group, in_feats, kernel, rest, out_act, tmp):
    expect(in_feats, torch.int8, "in_feats")
    expect(kernel, torch.int8, "kernel")
    expect(out_act, torch.float16, "out_act")
    for i, t in enumerate(rest):
        expect(t, torch.int8 if per_group and i < 2 else torch.float16, f"operand {i}")
    K = in_feats.size(-1)
    M, N = in_feats.numel() // K, kernel.size(0)
    if kernel.size(1) * 2 != K:
        raise RuntimeError(f"gemm_silu_and_mul: kernel {tuple(kernel.shape)} does not match K={K}")
    if out_act.numel() != M * (N // 2):
        raise RuntimeError(f"gemm_silu_and_mul: out_act has {out_act.numel()} elements, expected {M} x {N // 2}")
    if tmp is not None:
        expect(tmp, torch.float16, "tmp")
        if tmp.numel() < M * N:
            raise RuntimeError(f"gemm_silu_and_mul: tmp has {tmp.numel()} elements, needs {M} x {N}")
    fn = lib.qs_w4a8_per_group_gemm_silu_mul if per_group else lib.qs_w4a8_per_chn_gemm_silu_mul
    with guard(out_act):
        scratch = widened_scratch(M, N, K, in_feats) if per_group else None
        if scratch is not None:
            check(lib.qs_w4a8_per_group_gemm_silu_mul_scratch(ptr(in_feats), ptr(kernel), *[ptr(t) for t in rest], ptr(out_act),
                                                              ptr(tmp) if tmp is not None else 0, M, N, K, ptr(scratch), scratch.numel(), stream()),
                  "fused.gemm_silu_and_mul")
            return
        check(fn(ptr(in_feats), ptr(kernel), *[ptr(t) for t in rest], ptr(out_act), ptr(tmp) if tmp is not None else 0,
                 M, N, K, stream()), "fused.gemm_silu_and_mul")


def single_query_attention_quant(q, k, v, kv_pointers, length_per_sample, quant_out, quant_scale, memory_max_seqlen,
                                 tokens_per_block, size_per_token, timestep, rotary_embedding_dim, rotary_base,
                                 neox_rotary_style, int4_kv_cache, kv_cache_with_zeros, quant_sum=None):
    """attn = single_query_attention(q, k, v, ...) (fp16 [B, H, Dh], returned) and, in the same call,
    quant_out / quant_scale (/ quant_sum) = invoke_quant(_fuse_sum)(attn.reshape(B, -1)) - bit-identical to the pair
    (llama_w4a8_unpad.py:253-282); one launch where the attention kernel can finish the row itself."""
    for n, t in (("q", q), ("k", k), ("v", v)):
        expect(t, torch.float16, n, contiguous=False)
    expect(kv_pointers, torch.int64, "kv_pointers")
    expect(quant_out, torch.int8, "quant_out")
    expect(quant_scale, torch.float16, "quant_scale")
    if quant_sum is not None:
        expect(quant_sum, torch.float16, "quant_sum")
    batch = kv_pointers.size(0)
    nheads, nheads_kv, headdim = q.size(1), k.size(1), k.size(-1)
    if not (k.stride(2) == 1 and k.stride(1) == headdim and v.stride(2) == 1 and v.stride(1) == headdim):
        raise RuntimeError("k and v must have stride(2) == 1 and stride(1) == head_dim")
    if not (q.stride(2) == 1 and q.stride(1) == headdim):
        raise RuntimeError("q must have stride(2) == 1 and stride(1) == head_dim")
    if length_per_sample is not None:
        expect(length_per_sample, torch.int32, "length_per_sample")
    if quant_out.numel() != q.size(0) * nheads * headdim:
        raise RuntimeError("quant_out must hold batch x heads x head_dim int8 values")
    out = torch.empty((q.size(0), nheads, headdim), dtype=q.dtype, device=q.device)
    with guard(q):
        check(lib.qs_single_query_attention_quant(
            ptr(q), ptr(k), ptr(v), ptr(kv_pointers), ptr(length_per_sample), ptr(out), ptr(quant_out),
            ptr(quant_sum) if quant_sum is not None else 0, ptr(quant_scale), batch, nheads, nheads_kv, headdim,
            q.stride(0), k.stride(0), kv_pointers.size(-1), int(memory_max_seqlen), int(tokens_per_block),
            int(size_per_token), int(timestep), int(rotary_embedding_dim), float(rotary_base),
            int(bool(neox_rotary_style)), int(bool(int4_kv_cache)), int(bool(kv_cache_with_zeros)), stream()),
            "fused.single_query_attention_quant")
    return out


def _gemm_common(per_group, in_feats, kernel, rest):
    expect(in_feats, torch.int8, "in_feats")
    expect(kernel, torch.int8, "kernel")
    for i, t in enumerate(rest):
        expect(t, torch.int8 if per_group and i < 2 else torch.float16, f"operand {i}")
    K = in_feats.size(-1)
    M, N = in_feats.numel() // K, kernel.size(0)
    if kernel.size(1) * 2 != K:
        raise RuntimeError(f"w4a8 gemm: kernel {tuple(kernel.shape)} does not match K={K}")
    return M, N, K


# ---- K-slice planes: (row-parallel GEMM, add + norm + quant) with the GEMM's cross-workgroup reduction and epilogue moved into
# the row kernel that follows it anyway (include/qserve_amd.h, "K-slice PLANES") ------------------------------------------------
_PLANES_PLAN = {}


def gemm_planes_plan(M, N, K, per_group=False):
    """-> number of K slices the planes launch of this shape uses (0: no such launch, run the ordinary pair).  Deterministic
    in the shape (and in the library's A/B switch, which tests change): cached per shape while the switch is at its default."""
    import ctypes as C
    key = (int(M), int(N), int(K), bool(per_group))
    ks = _PLANES_PLAN.get(key)
    if ks is None or _PLANES_PLAN.get("nocache"):
        buf = (C.c_int * 4)()
        check(lib.qs_w4a8_gemm_planes_plan(int(key[3]), key[0], key[1], key[2], C.cast(buf, C.c_void_p)), "fused.gemm_planes_plan")
        ks = int(buf[0])
        _PLANES_PLAN[key] = ks
    return ks


def gemm_planes(in_feats, kernel, planes, zeros=None, scales_i8=None):
    """planes int32 [k_slices, M, N] (k_slices = gemm_planes_plan(M, N, K)): the W4A8 GEMM's partial sums per K slice,
    per-channel (zeros / scales_i8 None) or per-group."""
    per_group = zeros is not None
    M, N, K = _gemm_common(per_group, in_feats, kernel, (zeros, scales_i8) if per_group else ())
    expect(planes, torch.int32, "planes")
    if planes.dim() != 3 or planes.size(1) != M or planes.size(2) != N or not planes.is_contiguous():
        raise RuntimeError(f"gemm_planes: planes {tuple(planes.shape)} for a [{M}, {N}] product")
    ks = gemm_planes_plan(M, N, K, per_group)
    if ks == 0 or planes.size(0) != ks:
        raise RuntimeError(f"gemm_planes: planes {tuple(planes.shape)} but this shape runs as {ks} x [{M}, {N}]")
    with guard(in_feats):
        if per_group:
            check(lib.qs_w4a8_per_group_gemm_planes(ptr(in_feats), ptr(kernel), ptr(zeros), ptr(scales_i8), ptr(planes), M, N, K,
                                                    stream()), "fused.gemm_planes")
        else:
            check(lib.qs_w4a8_per_chn_gemm_planes(ptr(in_feats), ptr(kernel), ptr(planes), M, N, K, stream()), "fused.gemm_planes")


def add_residual_rms_norm_general_planes(out, hidden, planes, wscales, ascales, weight, scaling, epsilon, w_szs=None,
                                         a_ssums=None, input_sum=None):
    """== gemm(..., delta) ; add_residual_rms_norm_general(out, hidden, delta, weight, scaling, epsilon, input_sum) where the GEMM
    ran as gemm_planes: wscales / w_szs [hidden] and ascales / a_ssums [T] are that GEMM's epilogue operands (w_szs and a_ssums
    None together = per-group).  ascales / a_ssums may be the very tensors scaling / input_sum are written to."""
    expect(out, torch.int8, "out")
    expect(hidden, torch.float16, "hidden")
    expect(planes, torch.int32, "planes")
    for n, t in (("wscales", wscales), ("ascales", ascales), ("weight", weight), ("scaling", scaling)):
        expect(t, torch.float16, n)
    if (w_szs is None) != (a_ssums is None):
        raise RuntimeError("add_residual_rms_norm_general_planes: w_szs and a_ssums come together or not at all")
    for n, t in (("w_szs", w_szs), ("a_ssums", a_ssums), ("input_sum", input_sum)):
        if t is not None:
            expect(t, torch.float16, n)
    hid = hidden.size(-1)
    T = hidden.numel() // hid
    if planes.dim() != 3 or planes.size(1) != T or planes.size(2) != hid:
        raise RuntimeError(f"add_residual_rms_norm_general_planes: planes {tuple(planes.shape)} vs hidden [{T}, {hid}]")
    # the C entry takes pointers + a plane stride: everything it will read or write must be there (a wrong-sized tensor would be
    # read or written out of bounds on the device)
    if not planes[0].is_contiguous() or not hidden.is_contiguous() or not out.is_contiguous():
        raise RuntimeError("add_residual_rms_norm_general_planes: planes[i], hidden and out must be contiguous [T, hidden] blocks")
    if out.numel() != T * hid:
        raise RuntimeError(f"add_residual_rms_norm_general_planes: out has {out.numel()} elements, expected {T * hid}")
    for n, t, need in (("wscales", wscales, hid), ("w_szs", w_szs, hid), ("weight", weight, hid), ("ascales", ascales, T),
                       ("a_ssums", a_ssums, T), ("scaling", scaling, T), ("input_sum", input_sum, T)):
        if t is not None and (t.numel() < need or not t.is_contiguous()):
            raise RuntimeError(f"add_residual_rms_norm_general_planes: {n} needs {need} contiguous values, has {t.numel()}")
    with guard(out):
        check(lib.qs_add_residual_rms_norm_general_planes(
            ptr(out), ptr(hidden), ptr(planes), planes.size(0), planes.stride(0), ptr(wscales),
            ptr(w_szs) if w_szs is not None else 0, ptr(ascales), ptr(a_ssums) if a_ssums is not None else 0, ptr(weight),
            ptr(input_sum) if input_sum is not None else 0, ptr(scaling), float(epsilon), T, hid, stream()),
            "fused.add_residual_rms_norm_general_planes")


def add_residual_rms_norm_planes(out, hidden, hidden_out, planes, wscales, ascales, weight, epsilon, w_szs=None, a_ssums=None):
    """== gemm(..., delta) ; hidden_out = hidden + delta ; rms_norm(out, hidden_out, weight) where the GEMM left planes [k_slices, T, hidden]
    (k_slices 1, 2 or 4; its epilogue operands as in add_residual_rms_norm_general_planes).  hidden_out may be hidden."""
    expect(planes, torch.int32, "planes")
    hid = hidden.size(-1)
    T = hidden.numel() // hid
    _whole("add_residual_rms_norm_planes", torch.float16, (out, T * hid), (hidden, T * hid), (hidden_out, T * hid), (wscales, hid), (w_szs, hid), (weight, hid), (ascales, T),
           (a_ssums, T))
    if planes.dim() != 3 or planes.size(1) != T or planes.size(2) != hid or not planes.is_contiguous() or (w_szs is None) != (a_ssums is None):
        raise RuntimeError(f"add_residual_rms_norm_planes: planes {tuple(planes.shape)} vs hidden [{T}, {hid}]")
    with guard(out):
        check(lib.qs_add_residual_rms_norm_planes(ptr(out), ptr(hidden), ptr(hidden_out), ptr(planes), planes.size(0), planes.stride(0), ptr(wscales), _or0(w_szs),
                                                  ptr(ascales), _or0(a_ssums), ptr(weight), float(epsilon), T, hid, stream()), "fused.add_residual_rms_norm_planes")


# ---- the two ends of a prompt phase over sequences of one length (include/qserve_amd.h) -----------------------------------------------------

def prompt_layout(batch, tokens, device):
    """-> (lengths int32 [batch], first rows int32 [batch + 1], padding offsets int32 [batch * tokens]) of `batch` sequences of `tokens` tokens."""
    seq, cu, pad = (torch.empty((n,), dtype=torch.int32, device=device) for n in (batch, batch + 1, batch * tokens))
    with guard(seq):
        check(lib.qs_prompt_layout(ptr(seq), ptr(cu), ptr(pad), batch, tokens, stream()), "fused.prompt_layout")
    return seq, cu, pad


def embed_rms_norm_general(out, hidden, table, tokens, weight, scaling, epsilon, input_sum=None):
    """== hidden = table[tokens] ; rms_norm_general(_fuse_sum)(out, hidden, ...), the row sum in this library's order."""
    T, hid = hidden.shape
    _whole("embed_rms_norm_general", torch.int8, (out, T * hid))
    _whole("embed_rms_norm_general", torch.int64, (tokens, T))
    _whole("embed_rms_norm_general", torch.float16, (hidden, T * hid), (table, table.size(0) * hid), (weight, hid), (scaling, T), (input_sum, T))
    with guard(out):
        check(lib.qs_embed_rms_norm_general(ptr(out), ptr(hidden), ptr(table), ptr(tokens), table.size(0), ptr(weight), _or0(input_sum), ptr(scaling), float(epsilon), T, hid,
                                            stream()), "fused.embed_rms_norm_general")


def last_rows_rms_norm(out, hidden, hidden_out, delta, weight, epsilon, tokens, lengths):
    """hidden_out [B, hid] = the last of every `tokens` rows of hidden + delta ; rms_norm(out, hidden_out) ; lengths [B] = tokens + 1."""
    B, hid = hidden_out.shape
    _whole("last_rows_rms_norm", torch.float16, (out, B * hid), (hidden, B * tokens * hid), (hidden_out, B * hid), (delta, B * tokens * hid), (weight, hid))
    _whole("last_rows_rms_norm", torch.int32, (lengths, B))
    with guard(out):
        check(lib.qs_last_rows_rms_norm(ptr(out), ptr(hidden), ptr(hidden_out), ptr(delta), ptr(weight), float(epsilon), B, tokens, hid, ptr(lengths), stream()),
              "fused.last_rows_rms_norm")


# ---- products of one to four tokens with the row operation in front of them (include/qserve_amd.h, qs_*_w4a8_rows*) ---------------------

def _or0(t):
    return 0 if t is None else ptr(t)


def _whole(what, dtype, *pairs):
    """Every tensor there is: of this type, contiguous, with at least so many values (the C entries take bare pointers)."""
    for t, n in pairs:
        if t is not None:
            expect(t, dtype, what)
            if t.numel() < n or not t.is_contiguous():
                raise RuntimeError(f"{what}: a tensor of {t.numel()} values where {n} contiguous ones are read or written")


def _rows_weights(what, kernel, zeros, scales_i8, N, K):
    _whole(what, torch.int8, (kernel, N * K // 2), (zeros, N * K // 128), (scales_i8, N * K // 128))
    if (zeros is None) != (scales_i8 is None):
        raise RuntimeError(f"{what}: zeros and scales_i8 come together or not at all")


def rows_ok(M, N, K, k_slices, per_group=False):
    """Whether the products of few tokens take [M, K] x [N, K] in k_slices slices of K."""
    return bool(lib.qs_w4a8_rows_ok(int(per_group), int(M), int(N), int(K), int(k_slices)))


def rows_planes(in_feats, kernel, planes, zeros=None, scales_i8=None):
    """planes int32 [k_slices, M, N]: gemm_planes for M <= 4, in as many slices as planes has."""
    ks, M, N = planes.shape
    K = in_feats.numel() // M
    _whole("rows_planes", torch.int8, (in_feats, M * K))
    _whole("rows_planes", torch.int32, (planes, ks * M * N))
    _rows_weights("rows_planes", kernel, zeros, scales_i8, N, K)
    with guard(planes):
        check(lib.qs_w4a8_rows_planes(ptr(in_feats), ptr(kernel), _or0(zeros), _or0(scales_i8), ptr(planes), M, N, K, ks, stream()), "fused.rows_planes")


def norm_rows(out, hidden, hidden_out, planes, plane_wscales, plane_ascales, weight, epsilon, kernel, wscales, plane_wszs=None, plane_asums=None, w_szs=None, zeros=None,
              scales_i8=None, silu_mul=False):
    """== add_residual_rms_norm_general_planes (the sum into hidden_out, another tensor than hidden) and the product of its int8 rows with `kernel`: out fp16 [M, N], or
    with silu_mul silu(gate) * up [M, N / 2] of kernel = [gate rows | up rows]."""
    M, K = hidden.shape
    N = kernel.size(0)
    f16 = torch.float16
    _whole("norm_rows", f16, (out, M * N // (2 if silu_mul else 1)), (hidden, M * K), (hidden_out, M * K), (plane_wscales, K), (plane_wszs, K), (plane_ascales, M),
           (plane_asums, M), (weight, K), (wscales, N), (w_szs, N))
    _whole("norm_rows", torch.int32, (planes, planes.size(0) * M * K))
    _rows_weights("norm_rows", kernel, zeros, scales_i8, N, K)
    if planes.dim() != 3 or planes.size(1) != M or planes.size(2) != K:
        raise RuntimeError(f"norm_rows: planes {tuple(planes.shape)} vs hidden [{M}, {K}]")
    with guard(out):
        check(lib.qs_norm_w4a8_rows(ptr(out), int(silu_mul), ptr(hidden), ptr(hidden_out), ptr(planes), planes.size(0), planes.stride(0), ptr(plane_wscales),
                                    _or0(plane_wszs), ptr(plane_ascales), _or0(plane_asums), ptr(weight), float(epsilon), ptr(kernel), _or0(zeros), _or0(scales_i8),
                                    ptr(wscales), _or0(w_szs), M, N, K, stream()), "fused.norm_rows")


def quant_rows_planes(planes, act, scale, kernel, input_sum=None, zeros=None, scales_i8=None):
    """== invoke_quant(_fuse_sum) of act [M, K] (scale and, per-channel, input_sum [M] are written) and rows_planes of its int8 rows."""
    ks, M, N = planes.shape
    K = act.numel() // M
    _whole("quant_rows_planes", torch.float16, (act, M * K), (scale, M), (input_sum, M))
    _whole("quant_rows_planes", torch.int32, (planes, ks * M * N))
    _rows_weights("quant_rows_planes", kernel, zeros, scales_i8, N, K)
    with guard(planes):
        check(lib.qs_quant_w4a8_rows_planes(ptr(planes), ptr(act), ptr(scale), _or0(input_sum), ptr(kernel), _or0(zeros), _or0(scales_i8), M, N, K, ks, stream()),
              "fused.quant_rows_planes")
