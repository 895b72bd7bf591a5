"""Host-side mirror of the reference's attention call sites on top of the C ABI.

`AttentionContext.compute_val_lookup` has the argument meaning of
TAttentionComputer::ComputeValLookup (gpt/compute/gpt_cpu.cpp:391-441) / the Fp8Att launch
(gpt/compute/gpt_cuda.cu:503-507); `AttentionContext.compute_val_lookup_decode` that of
ComputeValLookup in gpt/train/cpu_infer.cpp:413-460 and `KVCache.add_vectors` that of
TAttentionVecHistory::AddVectors (:403-408).  torch tensors are used for device memory only; all
arithmetic happens in libtsattn.so.  There is no fallback path: a missing library raises.
"""
import ctypes
import functools

import numpy as np
import torch

from . import capi


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _stream_ptr():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _raw_stream():
    """The current device's current stream, as an integer."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _scale_arg(s):
    """tensor -> (tensor, 0.0); python number -> (None, value)."""
    if isinstance(s, torch.Tensor):
        assert s.dtype == torch.float32 and s.is_cuda and s.is_contiguous()
        return s, 0.0
    return None, float(s)


def _new(rows, cols, dtype, device):
    return torch.empty_strided((rows, cols), (cols, 1), dtype=dtype, device=device)


def alibi_layer_schedule(depth, wide_window):
    """Per-layer (attention width, ALiBi slope) of a TScale model of `depth` layers: the ALIBI_V3 rule of
    InitAlibi (gpt/model_params/model_dim.cpp:55-97): max(1, groups/6) leading pairs of width-1 layers,
    then pairs of (64, slope 0.5) and (wide, slope 0); a one-layer model is (wide, 0.1)."""
    if depth == 1:
        return [(wide_window, 0.1)]
    groups = (depth + 1) // 2
    w1 = max(1, groups // 6)
    out = []
    for _ in range(w1):
        out += [(1, 0.0), (1, 0.0)]
    for _ in range(w1, groups):
        out += [(64, 0.5), (wide_window, 0.0)]
    return out


class AttentionContext:
    """One per device, like the reference's per-device compute context (gpt_cuda.cu:1478-1573)."""

    def __init__(self, device=0, max_seqs=64, max_heads=16, max_head_dim=128, max_splits=32):
        self.lib = capi.load()
        if not torch.cuda.is_available():
            raise RuntimeError("tscale_amd needs a HIP device; there is no CPU path")
        cfg = capi.Config(device, max_seqs, max_heads, max_head_dim, max_splits)
        h = ctypes.c_void_p()
        capi.check(self.lib.tsattn_create(ctypes.byref(cfg), ctypes.byref(h)))
        self.handle = h
        self._h = h.value
        self._count = ctypes.c_int(0)  # where calls write a number of planes
        self._count_at = ctypes.addressof(self._count)
        self.device = torch.device("cuda", device)
        self._workspace = None  # scratch of the long-span prefill kernel, grown on demand

    def close(self):
        if self.handle:
            self.lib.tsattn_destroy(self.handle)
            self.handle = self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    # ---- producers of the path's inputs -------------------------------------------------------
    def quantize_rows(self, x, n_heads, dtype):
        """x: [n_rows, n_heads*d] float32 or bfloat16 -> (uint8 [n_rows, n_heads*d], f32 [n_heads, n_rows])."""
        assert x.is_cuda and x.is_contiguous() and x.dim() == 2
        n_rows, hd = x.shape
        src = capi.SRC_F32 if x.dtype == torch.float32 else capi.SRC_BF16
        assert x.dtype in (torch.float32, torch.bfloat16)
        q = _new(n_rows, hd, torch.uint8, x.device)
        scale = _new(n_heads, n_rows, torch.float32, x.device)
        capi.check(capi.native.quantize_rows(self._h, src, dtype, x, hd * (4 if src == capi.SRC_F32 else 2), n_rows, n_heads, hd // n_heads, q, hd, scale,
                                             n_rows, _raw_stream()))
        return q, scale

    def fill_rope_table(self, head_dim, max_len):
        """The table of FillRopeBuf (gpt/att/rope.cpp:4-24), computed on the host by the library, on the device."""
        host = torch.empty((max_len, head_dim), dtype=torch.float32)
        self.lib.tsattn_fill_rope_table(head_dim, max_len, ctypes.c_void_p(host.data_ptr()))
        return host.to(self.device)

    def _produce_args(self, n_rows, hd, device, n_heads, dtype, pos, rope, rotate_dir, vec_scale, scale_mult, row_major_scale, relu,
                      rope_heads, scale_heads, resid, resid_scale, source=(0, None, 0, 0, 0)):
        """The fields of the producer's arguments (source: dtype, data, pitch, planes, plane stride) and its two results."""
        q = _new(n_rows, hd, torch.uint8, device)
        n_scale = n_heads if scale_heads is None else scale_heads[1]
        if row_major_scale:
            scale, pitch, stride = _new(n_rows, n_scale, torch.float32, device), 1, n_scale
        else:
            scale, pitch, stride = _new(n_scale, n_rows, torch.float32, device), n_rows, 1
        first, count = (0, 0) if scale_heads is None else (int(scale_heads[0]), int(scale_heads[1]))
        resid_pitch = 0
        if resid is not None:
            assert resid.dtype == torch.float32 and resid.shape == (n_rows, hd) and resid.stride(1) == 1
            resid_pitch = resid.stride(0)
        src_dtype, src, src_pitch, planes, plane_stride = source
        return (src_dtype, dtype, n_rows, n_heads, hd // n_heads, src, src_pitch, pos, rope, 0 if rope is None else rope.shape[0], rotate_dir, vec_scale,
                scale_mult, q, hd, scale, pitch, stride, int(bool(relu)), planes, plane_stride, int(rope_heads), first, count, resid, resid_pitch,
                resid_scale), q, scale

    def rope_normalize_rows(self, x, n_heads, dtype, pos=None, rope=None, rotate_dir=1.0, vec_scale=1.0 / 24,
                            scale_mult=1.0, row_major_scale=False, relu=False, rope_heads=0, scale_heads=None,
                            resid=None, resid_scale=1.0):
        """ApplyRope + NormalizeState of the reference's inference path (cpu_infer.cpp:486-499): x [n_rows, H*d]
        float32 or int32 -> (uint8 [n_rows, H*d], f32 scale [H, n_rows], or [n_rows, H] with row_major_scale: what
        the cache append reads); pos int32 [n_rows] or None (no rotation); relu: negative results become 0 (:520-524).
        x may be int32 [planes, n_rows, H*d]: the parts of a split-K product, summed on the fly.  rope_heads: only the
        heads below it are rotated.  scale_heads = (begin, count): scales only for those heads.  resid (f32
        [n_rows, H*d]): resid += x * resid_scale first, in place, and the updated rows are normalised."""
        assert x.is_cuda and x.is_contiguous() and x.dtype in (torch.float32, torch.int32)
        planes = 1
        if x.dim() == 3:
            assert x.dtype == torch.int32
            planes = x.shape[0]
        n_rows, hd = x.shape[-2:]
        source = (capi.SRC_F32 if x.dtype == torch.float32 else capi.SRC_I32, x, hd, planes, n_rows * hd)
        fields, q, scale = self._produce_args(n_rows, hd, x.device, n_heads, dtype, pos, rope, rotate_dir, vec_scale, scale_mult, row_major_scale,
                                              relu, rope_heads, scale_heads, resid, resid_scale, source)
        capi.check(capi.calls.rope_normalize_rows(self._h, _raw_stream(), *fields))
        return q, scale

    def matmul_normalize(self, a, w, n_heads, dtype, scratch=None, **producer):
        """MulForward followed by rope_normalize_rows on its int32 result, as one library call: the projection with its
        normalising epilogue.  Large products with an int8 result never write the int32 sums (the product's kernel
        normalises its own tiles).  a uint8 [m, k], w uint8 [n, k]; scratch: int32 room for 16 * m * n sums (m <= 128) or
        m * n, made here if not given; producer: rope_normalize_rows' keyword arguments.  Returns (uint8 [m, n], scale)
        like rope_normalize_rows."""
        m, k = a.shape
        n = w.shape[0]
        assert w.shape[1] == k and a.stride(1) == 1 and w.stride(1) == 1
        room = (16 if m <= 128 else 1) * m * n
        if scratch is None:
            scratch = torch.empty(room, dtype=torch.int32, device=a.device)
        assert scratch.is_contiguous() and scratch.dtype == torch.int32 and scratch.numel() >= room
        kw = dict(pos=None, rope=None, rotate_dir=1.0, vec_scale=1.0 / 24, scale_mult=1.0, row_major_scale=False, relu=False, rope_heads=0,
                  scale_heads=None, resid=None, resid_scale=1.0)
        kw.update(producer)
        ep, q, scale = self._produce_args(m, n, a.device, n_heads, dtype, kw["pos"], kw["rope"], kw["rotate_dir"], kw["vec_scale"], kw["scale_mult"],
                                          kw["row_major_scale"], kw["relu"], kw["rope_heads"], kw["scale_heads"], kw["resid"], kw["resid_scale"])
        capi.check(capi.calls.matmul_i8(self._h, _raw_stream(), m, n, k, a, a.stride(0), w, w.stride(0), capi.MM_I32_PLANES, 1.0, scratch, n, None, 0,
                                        self._count_at, capi.calls.rope_normalize_rows.pack(*ep)))
        return q, scale

    def kv_product(self, k, value, n_heads, rep=4, mult=1.0):
        """KVProduct (cpu_infer.cpp:320-337): k uint8 (int8 bytes) [n, H*d], value f32/f16 [n, H*d] -> uint8 [n, H*d*rep]."""
        n, hd = k.shape
        assert value.shape == k.shape and value.is_contiguous() and k.stride(1) == 1
        kv = _new(n, hd * rep, torch.uint8, k.device)
        vdt = capi.OUT_F16 if value.dtype == torch.float16 else capi.OUT_F32
        capi.check(capi.native.kv_product(self._h, n, n_heads, hd // n_heads, rep, k, k.stride(0), vdt, value, hd, float(mult), kv, hd * rep,
                                          _raw_stream()))
        return kv

    def matmul_i8(self, a, w, mode=capi.MM_I32, scale=1.0, out=None, workspace=None):
        """MulForward / AddScaled (cpu_infer.cpp:294-316): a uint8 (int8 bytes) [m, k], w uint8 [n, k] (one row per
        output) -> out[m, n]: int32 sums (MM_I32), f32 sums * scale (MM_F32), or out += sums * scale (MM_ADD_SCALED,
        out given, f32)."""
        m, k = a.shape
        n = w.shape[0]
        assert w.shape[1] == k and a.stride(1) == 1 and w.stride(1) == 1
        if mode == capi.MM_I32_PLANES:
            # partial sums [planes, m, n] for a consumer that adds them up (rope_normalize_rows); returns the planes in use
            room = (16 if m <= 128 else 1) * m * n    # K is split only for few rows
            if out is None:
                out = torch.empty(room, dtype=torch.int32, device=a.device)
            assert out.is_contiguous() and out.dtype == torch.int32 and out.numel() >= room
            capi.check(capi.calls.matmul_i8(self._h, _raw_stream(), m, n, k, a, a.stride(0), w, w.stride(0), mode, 1.0, out, n, None, 0, self._count_at))
            planes = self._count.value if m and n else 0
            return out.view(-1)[:planes * m * n].view(planes, m, n)
        if out is None:
            assert mode != capi.MM_ADD_SCALED
            out = _new(m, n, torch.int32 if mode == capi.MM_I32 else torch.float32, a.device)
        assert out.stride(1) == 1 and out.dtype == (torch.int32 if mode == capi.MM_I32 else torch.float32)
        # workspace: a uint8 tensor the caller keeps, room for split-K partial sums when m is small
        room = 0 if workspace is None else workspace.numel() * workspace.element_size()
        capi.check(capi.calls.matmul_i8(self._h, _raw_stream(), m, n, k, a, a.stride(0), w, w.stride(0), mode, float(scale), out, out.stride(0), workspace, room))
        return out

    def embed_rows(self, labels, embed, embed_scale, out=None):
        """The embedding sum of ComputePrediction (cpu_infer.cpp:559-565): labels int32 [n_rows] or [n_rows, L], embed uint8
        (int8 bytes) [n_labels, dim] -> f32 [n_rows, dim]."""
        if labels.dim() == 1:
            labels = labels.view(-1, 1)
        n_rows, per_row = labels.shape
        n_labels, dim = embed.shape
        if out is None:
            out = _new(n_rows, dim, torch.float32, embed.device)
        assert labels.dtype == torch.int32 and labels.is_contiguous() and embed.stride(1) == 1 and out.stride(1) == 1
        capi.check(capi.native.embed_rows(self._h, n_rows, dim, labels, per_row, embed, embed.stride(0), n_labels, float(embed_scale), out, out.stride(0),
                                          _raw_stream()))
        return out

    def _head_scratch(self, n):
        """Scratch of one softmax or sampling call, from the current stream's allocator: calls on several streams may overlap."""
        if n <= capi.HEAD_CHUNK:
            return None, 0
        return torch.empty_strided((capi.HEAD_SCRATCH_BYTES // 4,), (1,), dtype=torch.int32, device=self.device), capi.HEAD_SCRATCH_BYTES

    def softmax_rows(self, vec, scale, bias=None, want_prob=True, argmax=None):
        """The final SoftMax of ComputePrediction (cpu_infer.cpp:340-355, base 2) and the greedy choice: vec int32 [n_rows, n]
        or [planes, n_rows, n] (parts of a split-K product) -> (prob f32 [n_rows, n] or None, argmax int32 [n_rows])."""
        planes = vec.shape[0] if vec.dim() == 3 else 1
        n_rows, n = vec.shape[-2:]
        assert vec.dtype == torch.int32 and vec.is_contiguous()
        prob = _new(n_rows, n, torch.float32, vec.device) if want_prob else None
        if argmax is None:
            argmax = torch.empty_strided((n_rows,), (1,), dtype=torch.int32, device=vec.device)
        capi.check(capi.native.softmax_rows(self._h, n_rows, n, vec, planes, n_rows * n, n, float(scale), bias, prob, n, argmax,
                                              *self._head_scratch(n), _raw_stream()))
        return prob, argmax

    def sample_rows(self, prob, temperature, rnd=None, seed=0, offset=0, choice=None):
        """SampleFromDistr (cpu_infer.cpp:585-599), the Gumbel-max choice: prob f32 [n_rows, n] -> int32 [n_rows].  rnd: the
        caller's uint32 words [n_rows, n], or None = the counter-based generator on (seed, offset)."""
        n_rows, n = prob.shape
        assert prob.dtype == torch.float32 and prob.stride(1) == 1
        if rnd is not None:
            assert rnd.shape == prob.shape and rnd.element_size() == 4 and rnd.stride(1) == 1
        if choice is None:
            choice = torch.empty_strided((n_rows,), (1,), dtype=torch.int32, device=prob.device)
        capi.check(capi.native.sample_rows(self._h, n_rows, n, prob, prob.stride(0), float(temperature), rnd, rnd.stride(0) if rnd is not None else 0,
                                           int(seed), int(offset), choice, *self._head_scratch(n), _raw_stream()))
        return choice

    def build_spans(self, seq_offset, n_tokens, window, doc_start_flag=None):
        """seq_offset: int32 [n_seqs+1] on the device.  Returns (span_start, span_finish) int32 [n_tokens]."""
        st = torch.empty_strided((n_tokens,), (1,), dtype=torch.int32, device=self.device)
        fi = torch.empty_strided((n_tokens,), (1,), dtype=torch.int32, device=self.device)
        capi.check(capi.native.build_spans(self._h, seq_offset.numel() - 1, seq_offset, n_tokens, doc_start_flag, int(window), st, fi, _raw_stream()))
        return st, fi

    def build_span_tiles(self, span_start, span_finish):
        """Per-128-row summary of a span list for compute_val_lookup(span_tiles=...); build once per batch and mask."""
        n = span_start.numel()
        tiles = _new((n + 127) // 128, capi.SPAN_TILE_INTS, torch.int32, self.device)
        capi.check(capi.native.build_span_tiles(self._h, n, span_start, span_finish, tiles, _raw_stream()))
        return tiles

    # ---- prefill --------------------------------------------------------------------------------
    def compute_val_lookup(self, dtype, n_heads, q, k, v, q_scale, k_scale, v_scale, span_start, span_finish,
                           alibi_slope, out=None, out_f16=False, sum_weight_log=None, k_global_scale=None,
                           debug_qk_acc=None, causal_period=0, span_tiles=None, kv_product=None, want_out=True,
                           span_len_hint=0, workspace=None):
        """q,k,v: uint8 [n_tokens, n_heads*d] (row pitch = stride(0)); scales f32 [n_heads, n_tokens] or numbers.
        causal_period: launch-order hint for batches of equal-length sequences under a wide causal window (the
        common sequence length); never changes the result.  span_tiles: what build_span_tiles made of these spans.
        kv_product = (k, kv_out, rep, mult): KVProduct of the f32 result with the tokens' K vectors, written by the same
        launch (k uint8 [n_tokens, H*d], kv_out uint8 [n_tokens, H*rep*d]); with want_out=False the result itself is
        not written and None is returned.
        span_len_hint: typical number of keys per row (the layer's attention width clipped to the sequence length); from
        capi.PREFILL_LONG_SPAN on, with head width 128 and no slope, the call goes through the long-span kernel, which needs a workspace
        (uint8 tensor; by default one that this context keeps and grows on demand)."""
        n_tokens, hd = q.shape
        d = hd // n_heads
        assert want_out or kv_product is not None
        if out is None and want_out:
            out = _new(n_tokens, hd, torch.float16 if out_f16 else torch.float32, q.device)
        qs, qs_const = _scale_arg(q_scale)
        ks, ks_const = _scale_arg(k_scale)
        vs, vs_const = _scale_arg(v_scale)
        pitch = None
        for plane in (qs, ks, vs, sum_weight_log):
            if plane is not None:
                at = plane.stride(0)
                assert pitch is None or at == pitch, "all scale planes must share one pitch"
                pitch = at
        parts = part_stride = 0
        if span_start.dim() == 2:      # rows with several spans: [n_parts, n_tokens], part i = every row's i-th span
            assert span_finish.shape == span_start.shape and span_start.stride(1) == 1 and span_finish.stride() == span_start.stride()
            parts, part_stride = span_start.shape[0], span_start.stride(0)
            assert span_tiles is None or (span_tiles.is_contiguous() and span_tiles.shape[0] == span_start.shape[0])
        out_f16 = out is not None and out.dtype == torch.float16
        kv_k = kv_out = None
        kv_k_pitch = kv_out_pitch = kv_rep = 0
        kv_mult = 0.0
        if kv_product is not None:
            kv_k, kv_out, kv_rep, kv_mult = kv_product
            assert kv_k.stride(1) == 1 and kv_out.stride(1) == 1
            kv_k_pitch, kv_out_pitch = kv_k.stride(0), kv_out.stride(0)
        room = 0
        if span_len_hint >= capi.PREFILL_LONG_SPAN:
            need = int(self.lib.tsattn_prefill_workspace_bytes(n_tokens, n_heads, d))
            if workspace is None and need > 0:
                if self._workspace is None or self._workspace.numel() < need or self._workspace.device != q.device:
                    self._workspace = torch.empty(need, dtype=torch.uint8, device=q.device)
                workspace = self._workspace
            if workspace is not None:
                room = workspace.numel() * workspace.element_size()
        else:
            workspace = None
        capi.check(capi.calls.prefill(
            self._h, _raw_stream(), dtype, capi.OUT_F16 if out_f16 else capi.OUT_F32, n_tokens, n_heads, d, q, k, v, q.stride(0), k.stride(0), v.stride(0),
            qs, ks, vs, n_tokens if pitch is None else pitch, qs_const, ks_const, vs_const, k_global_scale, span_start, span_finish, float(alibi_slope),
            out, 0 if out is None else out.stride(0) * (2 if out_f16 else out.element_size()), sum_weight_log,
            debug_qk_acc, 0 if debug_qk_acc is None else debug_qk_acc.stride(1), span_tiles, int(causal_period),
            kv_k, kv_k_pitch, kv_out, kv_out_pitch, int(kv_rep), float(kv_mult), workspace, room, int(span_len_hint), parts, part_stride))
        return out

    def merge_lookups(self, part_out, part_swl, out=None, out_f16=False, sum_weight_log=None):
        """part_out: f32 [n_parts, n_tokens, H*d], part_swl: f32 [n_parts, H, n_tokens]: prefill results over each row's
        i-th span; returns the attention result over all of a row's spans."""
        n_parts, n_tokens, hd = part_out.shape
        n_heads = part_swl.shape[1]
        if out is None:
            out = torch.empty((n_tokens, hd), dtype=torch.float16 if out_f16 else torch.float32, device=part_out.device)
        a = capi.MergeArgs()
        a.n_parts, a.n_tokens, a.n_heads, a.head_dim = n_parts, n_tokens, n_heads, hd // n_heads
        a.part_out, a.part_out_pitch, a.part_out_stride = _ptr(part_out), part_out.stride(1), part_out.stride(0)
        a.part_swl, a.scale_pitch, a.part_swl_stride = _ptr(part_swl), part_swl.stride(1), part_swl.stride(0)
        a.out_dtype = capi.OUT_F16 if out.dtype == torch.float16 else capi.OUT_F32
        a.out, a.out_pitch = _ptr(out), out.stride(0) * out.element_size()
        if sum_weight_log is not None:
            assert sum_weight_log.stride(0) == a.scale_pitch
            a.sum_weight_log = _ptr(sum_weight_log)
        capi.check(self.lib.tsattn_merge_lookups(self.handle, ctypes.byref(a), _stream_ptr()))
        return out

    def compute_val_lookup_multi(self, dtype, n_heads, q, k, v, q_scale, k_scale, v_scale, span_ptr, spans, alibi_slope,
                                 out_f16=False, sum_weight_log=None, merge=False):
        """Rows with any number of spans, as TAttentionInfo holds them (gpt/att/att.h:24-47): span_ptr int [n_tokens+1],
        spans int [n_spans, 2] (inclusive start, finish), both on the host.  Part i takes every row's i-th span; one
        launch walks all parts (n_span_parts of tsattn_prefill_args), or with merge=True one launch per part and one that
        combines them (tsattn_merge_lookups)."""
        n_tokens = q.shape[0]
        span_ptr = np.asarray(span_ptr, dtype=np.int64)
        spans = np.asarray(spans, dtype=np.int32).reshape(-1, 2)
        counts = span_ptr[1:] - span_ptr[:-1]
        n_parts = max(1, int(counts.max()) if n_tokens else 1)
        st = np.tile(np.arange(n_tokens, dtype=np.int32), (n_parts, 1))
        fi = st - 1                                   # rows that have no i-th span: an empty one
        for i in range(n_parts):
            rows = np.nonzero(counts > i)[0]
            st[i, rows] = spans[span_ptr[rows] + i, 0]
            fi[i, rows] = spans[span_ptr[rows] + i, 1]
        st_d, fi_d = torch.from_numpy(st).to(q.device), torch.from_numpy(fi).to(q.device)
        if not merge:
            return self.compute_val_lookup(dtype, n_heads, q, k, v, q_scale, k_scale, v_scale, st_d, fi_d, alibi_slope,
                                           out_f16=out_f16, sum_weight_log=sum_weight_log)
        part_out = torch.empty((n_parts, n_tokens, q.shape[1]), dtype=torch.float32, device=q.device)
        part_swl = torch.empty((n_parts, n_heads, n_tokens), dtype=torch.float32, device=q.device)
        for i in range(n_parts):
            self.compute_val_lookup(dtype, n_heads, q, k, v, q_scale, k_scale, v_scale, st_d[i], fi_d[i], alibi_slope,
                                    out=part_out[i], sum_weight_log=part_swl[i])
        return self.merge_lookups(part_out, part_swl, out_f16=out_f16, sum_weight_log=sum_weight_log)

    # ---- decode ---------------------------------------------------------------------------------
    def compute_val_lookup_decode(self, cache, q, q_scale, window, alibi_slope, out=None, n_splits=0,
                                  debug_qk_acc=None, max_len=None, append=None, kv_product=None, static_scratch=False):
        """q: uint8 [B, H*d] with q_scale f32 [B, H] (or a number), or bfloat16 [B, H*d] (quantised in the kernel).
        append = (k_new, k_scale_new, v_new, v_scale_new): KVCache.add_vectors fused into the same launches.
        kv_product = (k, kv_out, rep, mult): KVProduct of the result with the token's K vector, written by the same
        launches (k uint8 [B, H*d], kv_out uint8 [B, H*rep*d]).
        static_scratch: go through tsattn_decode_static, the entry point that needs no handle and allocates nothing."""
        B, H, d = cache.n_seqs, cache.n_heads, cache.head_dim
        if out is None:
            out = _new(B, H * d, torch.float32, q.device)
        bf16 = q.dtype == torch.bfloat16
        qs, qs_const = _scale_arg(q_scale if q_scale is not None else 1.0)
        ks, ks_const = _scale_arg(cache.k_scale)
        vs, vs_const = _scale_arg(cache.v_scale)
        seq_stride, head_stride, tok_stride, _ = cache.k.stride()
        s_seq_stride, s_head_stride, _ = (0, 0, 0) if ks is None else ks.stride()
        fields = (cache.dtype, capi.Q_BF16 if bf16 else capi.Q_8BIT, B, H, d, q, q.stride(0) * (2 if bf16 else q.element_size()), qs, qs_const,
                  cache.k, cache.v, seq_stride, head_stride, tok_stride, ks, vs, s_seq_stride, s_head_stride, ks_const, vs_const, cache.cache_len,
                  cache.max_len if max_len is None else int(max_len), int(window), float(alibi_slope), out, int(n_splits))
        if debug_qk_acc is not None or append is not None or kv_product is not None:
            k_new, ks_new, v_new, vs_new = append if append is not None else (None, None, None, None)
            kk, kv_out, rep, mult = kv_product if kv_product is not None else (None, None, 0, 0.0)
            fields += (debug_qk_acc, 0 if debug_qk_acc is None else debug_qk_acc.stride(1), k_new, v_new, 0 if k_new is None else k_new.stride(0),
                       ks_new, vs_new, kk, 0 if kk is None else kk.stride(0), kv_out, 0 if kk is None else kv_out.stride(0), int(rep), float(mult))
        if static_scratch:
            a = capi.DecodeArgs.from_buffer_copy(capi.calls.decode.pack(*fields))
            capi.check(self.lib.tsattn_decode_static(ctypes.byref(a), _stream_ptr()))
        else:
            capi.check(capi.calls.decode(self._h, _raw_stream(), *fields))
        return out


VEC_SCALE = 1.0 / 24      # gpt/train/cpu_infer.cpp:16
STATE_NORM_TILE = 128     # gpt/model_params/model_dim.h:22
COMBINER_REP = 4          # gpt/model_params/model_dim.h:12


def _product_scale_of(scale, width):
    f32 = np.float32
    return float(f32(scale) * f32(VEC_SCALE) * f32(np.sqrt(f32(1.0) / f32(width))))


_product_scale_of_float = functools.lru_cache(maxsize=4096)(_product_scale_of)


def _product_scale(scale, width):
    """A matrix's scale times VEC_SCALE * CalcDotScale(width), in single precision as the reference multiplies it up.  The scale is
    a number or an array or tensor of one; only a float's result is kept (a tensor may change in place)."""
    return (_product_scale_of_float if type(scale) is float else _product_scale_of)(scale, width)


def add_lookup_product(ctx, layer, cache, t, rope, state, workspace=None, scratch=None, pending=None, defer=False):
    """One layer of the int8 inference path for one new token per sequence: AddLookupProduct,
    gpt/train/cpu_infer.cpp:465-527: one library call (tsattn_layer_token) where it serves the shape, else a chain of nine or
    ten (as NTsAttn::TLayerComputer, the C++ form, makes them).
    layer: dict with uint8 (int8 bytes) matrices proj [4*H*d, dim] (the QK, QV, K and V matrices one after the other),
    combiner [dim, 4*H*d], expand [H*d, dim], contract [dim, H*d], floats qv_scale, combiner_scale, contract_scale, and
    width, slope.  cache: KVCache whose value scales are VEC_SCALE; t: int32 [B] positions; rope: table of
    fill_rope_table; state: f32 [B, dim], updated in place.  scratch: dict for buffers kept between calls.
    Returns the attention output [B, H*d].
    defer=True leaves the layer's last state update (contract's AddScaled) undone and returns (attention output,
    pending): the next layer's first normalisation does it when given `pending` (one launch less per layer), and
    flush_state does it after the last layer."""
    B, dim = state.shape
    H, d = cache.n_heads, cache.head_dim
    qsum = H * d
    groups = dim // STATE_NORM_TILE
    sc = scratch if scratch is not None else {}
    fused = _layer_token(ctx, layer, cache, t, rope, state, sc, pending)
    if fused is not None:
        if defer:
            return fused
        flush_state(ctx, fused[1], state)
        return fused[0]
    if "planes" not in sc:
        sc["planes"] = torch.empty((16, B, max(4 * qsum, dim, layer["expand"].shape[0])), dtype=torch.int32, device=state.device)
        sc["v_scale"] = torch.full((B, H), VEC_SCALE, dtype=torch.float32, device=state.device)
    planes_buf, v_scale = sc["planes"], sc["v_scale"]
    if pending is not None:   # the previous layer's contract product, still in parts: state += sum * scale, then normalise
        norm, _ = ctx.rope_normalize_rows(pending[0], groups, capi.I8, resid=state, resid_scale=pending[1])
    else:
        norm, _ = ctx.rope_normalize_rows(state, groups, capi.I8)
    # the four projections as one product; RoPE on the qk and qv heads, per-head normalisation of all four in one call
    proj = ctx.matmul_i8(norm, layer["proj"], mode=capi.MM_I32_PLANES, out=planes_buf)
    key_mult = _product_scale(layer["qv_scale"], dim)
    q4, qv_scale = ctx.rope_normalize_rows(proj, 4 * H, capi.I8, pos=t, rope=rope, scale_mult=key_mult, row_major_scale=True,
                                           rope_heads=2 * H, scale_heads=(H, H))
    qk, qv, k, v = q4[:, :qsum], q4[:, qsum:2 * qsum], q4[:, 2 * qsum:3 * qsum], q4[:, 3 * qsum:]
    if "kv" not in sc:
        sc["kv"] = torch.empty((B, qsum * COMBINER_REP), dtype=torch.uint8, device=state.device)
        sc["val"] = torch.empty((B, qsum), dtype=torch.float32, device=state.device)
    kv, val = sc["kv"], sc["val"]
    fused_kv = (k, kv, COMBINER_REP, 1.0)   # KVProduct written by the attention launches themselves
    if layer["width"] == 0:   # the token attends to the row being written: append first
        cache.add_vectors(qv, qv_scale, v, v_scale)
        ctx.compute_val_lookup_decode(cache, qk, VEC_SCALE, 0, layer["slope"], out=val, kv_product=fused_kv)
    else:
        ctx.compute_val_lookup_decode(cache, qk, VEC_SCALE, layer["width"], layer["slope"], out=val, append=(qv, qv_scale, v, v_scale),
                                      kv_product=fused_kv)
    # combiner; its AddScaled is done by the normalisation that follows
    delta = ctx.matmul_i8(kv, layer["combiner"], mode=capi.MM_I32_PLANES, out=planes_buf)
    norm, _ = ctx.rope_normalize_rows(delta, groups, capi.I8, resid=state,
                                      resid_scale=_product_scale(layer["combiner_scale"], qsum * COMBINER_REP))
    relu_src = ctx.matmul_i8(norm, layer["expand"], mode=capi.MM_I32_PLANES, out=planes_buf)
    relu, _ = ctx.rope_normalize_rows(relu_src, H, capi.I8, relu=True)
    relu_dim = relu_src.shape[-1]
    contract_scale = _product_scale(layer["contract_scale"], relu_dim)
    if defer:
        parts = ctx.matmul_i8(relu, layer["contract"], mode=capi.MM_I32_PLANES, out=planes_buf)
        return val, (parts, contract_scale)
    ctx.matmul_i8(relu, layer["contract"], mode=capi.MM_ADD_SCALED, out=state, workspace=workspace, scale=contract_scale)
    return val


def _layer_token(ctx, layer, cache, t, rope, state, sc, pending):
    """The layer in one library call (tsattn_layer_token: five launches instead of nine), where it serves the shape: returns
    (attention output, pending), or None."""
    B, dim = state.shape
    H, d = cache.n_heads, cache.head_dim
    proj, combiner, expand, contract = layer["proj"], layer["combiner"], layer["expand"], layer["contract"]
    relu_dim = expand.shape[0]
    qsum = H * d
    if (layer["width"] <= 0 or cache.dtype != capi.I8 or not isinstance(cache.k_scale, torch.Tensor) or not isinstance(cache.v_scale, torch.Tensor)
            or state.stride(1) != 1 or (pending is not None and pending[0].shape[0] not in (1, 2, 4))
            or not (proj.is_contiguous() and combiner.is_contiguous() and expand.is_contiguous() and contract.is_contiguous())):
        return None
    room = sc.get("fused")
    if room is None or sc.get("fused_shape") != (B, H, d, dim, relu_dim):
        need = int(ctx.lib.tsattn_layer_token_scratch_bytes(B, H, d, dim, relu_dim))
        if need == 0:
            return None
        room = sc["fused"] = torch.empty(need, dtype=torch.uint8, device=state.device)
        sc["fused_shape"] = (B, H, d, dim, relu_dim)
        planes = torch.empty((4, B, dim), dtype=torch.int32, device=state.device)
        sc["parts"] = {n: planes[:n] for n in (1, 2, 4)}
        sc["val"] = torch.empty((B, qsum), dtype=torch.float32, device=state.device)
    assert proj.shape == (4 * qsum, dim) and combiner.shape == (dim, 4 * qsum) and expand.shape == (relu_dim, dim) and contract.shape == (dim, relu_dim)
    assert t.dtype == torch.int32 and state.dtype == torch.float32 and cache.n_seqs == B
    parts, val = sc["parts"], sc["val"]
    seq_stride, head_stride, tok_stride, _ = cache.k.stride()
    s_seq_stride, s_head_stride, _ = cache.k_scale.stride()
    planes, planes_scale = (None, 0.0) if pending is None else pending
    capi.check(capi.calls.layer_token(
        ctx._h, _raw_stream(), B, H, d, dim, relu_dim, proj, combiner, expand, contract, VEC_SCALE, _product_scale(layer["qv_scale"], dim),
        _product_scale(layer["combiner_scale"], qsum * COMBINER_REP), t, rope, rope.shape[0], cache.k, cache.v, seq_stride, head_stride, tok_stride,
        cache.k_scale, cache.v_scale, s_seq_stride, s_head_stride, 0.0, cache.cache_len, cache.max_len, int(layer["width"]), float(layer["slope"]),
        state, state.stride(0), val, planes, 0 if planes is None else planes.shape[0], planes_scale, parts[4], ctx._count_at, room, room.numel()))
    return val, (parts[ctx._count.value], _product_scale(layer["contract_scale"], relu_dim))


def flush_state(ctx, pending, state):
    """The state update a deferred add_lookup_product left undone; returns NormalizeState of the updated state (what
    ComputePrediction multiplies with the final layer)."""
    norm, _ = ctx.rope_normalize_rows(pending[0], state.shape[1] // STATE_NORM_TILE, capi.I8, resid=state, resid_scale=pending[1])
    return norm


def add_lookup_product_prompt(ctx, layer, cache, seq_offset, pos, rope, state, span_start, span_finish, span_tiles=None,
                              causal_period=0, norm=None, want_norm=False, want_val=True):
    """The same layer for a whole batch of prompt tokens at once (sequences concatenated, seq_offset int32 [B+1], pos
    int32 [n_tokens] = each token's position in its sequence): every token's attention over the earlier tokens of its
    sequence is one tsattn_prefill launch, and the tokens' key and value rows go into the cache in one
    tsattn_cache_fill.  Token by token through add_lookup_product gives the same cache and the same states (a token's
    layer input does not depend on other tokens' outputs of the same layer).  state: f32 [n_tokens, dim], updated in
    place; the spans are those of the layer's width (build_spans).  Returns the attention output (None with
    want_val=False: KVProduct is the attention kernel's last step and nothing else reads the output).
    norm: NormalizeState(state) where the caller has it (the previous layer's second result); want_norm=True returns
    (attention output, NormalizeState(new state)), which the layer's last product then makes as its epilogue."""
    n, dim = state.shape
    H, d = cache.n_heads, cache.head_dim
    qsum = H * d
    groups = dim // STATE_NORM_TILE
    if norm is None:
        norm, _ = ctx.rope_normalize_rows(state, groups, capi.I8)
    # every product with its normalisation as epilogue (large products never write their int32 sums); one scratch
    # buffer for whichever falls back to two launches
    key_mult = _product_scale(layer["qv_scale"], dim)
    room = torch.empty((16 if n <= 128 else 1) * n * max(4 * qsum, dim, layer["expand"].shape[0]), dtype=torch.int32, device=state.device)
    q4, qv_scale = ctx.matmul_normalize(norm, layer["proj"], 4 * H, capi.I8, room, pos=pos, rope=rope, scale_mult=key_mult,
                                        rope_heads=2 * H, scale_heads=(H, H))      # scales as [head][token] planes
    qk, qv, k, v = q4[:, :qsum], q4[:, qsum:2 * qsum], q4[:, 2 * qsum:3 * qsum], q4[:, 3 * qsum:]
    # attention with KVProduct as its last step: the result itself is written only for a caller who wants it
    kv = torch.empty((n, qsum * COMBINER_REP), dtype=torch.uint8, device=state.device)
    val = ctx.compute_val_lookup(capi.I8, H, qk, qv, v, VEC_SCALE, qv_scale, VEC_SCALE, span_start, span_finish, layer["slope"],
                                 span_tiles=span_tiles, causal_period=causal_period, kv_product=(k, kv, COMBINER_REP, 1.0),
                                 want_out=want_val)
    cache.fill_from_prefill(seq_offset, qv, qv_scale, v)       # value scales: the cache's constant VEC_SCALE
    norm, _ = ctx.matmul_normalize(kv, layer["combiner"], groups, capi.I8, room, resid=state,
                                   resid_scale=_product_scale(layer["combiner_scale"], qsum * COMBINER_REP))
    del kv
    relu, _ = ctx.matmul_normalize(norm, layer["expand"], H, capi.I8, room, relu=True)
    relu_dim = relu.shape[-1]
    contract_scale = _product_scale(layer["contract_scale"], relu_dim)
    if want_norm:   # state += product * scale, and the updated state normalised for whoever comes next
        norm_next, _ = ctx.matmul_normalize(relu, layer["contract"], groups, capi.I8, room, resid=state, resid_scale=contract_scale)
        return val, norm_next
    del room
    ctx.matmul_i8(relu, layer["contract"], mode=capi.MM_ADD_SCALED, out=state, scale=contract_scale)
    return val


class KVCache:
    """Planar KV cache [n_seqs][n_heads][max_len][d] 8-bit with f32 row scales [n_seqs][n_heads][max_len];
    the device-resident counterpart of TAttentionVecHistory (gpt/train/cpu_infer.cpp:397-410)."""

    def __init__(self, ctx, dtype, n_seqs, n_heads, max_len, head_dim, const_scales=None):
        dev = ctx.device
        self.ctx, self.dtype = ctx, dtype
        self.n_seqs, self.n_heads, self.max_len, self.head_dim = n_seqs, n_heads, max_len, head_dim
        self.k = torch.zeros((n_seqs, n_heads, max_len, head_dim), dtype=torch.uint8, device=dev)
        self.v = torch.zeros_like(self.k)
        if const_scales is None:
            self.k_scale = torch.zeros((n_seqs, n_heads, max_len), dtype=torch.float32, device=dev)
            self.v_scale = torch.zeros_like(self.k_scale)
        else:
            self.k_scale, self.v_scale = const_scales
        self.cache_len = torch.zeros(n_seqs, dtype=torch.int32, device=dev)

    def add_vectors(self, k_new, k_scale_new, v_new, v_scale_new=None):
        """k_new, v_new: uint8 [n_seqs, n_heads*d]; scales f32 [n_seqs, n_heads] (None with constant scales)."""
        seq_stride, head_stride, tok_stride, _ = self.k.stride()
        planes = isinstance(self.k_scale, torch.Tensor)
        s_seq_stride, s_head_stride, _ = self.k_scale.stride() if planes else (0, 0, 0)
        capi.check(capi.calls.cache_append(
            self.ctx._h, _raw_stream(), self.n_seqs, self.n_heads, self.head_dim, k_new, v_new, k_new.stride(0), k_scale_new, v_scale_new, self.k, self.v,
            seq_stride, head_stride, tok_stride, self.k_scale if planes else None, self.v_scale if planes else None, s_seq_stride, s_head_stride,
            self.cache_len, self.max_len))

    def fill_from_prefill(self, seq_offset, k, k_scale, v, v_scale=None):
        """Append a prefill batch: k, v uint8 [n_tokens, n_heads*d]; scales f32 [n_heads, n_tokens] planes (None
        with constant scales); seq_offset int32 [n_seqs+1] on the device.  Equals add_vectors once per token."""
        n_tokens = k.shape[0]
        assert v.stride(0) == k.stride(0)
        pitches = [p.stride(0) for p in (k_scale, v_scale) if p is not None]
        assert len(set(pitches)) <= 1
        seq_stride, head_stride, tok_stride, _ = self.k.stride()
        planes = isinstance(self.k_scale, torch.Tensor)
        s_seq_stride, s_head_stride, _ = self.k_scale.stride() if planes else (0, 0, 0)
        capi.check(capi.calls.cache_fill(
            self.ctx._h, _raw_stream(), self.n_seqs, self.n_heads, self.head_dim, n_tokens, seq_offset, k, v, k.stride(0), k_scale, v_scale,
            pitches[0] if pitches else n_tokens, self.k, self.v, seq_stride, head_stride, tok_stride, self.k_scale if planes else None,
            self.v_scale if planes else None, s_seq_stride, s_head_stride, self.cache_len, self.max_len))
