"""TurboQuantKVCache: the reference's cache object (turboquant_mlx/cache.py:42-369) over the
HIP codec.  Storage layout, growth rule, fetch modes, serialisation strings and quirks follow
the reference member by member; new vectors are encoded by the GPU straight into the packed
storage (no staging copy) and prefill dequantises straight into the fp16 buffer.
"""
from __future__ import annotations

import torch

from . import attention, ops
from .kvcache import make_mask_for
from .quantizer import gaussian_boundaries, gaussian_codebook
from .rotation import random_diagonal_sign


def _checked_signs(signs, dim, device) -> torch.Tensor:
    """A caller's sign vector as the kernels take it: float32 [dim] of +-1 on `device`."""
    t = torch.as_tensor(signs)
    if t.dim() != 1 or t.numel() != dim:
        raise ValueError(f"a sign vector must have shape ({dim},), got {tuple(t.shape)}")
    t = t.detach().to(device=device, dtype=torch.float32).contiguous()
    if not bool((t.abs() == 1.0).all()):
        raise ValueError("a sign vector holds +1 and -1 only")
    return t


def _check_sign_stream(sign_stream):
    if sign_stream not in ("native", "mlx"):
        raise ValueError(f"sign_stream must be 'native' or 'mlx', got {sign_stream!r}")


class _Quantizer:
    """cache.py:33-39: signs (device) + codebook tables (host).  `signs` overrides the vector that
    random_diagonal_sign derives from `seed` (whose generator is this package's own, not MLX's): the way to
    read a cache written by the reference, which stores only the seed (cache.py:286)."""

    def __init__(self, dim, bits, seed, device, signs=None, sign_stream="native", made=None, tables=None):
        """made: the sign vector of `seed` where the caller has it already; tables: (centroids, boundaries) of `bits`."""
        self.dim = dim
        self.bits = bits
        if signs is not None:
            self.signs = _checked_signs(signs, dim, device)
        else:
            self.signs = made if made is not None else random_diagonal_sign(dim, seed=seed, device=device, stream=sign_stream)
        self.centroids, self.boundaries = tables if tables is not None else _tables(bits)


_TABLE_MASTERS = {}     # the widths' tables as first made outside any mode, never handed out: a cache's are copies (2 us, against 6)


def _tables(bits):
    """(centroids, boundaries) of a width, host tensors of the caller's own; under a mode whatever it makes of them."""
    if torch._C._len_torch_function_stack() or torch._C._len_torch_dispatch_stack():
        centroids = gaussian_codebook(bits)
        return centroids, gaussian_boundaries(centroids)
    if bits not in _TABLE_MASTERS:
        centroids = gaussian_codebook(bits)
        made = centroids, gaussian_boundaries(centroids)
        if any(torch._C._functorch.is_functorch_wrapped_tensor(t) for t in made):
            return made
        _TABLE_MASTERS[bits] = made
    return tuple(t.clone() for t in _TABLE_MASTERS[bits])


def _round_up(n, step):
    return ((n + step - 1) // step) * step


def _is_grouped(t: torch.Tensor, inner: int) -> bool:
    """Whether _group_stride can describe t."""
    if inner == 1 and t.dim() == 3:
        return t.stride(2) == 1 and t.stride(0) == t.shape[1] * t.stride(1)
    return (t.stride(3) == 1 and t.stride(2) == inner and t.stride(1) % inner == 0
            and t.stride(0) == t.shape[1] * t.stride(1))


def _group_stride(t: torch.Tensor, inner: int) -> int:
    """Rows between consecutive (b, h) groups of a [B, H, T, inner] (or [B, H, T] with inner=1)
    tensor whose rows are dense and whose batch stride is H head strides -- true for the cache's
    own allocations and for time-slices of them."""
    if t.is_contiguous():
        shape = t.shape
        if (len(shape) == 4 and shape[3] == inner) or (inner == 1 and len(shape) == 3):
            return shape[2]
    if not _is_grouped(t, inner):
        raise ValueError("cache storage must be row-contiguous [B, H, T, *]; call .contiguous() first")
    return t.stride(1) // inner


class TurboQuantKVCache:
    """PolarQuant KV cache with packed uint32 indices + float32 norms (cache.py:42-51).

    update_and_fetch returns, like the reference:
      fused=True   zero placeholders (attention reads the packed storage directly);
      v_only=True  (zero K placeholder, dequantised V);
      default      dequantised (K, V) from an incrementally maintained fp16 buffer.
    """

    step = 256                                               # cache.py:52

    _DTYPE_MAP = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
    _DTYPE_NAME = {v: k for k, v in _DTYPE_MAP.items()}

    def __init__(self, bits: int = 3, seed: int = 42, fused: bool = False,
                 sparse_v_threshold: float | None = None, v_only: bool = False,
                 encode_variant: str = "mlx", k_signs=None, v_signs=None, sign_stream: str = "native"):
        """k_signs / v_signs ([dim] of +-1, any tensor-like): the rotation's sign vectors, used instead of the ones
        derived from `seed` / `seed + 1` (cache.py:92,96).  sign_stream: which generator derives them when they
        are not given -- "native" (this package's) or "mlx" (the restated stream of rotation.py:47-49, for a
        cache the reference wrote with that seed).  Everything else as the reference (cache.py:54-61)."""
        _check_sign_stream(sign_stream)
        self.quant_bits = bits
        self.seed = seed
        self.offset = 0
        self.fused = fused
        self.sparse_v_threshold = sparse_v_threshold
        self.v_only = v_only
        # "mlx": packed bits equal to the pure-array quantiser (quantizer.py:85-106 + packing.py);
        # "metal": equal to the Metal encoder the reference cache calls (cache.py:140 -> metal.py:147).
        # The two differ only for values within an ulp of a decision boundary.
        self.encode_variant = encode_variant
        self._reset_fields()
        self._k_signs_given, self._v_signs_given = k_signs, v_signs
        self.sign_stream = sign_stream

    def _reset_fields(self):
        self.k_packed = None
        self.k_norms = None
        self.v_packed = None
        self.v_norms = None
        self._k_deq_buf = None
        self._v_deq_buf = None
        self._deq_offset = 0
        self._deq_alloc = 0
        self._k_q = None
        self._v_q = None
        self._k_dim = None
        self._v_dim = None
        self._k_pdim = None
        self._v_pdim = None
        self._dtype = None
        self._step, self._step_key = None, None
        self._k_signs_given, self._v_signs_given = None, None
        self.sign_stream = "native"

    # ---------------------------------------------------------------- setup (cache.py:90-123)
    def _device(self):
        for t in (self.v_packed, self.k_packed):
            if t is not None:
                return t.device
        return torch.device("cuda")

    def _ensure_quantizer(self, k_dim, v_dim, device=None, in_order=True, fill=None):
        """in_order: what uses the sign vectors runs on the current stream (or waits for it), as the inserts do.  False
        makes them with a blocking copy, for a restored cache that may be read from any stream at once.  fill: the sign
        vectors join it, and the caller takes the quantizers back should it not run."""
        new_k, new_v = not self.v_only and self._k_q is None, self._v_q is None
        if not (new_k or new_v):
            return
        device = torch.device(device) if device is not None else self._device()
        ask = []                                             # (seed, dim) of the vectors to derive
        if new_k and self._k_signs_given is None:
            ask.append((self.seed, k_dim))
        if new_v and self._v_signs_given is None:
            ask.append((self.seed + 1, v_dim))
        made = {}
        if in_order and ask and self.sign_stream == "native" and device.type == "cuda" and len({d for _, d in ask}) == 1:
            seeds = [s for s, _ in ask]
            made = dict(zip(seeds, (fill.signs if fill is not None else ops.random_signs)(seeds, ask[0][1], device).unbind(0)))
        tables = _tables(self.quant_bits)
        if new_k:
            self._k_q = _Quantizer(k_dim, self.quant_bits, self.seed, device, self._k_signs_given, self.sign_stream,
                                   made.get(self.seed), tables)
            self._k_dim = k_dim
            self._k_pdim = ops.packed_dim(k_dim, self.quant_bits)
        if new_v:
            self._v_q = _Quantizer(v_dim, self.quant_bits, self.seed + 1, device, self._v_signs_given, self.sign_stream,
                                   made.get(self.seed + 1), tables)
            self._v_dim = v_dim
            self._v_pdim = ops.packed_dim(v_dim, self.quant_bits)

    def _grow(self, old, shape, inner, prev, incoming, dtype, device, fill):
        """Fresh storage [B, H, n(, inner)] holding the first `prev` rows of `old`, zero from row prev + incoming on; the
        rows between are about to be written.  The copy and the zeros join `fill`."""
        new = torch.empty(shape, dtype=dtype, device=device)
        n = shape[2]
        if prev == 0:
            fill.add(new, inner, incoming, n, axis=2)
        elif old is None:                                    # rows that this side never held, as of a restored v_only cache: zeros
            fill.add(new, inner, 0, n, axis=2)
        elif old.dtype == dtype and old.device == new.device and old.shape[:2] == new.shape[:2] and _is_grouped(old, inner):
            fill.add(new, inner, prev + incoming, n, src=old, src_stride=_group_stride(old, inner), copy=prev,
                     axis=2)
        else:
            new.zero_()
            new[:, :, :prev] = old[:, :, :prev]
        return new

    def _ensure_storage(self, B, H, num_new, device, incoming=0):
        """Room for num_new more positions (cache.py:100-123); the caller writes the first `incoming` of them itself."""
        if self._lacks_room(num_new):
            self._reallocate(B, H, _round_up(self.offset + num_new, self.step), device, incoming)

    def _lacks_room(self, num_new):
        return self.v_packed is None or self.offset + num_new > self.v_packed.shape[2]

    def _reallocate(self, B, H, n, device, incoming=0):
        """Fresh contiguous storage of n positions per (b, h) holding the first `offset` positions."""
        fill = ops.StorageFill()
        new = self._grown_storage(B, H, n, device, incoming, fill)
        fill.run()
        self.__dict__.update(new)

    def _grown_storage(self, B, H, n, device, incoming, fill):
        """The tensors of _reallocate by name, whole once `fill` has run.  The cache keeps what it has until then: an
        allocation that fails on the way leaves it as it was."""
        prev, new = self.offset, {}
        if not self.v_only:
            new["k_packed"] = self._grow(self.k_packed, (B, H, n, self._k_pdim), self._k_pdim, prev, incoming, torch.uint32, device, fill)
            new["k_norms"] = self._grow(self.k_norms, (B, H, n), 1, prev, incoming, torch.float32, device, fill)
        new["v_packed"] = self._grow(self.v_packed, (B, H, n, self._v_pdim), self._v_pdim, prev, incoming, torch.uint32, device, fill)
        new["v_norms"] = self._grow(self.v_norms, (B, H, n), 1, prev, incoming, torch.float32, device, fill)
        return new

    # ---------------------------------------------------------------- codec calls
    def _encode(self, x, q, packed, norms, B, H, S, dim, prev):
        ops.encode_into(x.reshape(-1, dim), q.signs, q.boundaries, packed, norms,
                        n_groups=B * H, rows_per_group=S,
                        packed_group_stride=_group_stride(packed, packed.shape[3]),
                        norms_group_stride=_group_stride(norms, 1), dim=dim, bits=self.quant_bits,
                        variant=self.encode_variant, packed_row_offset=prev, norms_row_offset=prev)

    def _encode_pair(self, keys, values, B, H, S, k_dim, v_dim, prev):
        """Key and value rows at positions prev .. prev + S - 1, in one launch where one describes both."""
        gs = _group_stride(self.v_packed, self._v_pdim)
        if (keys.dtype == values.dtype and k_dim == v_dim and _group_stride(self.k_packed, self._k_pdim) == gs
                and _group_stride(self.k_norms, 1) == gs and _group_stride(self.v_norms, 1) == gs):
            kq, vq = self._k_q, self._v_q
            ops.encode_kv_into(keys, kq.signs, self.k_packed, self.k_norms, values, vq.signs, self.v_packed, self.v_norms,
                               vq.boundaries, n_groups=B * H, rows_per_group=S, group_stride=gs, dim=v_dim,
                               bits=self.quant_bits, variant=self.encode_variant, row_offset=prev)
        else:
            self._encode(values, self._v_q, self.v_packed, self.v_norms, B, H, S, v_dim, prev)
            self._encode(keys, self._k_q, self.k_packed, self.k_norms, B, H, S, k_dim, prev)

    def _sides(self):
        """(packed, norms, quantizer, dim) of the stored tensors."""
        v = (self.v_packed, self.v_norms, self._v_q, self._v_dim)
        return [v] if self.v_only else [(self.k_packed, self.k_norms, self._k_q, self._k_dim), v]

    def _dequant_rows(self, outs, B, H, start, count, out_start):
        """Positions start .. start + count - 1 of every (b, h) of each stored tensor into rows out_start .. of its
        contiguous [B, H, T, dim] tensor in `outs` (None: not wanted): one launch where one describes both."""
        sides = self._sides()
        if len(sides) == 2 and outs[0] is not None and outs[1] is not None:
            (kp, kn, kq, kd), (vp, vn, vq, vd) = sides
            ko, vo = outs
            gs = _group_stride(vp, vp.shape[3])
            if (ko.dtype == vo.dtype and ko.shape == vo.shape and _group_stride(kp, kp.shape[3]) == gs
                    and _group_stride(kn, 1) == gs and _group_stride(vn, 1) == gs and kq.centroids is vq.centroids):
                ops.dequant_kv_into(kp, kn, kq.signs, ko, vp, vn, vq.signs, vo, vq.centroids, n_groups=B * H,
                                    rows_per_group=count, group_stride=gs, out_group_stride=vo.shape[2], dim=vd,
                                    bits=self.quant_bits, row_offset=start, out_row_offset=out_start)
                return
        for (packed, norms, q, dim), out in zip(sides, outs):
            if out is None:
                continue
            ops.dequant_into(packed, norms, q.centroids, q.signs, out, n_groups=B * H, rows_per_group=count,
                             packed_group_stride=_group_stride(packed, packed.shape[3]),
                             norms_group_stride=_group_stride(norms, 1), out_group_stride=out.shape[2], dim=dim,
                             bits=self.quant_bits, packed_row_offset=start, norms_row_offset=start, out_row_offset=out_start)

    def _full_dequant(self, packed, norms, q, dim, B, H, total, dtype):
        """cache.py:125-129: every stored position, as a fresh [B, H, total, dim] tensor."""
        out = torch.empty((B, H, total, dim), dtype=dtype, device=packed.device)
        ops.dequant_into(packed, norms, q.centroids, q.signs, out, n_groups=B * H, rows_per_group=total,
                         packed_group_stride=_group_stride(packed, packed.shape[3]),
                         norms_group_stride=_group_stride(norms, 1),
                         out_group_stride=total, dim=dim, bits=self.quant_bits)
        return out

    def _buffers(self, B, H, n, dtypes, device):
        return [torch.empty((B, H, n, side[3]), dtype=dt, device=device) for side, dt in zip(self._sides(), dtypes)]

    def _incremental(self, bufs, B, H, prev, total, dtypes):
        """Decode step of cache.py:171-180 / 192-207: dequantise only the new rows, in half precision (dequant_fp16),
        cast to the cache dtype, into the persistent buffers."""
        if total > bufs[0].shape[2]:
            fill = ops.StorageFill()
            grown = self._buffers(B, H, _round_up(total, self.step), dtypes, bufs[0].device)
            for new, old in zip(grown, bufs):
                if new.dtype == old.dtype and new.shape[:2] == old.shape[:2] and new.shape[3] == old.shape[3]:
                    fill.add(new, new.shape[3], total, new.shape[2], src=old, src_stride=old.shape[2], copy=self._deq_offset, axis=2)
                else:                                        # rows of another dtype than before: cast, as a slice assignment does
                    new[:, :, :self._deq_offset] = old[:, :, :self._deq_offset]
                    fill.add(new, new.shape[3], total, new.shape[2], axis=2)
            fill.run()
            bufs = grown
        half = [dt == torch.float16 for dt in dtypes]
        if any(half):
            self._dequant_rows([buf if h else None for buf, h in zip(bufs, half)], B, H, prev, total - prev, prev)
        if not all(half):                                    # rows of another dtype: cast to theirs, then to the buffer's
            tmp = self._buffers(B, H, total - prev, [torch.float16] * len(bufs), bufs[0].device)
            self._dequant_rows([None if h else rows for rows, h in zip(tmp, half)], B, H, prev, total - prev, 0)
            for buf, rows, dt in zip(bufs, tmp, dtypes):
                if dt != torch.float16:
                    buf[:, :, prev:total].copy_(rows if buf.dtype == dt else rows.to(dt))
        return bufs

    # ---------------------------------------------------------------- cache.py:131-218
    def _zero_like(self, t: torch.Tensor, fill, made: dict) -> torch.Tensor:
        """A zero scalar of t's dtype on t's device, made once: the source of the stride-0 placeholders
        (a fresh one per step would cost a fill launch each).  A new one's bytes join `fill`, itself `made`, which
        the caller keeps once the fill has run."""
        key = (t.dtype, t.device)
        z = self.__dict__.setdefault("_zero_scalars", {}).get(key, made.get(key))
        if z is None:
            base = t.new_empty(8)
            fill.add(base, 1, 0, 8)
            z = made[key] = base[0]
        return z

    def reserve(self, B: int, H: int, n_positions: int, dim: int, device="cuda"):
        """Allocate storage for `n_positions` more positions now, so that steps recorded in a HIP graph keep
        their addresses for that long (storage otherwise grows in steps of 256, which reallocates)."""
        device = torch.device(device)
        self._ensure_quantizer(dim, dim, device)
        self._ensure_storage(B, H, n_positions, device)

    def decode_step(self, queries: torch.Tensor, keys: torch.Tensor, values: torch.Tensor, attn_scale: float,
                    position: torch.Tensor | None = None, out: torch.Tensor | None = None):
        """Encode one token and attend in one library call: the result of `update_and_fetch(keys, values)`
        followed by `turboquant_attention(queries, self, attn_scale, fused=True)` (no mask, no threshold) on
        a cache with packed keys and values.  queries (B, n_heads, 1, dim), keys / values (B, n_kv, 1, dim)
        -> (B, n_heads, 1, dim) in queries.dtype.  Not in the reference, where the two halves are separate
        calls of the model's attention layer (cache.py:131-165, fused_attention.py:20-125).

        With `position` (one-element int64 GPU tensor holding the cache's current offset) the kernels read the
        insert position and the attended length from it when they run, so the step can be recorded in a HIP
        graph once and replayed while the caller advances the tensor; set `offset` afterwards.  `out`
        (B, n_heads, dim) receives the result when given."""
        B, n_q, S_q, dim = queries.shape
        H = values.shape[1]
        ok = (not self.v_only and S_q == 1 and values.shape[2] == 1 and keys.shape == values.shape
              and keys.shape[3] == dim and n_q % H == 0 and values.is_cuda
              and queries.dtype in ops._DTYPES and keys.dtype in ops._DTYPES and values.dtype in ops._DTYPES
              and ops.vonly_sparse_supported(dim, self.quant_bits, n_q // H))
        if ok:
            self._dtype = keys.dtype
            self._ensure_quantizer(dim, dim, values.device)
            self._ensure_storage(B, H, 1, values.device)
            key = (self.k_packed.data_ptr(), self.k_norms.data_ptr(), self.v_packed.data_ptr(),
                   self.v_norms.data_ptr(), self.v_packed.shape[2], n_q)
            if self._step_key != key:
                try:
                    self._step = ops.PackedStep(self.k_packed, self.k_norms, self.v_packed, self.v_norms,
                                                self._k_q.signs, self._v_q.signs, self._v_q.boundaries,
                                                self._v_q.centroids, dim=dim, n_rep=n_q // H, bits=self.quant_bits,
                                                variant=self.encode_variant)
                    self._step_key = key
                except ValueError:                 # storage handed in through `state` as slices
                    ok = False
        if not ok:
            if position is not None:
                raise ValueError("a step with a device-side position needs one new token, dim 128, "
                                 "n_rep <= 16 and contiguous storage")
            self.update_and_fetch(keys, values)
            return attention.turboquant_attention(queries, self, attn_scale, fused=True)
        if position is not None and (position.dtype != torch.int64 or position.numel() != 1 or not position.is_cuda):
            raise ValueError("a device-side position must be a one-element int64 tensor on the GPU")
        sb, sh_, _, sd = self._step.shape
        if (sb, sh_, sd) != (B, H, dim) or values.shape[0] != B or not (queries.is_cuda and keys.is_cuda):
            raise ValueError(f"the cache stores {sb} x {sh_} groups of dim {sd} on the GPU; got queries {tuple(queries.shape)}, "
                             f"keys {tuple(keys.shape)} on {keys.device}")
        if out is None:
            res = torch.empty((B, n_q, 1, dim), dtype=queries.dtype, device=queries.device)
        elif out.numel() != B * n_q * dim or not out.is_contiguous() or not out.is_cuda or out.dtype not in ops._DTYPES:
            raise ValueError(f"out must be a contiguous GPU tensor of {B} x {n_q} x {dim} elements")
        else:
            res = out
        ops.step_call_unchecked(self._step, keys.contiguous(), values.contiguous(), queries.contiguous(),
                                self.offset if position is None else position, attn_scale, res, packed=True)
        self.offset += 1          # _deq_offset stays behind: the next unfused fetch dequantises the whole cache
        return res if res.dim() == 4 else res[:, :, None, :]

    def update_and_fetch(self, keys: torch.Tensor, values: torch.Tensor):
        B, H, S, k_dim = keys.shape
        v_dim = values.shape[3]
        device = values.device
        self._dtype = keys.dtype
        prev = self.offset
        total = prev + S
        fill = ops.StorageFill()
        held = self._k_q, self._v_q
        try:
            self._ensure_quantizer(k_dim, v_dim, device, fill=fill)
            new = self._grown_storage(B, H, _round_up(total, self.step), device, S, fill) if self._lacks_room(S) else {}
            dtypes = [values.dtype] if self.v_only else [keys.dtype, values.dtype]
            fresh = None if self.fused else self._fetch_buffers(B, H, prev, total, dtypes, device, fill)
            made = {}
            zeros = [self._zero_like(t, fill, made) for t in ((keys, values) if self.fused else (keys,) if self.v_only else ())]
            fill.run()                                       # every allocation has succeeded: now the cache may change
        except BaseException:
            self._k_q, self._v_q = held                      # their sign vectors may not have been made
            raise
        self.__dict__.update(new)
        if made:
            self._zero_scalars.update(made)
        if self.v_only:
            self._encode(values, self._v_q, self.v_packed, self.v_norms, B, H, S, v_dim, prev)
        else:
            self._encode_pair(keys, values, B, H, S, k_dim, v_dim, prev)
        self.offset = total

        if self.fused:
            # zero placeholders of the right shape that own no memory (stride-0 views)
            return zeros[0].expand(B, H, total, k_dim), zeros[1].expand(B, H, total, v_dim)
        out = self._fetch(fresh, B, H, prev, total, dtypes)
        if self.v_only:
            return zeros[0].expand(B, H, total, k_dim), out[0]
        return out[0], out[1]

    def _fetch_buffers(self, B, H, prev, total, dtypes, device, fill):
        """The dequantised buffers a fetch of the first `total` positions goes to: None where the new rows join the present
        ones (cache.py:171-180, 192-207), else fresh step-rounded ones, whose tails join `fill` (cache.py:182-188, 208-218)."""
        if total - prev <= 4 and self._v_deq_buf is not None and self._deq_offset == prev:
            return None
        bufs = self._buffers(B, H, _round_up(total, self.step), dtypes, device)
        for buf in bufs:
            fill.add(buf, buf.shape[3], total, buf.shape[2], axis=2)
        return bufs

    def _fetch(self, fresh, B, H, prev, total, dtypes):
        """Dequantise into the buffers of _fetch_buffers; views of their first `total` positions."""
        if fresh is None:
            bufs = self._incremental([self._v_deq_buf] if self.v_only else [self._k_deq_buf, self._v_deq_buf],
                                     B, H, prev, total, dtypes)
        else:
            bufs = fresh
            self._dequant_rows(bufs, B, H, 0, total, 0)
        self._v_deq_buf = bufs[-1]
        if not self.v_only:
            self._k_deq_buf = bufs[0]
        self._deq_alloc = self._v_deq_buf.shape[2]
        self._deq_offset = total
        return [buf[:, :, :total] for buf in bufs]

    def fetch_values(self, prev, dtype):
        """The dequantised values of a v_only cache whose positions from `prev` on an owner has encoded itself."""
        B, H = self.v_packed.shape[:2]
        fill = ops.StorageFill()
        fresh = self._fetch_buffers(B, H, prev, self.offset, [dtype], self.v_packed.device, fill)
        fill.run()
        return self._fetch(fresh, B, H, prev, self.offset, [dtype])[0]

    # ---------------------------------------------------------------- cache.py:220-247
    def empty(self):
        return self.v_packed is None if self.v_only else self.k_packed is None

    @property
    def nbytes(self):
        total = 0
        if self.k_packed is not None:
            B, H = self.k_packed.shape[:2]
            total += B * H * self.offset * (self.k_packed.shape[3] * 4 + 4)
        if self.v_packed is not None:
            B, H = self.v_packed.shape[:2]
            total += B * H * self.offset * (self.v_packed.shape[3] * 4 + 4)
        return total

    @property
    def compression_ratio(self) -> float:
        """FP16 bytes of the uncompressed K+V divided by packed + norm bytes (cache.py:234-247)."""
        total = self.nbytes
        if total == 0:
            return 1.0
        ref = self.v_packed if self.v_only else self.k_packed
        if ref is None:
            return 1.0
        B, H = ref.shape[0], ref.shape[1]
        fp16_bytes = B * H * self.offset * ((self._k_dim or 0) + (self._v_dim or 0)) * 2
        return fp16_bytes / total

    # ---------------------------------------------------------------- cache.py:249-297
    @property
    def state(self):
        if self.v_packed is None and self.k_packed is None:
            return []
        parts = []
        if self.k_packed is not None:
            parts += [self.k_packed[..., :self.offset, :], self.k_norms[..., :self.offset]]
        if self.v_packed is not None:
            parts += [self.v_packed[..., :self.offset, :], self.v_norms[..., :self.offset]]
        return parts

    @state.setter
    def state(self, v):
        if not v:
            return
        if len(v) == 4:
            self.k_packed, self.k_norms, self.v_packed, self.v_norms = v
            self.offset = self.k_packed.shape[2]
        elif len(v) == 2:
            self.v_packed, self.v_norms = v
            self.offset = self.v_packed.shape[2]
        else:
            raise ValueError(f"Expected 2 (v_only) or 4 arrays in state, got {len(v)}")

    @property
    def meta_state(self):
        dtype_str = self._DTYPE_NAME.get(self._dtype, "float16")
        return (f"{self.offset},{self.quant_bits},{self.seed},"
                f"{self._k_dim or 0},{self._v_dim or 0},{dtype_str}")

    @meta_state.setter
    def meta_state(self, v):
        parts = v.split(",")
        self.offset, self.quant_bits, self.seed = int(parts[0]), int(parts[1]), int(parts[2])
        self._k_dim = int(parts[3]) or None
        self._v_dim = int(parts[4]) or None
        self._dtype = self._DTYPE_MAP.get(parts[5], torch.float16) if len(parts) > 5 else torch.float16

    # ---------------------------------------------------------------- cache.py:299-334
    def is_trimmable(self):
        return True

    def trim(self, n):
        n = min(self.offset, n)
        self.offset -= n
        self._k_deq_buf = None
        self._v_deq_buf = None
        self._deq_offset = 0
        self._deq_alloc = 0
        return n

    def size(self):
        return self.offset

    def make_mask(self, N, return_array: bool = False, window_size=None):
        return make_mask_for(self.offset, N, return_array, window_size, self._device())

    # ---------------------------------------------------------------- cache.py:336-369
    @classmethod
    def from_state(cls, state, meta_state, k_signs=None, v_signs=None, sign_stream: str = "native"):
        """cache.py:336-369.  The serialised cache carries its seed, not its sign vectors (cache.py:286): a cache
        written with explicit signs -- or by the reference, whose seed-to-signs generator is MLX's -- restores
        correctly only with the same k_signs / v_signs given here, or, for a reference-written cache whose
        vectors were not kept, with sign_stream="mlx" (the seed is then expanded by the restated MLX stream)."""
        _check_sign_stream(sign_stream)
        obj = cls.__new__(cls)
        obj._reset_fields()
        obj._k_signs_given, obj._v_signs_given = k_signs, v_signs
        obj.sign_stream = sign_stream
        obj.fused = False
        obj.sparse_v_threshold = None
        obj.v_only = False
        obj.encode_variant = "mlx"
        obj.meta_state = meta_state
        obj.state = state
        if obj.k_packed is not None:
            obj._k_pdim = obj.k_packed.shape[-1]
        if obj.v_packed is not None:
            obj._v_pdim = obj.v_packed.shape[-1]
        if obj._k_dim is not None and obj._v_dim is not None:
            obj._ensure_quantizer(obj._k_dim, obj._v_dim, in_order=False)
        return obj

    # ---------------------------------------------------------------- from_kvcache
    @classmethod
    def from_kvcache(cls, kv, bits: int = 3, seed: int = 42, **kwargs):
        """Compress an existing uncompressed cache (anything with .keys/.values/.offset, layout
        [B, H, T, D]).  Defined as: construct an empty cache, then update_and_fetch with the valid
        prefix.  The reference tree has no such constructor; its README shows the name on the
        mixed-quant cache of its mlx-lm fork (README.md:41-46)."""
        obj = cls(bits=bits, seed=seed, **kwargs)
        if kv.keys is not None and kv.offset > 0:
            obj.update_and_fetch(kv.keys[..., :kv.offset, :], kv.values[..., :kv.offset, :])
        return obj
