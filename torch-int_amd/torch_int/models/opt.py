"""INT8 OPT blocks on the MI355X kernels (upstream ``torch_int/models/opt.py``).

``Int8OPTAttention`` and ``Int8OPTDecoderLayer`` keep upstream's constructor
signatures, sub-module names, scale algebra and forward semantics.  The
decoder / model / causal-LM wrappers carry their own small OPT scaffolding
(token + learned position embeddings with the +2 offset, additive causal
mask, final LayerNorm, fp ``lm_head``) instead of borrowing methods from a
particular ``transformers`` release; any object with OPTConfig's field names
works as ``config``.
"""
import ctypes
import threading
import weakref
from dataclasses import dataclass
from typing import List, Optional, Tuple

import torch
from torch import nn

from .. import _hip_ext
from ..nn._scalars import read_scalars
from ..nn.bmm import BMM_S8T_S8N_F32T, BMM_S8T_S8N_S8T
from ..nn.fused import LayerNormQ
from ..nn.linear import W8A8B8O8Linear, W8A8B8O8LinearReLU, W8A8BFP32OFP32Linear


class _KVBuffer:
    """Backing store of one growing K or V cache tensor: ``buf`` is [bsz, heads, capacity, head_dim] and the
    first ``filled`` positions hold tokens.  The tensors handed out as ``past_key_value`` are views
    ``buf[:, :, :n]`` that carry a reference to this object.  ``bare``: the tokens are still elsewhere, and the kernel that
    appends the next one moves them here."""
    __slots__ = ("buf", "filled", "bare", "__weakref__")

    def __init__(self, buf, filled, bare=False):
        self.buf, self.filled, self.bare = buf, filled, bare


def _kv_room(past, new):
    """The buffer behind ``past`` when ``new`` can be written right after it, else None."""
    kv = getattr(past, "_ti_kv", None)
    S, T = past.shape[2], new.shape[2]
    if (kv is not None and kv.filled == S and S + T <= kv.buf.shape[2] and past.data_ptr() == kv.buf.data_ptr()
            and past.stride() == kv.buf.stride() and past.shape[:2] == new.shape[:2] and past.shape[3] == new.shape[3]
            and past.dtype == new.dtype and past.device == new.device):
        return kv
    return None


def _kv_room_for(past, T):
    """``_kv_room`` for T new positions that will be written by a kernel (there is no tensor to compare with)."""
    kv = getattr(past, "_ti_kv", None)
    S = past.shape[2]
    if (kv is not None and kv.filled == S and S + T <= kv.buf.shape[2] and past.data_ptr() == kv.buf.data_ptr()
            and past.stride() == kv.buf.stride()):
        return kv
    return None


def _kv_empty(past, T):
    """A bare buffer for ``past`` with room for T + max(64, a quarter of the length) further positions."""
    S = past.shape[2]
    cap = -(-(S + T + max(64, (S + T) // 4)) // 16) * 16
    buf = torch.empty((past.shape[0], past.shape[1], cap, past.shape[3]), dtype=past.dtype, device=past.device)
    return _KVBuffer(buf, S, bare=True)


def _kv_fresh(past, T):
    """A new buffer holding ``past`` with room behind it."""
    kv = _kv_empty(past, T)
    kv.buf[:, :, :past.shape[2]].copy_(past)
    kv.bare = False
    return kv


_kv_lock = threading.Lock()


def _kv_claim(past):
    """The buffer with room for one more position behind ``past``, taken, or None: it counts as filled from here on, so that nobody
    else who continues the same past (another thread, while this one's layers are on their way) is given the same position."""
    with _kv_lock:
        kv = _kv_room_for(past, 1)
        if kv is not None:
            kv.filled = past.shape[2] + 1
        return kv


def _kv_rooms(past):
    """Buffers for one more position behind a layer's (key, value) cache, taken (``_kv_claim``), both of them bare where there is no
    room and the kernel that appends can read the cache as it lies; None when a kernel cannot write there."""
    kk, vv = _kv_claim(past[0]), _kv_claim(past[1])
    if kk is None or vv is None:
        new = _kv_empty if kk is None and vv is None and _hip_ext.cache_rows_movable(past) else _kv_fresh
        if kk is None:
            kk = new(past[0], 1)
            kk.filled += 1
        if vv is None:
            vv = new(past[1], 1)
            vv.filled += 1
    kb, vb = kk.buf, vv.buf
    if kb.data_ptr() % 16 or vb.data_ptr() % 16 or not (kb.is_contiguous() and vb.is_contiguous() and kb.shape == vb.shape):
        _kv_give_back((kk, vv))
        return None
    return kk, vv


def _kv_give_back(rooms):
    for kv in rooms:
        kv.filled -= 1


class _KVChain:
    """The cache buffers of the layers of a model, as the pass that appended to them last left them: what the pass that
    continues it compares the cache it is given with, instead of looking at every tensor of it anew.  Every buffer holds the same
    positions of the same heads.  It keeps none of them alive: the tensors of a cache do, each its own."""
    __slots__ = ("rooms", "keys", "values", "shape", "stride", "cap", "device")

    def __reduce__(self):   # a copied or pickled cache has buffers of its own
        return _no_plan, ()

    @staticmethod
    def of(rooms):
        """The chain of ``rooms`` ((key buffer, value buffer) for every layer), or None where they differ in size."""
        first = rooms[0][0].buf
        if any(kv.buf.shape != first.shape or kv.buf.device != first.device or kv.bare for pair in rooms for kv in pair):
            return None
        chain = _KVChain()
        chain.rooms = [(weakref.ref(kk), weakref.ref(vv)) for kk, vv in rooms]
        chain.keys, chain.values = (_hip_ext.pointers([pair[i].buf.data_ptr() for pair in rooms]) for i in (0, 1))
        chain.shape, chain.stride, chain.cap, chain.device = first.shape, first.stride(), first.shape[2], first.device
        return chain

    def claim(self, cache, S):
        """The buffers with position S - 1 taken in each, as ``_kv_claim`` takes it, when ``cache`` is what they hold before it,
        else None."""
        held = (self.shape[0], self.shape[1], S - 1, self.shape[3])
        if S > self.cap:
            return None
        rooms = []
        for i, (kk, vv) in enumerate(self.rooms):
            key, value = cache[i]
            pair = getattr(key, "_ti_kv", None), getattr(value, "_ti_kv", None)
            if not (pair[0] is not None and pair[1] is not None and kk() is pair[0] and vv() is pair[1] and key.shape == held
                    and value.shape == held and key.stride() == self.stride and value.stride() == self.stride
                    and key.data_ptr() == self.keys[i] and value.data_ptr() == self.values[i]):
                return None
            rooms.append(pair)
        with _kv_lock:
            if any(kk.filled != S - 1 or vv.filled != S - 1 for kk, vv in rooms):
                return None
            for kk, vv in rooms:
                kk.filled = vv.filled = S
        return rooms


def _kv_append_in_layer(plan, hidden, mask, rooms, past, S, **chain):
    """One layer's decode step, which appends to ``rooms`` (``_kv_rooms(past)``) and moves the past there if they are bare."""
    kk, vv = rooms
    _hip_ext.opt_layer_decode(plan, hidden, mask, kk.buf, vv.buf, S, past=past if kk.bare else None, **chain)
    kk.bare = vv.bare = False
    return _kv_view(kk, S), _kv_view(vv, S)


def _kv_view(kv, n):
    out = kv.buf.narrow(2, 0, n)
    out._ti_kv = kv
    return out


def _kv_append(past, new):
    """``torch.cat([past, new], dim=2)`` for [bsz, heads, len, head_dim] cache tensors without re-copying the
    past: when ``past`` is a view handed out by an earlier call and nothing was appended after it, ``new`` is
    written into the spare room behind it and a longer view of the same buffer is returned; the values
    ``past`` shows never change.  Otherwise (first decode step, a cache that was re-indexed or sliced by the
    caller, a second continuation of the same past, no room left) the result is built in a fresh buffer."""
    S, T = past.shape[2], new.shape[2]
    kv = _kv_room(past, new) or _kv_fresh(past, T)
    kv.buf[:, :, S:S + T].copy_(new)
    kv.filled = S + T
    return _kv_view(kv, S + T)


def _kv_append_pair(past_k, past_v, new_k, new_v):
    """``_kv_append`` for the key and the value cache of one layer, with a single copy kernel when both live
    in HIP buffers of the same shape."""
    S, T = past_k.shape[2], new_k.shape[2]
    if past_v.shape[2] != S or new_v.shape[2] != T:
        return _kv_append(past_k, new_k), _kv_append(past_v, new_v)
    kk = _kv_room(past_k, new_k) or _kv_fresh(past_k, T)
    vv = _kv_room(past_v, new_v) or _kv_fresh(past_v, T)
    if _hip_ext.can_kv_append(new_k, new_v, kk.buf, vv.buf):
        _hip_ext.kv_append(new_k, new_v, kk.buf, vv.buf, S, checked=True)
    else:
        kk.buf[:, :, S:S + T].copy_(new_k)
        vv.buf[:, :, S:S + T].copy_(new_v)
    kk.filled = vv.filled = S + T
    return _kv_view(kk, S + T), _kv_view(vv, S + T)


class Int8OPTAttention(nn.Module):
    """Multi-head self-attention with int8 projections and int8 Q.K^T / P.V products.

    upstream: ``torch_int/models/opt.py:22-199``.

    ``kv_cache_in_place`` (class attribute, default True): the (key, value) tensors returned for
    ``past_key_value`` reuse one buffer with spare room, so a decode step appends its token instead of
    re-copying the whole cache (see ``_kv_append``).  They are then views that are packed per head but not
    across heads; set it to False to get upstream's freshly concatenated contiguous tensors.
    """
    kv_cache_in_place = True
    # False: the probabilities come from upstream's own chain of torch ops between the two products (mask add,
    # clamp, softmax, * 127, round, int8 cast; models/opt.py:144-178) instead of the fused kernels, whose
    # e * (127 / sum) differs from (e / sum) * 127 by one LSB on a small fraction of the probabilities.
    fused_softmax = True

    def __init__(self, embed_dim: int, num_heads: int):
        super().__init__()
        self.embed_dim = embed_dim
        self.num_heads = num_heads
        self.head_dim = embed_dim // num_heads
        if self.head_dim * num_heads != embed_dim:
            raise ValueError(f"embed_dim must be divisible by num_heads (got `embed_dim`: {embed_dim}"
                             f" and `num_heads`: {num_heads}).")
        self.attention_weight_scale = 1.0
        self.qk_bmm = BMM_S8T_S8N_F32T(1.0)
        self.pv_bmm = BMM_S8T_S8N_S8T(1.0)
        self.k_proj = W8A8B8O8Linear(embed_dim, embed_dim)
        self.v_proj = W8A8B8O8Linear(embed_dim, embed_dim)
        self.q_proj = W8A8B8O8Linear(embed_dim, embed_dim)
        self.out_proj = W8A8BFP32OFP32Linear(embed_dim, embed_dim)

    @staticmethod
    @torch.no_grad()
    def from_float(module, input_scale: float, q_output_scale: float, k_output_scale: float,
                   v_output_scale: float, out_input_scale: float):
        """``module`` is an fp OPT attention (attributes embed_dim, num_heads, scaling,
        q/k/v/out_proj).  The 1/sqrt(d) factor is folded into q_proj, in place on ``module``."""
        q = Int8OPTAttention(module.embed_dim, module.num_heads)
        q_output_scale = q_output_scale * module.scaling
        module.q_proj.weight *= module.scaling
        module.q_proj.bias *= module.scaling
        q.q_proj = W8A8B8O8Linear.from_float(module.q_proj, input_scale, q_output_scale)
        q.k_proj = W8A8B8O8Linear.from_float(module.k_proj, input_scale, k_output_scale)
        q.v_proj = W8A8B8O8Linear.from_float(module.v_proj, input_scale, v_output_scale)
        q.out_proj = W8A8BFP32OFP32Linear.from_float(module.out_proj, out_input_scale)
        q.qk_bmm = BMM_S8T_S8N_F32T.from_scale(q_output_scale, k_output_scale)
        # probabilities are quantised with scale 1/127
        q.pv_bmm = BMM_S8T_S8N_S8T.from_scale(1.0 / 127, v_output_scale, out_input_scale)
        return q

    def _qkv_grouped(self, hidden_states):
        """(q, k, v) projections [bsz, tgt, embed] from one grouped call, or None when the three layers are not
        plain W8A8B8O8Linear of one shape on contiguous HIP tensors."""
        q, k, v = self.q_proj, self.k_proj, self.v_proj
        if not (type(q) is W8A8B8O8Linear and type(k) is W8A8B8O8Linear and type(v) is W8A8B8O8Linear):
            return None
        x = hidden_states.reshape(-1, hidden_states.shape[-1])
        (wq, bq), (wk, bk), (wv, bv) = q._wb(), k._wb(), v._wb()
        weights, biases = (wq, wk, wv), (bq.reshape(-1), bk.reshape(-1), bv.reshape(-1))
        if not _hip_ext.can_linear_group(x, weights, biases):
            return None
        outs = _hip_ext.linear_a8_w8_b8_o8_group(
            x, weights, biases, (q._scalar("a"), k._scalar("a"), v._scalar("a")),
            (q._scalar("b"), k._scalar("b"), v._scalar("b")), checked=True)
        lead = hidden_states.shape[:-1]
        return tuple(o.view(*lead, -1) for o in outs)

    def _qkv_head_major(self, hidden_states, bsz, tgt_len):
        """(q, k, v), each int8 [bsz, heads, tgt, head_dim] written in that layout by the projection GEMMs
        themselves, or None when the layers or tensors do not qualify."""
        q, k, v = self.q_proj, self.k_proj, self.v_proj
        if not (type(q) is W8A8B8O8Linear and type(k) is W8A8B8O8Linear and type(v) is W8A8B8O8Linear):
            return None
        x = hidden_states.reshape(-1, hidden_states.shape[-1])
        H, d = self.num_heads, self.head_dim
        wb = [lin._wb() for lin in (q, k, v)]
        weights, biases = [w for w, _ in wb], [b.reshape(-1) for _, b in wb]
        if not all(_hip_ext.can_linear_heads(x, w, b, bsz, tgt_len, H, d) for w, b in zip(weights, biases)):
            return None
        if (_hip_ext.can_linear_group(x, weights, biases)
                and _hip_ext.linear_group_is_one_launch(x.shape[0], weights[0].shape[0], x.shape[1], len(weights))):
            # one call; widths the 16x16-block tiles divide run as a single persistent launch
            return _hip_ext.linear_a8_w8_b8_o8_group_heads(
                x, weights, biases, [lin._scalar("a") for lin in (q, k, v)], [lin._scalar("b") for lin in (q, k, v)],
                bsz, tgt_len, H, d, checked=True)
        return tuple(_hip_ext.linear_a8_w8_b8_o8_heads(x, w, b, lin._scalar("a"), lin._scalar("b"), bsz, tgt_len, H, d,
                                                       checked=True)
                     for lin, w, b in zip((q, k, v), weights, biases))

    def _shape(self, tensor: torch.Tensor, seq_len: int, bsz: int):
        """[bsz, seq, embed] -> contiguous [bsz, heads, seq, head_dim]."""
        if seq_len < 0:
            seq_len = tensor.numel() // (bsz * self.embed_dim)
        return _hip_ext.split_heads(tensor, bsz, seq_len, self.num_heads, self.head_dim)

    @torch.no_grad()
    def _decode_fused(self, query4, key, value, past_key_value, attention_mask, output_attentions):
        """The whole attention of a decode step (cache append, Q.K^T, softmax-quant, P.V) as one kernel launch,
        or None when the shapes, the cache or the product modules do not allow it; same values as the separate
        steps of ``forward``."""
        past_k, past_v = past_key_value
        if not (type(self.qk_bmm) is BMM_S8T_S8N_F32T and type(self.pv_bmm) is BMM_S8T_S8N_S8T
                and past_k.dim() == 4 and past_v.shape == past_k.shape):
            return None
        bsz, H, T, d = query4.shape
        S0 = past_k.shape[2]
        if not _hip_ext.decode_attention_shape_ok(T, S0 + T, d):
            return None
        kk = _kv_room(past_k, key) or _kv_fresh(past_k, T)
        vv = _kv_room(past_v, value) or _kv_fresh(past_v, T)
        if not _hip_ext.can_decode_attention(query4, key, value, kk.buf, vv.buf, S0, attention_mask):
            return None   # (a buffer made above is simply dropped; the caller builds its own)
        ctx, probs = _hip_ext.decode_attention(query4, key, value, kk.buf, vv.buf, S0, attention_mask,
                                               self.qk_bmm._scalar("a"), self.pv_bmm._scalar("a"),
                                               want_probs=output_attentions, checked=True)
        kk.filled = vv.filled = S0 + T
        present = (_kv_view(kk, S0 + T), _kv_view(vv, S0 + T))
        probs_out = probs.view(bsz, H, T, S0 + T).float() if output_attentions else None
        ctx = _hip_ext.merge_heads(ctx, bsz, H, T, d)
        return self.out_proj(ctx), probs_out, present

    def decode_step_devlen(self, hidden_states, k_buf, v_buf, length, max_length):
        """Self-attention of one new token per sequence (int8 [bsz, 1, embed]) over cache buffers [bsz, heads, cap,
        head_dim] whose length after the append is read from the int32 HIP tensor ``length`` when the kernels run
        (``Int8OPTGraphDecoder`` records this once and replays it).  No mask, no head mask; the values of
        ``forward`` with a cache of ``length - 1`` positions.  Returns the fp32 output of ``out_proj``."""
        bsz, tgt_len, _ = hidden_states.shape
        flat = self._qkv_grouped(hidden_states)
        if flat is None or not (type(self.qk_bmm) is BMM_S8T_S8N_F32T and type(self.pv_bmm) is BMM_S8T_S8N_S8T):
            raise RuntimeError("Int8OPTAttention.decode_step_devlen: needs the stock int8 projections and products "
                               "on contiguous HIP tensors")
        query4, key, value = (self._shape(t, tgt_len, bsz) for t in flat)
        ctx = _hip_ext.decode_attention_devlen(query4, key, value, k_buf, v_buf, length, max_length,
                                               self.qk_bmm._scalar("a"), self.pv_bmm._scalar("a"))
        ctx = _hip_ext.merge_heads(ctx, bsz, self.num_heads, tgt_len, self.head_dim)
        return self.out_proj(ctx)

    def forward(self, hidden_states: torch.Tensor, key_value_states: Optional[torch.Tensor] = None,
                past_key_value: Optional[Tuple[torch.Tensor]] = None,
                attention_mask: Optional[torch.Tensor] = None,
                layer_head_mask: Optional[torch.Tensor] = None, output_attentions: bool = False,
                ) -> Tuple[torch.Tensor, Optional[torch.Tensor], Optional[Tuple[torch.Tensor]]]:
        """hidden_states: int8 [batch, time, channel] -> (fp32 output, probs or None, (k, v) int8 cache)."""
        cross = key_value_states is not None
        bsz, tgt_len, _ = hidden_states.size()
        H, d = self.num_heads, self.head_dim
        if attention_mask is not None and attention_mask.is_cuda and attention_mask.dtype in (torch.float16, torch.bfloat16):
            # the mask of an fp16 model: it is only ever added to the fp32 scores, where type promotion turns it into
            # these same fp32 values; the fused kernels read fp32
            attention_mask = attention_mask.float()

        # Self-attention on HIP tensors takes the q/k/v projections from one of two fused forms: a single
        # grouped launch for decode-sized inputs, or projections whose stores already produce the
        # [bsz, heads, seq, head_dim] layout; both give the values of the plain layers.
        proj = None  # (q, k, v), each [bsz, H, tgt, d]
        if not cross and hidden_states.is_cuda:
            if bsz * tgt_len <= 16:
                flat = self._qkv_grouped(hidden_states)
                if flat is not None:
                    proj = tuple(self._shape(t, tgt_len, bsz) for t in flat)
            else:
                proj = self._qkv_head_major(hidden_states, bsz, tgt_len)
        if proj is not None:
            query4, key, value = proj
        else:
            query4 = self._shape(self.q_proj(hidden_states), tgt_len, bsz)
        if cross and past_key_value is not None:
            key, value = past_key_value
        else:
            if proj is None:
                kv_src = key_value_states if cross else hidden_states
                key = self._shape(self.k_proj(kv_src), -1, bsz)
                value = self._shape(self.v_proj(kv_src), -1, bsz)
            if not cross and past_key_value is not None:
                if (self.kv_cache_in_place and self.fused_softmax and proj is not None and tgt_len <= 4
                        and layer_head_mask is None):
                    fused = self._decode_fused(query4, key, value, past_key_value, attention_mask, output_attentions)
                    if fused is not None:
                        return fused
                if self.kv_cache_in_place:
                    key, value = _kv_append_pair(past_key_value[0], past_key_value[1], key, value)
                else:
                    key = torch.cat([past_key_value[0], key], dim=2)
                    value = torch.cat([past_key_value[1], value], dim=2)
        present = (key, value)

        query = query4.view(bsz * H, -1, d)
        # cache views are packed per head; [bsz, H] merges into one batch dimension either way
        key = key.view(bsz * H, -1, d) if key.is_contiguous() else key.reshape(bsz * H, key.shape[2], d)
        value = value.view(bsz * H, -1, d) if value.is_contiguous() else value.reshape(bsz * H, value.shape[2], d)
        src_len = key.size(1)

        # Beyond 576 keys the fused kernels are taken for a plain prefill (tgt_len == src_len) only: the line was drawn where they
        # swept the keys three times and won through the key tiles that a causal mask kills (160 x 2048 x 2048: 0.99 ms against
        # 1.34 ms for the separate kernels).  With a row's scores in registers, up to 2048 keys, they no longer do; a prompt
        # continued over a longer cache has not been measured against them.
        long_ok = src_len <= 576 or tgt_len == src_len
        if (self.fused_softmax and long_ok and layer_head_mask is None and not output_attentions and tgt_len > 16
                and type(self.qk_bmm) is BMM_S8T_S8N_F32T and type(self.pv_bmm) is BMM_S8T_S8N_S8T
                and _hip_ext.can_attn_qk_softmax_q(query, key, attention_mask, bsz, H) and value.is_cuda
                and _hip_ext.attn_prefill_shape_ok(tgt_len, src_len, d)):
            # the whole attention (Q.K^T, softmax-quant, P.V, head merge) in one kernel on V transposed
            vt = _hip_ext.transpose_last2(value.contiguous())
            if _hip_ext.can_attn_prefill(query, key, vt, attention_mask, bsz, H):
                ctx = _hip_ext.attn_prefill(query, key, vt, attention_mask, self.qk_bmm._scalar("a"),
                                            self.pv_bmm._scalar("a"), H, checked=True)
                return self.out_proj(ctx), None, present
        probs_q = None
        if (self.fused_softmax and long_ok and layer_head_mask is None and tgt_len > 16
                and type(self.qk_bmm) is BMM_S8T_S8N_F32T and _hip_ext.can_attn_qk_softmax_q(query, key, attention_mask, bsz, H)):
            # Q.K^T, mask, clamp, softmax, *127, round and int8 cast in one kernel: the fp32 scores stay in registers
            probs_q = _hip_ext.attn_qk_softmax_q(query, key, attention_mask, self.qk_bmm._scalar("a"), H, checked=True)
            probs_out = probs_q.view(bsz, H, tgt_len, src_len).float() if output_attentions else None
        elif (not key.is_contiguous() and type(self.qk_bmm) is BMM_S8T_S8N_F32T
                and _hip_ext.can_bmm_strided(query, key)):
            scores = _hip_ext.bmm_s8t_s8n_f32t_strided(query, key, self.qk_bmm._scalar("a"), checked=True)
        else:
            scores = self.qk_bmm(query, key.contiguous())  # fp32 [bsz*H, tgt, src]
        if probs_q is None and scores.size() != (bsz * H, tgt_len, src_len):
            raise ValueError(f"Attention weights should be of size {(bsz * H, tgt_len, src_len)}, but is"
                             f" {scores.size()}")
        if attention_mask is not None and attention_mask.size() != (bsz, 1, tgt_len, src_len):
            raise ValueError(f"Attention mask should be of size {(bsz, 1, tgt_len, src_len)}, but is"
                             f" {attention_mask.size()}")
        if layer_head_mask is not None and layer_head_mask.size() != (H,):
            raise ValueError(f"Head mask for a single layer should be of size {(H,)}, but is"
                             f" {layer_head_mask.size()}")
        if probs_q is not None:
            pass
        elif self.fused_softmax and layer_head_mask is None and _hip_ext.can_fuse_softmax(scores, attention_mask, bsz, H):
            # mask add, clamp, softmax, *127, round and int8 cast in one kernel
            probs_q = _hip_ext.attn_softmax_q(scores, attention_mask, H, checked=True)
            probs_out = probs_q.view(bsz, H, tgt_len, src_len).float() if output_attentions else None
        else:
            if attention_mask is not None:
                scores = scores.view(bsz, H, tgt_len, src_len) + attention_mask
                scores = torch.clamp_min(scores, torch.finfo(scores.dtype).min)
                scores = scores.view(bsz * H, tgt_len, src_len)
            probs = nn.functional.softmax(scores, dim=-1)
            if layer_head_mask is not None:
                probs = (layer_head_mask.view(1, -1, 1, 1) * probs.view(bsz, H, tgt_len, src_len)
                         ).view(bsz * H, tgt_len, src_len)
            probs_out = probs.view(bsz, H, tgt_len, src_len) if output_attentions else None
            # The probabilities are scaled and rounded in place, so with output_attentions the
            # returned view holds round(127 p), which is what upstream returns too
            # (models/opt.py:166-178).
            probs_q = probs.mul_(127).round_().to(torch.int8)
        if tgt_len <= 16 and type(self.pv_bmm) is BMM_S8T_S8N_S8T and _hip_ext.can_bmm_rowmajor(probs_q, value):
            # few query rows (incremental decoding): stream V once, as the cache stores it
            ctx = _hip_ext.bmm_s8t_s8t_s8t(probs_q, value, self.pv_bmm._scalar("a"), checked=True)
        else:
            # P.V with V transposed to [bsz*H, d, src]: (P V) = P . (V^T)^T
            ctx = self.pv_bmm(probs_q, _hip_ext.transpose_last2(value.contiguous()))  # int8 [bsz*H, tgt, d]
        if ctx.size() != (bsz * H, tgt_len, d):
            raise ValueError(f"`attn_output` should be of size {(bsz, H, tgt_len, d)}, but is {ctx.size()}")
        ctx = _hip_ext.merge_heads(ctx, bsz, H, tgt_len, d)
        return self.out_proj(ctx), probs_out, present


class _DecodePlan:
    """``Int8OPTDecoderLayer`` flattened into the structure ``ti_opt_decoder_layer_decode`` reads, plus what it was
    built from: (dict that holds the tensor, its name, the tensor, its version) for every buffer and (dict, name, module)
    for every sub-module, so that a replaced or rewritten buffer and a replaced module are noticed."""
    __slots__ = ("ok", "half", "device", "struct", "addr", "sources", "modules", "embed", "heads", "head_dim", "ffn")

    def __reduce__(self):   # a copied or pickled layer makes a plan of its own tensors
        return _no_plan, ()

    def new_cache(self, hidden):
        """Empty key and value tensors [bsz, heads, tokens, head_dim] for a prefill of ``hidden``."""
        shape = (hidden.shape[0], self.heads, hidden.shape[1], self.head_dim)
        return (torch.empty(shape, dtype=torch.int8, device=self.device), torch.empty(shape, dtype=torch.int8, device=self.device))

    @staticmethod
    def build(layer, half, device):
        plan = _DecodePlan()
        plan.ok, plan.half, plan.device = False, half, device
        sources = []
        at = layer.self_attn
        plan.modules = tuple((holder._modules, name, getattr(holder, name)) for holder, names in (
            (layer, ("self_attn", "fc1", "fc2", "self_attn_layer_norm", "final_layer_norm")),
            (at, ("q_proj", "k_proj", "v_proj", "out_proj", "qk_bmm", "pv_bmm"))) for name in names)
        stock = (type(at.q_proj) is W8A8B8O8Linear and type(at.k_proj) is W8A8B8O8Linear
                 and type(at.v_proj) is W8A8B8O8Linear and type(at.out_proj) is W8A8BFP32OFP32Linear
                 and type(layer.fc1) is W8A8B8O8LinearReLU and type(layer.fc2) is W8A8BFP32OFP32Linear
                 and type(at.qk_bmm) is BMM_S8T_S8N_F32T and type(at.pv_bmm) is BMM_S8T_S8N_S8T
                 and type(layer.self_attn_layer_norm) is LayerNormQ and type(layer.final_layer_norm) is LayerNormQ)
        plan.sources = ()
        if not stock:
            return plan
        E, H, d, F = at.embed_dim, at.num_heads, at.head_dim, layer.fc1.out_features
        fdt = torch.float16 if half else torch.float32

        def tensor(mod, name, dtype, numel):
            holder = mod._buffers if mod._buffers.get(name) is not None else mod._parameters
            t = holder.get(name)
            if not (isinstance(t, torch.Tensor) and t.device == device and t.dtype is dtype and t.is_contiguous()
                    and t.numel() == numel and t.data_ptr() % 16 == 0):
                raise _NotStock
            sources.append((holder, name, t, t._version))
            return t.data_ptr()

        def scalar(mod, name):
            value = mod._scalar(name)
            t = mod._buffers.get(name)
            if isinstance(t, torch.Tensor):
                sources.append((mod._buffers, name, t, t._version))
            else:
                raise _NotStock   # a scale that is not a registered buffer cannot be watched
            return value

        try:
            qkv1 = (at.q_proj, at.k_proj, at.v_proj, layer.fc1)
            read_scalars([(m, "a") for m in qkv1 + (at.qk_bmm, at.pv_bmm, at.out_proj, layer.fc2)] + [(m, "b") for m in qkv1])
            for lin in (at.out_proj, layer.fc2):   # their fp32 bias may still be in the dtype a cast left (see _run)
                _, bias = lin._wb()
                if bias.dtype is not torch.float32:
                    lin.bias = bias.to(torch.float32)
            st = _hip_ext.OptDecodeLayer()
            st.embed, st.heads, st.head_dim, st.ffn, st.half = E, H, d, F, int(half)
            ln1, ln2 = layer.self_attn_layer_norm, layer.final_layer_norm
            st.ln1_eps, st.ln2_eps = float(ln1.eps), float(ln2.eps)
            st.ln1_gamma, st.ln1_beta = tensor(ln1, "weight", fdt, E), tensor(ln1, "bias", fdt, E)
            st.ln2_gamma, st.ln2_beta = tensor(ln2, "weight", fdt, E), tensor(ln2, "bias", fdt, E)
            st.wq, st.wk, st.wv = (tensor(m, "weight", torch.int8, E * E) for m in (at.q_proj, at.k_proj, at.v_proj))
            st.bq, st.bk, st.bv = (tensor(m, "bias", torch.int8, E) for m in (at.q_proj, at.k_proj, at.v_proj))
            st.alpha_q, st.alpha_k, st.alpha_v = (scalar(m, "a") for m in (at.q_proj, at.k_proj, at.v_proj))
            st.beta_q, st.beta_k, st.beta_v = (scalar(m, "b") for m in (at.q_proj, at.k_proj, at.v_proj))
            st.alpha_qk, st.alpha_pv = scalar(at.qk_bmm, "a"), scalar(at.pv_bmm, "a")
            st.wo, st.bo = tensor(at.out_proj, "weight", torch.int8, E * E), tensor(at.out_proj, "bias", torch.float32, E)
            st.alpha_o = scalar(at.out_proj, "a")
            st.w1, st.b1 = tensor(layer.fc1, "weight", torch.int8, F * E), tensor(layer.fc1, "bias", torch.int8, F)
            st.alpha_1, st.beta_1 = scalar(layer.fc1, "a"), scalar(layer.fc1, "b")
            st.w2, st.b2 = tensor(layer.fc2, "weight", torch.int8, E * F), tensor(layer.fc2, "bias", torch.float32, E)
            st.alpha_2 = scalar(layer.fc2, "a")
        except _NotStock:
            return plan
        finally:
            plan.sources = tuple(sources)
        if H * d != E or at.q_proj.in_features != E or layer.fc2.in_features != F:
            return plan
        plan.struct, plan.addr = st, ctypes.addressof(st)
        plan.embed, plan.heads, plan.head_dim, plan.ffn = E, H, d, F
        plan.ok = True
        return plan


class _NotStock(Exception):
    pass


def _no_plan():
    return None


def _mask_as_fp32(mask):
    """The additive mask as the fused kernels read it: fp32 on the device (None when it is neither that nor an fp16 /
    bf16 HIP tensor).  The mask of an fp16 model is only ever added to fp32 scores (see ``Int8OPTAttention.forward``).
    A copy is this call's own, on its stream and of the values there are now; a decoder makes one for all of its layers
    (``Int8OPTDecoder._layer_mask``)."""
    if not mask.is_cuda:
        return None
    if mask.dtype is torch.float32:
        return mask
    return mask.float() if mask.dtype is torch.float16 or mask.dtype is torch.bfloat16 else None


_GLOBAL_FORWARD_HOOKS = torch.nn.modules.module._global_forward_hooks
_GLOBAL_FORWARD_PRE_HOOKS = torch.nn.modules.module._global_forward_pre_hooks


class Int8OPTDecoderLayer(nn.Module):
    """Pre-LN OPT block on an fp residual stream: LayerNormQ -> int8 attention -> add ->
    LayerNormQ -> fc1 (ReLU, int8) -> fc2 (fp32) -> add.  The input tensor is updated in
    place, as upstream does (``torch_int/models/opt.py:202-299``)."""

    def __init__(self, embed_dim, num_attention_heads, ffn_dim):
        super().__init__()
        self.embed_dim = embed_dim
        self.self_attn = Int8OPTAttention(embed_dim=embed_dim, num_heads=num_attention_heads)
        self.self_attn_layer_norm = LayerNormQ(embed_dim)
        self.fc1 = W8A8B8O8LinearReLU(embed_dim, ffn_dim)
        self.fc2 = W8A8BFP32OFP32Linear(ffn_dim, embed_dim)
        self.final_layer_norm = LayerNormQ(embed_dim)

    @staticmethod
    def from_float(module, attn_input_scale: float, q_output_scale: float, k_output_scale: float,
                   v_output_scale: float, out_input_scale: float, fc1_input_scale: float,
                   fc2_input_scale: float):
        q = Int8OPTDecoderLayer(module.embed_dim, module.self_attn.num_heads, module.fc1.out_features)
        q.self_attn_layer_norm = LayerNormQ.from_float(module.self_attn_layer_norm, attn_input_scale)
        q.self_attn = Int8OPTAttention.from_float(module.self_attn, attn_input_scale, q_output_scale,
                                                  k_output_scale, v_output_scale, out_input_scale)
        q.final_layer_norm = LayerNormQ.from_float(module.final_layer_norm, fc1_input_scale)
        q.fc1 = W8A8B8O8LinearReLU.from_float(module.fc1, fc1_input_scale, fc2_input_scale)
        q.fc2 = W8A8BFP32OFP32Linear.from_float(module.fc2, fc2_input_scale)
        return q

    #: one new token per sequence with a KV cache: the layer's kernels are issued from one C call
    #: (``ti_opt_decoder_layer_decode``: the same entry points with the same arguments, so the same values) instead of
    #: one Python call per module; set to False to go through the modules
    decode_in_one_call = True

    def _decode_plan(self, half, device):
        """The layer as ``ti_opt_decoder_layer_decode`` reads it, built once and rebuilt when a tensor it was built from
        has been replaced or written to; None when the layer is not the stock int8 block on ``device``."""
        plan = self.__dict__.get("_ti_decode_plan")
        if plan is None or plan.half != half or plan.device != device or not _hip_ext.plan_current(plan.sources, plan.modules):
            if plan is not None and any(m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__
                                        for _, _, m in plan.modules):
                return None   # a hook on a sub-module, or a forward that replaces its own, wants to see that module's call
            plan = self.__dict__["_ti_decode_plan"] = _DecodePlan.build(self, half, device)
            if not _hip_ext.plan_current(plan.sources, plan.modules):
                return None
        return plan if plan.ok and not _GLOBAL_FORWARD_HOOKS and not _GLOBAL_FORWARD_PRE_HOOKS else None

    def _decode_checks(self, hs, mask, past_key_value):
        """(plan, positions after this step) when one new token per sequence over this KV cache can be issued from one C
        call, else None.  ``mask`` fp32 on the device or None."""
        past_k, past_v = past_key_value
        shape = past_k.shape
        if not (len(shape) == 4 and past_v.shape == shape and past_k.dtype is torch.int8 and past_v.dtype is torch.int8
                and past_k.device == hs.device and past_v.device == hs.device):
            return None
        plan = self._decode_plan(hs.dtype is torch.float16, hs.device)
        bsz, S = hs.shape[0], shape[2] + 1
        if (plan is None or shape[0] != bsz or shape[1] != plan.heads or shape[3] != plan.head_dim or hs.shape[2] != plan.embed
                or not _hip_ext.decode_attention_shape_ok_cached(1, S, plan.head_dim)
                or (mask is not None and mask.shape != (bsz, 1, 1, S))):
            return None
        return plan, S

    @staticmethod
    def _one_call_tensors(hs, attention_mask):
        """(whether the residual stream and the mask qualify for the C calls, the mask as they read it)."""
        for cls, forward in _STOCK_FORWARDS:
            if cls.forward is not forward:   # replaced for all modules of that class
                return False, None
        if not (hs.is_cuda and hs.is_contiguous() and (hs.dtype is torch.float32 or hs.dtype is torch.float16)):
            return False, None
        if attention_mask is None:
            return True, None
        mask = _mask_as_fp32(attention_mask)
        return (mask is not None and mask.is_contiguous() and mask.device == hs.device and mask.data_ptr() % 16 == 0), mask

    def _decode_in_one_call(self, hidden_states, attention_mask, past_key_value, use_cache):
        """``forward`` for one new token per sequence over a KV cache, or None when the tensors do not qualify."""
        ok, mask = self._one_call_tensors(hidden_states, attention_mask)
        if not ok or hidden_states.shape[0] > 64:
            return None
        found = self._decode_checks(hidden_states, mask, past_key_value)
        rooms = found and _kv_rooms(past_key_value)
        if not rooms:
            return None
        plan, S = found
        present = _kv_append_in_layer(plan, hidden_states, mask, rooms, past_key_value, S)
        if use_cache:
            return hidden_states, present
        return (hidden_states,)

    #: a prefill (more than 16 tokens per sequence, a multiple of 16) likewise: up to 4096 tokens a layer's kernels take less
    #: time than eight trips through Python (``ti_opt_decoder_layer_prefill``); as part of a model, any number of tokens
    prefill_in_one_call = True

    def _prefill_checks(self, hs, mask):
        """The plan when a prefill without a cache can be issued from one C call, else None."""
        bsz, T = hs.shape[0], hs.shape[1]
        if T % 16 or bsz == 0 or bsz > 65535 or bsz * T > 1 << 20 or (mask is not None and mask.shape != (bsz, 1, T, T)):
            return None
        plan = self._decode_plan(hs.dtype is torch.float16, hs.device)
        # up to 65535 matrices, what one transpose of all values takes, which more than 2048 keys need (beyond, ``_hip_ext.transpose_last2``
        # leaves them to torch)
        if (plan is None or hs.shape[2] != plan.embed or bsz * plan.heads > 65535
                or not _hip_ext.attn_prefill_shape_ok_cached(T, T, plan.head_dim)):
            return None
        return plan

    def _prefill_in_one_call(self, hidden_states, attention_mask, use_cache):
        """``forward`` without a cache on T > 16 tokens per sequence, or None when the tensors do not qualify."""
        ok, mask = self._one_call_tensors(hidden_states, attention_mask)
        plan = self._prefill_checks(hidden_states, mask) if ok and hidden_states.shape[0] * hidden_states.shape[1] <= 4096 else None
        if plan is None:
            return None
        key, value = plan.new_cache(hidden_states)
        _hip_ext.opt_layer_prefill(plan, hidden_states, mask, key, value,
                                   classes=_hip_ext.prefill_mask_classes(hidden_states, mask, plan.heads, plan.head_dim))
        if use_cache:
            return hidden_states, (key, value)
        return (hidden_states,)

    def decode_step_devlen(self, hidden_states, k_buf, v_buf, length, max_length):
        """``forward`` for one new token per sequence with the cache length read on the device (see
        ``Int8OPTAttention.decode_step_devlen``): updates ``hidden_states`` in place and appends to the cache."""
        residual = hidden_states
        x = self.self_attn_layer_norm(hidden_states)
        x = self.self_attn.decode_step_devlen(x, k_buf, v_buf, length, max_length)
        x = self.final_layer_norm(residual, add=x)
        x = self.fc1(x)
        if type(self.fc2) is W8A8BFP32OFP32Linear:
            self.fc2(x, add_to=residual)
        else:
            residual.add_(self.fc2(x).to(residual.dtype))
        return residual

    def forward(self, hidden_states: torch.Tensor, attention_mask: Optional[torch.Tensor] = None,
                layer_head_mask: Optional[torch.Tensor] = None, output_attentions: Optional[bool] = False,
                use_cache: Optional[bool] = False, past_key_value: Optional[Tuple[torch.Tensor]] = None):
        """hidden_states: fp [batch, time, embed_dim] residual stream -> tuple starting with it."""
        if (past_key_value is not None and self.decode_in_one_call and hidden_states.dim() == 3
                and hidden_states.shape[1] == 1 and layer_head_mask is None and not output_attentions
                and self.self_attn.kv_cache_in_place and self.self_attn.fused_softmax):
            out = self._decode_in_one_call(hidden_states, attention_mask, past_key_value, use_cache)
            if out is not None:
                return out
        elif (past_key_value is None and self.prefill_in_one_call and hidden_states.dim() == 3
                and 16 < hidden_states.shape[1] and layer_head_mask is None and not output_attentions
                and self.self_attn.fused_softmax):
            out = self._prefill_in_one_call(hidden_states, attention_mask, use_cache)
            if out is not None:
                return out
        residual = hidden_states
        x = self.self_attn_layer_norm(hidden_states)
        x, attn_weights, present = self.self_attn(
            hidden_states=x, past_key_value=past_key_value, attention_mask=attention_mask,
            layer_head_mask=layer_head_mask, output_attentions=output_attentions)
        x = self.final_layer_norm(residual, add=x)  # residual += x, then LayerNormQ
        x = self.fc1(x)
        if type(self.fc2) is W8A8BFP32OFP32Linear:
            self.fc2(x, add_to=residual)  # residual += fc2(x), added in the GEMM epilogue when residual is fp32
        else:
            residual.add_(self.fc2(x).to(residual.dtype))
        outputs = (residual,)
        if output_attentions:
            outputs += (attn_weights,)
        if use_cache:
            outputs += (present,)
        return outputs


#: the calls that a layer's one C call stands for, as their classes define them; the chain stands for the layer's own too
_STOCK_FORWARDS = tuple((cls, cls.forward) for cls in (
    Int8OPTAttention, LayerNormQ, W8A8B8O8Linear, W8A8B8O8LinearReLU, W8A8BFP32OFP32Linear, BMM_S8T_S8N_F32T,
    BMM_S8T_S8N_S8T))
_STOCK_LAYER_FORWARD = Int8OPTDecoderLayer.forward


# --------------------------------------------------------------------------------------
# OPT scaffolding around the int8 blocks
# --------------------------------------------------------------------------------------

@dataclass
class OPTConfigLite:
    """The OPTConfig fields the int8 model reads, with OPT-125m defaults."""
    vocab_size: int = 50272
    hidden_size: int = 768
    num_hidden_layers: int = 12
    ffn_dim: int = 3072
    num_attention_heads: int = 12
    max_position_embeddings: int = 2048
    word_embed_proj_dim: Optional[int] = None
    pad_token_id: int = 1
    do_layer_norm_before: bool = True
    _remove_final_layer_norm: bool = False
    use_cache: bool = True

    def __post_init__(self):
        if self.word_embed_proj_dim is None:
            self.word_embed_proj_dim = self.hidden_size


@dataclass
class BaseModelOutputWithPast:
    last_hidden_state: torch.Tensor = None
    past_key_values: Optional[tuple] = None
    hidden_states: Optional[tuple] = None
    attentions: Optional[tuple] = None


@dataclass
class CausalLMOutputWithPast:
    loss: Optional[torch.Tensor] = None
    logits: torch.Tensor = None
    past_key_values: Optional[tuple] = None
    hidden_states: Optional[tuple] = None
    attentions: Optional[tuple] = None


class OPTLearnedPositionalEmbedding(nn.Embedding):
    """Learned absolute positions; OPT reserves the first two rows, so indices are offset by 2."""
    offset = 2

    def __init__(self, num_embeddings: int, embedding_dim: int):
        super().__init__(num_embeddings + self.offset, embedding_dim)

    def forward(self, attention_mask: torch.Tensor, past_key_values_length: int = 0):
        mask = attention_mask.long()
        positions = torch.cumsum(mask, dim=1) * mask - 1  # padded slots get -1
        return super().forward(positions[:, past_key_values_length:] + self.offset)


def _additive_decoder_mask(attention_mask, tgt_len, past_len, dtype, device):
    """[bsz, 1, tgt, past+tgt] mask: 0 where attention is allowed, finfo.min where the
    key is in the future or is padding (both conditions add up)."""
    bsz, src_len = attention_mask.shape
    neg = torch.finfo(dtype).min
    keep = attention_mask[:, None, None, :].to(dtype)
    pad = (1.0 - keep).masked_fill((1.0 - keep).bool(), neg).expand(bsz, 1, tgt_len, src_len)
    if tgt_len <= 1:
        return pad.contiguous()
    q_pos = torch.arange(past_len, past_len + tgt_len, device=device)[:, None]
    k_pos = torch.arange(src_len, device=device)[None, :]
    causal = torch.zeros((tgt_len, src_len), dtype=dtype, device=device).masked_fill(k_pos > q_pos, neg)
    return pad + causal[None, None]


def _causal_mask(bsz, tgt_len, dtype, device):
    """``_additive_decoder_mask`` of tokens that are all attended and have no past, as the layers read it: fp32 with the lowest
    value of ``dtype``."""
    return torch.full((bsz, 1, tgt_len, tgt_len), torch.finfo(dtype).min, dtype=torch.float32, device=device).triu_(1)


_STOCK_POSITIONS_FORWARD = OPTLearnedPositionalEmbedding.forward


class Int8OPTDecoder(nn.Module):
    """Stack of ``Int8OPTDecoderLayer`` with fp embeddings and final LayerNorm
    (upstream ``torch_int/models/opt.py:302-398``).  Without a KV cache the token dimension
    is padded to a multiple of 16 with <pad> (id 1, masked out) and the result sliced back,
    exactly as upstream; with a cache the new tokens are used as they are."""

    def __init__(self, config):
        super().__init__()
        self.config = config
        self.padding_idx = config.pad_token_id
        self.max_target_positions = config.max_position_embeddings
        self.vocab_size = config.vocab_size
        D, E = config.hidden_size, config.word_embed_proj_dim
        self.embed_tokens = nn.Embedding(config.vocab_size, E, self.padding_idx)
        self.embed_positions = OPTLearnedPositionalEmbedding(config.max_position_embeddings, D)
        self.project_out = nn.Linear(D, E, bias=False) if E != D else None
        self.project_in = nn.Linear(E, D, bias=False) if E != D else None
        if config.do_layer_norm_before and not getattr(config, "_remove_final_layer_norm", False):
            self.final_layer_norm = nn.LayerNorm(D)
        else:
            self.final_layer_norm = None
        self.layers = nn.ModuleList(
            [Int8OPTDecoderLayer(D, config.num_attention_heads, config.ffn_dim)
             for _ in range(config.num_hidden_layers)])

    def get_input_embeddings(self):
        return self.embed_tokens

    def set_input_embeddings(self, value):
        self.embed_tokens = value

    @staticmethod
    def from_float(module, decoder_layer_scales):
        q = Int8OPTDecoder(module.config)
        q.embed_tokens = module.embed_tokens
        q.embed_positions = module.embed_positions
        q.project_out = module.project_out
        q.project_in = getattr(module, "project_in", None)
        q.final_layer_norm = module.final_layer_norm
        for i, layer in enumerate(module.layers):
            q.layers[i] = Int8OPTDecoderLayer.from_float(layer, **decoder_layer_scales[i])
        return q

    def _chain_layers(self, hidden, attention_mask, past_key_values, use_cache):
        """The loop over the layers with one C call per layer and the last addition of a layer left to the next one's first
        kernel (``chain`` in ``_hip_ext.opt_layer_decode``): updates ``hidden`` in place and returns the cache, or None
        when a layer, its hooks or the tensors want the ordinary calls.  Values of the loop over ``layer(hidden, ...)``."""
        layers = list(self.layers)
        count, decode = len(layers), bool(past_key_values)
        if count == 0 or (hidden.shape[1] != 1 or hidden.shape[0] > 64 if decode else hidden.shape[1] <= 16):
            return None
        ok, mask = Int8OPTDecoderLayer._one_call_tensors(hidden, attention_mask)
        if not ok or Int8OPTDecoderLayer.forward is not _STOCK_LAYER_FORWARD or (decode and len(past_key_values) != count):
            return None
        chain = getattr(past_key_values[0][0], "_ti_chain", None) if decode else None
        if chain is not None and len(chain.rooms) == count:
            cache = self._continue_chain(layers, chain, hidden, mask, past_key_values)
            if cache is not None:
                return cache
        found = []
        for i, layer in enumerate(layers):
            if (type(layer) is not Int8OPTDecoderLayer or layer._forward_hooks or layer._forward_pre_hooks
                    or "forward" in layer.__dict__):
                return None
            attn = layer.self_attn
            if not (type(attn) is Int8OPTAttention and attn.fused_softmax and (attn.kv_cache_in_place or not decode)
                    and (layer.decode_in_one_call if decode else layer.prefill_in_one_call)):
                return None
            hit = layer._decode_checks(hidden, mask, past_key_values[i]) if decode else layer._prefill_checks(hidden, mask)
            if hit is None:
                return None
            found.append(hit)
        # The carry: fc2's output on its way from one layer to the next, and in a prefill out_proj's too; memory of this pass, so
        # that passes of other threads on the same stream do not meet in it.  A decode step on an fp32 stream has none (fc2's
        # GEMM adds its output itself).  On an fp16 stream of up to 4 or more than 64 rows nothing is left in it either: it is what
        # lets a prefill's layers do with the smaller scratch.
        carry = self._carry(hidden, count, decode)
        links = [0 if carry is None else (_hip_ext.CHAIN_ADD if i else 0) | (_hip_ext.CHAIN_LEAVE if i + 1 < count else 0)
                 for i in range(count)]
        cache = []
        if decode:
            rooms = [_kv_rooms(past) for past in past_key_values]
            if not all(rooms):
                _kv_give_back(kv for pair in rooms if pair for kv in pair)
                return None
            scratch = _hip_ext.opt_decode_scratch([plan for plan, _ in found], hidden)
            for (plan, S), room, past, chain in zip(found, rooms, past_key_values, links):
                present = _kv_append_in_layer(plan, hidden, mask, room, past, S, chain=chain, carry=carry, scratch=scratch)
                if use_cache:
                    cache.append(present)
            if use_cache:
                cache[0][0]._ti_chain = _KVChain.of(rooms)
        else:
            memory = _hip_ext.opt_prefill_scratch(found, hidden)
            widest = max(found, key=lambda plan: plan.heads)
            classes = _hip_ext.prefill_mask_classes(hidden, mask, widest.heads, widest.head_dim)
            for plan, chain in zip(found, links):
                key, value = plan.new_cache(hidden)
                _hip_ext.opt_layer_prefill(plan, hidden, mask, key, value, chain=chain, carry=carry, memory=memory, classes=classes)
                if use_cache:
                    cache.append((key, value))
        return tuple(cache)

    @staticmethod
    def _carry(hidden, count, decode):
        if count < 2 or (decode and hidden.dtype is torch.float32):
            return None
        return torch.empty((hidden.shape[0] * hidden.shape[1], hidden.shape[2]), dtype=torch.float32, device=hidden.device)

    def _continue_chain(self, layers, chain, hidden, mask, past_key_values):
        """``_chain_layers`` for a decode step whose cache is as the step before left it: the layers are looked at as there, their
        caches together, and one C call issues them all.  (The loop there is some 12 us of Python a layer, what four of its five launches cost
        the host, and a small model's step is bound by it.)"""
        bsz, heads, _, d = chain.shape
        S = past_key_values[0][0].shape[2] + 1
        half, device = hidden.dtype is torch.float16, hidden.device
        if (bsz != hidden.shape[0] or device != chain.device or not _hip_ext.decode_attention_shape_ok_cached(1, S, d)
                or (mask is not None and mask.shape != (bsz, 1, 1, S))):
            return None
        plans = []
        for layer in layers:
            own = layer.__dict__
            if (type(layer) is not Int8OPTDecoderLayer or own["_forward_hooks"] or own["_forward_pre_hooks"] or "forward" in own
                    or not layer.decode_in_one_call):
                return None
            attn = own["_modules"]["self_attn"]
            if type(attn) is not Int8OPTAttention or not attn.fused_softmax or not attn.kv_cache_in_place:
                return None
            plan = layer._decode_plan(half, device)
            if plan is None or plan.heads != heads or plan.head_dim != d or plan.embed != hidden.shape[2]:
                return None
            plans.append(plan)
        rooms = chain.claim(past_key_values, S)
        if rooms is None:
            return None
        _hip_ext.opt_layers_decode(plans, hidden, mask, chain.keys, chain.values, chain.cap, S)
        cache = tuple((_kv_view(kk, S), _kv_view(vv, S)) for kk, vv in rooms)
        cache[0][0]._ti_chain = chain
        return cache

    def _positions_in_order(self, past_len, count):
        """The position embeddings [1, count, width] of tokens past_len, past_len + 1, ..., as a view of the table, or None where
        the table's module is not the stock one or is shorter (its lookup then says so)."""
        m = self.embed_positions
        if (type(m) is not OPTLearnedPositionalEmbedding or m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__
                or OPTLearnedPositionalEmbedding.forward is not _STOCK_POSITIONS_FORWARD or m.max_norm is not None
                or _GLOBAL_FORWARD_HOOKS or _GLOBAL_FORWARD_PRE_HOOKS or past_len + count + m.offset > m.weight.shape[0]):
            return None
        return m.weight[past_len + m.offset:past_len + m.offset + count].unsqueeze(0)

    @staticmethod
    def _layer_mask(attention_mask, tgt_len, past_len, inputs_embeds):
        mask = _additive_decoder_mask(attention_mask, tgt_len, past_len, inputs_embeds.dtype, inputs_embeds.device)
        if mask.is_cuda and mask.dtype in (torch.float16, torch.bfloat16):
            mask = mask.float()  # once here instead of once per layer (see Int8OPTAttention.forward)
        return mask

    @torch.no_grad()
    def forward(self, input_ids: torch.LongTensor = None, attention_mask: Optional[torch.Tensor] = None,
                head_mask: Optional[torch.Tensor] = None,
                past_key_values: Optional[List[Tuple[torch.Tensor]]] = None,
                inputs_embeds: Optional[torch.Tensor] = None, use_cache: Optional[bool] = None,
                output_attentions: Optional[bool] = None, output_hidden_states: Optional[bool] = None,
                return_dict: Optional[bool] = None):
        use_cache = bool(use_cache) if use_cache is not None else False
        if inputs_embeds is None:
            input_ids = input_ids.view(-1, input_ids.shape[-1])
        input_len = (input_ids if input_ids is not None else inputs_embeds).shape[1]
        past_len = past_key_values[0][0].shape[2] if past_key_values else 0

        pad_len = (-input_len) % 16 if (past_len == 0 and inputs_embeds is None) else 0
        if pad_len:
            input_ids = nn.functional.pad(input_ids, (0, pad_len), value=1)
            if attention_mask is not None:
                attention_mask = nn.functional.pad(attention_mask, (0, pad_len), value=0)
        if inputs_embeds is None:
            inputs_embeds = self.embed_tokens(input_ids)
        bsz, tgt_len = inputs_embeds.shape[:2]
        # Without an attention mask every key up to a token is attended and positions follow the past: a slice of the
        # position table and, in a prefill, one triangle take the place of some fifteen kernels.
        pos = self._positions_in_order(past_len, tgt_len) if attention_mask is None and inputs_embeds.is_cuda else None
        in_order = pos is not None and inputs_embeds.dtype in (torch.float16, torch.bfloat16, torch.float32)
        if in_order and (tgt_len == 1 or past_len == 0):
            mask = None if tgt_len == 1 else _causal_mask(bsz, tgt_len, inputs_embeds.dtype, inputs_embeds.device)
        else:
            if attention_mask is None:
                attention_mask = torch.ones((bsz, past_len + tgt_len), dtype=torch.bool, device=inputs_embeds.device)
            pos = self.embed_positions(attention_mask, past_len)
            mask = self._layer_mask(attention_mask, tgt_len, past_len, inputs_embeds)
        if self.project_in is not None:
            inputs_embeds = self.project_in(inputs_embeds)
        hidden = inputs_embeds + pos  # a fresh tensor: the layers update it in place

        all_hidden = () if output_hidden_states else None
        all_attn = () if output_attentions else None
        cache = () if use_cache else None
        chained = None
        if head_mask is None and not output_attentions and not output_hidden_states:
            chained = self._chain_layers(hidden, mask, past_key_values, use_cache)
        if chained is not None:
            cache = chained if use_cache else None
        elif mask is None:   # layers called by themselves are handed the mask of zeros
            attention_mask = torch.ones((bsz, past_len + tgt_len), dtype=torch.bool, device=hidden.device)
            mask = self._layer_mask(attention_mask, tgt_len, past_len, inputs_embeds)
        for i, layer in enumerate(self.layers if chained is None else ()):
            if output_hidden_states:
                all_hidden += (hidden.clone(),)
            out = layer(hidden, attention_mask=mask,
                        layer_head_mask=head_mask[i] if head_mask is not None else None,
                        output_attentions=bool(output_attentions), use_cache=use_cache,
                        past_key_value=past_key_values[i] if past_key_values else None)
            hidden = out[0]
            if output_attentions:
                all_attn += (out[1],)
            if use_cache:
                cache += (out[-1],)
        if self.final_layer_norm is not None:
            hidden = self.final_layer_norm(hidden)
        if self.project_out is not None:
            hidden = self.project_out(hidden)
        if output_hidden_states:
            all_hidden += (hidden,)
        if pad_len:
            hidden = hidden[:, :input_len, :]
        return BaseModelOutputWithPast(last_hidden_state=hidden, past_key_values=cache,
                                       hidden_states=all_hidden, attentions=all_attn)


class Int8OPTModel(nn.Module):
    """upstream ``torch_int/models/opt.py:401-417``."""

    def __init__(self, config):
        super().__init__()
        self.config = config
        self.decoder = Int8OPTDecoder(config)

    def get_input_embeddings(self):
        return self.decoder.embed_tokens

    def set_input_embeddings(self, value):
        self.decoder.embed_tokens = value

    def get_decoder(self):
        return self.decoder

    @staticmethod
    def from_float(module, decoder_layer_scales):
        q = Int8OPTModel(module.config)
        q.decoder = Int8OPTDecoder.from_float(module.decoder, decoder_layer_scales)
        return q

    def forward(self, *args, **kwargs):
        return self.decoder(*args, **kwargs)


class Int8OPTForCausalLM(nn.Module):
    """Int8 decoder + fp ``lm_head`` (not quantised; upstream ``torch_int/models/opt.py:420-450``)."""
    _keys_to_ignore_on_load_missing = [r"lm_head.weight"]

    def __init__(self, config):
        super().__init__()
        self.config = config
        self.model = Int8OPTModel(config)
        self.lm_head = nn.Linear(config.word_embed_proj_dim, config.vocab_size, bias=False)
        # Upstream's post_init ties the output projection to the token embedding (OPTConfig.tie_word_embeddings
        # defaults to True), and exported checkpoints then carry no ``lm_head.weight``.
        if getattr(config, "tie_word_embeddings", True):
            self.lm_head.weight = self.model.decoder.embed_tokens.weight
        self._register_load_state_dict_pre_hook(self._fill_tied_lm_head)

    def _fill_tied_lm_head(self, state_dict, prefix, *unused):
        """A state dict without ``lm_head.weight`` (tied weights are stored once) loads the embedding there."""
        head, emb = prefix + "lm_head.weight", prefix + "model.decoder.embed_tokens.weight"
        if head not in state_dict and emb in state_dict and self.lm_head.weight.shape == state_dict[emb].shape:
            state_dict[head] = state_dict[emb]

    @staticmethod
    def from_float(module, decoder_layer_scales):
        q = Int8OPTForCausalLM(module.config)
        q.model = Int8OPTModel.from_float(module.model, decoder_layer_scales)
        q.lm_head = module.lm_head
        return q

    def get_input_embeddings(self):
        return self.model.decoder.embed_tokens

    def set_input_embeddings(self, value):
        self.model.decoder.embed_tokens = value

    def get_output_embeddings(self):
        return self.lm_head

    def set_output_embeddings(self, new_embeddings):
        self.lm_head = new_embeddings

    def set_decoder(self, decoder):
        self.model.decoder = decoder

    def get_decoder(self):
        return self.model.decoder

    @torch.no_grad()
    def forward(self, input_ids: torch.LongTensor = None, attention_mask: Optional[torch.Tensor] = None,
                head_mask: Optional[torch.Tensor] = None, past_key_values=None,
                inputs_embeds: Optional[torch.Tensor] = None, labels: Optional[torch.LongTensor] = None,
                use_cache: Optional[bool] = None, output_attentions: Optional[bool] = None,
                output_hidden_states: Optional[bool] = None, return_dict: Optional[bool] = None):
        out = self.model.decoder(input_ids=input_ids, attention_mask=attention_mask, head_mask=head_mask,
                                 past_key_values=past_key_values, inputs_embeds=inputs_embeds,
                                 use_cache=use_cache, output_attentions=output_attentions,
                                 output_hidden_states=output_hidden_states)
        logits = self.lm_head(out.last_hidden_state.to(self.lm_head.weight.dtype)).contiguous()
        loss = None
        if labels is not None:
            shift = logits[..., :-1, :].contiguous()
            loss = nn.functional.cross_entropy(shift.view(-1, shift.size(-1)),
                                               labels[..., 1:].contiguous().view(-1).to(logits.device))
        return CausalLMOutputWithPast(loss=loss, logits=logits, past_key_values=out.past_key_values,
                                      hidden_states=out.hidden_states, attentions=out.attentions)

    def prepare_inputs_for_generation(self, input_ids, past_key_values=None, attention_mask=None, **kwargs):
        if past_key_values:
            input_ids = input_ids[:, -1:]
        return {"input_ids": input_ids, "attention_mask": attention_mask,
                "past_key_values": past_key_values, "use_cache": kwargs.get("use_cache")}

    @staticmethod
    def _reorder_cache(past, beam_idx):
        return tuple(tuple(s.index_select(0, beam_idx) for s in layer) for layer in past)


class Int8OPTGraphDecoder:
    """Token-by-token decoding of an ``Int8OPTForCausalLM`` on HIP with the decoder layers of a step replayed from
    one HIP graph (no counterpart upstream, whose ``generate`` re-issues every launch from Python).

    A decode step of a small or medium model is bound by the host: seven launches per layer and the Python around
    them.  Here the layers are recorded once, on fixed buffers: the residual stream of the new token, the key /
    value caches (buffers with room for ``max_new_tokens`` more positions) and an int32 tensor holding the cache
    length, which the attention kernel reads when it runs, so the same recording serves every step.  Embeddings,
    the final LayerNorm and ``lm_head`` stay ordinary torch calls around the replay.  No padding inside the batch
    (every sequence has the same length) and no head mask.  Values are those of ``lm(ids, past_key_values=...)``.

        out = lm(prompt_ids, use_cache=True)
        dec = Int8OPTGraphDecoder(lm, out.past_key_values, max_new_tokens=128)
        tok = out.logits[:, -1].argmax(-1, keepdim=True)
        for _ in range(128):
            tok = dec.step(tok)[:, -1].argmax(-1, keepdim=True)
    """

    @torch.no_grad()
    def __init__(self, lm, past_key_values, max_new_tokens):
        dec = lm.model.decoder
        k0 = past_key_values[0][0]
        if not (k0.is_cuda and k0.dtype is torch.int8 and k0.dim() == 4 and len(past_key_values) == len(dec.layers)):
            raise RuntimeError("Int8OPTGraphDecoder: needs the int8 HIP key/value caches of every decoder layer")
        bsz, H, S0, d = k0.shape
        self.lm, self.filled, self.max_length = lm, S0, S0 + int(max_new_tokens)
        if max_new_tokens < 1 or self.max_length > dec.max_target_positions:
            raise RuntimeError(f"Int8OPTGraphDecoder: {S0} cached + {max_new_tokens} new positions exceed the model's "
                               f"{dec.max_target_positions}")
        if not _hip_ext.decode_attention_shape_ok(1, self.max_length, d):
            raise RuntimeError(f"Int8OPTGraphDecoder: the decode attention kernel does not take {self.max_length} "
                               f"positions of head size {d}")
        cap = -(-self.max_length // 16) * 16
        self.caches = []
        for k, v in past_key_values:
            kb = torch.empty((bsz, H, cap, d), dtype=torch.int8, device=k0.device)
            vb = torch.empty_like(kb)
            kb[:, :, :S0].copy_(k)
            vb[:, :, :S0].copy_(v)
            self.caches.append((kb, vb))
        stream_dtype = dec.embed_positions.weight.dtype
        self.hidden = torch.zeros((bsz, 1, dec.embed_positions.weight.shape[1]), dtype=stream_dtype, device=k0.device)
        self.length = torch.full((1,), S0 + 1, dtype=torch.int32, device=k0.device)
        self._ones = torch.ones((bsz, self.max_length), dtype=torch.bool, device=k0.device)

        def layers():
            for layer, (kb, vb) in zip(dec.layers, self.caches):
                layer.decode_step_devlen(self.hidden, kb, vb, self.length, self.max_length)
        # one eager pass first: scalar caches, kernel attributes and the allocator's pools are then warm, and nothing
        # in the recording synchronises.  It writes position S0 of the caches, which the first real step overwrites.
        side = torch.cuda.Stream(device=k0.device)
        side.wait_stream(torch.cuda.current_stream(k0.device))
        with torch.cuda.stream(side):
            layers()
        torch.cuda.current_stream(k0.device).wait_stream(side)
        # recorded on the stream of the eager pass: the library's per-stream state (split-K workspace and arrival
        # counters, placement probe) is then ready, and nothing in the recording has to fall back or synchronise
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph, stream=side):
            layers()

    @torch.no_grad()
    def step(self, input_ids):
        """Logits [bsz, 1, vocab] for one new token per sequence (``input_ids`` [bsz, 1]); the caches grow by one."""
        if self.filled >= self.max_length:
            raise RuntimeError("Int8OPTGraphDecoder: max_new_tokens steps have been taken")
        dec = self.lm.model.decoder
        embeds = dec.embed_tokens(input_ids)
        pos = dec.embed_positions(self._ones[:, :self.filled + 1], self.filled)
        if dec.project_in is not None:
            embeds = dec.project_in(embeds)
        self.hidden.copy_(embeds + pos)
        self.length.fill_(self.filled + 1)
        self.graph.replay()
        self.filled += 1
        hidden = self.hidden
        if dec.final_layer_norm is not None:
            hidden = dec.final_layer_norm(hidden)
        if dec.project_out is not None:
            hidden = dec.project_out(hidden)
        return self.lm.lm_head(hidden.to(self.lm.lm_head.weight.dtype)).contiguous()

    @property
    def past_key_values(self):
        """The caches as ``forward`` would return them: per layer (key, value) int8 [bsz, heads, filled, head_dim]."""
        return tuple((kb[:, :, :self.filled], vb[:, :, :self.filled]) for kb, vb in self.caches)

