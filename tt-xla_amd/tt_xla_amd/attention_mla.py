"""vLLM attention backend for multi-head latent attention (MLA) on MI355X.

Mirrors the interface of tt-xla's
``integrations/vllm_plugin/vllm_tt/attention_impls/attention_mla.py``: backend name and
static methods (:67-110), the constructor's arguments and refusals (:118-165), ``forward``'s
signature, its prefill / decode dispatch and its output contract (:184-422).  The latent
cache is ONE tensor ``[num_blocks, 1, block_size, kv_lora_rank + qk_rope_head_dim]`` per layer
(K and V share it: V is the leading ``kv_lora_rank`` features of K).

What a forward pass does, in the order of the reference:
  1. absorb ``W_UK_T`` into the no-position part of the query (:230-244) and concatenate the
     rotary part: latent query ``[users, S, N, L + R]``; latent key of the new tokens
     ``[users, S, 1, L + R]`` from ``kv_c_normed`` and ``k_pe`` (:246-248);
  2. prefill (more than one token per user, :283-297): causal attention of the new tokens
     against themselves (``tt::flash_mla_prefill``), then the new latent keys go into the paged
     cache through the fill page table (:337-359);
     decode: the new token's latent key goes into the cache at ``cache_position`` first
     (:379-389), then ``tt::paged_flash_mla_decode`` attends over the paged cache (:394-405);
  3. expand the latent output with ``W_UV`` and write ``[tokens, N * v_head_dim]`` (:322-335,
     :408-422).
Differences from the reference, invisible in results: a causal prompt pass of more than 64 tokens at the
head shape 128 + 64 / 128 expands K and V per head instead of absorbing the query (``_expands_prompts``: the
same sums with the products grouped the other way; four prompts of 2048 tokens, 16 heads: 763 -> 164 us, and
the error against a 64-bit evaluation is 3.37e-3 of the output where the absorbed form's is 3.45e-3); a causal decode pass at that shape and a
latent width of 512 is one operator (``tt::latent_decode_step_``: the same steps and roundings without the
copies between them; 128 users, 16 heads: 168 -> 94 us); the cache writes use the in-place
operators (one batched fill instead of a per-user loop over functional fills followed by a
copy of the whole cache); ``functional_cache_ops=True`` restores the reference's call sequence.

The two latent attention operators sit on ``ttpa_paged_mla_decode``.
"""

from __future__ import annotations

from typing import List, Optional, Tuple

import torch

from . import _native
from . import custom_ops  # (registers torch.ops.tt.*)
from .attention import TTAttentionMetadataBuilder, TTMetadata

# the operator namespace, looked up once: host-logic tests substitute it
_ops = torch.ops.tt

try:  # pragma: no cover - vLLM is not part of the test image
    from vllm.v1.attention.backend import AttentionBackend as _BackendBase
    from vllm.v1.attention.backend import MLAAttentionImpl as _ImplBase
except Exception:  # vLLM absent: same surface, no base classes
    _BackendBase = object
    _ImplBase = object


class TTMLAAttentionBackend(_BackendBase):
    """Backend descriptor for the latent-attention layers (reference :67-110)."""

    @staticmethod
    def get_name() -> str:
        return "FLASH_ATTN_MLA"

    @staticmethod
    def get_impl_cls():
        return TTMLAAttentionBackendImpl

    @staticmethod
    def get_builder_cls():
        return TTAttentionMetadataBuilder  # the same stub builder as the non-latent backend

    @staticmethod
    def get_kv_cache_shape(num_blocks: int, block_size: int, num_kv_heads: int, head_size: int,
                           cache_dtype_str: str = "auto") -> Tuple[int, ...]:
        # one concatenated latent tensor per slot: head_size = kv_lora_rank + qk_rope_head_dim
        assert num_kv_heads == 1, "num_kv_heads must be 1 for MLA"
        return (num_blocks, num_kv_heads, block_size, head_size)

    @staticmethod
    def get_page_size(vllm_config) -> int:
        return 32

    @staticmethod
    def swap_blocks(src_kv_cache, dst_kv_cache, src_to_dst) -> None:
        raise RuntimeError("swap_blocks is not used for the TT MLA backend.")


class TTMLAAttentionBackendImpl(_ImplBase):
    def __init__(
        self,
        num_heads: int,
        head_size: int,
        scale: float,
        num_kv_heads: int,
        alibi_slopes: Optional[List[float]],
        sliding_window: Optional[int],
        kv_cache_dtype: str,
        logits_soft_cap: Optional[float],
        attn_type: str,
        kv_sharing_target_layer_name: Optional[str],
        q_lora_rank: Optional[int] = None,
        kv_lora_rank: int = 0,
        qk_nope_head_dim: int = 0,
        qk_rope_head_dim: int = 0,
        qk_head_dim: int = 0,
        v_head_dim: int = 0,
        kv_b_proj=None,
        indexer: Optional[object] = None,
        q_pad_num_heads: Optional[int] = None,
        functional_cache_ops: bool = False,
        **kwargs,
    ) -> None:
        self.num_heads = num_heads
        self.head_size = head_size
        self.scale = scale
        self.num_kv_heads = num_kv_heads
        self.kv_cache_dtype = kv_cache_dtype
        self.q_lora_rank = q_lora_rank
        self.kv_lora_rank = kv_lora_rank
        self.qk_nope_head_dim = qk_nope_head_dim
        self.qk_rope_head_dim = qk_rope_head_dim
        self.qk_head_dim = qk_head_dim
        self.v_head_dim = v_head_dim
        self.functional_cache_ops = functional_cache_ops
        if alibi_slopes is not None:
            raise NotImplementedError("Alibi slopes are not supported for MLA on TT.")
        if kv_cache_dtype != "auto":
            raise NotImplementedError(
                f"Quantized MLA KV cache ({kv_cache_dtype}) is not yet supported on TT."
            )

    # vLLM's generic MLA entry points are bypassed by the layer, which calls forward() directly
    def forward_mha(self, *args, **kwargs) -> None:
        raise RuntimeError(
            "TTMLAAttentionBackendImpl.forward_mha should never be called; the TT MLA layer "
            "routes through forward() directly."
        )

    def forward_mqa(self, *args, **kwargs):
        raise RuntimeError(
            "TTMLAAttentionBackendImpl.forward_mqa should never be called; the TT MLA layer "
            "routes through forward() directly."
        )

    # ------------------------------------------------------------------ forward
    def forward(
        self,
        q: Tuple[torch.Tensor, torch.Tensor],
        kv_c_normed: torch.Tensor,
        k_pe: torch.Tensor,
        kv_cache: torch.Tensor,
        attn_metadata: Optional[TTMetadata],
        layer,
        output: Optional[torch.Tensor] = None,
        **kwargs,
    ) -> None:
        """q = (q_nope [tokens, N, P], q_pe [tokens, N, R]); kv_c_normed [tokens, L];
        k_pe [tokens, 1, R]; kv_cache [num_blocks, 1, block_size, L + R]; the result is written
        into ``output`` [tokens, N * v_head_dim].  ``layer`` carries ``W_UK_T`` [N, P, L] and
        ``W_UV`` [N, L, V]."""
        assert output is not None, "TTMLAAttentionBackendImpl.forward requires an output tensor."
        if self._forward_native(q, kv_c_normed, k_pe, kv_cache, attn_metadata, layer, output):
            return
        q_nope, q_pe = q
        prefill = self._infer_is_prefill(q_nope, attn_metadata)
        users = 1
        if attn_metadata is not None and attn_metadata.cache_position is not None:
            users = attn_metadata.cache_position.shape[0]
        tokens = q_nope.shape[0]
        assert tokens % users == 0, f"total_tokens ({tokens}) not divisible by users ({users})."
        s = tokens // users
        n, lat, rope, nope = self.num_heads, self.kv_lora_rank, self.qk_rope_head_dim, self.qk_nope_head_dim

        if prefill and self._expands_prompts(q_nope, q_pe, kv_c_normed, k_pe, kv_cache, attn_metadata, layer, s, output):
            form = self._forward_prefill_short if s <= 64 else self._forward_prefill_expanded
            form(q_nope, q_pe, kv_c_normed, k_pe, kv_cache, attn_metadata, layer, s, users, output)
            return

        if not prefill and self._steps_at_once(q_nope, q_pe, kv_c_normed, k_pe, kv_cache, attn_metadata, layer, output):
            # projections, cache write and attention without the copies in between
            torch.ops.tt.latent_decode_step_(
                q_nope, q_pe, kv_c_normed.view(users, lat), k_pe.view(users, rope), layer.W_UK_T, layer.W_UV, kv_cache,
                attn_metadata.page_table, attn_metadata.cache_position, output.view(users, n, self.v_head_dim), float(self.scale))
            return

        act_dtype, device = q_pe.dtype, q_nope.device
        # W_UK_T is a plain attribute of the layer, not a parameter: it may still sit elsewhere
        w_uk_t = layer.W_UK_T.to(device=device)
        q_abs = torch.einsum("bsnp,npl->bsnl", q_nope.view(users, s, n, nope), w_uk_t).to(act_dtype)
        q_lat = torch.cat([q_abs, q_pe.view(users, s, n, rope)], dim=-1)             # [users, S, N, L+R]
        k_lat = torch.cat([kv_c_normed.view(users, s, 1, lat), k_pe.view(users, s, 1, rope)], dim=-1)

        if prefill:
            out = self._forward_prefill(q_lat, k_lat, kv_cache, attn_metadata, layer, s, users)
        else:
            out = self._forward_decode(q_lat, k_lat, kv_cache, attn_metadata, layer, users)
        output.copy_(out.to(act_dtype).reshape_as(output))

    def _forward_native(self, q, kv_c_normed, k_pe, kv_cache, attn_metadata, layer, output) -> bool:
        """The ordinary eager pass (causal, the head shape that the operators below are built for, with a cache) as one native
        call; False: not such a pass, nothing has been issued.  A prompt of 32 tokens took 100 us through views, batched
        products and operators, whatever the GPU did meanwhile."""
        if (
            attn_metadata is None
            or self.functional_cache_ops
            or (self.qk_nope_head_dim, self.qk_rope_head_dim, self.kv_lora_rank, self.v_head_dim) != (128, 64, 512, 128)
            or attn_metadata.attn_mask is not None
            or not attn_metadata.is_causal
            or torch.compiler.is_compiling()
        ):
            return False
        status = _native.latent_pass(
            q[0], q[1], kv_c_normed, k_pe, kv_cache, attn_metadata.page_table, attn_metadata.cache_position, attn_metadata.fill_page_table,
            layer.W_UK_T, layer.W_UV, output, self.num_heads, self.scale, custom_ops._workspace)
        if status is None:
            return False
        if status != 0:
            _native.check(*status)
        return True

    @staticmethod
    def _infer_is_prefill(q_nope: torch.Tensor, attn_metadata: Optional[TTMetadata]) -> bool:
        """More than one token per user.  A pass is all prefill or all decode (the scheduler
        guarantees it); a pass without metadata is a profiling run and counts as prefill."""
        if attn_metadata is None or attn_metadata.cache_position is None:
            return True
        users = attn_metadata.cache_position.shape[0]
        assert users > 0, "Invalid number of users"
        return q_nope.shape[0] // users > 1

    @staticmethod
    def _has_cache(kv_cache) -> bool:
        return isinstance(kv_cache, torch.Tensor) and kv_cache.numel() > 0

    def _expand(self, out_lat: torch.Tensor, layer, pattern: str) -> torch.Tensor:
        return torch.einsum(pattern, out_lat, layer.W_UV.to(device=out_lat.device))

    def _bf16_on_gpu(self, *tensors) -> bool:
        """bfloat16 on one GPU.  (The weights are plain attributes and may sit elsewhere: such a pass moves them.)
        Not if autograd, a forward-mode derivative or a functional transform may look at one of them: the operators
        that take a pass at once have no derivative, while the products around the attention have."""
        device = tensors[0].device
        if device.type != "cuda":
            return False
        bf16, watched = torch.bfloat16, torch.is_grad_enabled()
        for t in tensors:  # (a loop: a short prompt is bound by the host)
            if t.dtype is not bf16 or t.device != device or (watched and t.requires_grad):
                return False
        return torch.compiler.is_compiling() or (
            torch.autograd.forward_ad._current_level < 0 and torch._C._functorch.peek_interpreter_stack() is None)

    def _steps_at_once(self, q_nope, q_pe, kv_c_normed, k_pe, kv_cache, attn_metadata, layer, output) -> bool:
        """Whether a decode pass is one ``tt::latent_decode_step_``: the head shape it is built for, causal, with a
        cache to write.  (Without a cache the pass is a profiling run, which the operators in turn refuse.)"""
        if (self.qk_nope_head_dim, self.qk_rope_head_dim, self.kv_lora_rank, self.v_head_dim) != (128, 64, 512, 128):
            return False
        if self.functional_cache_ops or not attn_metadata.is_causal or not self._has_cache(kv_cache) or not kv_cache.is_contiguous():
            return False
        if self.scale is None:  # (the operators' default is theirs to choose)
            return False
        if not self._bf16_on_gpu(q_nope, q_pe, kv_c_normed, k_pe, layer.W_UK_T, layer.W_UV, kv_cache, output):
            return False
        return output.is_contiguous()  # (its address is the operator's business: a traced tensor has none)

    def _expands_prompts(self, q_nope, q_pe, kv_c_normed, k_pe, kv_cache, attn_metadata, layer, s, output) -> bool:
        """A prompt pass attends only its own tokens, so K and V can be expanded per head (scores over
        nope + rope features, values of v_head_dim) where the absorbed form works on kv_lora_rank +
        rope features for every head: 3.4 times fewer matrix operations at 128 + 64 / 128 over a rank of 512, and
        the expansion costs what absorption and output expansion cost.  Built for that head shape, causal."""
        if (self.qk_nope_head_dim, self.qk_rope_head_dim, self.v_head_dim) != (128, 64, 128) or s % 32 or self.functional_cache_ops:
            return False
        if attn_metadata is not None and (attn_metadata.attn_mask is not None or not attn_metadata.is_causal):
            return False
        if not self._bf16_on_gpu(q_nope, q_pe, kv_c_normed, k_pe, layer.W_UK_T, layer.W_UV, output) or self.scale is None or not self.scale > 0:
            return False
        if attn_metadata is not None and self._has_cache(kv_cache) and kv_cache.dtype != torch.bfloat16:
            return False
        return output.is_contiguous()  # (its address is the operator's business: a traced tensor has none)

    def _forward_prefill_short(self, q_nope, q_pe, kv_c_normed, k_pe, kv_cache, attn_metadata, layer, s, users, output):
        """A prompt of up to 64 tokens in the absorbed form: its error against a 64-bit evaluation is smaller there (a latent
        output of few keys is rounded less than each of their values; 16 heads, 32 / 64 / 96 / 160 tokens: 2.851e-3 / 2.975e-3 /
        3.062e-3 / 3.155e-3 against 2.871e-3 / 2.993e-3 / 3.056e-3 / 3.140e-3 expanded), and so short a pass is bound by
        the host: the steps of the operators in turn in fewer calls, one prompt of 32 tokens 165 -> 112 us (100 expanded)."""
        n, lat, rope = self.num_heads, self.kv_lora_rank, self.qk_rope_head_dim
        rows = lambda w: w if w.stride(-1) == 1 else w.contiguous()  # noqa: E731  (no batched product with a transposed right operand)
        latent, rotary = kv_c_normed.view(users, s, lat), k_pe.view(users, s, rope)
        heads = lambda t, width: t.view(users * s, n, width).transpose(0, 1)  # noqa: E731
        q_abs = torch.bmm(heads(q_nope, self.qk_nope_head_dim), rows(layer.W_UK_T))             # [N, tokens, L]
        q_lat = torch.cat([q_abs, heads(q_pe, rope)], -1).view(n, users, s, lat + rope).transpose(0, 1)
        out_lat = _ops.flash_mla_prefill(query=q_lat, key=torch.cat([latent, rotary], -1).unsqueeze(1), head_dim_v=lat, scale=self.scale)
        out = torch.bmm(out_lat.transpose(0, 1).reshape(n, users * s, lat), rows(layer.W_UV))   # [N, tokens, V]
        heads(output, self.v_head_dim).copy_(out)
        if attn_metadata is not None and self._has_cache(kv_cache):
            torch.ops.tt.paged_fill_latent_cache_(kv_cache, latent, rotary, attn_metadata.fill_page_table)

    def _forward_prefill_expanded(self, q_nope, q_pe, kv_c_normed, k_pe, kv_cache, attn_metadata, layer, s, users, output):
        n, lat, rope, nope, vd = self.num_heads, self.kv_lora_rank, self.qk_rope_head_dim, self.qk_nope_head_dim, self.v_head_dim
        latent = kv_c_normed.view(users, s, lat)
        rotary = k_pe.view(users, s, rope)
        rows = latent.reshape(users * s, lat)
        k_nope = torch.mm(rows, layer.W_UK_T.reshape(n * nope, lat).t())                      # [tokens, N * P]
        v = torch.mm(rows, layer.W_UV.transpose(0, 1).reshape(lat, n * vd))                   # [tokens, N * V]
        heads = lambda t, width: t.view(users, s, n, width).transpose(1, 2)  # noqa: E731
        torch.ops.tt.split_key_prefill_out(
            heads(q_nope, nope), heads(q_pe, rope), heads(k_nope, nope), rotary.unsqueeze(1), heads(v, vd),
            heads(output, vd), float(self.scale))
        # the new tokens' latent keys go into the paged cache (skipped in profiling runs)
        if attn_metadata is not None and self._has_cache(kv_cache):
            torch.ops.tt.paged_fill_latent_cache_(kv_cache, latent, rotary, attn_metadata.fill_page_table)

    def _forward_prefill(self, q_lat, k_lat, kv_cache, attn_metadata, layer, seq_len, users):
        out_lat = _ops.flash_mla_prefill(
            query=q_lat.transpose(1, 2).contiguous(),        # [users, N, S, L+R]
            key=k_lat.transpose(1, 2).contiguous(),          # [users, 1, S, L+R]
            head_dim_v=self.kv_lora_rank,
            value=None,
            attn_mask=attn_metadata.attn_mask if attn_metadata is not None else None,
            is_causal=attn_metadata.is_causal if attn_metadata is not None else True,
            scale=self.scale,
        )                                                    # [users, N, S, L]
        out = self._expand(out_lat, layer, "bnsl,nlv->bnsv")  # [users, N, S, V]
        out = out.transpose(1, 2).reshape(users * seq_len, self.num_heads * self.v_head_dim)

        # the new tokens' latent keys go into the paged cache (skipped in profiling runs)
        if attn_metadata is not None and self._has_cache(kv_cache):
            fill = k_lat.transpose(1, 2)                     # [users, 1, S, L+R], a view
            table = attn_metadata.fill_page_table
            if self.functional_cache_ops:
                filled = kv_cache
                for u in range(users):
                    filled = _ops.paged_fill_cache(
                        filled, fill[u : u + 1], table,
                        batch_idx=torch.tensor([u], dtype=torch.int32, device=kv_cache.device))
                kv_cache.copy_(filled)
            else:
                _ops.paged_fill_cache_(
                    kv_cache, fill, table,
                    torch.arange(users, dtype=torch.int32, device=kv_cache.device))
        return out

    def _forward_decode(self, q_lat, k_lat, kv_cache, attn_metadata, layer, users):
        # the new token's latent key goes into the cache first (skipped in profiling runs)
        if self._has_cache(kv_cache):
            fresh = k_lat.transpose(0, 1)                    # [1, users, 1, L+R]
            if self.functional_cache_ops:
                kv_cache.copy_(_ops.paged_update_cache(
                    kv_cache, fresh, attn_metadata.cache_position, attn_metadata.page_table))
            else:
                _ops.paged_update_cache_(
                    kv_cache, fresh, attn_metadata.cache_position, attn_metadata.page_table)
        is_causal = attn_metadata.is_causal if attn_metadata is not None else True
        out_lat = _ops.paged_flash_mla_decode(
            query=q_lat.transpose(0, 1),                     # [1, users, N, L+R]
            key=kv_cache,
            head_dim_v=self.kv_lora_rank,
            page_table=attn_metadata.page_table,
            value=None,
            is_causal=is_causal,
            attn_mask=None if is_causal else attn_metadata.attn_mask,
            cur_pos_tensor=attn_metadata.cache_position,
            scale=self.scale,
        )                                                    # [1, users, N, L]
        out = self._expand(out_lat.reshape(users, self.num_heads, self.kv_lora_rank), layer, "bnl,nlv->bnv")
        return out.reshape(users, self.num_heads * self.v_head_dim)
