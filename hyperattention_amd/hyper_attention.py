"""HyperAttention module: same constructor and forward signature as the reference
(hyper_attention.py:9-132), computed by the HIP library.

The host path of a call is native (csrc/torch_host.cpp).  Without gradients a forward is one library call
(ha_forward: q and k hashed in one launch, the rows ranked once for all levels, leaves, then each level merged in
place).  With inputs that require grad it is one autograd node that keeps what the backward needs: q and k
are hashed in one launch and the rows ranked once for all levels (ha_forward_sort), every attention call of
the recursion works on segments of the whole tensors, one pass merges their results, and in the backward the
calls' gradients are accumulated by the kernels.

The residual estimator is composed here from the same HIP operators, following the reference's recursion step by step.
"""
from __future__ import annotations

import math

import torch

from . import _lib, ops
from .angular_lsh import AngularLSH


class HyperAttention(torch.nn.Module):

    def __init__(self, input_dim=64, lsh_num_projs=8, block_size=256, sample_size=256, min_seq_len=2048,
                 smooth_block=False, **kwargs):
        """
        - block_size and sample_size must be divisible by 128
        Optional keyword hooks (not in the reference, for reproducible runs): `rng` (torch.Generator
        for the projection), `proj_dir` (explicit (input_dim, lsh_num_projs) projection) and
        `sampled_idx` (explicit sampled key rows, shape (sample_size,); with gradients and without mask also a list
        per key/value head, (heads, sample_size) or (batch, heads, sample_size)).
        `residual_estimator=True` (not in the reference either; the estimator of the HyperAttention paper):
        every hashed call weights its sampled keys by n_key / sample_size and leaves out those that are
        already among the block keys of the query.  Forward only, head dims 64 and 128.
        """
        super().__init__()
        self.input_dim = input_dim
        self.lsh_num_projs = lsh_num_projs
        self.block_size = block_size
        self.sample_size = sample_size
        self.min_seq_len = min_seq_len
        self.smooth_block = smooth_block
        self.lsh = AngularLSH(num_projs=self.lsh_num_projs, dim=(1, 1, input_dim), rng=kwargs.get('rng'))
        if kwargs.get('proj_dir') is not None:
            proj = torch.as_tensor(kwargs['proj_dir']).reshape(1, 1, input_dim, lsh_num_projs)
            self.lsh.proj_dir = proj.to(self.lsh.proj_dir.dtype).clone()
        self.sampled_idx = kwargs.get('sampled_idx')
        self.residual_estimator = bool(kwargs.get('residual_estimator', False))
        # for callers that run the one-call forward through ops.hyper_forward and keep its workspace with the module
        self._workspace = ops.WorkspaceCache()

    def forward(self, query: torch.tensor, key: torch.tensor, value: torch.tensor, scale=None, causal=False,
                return_lse=False):
        """
        inputs:
            - query, key, value: (batch, heads, seq_len, dim); same sequence lengths
            - sequence lengths must be divisible by block_size
        output:
            - attn: (approximation of) the attention output (batch, heads, seq_len, dim_v)
            - lse: (approximation of) log-sum-exp of the scaled qk matrix, (batch, heads, seq_len, 1)
        """
        dim, dim_v = key.shape[-1], value.shape[-1]
        proj = self.lsh.proj_dir
        if self.residual_estimator:
            return self._forward_residual_estimator(query, key, value, scale or dim ** (-0.5), causal, return_lse)
        sampled = self._sampled(query, key, value, causal) if self.sampled_idx is not None else None
        run = _lib.host().forward
        result = run(query, key, value, proj, sampled, scale or 0.0, causal is not False, self.lsh_num_projs,
                     self.block_size, self.sample_size, self.min_seq_len, bool(self.smooth_block))
        if result is None:
            # Head dims that are multiples of 8 run as they are, without gradients with a value dim apart from the
            # q/k dim.  Others run zero-padded: zero columns change neither the projections, nor q.k, nor the
            # wanted outputs
            wide = ops.padded_head_dim(max(dim, dim_v))
            pad = lambda x: torch.nn.functional.pad(x, (0, wide - x.shape[-1]))
            attn, lse = run(pad(query), pad(key), pad(value), torch.nn.functional.pad(proj, (0, 0, 0, wide - dim)), sampled,
                            scale or dim ** (-0.5), causal is not False, self.lsh_num_projs, self.block_size,
                            self.sample_size, self.min_seq_len, bool(self.smooth_block))
            result = attn[..., :dim_v], lse
        return result if return_lse else result[0]

    def _sampled(self, query, key, value, causal):
        """The module's explicit sample list as an int32 device tensor, checked against the shortest hashed call (the
        list serves every level); None where no call is hashed.  One list for all heads; the one call of a pass with
        gradients and without mask takes a list per key/value head too, as hyper_attn_func does."""
        shortest = ops.smallest_hashed_key_length(query.shape[2], self.min_seq_len, causal is not False)
        if shortest is None:
            return None
        ops.check_sampled_idx(self.sampled_idx, shortest)
        sampled = self.sampled_idx.to(device=query.device, dtype=torch.int32).contiguous()
        shapes, heads = [(self.sample_size,)], key.shape[1]
        if causal is False and ops._wants_grad(query, key, value):
            shapes += [(heads, self.sample_size), (key.shape[0], heads, self.sample_size)]
        assert sampled.shape in shapes, f"the module's sampled_idx must have one of the shapes {shapes}"
        return sampled

    def _forward_residual_estimator(self, query, key, value, scale, causal, return_lse):
        if ops._wants_grad(query, key, value):
            raise NotImplementedError("residual_estimator has no backward")
        n_query, n_key = query.shape[2], key.shape[2]
        assert n_query == n_key
        dim, dim_v = key.shape[-1], value.shape[-1]
        proj = self.lsh.proj_dir
        if dim % 8 or dim_v % 8:
            assert dim <= 128 and dim_v <= 128, "FlashAttention only support head dimensions up to 128"
            wide = ops.padded_head_dim(max(dim, dim_v))
            pad = lambda x: torch.nn.functional.pad(x, (0, wide - x.shape[-1]))
            query, key, value = pad(query), pad(key), pad(value)
            proj = torch.nn.functional.pad(proj, (0, 0, 0, wide - dim))
        if key.shape[1] != query.shape[1] and causal is not False:
            # grouped-query inputs on the operator-by-operator recursion: it follows the reference, which
            # folds halves into heads (hyper_attention.py:67-68), and that needs as many k/v heads as q
            # heads; a single un-masked call takes the groups as they are
            group = query.shape[1] // key.shape[1]
            key, value = key.repeat_interleave(group, dim=1), value.repeat_interleave(group, dim=1)
        attn, lse = self._forward_composed(query.contiguous(), key.contiguous(), value.contiguous(), scale, causal, proj)
        attn = attn[..., :dim_v]
        if causal is not False and n_key <= self.min_seq_len:
            # a top-level leaf: the exact kernel's padded 3-d lse
            lse = torch.nn.functional.pad(lse.squeeze(-1), (0, -(-n_key // 128) * 128 - n_key))
        return (attn, lse) if return_lse else attn

    # ---- the reference's recursion, operator by operator (the residual estimator; a check of the others) --------
    def _forward_composed(self, query, key, value, scale, causal, proj=None):
        batch_size, n_heads, n_key, dim = key.shape
        n_query = query.shape[2]
        if causal is False:
            return self.forward_no_causal_mask(query, key, value, scale, proj)
        if n_key <= self.min_seq_len:
            attn, lse = ops.flash_attn_func(query.transpose(1, 2), key.transpose(1, 2), value.transpose(1, 2),
                                            None, True, scale)
            return attn.transpose(1, 2), lse[:, :, :n_query].unsqueeze(-1)
        if n_query % 2:
            query = torch.nn.functional.pad(query, (0, 0, 0, 1), mode='constant', value=0.)
            key = torch.nn.functional.pad(key, (0, 0, 0, 1), mode='constant', value=0.)
            value = torch.nn.functional.pad(value, (0, 0, 0, 1), mode='constant', value=0.)
        half = key.shape[2] // 2
        q_bd = query.view(batch_size, 2 * n_heads, half, query.shape[-1])
        k_bd = key.view(batch_size, 2 * n_heads, half, key.shape[-1])
        v_bd = value.view(batch_size, 2 * n_heads, half, value.shape[-1])
        attn_bd, lse_bd = self._forward_composed(q_bd, k_bd, v_bd, scale, True, proj)
        attn_bd = attn_bd.contiguous().view(batch_size, n_heads, -1, value.shape[-1])
        lse_bd = lse_bd.contiguous().view(batch_size, n_heads, -1, 1)
        attn_unmasked, lse_unmasked = self.forward_no_causal_mask(
            query[:, :, half:, :], key[:, :, :half, :], value[:, :, :half, :], scale, proj)
        attn_down, lse_down = ops.add_self_attentions(attn_bd[:, :, half:, :], lse_bd[:, :, half:, :],
                                                      attn_unmasked, lse_unmasked)
        attn = torch.cat((attn_bd[:, :, :half, :], attn_down), dim=-2)
        lse = torch.cat((lse_bd[:, :, :half, :], lse_down), dim=-2)
        if n_query % 2:
            attn = attn[:, :, :-1, :]
            lse = lse[:, :, :-1, :]
        return attn, lse

    def forward_no_causal_mask(self, query, key, value, scale, proj=None):
        """
            - sequence lengths must be divisible by block_size
            - proj (not in the reference): projection to hash with instead of the module's own
        """
        batch_size, head_size, n_query, dim = query.shape

        if self.min_seq_len > n_query:
            attn, lse = ops.flash_attn_func(query.transpose(1, 2), key.transpose(1, 2), value.transpose(1, 2),
                                            None, False, scale)
            lse = lse[:, :, :n_query]
        else:
            num_keys = 1 << self.lsh_num_projs
            query_sort_idx = ops.bucket_argsort(self.lsh.hash(query, proj), num_keys)
            key_sort_idx = ops.bucket_argsort(self.lsh.hash(key, proj), num_keys)
            estimator = {}
            if self.residual_estimator and self.sample_size > 0:
                estimator = dict(sample_bias=math.log(key.shape[2] / self.sample_size), mask_sampled_in_block=True)
            attn, lse = ops.hyper_attn_func(query.transpose(1, 2), key.transpose(1, 2), value.transpose(1, 2),
                                            query_sort_idx.transpose(1, 2), key_sort_idx.transpose(1, 2),
                                            self.block_size, self.sample_size, scale, self.smooth_block,
                                            sampled_idx=self.sampled_idx, **estimator)
        attn = attn.transpose(1, 2)
        return attn, lse.unsqueeze(-1)
