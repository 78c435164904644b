"""Prompt portions of attention through a latent with the heads' own keys and values, and when that serves a step."""
from __future__ import annotations

import ctypes
from typing import Optional

import torch

from . import library
from .attention_fast import compute_units
from .kernels import KernelError, _check, _check_cache2, _check_table, _ptr, _stream

c_float = ctypes.c_float
TILE = 64                    # keys of a tile (csrc/latent_prompt.hip)
QUERIES = 128                # queries of a workgroup
MAX_BYTES = 1 << 31          # of the keys and values that a step lays out


def supported(dim: int, rot_dim: int, value_dim: int, rank: int) -> bool:
    return all(n in (32, 64, 128) for n in (dim, rot_dim, value_dim)) and rank % 32 == 0 and 32 <= rank <= 256


def bucket(tiles: int) -> int:
    """Room for so many tiles: the next of 2^k and 3 2^k, so that a recorded step serves contexts of a range of lengths."""
    room = 16
    while room < tiles:
        if room * 3 // 2 >= tiles:
            return room * 3 // 2
        room *= 2
    return room


class LatentPrompt:
    """Attention of a step's portions; a step's single tokens, in front of them, are served in the latent's space.  ``uk`` [H dim, rank], ``uv`` [H value_dim, rank]: the heads' key and value matrices, bfloat16."""

    def __init__(self, heads: int, dim: int, rot_dim: int, value_dim: int, rank: int, scale: float, uk: torch.Tensor, uv: torch.Tensor):
        self.heads, self.d, self.r, self.dv, self.rank, self.scale = heads, dim, rot_dim, value_dim, rank, float(scale)
        if tuple(uk.shape) != (heads * dim, rank) or tuple(uv.shape) != (heads * value_dim, rank) or uk.dtype != torch.bfloat16 \
                or uv.dtype != torch.bfloat16 or not uk.is_contiguous() or not uv.is_contiguous():
            raise KernelError("latent prompt: the heads' matrices must be contiguous bfloat16 [heads * entries, latent]")
        self.uk, self.uv = uk, uv
        self.lib = library.latent_prompt_library(dim, rot_dim, value_dim, rank)
        self.slots = max(1, 2 * compute_units() // heads)      # workgroups a head: two a compute unit in all
        self.least = 4                                         # tiles of keys that a workgroup has at least

    @staticmethod
    def pays(tokens: int, keys: int, singles: int) -> bool:
        """Whether a step's portions, of so many tokens that see so many keys, are served here.  What is paid here is a key's
        product (12 heads: 27 us for 6,144 keys) and in the latent's space a query's.  Microseconds, latent's space / here, 12 heads of
        128 + 64 and 128 and a latent of 256: 8 tokens behind 0, 1,000 and 8,000: 19 / 17, 25 / 29, 36 / 58; 32: 23 / 17, 29 / 31, 48 / 60;
        48: 28 / 17, 33 / 31, 69 / 61; 64: 28 / 17, 37 / 31, 72 / 62; 128: 53 / 21, 69 / 34, 142 / 68 (28 heads cross at the same places).
        With single tokens in front of the portions these need launches of their own (about 25 us), which 96 tokens earn."""
        if singles:
            return tokens >= 96
        return tokens >= 48 or keys <= 16 * tokens

    def plan(self, ctx) -> Optional[tuple]:
        """(single tokens in front, room for tiles of keys) if the step's portions are served here, else None.  Decided on the
        host from the shape of the step, once for all layers; the filler of a recorded step does not count, only its room."""
        key = ("latent_prompt", self.heads, self.d, self.r, self.dv, self.rank)
        if key not in ctx.shared:
            ctx.shared[key] = self._plan(ctx)
        return ctx.shared[key]

    def _plan(self, ctx) -> Optional[tuple]:
        if ctx.all_decode or "cu_seqlens" not in ctx.host or "context_lens" not in ctx.host:
            return None
        B, cu, filler = ctx.num_seqs, ctx.host["cu_seqlens"], int(ctx.host.get("filler", 0))
        real, lead = B - filler, 0
        while lead < real and cu[lead + 1] - cu[lead] == 1:
            lead += 1
        contexts = [int(c) for c in ctx.host["context_lens"][lead:real]]
        tokens = int(cu[real] - cu[lead])
        if not contexts or not self.pays(tokens, sum(contexts), lead):
            return None
        room = bucket(sum(-(-c // TILE) for c in contexts)) + (-(-ctx.num_tokens // TILE) if filler else 0)
        fits = room * TILE * self.heads * (self.d + self.dv) * 2 <= MAX_BYTES and (ctx.num_tokens // QUERIES + B) * room < 1 << 30
        return (lead, room) if fits else None

    def __call__(self, q: torch.Tensor, table: torch.Tensor, cache, block_table: torch.Tensor, ctx, plan: tuple, out: torch.Tensor,
                 gate: Optional[torch.Tensor] = None) -> torch.Tensor:
        """q [T, >= heads (dim + rot_dim)], unturned; writes rows of ``out`` [T, heads value_dim] from the first portion's on."""
        lead, room = plan
        first = int(ctx.host["cu_seqlens"][lead])
        return self.run(q, table, cache.k, cache.v, block_table[lead:], ctx.cu_seqlens[lead:], ctx.context_lens[lead:],
                        ctx.num_seqs - lead, first, room, out, gate)

    def run(self, q, table, k_cache, v_cache, block_table, cu_seqlens, context_lens, num_seqs: int, first: int, room: int,
            out: torch.Tensor, gate: Optional[torch.Tensor] = None) -> torch.Tensor:
        H, T, dev = self.heads, q.shape[0], q.device
        pages, P = _check_cache2(k_cache, v_cache, 1, self.rank + self.r, self.rank)
        for t in (q, k_cache, out) + ((gate,) if gate is not None else ()):
            if not t.is_cuda or t.dtype != torch.bfloat16:
                raise KernelError("latent prompt: bfloat16 tensors on the GPU")
        for t, cols, what in ((q, H * (self.d + self.r), "queries"), (out, H * self.dv, "outputs"), (gate, H, "gates")):
            if t is not None and (t.dim() != 2 or t.shape[0] != T or t.stride(1) != 1 or t.shape[1] < cols):
                raise KernelError(f"latent prompt: {what} must be [T, >= {cols}] with unit stride along the row")
        if block_table.dtype != torch.int32 or block_table.dim() != 2 or not block_table.is_contiguous() or block_table.shape[0] < num_seqs:
            raise KernelError("block_table must be contiguous int32 [sequences, pages]")
        for t, n in ((cu_seqlens, num_seqs + 1), (context_lens, num_seqs)):
            if t.dtype != torch.int32 or t.numel() < n or not t.is_contiguous():
                raise KernelError("sequence metadata must be contiguous int32")
        _check_table(table, T, self.r // 2)
        kx = torch.empty(room * H * TILE * self.d, dtype=torch.bfloat16, device=dev)
        vx = torch.empty(room * H * TILE * self.dv, dtype=torch.bfloat16, device=dev)
        kr = torch.empty(room * TILE * self.r, dtype=torch.bfloat16, device=dev)
        part = torch.empty(H * self.slots * 2 * QUERIES * (self.dv + 4), dtype=torch.float32, device=dev)
        _check(self.lib, self.lib.pico_latent_prompt(
            _ptr(q), q.stride(0) if T > 1 else q.shape[1], _ptr(table), _ptr(k_cache), _ptr(self.uk), _ptr(self.uv), _ptr(block_table),
            block_table.shape[1], _ptr(cu_seqlens), _ptr(context_lens), num_seqs, first, T, _ptr(kx), _ptr(vx), _ptr(kr), room, _ptr(part),
            self.slots, self.least, _ptr(out), out.stride(0) if T > 1 else out.shape[1], _ptr(gate),
            0 if gate is None else (gate.stride(0) if T > 1 else gate.shape[1]), H, self.d, self.r, self.dv, self.rank, P, pages,
            c_float(self.scale), _stream()))
        return out
