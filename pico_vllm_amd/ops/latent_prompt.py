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
MAX_BYTES = 1 << 31          # of the keys and values that a step lays out, where memory for them is left (``LatentPrompt.limit``)


def supported(dim: int, rot_dim: int, value_dim: int, rank: int) -> bool:
    return all(n in (32, 64, 128) for n in (dim, rot_dim, value_dim)) and rank % 32 == 0 and 32 <= rank <= 256


def bucket(tiles: int) -> int:
    """Room of a recorded step for so many tiles: the next of 64 4^k, so that three recordings serve contexts of up to 65,536 tokens."""
    room = 64
    while room < tiles:
        room *= 4
    return room


class LatentPrompt:
    """Attention of a step's portions; a step's single tokens, in front of them, are served in the latent's space.  ``uk`` [H dim, rank], ``uv`` [H value_dim, rank]: the heads' key and value matrices, bfloat16."""

    def __init__(self, heads: int, dim: int, rot_dim: int, value_dim: int, rank: int, scale: float, uk: torch.Tensor, uv: torch.Tensor):
        self.heads, self.d, self.r, self.dv, self.rank, self.scale = heads, dim, rot_dim, value_dim, rank, float(scale)
        if tuple(uk.shape) != (heads * dim, rank) or tuple(uv.shape) != (heads * value_dim, rank) or uk.dtype != torch.bfloat16 \
                or uv.dtype != torch.bfloat16 or not uk.is_contiguous() or not uv.is_contiguous():
            raise KernelError("latent prompt: the heads' matrices must be contiguous bfloat16 [heads * entries, latent]")
        # (read in sixteens of bytes)
        self.uk, self.uv = (t if t.data_ptr() % 16 == 0 else t.clone() for t in (uk, uv))
        self.lib = library.latent_prompt_library(dim, rot_dim, value_dim, rank)
        self.slots = max(1, 2 * compute_units() // heads)      # workgroups a head: two a compute unit in all
        self.least = 4                                         # tiles of keys that a workgroup has at least
        self.limit: Optional[int] = None                       # bytes of a step's workspaces, if something limits them

    def gain(self, portions, singles: int) -> float:
        """Microseconds that a step's portions, pairs (new tokens, context), are expected to take less here than in the latent's space.
        Here a portion pays for its keys, whoever reads them: their way into memory and out of it, and products for whole tiles of
        queries; there for its tokens' products and for every pair, and from 65 rows on for the batched products' launches and copies
        and for the longest context, which few workgroups walk.  With single tokens in front of the portions these need launches of
        their own.  A fit to 196 steps of seven sets of sizes (12 to 28 heads, latents of 32 to 256, 1 to 16 portions of 4 to 2,048 tokens
        behind up to 8,000), of which it sends 11 the slower way, by 10 % at most; 4 of 140 drawn ones of five other sets, by 27 %.  Microseconds, latent's space / here, 12 heads of
        128 + 64 and 128, latents of 256 and 64: 32 tokens 31 / 24 and 22 / 22, behind 8,000 56 / 68 and 35 / 56; 64 behind 8,000 85 / 72 and 49 /
        60; six portions of 16 behind 8,000 154 / 234 and 87 / 207; 200 83 / 41 and 62 / 38; 2,048 behind 4,096 478 / 170 and 254 / 154."""
        tokens, keys = sum(n for n, _ in portions), sum(c for _, c in portions)
        pairs, tiles = sum(n * c for n, c in portions), sum(-(-n // QUERIES) * QUERIES * c for n, c in portions)
        many = tokens + singles >= 65
        H, outputs = self.heads, self.heads * (self.d + self.dv)
        return ((23.0 + 4.0e-3 * max(c for _, c in portions) if many else 0.0) + 4.5e-8 * tokens * outputs * self.rank
                + (5.6e-9 if many else 7.9e-9) * pairs * H * (2 * self.rank + self.r)
                - 5.2e-7 * keys * outputs - 2.4e-9 * tiles * H * (self.d + self.r + self.dv) - (16.5 if singles else 0.0) - (2.0 if len(portions) > 1 else 0.0))

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
        portions = [(int(cu[b + 1] - cu[b]), int(ctx.host["context_lens"][b])) for b in range(lead, real) if cu[b + 1] > cu[b]]
        if not portions or self.gain(portions, lead) <= 0:
            return None
        need = sum(-(-int(c) // TILE) for c in ctx.host["context_lens"][lead:real])
        behind = -(-ctx.num_tokens // TILE) if filler else 0
        most = (MAX_BYTES if self.limit is None else max(0, min(MAX_BYTES, self.limit - self.part_bytes))) // self.tile_bytes - behind
        room = (min(bucket(need), most) if filler else need) + behind
        return (lead, room) if need <= most and (ctx.num_tokens // QUERIES + B) * room < 1 << 30 else None

    @property
    def tile_bytes(self) -> int:
        """Keys and values of a tile."""
        return TILE * (self.heads * (self.d + self.dv) + self.r) * 2

    @property
    def part_bytes(self) -> int:
        """Sums of the tiles of queries whose keys several workgroups share."""
        return self.heads * self.slots * 2 * QUERIES * (self.dv + 4) * 4

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
        part = torch.empty(self.part_bytes // 4, dtype=torch.float32, device=dev)
        _check(self.lib, self.lib.pico_latent_prompt(
            _ptr(q), q.stride(0) if T > 1 else q.shape[1], _ptr(table), _ptr(k_cache), _ptr(self.uk), _ptr(self.uv), _ptr(block_table),
            block_table.shape[1], _ptr(cu_seqlens), _ptr(context_lens), num_seqs, first, T, _ptr(kx), _ptr(vx), _ptr(kr), room, _ptr(part),
            self.slots, self.least, _ptr(out), out.stride(0) if T > 1 else out.shape[1], _ptr(gate),
            0 if gate is None else (gate.stride(0) if T > 1 else gate.shape[1]), H, self.d, self.r, self.dv, self.rank, P, pages,
            c_float(self.scale), _stream()))
        return out
