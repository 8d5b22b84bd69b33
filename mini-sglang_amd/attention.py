"""HipAttnBackend: the MI355X attention backend behind the reference's plugin API.

Implements the five abstract methods of BaseAttnBackend (P/attention/base.py:18-34) and the
metadata contract (`get_last_indices`, P/attention/base.py:12-15, fa.py:32-33) with the gfx950
kernels.  Differences from the reference backends that matter for speed, none for results:

* the page table is read IN PLACE: the kernels walk `ctx.page_table[req.table_idx, :len]`
  (token slots, page-size agnostic) directly, so `prepare_metadata` builds no per-step
  `[B, max_k / page]` table (cf. fa.py:92-97: B slice views + a stack + a div per step) and
  graph replay copies two `[B]` int vectors instead of a `[B, max_seq/page]` table;
* all per-batch integers travel in ONE pinned host buffer / ONE async H2D copy;
* decode work is split by a device-side plan (no host sync, fixed grids => graph-safe).
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Any, Dict, List, Optional

import numpy as np
import torch

from . import _lib, ops
from . import core as _core


@dataclass
class HipAttnMetadata:
    cu_seqlens_q: torch.Tensor  # [B+1] int32, device
    seq_lens: torch.Tensor      # [B]   int32, device (= cache_seqlens / device_len)
    req_rows: torch.Tensor      # [B]   int32, device (= req.table_idx)
    batch: int
    max_seqlen_q: int
    max_seqlen_k: int
    tile_cu: Optional[torch.Tensor] = None  # [B+1] int32 (prefill only)
    total_tiles: int = 0
    tile_order: Optional[torch.Tensor] = None  # [total_tiles] int32: q tiles, most keys first (prefill only)
    ranges: tuple = (1, 0)                  # key ranges of a q tile, 64-key tiles of each (prefill only)
    scratch: Optional[torch.Tensor] = None  # their partial sums, or those of one-token prompts, from the first layer on
    pairs: bool = False                     # two heads a workgroup (prefill only)
    fresh: bool = False                     # short prompts that have nothing in the pool (prefill only)
    plan: Optional[torch.Tensor] = None     # decode work list (device)
    chunks: Optional[tuple] = None          # recurrent layers: (items [n, 3], item_first [B + 1], n) of long portions cut in pieces
    delta_chunks: Optional[tuple] = None    # the same list at the delta-rule layers' piece size
    ssd_chunks: Optional[tuple] = None      # the same list at the state-space layers' piece size

    def get_last_indices(self, bs: int) -> torch.Tensor:
        return self.cu_seqlens_q[1: 1 + bs] - 1


def prefill_tile_order(seqlens_q: np.ndarray, seqlens_k: np.ndarray, tiles: np.ndarray,
                       q_tile: Optional[int] = None) -> np.ndarray:
    """Launch order of the q tiles (q_tile rows each; default: the default prefill kernel's) of a prefill batch: by
    decreasing number of keys the tile attends (tile t of request b sees keys [0, min(k_b, k_b - q_b + min((t + 1) *
    q_tile, q_b)))), ties in natural order.  A scheduling hint only (longest-processing-time first shortens the launch
    tail); results do not depend on it."""
    if q_tile is None:
        q_tile = ops.prefill_q_tile()
    total = int(tiles.sum())
    req = np.repeat(np.arange(len(tiles)), tiles)
    first = np.cumsum(tiles) - tiles
    t_in = np.arange(total) - first[req]
    q, k = seqlens_q[req], seqlens_k[req]
    kend = np.minimum(k, k - q + np.minimum((t_in + 1) * q_tile, q))
    return np.argsort(-kend, kind="stable").astype(np.int32)


def fill_metadata_host(h: np.ndarray, seqlens_q: np.ndarray, seqlens_k: np.ndarray, rows: np.ndarray,
                       decode: bool, q_tile: int = _lib.PREFILL_QTILE) -> None:
    """Per-batch integers of `prepare_metadata` (fa.py:67-105) in one int32 buffer of 4 B + 2 (+ tiles) words:
    [seq_lens = device_len (cache_seqlens) | rows = table_idx | cu_seqlens_q [B+1] | tile_cu [B+1] | tile_order].
    cu_seqlens_q is the reference's in all three regimes (arange for decode, = cu_seqlens_k without a cache
    hit, own cumsum with one): it is always the exclusive prefix of extend_len."""
    bs = len(seqlens_q)
    h[:bs] = seqlens_k
    h[bs: 2 * bs] = rows
    h[2 * bs] = 0
    h[2 * bs + 1: 3 * bs + 1] = np.cumsum(seqlens_q)
    if not decode:
        tiles = (seqlens_q + q_tile - 1) // q_tile
        h[3 * bs + 1] = 0
        h[3 * bs + 2: 4 * bs + 2] = np.cumsum(tiles)
        h[4 * bs + 2:] = prefill_tile_order(seqlens_q, seqlens_k, tiles, q_tile)


SMALL_DECODE_HEADS = 32  # (request, kv head) pairs up to which decode attention takes the small-batch kernel whatever the table's width


class HipAttnBackend:
    """Paged attention (prefill + decode) over the reference's KV pool and global page table."""

    def __init__(self, config: Any, ctx: Any = None, *, tp_size: int = 1, decode_capacity: int = 0) -> None:
        ctx = ctx if ctx is not None else _core.get_global_ctx()
        self.ctx = ctx
        self.config = config
        self.kvcache = ctx.kv_cache
        self.page_size = ctx.page_size
        # aligned runs of this many positions never cross a page => consecutive slots (cache.py:42-53)
        self.slot_run = self.page_size & -self.page_size
        self.device = self.kvcache.device
        self.head_dim = config.head_dim
        self.scale = config.head_dim ** -0.5
        self.tp_size = tp_size
        self._q_tile = ops.prefill_q_tile()  # query rows per tile of the prefill kernel in use (unit of tile_cu / tile_order)
        self.qo_heads = config.num_qo_heads // tp_size
        self.kv_heads = max(config.num_kv_heads // tp_size, 1)
        self.max_bs = int(ctx.page_table.shape[0])
        self.capacity = decode_capacity or max(4096, 4 * self.max_bs)
        self._plan_words = ops.attn_decode_plan_words(self.max_bs, self.capacity)
        self._small_heads = 0  # requests x kv heads of a decode batch up to which `small_decode` says yes
        if self.head_dim == 128 and self.qo_heads % self.kv_heads == 0 and self.qo_heads // self.kv_heads <= 8:
            self._small_heads = SMALL_DECODE_HEADS * (2 if self.kv_heads <= 2 or int(ctx.page_table.shape[1]) <= 4096 else 1)
        # decode steps only: one at a time per backend (prompts have scratch of their own)
        small = (ops.attn_decode_small_workspace_bytes(b, ops.attn_decode_small_ranges(b, self.kv_heads, ctx.page_table.shape[1]), self.qo_heads)
                 for b in range(1, self._small_heads // self.kv_heads + 1))
        self._workspace = torch.empty(max([ops.attn_decode_workspace_bytes(self.capacity, self.qo_heads, self.head_dim), *small]),
                                      dtype=torch.uint8, device=self.device)
        self._layers_workspaces: Dict[tuple, torch.Tensor] = {}  # (layers, hidden size, intermediate size) -> what decode_layers' workgroups meet in
        self._layers_failed: Dict[tuple, tuple] = {}  # likewise: (pinned copy of its error word, event behind the copy)
        self._md_calls = 0
        # graph state
        self.capture_bs: List[int] = []
        self.max_graph_bs = 0
        self._cap_seq: Optional[torch.Tensor] = None
        self._cap_rows: Optional[torch.Tensor] = None
        self._cap_plan: Optional[torch.Tensor] = None
        self._cap_cu_q: Optional[torch.Tensor] = None
        self._cap_planned: set = set()  # captured batch sizes whose attention reads the work plan

    # ------------------------------------------------------------------ forward
    def _kv_tokens(self, layer_id: int):
        k = self.kvcache.k_cache(layer_id)
        v = self.kvcache.v_cache(layer_id)
        return k.view(-1, k.shape[-2], k.shape[-1]), v.view(-1, v.shape[-2], v.shape[-1])

    def small_decode(self, batch: Any) -> bool:
        """Whether the batch's decode attention takes the kernel that does the new tokens' row work itself
        (csrc/attn_decode_small.hip), in place of row work, planned kernel and merge.  us of a step saved by it per layer, inside
        captured steps of Qwen3-0.6B (28 layers, 16 heads on 8) | of six layers of a 14B model (40 on 8), bf16:
          table of 40960 tokens   1 request of 533 4.8 | 8.8     4 of 533 2.0 | 5.2     8 of 533 1.8 | 4.7     5 of 8000 - | 1.1
          just wide enough        4 of 533 6.6 | 9.9             8 of 533 2.5 | 5.7     8 of 2000 2.4 | 4.4    8 of 4000 1.5 | 1.3
        Its requests are half lines, and it loses once the stream is long: 8 of 8000 - | -0.8, 8 of 16000 - | -23.  A captured step does
        not know its lengths, so more than 32 (request, kv head) pairs take it only where the table ends at 4096 tokens.  At 4
        requests it is ahead up to 12000 tokens (8000 - | 5.8, 12000 - | 2.3) and loses from 14000 on with three and more heads a kv
        head (16000 30 | -1.7, 32000 - | -13.6, of some 250), which the shorter ones are worth.  With 1 or 2 kv heads it is ahead
        up to 64 pairs at all lengths (a chain of attention alone, 10 on 2, 32 requests: 533 tokens 20.1 / 16.7, 16000 105.4 / 104.6;
        5 on 1, 64: 533 20.1 / 16.6, 16000 107.0 / 101.6)."""
        md = batch.attn_metadata
        return md.max_seqlen_q == 1 and md.batch * self.kv_heads <= self._small_heads

    def _decode_scratch(self, batch: Any) -> torch.Tensor:
        """The decode kernels' partial sums: decode steps share the backend's; a prompt that extends by one token a request, which may run beside a
        step on another stream, has its own for its layers one after the other."""
        if self._decode_phase(batch):
            return self._workspace
        md: HipAttnMetadata = batch.attn_metadata
        if md.scratch is None:
            md.scratch = torch.empty_like(self._workspace)
        return md.scratch

    def _attend_small(self, q, k, v, layer_id: int, batch: Any, **row_work) -> torch.Tensor:
        md: HipAttnMetadata = batch.attn_metadata
        k_tok, v_tok = self._kv_tokens(layer_id)
        table = self.ctx.page_table
        out = torch.empty((q.shape[0], q.shape[1]), dtype=q.dtype, device=q.device)
        ranges = ops.attn_decode_small_ranges(md.batch, self.kv_heads, table.shape[1])
        ops.attn_decode_small(out, q, k, v, k_tok, v_tok, batch.out_loc, table, md.req_rows, md.seq_lens, self._decode_scratch(batch), ranges, self.scale, **row_work)
        return out.view(q.shape[0], self.qo_heads, self.head_dim)

    def attend_new(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, q_norm_w, k_norm_w, eps: float, positions: torch.Tensor,
                   cos_sin: torch.Tensor, layer_id: int, batch: Any) -> torch.Tensor:
        """qk-norm, RoPE, K / V store and attention of a batch that `small_decode` says yes to, from the projection's rows."""
        return self._attend_small(q, k, v, layer_id, batch, q_norm_w=q_norm_w, k_norm_w=k_norm_w, eps=eps, positions=positions, cos_sin_cache=cos_sin)

    def takes_layers(self, batch: Any, hidden: int, intermediate: int, layers: int) -> bool:
        """Whether all layers of the batch's decode step go in one launch (csrc/decode_layers.hip): a batch of `small_decode` whose layer fits the compute units'
        LDS, where that launch was ahead at every length.  Separate launches against it, % of a step in an engine as wide as its requests, or wider than 4096
        tokens for longer ones (hidden size, heads on kv heads; 12 - 28 layers, bf16):
          8 and more kv heads: 1 - 8 requests of 16 - 40000 tokens, 1024 and 768 columns, 16 on 8, 8 on 8, 10 on 10: -26 .. -1 (8 x 4000 -3 .. -1, 1 x 32000 -14 .. -2)
          3 - 5: up to 4 requests in up to 4096 tokens -24 .. -3 (12, 16, 24 on 4, 10 on 5, 6 on 3), 6 x 1000 -5, but 8 x 533 -3 .. 0 and 8 x 1000 on 16 on 4 +4; longer
            ones 1 x 8000 +8 .. +10, 1 x 32000 +5 .. +9
          1, 2: up to 3 in up to 4096 -29 .. 0, but 4 x 4080 -5 .. +3, 8 x 2000 -1 .. +6, 8 x 4000 up to +12, 1 x 8000 0 .. +5
          512 columns (half of the compute units have rows of a product): 1 x 533 -16 .. -14, but 1 x 4000 -2 .. +2, 8 requests -6 .. +15, 1 x 32000 +6 .. +9
        A captured step does not know its lengths.  Not prompts that extend by one token: what the launch's workgroups meet in is one for all decode steps, which may
        run beside a prompt.  Nor a capture that no step of the model came before: the zeros that the first launch starts from would be written when the graph is
        replayed, and by every replay."""
        few = 4 if self.kv_heads >= 3 else 3
        return (self._decode_phase(batch) and batch.positions.dtype == batch.out_loc.dtype == torch.int32
                and hidden >= 3 * int(_lib.lib().msgl_device_cu_count()) and self.small_decode(batch)
                and (self.kv_heads >= 8 or batch.attn_metadata.batch <= few and int(self.ctx.page_table.shape[1]) <= 4096)
                and ops.decode_layers_supported(batch.attn_metadata.batch, hidden, self.qo_heads, self.kv_heads, intermediate)
                and ((layers, hidden, intermediate) in self._layers_workspaces or not torch.cuda.is_current_stream_capturing()))

    def _layers_workspace(self, layers: int, hidden: int, intermediate: int) -> torch.Tensor:
        """Zeros for a model's decode steps of all batches; like the decode workspace: one step at a time."""
        at = (layers, hidden, intermediate)
        if at not in self._layers_workspaces:
            need = max(ops.decode_layers_workspace_bytes(b, layers, hidden, self.qo_heads, self.kv_heads, intermediate)
                       for b in range(1, self._small_heads // self.kv_heads + 1)
                       if ops.decode_layers_supported(b, hidden, self.qo_heads, self.kv_heads, intermediate))
            self._layers_workspaces[at] = torch.zeros(need, dtype=torch.uint8, device=self.device)
        return self._layers_workspaces[at]

    def poll_errors(self) -> None:
        """Raise if a workgroup of a one-launch step ever gave up waiting for another one's rows (the step's logits were NaN then, not a partial result).  One
        4-byte asynchronous copy: it looks at the word that the previous poll asked for, complete by now in any loop that synchronises once per step."""
        for at, workspace in self._layers_workspaces.items():
            word, done = self._layers_failed.get(at, (None, None))
            if word is None:
                word = torch.zeros(1, dtype=torch.int32, pin_memory=True)
            elif not done.query():
                continue
            if int(word[0]):
                raise _lib.MsglError(f"decode_layers: a workgroup gave up waiting in launch {int(word[0]) & 0xffffffff}; its step's logits are NaN")
            word.copy_(ops.decode_layers_failed(workspace), non_blocking=True)
            done = torch.cuda.Event()
            done.record()
            self._layers_failed[at] = word, done

    def decode_layers(self, x: torch.Tensor, layers: Any, interleaved: bool, eps: float, positions: torch.Tensor, cos_sin: torch.Tensor, batch: Any):
        """Every layer of a batch that `takes_layers` says yes to: the last down projection's rows and the residual stream without them."""
        md: HipAttnMetadata = batch.attn_metadata
        tokens = [self._kv_tokens(i) for i in range(len(layers))]
        return ops.decode_layers(x, layers, [k for k, _ in tokens], [v for _, v in tokens], positions, cos_sin, batch.out_loc, self.ctx.page_table, md.req_rows,
                                 md.seq_lens, self._layers_workspace(len(layers), x.shape[1], layers[0].down.shape[1]), self.qo_heads, interleaved, eps, self.scale)

    def forward(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, layer_id: int, batch: Any) -> torch.Tensor:
        """Reference contract (fa.py:48-65): persist k, v at batch.out_loc, then attend.  A decode batch's out_loc is where its requests'
        last table entries point, as the scheduler allocates them."""
        if self.small_decode(batch):
            q2, k2, v2 = (t.reshape(t.shape[0], -1) for t in (q, k, v))
            if (batch.out_loc.dtype == torch.int32 and batch.out_loc.is_contiguous() and {t.dtype for t in (q, k, v)} == {self.kvcache.dtype}
                    and all(t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0 for t in (q2, k2, v2))):
                return self._attend_small(q2, k2, v2, layer_id, batch)
        if batch.attn_metadata.fresh and self._takes_fresh(q, k, v, batch):
            return self._attend_fresh(q, k, v, layer_id, batch)
        self.kvcache.store_kv(k, v, batch.out_loc, layer_id)
        return self.attend(q, layer_id, batch)

    def _takes_fresh(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, batch: Any) -> bool:
        """Whether a batch of short prompts with nothing cached goes from its rows as they come, and into the pool, in one launch (one stride, 16-byte pieces, no key
        ranges or pairs of heads; the default kernel).  Its page table then says of the new tokens what out_loc says, as the scheduler allocates them."""
        md, loc = batch.attn_metadata, batch.out_loc
        if md.ranges[0] > 1 or md.pairs or ops.PREFILL_IMPL not in (0, 4) or self.head_dim != 128 or loc.dtype != torch.int32 or not loc.is_contiguous():
            return False
        k2, v2 = (t.view(t.shape[0], -1) for t in (k, v))
        return (q.shape[0] == k2.shape[0] == loc.numel() and {q.dtype, k.dtype, v.dtype} == {self.kvcache.dtype} and k2.shape[1] == self.kv_heads * self.head_dim
                and k2.shape == v2.shape and k2.stride() == v2.stride() and k2.stride(1) == 1 and k2.stride(0) % 8 == 0
                and k2.data_ptr() % 16 == 0 and v2.data_ptr() % 16 == 0)

    def _attend_fresh(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, layer_id: int, batch: Any) -> torch.Tensor:
        md: HipAttnMetadata = batch.attn_metadata
        q = q.view(-1, self.qo_heads, self.head_dim)
        out = torch.empty((q.shape[0], self.qo_heads, self.head_dim), dtype=q.dtype, device=q.device)
        ops.attn_prefill_fresh(out, q, k.view(k.shape[0], -1), v.view(v.shape[0], -1), *self._kv_tokens(layer_id), batch.out_loc, md.seq_lens, md.cu_seqlens_q,
                               md.tile_cu, md.batch, md.total_tiles, self.scale, tile_order=md.tile_order)
        return out

    def attend(self, q: torch.Tensor, layer_id: int, batch: Any) -> torch.Tensor:
        """Attention only (K/V for this batch already in the pool, e.g. via the fused
        qk-norm + RoPE + store kernel)."""
        md: HipAttnMetadata = batch.attn_metadata
        q = q.view(-1, self.qo_heads, self.head_dim)
        out = torch.empty((q.shape[0], self.qo_heads, self.head_dim), dtype=q.dtype, device=q.device)
        k_tok, v_tok = self._kv_tokens(layer_id)
        table = self.ctx.page_table
        if md.max_seqlen_q == 1:
            if md.plan is None:  # prepared for replay but run eagerly by the host: plan on first use
                md.plan = torch.empty(self._plan_words, dtype=torch.int32, device=self.device)
                ops.attn_decode_plan(md.plan, md.seq_lens, md.batch, self.max_bs, self.capacity, self.qo_heads,
                                     self.kv_heads)
            elif md.plan is self._cap_plan:
                self._cap_planned.add(md.batch)
            ops.attn_decode(out, q, k_tok, v_tok, table, md.req_rows, md.seq_lens, md.plan, self._decode_scratch(batch),
                            md.batch, self.max_bs, self.capacity, self.scale, slot_run=self.slot_run)
        else:
            if md.ranges[0] > 1 and md.scratch is None:
                # this batch's own, for its layers one after the other: other batches may run beside it on other streams, decode steps among them
                md.scratch = torch.empty(ops.prefill_ranges_workspace_bytes(md.total_tiles * self.qo_heads * md.ranges[0]), dtype=torch.uint8, device=self.device)
            ops.attn_prefill(out, q, k_tok, v_tok, table, md.req_rows, md.seq_lens, md.cu_seqlens_q, md.tile_cu,
                             md.batch, md.total_tiles, self.scale, tile_order=md.tile_order,
                             ranges=md.ranges, workspace=md.scratch, pairs=md.pairs)
        return out

    # ------------------------------------------------------------------ metadata
    def prepare_metadata(self, batch: Any) -> None:
        self._md_calls += 1
        if self.tp_size > 1:
            # driven by the reference's scheduler nobody else sees the communicator once decode runs from captured
            # graphs: every 16th step look at the peer-to-peer error word (one 4-byte async copy; raises on a timeout)
            if self._md_calls % 16 == 0:
                from .kernel import poll_communicator_errors

                poll_communicator_errors(sync=False)
        if self._layers_workspaces and self._md_calls % 64 == 0 and not torch.cuda.is_current_stream_capturing():  # captured one-launch steps likewise
            self.poll_errors()
        reqs = batch.padded_reqs
        bs = len(reqs)
        seqlens_q = np.fromiter((r.extend_len for r in reqs), dtype=np.int64, count=bs)
        seqlens_k = np.fromiter((r.device_len for r in reqs), dtype=np.int64, count=bs)
        rows = np.fromiter((r.table_idx for r in reqs), dtype=np.int64, count=bs)
        max_q, max_k = int(seqlens_q.max()), int(seqlens_k.max())
        decode = max_q == 1
        q_tile = self._q_tile
        total_tiles = 0 if decode else int(((seqlens_q + q_tile - 1) // q_tile).sum())
        # one pinned buffer, one async H2D copy: [seq_lens | rows | cu_q | tile_cu | tile_order]
        host = torch.empty(4 * bs + 2 + total_tiles, dtype=torch.int32, pin_memory=True)
        fill_metadata_host(host.numpy(), seqlens_q, seqlens_k, rows, decode, q_tile)
        dev = host.to(self.device, non_blocking=True)
        md = HipAttnMetadata(
            cu_seqlens_q=dev[2 * bs: 3 * bs + 1], seq_lens=dev[:bs], req_rows=dev[bs: 2 * bs], batch=bs,
            max_seqlen_q=max_q, max_seqlen_k=max_k, tile_cu=None if decode else dev[3 * bs + 1: 4 * bs + 2],
            total_tiles=total_tiles, tile_order=None if decode else dev[4 * bs + 2:],
            ranges=(1, 0) if decode else ops.prefill_ranges(total_tiles, self.qo_heads, max_q, max_k),
            pairs=not decode and ops.prefill_pairs(total_tiles, self.qo_heads, self.kv_heads, seqlens_q, seqlens_k),
            fresh=not decode and max_q <= ops.FRESH_TOKENS and bool((seqlens_q == seqlens_k).all()),
        )
        if decode and not self._replayed_from_graph(batch, bs):
            # runs eagerly: plan now (device side, no sync).  Only batches the engine will REPLAY are planned
            # later, in prepare_for_replay; replay is keyed on the phase (P/engine/graph.py:149-150
            # can_use_cuda_graph = batch.is_decode and size <= max_graph_bs), NOT on max_q == 1: a prefill
            # batch whose every request extends by one token (radix full hit on a repeated prompt at
            # page_size 1, P/scheduler/cache.py:27-30; a one-token chunk remainder) takes this kernel eagerly
            md.plan = torch.empty(self._plan_words, dtype=torch.int32, device=self.device)
            ops.attn_decode_plan(md.plan, md.seq_lens, bs, self.max_bs, self.capacity, self.qo_heads, self.kv_heads)
        batch.attn_metadata = md

    @staticmethod
    def _decode_phase(batch: Any) -> bool:
        phase = getattr(batch, "phase", None)
        return phase == "decode" if phase is not None else True

    def _replayed_from_graph(self, batch: Any, padded_bs: int) -> bool:
        return bool(self._decode_phase(batch) and self._cap_plan is not None and padded_bs in self.capture_bs
                    and len(batch.reqs) <= self.max_graph_bs)

    # ------------------------------------------------------------------ graph hooks
    def init_capture_graph(self, max_seq_len: int, bs_list: List[int]) -> None:
        assert self._cap_plan is None, "Capture already initialized."
        max_bs = max(bs_list)
        assert max_bs <= self.max_bs
        self.max_graph_bs = max_bs
        self.capture_bs = sorted(bs_list)
        self._cap_seq = torch.ones(max_bs, dtype=torch.int32, device=self.device)
        self._cap_rows = torch.zeros(max_bs, dtype=torch.int32, device=self.device)
        self._cap_cu_q = torch.arange(0, max_bs + 1, dtype=torch.int32, device=self.device)
        self._cap_plan = torch.zeros(self._plan_words, dtype=torch.int32, device=self.device)

    def prepare_for_capture(self, batch: Any) -> None:
        bs = batch.size
        assert bs in self.capture_bs and self._cap_plan is not None
        # dummy requests: length 1, all rows = the dummy request's table row
        self._cap_rows[:bs].fill_(batch.reqs[0].table_idx)
        self._cap_seq[:bs].fill_(1)
        ops.attn_decode_plan(self._cap_plan, self._cap_seq, bs, self.max_bs, self.capacity, self.qo_heads, self.kv_heads)
        batch.attn_metadata = HipAttnMetadata(
            cu_seqlens_q=self._cap_cu_q[: bs + 1], seq_lens=self._cap_seq[:bs], req_rows=self._cap_rows[:bs],
            batch=bs, max_seqlen_q=1, max_seqlen_k=int(self.ctx.page_table.shape[1]), plan=self._cap_plan,
        )

    def prepare_for_replay(self, batch: Any) -> None:
        md, bs = batch.attn_metadata, batch.padded_size
        assert isinstance(md, HipAttnMetadata) and bs in self.capture_bs and self._cap_plan is not None
        self._cap_seq[:bs].copy_(md.seq_lens)
        self._cap_rows[:bs].copy_(md.req_rows)
        if bs in self._cap_planned:
            ops.attn_decode_plan(self._cap_plan, self._cap_seq, bs, self.max_bs, self.capacity, self.qo_heads, self.kv_heads)


class MixAttnBackend:
    """Batch metadata for the hybrid decoders (latent attention + linear recurrence): the same three vectors the paged
    backend hands its kernels -- keys per request after this forward, page-table row, exclusive prefix of new tokens -- in
    one pinned buffer and one asynchronous copy.  Their kernels take prompt portions, single decoded tokens and any mix of
    the two in one launch, so there is no prefill / decode split and no work plan; the recurrent layers use the table row
    as the request's state slot.  Graph capture keeps static copies of the vectors, refreshed before every replay."""

    RECURRENT_CHUNK = 128
    DELTA_CHUNK = 256
    SSD_CHUNK = 64
    SCAN_CHUNK = 64

    def __init__(self, config: Any, ctx: Any = None, *, tp_size: int = 1) -> None:
        ctx = ctx if ctx is not None else _core.get_global_ctx()
        self.ctx, self.config = ctx, config
        self.kvcache = ctx.kv_cache
        self.device = self.kvcache.device
        self.max_bs = int(ctx.page_table.shape[0])
        self.capture_bs: List[int] = []
        self._cap: Optional[torch.Tensor] = None
        self._kinds = {getattr(s, "kind", "") for s in getattr(config, "layers", ())}
        self._decay_heads = max((s.heads for s in getattr(config, "layers", ()) if getattr(s, "kind", "") in ("retention", "gla")), default=0)
        parts = [p for s in getattr(config, "layers", ()) for p in (getattr(s, "left", None), getattr(s, "right", None)) if p]
        self._kinds |= {getattr(p, "kind", "") for p in parts}
        self._delta_pieces = any(not _lib.mix_lib().msgl_mix_delta_rule_block_floats(s.dim, s.vdim) for s in [*getattr(config, "layers", ()), *parts]
                                 if getattr(s, "kind", "") in ("delta", "channel_delta"))

    @staticmethod
    def decay_chunk(tokens: int, heads: int) -> int:
        """Piece size of the decay recurrences in a step of `tokens` new tokens: as many (piece, head) workgroups as the chip holds at a
        time (two per compute unit), in whole 16-token pieces, between 32 and 512 tokens."""
        return min(max(-(-tokens * heads // (512 * 16)) * 16, 32), 512)

    def prepare_metadata(self, batch: Any) -> None:
        reqs = batch.padded_reqs
        bs = len(reqs)
        q = np.fromiter((r.extend_len for r in reqs), dtype=np.int64, count=bs)
        k = np.fromiter((r.device_len for r in reqs), dtype=np.int64, count=bs)
        rows = np.fromiter((r.table_idx for r in reqs), dtype=np.int64, count=bs)
        # a long portion's recurrence runs as pieces in parallel (their states joined by a scan): RECURRENT_CHUNK tokens for the
        # decay-only recurrence, DELTA_CHUNK for the delta rule, whose scan step is a [d, d] x [d, dv] product per piece (head sizes that
        # have no form in blocks; the others take the blocks for any portion of that length and read no list)
        lists = []
        if int(q.max()) >= 2 * self.RECURRENT_CHUNK and self._kinds & {"lightning"}:
            lists.append(("chunks", self.RECURRENT_CHUNK))
        if self._delta_pieces and int(q.max()) >= 2 * self.DELTA_CHUNK:
            lists.append(("delta_chunks", self.DELTA_CHUNK))
        if int(q.max()) >= 2 * self.SSD_CHUNK and "state_space" in self._kinds:
            lists.append(("ssd_chunks", self.SSD_CHUNK))
        if int(q.max()) >= 2 * self.SCAN_CHUNK and "mamba1" in self._kinds:
            lists.append(("scan_chunks", self.SCAN_CHUNK))
        if self._decay_heads:
            c = self.decay_chunk(int(q.sum()), self._decay_heads)
            if int(q.max()) >= 2 * c:
                lists.append(("decay_chunks", c))
        pieces = [-(-q // c) for _, c in lists]
        extra = sum(3 * int(p.sum()) + bs + 1 for p in pieces)
        host = torch.empty(3 * bs + 1 + extra, dtype=torch.int32, pin_memory=True)
        h = host.numpy()
        h[:bs], h[bs: 2 * bs], h[2 * bs] = k, rows, 0
        h[2 * bs + 1: 3 * bs + 1] = np.cumsum(q)
        at, where = 3 * bs + 1, []
        for (name, c), p in zip(lists, pieces):
            n_items = int(p.sum())
            req = np.repeat(np.arange(bs), p)
            first = np.cumsum(p) - p
            begin = (np.arange(n_items) - first[req]) * c
            items = h[at: at + 3 * n_items].reshape(n_items, 3)
            items[:, 0], items[:, 1], items[:, 2] = req, begin, np.minimum(begin + c, q[req])
            h[at + 3 * n_items] = 0
            h[at + 3 * n_items + 1: at + 3 * n_items + bs + 1] = np.cumsum(p)
            where.append((name, at, n_items))
            at += 3 * n_items + bs + 1
        dev = host.to(self.device, non_blocking=True)
        batch.attn_metadata = HipAttnMetadata(cu_seqlens_q=dev[2 * bs: 3 * bs + 1], seq_lens=dev[:bs], req_rows=dev[bs: 2 * bs], batch=bs,
                                              max_seqlen_q=int(q.max()), max_seqlen_k=int(k.max()))
        for name, at, n_items in where:
            setattr(batch.attn_metadata, name, (dev[at: at + 3 * n_items], dev[at + 3 * n_items: at + 3 * n_items + bs + 1], n_items))

    # ------------------------------------------------------------------ graph hooks
    def init_capture_graph(self, max_seq_len: int, bs_list: List[int]) -> None:
        assert self._cap is None, "Capture already initialized."
        n = max(bs_list)
        assert n <= self.max_bs
        self.capture_bs = sorted(bs_list)
        self._cap = torch.zeros(3 * n + 1, dtype=torch.int32, device=self.device)
        self._cap_n = n

    def _static(self, bs: int) -> HipAttnMetadata:
        n, c = self._cap_n, self._cap
        return HipAttnMetadata(cu_seqlens_q=c[2 * n: 2 * n + bs + 1], seq_lens=c[:bs], req_rows=c[n: n + bs], batch=bs,
                               max_seqlen_q=1, max_seqlen_k=int(self.ctx.page_table.shape[1]))

    def prepare_for_capture(self, batch: Any) -> None:
        bs, n = batch.size, self._cap_n
        assert bs in self.capture_bs
        self._cap[:bs].fill_(1)
        self._cap[n: n + bs].fill_(batch.reqs[0].table_idx)
        self._cap[2 * n: 2 * n + bs + 1].copy_(torch.arange(bs + 1, dtype=torch.int32, device=self.device))
        batch.attn_metadata = self._static(bs)

    def prepare_for_replay(self, batch: Any) -> None:
        md, bs, n = batch.attn_metadata, batch.padded_size, self._cap_n
        assert bs in self.capture_bs
        self._cap[:bs].copy_(md.seq_lens)
        self._cap[n: n + bs].copy_(md.req_rows)
        self._cap[2 * n: 2 * n + bs + 1].copy_(md.cu_seqlens_q)
