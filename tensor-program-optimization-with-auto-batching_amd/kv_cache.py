"""Paged caches: host-side page bookkeeping around the HIP attention kernels.

Keeps the host protocol of the reference's cache object
(`tvm/llama_auto_batcher/llama_exec_graph.py:41-46,66,75-79,85,121-127`):
    add_sequence(sid) ; begin_forward(seq_ids, append_lens) ; attention_with_fused_qkv(layer, qkv, n_q_heads) ;
    end_forward()
with RoPE applied inside the cache operator (`llama_for_causal_lm.py:148-174`: rotary_dim = head_dim,
scale 1, no sliding window).  Keys are stored already rotated, which is equivalent to rotating them at
read time and saves the per-step re-rotation of the whole context.

A finished sequence gives its pages and its slot back with free_sequence(sid).

Device layout of PagedKVCache per layer: k [n_pages, Hkv, 16, D], v [n_pages, Hkv, D, 16] (fp16), one int32 block table
[max_seqs, max_blocks], fp32 RoPE tables [max_pos, D/2].
"""
from __future__ import annotations

import numpy as np
import torch

from . import ops
from .decoder_ops import PrefillPlan, TimeMixPlan

PAGE = 16
AT_ONCE = 128       # sequences from which on a pass looks its pages up in one indexing


def rope_tables(head_dim: int, theta: float, max_pos: int):
    """cos/sin [max_pos, head_dim/2] float32 (float64 math, rounded once)."""
    inv_freq = theta ** (-(np.arange(0, head_dim, 2, dtype=np.float64) / head_dim))
    ang = np.arange(max_pos, dtype=np.float64)[:, None] * inv_freq[None, :]
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


class PageTable:
    """The host side of a paged cache: which pages of the pool belong to which sequence, and the protocol of a forward
    pass.  What lies in a page is up to the subclass."""

    def __init__(self, n_pages, max_seqs, max_blocks, max_pos, device, free_pages=None, page_size=PAGE):
        if page_size != PAGE:
            raise ValueError(f"page_size must be {PAGE}")
        self.n_pages, self.max_seqs, self.max_blocks, self.max_pos = n_pages, max_seqs, max_blocks, max_pos
        self.device = torch.device(device)
        self.free = list(range(n_pages)) if free_pages is None else [int(p) for p in free_pages]
        if sorted(self.free) != list(range(n_pages)):
            raise ValueError("free_pages must be a permutation of range(n_pages)")
        # host mirrors (integer bookkeeping is host logic, as in the reference's runtime)
        self.table_h = np.full((max_seqs, max_blocks), -1, dtype=np.int32)
        self.lens = {}          # sid -> committed length
        self.slot = {}          # sid -> row of the block table
        self.free_slots = list(range(max_seqs))
        self.block_table = torch.from_numpy(self.table_h.copy()).to(self.device)
        self._dirty = False
        self._cur = None
        self._staged = None     # (raw stream, event) of arrays queued last
        self._users = {}        # raw stream -> (stream, event behind the last pass's work or None): streams whose work reads the arrays

    # ------------------------------------------------------------------ protocol
    def add_sequence(self, sid):
        if sid in self.slot:
            raise ValueError(f"sequence with id {sid} has already been added")
        if not self.free_slots:
            raise RuntimeError("paged KV cache: no sequence slot left")
        self.slot[sid] = self.free_slots.pop(0)
        self.lens[sid] = 0

    def free_sequence(self, sid):
        """Give back the pages and the slot of a finished sequence."""
        if self._cur is not None:
            raise RuntimeError("free_sequence between begin_forward and end_forward")
        row = self.slot.pop(sid)
        del self.lens[sid]
        self.free.extend(int(p) for p in self.table_h[row] if p >= 0)
        self.table_h[row] = -1
        self.free_slots.insert(0, row)
        self._dirty = True

    def begin_forward(self, seq_ids, append_lens, device_meta=None):
        """Reserve pages for the appended tokens and stage the per-token (sequence, position) arrays."""
        if self._cur is not None:
            raise RuntimeError("begin_forward called twice without end_forward")
        if len(seq_ids) != len(append_lens):
            raise ValueError("seq_ids and append_lens differ in length")
        # Which sequences lack a page (they are handed out in order: the last one needed is missing).  us a step without host-made arrays, one by one / all at
        # once: one sequence 2.5 / 15.5, four 3.6 / 16.3, 64 29 / 34, 212 94 / 81
        if len(seq_ids) < AT_ONCE:
            short = []
            for sid, n in zip(seq_ids, append_lens):
                row, new_len = self.slot[sid], self.lens[sid] + n
                need = -(-new_len // PAGE)
                if new_len > self.max_pos or need > self.max_blocks:
                    raise RuntimeError(f"sequence {sid}: length {new_len} exceeds the cache geometry")
                if need > 0 and self.table_h[row, need - 1] < 0:
                    short.append((row, need))
        else:
            rows, base = self._rows_and_lens(seq_ids)
            new_len = base + np.asarray(append_lens, dtype=np.int64)
            need = -(-new_len // PAGE)
            beyond = (new_len > self.max_pos) | (need > self.max_blocks)
            if beyond.any():
                i = int(beyond.argmax())
                raise RuntimeError(f"sequence {seq_ids[i]}: length {new_len[i]} exceeds the cache geometry")
            short = [(rows[i], int(need[i])) for i in np.flatnonzero((need > 0) & (self.table_h[rows, np.maximum(need, 1) - 1] < 0))]
        for row, need in short:
            for j in range(int((self.table_h[row] >= 0).sum()), need):
                if not self.free:
                    raise RuntimeError("paged KV cache out of pages")
                self.table_h[row, j] = self.free.pop(0)
                self._dirty = True
        self._enter()
        staged = self._dirty or device_meta is None
        if self._dirty:
            self.block_table.copy_(ops.upload(torch.from_numpy(self.table_h), self.device))
            self._dirty = False
        decode = all(n == 1 for n in append_lens)
        if device_meta is not None:
            tok_seq, tok_pos, ctx = device_meta
        elif decode:
            rows, base = self._rows_and_lens(seq_ids)
            tok_seq, tok_pos, ctx = ops.upload(torch.from_numpy(np.stack([rows, base, base + 1])), self.device)
        else:
            rows, base = self._rows_and_lens(seq_ids)
            ts = np.repeat(rows, append_lens).astype(np.int32)
            tp = np.concatenate([b + np.arange(n, dtype=np.int32) for b, n in zip(base, append_lens)]).astype(np.int32)
            tok_seq, tok_pos = ops.upload(torch.from_numpy(np.stack([ts, tp])), self.device)
            ctx = None
        if staged:
            self._stage()
        self._cur = (list(seq_ids), list(append_lens), decode, tok_seq, tok_pos, ctx)

    def _rows_and_lens(self, seq_ids):
        """Block-table rows and lengths of sequences."""
        return np.asarray([self.slot[s] for s in seq_ids], dtype=np.int32), np.asarray([self.lens[s] for s in seq_ids], dtype=np.int32)

    # Host-made arrays are queued on the stream that is current, not waited for, and the next pass overwrites the block table.  So a
    # stream that goes on with a pass waits for its arrays, and the stream that begins the next one waits for all that the last was
    # queued on.  No event from outside may enter a capture: one begins behind a wait for the whole device, or on a stream that its
    # caller has ordered.
    def _raw_stream(self):
        return torch._C._cuda_getCurrentRawStream(self.block_table.device.index)

    def _enter(self):
        """A pass begins on the current stream."""
        if self.device.type != "cuda" or torch.cuda.is_current_stream_capturing():
            return
        raw = self._raw_stream()
        stream = self._users[raw][0] if raw in self._users else torch.cuda.current_stream(self.device)
        for r, (other, behind) in self._users.items():
            if r != raw:
                stream.wait_stream(other) if behind is None else stream.wait_event(behind)
        self._users = {raw: (stream, None)}

    def _stage(self):
        """Arrays of the pass have been queued on the current stream."""
        if self.device.type == "cuda" and not torch.cuda.is_current_stream_capturing():
            raw = self._raw_stream()
            if raw not in self._users:
                self._users[raw] = (torch.cuda.current_stream(self.device), None)
            self._staged = (raw, self._users[raw][0].record_event())

    def _join(self):
        """The pass goes on on the current stream."""
        if self.device.type != "cuda":
            return
        raw = self._raw_stream()
        elsewhere = self._staged is not None and raw != self._staged[0]
        if (raw in self._users and not elsewhere) or torch.cuda.is_current_stream_capturing():
            return
        stream = torch.cuda.current_stream(self.device)
        self._users[raw] = (stream, None)
        if elsewhere:
            stream.wait_event(self._staged[1])
            for t in self._pass_arrays():          # their memory may be given out again, to the stream they were made on
                t.record_stream(stream)

    def __getstate__(self):
        """A copy, or a pickle, is made behind all that the passes have queued and knows no streams (which neither takes)."""
        self._enter()
        return {**self.__dict__, "_staged": None, "_users": {}}

    def _pass_arrays(self):
        """Arrays that were made for the current pass."""
        return [t for t in self._cur[3:] if t is not None]

    def end_forward(self):
        seq_ids, append_lens = self._cur[0], self._cur[1]
        for sid, n in zip(seq_ids, append_lens):
            self.lens[sid] += n
        self._cur = None
        for raw, (stream, _) in self._users.items():         # (the default stream outlives every pass: no event before one is waited for)
            if raw and not torch.cuda.is_current_stream_capturing():
                self._users[raw] = (stream, stream.record_event())

    # ------------------------------------------------------------------ helpers
    def pages_of(self, sid):
        row = self.table_h[self.slot[sid]]
        return row[row >= 0].tolist()


class PagedKVCache(PageTable):
    def __init__(self, n_layers, n_pages, n_kv_heads, head_dim, max_seqs, max_blocks, rope_theta, max_pos,
                 device="cuda:0", free_pages=None, page_size=PAGE):
        super().__init__(n_pages, max_seqs, max_blocks, max_pos, device, free_pages, page_size)
        self.n_layers, self.Hkv, self.D = n_layers, n_kv_heads, head_dim
        if head_dim % 32:
            raise ValueError("head_dim must be a multiple of 32")
        # keys in matrix-core fragment order: element (token, d) of a page at [d // 32, (d % 32) // 8, token, d % 8]
        self.k = torch.zeros((n_layers, n_pages, n_kv_heads, head_dim // 32, 4, PAGE, 8), dtype=torch.float16, device=self.device)
        self.v = torch.zeros((n_layers, n_pages, n_kv_heads, head_dim, PAGE), dtype=torch.float16, device=self.device)
        cos, sin = rope_tables(head_dim, rope_theta, max_pos)
        self.rope_cos = torch.from_numpy(cos).to(self.device)
        self.rope_sin = torch.from_numpy(sin).to(self.device)

    def k_rowmajor(self, layer: int) -> torch.Tensor:
        """The layer's rotated keys as [n_pages, Hkv, 16, D] (a copy, for inspection)."""
        k = self.k[layer]
        return k.permute(0, 1, 4, 2, 3, 5).reshape(self.n_pages, self.Hkv, PAGE, self.D).contiguous()

    def attention_with_fused_qkv(self, layer, qkv, n_q_heads, out=None, frag=False, o_shrink=None):
        """qkv [T, Hq + 2 Hkv, D] (or [T, (Hq + 2 Hkv) * D]) fp16, token-major in begin_forward order.
        Rotates q in place, appends rotated k and v, attends causally; returns [T, Hq * D] fp16
        (frag=True: as a FragActivation ready for the o_proj product).  o_shrink (a decode step only): see
        ops.paged_attn_decode - the call then returns (attention output, head shares of the o projection's shrink)."""
        if self._cur is None:
            raise RuntimeError("attention_with_fused_qkv outside begin_forward/end_forward")
        self._join()
        _, append_lens, decode, tok_seq, tok_pos, ctx = self._cur
        T = sum(append_lens)
        qkv = qkv.view(T, n_q_heads + 2 * self.Hkv, self.D)
        ops.rope_kv_append(qkv, self.k[layer], self.v[layer], self.block_table, tok_seq, tok_pos,
                           self.rope_cos, self.rope_sin, n_q_heads, self.Hkv, self.D)
        if decode:
            return ops.paged_attn_decode(qkv, self.k[layer], self.v[layer], self.block_table, tok_seq, ctx,
                                         n_q_heads, self.Hkv, self.D, out=out, frag=frag, o_shrink=o_shrink)
        if o_shrink is not None:
            raise ValueError("attention_with_fused_qkv: o_shrink is for decode steps")
        return ops.paged_attn_prefill(qkv, self.k[layer], self.v[layer], self.block_table, tok_seq, tok_pos,
                                      n_q_heads, self.Hkv, self.D, out=out, frag=frag)

    def kv_bytes_read_per_step(self, seq_ids):
        """Algorithmic K+V bytes one decode step reads for these sequences, all layers."""
        per_pos = self.n_layers * 2 * self.Hkv * self.D * 2
        return int(sum(self.lens[s] + 1 for s in seq_ids)) * per_pos


class PagedLatentCache(PageTable):
    """Pages of latent attention: per layer one vector per token, the normed latent and the rotated key part, in the page
    layout of latent_attention.hip.  A layer may read another layer's pages instead of having its own."""

    def __init__(self, layers, n_pages, max_seqs, max_blocks, max_pos, dtype, device="cuda:0", free_pages=None, page_size=PAGE):
        """layers: per layer (kv_rank, rot_dim, rotation, owner): owner is the layer whose pages this one reads (itself,
        if it has its own); rotation: rotary.Rotation."""
        super().__init__(n_pages, max_seqs, max_blocks, max_pos, device, free_pages, page_size)
        self.dtype = dtype
        self.owner = [o for *_, o in layers]
        self.pages = []
        self.rope = []
        tables = {}
        for l, (rank, rot_dim, rotation, o) in enumerate(layers):
            blocks = -(-rank // 32) + -(-rot_dim // 32)
            # padding between and behind the two parts is read by the matrix cores: it stays zero
            self.pages.append(torch.zeros((n_pages, blocks, 4, PAGE, 8), dtype=dtype, device=self.device) if o == l else self.pages[o])
            key = (rotation, rot_dim)
            if key not in tables:
                tables[key] = tuple(torch.from_numpy(t).to(self.device) for t in rotation.tables(rot_dim, max_pos))
            self.rope.append(tables[key])
        self._plan = None

    def latents(self, layer, sid):
        """The cached vectors [length, blocks * 32] of a sequence (a copy, for inspection)."""
        n = self.lens[sid]
        p = self.pages[layer][torch.tensor(self.pages_of(sid), device=self.device, dtype=torch.int64)]
        return p.permute(0, 3, 1, 2, 4).reshape(-1, p.shape[1] * 32)[:n].contiguous()

    def latent_attention(self, layer, qkv, att, out=None):
        """The mixer of `layer` behind its input projection: qkv [T, att.proj_rows] in begin_forward order (att:
        latent_attention.LatentAttention) -> the heads' outputs, concatenated (`out`: an activation of att.out_cols
        columns)."""
        if self._cur is None:
            raise RuntimeError("latent_attention outside begin_forward/end_forward")
        self._join()
        seq_ids, append_lens, _, tok_seq, tok_pos, _ = self._cur
        ctx = [self.lens[s] + n for s, n in zip(seq_ids, append_lens)]
        return att.attend(qkv, self.pages[layer], self.block_table, tok_seq, tok_pos, *self.rope[layer], max_ctx=max(ctx),
                          store=self.owner[layer] == layer, plan=self.attention_plan(att), out=out)

    def _pass_arrays(self):
        plan = self._plan[1] if self._plan is not None and self._plan[0] is self._cur else None
        return super()._pass_arrays() + ([plan.tiles, plan.phys] if plan is not None else [])

    def attention_plan(self, att):
        """The pass's plan for the prompt form where `att` takes that (one serves all layers), else None."""
        seq_ids, append_lens, decode = self._cur[:3]
        if decode:
            return None
        ctx = [self.lens[s] + n for s, n in zip(seq_ids, append_lens)]
        if not att.prompt_form_pays(list(zip(append_lens, ctx))):
            return None
        if self._plan is None or self._plan[0] is not self._cur:
            self._plan = (self._cur, PrefillPlan([(self.pages_of(s), n, c) for s, n, c in zip(seq_ids, append_lens, ctx)], self.device, wait=False))
            self._stage()
        return self._plan[1]


class PagedStateCache(PageTable):
    """What the layers of a model with recurrent and attention layers keep per sequence, one entry per layer run (a layer that
    runs several times has one for every pass): pages of tied attention, or a state per slot.  A slot needs no clearing:
    kernels start a sequence's state from zero at its position 0."""

    def __init__(self, runs, width_p, n_pages, max_seqs, max_blocks, max_pos, dtype, device="cuda:0", free_pages=None, page_size=PAGE):
        """runs: per layer run the mixer's spec, whose cache_entry says what is kept; width_p: columns of the residual stream."""
        super().__init__(n_pages, max_seqs, max_blocks, max_pos, device, free_pages, page_size)
        self.dtype = dtype
        self.entries = [tuple(torch.zeros(shape, dtype=dtype if elements else torch.float32, device=self.device)
                              for shape, elements in s.cache_entry(n_pages, max_seqs, PAGE, width_p)) for s in runs]
        self._meta = None

    def values(self, run, sid):
        """The cached values [length, G, columns] of a sequence (a copy, for inspection)."""
        p = self.entries[run][0][torch.tensor(self.pages_of(sid), device=self.device, dtype=torch.int64)]
        return p.permute(0, 4, 1, 2, 3, 5).reshape(-1, p.shape[1], p.shape[2] * 32)[: self.lens[sid]].contiguous()

    def state(self, run, sid):
        """The matrix states [H, D, D] of a sequence (a view)."""
        return self.entries[run][0][self.slot[sid]]

    def shift(self, run):
        """The previous tokens' rows [slots, columns] of a recurrent layer run."""
        return self.entries[run][1]

    def _pass(self):
        """Of the current pass, made once for all its layers: {"last": the last token of every token's sequence, "segs": [n][4]
        {slot, first token, tokens, position}} - both None in a decode step - and the plans of the prompt forms, once taken."""
        if self._cur is None:
            raise RuntimeError("outside begin_forward/end_forward")
        self._join()
        if self._meta is None or self._meta[0] is not self._cur:
            seq_ids, lens, decode = self._cur[:3]
            m = {"last": None, "segs": None, "plan": None, "ranges": {}, "host": None}
            if not decode:
                ends = np.cumsum(lens)
                m["host"] = segs = [(self.slot[s], int(e) - n, n, self.lens[s]) for s, n, e in zip(seq_ids, lens, ends)]
                both = np.concatenate([np.asarray(segs, dtype=np.int32).reshape(-1), np.repeat(ends - 1, lens).astype(np.int32)])
                both = ops.upload(torch.from_numpy(both), self.device)
                self._stage()
                m["segs"], m["last"] = both[: 4 * len(segs)].view(-1, 4), both[4 * len(segs):]
            self._meta = (self._cur, m)
        return self._meta[1]

    def _pass_arrays(self):
        out, m = super()._pass_arrays(), self._meta[1] if self._meta is not None and self._meta[0] is self._cur else {}
        if m.get("segs") is not None:
            out += [m["segs"], m["last"]]
        if m.get("plan") is not None:
            out += [m["plan"].tiles, m["plan"].phys]
        return out + [a for r in m.get("ranges", {}).values() for a in (r.ranges, r.seqs)]

    def token_meta(self):
        """(sequence, position, last token of its sequence in the pass) per token."""
        return self._cur[3], self._cur[4], self._pass()["last"]

    def time_mix(self, run, mixes, mixer):
        """The recurrence of a layer run on the five mixes of the pass (mixer: time_mix.TimeMix)."""
        m = self._pass()
        return mixer.run(mixes, self.entries[run][0], m["segs"], self._cur[3], self._cur[4], self.time_mix_plan(mixer))

    def time_mix_plan(self, mixer):
        """The pass's ranges where `mixer` takes the prompt form, else None."""
        m, heads = self._pass(), mixer.spec.heads
        if m["host"] is None or not mixer.prompt_form:
            return None
        if heads not in m["ranges"]:
            m["ranges"][heads] = TimeMixPlan(m["host"], heads, self.device, wait=False)
            self._stage()
        return m["ranges"][heads]

    def attention_plan(self, att):
        """The pass's plan where `att` takes the prompt form, else None."""
        m = self._pass()
        seq_ids, append_lens, decode = self._cur[:3]
        seqs = [(n, self.lens[s] + n) for s, n in zip(seq_ids, append_lens)]
        if decode or not att.prompt_form_pays(seqs):
            return None
        if m["plan"] is None:
            m["plan"] = PrefillPlan([(self.pages_of(s), n, c) for s, (n, c) in zip(seq_ids, seqs)], self.device, wait=False)
            self._stage()
        return m["plan"]

    def tied_attention(self, run, y, att):
        """The attention of a layer run behind its input projection y (att: tied_attention.TiedAttention)."""
        if self._cur is None:
            raise RuntimeError("outside begin_forward/end_forward")
        seq_ids, append_lens, _, tok_seq, tok_pos, _ = self._cur
        max_ctx = max(self.lens[s] + n for s, n in zip(seq_ids, append_lens))
        return att.attend(y, *self.entries[run], self.block_table, tok_seq, tok_pos, max_ctx=max_ctx, plan=self.attention_plan(att))
