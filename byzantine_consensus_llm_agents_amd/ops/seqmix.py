"""HIP bindings of the fp32-stream mixer kernels (csrc/kernels/seqmix_*.hip).

Activations are bf16 or fp32 (one template instance each; fp32 is the exact mode: true-fp32
MFMAs, fp32 vendor GEMMs); the residual stream, norm weights, router and gate are fp32 always.
Every wrapper checks shapes, dtypes and contiguity on the host before it launches, and launches
on the current stream (graph-capturable: no host synchronisation, scratch from the caching
allocator).  Semantics: the functions of the same names in ``reference.py``.
"""

import ctypes
import functools
import math

import torch

c_void_p = ctypes.c_void_p


def _p(t):
    return c_void_p(t.data_ptr()) if t is not None else None


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _req(cond, msg):
    if not cond:
        raise ValueError(msg)


def _check(rc, name):
    if rc != 0:
        raise RuntimeError(f"{name} launch failed (rc={rc})")


def _act(t):
    _req(t.dtype in (torch.bfloat16, torch.float32), "activations: bf16 or fp32")
    return int(t.dtype == torch.float32)


ACT_CODES = {"gelu_tanh": 0, "relu2": 1, "silu": 2, "clamped_glu": 3}
EXPERT_ACTS = {"silu_gated": "silu", "clamped_glu": "clamped_glu"}   # gated experts -> activation of their hidden values

CUS = 256          # compute units of the GPU
WIDE_ROWS = 256    # rows of a position tile of the 256 x 256 expert products
WIDE_SLOTS = 64    # ... taken from this many routed rows per expert on (see `_wide_experts`)

FEW_SLOTS, FEW_WEIGHT = 24, 1 << 18    # position tiles of 32 rows: most routed rows per expert, least weights of a matrix (see `few_row_tiles`)


@functools.lru_cache(maxsize=1024)
def _likely_tiles(n_slots, E, rows):
    """How many tiles of `rows` rows hold n_slots slots that go to E experts at random (an expert has c slots, Poisson): the experts with
    a slot, two standard deviations more than their mean, and the mean of their further tiles."""
    mean, p, below, more = n_slots / E, math.exp(-n_slots / E), 0.0, 0.0
    some = E * (1.0 - p)
    for c in range(4 * rows + 1):
        below, p = below + p, p * mean / (c + 1)
        if c and c % rows == 0:
            more += E * max(0.0, 1.0 - below)     # experts of more than c slots
    return max(1, round(min(E, n_slots, some + 2 * math.sqrt(some * (1.0 - some / E))) + more))


def few_row_tiles(n_slots, E, W, ff, rows):
    """The tiles that are likely to hold rows if an expert layer's products stream the weights past position tiles of 32 rows (csrc/kernels/
    moe_rows.hip), 0 if they do not: up to FEW_SLOTS routed rows per expert, where few experts have a second tile that streams their
    weight again.  All four launches, tiles of 64 rows -> of 32, us: 8 gated experts of 2048 x 2048, top 2: 4 rows per expert 96 -> 53,
    16: 97 -> 54; past the line 25: 95 -> 61, 32: 91 -> 75, 40: 97 -> 121; 4096 x 3072: 16: 194 -> 118, 32: 189 -> 180.
    Ratios of the times over 2 to 256 experts, widths 512 to 4096, hidden widths 256 to 3072, 1 to 768 tokens, top 2 and 8:
    * up to 40 tiles 0.24 to 1.03, but up to 1.07 with experts of 512 x 256: most waves have no part of K there;
    * more tiles get a few workgroups each: 0.61 to 1.04 where these fill the 256 CUs to 0.85 and the experts are
      1024 wide and have 2^20 weights a matrix and more; less filled 0.95 to 1.31 (128 experts, 128 slots: 92 tiles, 2 workgroups
      each), smaller experts 0.86 to 1.4 (256 of 1024 x 256)."""
    if n_slots > FEW_SLOTS * E or W % 64 or ff % 64 or max(W, ff) > 32768 or W * ff < FEW_WEIGHT:
        return 0
    held = _likely_tiles(n_slots, E, rows)
    if held > 40 and (W < 1024 or ff < 512 or W * ff < 1 << 20 or held * (CUS // held) < 0.85 * CUS):
        return 0
    return held


def seqmix_ops(lib, linear, counters):
    from .hip import part_rule

    split_keys = lib.bcg_multimap_split_keys()
    tile_rows = lib.bcg_moe_tile_rows()
    few_rows = lib.bcg_moe_rows_tile()

    def embed_scale_rmsnorm(tokens, table, scale, w, eps, w_offset, out_dtype, add=None):
        _req(tokens.dtype == torch.int32 and tokens.is_contiguous() and tokens.dim() == 1, "tokens int32 [T]")
        _req(table.dim() == 2 and table.is_contiguous() and table.dtype == out_dtype, "table [V, W] in the activation dtype")
        T, W = tokens.numel(), table.shape[1]
        _req(w.dtype == torch.float32 and w.shape == (W,) and w.is_contiguous(), "norm weight fp32 [W]")
        _req(add is None or (add.dtype == torch.float32 and add.shape == (W,) and add.is_contiguous()), "added vector fp32 [W]")
        resid = torch.empty(T, W, dtype=torch.float32, device=table.device)
        out = torch.empty(T, W, dtype=out_dtype, device=table.device)
        _check(lib.bcg_embed_scale_rmsnorm(_p(tokens), _p(table), scale, _p(add), _p(w), eps, w_offset, _p(resid), _p(out), T, W,
                                           table.shape[0], _act(table), _stream()), "embed_scale_rmsnorm")
        return out, resid

    def embed_position(tokens, positions, table, pos_table, out_dtype):
        _req(tokens.dtype == torch.int32 and tokens.is_contiguous() and tokens.dim() == 1, "tokens int32 [T]")
        T, W = tokens.numel(), table.shape[1]
        _req(positions.dtype == torch.int32 and positions.is_contiguous() and positions.numel() == T, "positions int32 [T]")
        for t in (table, pos_table):
            _req(t.dim() == 2 and t.is_contiguous() and t.dtype == out_dtype and t.shape[1] == W and t.shape[0] >= 1,
                 "embedding / position table [rows, W] in the activation dtype")
        x = torch.empty(T, W, dtype=torch.float32, device=table.device)
        out = torch.empty(T, W, dtype=out_dtype, device=table.device)
        _check(lib.bcg_embed_position(_p(tokens), _p(positions), _p(table), _p(pos_table), _p(x), _p(out), T, W, table.shape[0],
                                      pos_table.shape[0], _act(table), _stream()), "embed_position")
        return x, out

    def residual_add_rmsnorm32(residual, parts, w, eps, w_offset, out_dtype, gate=None, gated=None):
        _req(residual.dtype == torch.float32 and residual.dim() == 2 and residual.is_contiguous(), "residual fp32 [T, W]")
        T, W = residual.shape
        typed, f32 = [], []
        for p in parts:
            _req(p.shape == (T, W) and p.is_contiguous(), "residual part [T, W] contiguous")
            (f32 if p.dtype == torch.float32 and out_dtype != torch.float32 else typed).append(p)
        if out_dtype == torch.float32 and len(typed) > 2:
            f32, typed = typed[2:], typed[:2]
        _req(len(typed) <= 2 and len(f32) <= 1 and all(p.dtype == out_dtype for p in typed)
             and all(p.dtype == torch.float32 for p in f32), "residual parts: <= 2 activation-typed + <= 1 fp32")
        if gated is not None:
            _req(gated.shape == (T, W) and gated.is_contiguous() and gated.dtype == out_dtype and gate is not None
                 and gate.dtype == torch.float32 and gate.numel() == T and gate.is_contiguous(), "gated part / gate")
        out = None
        if w is not None:
            _req(w.dtype == torch.float32 and w.shape == (W,) and w.is_contiguous(), "norm weight fp32 [W]")
            out = torch.empty(T, W, dtype=out_dtype, device=residual.device)
        typed = typed + [None, None]
        _check(lib.bcg_residual_add_rmsnorm32(_p(residual), _p(typed[0]), _p(typed[1]), _p(f32[0]) if f32 else None,
                                              _p(gate) if gated is not None else None, _p(gated), _p(w), eps, w_offset,
                                              _p(out), T, W, int(out_dtype == torch.float32), _stream()),
               "residual_add_rmsnorm32")
        return out

    def rmsnorm32(x, w, eps, w_offset, out_dtype):
        return residual_add_rmsnorm32(x, [], w, eps, w_offset, out_dtype)

    def act_fn(x, kind):
        _req(x.dim() == 2 and x.stride(1) == 1, "act_fn: [rows, n] with unit column stride")
        rows, n = x.shape
        out = torch.empty(rows, n, dtype=x.dtype, device=x.device)
        code = ACT_CODES[kind]
        _check(lib.bcg_act_fn(_p(x), _p(out), rows, n, x.stride(0), code, _act(x), _stream()), "act_fn")
        return out

    def _cache_ok(k_cache, v_cache, n_kv, kd, vdim, dtype):
        _req(k_cache.dim() == 4 and v_cache.dim() == 4 and k_cache.is_contiguous() and v_cache.is_contiguous()
             and k_cache.dtype == dtype and v_cache.dtype == dtype, "KV cache: contiguous, activation dtype")
        NB, G, BS, KD = k_cache.shape
        _req(G == n_kv and KD == kd and v_cache.shape == (NB, n_kv, vdim, BS) and BS % 16 == 0,
             "KV cache: K [NB, G, BS, maps dim], V [NB, G, vdim, BS], BS % 16 == 0")
        return NB, BS

    def kv_from_logical(k, v):
        """The cache tensors the kernels read, from logical K [NB, G, BS, KD] / V [NB, G, vdim, BS]
        (tests, tools): with KD % 4 == 0 every (page, head) slab is stored fragment-major, K as
        [KD / 4][BS][4] and V as [BS / 4][vdim][4]; the shapes stay the logical ones."""
        NB, G, BS, KD = k.shape
        if KD % 4:
            return k.contiguous(), v.contiguous()
        vd = v.shape[2]
        kp = k.reshape(NB, G, BS, KD // 4, 4).permute(0, 1, 3, 2, 4).contiguous().view(NB, G, BS, KD)
        vp = v.reshape(NB, G, vd, BS // 4, 4).permute(0, 1, 3, 2, 4).contiguous().view(NB, G, vd, BS)
        return kp, vp

    def kv_to_logical(k, v):
        """Inverse of `kv_from_logical`."""
        NB, G, BS, KD = k.shape
        if KD % 4:
            return k, v
        vd = v.shape[2]
        kl = k.reshape(NB, G, KD // 4, BS, 4).permute(0, 1, 3, 2, 4).contiguous().view(NB, G, BS, KD)
        vl = v.reshape(NB, G, BS // 4, vd, 4).permute(0, 1, 3, 2, 4).contiguous().view(NB, G, vd, BS)
        return kl, vl

    def rope_multi_kv_write(qkv, positions, slots, n_q, n_kv, maps, dim, vdim, inv_freq, k_cache, v_cache):
        T = qkv.shape[0]
        qw, kw, vw = n_q * maps * dim, n_kv * maps * dim, n_kv * vdim
        _req(qkv.dim() == 2 and qkv.stride(1) == 1 and qkv.shape[1] >= qw + kw + vw, "fused projection row [q | k | v | ...]")
        _req(positions.dtype == torch.int32 and slots.dtype == torch.int32 and positions.numel() == T
             and slots.numel() == T and positions.is_contiguous() and slots.is_contiguous(), "positions / slots int32 [T]")
        half = inv_freq.numel()
        _req(inv_freq.dtype == torch.float32 and inv_freq.is_contiguous() and 2 * half <= dim, "inv_freq fp32 [rot/2]")
        NB, BS = _cache_ok(k_cache, v_cache, n_kv, maps * dim, vdim, qkv.dtype)
        q = torch.empty(T, n_q, maps * dim, dtype=qkv.dtype, device=qkv.device)
        _check(lib.bcg_rope_multi_kv_write(_p(qkv), qkv.stride(0), _p(positions), _p(slots), _p(inv_freq), half, _p(q),
                                           _p(k_cache), _p(v_cache), T, n_q, n_kv, maps, dim, vdim, BS, NB, _act(qkv),
                                           _stream()), "rope_multi_kv_write")
        return q

    def multimap_tile_rows(dim, vdim):
        """Query rows per prefill tile (the tile table the engine builds) for these head sizes."""
        return 64  # four waves x 16 rows

    def multimap_attention(q, k_cache, v_cache, meta, scale, maps, lam, head_eps, out_scale, vdim, window=0, sink=None,
                           chunk=0, softcap=0.0, slopes=None, keep=0, parts=None):
        """Prefill tiles (``meta.tiles``) on the MFMA kernel, one-token rows (``meta.single``, or
        every row of a decode step) by pairs or splits of their keys (``parts``: every pair in that many).  ``window`` / ``chunk`` / ``sink``
        (one-map heads): sliding window in keys, or a chunk mask (a query sees the keys of its own
        ``chunk``-aligned block of positions only); fp32 [H] sink logits of the softmax denominator.
        ``softcap`` / ``slopes`` (one-map heads): scaled scores capped by tanh, then fp32 [H] slopes
        times the distance to the key taken off.  ``keep`` (with a window): the sequence's first ``keep``
        keys stay visible."""
        T, H, qd = q.shape
        _req(q.is_contiguous() and qd % maps == 0, "q [T, H, maps dim] contiguous")
        dim = qd // maps
        G = k_cache.shape[1]
        NB, BS = _cache_ok(k_cache, v_cache, G, qd, vdim, q.dtype)
        _req(H % G == 0 and maps in (1, 2) and dim <= (512 if maps == 1 else 128)
             and vdim <= (512 if maps == 1 else 256), "multimap attention: maps <= 2, dim <= 128 and vdim <= 256 (one map: 512)")
        bt = meta.block_tables
        lens = meta.seq_lens if meta.attn_seq_lens is None else meta.attn_seq_lens
        _req(bt.dtype == torch.int32 and bt.dim() == 2 and bt.is_contiguous() and lens.dtype == torch.int32
             and lens.is_contiguous() and lens.numel() == bt.shape[0], "block tables int32 [B, max_blocks], lens int32 [B]")
        out = torch.empty(T, H * vdim, dtype=q.dtype, device=q.device)
        f32 = _act(q)
        tile_rows = meta.tile_rows if not meta.decode else 64
        _req(tile_rows == 64, "prefill tiles: 64 query rows")
        window, chunk = int(window or 0), int(chunk or 0)
        _req(window >= 0 and chunk >= 0 and not (window and chunk)
             and (maps == 1 or (window == 0 and chunk == 0 and sink is None)), "window / chunk / sink: one-map heads, one mask")
        if sink is not None:
            _req(sink.dtype == torch.float32 and sink.numel() == H and sink.is_contiguous(), "sink fp32 [H]")
        softcap = float(softcap or 0.0)
        _req(softcap >= 0 and (maps == 1 or (softcap == 0 and slopes is None)), "softcap / slopes: one-map heads")
        if slopes is not None:
            _req(slopes.dtype == torch.float32 and slopes.numel() == H and slopes.is_contiguous(), "slopes fp32 [H]")
        keep = int(keep or 0) if window else 0   # (without a window nothing is hidden but the future)
        _req(keep >= 0 and (keep == 0 or (softcap == 0 and slopes is None)), "kept first keys: without softcap / slopes")
        common = (H, G, maps, dim, vdim, BS, NB, scale, lam, head_eps, out_scale, tile_rows, f32, window, chunk, _p(sink), softcap,
                  _p(slopes), keep)

        def decode(work, n_items):
            if (not f32 and BS == 16 and n_items <= 65535 and (k_cache.data_ptr() | v_cache.data_ptr()) % 16 == 0
                    and lib.bcg_multimap_pairs(maps, dim, vdim, int(softcap > 0 or slopes is not None), keep)):
                span = bt.shape[1] * BS
                if window or chunk:   # (whole chunks of 32 keys, of the kept ones too)
                    span = min(span, keep + max(window, chunk) + 64)
                pairs = n_items * G * -(-(H // G) // 16)
                if parts is not None:
                    rule = (parts, 0, 0, 0, pairs * (parts - 1))
                    _req(1 <= parts <= 16 and rule[4] <= 1 << 16, "decode parts")
                elif n_items <= 2048:
                    rule = part_rule(pairs, 64 * (maps * dim + vdim), -(-span // 32))
                else:   # (every long row's workgroup looks over all of them)
                    rule = (1, 0, 1, 0, 0)
                ws = torch.empty(2 * rule[4] * 16 * (2 * maps + maps * vdim), dtype=torch.float32, device=q.device) if rule[4] else None
                _check(lib.bcg_multimap_attention(2, _p(q), _p(k_cache), _p(v_cache), _p(bt), bt.shape[1], None, _p(lens), _p(work), n_items,
                                                  _p(out), _p(ws), rule[0], *common, *rule[1:], _p(counters(q.device)) if rule[4] else None,
                                                  _stream()), "multimap decode")
                return
            _req(parts is None, "parts: of the heads that a workgroup takes in pairs")
            n_splits = max(1, (bt.shape[1] * BS + split_keys - 1) // split_keys)
            if window or chunk:  # splits are counted from the window's (chunk's) first: it touches this many at most
                n_splits = min(n_splits, (keep + split_keys - 1) // split_keys + (max(window, chunk) + split_keys - 1) // split_keys + 1)
            ws = torch.empty(n_items * H * n_splits * (2 * maps + maps * vdim), dtype=torch.float32, device=q.device)
            _check(lib.bcg_multimap_attention(1, _p(q), _p(k_cache), _p(v_cache), _p(bt), bt.shape[1], None, _p(lens),
                                              _p(work), n_items, _p(out), _p(ws), n_splits, *common, 0, 0, 0, 0, None, _stream()), "multimap decode")

        if meta.decode:
            _req(T == bt.shape[0], "decode step: one row per sequence")
            decode(None, T)
            return out
        tiles, single = meta.tiles, meta.single
        _req(tiles is not None and tiles.dtype == torch.int32 and tiles.dim() == 2 and tiles.shape[1] == 3
             and tiles.is_contiguous() and meta.q_start.dtype == torch.int32, "prefill tiles int32 [n, 3]")
        if tiles.shape[0]:
            _check(lib.bcg_multimap_attention(0, _p(q), _p(k_cache), _p(v_cache), _p(bt), bt.shape[1], _p(meta.q_start),
                                              _p(lens), _p(tiles), tiles.shape[0], _p(out), None, 0, *common, 0, 0, 0, 0, None, _stream()),
                   "multimap prefill")
        if single is not None and single.shape[0]:
            _req(single.dtype == torch.int32 and single.dim() == 2 and single.shape[1] == 2 and single.is_contiguous(),
                 "single rows int32 [n, 2]")
            decode(single, single.shape[0])
        return out

    def moe_route(h, router_w, router_b, top, gate_w=None):
        T, W = h.shape
        E = router_w.shape[0]
        _req(h.is_contiguous() and router_w.dtype == torch.float32 and router_w.shape == (E, W) and router_w.is_contiguous()
             and (router_b is None or (router_b.dtype == torch.float32 and router_b.numel() == E))
             and 1 <= top <= E <= 256, "moe_route: fp32 router [E, W], E <= 256")
        idx = torch.empty(T, top, dtype=torch.int32, device=h.device)
        wts = torch.empty(T, top, dtype=torch.float32, device=h.device)
        gate = None
        if gate_w is not None:
            _req(gate_w.dtype == torch.float32 and gate_w.numel() == W and gate_w.is_contiguous(), "gate fp32 [W]")
            gate = torch.empty(T, dtype=torch.float32, device=h.device)
        _check(lib.bcg_moe_route(_p(h), _p(router_w), _p(router_b), _p(gate_w), _p(idx), _p(wts), _p(gate), T, W, E, top,
                                 _act(h), _stream()), "moe_route")
        return idx, wts, gate

    def moe_route_scored(h, router_w, corr, top, groups, keep, scale):
        T, W = h.shape
        E = router_w.shape[0]
        _req(h.is_contiguous() and router_w.dtype == torch.float32 and router_w.shape == (E, W) and router_w.is_contiguous()
             and (corr is None or (corr.dtype == torch.float32 and corr.numel() == E and corr.is_contiguous()))
             and 1 <= top <= E <= 256, "moe_route_scored: fp32 router [E, W], fp32 correction [E], E <= 256")
        _req(groups >= 1 and E % groups == 0 and 1 <= keep <= groups and top <= keep * (E // groups),
             "moe_route_scored: equal groups, `top` experts inside the kept groups")
        idx = torch.empty(T, top, dtype=torch.int32, device=h.device)
        wts = torch.empty(T, top, dtype=torch.float32, device=h.device)
        _check(lib.bcg_moe_route_scored(_p(h), _p(router_w), _p(corr), _p(idx), _p(wts), T, W, E, top, groups, keep,
                                        float(scale), _act(h), _stream()), "moe_route_scored")
        return idx, wts

    def moe_pair_rows(gate, up):
        """The [2 ff, W] weight of one gated expert as `moe_experts` (kinds "silu_gated", "clamped_glu") reads it:
        gate and up rows in alternating groups of 16 when ff is a multiple of 16 (the product's
        epilogue then forms the hidden values), else [gate; up]."""
        ff, W = gate.shape
        if ff % 16:
            return torch.cat([gate, up])
        return torch.stack([gate.reshape(ff // 16, 16, W), up.reshape(ff // 16, 16, W)], 1).reshape(2 * ff, W)

    def _wide_experts(n_slots, E, W, ff, kind, h, up, down):
        """Whether the products run on position tiles of 256 rows: from WIDE_SLOTS routed rows per expert on.  Two gated
        products of 8 experts, top 2, 64-row tiles -> 256-row tiles, us: width 2048, ff 2048: 32 rows per expert 71 -> 97,
        64: 89 -> 98, 256: 211 -> 103, 2046: 818 -> 424; width 4096, ff 3072: 32: 190 -> 192, 64: 294 -> 194, 256: 629 ->
        271, 2046: 2285 -> 1063 (1.16 PFLOP/s of 0.54)."""
        if h.dtype != torch.bfloat16 or W % 64 or ff % 64 or (kind in EXPERT_ACTS and ff % 128) or n_slots < WIDE_SLOTS * E:
            return False
        rows = n_slots + E * (WIDE_ROWS - 1) + 2 * WIDE_ROWS    # (with a tile to spare: the kernel's offsets are 32-bit)
        n_up = up.shape[1]
        return (2 * rows * max(W, n_up) < 1 << 31 and 2 * (max(W, n_up) + 256) * max(W, ff) < 1 << 31
                and all(t.data_ptr() % 16 == 0 for t in (h, up, down)))

    def _expert_products(h, up, down, idx, kind, limit, by_table=None):
        """Both products of the experts' rows: (y, pos), a slot's row at pos[slot], or at the slot where pos is None.  ``by_table``: (tokens,
        table) by which `idx` is filled first."""
        T, W = h.shape
        E, n_up, _ = up.shape
        top = idx.shape[1]
        gated = kind in EXPERT_ACTS
        ff = n_up // 2 if gated else n_up
        n_slots = T * top
        dev, f32 = h.device, _act(h)
        tokens, table = by_table or (None, None)
        route = (_p(tokens), _p(table), 0 if table is None else table.shape[0], 0 if table is None else table.stride(0), top)
        wide = _wide_experts(n_slots, E, W, ff, kind, h, up, down)
        held = 0
        if not wide and h.dtype == torch.bfloat16 and all(t.data_ptr() % 16 == 0 for t in (h, up, down)):
            held = few_row_tiles(n_slots, E, W, ff, few_rows)
        rows = WIDE_ROWS if wide else few_rows if held else tile_rows
        n_tiles = (n_slots + E * (rows - 1) + rows - 1) // rows
        cap = n_tiles * rows
        sorted_ = torch.empty(cap, dtype=torch.int32, device=dev)
        tile_e = torch.empty(n_tiles, dtype=torch.int32, device=dev)
        if wide:
            place = torch.empty(n_slots + 1, dtype=torch.int32, device=dev)   # every slot's position; the tiles in use
            pos, used = place[:n_slots], place[n_slots:]
            _check(lib.bcg_moe_align(_p(idx), n_slots, E, _p(sorted_), cap, _p(tile_e), n_tiles, rows, _p(pos), _p(used),
                                     *route, _stream()), "moe_align")
            hidden = torch.empty(cap, ff, dtype=h.dtype, device=dev)
            _check(lib.bcg_gemm_w4_grouped(3 if gated else 4, _p(h), _p(up), _p(hidden), _p(tile_e), _p(used), n_tiles, n_up, W,
                                           limit if kind == "clamped_glu" else 0.0, _p(sorted_), top, T, _stream()), "moe gate / up")
            y = torch.empty(cap, W, dtype=h.dtype, device=dev)
            _check(lib.bcg_gemm_w4_grouped(0, _p(hidden), _p(down), _p(y), _p(tile_e), _p(used), n_tiles, W, ff, 0.0, None, 1, 0,
                                           _stream()), "moe down")
            return y, pos
        _check(lib.bcg_moe_align(_p(idx), n_slots, E, _p(sorted_), cap, _p(tile_e), n_tiles, rows, None, None, *route,
                                 _stream()), "moe_align")
        if held:
            code = ACT_CODES[EXPERT_ACTS[kind]] if gated else 1
            used = (n_slots + min(E, n_slots) * (rows - 1)) // rows     # `align` packs the tiles in use at the front, this many at most
            hidden = torch.empty(cap, ff, dtype=h.dtype, device=dev)
            _check(lib.bcg_moe_rows(_p(h), T, W, _p(up), _p(hidden), ff, _p(sorted_), _p(tile_e), used, held, n_up, W, top, 1, 0,
                                    code, limit, _stream()), "moe up rows")
            y = torch.empty(n_slots, W, dtype=h.dtype, device=dev)
            _check(lib.bcg_moe_rows(_p(hidden), cap, ff, _p(down), _p(y), W, _p(sorted_), _p(tile_e), used, held, W, ff, top, 0, 1,
                                    0, 0.0, _stream()), "moe down rows")
            return y, None
        code = ACT_CODES[EXPERT_ACTS[kind]] if gated else 1
        if gated and ff % 16 == 0:   # rows paired by `moe_pair_rows`: the hidden values in the product's epilogue
            hidden = torch.empty(cap, ff, dtype=h.dtype, device=dev)
            _check(lib.bcg_moe_gemm(_p(h), W, _p(up), _p(hidden), ff, _p(sorted_), _p(tile_e), n_tiles, n_up, W, top, 1, 0, code,
                                    limit, f32, _stream()), "moe gate / up")
        elif gated:   # the stacked projection, then the hidden values from its halves
            both = torch.empty(cap, n_up, dtype=h.dtype, device=dev)
            _check(lib.bcg_moe_gemm(_p(h), W, _p(up), _p(both), n_up, _p(sorted_), _p(tile_e), n_tiles, n_up, W, top, 1, 0, 0,
                                    0.0, f32, _stream()), "moe gate / up")
            hidden = torch.empty(cap, ff, dtype=h.dtype, device=dev)
            _check(lib.bcg_gated_act(_p(both), _p(hidden), cap, ff, code, limit, f32, _stream()), "gated_act")
        else:
            hidden = torch.empty(cap, ff, dtype=h.dtype, device=dev)
            _check(lib.bcg_moe_gemm(_p(h), W, _p(up), _p(hidden), ff, _p(sorted_), _p(tile_e), n_tiles, ff, W, top, 1, 0, 1,
                                    0.0, f32, _stream()), "moe up")
        y = torch.empty(n_slots, W, dtype=h.dtype, device=dev)
        _check(lib.bcg_moe_gemm(_p(hidden), ff, _p(down), _p(y), W, _p(sorted_), _p(tile_e), n_tiles, W, ff, top, 0, 1, 0,
                                0.0, f32, _stream()), "moe down")
        return y, None

    def _check_experts(h, up, down, kind, limit):
        T, W = h.shape
        E, n_up, _ = up.shape
        _req(kind == "relu2" or kind in EXPERT_ACTS, "moe_experts: relu2, silu-gated or clamped gated experts")
        _req(kind != "clamped_glu" or limit > 0, "clamped experts: a positive limit")
        gated = kind in EXPERT_ACTS
        _req(not gated or n_up % 2 == 0, "gated experts: [gate; up] rows")
        ff = n_up // 2 if gated else n_up
        _req(h.is_contiguous() and up.shape == (E, n_up, W) and down.shape == (E, W, ff) and up.is_contiguous()
             and down.is_contiguous() and up.dtype == h.dtype and down.dtype == h.dtype, "expert weights [E, ff, W] / [E, W, ff]")

    def moe_experts(h, up, down, idx, weights, kind="relu2", limit=0.0):
        T, W = h.shape
        top = idx.shape[1]
        _check_experts(h, up, down, kind, limit)
        _req(idx.dtype == torch.int32 and idx.shape == (T, top) and idx.is_contiguous() and weights.dtype == torch.float32
             and weights.shape == (T, top) and weights.is_contiguous(), "routing tables [T, top]")
        if T * top == 0:
            return torch.zeros(T, W, dtype=torch.float32, device=h.device)
        y, pos = _expert_products(h, up, down, idx, kind, limit)
        out = torch.empty(T, W, dtype=torch.float32, device=h.device)
        _check(lib.bcg_moe_combine(_p(y), _p(weights), _p(pos), _p(idx), up.shape[0], _p(out), T, W, top, _act(h), _stream()), "moe_combine")
        return out

    return dict(embed_scale_rmsnorm=embed_scale_rmsnorm, embed_position=embed_position, residual_add_rmsnorm32=residual_add_rmsnorm32,
                rmsnorm32=rmsnorm32, act_fn=act_fn, rope_multi_kv_write=rope_multi_kv_write,
                kv_from_logical=kv_from_logical, kv_to_logical=kv_to_logical,
                multimap_attention=multimap_attention, multimap_tile_rows=multimap_tile_rows, moe_route=moe_route, moe_experts=moe_experts,
                _experts=(moe_experts, _check_experts, _expert_products),
                moe_pair_rows=moe_pair_rows, moe_route_scored=moe_route_scored)
