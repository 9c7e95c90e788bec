"""Host logic of the boundary: the Python twin of ``sparse_matmul`` in
``sparse/native/sparse_kernels.cc:7-50`` (layout pick, M/N/K rules, batch
flattening, output allocation, dtype dispatch) plus the argument checks the
reference does not make.  ``sparse_matmul`` keeps the reference's positional
signature (``native/sparse_ops.h:10-14``); the softmax entry points keep those of
``sparse_softmax.cu:208-210,233-236`` with ``scale`` / ``causal`` appended.
"""
import functools
import threading

import torch

from . import kernel as _k

BLOCK = 32
# tuning of the wavefront schedules: (target pairs per wavefront, wavefronts per workgroup)
# (cap, waves, split long groups, no row slicing, -, longest chunks first)
# Group walks (DSD, DDS).  A launch of few pairs is one generation of waves and lasts as long as its fullest SIMD: shorter chunks,
# spread over more of them.  Counted are the pairs of all batch entries and 64-column strips.  A table whose longest group fits
# the workgroup of a large launch is not cut by shorter chunks either (_group_walk_kinds): no launch needs a workspace that another
# batch count of the same layout does not need.  us, median of a graph of 20 launches, chunks of 12 -> now (fp16 DSD, longest row in
# brackets): 506 pairs (12) 6.6 -> 4.4, 628 (5) 4.8 -> 4.3, 2024 (12) 6.8 -> 4.6, 4048 (12) 7.0 -> 5.3, 6072 (12) 7.1 -> 6.8,
# 6120 (20) 6.9 -> 6.4, 9432 (12) 10.0 -> 8.4, 12144 (12) 13.0 -> 10.3, 12240 (20) 10.4 -> 8.7, 13344 (9) 11.8 -> 10.3; 16192 (12) would
# be 14.1 -> 13.9, 17792 (9) 12.7 -> 13.0.  Tables with longer groups gain little in fp16 (columns of 64, chunks of 10 against 4 and 6:
# 506 to 4048 pairs within 6 %, 8096 8.7 against 9.6 and 9.0, 12144 12.2 against 12.8 and 13.0; of 128: 6120 8.4 against 9.8 and 9.6).
SCHEDULE_GROUP_WALK = (4, 4, True, -1, 2, True)          # groups of at most GROUP_WALK_LONG pairs (rows of attention masks)
SCHEDULE_GROUP_WALK_MIDDLE = (6, 4, True, -1, 2, True)
SCHEDULE_GROUP_WALK_LARGE = (12, 4, True, -1, 2, True)
SCHEDULE_GROUP_WALK_LONG = (10, 4, True, -1, 2, True)    # tables with longer groups (columns of causal / strided masks)
GROUP_WALK_LONG = 24
GROUP_WALK_SMALL_PAIRS, GROUP_WALK_MIDDLE_PAIRS = 4096, 14000
SCHEDULE_SDD = (4, 2)
# SDD of few blocks (of all batch entries, times 64-value pieces of the inner dimension): more waves of two blocks each.  fp16, us,
# chunks of 4 -> 2: 506 blocks 3.5 -> 3.0, 2024 4.2 -> 3.7, 4048 4.5 -> 4.4, 6120 5.0 -> 4.9, 7084 5.9 -> 6.0; 8096 would be 5.6 -> 5.6,
# 12240 7.2 -> 7.3.  The same bits.
SCHEDULE_SDD_SMALL = (2, 2)
SDD_SMALL_BLOCKS = 8000
# fp32: a wave splits its row's operands into bf16 parts once, so chunks pay where the products are split: from as many blocks on as
# bsa_matmul splits them (SDD_F32_SPLIT_BLOCKS in csrc/matmul.hip, with both sides' times).  us, the fp32 instruction in chunks of 1
# in 4 waves -> split in chunks of 4 in 2, k = 64: 1012 blocks 6.2 -> 7.9, 2368 8.2 -> 8.8, 3552 10.3 -> 9.3, 8096 18.6 -> 15.0,
# 24480 46.5 -> 38, 73440 120 -> 98.
SCHEDULE_SDD_F32 = (1, 4)
SCHEDULE_SDD_F32_LARGE = (4, 2)
SDD_F32_LARGE_BLOCKS = 3000            # of all batch entries together, at k = 64 and more
# fp32: a pair keeps its SIMD's matrix pipe for 2048 clocks, so the chunks of the fullest SIMD are the launch.  us, chunks of 6 (10
# in tables with longer groups) -> now.  Rows of up to 12: 506 pairs 11.0 -> 7.4, 2024 11.2 -> 7.8, 4048 11.6 -> 10.9, 8096 19.6 -> 18.3,
# 10120 24.9 -> 21.2; of 5: 628 10.0 -> 7.4, 5024 13.8 -> 14.2; of 20 (chunks of 5 hold them): 6120 18.9 -> 16.3, 9180 23.3 -> 21.9.
# Columns of 64: 506 17.1 -> 10.4, 2024 17.6 -> 11.0, 4048 18.0 -> 13.2, 8096 24.4 -> 20.9, 10120 25.8 -> 22.1; of 128: 6120 21.4 -> 17.9,
# 9180 28.2 -> 22.5.  The line at 11000 lies where chunks of 4 stop being ahead for rows: 12144 pairs would be 25.4 -> 25.6 (12), 12240
# 24.3 -> 23.3 (20); for columns they still would be at some sizes: 12144 28.7 -> 26.7 and 14674 34.7 -> 31.0 (64), 12240 26.1 -> 26.4 (128).
SCHEDULE_GROUP_WALK_F32 = (3, 4, True, -1, 2, True)
SCHEDULE_GROUP_WALK_F32_MIDDLE = (4, 4, True, -1, 2, True)
SCHEDULE_GROUP_WALK_F32_LARGE = (6, 4, True, -1, 2, True)      # 73440 pairs, chunks of 12 -> 6: 114 -> 114
GROUP_WALK_F32_MIDDLE_PAIRS = 11000
SCHEDULE_SOFTMAX = (4, 4)
SOFTMAX_LONGEST_FIRST = True     # long rows are dispatched first: they would otherwise finish on a draining machine
SOFTMAX_WAVES_LONG_ROWS = 8
SCHEDULE_BLOCK64 = (4, 2, False)        # coarse pairs (64x64 blocks = four tiles) per wavefront; never split
# DSD on a block=64 layout: True takes the kernel whose wavefronts own whole 64x64 blocks, False walks the layout's
# 32x32 tiles.  Measured at 4096 tokens, 16 heads, 399 blocks of 64 (bench.py, rows block64_mask_*): 17.9-18.8 us
# against 17.1-18.4 us for the group walk over the tiles and 16.5 us for the run walk over them; a wavefront that
# holds a 64 x 64 fp32 tile needs 227 registers (two waves per SIMD), so the tile walks stay the default.
USE_BLOCK64_KERNEL = False
# DSD over a row table with the dense operand stored [K][N]: runs of consecutive block rows whose dense strips stay
# in LDS (bsa_matmul_dsd_runs), when the table is eligible, a fetched strip serves at least RUN_WALK_MIN_REUSE pairs
# and the launch is large enough to give every compute unit a run of RUN_WALK_PAIRS_MIN pairs.  A run is one
# workgroup with a compute unit to itself; the launch is cut into a whole number of generations of about
# RUN_WALK_PAIRS pairs per run (workgroups a few above a multiple of the compute units would cost a generation of
# their own).  Measured at 4096 tokens (1530 blocks per head), DSD fp16, against the walk of bsa_matmul:
# 10.2 / 10.8 / 16.1 / 24.3 / 29.4 / 42.0 us against 12.3 / 12.9 / 16.9 / 26.1 / 33.5 / 44.8 us at
# 4 / 8 / 16 / 24 / 32 / 48 heads.
RUN_WALK = True
RUN_WALK_WAVES = 8
RUN_WALK_PAIRS = 96
RUN_WALK_PAIRS_MIN = 48
RUN_WALK_STRIPS = 32             # 4 per wave; with 10 waves and up to 39 strips (rows of 33-39 blocks) the walk of
                                 # bsa_matmul is 3-6 % faster at 8192 tokens
RUN_WALK_MIN_REUSE = 2.0
# DDS over many dense rows (a block-sparse linear layer): panels of the dense operand shared by eight groups
# (bsa_matmul_dds_panels), when the mask is dense enough that a panel serves several of them and the launch has
# workgroups for most of the machine, both reckoned in tiles of PANEL_ROWS rows.  bf16, us, group walk -> panels: 0.1 of 64 x 64
# blocks, 4 x 1056 rows 31.8 -> 19.2, with a full column 34.6 -> 21.5; 0.12 of 96 x 96, 8 x 1024 rows 112 -> 64.5 and 127 -> 68.6;
# 0.25 of 64 x 64, 1920 rows (160 tiles) 28.9 -> 12.9 and 32.2 -> 16.2.  At the lines the panels are well ahead, and they stay ahead
# for some way below them (1056 rows, 88 tiles 18.3 -> 11.7 and 19.6 -> 14.8; 0.1 at 1344 rows, 112 tiles 12.8 -> 9.5 and 13.7 -> 13.7).
PANEL_WALK = True
PANEL_ROWS, PANEL_MAX_KBLOCKS, PANEL_MAX_NNZ = _k.dds_panel_limits()      # of a workgroup, of a launch
PANEL_GROUPS = 8                       # of a workgroup
PANEL_MIN_WORKGROUPS = 160
PANEL_MIN_DENSITY = 0.08
# Its weight gradient (bsa_weight_grad) against a stack per batch entry and a sum over them, us: 0.09 stored (96 x 96 blocks, 8192
# tokens) 81 -> 87, 0.13 121 -> 94, 0.19 196 -> 107; 0.11 (64 x 64, 4224 tokens) 63 -> 27, 0.26 67 -> 36; 0.2, 1056 tokens
# 60 -> 23; 0.3 (16 x 16), 256 tokens 12 -> 16.
WEIGHT_GRAD_MIN_TOKENS = 1024
WEIGHT_GRAD_MIN_DENSITY = 0.10
ATTENTION_WAVES_LONG_GROUPS = 8
ATTENTION_COLUMN_WAVES_128 = 4    # waves of a workgroup the column walk takes at head dim 128
ATTENTION_SPLIT_ROWS = True       # groups longer than cap * waves are cut into parts across workgroups
SCHEDULE_ATTENTION = (12, 4)           # forward: rows of more than 48 blocks are split across workgroups
SCHEDULE_ATTENTION_BACKWARD = (12, 4)
SCHEDULE_ATTENTION_BACKWARD_COLUMNS = (12, 2)
# A launch of few blocks is one generation of waves and lasts as long as its longest chunk: shorter chunks.  Measured,
# causal local-4 + stride-8 mask of 4096 tokens, head dim 64, chunks of 12 -> 6 (forward, rows, columns): 1 batch entry
# (1530 blocks) 10.6 / 12.8 / 18.2 -> 8.1 / 10.0 / 16.2 us; 4 entries (6120) 11.6 / 13.8 / 18.3 -> 10.7 / 13.2 / 17.8; 8
# entries of a random mask (13100) 15.2 / 18.0 / 19.5 -> 15.8 / 20.5 / 22.1.
# The workgroup's share (cap * waves) stays what it is for a large launch wherever a group is longer than 24 blocks
# (_attention_kinds): no launch needs a workspace that another batch count of the same layout does not need.  Chunks of 6
# in 4 and in 8 waves, one entry, forward / backward: causal local-4 + stride-8 of 8192 tokens (rows of up to 36) 9.5 / 30.0 ->
# 8.7 / 30.1 us, a quarter of 128 x 128 blocks (44) 10.8 / 21.9 -> 10.5 / 22.0, at head dim 128 14.5 / 35.3 -> 15.4 / 37.5.
SCHEDULE_ATTENTION_SMALL = (6, 4)
ATTENTION_SMALL_BLOCKS = 8192          # blocks of all batch entries together
# block rows of at most this many blocks are handed whole to SOFTMAX_SLICES wavefronts (8 element rows
# each), which keep them in registers and need no exchange; per dtype: forward, backward (the
# backward walk keeps two inputs)
SOFTMAX_SLICE_MAX = {torch.float16: (48, 24), torch.bfloat16: (48, 24), torch.float32: (24, 24)}
SOFTMAX_SLICES = {torch.float16: (4, 4), torch.bfloat16: (4, 4), torch.float32: (4, 8)}      # forward, backward

_DTYPES = {torch.float32: _k.BSA_F32, torch.float16: _k.BSA_F16, torch.bfloat16: _k.BSA_BF16}


class Schedule:
    """Device-resident wavefront schedule of one offset table."""

    def __init__(self, offsets: torch.Tensor, nnz: int, cap: int, waves: int, allow_split: bool = True,
                 slice_max: int = -1, slices: int = 2, longest_first: bool = False):
        groups = offsets.numel() - 1
        capacity = _k.lib.bsa_schedule_capacity(groups, nnz, cap, waves)
        self.table = torch.empty(4 * capacity, dtype=torch.int32, device=offsets.device)
        counts = torch.empty(4, dtype=torch.int32, device=offsets.device)
        with _k.on_device(offsets.device):
            _k.check(_k.lib.bsa_schedule_build(offsets.data_ptr(), groups, cap, waves,
                                               int(bool(allow_split)) | (2 if longest_first else 0), slice_max,
                                               slices, self.table.data_ptr(), capacity, counts.data_ptr(),
                                               _k.current_stream()))
        self.workgroups, self.tile_slots, self.split_groups, self.slots = (int(v) for v in counts.tolist())
        if self.workgroups < 0:
            raise _k.BsaError("schedule table too small for this offset table")
        self.groups = groups
        self.waves = waves
        self.cap = cap
        self._workspaces = {}
        self._captured = {}
        self._spares = {}
        self._spaces = {}

    def __getstate__(self):
        """A copy (of the layout) has no launches, graphs and plans yet: it gets the spares, which are always zero."""
        with self._lock:
            return {**self.__dict__, "_workspaces": {}, "_captured": {}, "_spaces": {},
                    "_spares": {key: list(spares) for key, spares in self._spares.items()}}

    def workspace(self, mode: int, batches: int, size_m: int, size_n: int, stream: int):
        """Zeroed scratch for split groups, one per (shape, stream): launches on one stream run in
        order and each leaves the buffer zero again; launches on different streams may overlap.
        Returns the buffer, its bytes and the key it is kept under (``None, 0, None`` where nothing is needed)."""
        if self.tile_slots == 0:
            return None, 0, None
        need = _k.lib.bsa_matmul_workspace_bytes(mode, self.tile_slots, self.split_groups, batches, size_m, size_n)
        return self._kept((mode, batches, size_m, size_n, stream), need)

    def attention_workspace(self, batches: int, head_dim: int, stream: int):
        """The same for the split rows of the fused attention forward."""
        if self.tile_slots == 0:
            return None, 0, None
        need = _k.lib.bsa_attention_workspace_bytes(self.tile_slots, self.split_groups, batches, head_dim)
        return self._kept(("attention", batches, head_dim, stream), need)

    def attention_backward_workspace(self, columns, batches: int, head_dim: int, stream: int):
        """The same for the backward walks: this schedule walks the rows, ``columns`` (or None) the columns."""
        ct, cg = (columns.tile_slots, columns.split_groups) if columns is not None else (0, 0)
        need = _k.lib.bsa_attention_backward_workspace_bytes(self.tile_slots, self.split_groups, ct, cg, batches,
                                                             head_dim)
        return self._kept(("attention_backward", ct, cg, batches, head_dim, stream), need)

    def _kept(self, key, need):
        ws, need = self._zeroed(key, need)
        return ws, need, key if ws is not None else None

    def has_workspace(self, key):
        """Whether a launch that is being captured can be given the workspace of ``key`` (its last item is the stream): one
        that the stream has, or a spare.  What a graph of another stream has is that graph's."""
        with self._lock:
            return key in self._captured or key in self._workspaces or bool(self._spares.get(key[:-1]))

    _spaces = {}             # of a schedule that no plan launches by
    _lock = threading.RLock()          # of what the schedules keep; none of the schedule's own, which is copied with its layout
    MAX_WORKSPACES = 16      # eager ones per schedule; the least recently used one goes first

    def _zeroed(self, key, need):
        """Workspace of ``need`` zero bytes for ``key`` (its last item is the stream).  A buffer must be
        zero before its first launch, and under graph capture nothing can be zeroed (a fill recorded
        there only runs at replay, possibly after another graph has used the buffer): every eager call
        keeps one zeroed spare per shape ready, which a first use under capture takes.

        A buffer handed out under capture is never dropped: the captured graph holds its raw address and
        may be replayed at any time.  An eager one is dropped only after the stream it was used on has
        drained (a launch still in flight parks partial tiles there).

        Plans launch with an eager workspace without coming here (``plan_space``); they lose it, and the next call
        comes here again, where it is dropped and where a capture took the shape's spare."""
        if need == 0:
            return None, 0
        gone = []
        with self._lock:
            ws = self._hand_out(key, need, gone)
        for stream, _ in gone:
            self._drain(stream)
        return ws, need

    def _hand_out(self, key, need, gone):
        """``_zeroed`` under the lock: filling a buffer lets other threads in.  What is dropped goes to ``gone``, with its stream."""
        capturing = torch.cuda.is_current_stream_capturing()
        spares = self._spares.setdefault(key[:-1], [])
        ws = self._captured.get(key)
        if ws is not None:                              # the graph that owns it is being extended or re-captured
            if not capturing and not spares:
                spares.append(torch.zeros(need, dtype=torch.uint8, device=self.table.device))
            return ws
        ws = self._workspaces.pop(key, None)
        if ws is None:
            if capturing:
                if not spares:
                    raise RuntimeError("this operator and shape has never run outside graph capture: call it once "
                                       "eagerly before capturing (its workspace must be zeroed first)")
                ws = spares.pop()
                for other in [k for k in self._spaces if k[:-1] == key[:-1]]:
                    self._forget_plans(other)           # one of their calls puts a spare back
            else:
                ws = torch.zeros(need, dtype=torch.uint8, device=self.table.device)
        if not capturing and not spares:
            spares.append(torch.zeros(need, dtype=torch.uint8, device=self.table.device))
        if capturing:
            self._captured[key] = ws
            return ws
        self._workspaces[key] = ws                      # most recently used last
        while len(self._workspaces) > self.MAX_WORKSPACES:
            old_key = next(iter(self._workspaces))
            self._forget_plans(old_key)
            gone.append((old_key[-1], self._workspaces.pop(old_key)))
        return ws

    def _drain(self, stream_handle):
        """Waits for the stream a workspace was used on before the workspace is given back to the allocator."""
        torch.cuda.ExternalStream(stream_handle, device=self.table.device).synchronize()

    def plan_space(self, key, ws):
        """What the plans that launch with the workspace ``ws`` of ``key`` share, and lose together."""
        with self._lock:
            if key not in self._spaces:
                self._spaces[key] = _k.host_calls.new_space(ws)
            return self._spaces[key]

    def _forget_plans(self, key):
        space = self._spaces.pop(key, None)
        if space is not None:
            _k.host_calls.drop_space(space)

    def discard(self, key):
        """Forget the workspace of ``key``: a launch that failed may have left its counters non-zero."""
        with self._lock:
            self._forget_plans(key)
            self._workspaces.pop(key, None)
            self._captured.pop(key, None)


class RunSchedule:
    """Runs of consecutive block rows of a row table (bsa_run_schedule_build)."""

    def __init__(self, blocks: torch.Tensor, offsets: torch.Tensor, target_pairs: int, max_strips: int):
        rows, nnz = offsets.numel() - 1, blocks.numel() // 2
        need = _k.lib.bsa_run_schedule_bytes(rows, nnz)
        self.table = torch.empty(need, dtype=torch.uint8, device=offsets.device)
        counts = torch.empty(4, dtype=torch.int32, device=offsets.device)
        with _k.on_device(offsets.device):
            _k.check(_k.lib.bsa_run_schedule_build(blocks.data_ptr(), offsets.data_ptr(), rows, nnz, target_pairs,
                                                   max_strips, self.table.data_ptr(), need, counts.data_ptr(),
                                                   _k.current_stream()))
        self.runs, self.strips, self.strips_total, self.pairs = (int(v) for v in counts.tolist())
        self.reuse = nnz / self.strips_total if self.strips_total else 0.0


@functools.lru_cache(maxsize=None)
def _compute_units(device_index: int) -> int:
    return torch.cuda.get_device_properties(device_index).multi_processor_count


def _run_schedule(layout, batches, strips_n):
    """Run schedule of a row table for a launch of ``batches`` x ``strips_n`` (64-column strips of the result)
    entries, or None when the table is not eligible, the launch is too small to fill the machine with runs, or
    its rows share too few columns for resident strips to pay."""
    blocks, offsets = layout
    nnz = blocks.numel() // 2
    entries = batches * strips_n
    cus = _compute_units(offsets.device.index)
    if nnz * entries < cus * RUN_WALK_PAIRS_MIN:
        return None
    generations = max(1, round(nnz * entries / (cus * RUN_WALK_PAIRS)))
    runs_wanted = max(1, cus * generations // entries)
    cache = getattr(offsets, "_bsa_runs", None)
    if cache is None:
        cache = {}
        offsets._bsa_runs = cache
    if runs_wanted not in cache:
        if torch.cuda.is_current_stream_capturing():
            return None                     # building synchronises: the first call for a shape runs eagerly
        target = max(RUN_WALK_PAIRS_MIN, -(-nnz // runs_wanted))
        for _ in range(4):                  # a cut forced by the strips can leave one run too many: aim higher
            rs = RunSchedule(blocks, offsets, target, RUN_WALK_STRIPS)
            if rs.runs <= runs_wanted:
                break
            target = -(-target * 11 // 10)
        cache[runs_wanted] = rs
    rs = cache[runs_wanted]
    if rs.runs == 0 or rs.reuse < RUN_WALK_MIN_REUSE:
        return None
    rs.waves = RUN_WALK_WAVES
    return rs if rs.strips <= 4 * rs.waves and rs.pairs <= 64 * rs.waves else None


def _launch(sched, key, status):
    """Raise on a failed C-ABI call; the workspace the call was given, ``key`` (or None), is dropped first, because a launch
    that failed midway may have left its counters non-zero and every later call would sum stale parts."""
    if status != 0 and key is not None:
        sched.discard(key)
    _k.check(status)


def schedule_for(layout, kind):
    """Schedule of a ``(blocks, offset_table)`` tuple, built on first use and kept
    on the offset tensor (the reference's boundary passes only the two tensors)."""
    blocks, offsets = layout
    cache = getattr(offsets, "_bsa_schedules", None)
    if cache is None:
        cache = {}
        offsets._bsa_schedules = cache
    if kind not in cache:
        cache[kind] = Schedule(offsets, blocks.numel() // 2, *kind)
    return cache[kind]


def _has_schedule(layout, kind) -> bool:
    """Whether ``schedule_for(layout, kind)`` has nothing to build."""
    return kind in getattr(layout[1], "_bsa_schedules", ())


def _longest_group(offsets) -> int:
    """Pairs in the longest group of a table; measured once and kept on the offsets tensor."""
    longest = getattr(offsets, "_bsa_longest", None)
    if longest is None:
        longest = int((offsets[1:] - offsets[:-1]).max().item()) if offsets.numel() > 1 else 0
        offsets._bsa_longest = longest
    return longest


def _group_walk_kinds(longest, dtype, pairs, of_others=True):
    """Schedules of a group walk over ``pairs`` pairs of all batch entries and strips: the one it takes, then what else serves
    where that one cannot be built (the others of this type; with ``of_others`` also what calls of another type have built)."""
    short = longest <= GROUP_WALK_LONG
    large = SCHEDULE_GROUP_WALK_LARGE if short else SCHEDULE_GROUP_WALK_LONG
    half = [SCHEDULE_GROUP_WALK, SCHEDULE_GROUP_WALK_MIDDLE, large] if short else [large]
    single = [SCHEDULE_GROUP_WALK_F32, SCHEDULE_GROUP_WALK_F32_MIDDLE, SCHEDULE_GROUP_WALK_F32_LARGE if short else large]
    if dtype == torch.float32:
        kinds, others, lines = single, half, (GROUP_WALK_SMALL_PAIRS, GROUP_WALK_F32_MIDDLE_PAIRS)
    else:
        kinds, others, lines = half, single, (GROUP_WALK_SMALL_PAIRS, GROUP_WALK_MIDDLE_PAIRS) if short else ()
    first = kinds[sum(pairs > line for line in lines)]

    def whole(kind):                # chunks that cut no group which the largest launches leave whole
        cap, waves = kind[:2]
        return (max(cap, -(-longest // waves)),) + kind[1:] if longest <= large[0] * large[1] else kind

    return tuple(dict.fromkeys(whole(kind) for kind in [first] + kinds + (others if of_others else [])))


def _group_walk_schedule(layout, dtype=torch.float16, entries=None, key=None):
    """Schedule of a group walk over ``entries`` batch entries times strips (None: as many as fill the machine).  Under graph
    capture the first that is there and has the launch's workspace, ``key`` (without its stream)."""
    pairs = layout[0].numel() // 2 * entries if entries is not None else 2 ** 62
    kinds = _group_walk_kinds(_longest_group(layout[1]), dtype, pairs)
    if torch.cuda.is_current_stream_capturing():
        there = [layout[1]._bsa_schedules[kind] for kind in kinds if _has_schedule(layout, kind)]
        with _k.on_device(layout[1].device):
            stream = _k.current_stream()
        for sched in there:
            if sched.tile_slots == 0 or key is None or sched.has_workspace(key + (stream,)):
                return sched
        if there:
            return there[0]
    return schedule_for(layout, kinds[0])


def _sdd_schedule(layout, dtype, batches, k):
    if dtype != torch.float32:
        small = layout[0].numel() // 2 * batches * -(-k // 64) <= SDD_SMALL_BLOCKS
        kinds = (SCHEDULE_SDD_SMALL, SCHEDULE_SDD) if small else (SCHEDULE_SDD, SCHEDULE_SDD_SMALL)
        return _schedule_or(layout, *kinds, SCHEDULE_SDD_F32)
    if layout[0].numel() // 2 * batches * min(k, 64) >= 64 * SDD_F32_LARGE_BLOCKS:
        return _schedule_or(layout, SCHEDULE_SDD_F32_LARGE, SCHEDULE_SDD_F32, SCHEDULE_SDD_SMALL)
    return _schedule_or(layout, SCHEDULE_SDD_F32, SCHEDULE_SDD_F32_LARGE, SCHEDULE_SDD_SMALL)


def _schedule_or(layout, kind, *others):
    """The schedule ``kind``, or, where a graph is being captured and it is not there, the first of ``others`` that is (they may
    be what calls of another type have built): building synchronises."""
    there = getattr(layout[1], "_bsa_schedules", ())
    if kind in there:
        return there[kind]
    if torch.cuda.is_current_stream_capturing():
        kind = next((other for other in others if other in there), kind)
    return schedule_for(layout, kind)


def _captured_without(layout, kind) -> bool:
    """Whether a graph is being captured and the schedule ``kind`` of the table (None: of its 16-bit group walk) is not there:
    building one synchronises.  Calls that used a walk without a schedule eagerly stay with it then."""
    if kind is None:
        longest = getattr(layout[1], "_bsa_longest", None)
        kinds = () if longest is None else _group_walk_kinds(longest, torch.float16, 0, of_others=False)
    else:
        kinds = (SCHEDULE_SDD, SCHEDULE_SDD_SMALL) if kind == SCHEDULE_SDD else (kind,)
    return not any(_has_schedule(layout, k) for k in kinds) and torch.cuda.is_current_stream_capturing()


def _attention_kind(layout, kind, split, most_waves=ATTENTION_WAVES_LONG_GROUPS):
    """Arguments of the schedule of a fused attention walk.  With ``split`` (what every caller passes while
    ``ATTENTION_SPLIT_ROWS`` is set) a group longer than the workgroup's share is cut into parts that
    meet in a workspace; without it such a table gets the most waves a workgroup holds instead."""
    cap, waves = kind
    if not split and _longest_group(layout[1]) > cap * waves:
        waves = most_waves
    return cap, waves, bool(split)


def _attention_schedule(layout, kind, split=False, most_waves=ATTENTION_WAVES_LONG_GROUPS):
    return schedule_for(layout, _attention_kind(layout, kind, split, most_waves))


def _attention_kinds(layout, kind, few_blocks):
    """Schedules to consider for a launch, in this order: the first that cuts no group into parts, else the last."""
    if not few_blocks:
        return (kind,)
    cap, waves = SCHEDULE_ATTENTION_SMALL
    same_share = cap, kind[0] * kind[1] // cap
    some_group_is_longer = layout[0].numel() // 2 > cap * waves * (layout[1].numel() - 1)      # longer than the average
    return (same_share,) if some_group_is_longer else (SCHEDULE_ATTENTION_SMALL, same_share)


def _attention_schedule_for(layout, kind, batches, most_waves=ATTENTION_WAVES_LONG_GROUPS):
    """Schedule of a fused attention walk over ``batches`` entries: ``kind``, or shorter chunks for a small launch.  Nothing
    can be built under graph capture: there the other length serves when only that one has been used eagerly."""
    few = layout[0].numel() // 2 * batches <= ATTENTION_SMALL_BLOCKS
    chosen = getattr(layout[1], "_bsa_attention", None)
    if chosen is None:
        chosen = layout[1]._bsa_attention = {}
    key = (kind, few, ATTENTION_SPLIT_ROWS, most_waves)
    if key in chosen:
        return chosen[key]
    for few_blocks in (few, not few):
        kinds = _attention_kinds(layout, kind, few_blocks)
        for k in kinds:
            if not _has_schedule(layout, _attention_kind(layout, k, ATTENTION_SPLIT_ROWS, most_waves)) \
                    and torch.cuda.is_current_stream_capturing():
                break
            sched = _attention_schedule(layout, k, ATTENTION_SPLIT_ROWS, most_waves)
            if sched.split_groups == 0 or k == kinds[-1]:
                if few_blocks == few:
                    chosen[key] = sched
                return sched
    raise RuntimeError("fused attention has never run on this layout outside graph capture: call it once eagerly before "
                       "capturing (building its schedule synchronises)")


def _softmax_schedule(layout, dtype, backward):
    cap, waves = SCHEDULE_SOFTMAX
    which = 1 if backward else 0
    slice_max, slices = SOFTMAX_SLICE_MAX[dtype][which], SOFTMAX_SLICES[dtype][which]
    if _longest_group(layout[1]) > slice_max:
        # a row too long for the register-resident walk is streamed by the waves of ONE workgroup (a row
        # cannot be split across workgroups): as many waves as a workgroup holds keep its chunks short
        waves = SOFTMAX_WAVES_LONG_ROWS
    waves = max(waves, slices)          # the slices of a row share a workgroup
    return schedule_for(layout, (cap, waves, False, slice_max, slices, SOFTMAX_LONGEST_FIRST))


def _is_table(t):
    return (isinstance(t, torch.Tensor) and t.dtype == torch.int32 and t.is_cuda and t.dim() == 1
            and t.is_contiguous())


def _check_layout(layout, name):
    blocks, offsets = layout
    if not (_is_table(blocks) and _is_table(offsets)):
        what = "offset_table" if _is_table(blocks) else "blocks"
        raise ValueError(f"{name}.{what} must be a contiguous 1-D int32 tensor on the GPU")
    if blocks.numel() % 2 or offsets.numel() < 2:
        raise ValueError(f"{name} is malformed")


def _matmul_route(a, b, mode, row_layout, col_layout, trans_a, trans_b):
    """Checks a product and says how it goes: (walk, its schedule, the table it walks, contiguous operands, shape of the
    result, whether the batch shares the sparse operand, batch entries, M, N, K)."""
    if mode not in _k.MODES:
        raise ValueError(f"mode must be one of 'sdd', 'dsd', 'dds', got {mode!r}")
    if a.dtype != b.dtype or a.dtype not in _DTYPES:
        raise TypeError(f"operands must both be float32, float16 or bfloat16, got {a.dtype} and {b.dtype}")
    if not (a.is_cuda and b.is_cuda) or a.device != b.device:
        raise ValueError("operands must live on the same GPU")
    _check_layout(row_layout, "row_layout")
    _check_layout(col_layout, "col_layout")
    trans_a, trans_b = bool(trans_a), bool(trans_b)

    # sparse_kernels.cc:12 : which table the walk uses
    use_row = mode == "sdd" or (mode == "dsd" and not trans_a) or (mode == "dds" and trans_b)
    layout = row_layout if use_row else col_layout
    if layout[0].device != a.device:
        raise ValueError("layout tables and operands must live on the same GPU")
    num_blocks = layout[0].numel() // 2
    mask_rows, mask_cols = row_layout[1].numel() - 1, col_layout[1].numel() - 1
    sparse_width = (layout[1].numel() - 1) * BLOCK                      # :14

    a_dense, b_dense = mode[1] == "d", mode[2] == "d"
    # a sparse INPUT without batch dimensions is shared by every batch entry of the dense operand
    shared = (not a_dense and a.dim() == 3) or (not b_dense and b.dim() == 3)
    if (a_dense and a.dim() < 3) or (b_dense and b.dim() < 3) or (not a_dense and a.dim() < 3) \
            or (not b_dense and b.dim() < 3):
        raise ValueError("operands need at least one batch dimension "
                         "(dense [..., rows, cols], sparse [..., nnz, 32, 32]; a sparse input may "
                         "also be [nnz, 32, 32], shared by the whole batch)")
    for t, dense, name in ((a, a_dense, "a"), (b, b_dense, "b")):
        if not dense and tuple(t.shape[-3:]) != (num_blocks, BLOCK, BLOCK):
            raise ValueError(f"sparse operand {name} must be [..., {num_blocks}, 32, 32], got {tuple(t.shape)}")

    # sparse_kernels.cc:17-19
    size_m = a.size(-1 if trans_a else -2) if a_dense else sparse_width
    size_n = b.size(-2 if trans_b else -1) if b_dense else sparse_width
    size_k = b.size(-1 if trans_b else -2) if b_dense else a.size(-2 if trans_a else -1)
    if a_dense and b_dense and a.size(-2 if trans_a else -1) != size_k:
        raise ValueError("inner dimensions of op(a) and op(b) differ")

    batch_a = tuple(a.shape[:-2] if a_dense else a.shape[:-3])
    batch_b = tuple(b.shape[:-2] if b_dense else b.shape[:-3])
    if shared:
        batch_a = batch_b = batch_a if a_dense else batch_b
    if batch_a != batch_b:
        raise ValueError(f"batch dimensions differ: {batch_a} vs {batch_b} (only a sparse input without "
                         f"batch dimensions is broadcast)")
    batches = 1
    for s in batch_a:
        batches *= s
    if batches < 1:
        raise ValueError("empty batch")

    # :22-37 : flatten the batch, allocate the result
    a = a.contiguous()
    b = b.contiguous()
    if mode[0] == "d":
        shape = batch_a + (size_m, size_n)
    else:
        shape = batch_a + (num_blocks, BLOCK, BLOCK)
    def route(walk, sched=None):
        return walk, sched, layout, a, b, shape, shared, batches, size_m, size_n, size_k

    coarse = getattr(row_layout[1], "_bsa_coarse", None)
    if (USE_BLOCK64_KERNEL and coarse is not None and mode == "dsd" and not trans_a and not trans_b
            and a.dtype != torch.float32 and size_n % 64 == 0 and num_blocks > 0):
        return route("block64", schedule_for(coarse[0], SCHEDULE_BLOCK64))

    if (RUN_WALK and mode == "dsd" and not trans_a and not trans_b and a.dtype != torch.float32
            and size_n % 64 == 0):
        runs = _run_schedule(layout, batches, size_n // 64)
        if runs is not None:
            return route("runs", runs)

    if (PANEL_WALK and mode == "dds" and not trans_a and a.dtype != torch.float32
            and size_m % BLOCK == 0 and size_k == BLOCK * (mask_cols if trans_b else mask_rows)
            and a.data_ptr() % 16 == 0 and b.data_ptr() % 16 == 0
            and _takes_panels(num_blocks, size_m * batches if shared else size_m, 1 if shared else batches,
                              size_k // BLOCK, size_n // BLOCK, lambda: _captured_without(layout, None))):
        return route("panels")

    if mode == "sdd":
        return route("walk", _sdd_schedule(layout, a.dtype, batches, size_k))
    strips = -(-(size_n if mode == "dsd" else size_m) // 64)
    return route("walk", _group_walk_schedule(layout, a.dtype, batches * strips, (_k.MODES[mode], batches, size_m, size_n)))


def sparse_matmul(a, b, mode, row_layout, col_layout, trans_a=False, trans_b=False):
    """``c = op(a) @ op(b)`` with one of a, b, c block-sparse (sparse_kernels.cc:7-50)."""
    walk, sched, layout, a, b, shape, shared, batches, size_m, size_n, size_k = _matmul_route(
        a, b, mode, row_layout, col_layout, trans_a, trans_b)
    c = torch.empty(shape, dtype=a.dtype, device=a.device)
    dtype, num_blocks, sparse_batches = _DTYPES[a.dtype], layout[0].numel() // 2, 1 if shared else batches
    mask_rows, mask_cols = row_layout[1].numel() - 1, col_layout[1].numel() - 1
    with _k.on_device(a.device):
        stream = _k.current_stream()
        if walk == "block64":
            (cblocks, coffsets), crows, ccols = row_layout[1]._bsa_coarse
            _k.check(_k.lib.bsa_matmul_dsd_block64(
                dtype, a.data_ptr(), b.data_ptr(), c.data_ptr(), cblocks.data_ptr(), coffsets.data_ptr(),
                sched.table.data_ptr(), sched.workgroups, sched.waves, crows, ccols, cblocks.numel() // 2, batches,
                sparse_batches, size_n, stream))
        elif walk == "runs":
            _k.check(_k.lib.bsa_matmul_dsd_runs(
                dtype, a.data_ptr(), b.data_ptr(), c.data_ptr(), layout[0].data_ptr(), layout[1].data_ptr(),
                sched.table.data_ptr(), sched.runs, sched.strips, sched.pairs, sched.waves, mask_rows, mask_cols, num_blocks,
                batches, sparse_batches, size_n, stream))
        elif walk == "panels":
            _k.check(_k.lib.bsa_matmul_dds_panels(
                dtype, a.data_ptr(), b.data_ptr(), c.data_ptr(), layout[0].data_ptr(), layout[1].data_ptr(),
                mask_rows, mask_cols, num_blocks, batches, sparse_batches, size_m, int(bool(trans_b)), stream))
        else:
            ws, ws_bytes, key = sched.workspace(_k.MODES[mode], batches, size_m, size_n, stream)
            _launch(sched, key, _k.lib.bsa_matmul(
                _k.MODES[mode], dtype, a.data_ptr(), b.data_ptr(), c.data_ptr(),
                layout[0].data_ptr(), layout[1].data_ptr(), layout[1].numel() - 1,
                sched.table.data_ptr(), sched.workgroups, sched.waves, sched.tile_slots, sched.split_groups,
                ws.data_ptr() if ws is not None else None, ws_bytes,
                mask_rows, mask_cols, num_blocks, batches, sparse_batches, size_m, size_n, size_k,
                int(bool(trans_a)), int(bool(trans_b)), stream))
    return c


def _takes_panels(nnz, rows, entries, kblocks, groups, without_choice=lambda: False):
    """Whether a DDS product of ``entries`` matrices of ``rows`` dense rows takes the panel walk
    (bsa_matmul_dds_panels): where it is the faster one, or, ``without_choice()``, wherever it can."""
    tiles, sets = -(-rows // PANEL_ROWS), -(-groups // PANEL_GROUPS)
    if (kblocks > PANEL_MAX_KBLOCKS or nnz > PANEL_MAX_NNZ or entries > 65535 or rows > 2 ** 30
            or (rows // 64 + 1) * (groups // 8 + 1) >= 2 ** 28):
        return False
    return ((tiles * sets * entries >= PANEL_MIN_WORKGROUPS
             and nnz * rows >= PANEL_MIN_DENSITY * kblocks * groups * tiles * PANEL_ROWS) or without_choice())


def sparse_weight_gradient(a, b, row_layout, col_layout, trans_a, trans_b):
    """``sparse_matmul(a, b, 'sdd', ..)`` summed over the batch: the gradient of a sparse operand that the batch shared.
    With both operands stored tokens-first (``trans_a``, not ``trans_b``) the batch and the tokens are one contraction,
    summed in fp32 by bsa_weight_grad; the other forms write a stack per batch entry and add them up."""
    if _folds(a, b, row_layout, col_layout, trans_a, trans_b):
        a, b = a.contiguous(), b.contiguous()
        if a.data_ptr() % 16 == 0 and b.data_ptr() % 16 == 0:
            return _folded_weight_gradient(a, b, row_layout, col_layout)
    stack = sparse_matmul(a, b, "sdd", row_layout, col_layout, trans_a, trans_b)
    return stack.sum(dim=tuple(range(stack.dim() - 3)))


def _folds(a, b, row_layout, col_layout, trans_a, trans_b):
    nnz = row_layout[0].numel() // 2
    rows, cols = row_layout[1].numel() - 1, col_layout[1].numel() - 1
    tokens = a.numel() // max(a.size(-1), 1)
    return (trans_a and not trans_b and a.dtype in (torch.float16, torch.bfloat16) and a.dtype == b.dtype
             and a.shape[:-1] == b.shape[:-1] and a.size(-2) % BLOCK == 0 and BLOCK <= tokens < 2 ** 31
             and a.size(-1) == BLOCK * rows and b.size(-1) == BLOCK * cols and a.is_cuda and a.device == b.device
             and row_layout[0].device == a.device and nnz > 0
             and ((tokens >= WEIGHT_GRAD_MIN_TOKENS and nnz >= WEIGHT_GRAD_MIN_DENSITY * rows * cols)
                  or _captured_without(row_layout, SCHEDULE_SDD)))


def _folded_weight_gradient(a, b, row_layout, col_layout):
    _check_layout(row_layout, "row_layout")
    nnz, tokens = row_layout[0].numel() // 2, a.numel() // a.size(-1)
    rows, cols = row_layout[1].numel() - 1, col_layout[1].numel() - 1
    out = torch.empty((nnz, BLOCK, BLOCK), dtype=a.dtype, device=a.device)
    shares = _k.lib.bsa_weight_grad_shares(rows, cols, tokens)
    parts = torch.empty(shares * nnz * BLOCK * BLOCK, dtype=torch.float32, device=a.device)
    with _k.on_device(a.device):
        _k.check(_k.lib.bsa_weight_grad(
            _DTYPES[a.dtype], a.data_ptr(), b.data_ptr(), out.data_ptr(), row_layout[0].data_ptr(),
            row_layout[1].data_ptr(), rows, cols, nnz, tokens, shares, parts.data_ptr(), 4 * parts.numel(),
            _k.current_stream()))
    return out


def _softmax_common(x, row_layout, col_layout, name):
    if x.dtype not in _DTYPES:
        raise TypeError(f"{name} must be float32, float16 or bfloat16, got {x.dtype}")
    if not x.is_cuda:
        raise ValueError(f"{name} must live on the GPU")
    _check_layout(row_layout, "row_layout")
    num_blocks = row_layout[0].numel() // 2
    if x.dim() < 4 or tuple(x.shape[-3:]) != (num_blocks, BLOCK, BLOCK):
        raise ValueError(f"{name} must be [..., {num_blocks}, 32, 32] with at least one batch "
                         f"dimension, got {tuple(x.shape)}")
    mask_rows = row_layout[1].numel() - 1
    mask_cols = col_layout[1].numel() - 1 if col_layout is not None else 65535
    batches = x.numel() // max(num_blocks * BLOCK * BLOCK, 1) if num_blocks else 1
    return num_blocks, mask_rows, mask_cols, max(batches, 1)


def sparse_softmax_forward(x, row_blocks, row_table, scale=1.0, causal=False, col_layout=None):
    """``y = softmax(scale * x)`` over the stored blocks of each row (sparse_softmax.cu:208-231)."""
    row_layout = (row_blocks, row_table)
    nnz, mask_rows, mask_cols, batches = _softmax_common(x, row_layout, col_layout, "x")
    x = x.contiguous()
    y = torch.empty_like(x)
    if nnz == 0 or x.numel() == 0:
        return y
    sched = _softmax_schedule(row_layout, x.dtype, False)
    with _k.on_device(x.device):
        _k.check(_k.lib.bsa_softmax_forward(
            _DTYPES[x.dtype], x.data_ptr(), y.data_ptr(), row_blocks.data_ptr(), row_table.data_ptr(),
            sched.table.data_ptr(), sched.workgroups, sched.waves, mask_rows, mask_cols, nnz, batches,
            float(scale), int(bool(causal)), _k.current_stream()))
    return y


def sparse_softmax_backward(y, dy, row_blocks, row_table, scale=1.0, col_layout=None):
    """``dx = scale * (dy - sum(dy * y)) * y`` per row (sparse_softmax.cu:233-258)."""
    row_layout = (row_blocks, row_table)
    nnz, mask_rows, mask_cols, batches = _softmax_common(y, row_layout, col_layout, "y")
    if dy.shape != y.shape or dy.dtype != y.dtype or dy.device != y.device:
        raise ValueError("dy must match y in shape, dtype and device")
    y = y.contiguous()
    dy = dy.contiguous()
    dx = torch.empty_like(y)
    if nnz == 0 or y.numel() == 0:
        return dx
    sched = _softmax_schedule(row_layout, y.dtype, True)
    with _k.on_device(y.device):
        _k.check(_k.lib.bsa_softmax_backward(
            _DTYPES[y.dtype], y.data_ptr(), dy.data_ptr(), dx.data_ptr(), row_blocks.data_ptr(),
            row_table.data_ptr(), sched.table.data_ptr(), sched.workgroups, sched.waves,
            mask_rows, mask_cols, nnz, batches, float(scale), _k.current_stream()))
    return dx


def _attention_common(q, k, v, row_blocks, row_table, col_layout):
    row_layout = (row_blocks, row_table)
    _check_layout(row_layout, "row_layout")
    for t, name in ((q, "q"), (k, "k"), (v, "v")):
        if t.dtype not in (torch.float16, torch.bfloat16) or t.dtype != q.dtype:
            raise TypeError(f"q, k, v must all be float16 or all bfloat16, got {name}: {t.dtype}")
        if not t.is_cuda or t.device != q.device:
            raise ValueError("q, k, v must live on the same GPU")
        if t.dim() < 3:
            raise ValueError(f"{name} needs at least one batch dimension, got shape {tuple(t.shape)}")
    if row_blocks.device != q.device:
        raise ValueError("layout tables and operands must live on the same GPU")
    if col_layout is None:
        raise ValueError("col_layout is needed for the number of block columns")
    mask_rows, mask_cols = row_table.numel() - 1, col_layout[1].numel() - 1
    head = q.size(-1)
    if q.size(-2) != mask_rows * BLOCK or k.size(-2) != mask_cols * BLOCK or k.shape != v.shape \
            or k.size(-1) != head or q.shape[:-2] != k.shape[:-2]:
        raise ValueError(f"q {tuple(q.shape)}, k {tuple(k.shape)}, v {tuple(v.shape)} do not fit a "
                         f"{mask_rows} x {mask_cols} block layout")
    batches = q.numel() // max(q.size(-1) * q.size(-2), 1)
    return row_layout, mask_rows, mask_cols, row_blocks.numel() // 2, head, batches


def _at_16_bytes(*operands):
    """Contiguous operands at multiples of 16 bytes: the attention walks load them straight to LDS, 16 bytes a lane, and a
    contiguous view may start anywhere in its storage."""
    return tuple(t if t.data_ptr() & 15 == 0 else t.clone() for t in operands)


def sparse_attention_forward(q, k, v, row_blocks, row_table, scale=1.0, causal=False, col_layout=None,
                             return_lse=False):
    """``softmax(scale * q k^T on the stored blocks) v`` in one launch: the chain of
    ``sparse_matmul('sdd', trans_b)``, the softmax and ``sparse_matmul('dsd')`` (sparse/matmul.py:57,
    sparse_softmax.cu:208-231) without the scores in memory.  fp16 / bf16, head dim 64 or 128.
    With ``return_lse`` also the fp32 row statistics the backward pass needs."""
    row_layout, mask_rows, mask_cols, nnz, head, batches = _attention_common(q, k, v, row_blocks, row_table,
                                                                              col_layout)
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    if (q.data_ptr() | k.data_ptr() | v.data_ptr()) & 15:
        q, k, v = _at_16_bytes(q, k, v)
    out = torch.empty_like(q)
    lse = torch.empty(q.shape[:-1], dtype=torch.float32, device=q.device) if return_lse else None
    if out.numel() > 0:
        sched = _attention_schedule_for(row_layout, SCHEDULE_ATTENTION, batches)
        with _k.on_device(q.device):
            stream = _k.current_stream()
            ws, ws_bytes, key = sched.attention_workspace(batches, head, stream)
            _launch(sched, key, _k.lib.bsa_attention_forward(
                _DTYPES[q.dtype], q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                lse.data_ptr() if lse is not None else None,
                row_blocks.data_ptr(), row_table.data_ptr(), sched.table.data_ptr(), sched.workgroups, sched.waves,
                sched.tile_slots, sched.split_groups, ws.data_ptr() if ws is not None else None, ws_bytes,
                mask_rows, mask_cols, nnz, batches, head, float(scale), int(bool(causal)), stream))
    return (out, lse) if return_lse else out


def sparse_attention_backward_scores(q, k, v, dout, out, lse, row_blocks, row_table, scale=1.0, causal=False,
                                     col_layout=None, with_dq=True):
    """Probabilities and score gradients of every stored block, ``[..., nnz, 32, 32]`` each, and (with
    ``with_dq``, else ``None``) the gradient of ``q``, in one launch: what ``sparse_matmul('sdd')``, the
    softmax forward, ``sparse_matmul('sdd')`` on ``dout, v``, the softmax backward
    (sparse_softmax.cu:165-205) and ``sparse_matmul('dsd')`` on ``ds, k`` give with five."""
    row_layout, mask_rows, mask_cols, nnz, head, batches = _attention_common(q, k, v, row_blocks, row_table,
                                                                              col_layout)
    if dout.shape != q.shape or out.shape != q.shape or dout.dtype != q.dtype or out.dtype != q.dtype:
        raise ValueError("dout and out must match q in shape and dtype")
    if lse.dtype != torch.float32 or lse.shape != q.shape[:-1]:
        raise ValueError("lse must be the float32 row statistics of the forward pass")
    q, k, v, dout, out, lse = (t.contiguous() for t in (q, k, v, dout, out, lse))
    if (q.data_ptr() | k.data_ptr() | v.data_ptr() | dout.data_ptr()) & 15:
        q, k, v, dout = _at_16_bytes(q, k, v, dout)
    shape = q.shape[:-2] + (nnz, BLOCK, BLOCK)
    p = torch.empty(shape, dtype=q.dtype, device=q.device)
    ds = torch.empty(shape, dtype=q.dtype, device=q.device)
    dq = torch.empty_like(q) if with_dq else None
    if q.numel() > 0:
        sched = _attention_schedule(row_layout, SCHEDULE_ATTENTION_BACKWARD, split=ATTENTION_SPLIT_ROWS)
        with _k.on_device(q.device):
            stream = _k.current_stream()
            ws, ws_bytes, key = sched.attention_backward_workspace(None, batches, head, stream) if with_dq else (None, 0, None)
            _launch(sched, key, _k.lib.bsa_attention_backward_scores(
                _DTYPES[q.dtype], q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), out.data_ptr(),
                lse.data_ptr(), p.data_ptr(), ds.data_ptr(), dq.data_ptr() if with_dq else None,
                row_blocks.data_ptr(), row_table.data_ptr(),
                sched.table.data_ptr(), sched.workgroups, sched.waves, sched.tile_slots, sched.split_groups,
                ws.data_ptr() if ws is not None else None, ws_bytes, mask_rows, mask_cols, nnz, batches, head,
                float(scale), int(bool(causal)), stream))
    return p, ds, dq


def _attention_backward_schedules(row_layout, col_layout, batches, head, with_dkdv):
    rs = _attention_schedule_for(row_layout, SCHEDULE_ATTENTION_BACKWARD, batches)
    cs = _attention_schedule_for(col_layout, SCHEDULE_ATTENTION_BACKWARD_COLUMNS, batches,
                                 ATTENTION_WAVES_LONG_GROUPS if head == 64 else ATTENTION_COLUMN_WAVES_128) \
        if with_dkdv else None
    return rs, cs


def sparse_attention_backward(q, k, v, dout, out, lse, row_blocks, row_table, col_blocks, col_table, scale=1.0,
                              causal=False, with_dkdv=True):
    """``(dq, dk, dv)`` of the fused attention in two launches (a walk over the rows, one over the
    columns), the probabilities and score gradients rebuilt in registers in both instead of stored:
    the seven launches of the unfused backward chain (sparse/matmul.py:27-52, sparse_softmax.cu:165-205)
    without a block stack in memory.  fp16 / bf16, head dim 64 or 128.  ``with_dkdv=False``: dq alone (None for the
    others), one launch."""
    col_layout = (col_blocks, col_table)
    _check_layout(col_layout, "col_layout")
    row_layout, mask_rows, mask_cols, nnz, head, batches = _attention_common(q, k, v, row_blocks, row_table,
                                                                              col_layout)
    if dout.shape != q.shape or out.shape != q.shape or dout.dtype != q.dtype or out.dtype != q.dtype:
        raise ValueError("dout and out must match q in shape and dtype")
    if lse.dtype != torch.float32 or lse.shape != q.shape[:-1]:
        raise ValueError("lse must be the float32 row statistics of the forward pass")
    q, k, v, dout, out, lse = (t.contiguous() for t in (q, k, v, dout, out, lse))
    if (q.data_ptr() | k.data_ptr() | v.data_ptr() | dout.data_ptr()) & 15:
        q, k, v, dout = _at_16_bytes(q, k, v, dout)
    dq = torch.empty_like(q)
    dk, dv = (torch.empty_like(k), torch.empty_like(v)) if with_dkdv else (None, None)
    if q.numel() > 0:
        delta = torch.empty_like(lse)
        rs, cs = _attention_backward_schedules(row_layout, col_layout, batches, head, with_dkdv)
        columns = (cs.table.data_ptr(), cs.workgroups, cs.waves, cs.tile_slots, cs.split_groups) if with_dkdv \
            else (None, 0, 0, 0, 0)
        with _k.on_device(q.device):
            stream = _k.current_stream()
            ws, ws_bytes, key = rs.attention_backward_workspace(cs, batches, head, stream)
            _launch(rs, key, _k.lib.bsa_attention_gradients(
                _DTYPES[q.dtype], q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), out.data_ptr(),
                lse.data_ptr(), dq.data_ptr(), dk.data_ptr() if with_dkdv else None, dv.data_ptr() if with_dkdv else None,
                delta.data_ptr(),
                row_blocks.data_ptr(), row_table.data_ptr(), rs.table.data_ptr(), rs.workgroups, rs.waves,
                rs.tile_slots, rs.split_groups,
                col_blocks.data_ptr(), col_table.data_ptr(), *columns, ws.data_ptr() if ws is not None else None, ws_bytes,
                mask_rows, mask_cols, nnz, batches, head, float(scale), int(bool(causal)), stream))
    return dq, dk, dv


# ---- plans: what csrc/host_calls.cpp needs to make a call of these shapes again without asking Python ----------------
_LIB = _k.lib
_MATMUL, _WEIGHT, _SOFTMAX, _SOFTMAX_BACKWARD, _ATTENTION, _ATTENTION_BACKWARD = range(6)
_ROUTES = {"walk": 0, "runs": 1, "panels": 2}


def _plans(layout, *operands):
    """The layout's plans where a call on these operands may be planned: nothing under capture (what is missing there is not
    built, and the walk that serves is not the one an eager call takes), nothing for operands off 16 bytes, which some walks do
    not take, and nothing while the library is replaced."""
    if _k.lib is not _LIB or torch.cuda.is_current_stream_capturing() or any(t.data_ptr() & 15 for t in operands):
        return None
    return getattr(layout, "_plans", None)


def _planned(make):
    """``make`` returns whether it left a plan; what it cannot do the general path does, or says why not."""
    @functools.wraps(make)
    def planned(*args):
        try:
            with _k.on_device(args[0].device):
                return make(*args)
        except Exception:
            return False
    return planned


def _add(plans, op, flags, a, b, route, ints, tables, out=(), workspace=(None, 0, None), sched=None, aligned=False):
    ws, ws_bytes, key = workspace
    _k.host_calls.add_plan(plans, op, flags, a, b, route, _DTYPES[a.dtype], aligned, ints, tables, out,
                           sched.plan_space(key, ws) if ws is not None else None, ws_bytes, _k.current_stream(), sched, key)
    return True


@_planned
def plan_matmul(a, b, mode, layout, trans_a, trans_b):
    plans = _plans(layout, a, b)
    if plans is None:
        return False
    rows, cols = layout.row_layout, layout.col_layout
    walk, sched, table, _, _, shape, shared, batches, m, n, k = _matmul_route(a, b, mode, rows, cols, trans_a, trans_b)
    if walk not in _ROUTES:
        return False
    counts = (rows[1].numel() - 1, cols[1].numel() - 1, table[0].numel() // 2, batches, 1 if shared else batches)
    flags = _k.MODES[mode] << 2 | bool(trans_a) << 1 | bool(trans_b)
    add = functools.partial(_add, plans, _MATMUL, flags, a, b, _ROUTES[walk], out=tuple(shape))
    if walk == "runs":
        return add((sched.runs, sched.strips, sched.pairs, sched.waves) + counts + (n,), table + (sched.table,))
    if walk == "panels":
        return add(counts + (m, int(bool(trans_b))), table, aligned=True)
    space = sched.workspace(_k.MODES[mode], batches, m, n, _k.current_stream())
    return add((_k.MODES[mode], table[1].numel() - 1, sched.workgroups, sched.waves, sched.tile_slots, sched.split_groups) + counts +
               (m, n, k, int(bool(trans_a)), int(bool(trans_b))), table + (sched.table,), workspace=space, sched=sched)


@_planned
def plan_weight(a, b, layout, trans_a, trans_b):
    plans = _plans(layout, a, b)
    rows, cols = layout.row_layout, layout.col_layout
    if plans is None or not _folds(a, b, rows, cols, trans_a, trans_b):
        return False
    _check_layout(rows, "row_layout")
    nnz, tokens = rows[0].numel() // 2, a.numel() // a.size(-1)
    mask = rows[1].numel() - 1, cols[1].numel() - 1
    shares = _k.lib.bsa_weight_grad_shares(*mask, tokens)
    floats = shares * nnz * BLOCK * BLOCK
    if floats >= 2 ** 31:
        return False
    return _add(plans, _WEIGHT, bool(trans_a) << 1 | bool(trans_b), a, b, 0, mask + (nnz, tokens, shares, floats), rows,
                (nnz, BLOCK, BLOCK), aligned=True)


def _plan_softmax(x, layout, backward):
    plans = _plans(layout, x)
    if plans is None:
        return False
    nnz, mask_rows, mask_cols, batches = _softmax_common(x, layout.row_layout, layout.col_layout, "x")
    if nnz == 0 or x.numel() == 0:
        return False
    sched = _softmax_schedule(layout.row_layout, x.dtype, backward)
    return _add(plans, _SOFTMAX_BACKWARD if backward else _SOFTMAX, 0, x, None, 0,
                (sched.workgroups, sched.waves, mask_rows, mask_cols, nnz, batches), layout.row_layout + (sched.table,))


@_planned
def plan_softmax(x, layout):
    return _plan_softmax(x, layout, False)


@_planned
def plan_softmax_backward(y, layout):
    return _plan_softmax(y, layout, True)


def _figures(sched):
    return sched.workgroups, sched.waves, sched.tile_slots, sched.split_groups


@_planned
def plan_attention(q, k, v, layout):
    plans = _plans(layout, q, k, v)
    if plans is None or q.numel() == 0:
        return False
    rows, *counts = _attention_common(q, k, v, *layout.row_layout, layout.col_layout)
    mask_rows, mask_cols, nnz, head, batches = counts
    sched = _attention_schedule_for(rows, SCHEDULE_ATTENTION, batches)
    space = sched.attention_workspace(batches, head, _k.current_stream())
    return _add(plans, _ATTENTION, 0, q, k, 0, _figures(sched) + (mask_rows, mask_cols, nnz, batches, head), rows + (sched.table,),
                workspace=space, sched=sched)


@_planned
def plan_attention_backward(q, k, v, layout, with_dkdv):
    plans = _plans(layout, q, k, v)
    if plans is None or q.numel() == 0:
        return False
    cols = layout.col_layout
    _check_layout(cols, "col_layout")
    rows, mask_rows, mask_cols, nnz, head, batches = _attention_common(q, k, v, *layout.row_layout, cols)
    rs, cs = _attention_backward_schedules(rows, cols, batches, head, with_dkdv)
    space = rs.attention_backward_workspace(cs, batches, head, _k.current_stream())
    return _add(plans, _ATTENTION_BACKWARD, int(bool(with_dkdv)), q, k, 0,
                _figures(rs) + (_figures(cs) if with_dkdv else (0, 0, 0, 0)) + (mask_rows, mask_cols, nnz, batches, head),
                rows + (rs.table,) + cols + (cs.table if with_dkdv else None,), workspace=space, sched=rs)


def failed(status, sched, key):
    """Raises for a failed launch; its workspace is forgotten first (``_launch``)."""
    if sched is not None:
        sched.discard(key)
    _k.check(status)
