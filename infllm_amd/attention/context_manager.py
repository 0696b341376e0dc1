"""ContextManager: the streaming memory behind the "inf-llm" attention type.

Same constructor, ``append`` and ``size``/``length`` as
inf_llm/attention/context_manager.py:196-816, re-designed around absolute
stream positions and device-resident rings instead of torch.cat/trim:

* new tokens are written once into per-layer rings (raw K, RoPE'd K, V, fp32
  score track) by the prologue kernel, row = position % ring_cap; the local
  window and the "remainder" of the reference are index ranges of that ring;
* the local stage is one launch of the MFMA kernel over the ring with the
  causal sliding-window mask; the global stage is one launch over a page table
  of 64-key tiles (cached memory units, init tokens, overflow remainder) - the
  reference's global_buffer copies do not exist;
* both stages leave partials that the merge kernel joins into the joint
  softmax; the local score (probability column sums) is a third kernel that
  needs the merged log-sum-exp;
* memory units live in HBM where there is room for them (``resident_bytes``):
  a whole append() call is then enqueued by one native call
  (infllm_resident_append), the selections become page tables on the device,
  and the host only keeps the residency policy's books from a pinned log;
* otherwise - beyond that budget, with the lru-s policy, with retrieval in
  chunks, and while selections are recorded or stepped through - the host
  drives every block: units live in pinned host memory and in a slab of
  ``max_cached_block`` device slots managed by the reference's lru / lru-s
  policy (plus fifo; native, infllm_cache_*); the misses of a block are moved
  by the DMA engines (short blocks: read from the pinned pages by one kernel
  on a side stream), for lru / fifo starting from the selection's candidates a
  block ahead of the selection itself (``fetch_ahead``).

The state machine is in absolute positions (context_manager.py:614-679
restated): ``cursor`` is the first token not yet carved, tokens [0, init_len)
are the attention sinks, unit u is tokens [n_init + u*bs, n_init + (u+1)*bs).
Driven by the host, the device work of one execution block is issued by three
native calls: infllm_block_front, infllm_block_select (the one host wait, for
the retrieved unit ids, which overlaps the local stage; then cache policy and
fetch) and infllm_block_back, plus infllm_block_prefetch for the next block.
"""
import contextlib
import ctypes
import functools
import os
import struct
import threading
import weakref

import torch

from .. import _lib
from .._lib import BackArgs, FrontArgs, LayerDesc, ResidentCall, ResidentDesc, check
from ..ops import HEAD_DIM, KEY_TILE, current_stream, rows16

from ._rows import check_head_dim, narrow as _narrow, wide_inv_freq, widen as _widen

_SIDE_STREAM = None          # one process-wide side stream, like GLOBAL_STREAM (context_manager.py:193)
# (device, stream, geometry) -> the buffers of a call prepared in one go, shared by the managers that are alive
_CALL_BUFFERS = weakref.WeakValueDictionary()
_HOST_CHUNK_UNITS = 64       # units per pinned host allocation
_UNIT_CHUNK = 64             # units per allocation of their home in HBM, at most ...
_CHUNK_BYTES = 96 << 20      # ... fewer where that many would take more than this (a batch), but four at least
_SPARE = 8                   # by default units do not take the last eighth of a device's memory; the driver is asked again when
_ASK_BYTES = 1 << 30         # this much has been taken (5 us, 60 beside a running kernel: 0.3 % of a long prompt at every step)
_LOG_SLOTS = 256             # selections whose bookkeeping may be outstanding
_MAX_SPLITS = 16             # key splits of one attention stage
_NUM_CUS = 256               # MI355X
_PAGE_SLOTS = 4
_CARVE_SLOTS = 4             # staging slots of the carve, used in turn (more of them serve more misses on the device - 16: 18 %,
                             # 64: 57 % of the benchmark stream's - but the stream is no faster for it, measured)


_CALL_ROWS = struct.Struct("@3P9qP4q")      # the first fields of an infllm_resident_call, d_q to n


@functools.lru_cache(None)
def _device_bytes(index):
    return torch.cuda.get_device_properties(index).total_memory


def _addressed(t):
    """rows16(t), with its address and strides"""
    strides, ptr = t.stride(), t.data_ptr()
    if strides[3] != 1 or (strides[0] | strides[1] | strides[2]) & 7 or ptr & 15:
        t = t.clone(memory_format=torch.contiguous_format)
        strides, ptr = t.stride(), t.data_ptr()
    return t, ptr, strides


class _Buffers(dict):
    """Workspaces of a call, shared by the managers that work on one stream.  Whoever enqueues launches on them holds the lock
    until the call's last one is enqueued: the stream orders whole calls, not the launches that two threads enqueue by turns."""

    def __init__(self, **tensors):
        super().__init__(**tensors)
        self.lock = threading.Lock()


class _Units:
    """What the resident units of all managers take of a device's memory, and the pinned logs between managers."""
    lock = threading.RLock()  # (a manager that the interpreter collects while it holds the lock gives its share back then)
    used = {}                 # device index -> bytes
    logs = {}                 # (device index, ints) -> [(log, last sequence number written or on its way)]
    max_logs = 64             # logs kept per size
    asked = {}                # device index -> bytes that may be taken before the driver is asked for its free memory again
    lost = []                 # logs whose launches could not be waited for

    @classmethod
    def take(cls, dev, n, limit):
        with cls.lock:
            cls.used[dev] = cls.used.get(dev, 0) + n
            if cls.used[dev] <= limit:
                return True
            cls.used[dev] -= n
        return False

    @classmethod
    def give(cls, dev, n):
        with cls.lock:
            cls.used[dev] = cls.used.get(dev, 0) - n

    @classmethod
    def take_log(cls, dev, stride):
        """A pinned log and the sequence number to go on from: one whose last selection has arrived, or a new one."""
        n = _LOG_SLOTS * stride
        with cls.lock:
            pool = cls.logs.setdefault((dev, n), [])
            for i, (log, seq) in enumerate(pool):
                if seq == 0 or ctypes.c_int32.from_address(log.data_ptr() + 4 * ((seq % _LOG_SLOTS) * stride + stride - 1)).value == seq:
                    del pool[i]
                    return log, seq
        return torch.zeros((n,), dtype=torch.int32, pin_memory=True), 0

    @classmethod
    def give_log(cls, dev, log, seq):
        with cls.lock:
            pool = cls.logs.setdefault((dev, log.numel()), [])
            if seq < 1 << 30 and len(pool) < cls.max_logs:
                pool.append((log, seq))
                return
        torch.cuda.synchronize(dev)               # kernels may still be on their way to it


class CachePolicy:
    """Residency policy of one batch row (context_manager.py:246-265, 495-515): a handle on the native
    object (infllm_cache_*), which ContextManager also drives directly from infllm_block_select.

    ``cached`` is the reference's insertion-ordered dict unit -> value; eviction walks it in
    ascending value (stable), skipping the units selected for this block.
    """

    def __init__(self, capacity, strategy, score_decay):
        self.capacity, self.strategy, self.score_decay = capacity, strategy, score_decay
        self._lib = _lib.load()
        self.handle = self._lib.infllm_cache_create(capacity, _lib.CACHE_STRATEGY[strategy],
                                                    float(score_decay) if score_decay is not None else 0.0)
        if not self.handle:
            raise _lib.InfLLMHipError((self._lib.infllm_last_error() or b"").decode())
        self.evicted_log = None             # set to a list to record the evictions of every block
        self._units = (ctypes.c_int32 * capacity)()
        self._slots = (ctypes.c_int32 * capacity)()
        self._values = (ctypes.c_double * capacity)()

    def __del__(self):
        if getattr(self, "handle", None):
            self._lib.infllm_cache_destroy(self.handle)
            self.handle = None

    def touch(self, selected):
        """Returns (misses, evicted) and updates values; slots of evicted units are freed."""
        n = len(selected)
        assert n <= self.capacity, "topk exceeds max_cached_block"
        sel = (ctypes.c_int32 * max(n, 1))(*selected)
        slots, mu, ms = ((ctypes.c_int32 * max(n, 1))() for _ in range(3))
        ev, n_ev = (ctypes.c_int32 * self.capacity)(), ctypes.c_int32(0)
        n_miss = self._lib.infllm_cache_touch(self.handle, sel, n, slots, mu, ms, ev, ctypes.byref(n_ev))
        if n_miss < 0:
            check(n_miss, "infllm_cache_touch")
        evicted = list(ev[:n_ev.value])
        if self.evicted_log is not None:
            self.evicted_log.append(evicted)
        return list(mu[:n_miss]), evicted

    def add_scores(self, units, unit_scores):
        n = len(units)
        check(self._lib.infllm_cache_add_scores(self.handle, (ctypes.c_int32 * max(n, 1))(*units),
                                                (ctypes.c_double * max(n, 1))(*unit_scores[:n]), n), "infllm_cache_add_scores")

    def _residents(self):
        n = self._lib.infllm_cache_residents(self.handle, self._units, self._values, self._slots, self.capacity)
        if n < 0:
            check(n, "infllm_cache_residents")
        return n

    @property
    def cached(self):
        n = self._residents()
        as_int = self.strategy != "lru-s"
        return {self._units[i]: (int(self._values[i]) if as_int else self._values[i]) for i in range(n)}

    @property
    def slot_of(self):
        n = self._residents()
        return {self._units[i]: self._slots[i] for i in range(n)}

    @property
    def free(self):
        used = set(self.slot_of.values())
        return [s for s in range(self.capacity) if s not in used]


class ContextManager:
    select_in_steps = False     # True: drive wait / policy / fetch from here (slower), instead of infllm_block_select
    fetch_ahead = True          # start the next block's fetch from its candidates (infllm_block_prefetch)
    call_tokens = 8192          # tokens of an append() call prepared in one go (prologue, mean queries and the local
                                # stage of all their blocks: infllm_call_front); 0: every block runs its own.
                                # INFLLM_CALL_TOKENS overrides it.  Needs exc_block_size to be a multiple of 32.
    local_group_blocks = None   # blocks of a prepared call per launch of the local stage (INFLLM_LOCAL_GROUP overrides it);
                                # None: two where the host drives, else as many as pay
    resident_bytes = None       # HBM that the units of all managers of this process may take together on a device; None: a
                                # quarter of it, and not the last eighth of what is free.  0 keeps units in pinned host
                                # memory, max_cached_block of them on the device (so does INFLLM_NO_RESIDENT=1).

    rows_by_token = False       # set for the next append() by a caller that takes a token's rows next to each other (the view
                                # [B, H, n, D] of a tensor [B, n, H, D], where the path has one to give): spares it a copy

    def __init__(self, position_embedding, n_init, n_local, block_size, max_cached_block, topk, exc_block_size,
                 score_decay=None, fattn=False, repr_topk=1, cache_strategy="lru", chunk_topk_calc=None,
                 async_global_stream=False, pin_memory=False, faiss=False, perhead=False):
        assert exc_block_size <= n_local                       # no global token inside the input block
        assert cache_strategy in ("lru", "lru-s", "fifo")
        if faiss:
            raise NotImplementedError("the faiss representative store is not available in this build")
        if cache_strategy == "lru-s":
            assert score_decay is not None, "cache_strategy='lru-s' needs score_decay"
        if chunk_topk_calc is not None:
            assert chunk_topk_calc >= exc_block_size, "chunk_topk_calc must cover at least one execution block"
        self.length = 0
        self.position_embedding = position_embedding
        self.n_init, self.n_local = n_init, n_local
        self.block_size, self.max_cached_block = block_size, max_cached_block
        self.topk, self.exc_block_size = topk, exc_block_size
        self.score_decay, self.fattn, self.repr_topk = score_decay, fattn, repr_topk
        self.cache_strategy = cache_strategy
        self.chunk_topk_calc = chunk_topk_calc
        self.async_global_stream = async_global_stream
        self.pin_memory = pin_memory           # host copies are always pinned here
        self.perhead = perhead
        self.initialized = False
        self.load_count = 0
        self.record_trace = False
        self.trace_blocks, self.trace_units = [], []
        self._call_scores = None      # [blocks of a call, B, units]: scores of every unit under every block's mean query
        self._host_copies_open = False
        self._stats = dict(blocks=0, hits=0, misses=0, evictions=0)
        self._policy = []
        self._layer = None
        self._resident = None         # native handle while the units are resident in HBM
        self._timing_cap, self._timing_stride = 0, 1
        self._mass_units = None                # lru-s: selections of the block whose unit masses are still on the device
        global _SIDE_STREAM
        if async_global_stream and _SIDE_STREAM is None and torch.cuda.is_available():
            _SIDE_STREAM = torch.cuda.Stream()

    def __del__(self):
        layer, self._layer = getattr(self, "_layer", None), None
        try:
            if layer:
                _lib.load().infllm_layer_destroy(layer)       # waits for this layer's own work, not for the device
            self._drop_resident()
        except Exception:
            pass

    # ------------------------------------------------------------------ setup
    def _wants_resident(self):
        """Whether the units may live in HBM: nothing asks for the host between a block's selection and its fetch."""
        return not (self.record_trace or self.select_in_steps or not self.fetch_ahead)

    def _init(self, q, k, resident=None):
        """q, k: rows of the heads' own width.  resident: False to have the host drive, None to choose."""
        B, H = q.shape[0], q.shape[1]
        Hkv = k.shape[1]
        dev = q.device
        if self.topk > self.max_cached_block:
            raise ValueError("topk must not exceed max_cached_block")
        if self.topk > 64:
            raise ValueError("this build selects at most 64 units per block (topk <= 64)")
        if self.repr_topk > self.block_size:
            raise ValueError("repr_topk must not exceed block_size")
        if self.position_embedding.inv_freq.numel() != self.dim_head // 2:
            raise ValueError(f"the rotary embedding is built for head_dim {2 * self.position_embedding.inv_freq.numel()}, "
                             f"the heads have {self.dim_head}")
        self.batch_size = self.num_units = B
        self.num_heads = self.unit_size = H
        self.num_heads_kv = self.unit_size_kv = Hkv
        self.dtype = q.dtype
        self.device = dev
        self._dev_index = dev.index if dev.index is not None else torch.cuda.current_device()
        self._lib = _lib.load()
        bs, exc, topk = self.block_size, self.exc_block_size, self.topk
        ct = int(os.environ.get("INFLLM_CALL_TOKENS", self.call_tokens))
        self._call_tokens = min(ct, 16 * exc) // exc * exc if (ct >= exc and exc % 32 == 0) else 0
        group = os.environ.get("INFLLM_LOCAL_GROUP", self.local_group_blocks)
        # the rings hold the local window, the remainder that waits to fill a unit, and what is prepared ahead of the
        # block being attended: one block, or the rest of a call prepared in one go
        cap = self.n_local + exc + bs + max(exc, self._call_tokens)
        self.ring_cap = (cap + KEY_TILE - 1) // KEY_TILE * KEY_TILE + KEY_TILE
        tiles_per_unit = (bs + KEY_TILE - 1) // KEY_TILE
        self.max_pages = topk * tiles_per_unit + (self.n_init + KEY_TILE - 1) // KEY_TILE + (exc + bs) // KEY_TILE + 3
        self.cursor = 0
        self.init_len = 0
        self.num_global_block = 0
        self._policy = [CachePolicy(self.max_cached_block, self.cache_strategy, self.score_decay) for _ in range(B)]
        if self.record_trace:
            for pol in self._policy:
                pol.evicted_log = []
        desc = None if resident is False else self._can_be_resident()
        resident = desc is not None
        # Blocks per launch of the local stage.  With the host between the blocks two: a launch covers the wait for a fetch.
        # Without it as many as a call has (131,072 tokens: 33.0 -> 32.4 ms, 24,300 of the smaller geometry: 5.2 -> 4.7), unless
        # launches are timed one by one: a sample is a launch of two blocks.
        self._local_group = int(group) if group is not None else 16 if resident and not self._timing_cap else 2
        # rows of 64 are the kernels' own width where the units are resident; everything else travels in rows of 128
        self.head_width = D = 64 if resident and self.dim_head == 64 else HEAD_DIM
        bf = dict(dtype=torch.bfloat16, device=dev)
        f32 = dict(dtype=torch.float32, device=dev)
        self.ring_k_raw, self.ring_k_rot, self.ring_v = torch.empty((3, B, Hkv, self.ring_cap, D), **bf).unbind(0)
        self.ring_score = torch.empty((B, H, self.ring_cap), **f32)
        self.init_kv = torch.empty((B, 2, Hkv, max(self.n_init, 1), D), **bf)
        self.reps = torch.empty((B, 16, H * D), **bf)
        self.unit_scores = torch.empty((B, 16), **f32)
        inv_freq = self.position_embedding.inv_freq
        if D != self.dim_head:
            inv_freq = wide_inv_freq(inv_freq, dev)
        elif inv_freq.device != dev or inv_freq.dtype != torch.float32 or not inv_freq.is_contiguous():
            inv_freq = inv_freq.to(device=dev, dtype=torch.float32).contiguous()
        self.inv_freq = inv_freq
        self.slot_bytes = 2 * Hkv * bs * D * 2              # one unit of one batch row
        self.unit_bytes = B * self.slot_bytes               # one unit, all batch rows
        self._init_resident(desc) if resident else self._init_host()
        self._call_stream = None               # stream the call buffers were taken for (they are bound at the first append)
        self.initialized = True

    # ------------------------------------------------------ units resident in HBM
    def _resident_limit(self):
        if os.environ.get("INFLLM_NO_RESIDENT", "0") not in ("", "0"):
            return 0
        if self.resident_bytes is not None:
            return self.resident_bytes
        return _device_bytes(self._dev_index) // 4

    def _leaves_room(self, n):
        """Whether the device still has memory for its other users once the units take n bytes more: units that found a home in
        HBM are not moved out of it when an allocation of the caller fails.  A budget set by the caller is taken at its word."""
        dev, at = self._dev_index, _Units.asked
        if self.resident_bytes is not None:
            return True
        if at.get(dev, 0) >= n:
            at[dev] -= n
            return True
        free, total = torch.cuda.mem_get_info(dev)
        if free - n < total // _SPARE:
            free += torch.cuda.memory_reserved(dev) - torch.cuda.memory_allocated(dev)
        if free - n < total // _SPARE:
            return False
        at[dev] = min(_ASK_BYTES, free - n - total // _SPARE)
        return True

    @staticmethod
    def _units_per_chunk(unit_bytes):
        """The step in which a manager takes memory, also for its first unit (a batch of 8 in 32 layers of the reference's
        geometry: 2 GiB, where 64 units a step would be 8, and a cache of 32 slots 4)."""
        n = _UNIT_CHUNK
        while n > 4 and n * unit_bytes > _CHUNK_BYTES:
            n //= 2
        return n

    def _resident_desc(self, D):
        """The descriptor of a resident memory with rows of D elements; its buffers are not in it yet."""
        d = ResidentDesc()
        d.B, d.H, d.Hkv, d.dim = self.num_units, self.unit_size, self.unit_size_kv, D
        d.n_local, d.n_init, d.block_size, d.exc = self.n_local, self.n_init, self.block_size, self.exc_block_size
        d.topk, d.repr_topk, d.max_cached = self.topk, self.repr_topk, self.max_cached_block
        d.max_splits, d.num_cus, d.call_tokens, d.group_blocks = _MAX_SPLITS, _NUM_CUS, self._call_tokens, 1
        unit_bytes = 2 * self.num_units * self.unit_size_kv * self.block_size * D * 2
        d.max_pages, d.units_per_chunk, d.log_slots = self.max_pages, self._units_per_chunk(unit_bytes), _LOG_SLOTS
        d.ring_cap, d.init_cap = self.ring_cap, max(self.n_init, 1)
        return d

    def _can_be_resident(self):
        """The descriptor of the resident memory, or None: the host drives."""
        if not self._wants_resident() or self.cache_strategy == "lru-s" or self.chunk_topk_calc is not None or self.topk < 1:
            return None
        # the switches that choose between ways of the host-driven path ask for that path
        if any(name in os.environ for name in ("INFLLM_FETCH_AHEAD_ALWAYS", "INFLLM_NO_DMA_FETCH", "INFLLM_NO_DMA_ENGINE", "INFLLM_NO_STAGING_COPY",
                                               "INFLLM_NO_CALL_LISTS", "INFLLM_CALL_LISTS_ROOM", "INFLLM_PAGE_TABLE_KERNEL", "INFLLM_SCORE_MERGE_APART")):
            return None
        limit = self._resident_limit()
        if not limit or _Units.used.get(self._dev_index, 0) >= limit:
            return None
        d = self._resident_desc(64 if self.dim_head == 64 else HEAD_DIM)
        return d if self._lib.infllm_resident_fits(ctypes.byref(d)) == 1 else None

    def _init_resident(self, d):
        dev, B, topk = self.device, self.num_units, self.topk
        self._chunks = []                       # homes of the units: [_chunk_units, B, 2, Hkv, bs, D] each
        self._chunk_units = d.units_per_chunk
        self._chunk_bytes = self._chunk_units * self.unit_bytes
        self._chunk_host = (ctypes.c_uint64 * 16)()
        # addresses of the units' homes, and behind the 16 of them a page table and a selection
        page_words = B * self.max_pages * ctypes.sizeof(_lib.Page) // 8
        self._chunk_dev = self._tables = torch.empty((16 + page_words + (B * topk + 1) // 2,), dtype=torch.int64, device=dev)
        self._log, seq = _Units.take_log(self._dev_index, B * topk + 1)
        self._caches = (ctypes.c_void_p * B)(*[pol.handle for pol in self._policy])
        d.group_blocks = self._local_group
        d.d_ring_k_raw, d.d_ring_k_rot = self.ring_k_raw.data_ptr(), self.ring_k_rot.data_ptr()
        d.d_ring_v, d.d_ring_score, d.d_init_kv = self.ring_v.data_ptr(), self.ring_score.data_ptr(), self.init_kv.data_ptr()
        d.d_pages = self._tables.data_ptr() + 8 * 16
        d.d_ids = d.d_pages + 8 * page_words
        d.d_log, d.h_log = self._lib.infllm_host_device_pointer(self._log.data_ptr()), self._log.data_ptr()
        d.h_caches, d.d_inv_freq = ctypes.addressof(self._caches), self.inv_freq.data_ptr()
        d.distance_scale, d.softmax_scale = float(self.position_embedding.distance_scale), 1.0 / (self.dim_head ** 0.5)
        d.first_seq = seq
        self._part_rows2 = int(self._lib.infllm_resident_part_rows(ctypes.byref(d)))
        self._resident = self._lib.infllm_resident_create(ctypes.byref(d))
        if not self._resident:
            raise _lib.InfLLMHipError("infllm_resident_create failed: " + (self._lib.infllm_last_error() or b"").decode())
        if self._timing_cap:
            check(self._lib.infllm_resident_timing(self._resident, self._timing_cap, self._timing_stride), "infllm_resident_timing")
        self._state = (ctypes.c_int64 * 10)()
        self._streams = {torch._C._cuda_getCurrentRawStream(self._dev_index)}
        self._rc = ResidentCall()
        self._rc_ref = ctypes.byref(self._rc)
        self._rc.h_chunks, self._rc.d_chunks = ctypes.addressof(self._chunk_host), self._chunk_dev.data_ptr()
        self._rc.call_tokens = self._call_tokens
        self._rc.max_tokens = max(self._call_tokens, self.exc_block_size)
        self._bind_resident_reps()

    def _bind_resident_reps(self):
        rc = self._rc
        rc.d_reps, rc.rep_sb, rc.rep_su, rc.rep_rows = self.reps.data_ptr(), self.reps.stride(0), self.reps.stride(1), self.reps.shape[1]
        rc.d_unit_scores, rc.unit_scores_sb = self.unit_scores.data_ptr(), self.unit_scores.stride(0)

    def _add_chunks(self, n_units):
        """Homes for n_units units; False when the budget or the memory does not have them."""
        while len(self._chunks) * self._chunk_units < n_units:
            if not self._leaves_room(self._chunk_bytes) or not _Units.take(self._dev_index, self._chunk_bytes, self._resident_limit()):
                return False
            try:
                t = torch.empty((self._chunk_units, self.num_units, 2, self.unit_size_kv, self.block_size, self.head_width), dtype=torch.bfloat16,
                                device=self.device)
            except torch.OutOfMemoryError:
                _Units.give(self._dev_index, self._chunk_bytes)
                return False
            n = len(self._chunks)
            self._chunks.append(t)
            if n == len(self._chunk_host):
                grown = (ctypes.c_uint64 * (2 * n))()
                grown[:n] = self._chunk_host[:]
                table = torch.empty((2 * n,), dtype=torch.int64, device=self.device)
                table[:n] = self._chunk_dev[:n]
                self._retire(self._chunk_dev)
                self._chunk_host, self._chunk_dev = grown, table
                self._rc.h_chunks, self._rc.d_chunks = ctypes.addressof(grown), table.data_ptr()
            self._chunk_host[n] = t.data_ptr()
            self._chunk_dev[n].fill_(t.data_ptr())
        self._rc.n_chunks = len(self._chunks)
        return True

    @staticmethod
    def _retire(*buffers):
        """Buffers that are replaced: a stream other than the one they were made on may still have launches that use them."""
        for t in buffers:
            if t is not None and t.is_cuda:
                t.record_stream(torch.cuda.current_stream(t.device))

    def _drop_resident(self):
        handle, self._resident = getattr(self, "_resident", None), None
        if not handle:
            return
        self._lib.infllm_resident_state(handle, 0, self._state)
        log, self._log = self._log, None
        try:
            # Work on several streams is waited for: the newest selection may be in the log while an older one, on another
            # stream, is still to be written there; and the buffers go back to the allocator for the stream they were made on.
            if len(self._streams) > 1:
                torch.cuda.synchronize(self.device)
            _Units.give_log(self._dev_index, log, int(self._state[9]))
        except Exception:
            _Units.lost.append(log)                        # (launches may still write to it: never handed out or freed)
            raise
        finally:
            _Units.give(self._dev_index, len(self._chunks) * self._chunk_bytes)
            self._lib.infllm_resident_destroy(handle)
            self._chunks = []

    def _resident_books(self, wait):
        """The bookkeeping of the selections so far (wait: of all of them) into the counters."""
        check(self._lib.infllm_resident_state(self._resident, 1 if wait else 0, self._state), "infllm_resident_state")
        for i, name in ((4, "blocks"), (5, "hits"), (6, "misses"), (7, "evictions")):
            self._stats[name] = int(self._state[i])

    @property
    def stats(self):
        """Blocks worked off and the residency counters: hits, misses and evictions of the unit cache of max_cached_block
        slots (of the books, where the units are resident and nothing has to move)."""
        if self._resident:
            self._resident_books(True)
        return self._stats

    @property
    def policy(self):
        if self._resident:
            self._resident_books(True)
        return self._policy

    def _leave_resident(self):
        """From here on the host drives (selections are to be recorded, or the units outgrew their budget): the state moves
        over as export_state / load_state move it, the policies stay, and the slots they hand out are filled."""
        policy, stats, length, timing = self.policy, self.stats, self.length, (self._timing_cap, self._timing_stride)
        units, per, n = self._chunks, self._chunk_units, self.num_global_block
        state = self.export_state(with_units=False)
        state["units"] = None
        self._drop_resident()
        self.initialized, self.length = False, 0
        self._load(state, resident=False, unit_at=lambda u: units[u // per][u % per])
        self._policy, self._stats = policy, stats
        for u, pol in enumerate(policy):
            if self.record_trace and pol.evicted_log is None:
                pol.evicted_log = []
            self._caches[u] = pol.handle
            for unit, slot in pol.slot_of.items():
                home = units[unit // per][unit % per, u]
                self.slab[u, slot] = _widen(home, self.dim_head) if self.head_width != home.shape[-1] else home
        torch.cuda.synchronize(self.device)
        assert self.length == length and self.num_global_block == n

    def _append_resident(self, q, k, v, n, by_token=False):
        """One append() call on resident units; None when the units no longer fit (nothing has been done then)."""
        rc, length = self._rc, self.length
        units = max(0, (length + n - self.n_init - self.n_local) // self.block_size)
        if units > len(self._chunks) * self._chunk_units and not self._add_chunks(units):
            return None
        if units > self.reps.shape[1]:
            self._grow_reps(units)
        stream = current_stream()
        if self._call_stream != stream:
            self._bind_resident_buffers(stream)
        if n > 1 and units > self.topk and (self._call_scores is None or self._call_scores.shape[2] < units):
            cols = max(-(-units // 256) * 256, 2 * (self._call_scores.shape[2] if self._call_scores is not None else 0))
            self._retire(self._call_scores)
            self._call_scores = torch.empty((-(-rc.max_tokens // self.exc_block_size), self.num_units, cols), dtype=torch.float32, device=self.device)
            rc.d_call_scores, rc.scores_cols = self._call_scores.data_ptr(), cols
        B, H, D = self.num_units, self.unit_size, self.head_width
        by_token = by_token and n > 1                            # (one token's rows lie the same either way)
        out = torch.empty((B, n, H, D) if by_token else (B, H, n, D), dtype=torch.bfloat16, device=q.device)
        (q, q_ptr, q_st), (k, k_ptr, k_st), (v, v_ptr, v_st) = _addressed(q), _addressed(k), _addressed(v)
        o_sh, o_sl = (D, H * D) if by_token else (n * D, D)
        _CALL_ROWS.pack_into(rc, 0, q_ptr, k_ptr, v_ptr, *q_st[:3], *k_st[:3], *v_st[:3], out.data_ptr(), n * H * D, o_sh, o_sl, n)
        with self._call_buf.lock:
            status = self._lib.infllm_resident_append(self._resident, self._rc_ref, stream)
        if status:
            check(status, "infllm_resident_append")
        self.length = length + n
        self.num_global_block = units
        self.init_len = min(self.n_init, max(self.length - self.n_local, 0))
        self.cursor = self.init_len + units * self.block_size
        if self.cache_strategy == "lru":
            self.load_count += -(-n // self.exc_block_size)
        return out.transpose(1, 2) if by_token else out

    def _bind_resident_buffers(self, stream):
        """Workspaces of a call: dead between append() calls, so the managers that work on one stream share one set; the set's
        lock keeps the launches of two threads' calls apart."""
        B, H, D, exc, T = self.num_units, self.unit_size, self.head_width, self.exc_block_size, self._rc.max_tokens
        blocks = -(-T // exc)
        part_rows = max(8, 2 * min(self._local_group, blocks)) * B * H * exc       # (at most two key splits of several blocks)
        key = ("resident", self._dev_index, stream, B, H, D, T, exc, self.n_local, self.topk, part_rows, self._part_rows2)
        buf = _CALL_BUFFERS.get(key)
        if buf is None:
            bf = dict(dtype=torch.bfloat16, device=self.device)
            f32 = dict(dtype=torch.float32, device=self.device)
            f16 = dict(dtype=torch.float16, device=self.device)
            buf = _Buffers(q_loc=torch.empty((B * H * T * D,), **bf), q_glb=torch.empty((B * H * T * D,), **bf),
                           qpart=torch.empty((B * ((T + 15) // 16) * H * D,), **f32), qbar=torch.empty((blocks * B * H * D,), **f32),
                           o_part=torch.empty((part_rows * D,), **f16), lse_part=torch.empty((part_rows,), **f32),
                           o_part2=torch.empty((self._part_rows2 * D,), **f16), lse_part2=torch.empty((self._part_rows2,), **f32),
                           lse=torch.empty((B * H * max(T, exc),), **f32), logits=torch.empty((B * H * self.n_local,), **f32),
                           base=torch.empty((blocks * B * self.topk,), dtype=torch.int32, device=self.device),
                           ticket=torch.zeros((1,), dtype=torch.int32, device=self.device))
            buf.addresses = [("d_" + name, t.data_ptr()) for name, t in buf.items()]
            _CALL_BUFFERS[key] = buf
        self._call_buf = buf
        rc = self._rc
        for name, address in buf.addresses:
            setattr(rc, name, address)
        rc.part_rows, rc.part_rows2 = part_rows, self._part_rows2
        self._call_stream = stream
        self._streams.add(stream)

    # -------------------------------------------------------- the host drives
    def _init_host(self):
        B, H, Hkv, D, dev, cap = self.num_units, self.unit_size, self.unit_size_kv, self.head_width, self.device, self.ring_cap
        bs, exc, topk = self.block_size, self.exc_block_size, self.topk
        bf = dict(dtype=torch.bfloat16, device=dev)
        f32 = dict(dtype=torch.float32, device=dev)
        self.slab = torch.empty((B, self.max_cached_block, 2, Hkv, bs, D), **bf)
        self.host_chunks, self._host_base, self._host_dev_base = [], [], []
        self._chunk_base = (ctypes.c_uint64 * 64)()           # device-visible chunk addresses, as the native side reads them
        # workspaces of one execution block
        self.q_loc = torch.empty((2, B * H * exc * D), **bf)        # two slots: this block / the one prepared ahead
        self.q_glb = torch.empty((2, B * H * exc * D), **bf)
        self.qbar = torch.empty((2, B, H * D), **f32)
        self.qpart = torch.empty((2, B, (exc + 15) // 16, H * D), **f32)
        n_part = 2 * _MAX_SPLITS
        self.o_part = torch.empty((n_part * B * H * exc * D,), dtype=torch.float16, device=self.device)
        self.lse_part = torch.empty((n_part * B * H * exc,), **f32)
        self.lse = torch.empty((B * H * exc,), **f32)
        self.topk_idx = torch.zeros((B, max(topk, 1)), dtype=torch.int32, device=dev)
        self.topk_idx_host = torch.zeros((B, max(topk, 1)), dtype=torch.int32, pin_memory=True)
        page_bytes = ctypes.sizeof(_lib.Page)
        self.pages_dev = torch.empty((B * self.max_pages * page_bytes,), dtype=torch.uint8, device=dev)
        self.pages_host = torch.empty((_PAGE_SLOTS * B * self.max_pages * page_bytes,), dtype=torch.uint8, pin_memory=True)
        self.max_carve = (exc + self.n_init) // bs + 2
        self.carve_stage = torch.empty((_CARVE_SLOTS, self.max_carve, B, 2, Hkv, bs, D), **bf)

        d = LayerDesc()
        d.B, d.H, d.Hkv = B, H, Hkv
        d.n_local, d.n_init, d.block_size, d.exc = self.n_local, self.n_init, bs, exc
        d.topk, d.repr_topk, d.max_cached = topk, self.repr_topk, self.max_cached_block
        d.max_splits, d.num_cus, d.ring_cap = _MAX_SPLITS, _NUM_CUS, cap
        d.d_ring_k_raw, d.d_ring_k_rot = self.ring_k_raw.data_ptr(), self.ring_k_rot.data_ptr()
        d.d_ring_v, d.d_ring_score = self.ring_v.data_ptr(), self.ring_score.data_ptr()
        d.d_init_kv, d.init_cap, d.d_slab = self.init_kv.data_ptr(), self.init_kv.shape[3], self.slab.data_ptr()
        d.d_q_loc, d.d_q_glb, d.d_qbar = self.q_loc.data_ptr(), self.q_glb.data_ptr(), self.qbar.data_ptr()
        d.d_qpart = self.qpart.data_ptr()
        d.d_o_part, d.d_lse_part, d.d_lse = self.o_part.data_ptr(), self.lse_part.data_ptr(), self.lse.data_ptr()
        # the top-k kernel writes the ids straight into pinned host memory (no copy in the chain)
        d.d_topk_idx = self._lib.infllm_host_device_pointer(self.topk_idx_host.data_ptr())
        d.h_topk_idx = None
        if not d.d_topk_idx:
            d.d_topk_idx, d.h_topk_idx = self.topk_idx.data_ptr(), self.topk_idx_host.data_ptr()
        else:                                      # the host polls a sequence number stored behind the ids
            self.topk_flag_host = torch.zeros((16,), dtype=torch.int32, pin_memory=True)
            d.d_topk_flag = self._lib.infllm_host_device_pointer(self.topk_flag_host.data_ptr())
            d.h_topk_flag = self.topk_flag_host.data_ptr() if d.d_topk_flag else None
        d.d_pages, d.h_pages = self.pages_dev.data_ptr(), self.pages_host.data_ptr()
        d.max_pages, d.page_slots = self.max_pages, _PAGE_SLOTS
        d.d_carve_stage, d.max_carve, d.carve_slots = self.carve_stage.data_ptr(), self.max_carve, _CARVE_SLOTS
        d.d_inv_freq = self.inv_freq.data_ptr()
        d.distance_scale = float(self.position_embedding.distance_scale)
        d.softmax_scale = 1.0 / (self.dim_head ** 0.5)
        self._layer = self._lib.infllm_layer_create(ctypes.byref(d))
        if not self._layer:
            raise _lib.InfLLMHipError("infllm_layer_create failed: " + (self._lib.infllm_last_error() or b"").decode())
        if self._timing_cap:
            check(self._lib.infllm_layer_timing(self._layer, self._timing_cap, self._timing_stride), "infllm_layer_timing")
        # argument blocks and host arrays reused by every block
        self._fa, self._ba = FrontArgs(), BackArgs()
        self._sel_slots = (ctypes.c_int32 * (B * max(topk, 1)))()
        self._miss_row = (ctypes.c_int32 * (B * max(topk, 1)))()
        self._miss_slot = (ctypes.c_int32 * (B * max(topk, 1)))()
        self._miss_unit = (ctypes.c_int32 * (B * max(topk, 1)))()
        self._miss_src = (ctypes.c_void_p * (B * max(topk, 1)))()
        self._carve_dst = (ctypes.c_void_p * self.max_carve)()
        ba = self._ba
        ba.h_sel_slots = ctypes.addressof(self._sel_slots)
        ba.h_miss_row, ba.h_miss_slot = ctypes.addressof(self._miss_row), ctypes.addressof(self._miss_slot)
        ba.h_miss_unit = ctypes.addressof(self._miss_unit)
        ba.h_miss_src, ba.h_carve_dst = ctypes.addressof(self._miss_src), ctypes.addressof(self._carve_dst)
        if self.cache_strategy == "lru-s":
            # context_manager.py:454-470: per-unit attention mass of every block, read back by the host
            self.mass_host = torch.zeros((B, max(topk, 1)), dtype=torch.float32, pin_memory=True)
            self.mass_scratch = torch.empty((B, max(topk, 1), H, bs), **f32)
            ba.d_unit_mass = self._lib.infllm_host_device_pointer(self.mass_host.data_ptr())
            if not ba.d_unit_mass:
                raise _lib.InfLLMHipError("pinned host memory is not device-mapped: " + (self._lib.infllm_last_error() or b"").decode())
            ba.d_mass_scratch = self.mass_scratch.data_ptr()
        # selection -> cache policy -> fetch runs natively (infllm_block_select) on these arrays
        n_ids = B * max(topk, 1)
        self._sel_ids = (ctypes.c_int32 * n_ids)()
        self._evicted = (ctypes.c_int32 * n_ids)()
        self._n_evicted, self._n_miss_row = (ctypes.c_int32 * B)(), (ctypes.c_int32 * B)()
        self._caches = (ctypes.c_void_p * B)(*[pol.handle for pol in self._policy])
        sa = self._sa = _lib.SelectArgs()
        sa.caches = ctypes.addressof(self._caches)
        sa.h_chunk_base, sa.n_chunks, sa.units_per_chunk = ctypes.addressof(self._chunk_base), 0, _HOST_CHUNK_UNITS
        sa.unit_bytes, sa.row_bytes = self.unit_bytes, self.slot_bytes
        sa.h_sel_slots = ba.h_sel_slots
        sa.h_miss_row, sa.h_miss_slot, sa.h_miss_unit, sa.h_miss_src = ba.h_miss_row, ba.h_miss_slot, ba.h_miss_unit, ba.h_miss_src
        sa.h_evicted, sa.h_n_evicted, sa.h_n_miss = (ctypes.addressof(self._evicted), ctypes.addressof(self._n_evicted),
                                                      ctypes.addressof(self._n_miss_row))
        self._sa_ref = ctypes.byref(sa)
        self._fa_ref, self._ba_ref = ctypes.byref(self._fa), ctypes.byref(self._ba)
        self._bind_reps()

    def _bind_call_buffers(self, stream):
        """Buffers of a call prepared in one go: the rotated queries of up to call_tokens tokens, the blocks' mean
        queries and the local stage's partial rows.  They are dead between append() calls, so the layers that work on
        one stream share one set; the set's lock keeps the launches of two threads' calls apart."""
        B, H, D, exc, T = self.num_units, self.unit_size, self.head_width, self.exc_block_size, self._call_tokens
        group = self._local_group
        blocks = max(8, 4 * group)            # partial rows: two groups of blocks, up to two key splits each
        key = (self._dev_index, stream, B, H, D, T, exc, blocks)
        buf = _CALL_BUFFERS.get(key)
        if buf is None:
            bf = dict(dtype=torch.bfloat16, device=self.device)
            f32 = dict(dtype=torch.float32, device=self.device)
            buf = _Buffers(
                q_loc=torch.empty((B, H, T, D), **bf), q_glb=torch.empty((B, H, T, D), **bf),
                qpart=torch.empty((B, (T + 15) // 16, H * D), **f32), qbar=torch.empty((T // exc, B, H * D), **f32),
                o_part=torch.empty((blocks * B * H * exc, D), dtype=torch.float16, device=self.device),
                lse_part=torch.empty((blocks * B * H * exc,), **f32))
            _CALL_BUFFERS[key] = buf
        self._call_buf = buf
        bd = _lib.BatchDesc()
        bd.d_q_loc, bd.d_q_glb = buf["q_loc"].data_ptr(), buf["q_glb"].data_ptr()
        bd.d_qpart, bd.d_qbar = buf["qpart"].data_ptr(), buf["qbar"].data_ptr()
        bd.d_o_part, bd.d_lse_part = buf["o_part"].data_ptr(), buf["lse_part"].data_ptr()
        bd.part_rows, bd.max_tokens, bd.group_blocks = blocks * B * H * exc, T, group
        check(self._lib.infllm_layer_set_batch(self._layer, ctypes.byref(bd)), "infllm_layer_set_batch")
        self._call_stream = stream

    def size(self, *args, **kwargs):
        return self.length

    # ------------------------------------------------------------ host memory
    def _host_unit_addr(self, unit):
        """Address of the pinned host copy [B, 2, Hkv, bs, D] of a unit."""
        chunk, idx = divmod(unit, _HOST_CHUNK_UNITS)
        while chunk >= len(self.host_chunks):
            t = torch.empty((_HOST_CHUNK_UNITS, self.num_units, 2, self.unit_size_kv, self.block_size, self.head_width),
                            dtype=torch.bfloat16, pin_memory=True)
            self.host_chunks.append(t)
            self._host_base.append(t.data_ptr())
            dev = self._lib.infllm_host_device_pointer(t.data_ptr())       # address the fetch kernel reads through
            if not dev:
                raise _lib.InfLLMHipError((self._lib.infllm_last_error() or b"").decode())
            self._host_dev_base.append(dev)
            if len(self._host_dev_base) > len(self._chunk_base):
                grown = (ctypes.c_uint64 * (2 * len(self._chunk_base)))()
                grown[:len(self._chunk_base)] = self._chunk_base[:]
                self._chunk_base = grown
                self._sa.h_chunk_base = ctypes.addressof(grown)
            self._chunk_base[len(self._host_dev_base) - 1] = dev
            self._sa.n_chunks = len(self._host_dev_base)
        return self._host_base[chunk] + idx * self.unit_bytes

    def _host_unit_rows(self, unit):
        chunk, idx = divmod(unit, _HOST_CHUNK_UNITS)
        return self.host_chunks[chunk][idx]

    def _finish_host_copies(self):
        """append() leaves the copy of the units it carved last to their pinned home in flight; this sees it through."""
        if self._host_copies_open and self._layer:
            check(self._lib.infllm_layer_flush(self._layer, self._copy_raw), "infllm_layer_flush")
            torch.cuda.synchronize(self.device)            # (the copy-stream form of that copy is only ordered by its stream)
            self._host_copies_open = False

    def host_unit(self, unit):
        """Pinned host tensor [B, 2, Hkv, bs, D] of a carved unit (K at index 0, V at 1); a copy where the unit is resident in
        HBM, and for heads narrower than 128 one with the real dimensions picked out."""
        if self._resident:
            t = self._chunks[unit // self._chunk_units][unit % self._chunk_units]
            host = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
            return _narrow(host.copy_(t), self.dim_head) if t.shape[-1] != self.dim_head else host.copy_(t)
        self._finish_host_copies()
        return _narrow(self._host_unit_rows(unit), self.dim_head)

    def rep_rows(self, row, lo, hi):
        """Representatives of units [lo, hi) of batch row `row` as a CPU fp32 tensor [hi - lo, H * D]."""
        r = self.reps[row, lo:hi].view(hi - lo, self.unit_size, self.head_width)
        return self._own_width(r).reshape(hi - lo, -1).float().cpu()

    def _own_width(self, t):
        """rows of head_width elements -> rows of the heads' own width"""
        return t if t.shape[-1] == self.dim_head else _narrow(t, self.dim_head)

    # ----------------------------------------------------------------- timing
    def enable_timing(self, capacity, stride=1):
        """Event-time every `stride`-th local / global stage launch (up to `capacity` of each) for benchmarks."""
        self._timing_cap, self._timing_stride = capacity, stride
        if self._layer:
            check(self._lib.infllm_layer_timing(self._layer, capacity, stride), "infllm_layer_timing")
        if self._resident:
            check(self._lib.infllm_resident_timing(self._resident, capacity, stride), "infllm_resident_timing")

    def prefetch_stats(self):
        """(guesses made, guesses that turned out to be the selection) of the fetch ahead of the selection."""
        issued, confirmed = ctypes.c_int64(0), ctypes.c_int64(0)
        if self._layer:
            check(self._lib.infllm_layer_prefetch_stats(self._layer, ctypes.byref(issued), ctypes.byref(confirmed)),
                  "infllm_layer_prefetch_stats")
        return issued.value, confirmed.value

    def staged_units(self):
        """Missed units that were copied from a carve staging slot instead of coming from pinned host memory."""
        return int(self._lib.infllm_layer_staged_units(self._layer)) if self._layer else 0

    def path_counts(self):
        """Which interchangeable paths this layer's blocks took (infllm_layer_path_counts)."""
        counts = (ctypes.c_int64 * 6)()
        if self._layer:
            check(self._lib.infllm_layer_path_counts(self._layer, counts), "infllm_layer_path_counts")
        if self._resident:
            self._resident_books(False)
            counts[5] = self._state[8]
        return dict(zip(("tables_inline", "tables_kernel", "tables_upload", "score_merged", "score_apart", "call_ranked"),
                        (int(c) for c in counts)))

    def fetched_units(self):
        """Units moved from pinned host memory to the device cache so far (wrongly guessed ones and repairs included)."""
        return int(self._lib.infllm_layer_fetched_units(self._layer)) if self._layer else 0

    def read_timing(self, which):
        """[(ms, n_queries, n_keys)] of the timed launches; which = 0 local stage, 1 global stage."""
        cap = self._timing_cap
        ms, nq, nk = (ctypes.c_float * cap)(), (ctypes.c_int32 * cap)(), (ctypes.c_int32 * cap)()
        n = (self._lib.infllm_resident_read_timing(self._resident, which, ms, nq, nk, cap) if self._resident
             else self._lib.infllm_layer_read_timing(self._layer, which, ms, nq, nk, cap))
        if n < 0:
            check(n, "infllm_layer_read_timing")
        return [(ms[i], nq[i], nk[i]) for i in range(n)]

    # -------------------------------------------------------- one exec block
    def _block(self, st, n, out_ptr, n_next, preselected=None):
        lib, layer, fa, ba = self._lib, self._layer, self._fa, self._ba
        B, bs, topk = self.num_units, self.block_size, self.topk
        b0 = self.length + st
        b1 = b0 + n
        N = self.num_global_block
        fa.d_q = self._q_ptr + st * self._q_step
        fa.d_k = self._k_ptr + st * self._k_step
        fa.d_v = self._v_ptr + st * self._v_step
        fa.n, fa.n_units, fa.b0 = n, N, b0
        fa.n_next = n_next
        fa.flags = ba.flags = _lib.NO_RETRIEVAL if preselected is not None else 0
        if n_next:
            fa.d_q_next = fa.d_q + n * self._q_step
            fa.d_k_next = fa.d_k + n * self._k_step
            fa.d_v_next = fa.d_v + n * self._v_step
        rc = lib.infllm_block_front(layer, self._fa_ref, self._main_raw)
        if rc:
            check(rc, "infllm_block_front")
        # ---- retrieval result (context_manager.py:366-383) -> cache policy (495-515) -> fetch, in one native call:
        #      this stretch is on the chain from one block's selection to the next, the rest of the host's work is not
        sa = self._sa
        stats = self._stats
        if self._mass_units is not None:                     # lru-s: the previous block's masses decide this eviction
            check(lib.infllm_layer_wait_mass(layer), "infllm_layer_wait_mass")
            masses = self.mass_host.tolist()
            for u in range(B):
                self._policy[u].add_scores(self._mass_units[u], masses[u][:len(self._mass_units[u])])
            self._mass_units = None
        # ---- state machine after the block (context_manager.py:614-679): it does not depend on the selection, so the
        #      arguments of the block's second half are ready before the host waits for the ids
        cursor, init_len = self.cursor, self.init_len
        live = b1 - cursor
        take = 0
        if init_len < self.n_init and live > self.n_local:
            take = min(self.n_init - init_len, live - self.n_local)
            live -= take
        c = max((live - self.n_local) // bs, 0)
        ba.n, ba.b0 = n, b0
        ba.init_len, ba.cursor = init_len, cursor
        ba.d_out = out_ptr
        ba.init_take, ba.n_carve, ba.n_units = take, c, N
        idx_out = None
        if c:
            if N + c > self.reps.shape[1]:
                self._grow_reps(N + c)
            ba.d_rep_out = self._reps_ptr + N * self._rep_su_bytes
            for i in range(c):
                self._carve_dst[i] = self._host_unit_addr(N + i)
            if self.record_trace:
                idx_out = torch.empty((B, c, self.unit_size, self.repr_topk), dtype=torch.int32, device=self.device)
            ba.d_repr_idx = idx_out.data_ptr() if idx_out is not None else None
        if self.select_in_steps:
            n_sel, n_miss, selected = self._select_stepwise(preselected, N)
            ba.n_sel, ba.n_miss = n_sel, n_miss
            rc = lib.infllm_block_back(layer, self._ba_ref, self._main_raw, self._copy_raw)
            if rc:
                check(rc, "infllm_block_back")
        else:
            if preselected is not None or N <= topk:
                # chosen for the whole chunk (context_manager.py:381-382), or every unit there is
                selected = preselected if preselected is not None else [list(range(N))] * B
                n_sel = len(selected[0])
                for u in range(B):
                    self._sel_ids[u * n_sel:(u + 1) * n_sel] = selected[u]
                sa.h_selected, sa.n_sel, sa.wait_topk = ctypes.addressof(self._sel_ids), n_sel, 0
            else:
                n_sel = topk
                sa.h_selected, sa.n_sel, sa.wait_topk = self.topk_idx_host.data_ptr(), n_sel, 1   # the one host wait of a block
                selected = None                                   # read back below, off the chain
            ba.n_sel = n_sel
            # selection -> policy -> fetch, then the block's second half at once: next to nothing of the interpreter sits
            # between the arrival of the ids and the launch of the global stage (one native call for both measured no faster)
            n_miss = lib.infllm_block_select(layer, self._sa_ref, self._main_raw, self._copy_raw)
            if n_miss < 0:
                check(n_miss, "infllm_block_select")
            ba.n_miss = n_miss
            rc = lib.infllm_block_back(layer, self._ba_ref, self._main_raw, self._copy_raw)
            if rc:
                check(rc, "infllm_block_back")
            if selected is None and (self.record_trace or self.cache_strategy == "lru-s"):
                # from the library's copy: the pinned ids belong to the next selection once the second half is enqueued
                got = lib.infllm_layer_last_selection(layer, self._sel_ids, len(self._sel_ids))
                if got != B * n_sel:
                    check(min(got, -1), "infllm_layer_last_selection")
                selected = [self._sel_ids[u * n_sel:(u + 1) * n_sel] for u in range(B)]
            stats["evictions"] += sum(self._n_evicted[:B])
            for u in range(B):
                if self._policy[u].evicted_log is not None:
                    self._policy[u].evicted_log.append(list(self._evicted[u * n_sel:u * n_sel + self._n_evicted[u]]))
        stats["hits"] += B * n_sel - n_miss
        stats["misses"] += n_miss
        if self.cache_strategy == "lru":
            self.load_count += 1
        if n_next and preselected is None and self.fetch_ahead and not self.select_in_steps and self.cache_strategy != "lru-s":
            sa.n_sel = topk
            rc = lib.infllm_block_prefetch(layer, self._sa_ref, self._main_raw, self._copy_raw)
            if rc < 0:
                check(rc, "infllm_block_prefetch")
        if self.cache_strategy == "lru-s" and n_sel:
            self._mass_units = selected
        if self.record_trace:
            self.trace_blocks.append(dict(b0=b0, b1=b1, selected=[sorted(s) for s in selected], order=[list(s) for s in selected],
                                          n_units=N, init_len=init_len))
            if c:
                self.trace_units.append((N, c, idx_out))
        stats["blocks"] += 1
        self.init_len = init_len + take
        self.cursor = cursor + take + c * bs
        self.num_global_block = N + c

    def _select_stepwise(self, preselected, N):
        """The same as infllm_block_select in the separate steps the C ABI also offers (a caller with a policy of
        its own would use them): wait for the ids, one infllm_cache_touch per row, build the lists, issue the fetch."""
        lib, layer, B = self._lib, self._layer, self.num_units
        if preselected is not None:
            selected = preselected
        elif N <= self.topk:
            selected = [list(range(N))] * B
        else:
            check(lib.infllm_layer_wait_topk(layer), "infllm_layer_wait_topk")
            selected = self.topk_idx_host.tolist()
        n_sel, n_miss = len(selected[0]), 0
        for u in range(B):
            pol = self._policy[u]
            misses, evicted = pol.touch(selected[u])
            self._stats["evictions"] += len(evicted)
            slot_of = pol.slot_of
            for i, unit in enumerate(selected[u]):
                self._sel_slots[u * n_sel + i] = slot_of[unit]
            for unit in misses:
                chunk, idx = divmod(unit, _HOST_CHUNK_UNITS)
                self._miss_row[n_miss], self._miss_slot[n_miss], self._miss_unit[n_miss] = u, slot_of[unit], unit
                self._miss_src[n_miss] = self._host_dev_base[chunk] + idx * self.unit_bytes + u * self.slot_bytes
                n_miss += 1
        check(lib.infllm_block_fetch(layer, n_miss, self._miss_row, self._miss_slot, self._miss_unit, self._miss_src,
                                     self._main_raw, self._copy_raw), "infllm_block_fetch")
        return n_sel, n_miss, selected

    def _chunk_topk(self, q, c0, c1):
        """Selections of every execution block of q[:, :, c0:c1] against the units that exist now
        (get_batched_topk, context_manager.py:548-612); one host wait for the whole chunk."""
        B, N, topk, exc = self.num_units, self.num_global_block, self.topk, self.exc_block_size
        n_blocks = -(-(c1 - c0) // exc)
        if N <= topk:
            return [[list(range(N))] * B for _ in range(n_blocks)]
        C = self.unit_size * self.head_width
        qbar = torch.empty((B, n_blocks, C), dtype=torch.float32, device=self.device)
        check(self._lib.infllm_chunk_qbar(q.data_ptr() + c0 * q.stride(2) * 2, q.stride(0), q.stride(1), q.stride(2), B,
                                          self.unit_size, c1 - c0, exc, self.inv_freq.data_ptr(),
                                          float(self.position_embedding.distance_scale), self.n_local - 1,
                                          qbar.data_ptr(), self._main_raw), "infllm_chunk_qbar")
        # every block's mean query over the same units: the representatives are read once per eight blocks
        scores = torch.empty((n_blocks, N), dtype=torch.float32, device=self.device)
        idx = torch.empty((n_blocks, B, topk), dtype=torch.int32, device=self.device)
        for u in range(B):
            rc = self._lib.infllm_score_topk_queries(self.reps[u].data_ptr(), self.reps.stride(1), N, C, qbar[u].data_ptr(), qbar.stride(1),
                                                     n_blocks, topk, scores.data_ptr(), scores.stride(0), idx[:, u].data_ptr(),
                                                     idx.stride(0), self._main_raw)
            if rc == 1:                                      # row lengths without that kernel: one block at a time
                for j in range(n_blocks):
                    check(self._lib.infllm_score_topk(self.reps[u].data_ptr(), self.reps.stride(1), N, C, qbar[u, j].data_ptr(),
                                                      topk, scores.data_ptr(), idx[j, u].data_ptr(), self._main_raw),
                          "infllm_score_topk")
            else:
                check(rc, "infllm_score_topk_queries")
        return idx.cpu().tolist()

    def _grow_reps(self, need):
        B, N = self.num_units, self.num_global_block
        rows = max(2 * self.reps.shape[1], need)
        grown = torch.empty((B, rows, self.reps.shape[2]), dtype=torch.bfloat16, device=self.device)
        grown[:, :N] = self.reps[:, :N]
        scores = torch.empty((B, rows), dtype=torch.float32, device=self.device)
        scores[:, :N] = self.unit_scores[:, :N]          # scores prepared ahead for the next block
        self._retire(self.reps, self.unit_scores)
        self.reps, self.unit_scores = grown, scores
        self._bind_resident_reps() if self._resident else self._bind_reps()

    def _bind_reps(self):
        fa, ba = self._fa, self._ba
        self._reps_ptr = self.reps.data_ptr()
        self._rep_su_bytes = self.reps.stride(1) * 2
        fa.d_reps, fa.rep_sb, fa.rep_su = self._reps_ptr, self.reps.stride(0), self.reps.stride(1)
        fa.d_unit_scores, fa.unit_scores_sb = self.unit_scores.data_ptr(), self.unit_scores.stride(0)
        ba.rep_sb, ba.rep_su = self.reps.stride(0), self.reps.stride(1)
        ba.d_reps, ba.d_unit_scores, ba.unit_scores_sb = fa.d_reps, fa.d_unit_scores, fa.unit_scores_sb

    # ----------------------------------------------------------------- append
    def append(self, local_q, local_k, local_v, global_q, global_k, global_v):
        """The next tokens of the stream: their output rows [B, H, n, D], contiguous (unless ``rows_by_token`` was set)."""
        by_token, self.rows_by_token = self.rows_by_token, False
        if not (global_q is local_q and global_k is local_k and global_v is local_v):
            if not (global_q.data_ptr() == local_q.data_ptr() and global_k.data_ptr() == local_k.data_ptr()
                    and global_v.data_ptr() == local_v.data_ptr()):
                raise ValueError("local and global q/k/v must be the same tensors (as inf_llm_forward passes them)")
        q, k, v = local_q, local_k, local_v
        bf, dev = torch.bfloat16, q.device                      # (the native calls take addresses: nothing behind here checks them)
        if q.dtype is not bf or k.dtype is not bf or v.dtype is not bf:
            raise TypeError(f"the HIP path computes in bfloat16; got {q.dtype}, {k.dtype}, {v.dtype}")
        if k.device != dev or v.device != dev:
            raise ValueError(f"q, k and v must be on one device, got {dev}, {k.device}, {v.device}")
        batch_size, heads, input_length, width = q.shape
        kv_shape = k.shape
        t0, heads_kv, t2, t3 = kv_shape
        assert t0 == batch_size and t2 == input_length and t3 == width and v.shape == kv_shape, "q, keys and values differ in shape"
        assert q.is_cuda
        units, unit_heads, unit_heads_kv = batch_size, heads, heads_kv
        if self.perhead:                                        # context_manager.py:690-704
            rep = lambda t: (t.reshape(batch_size, heads_kv, 1, input_length, -1)
                              .expand(batch_size, heads_kv, heads // heads_kv, input_length, -1)
                              .reshape(batch_size * heads, 1, input_length, -1))
            q, k, v = q.reshape(batch_size * heads, 1, input_length, -1), rep(k), rep(v)
            units, unit_heads, unit_heads_kv = batch_size * heads, 1, 1
        if not self.initialized:
            self.dim_head = width
            check_head_dim(width)
            self._init(q, k)
        elif width != self.dim_head:
            raise ValueError(f"head_dim changed from {self.dim_head} to {width}")
        if self._resident and not self._wants_resident():
            self._leave_resident()
        if self.head_width != width:
            q, k, v = _widen(q, width), _widen(k, width), _widen(v, width)
        assert units == self.num_units and unit_heads == self.unit_size and unit_heads_kv == self.unit_size_kv

        if self._resident:
            out = self._append_resident(q, k, v, input_length, by_token)
            if out is not None:
                if self.head_width != width:
                    out = self._own_width(out)
                return out.reshape(batch_size, heads, input_length, -1) if self.perhead else out
            self._leave_resident()
            if self.head_width != q.shape[-1]:
                q, k, v = (_widen(t, self.dim_head) for t in (q, k, v))
        q, k, v = rows16(q), rows16(k), rows16(v)
        out = torch.empty((self.num_units, self.unit_size, input_length, self.head_width), dtype=torch.bfloat16, device=q.device)
        fa, ba = self._fa, self._ba
        fa.q_sb, fa.q_sh, fa.q_sl = q.stride(0), q.stride(1), q.stride(2)
        fa.k_sb, fa.k_sh, fa.k_sl = k.stride(0), k.stride(1), k.stride(2)
        fa.v_sb, fa.v_sh, fa.v_sl = v.stride(0), v.stride(1), v.stride(2)
        ba.o_sb, ba.o_sh, ba.o_sl = out.stride(0), out.stride(1), out.stride(2)
        self._q_ptr, self._k_ptr, self._v_ptr = q.data_ptr(), k.data_ptr(), v.data_ptr()
        self._q_step, self._k_step, self._v_step = q.stride(2) * 2, k.stride(2) * 2, v.stride(2) * 2
        main = torch.cuda.current_stream()
        self._main_raw = main.cuda_stream
        self._copy_raw = _SIDE_STREAM.cuda_stream if self.async_global_stream else self._main_raw
        if self._call_tokens and self._call_stream != self._main_raw:
            self._bind_call_buffers(self._main_raw)
        out_ptr, out_step = out.data_ptr(), out.stride(2) * 2
        exc = self.exc_block_size
        use_chunks = self.chunk_topk_calc is not None and input_length > 1      # context_manager.py:749-760
        if use_chunks:
            per_chunk = self.chunk_topk_calc // exc
            cuts = [i * exc for i in range(0, input_length // exc + 1, per_chunk)]
            if cuts[-1] < input_length:
                cuts.append(input_length)
            cut_i, plan, plan_pos = -1, None, 0
        shared = self._call_tokens and input_length > exc       # (a call of one block has workspaces of its own)
        with self._call_buf.lock if shared else contextlib.nullcontext():
            call_end = 0
            for st in range(0, input_length, exc):
                n = min(exc, input_length - st)
                if self._call_tokens and st == call_end:
                    # the next stretch of the call in one go: prologue, mean queries, first retrieval, local stage
                    call_end = min(st + self._call_tokens, input_length)
                    if self.length + call_end - self.cursor > self.ring_cap:
                        raise RuntimeError(f"a call of {call_end} tokens at {self.length} does not fit the rings "
                                           f"({self.ring_cap} rows, carving cursor {self.cursor})")
                    if call_end - st > exc:          # a single block (a decode step) gains nothing from being prepared apart
                        fa.d_q, fa.d_k, fa.d_v = (self._q_ptr + st * self._q_step, self._k_ptr + st * self._k_step,
                                                  self._v_ptr + st * self._v_step)
                        fa.n, fa.n_units, fa.b0 = call_end - st, self.num_global_block, self.length + st
                        fa.flags = _lib.NO_RETRIEVAL if use_chunks else 0
                        # room for every block's scores of the units there are and of those the call can carve
                        blocks, cols = -(-self._call_tokens // exc), self.num_global_block + (call_end - st) // self.block_size + 2
                        if self._call_scores is None or self._call_scores.shape[2] < cols or self._call_scores.shape[0] < blocks:
                            cols = max(-(-cols // 256) * 256, 2 * (self._call_scores.shape[2] if self._call_scores is not None else 0))
                            self._retire(self._call_scores)
                            self._call_scores = torch.empty((blocks, self.num_units, cols), dtype=torch.float32, device=self.device)
                        fa.d_call_scores, fa.call_scores_cols = self._call_scores.data_ptr(), self._call_scores.shape[2]
                        check(self._lib.infllm_call_front(self._layer, self._fa_ref, self._main_raw), "infllm_call_front")
                elif not self._call_tokens:
                    call_end = input_length
                chosen = None
                if use_chunks:
                    if cuts[cut_i + 1] < st + n:
                        cut_i += 1
                        plan, plan_pos = self._chunk_topk(q, cuts[cut_i], cuts[cut_i + 1]), 0
                    chosen = plan[plan_pos]
                    plan_pos += 1
                self._block(st, n, out_ptr + st * out_step, min(exc, call_end - st - n), chosen)
        self.length += input_length
        # (the last carved units go on to their pinned home in the background: _finish_host_copies before reading them)
        check(self._lib.infllm_layer_end_call(self._layer, self._copy_raw), "infllm_layer_end_call")
        self._host_copies_open = True
        out = self._own_width(out)
        if self.perhead:
            out = out.view(batch_size, heads, input_length, -1)
        return out

    # ------------------------------------------------------- state in / out
    # The reference keeps its state only in the live object (context_manager.py:292-363); these two
    # methods let a harness start from a prepared memory (e.g. 8192 units with representatives) or resume.
    def export_state(self, with_units=True):
        """Snapshot after an append(): everything a fresh ContextManager needs to continue the stream.
        with_units=False leaves the units out (4 GiB at a million tokens): host_unit(u) still reads them in place."""
        self._finish_host_copies()
        torch.cuda.synchronize()
        T, cur, cap = self.length, self.cursor, self.ring_cap
        rows = torch.arange(cur, T, device=self.device) % cap
        if with_units and self._resident and self.num_global_block:
            units = self._own_width(torch.cat([c.cpu() for c in self._chunks])[:self.num_global_block])
        else:
            units = [self.host_unit(u).clone() for u in range(self.num_global_block)] if with_units else []
            units = torch.stack(units) if units else None
        own, n = self._own_width, self.num_global_block
        reps = own(self.reps[:, :n].view(self.num_units, n, self.unit_size, self.head_width)).reshape(self.num_units, n, -1)
        return dict(length=T, n_units=n, init_len=self.init_len,
                    tail_k=own(self.ring_k_raw[:, :, rows]).clone(), tail_v=own(self.ring_v[:, :, rows]).clone(),
                    tail_score=self.ring_score[:, :, rows].clone(),
                    init_k=own(self.init_kv[:, 0, :, :self.init_len]).clone(),
                    init_v=own(self.init_kv[:, 1, :, :self.init_len]).clone(),
                    units=units, reps=reps.clone())

    def load_state(self, state):
        """Start from a prepared memory.  ``state``: length T; tail_k/tail_v [B,Hkv,T-cursor,D] (un-rotated,
        the tokens not carved yet, which include the local window); tail_score [B,H,T-cursor] fp32 or None;
        init_k/init_v [B,Hkv,init_len,D]; units [n_units,B,2,Hkv,bs,D] (any device) or None; reps
        [B,n_units,H*D].  The counts must satisfy the stream's closed forms (context_manager.py:614-679):
        init_len = min(n_init, max(T-n_local, 0)), n_units = max(0, (T-n_init-n_local)//block_size)."""
        return self._load(state)

    def _load(self, state, resident=None, unit_at=None):
        """load_state; unit_at(u): a unit in rows of any width, in place of state["units"]."""
        from .. import ops
        assert not self.initialized and self.length == 0, "load_state needs a fresh ContextManager"
        tail_k, tail_v = state["tail_k"], state["tail_v"]
        T = int(state["length"])
        B, Hkv, n_tail, D = tail_k.shape
        reps = state["reps"]
        H = reps.shape[2] // D if reps is not None and reps.numel() else state["tail_score"].shape[1] if state.get("tail_score") is not None else state["num_heads"]
        init_len = min(self.n_init, max(T - self.n_local, 0))
        n_units = max(0, (T - self.n_init - self.n_local) // self.block_size)
        cursor = init_len + n_units * self.block_size
        assert n_tail == T - cursor, f"tail holds {n_tail} tokens, the stream state needs {T - cursor}"
        assert state["init_k"].shape[2] == init_len and (n_units == 0 or unit_at is not None or state["units"].shape[0] == n_units)
        check_head_dim(D)
        self.dim_head = D
        q_like = torch.empty((B, H, 1, D), dtype=torch.bfloat16, device=tail_k.device)
        self._init(q_like, tail_k[:, :, :1], resident)
        if self._resident and n_units and not self._add_chunks(n_units):
            self._drop_resident()
            self._init(q_like, tail_k[:, :, :1], False)
        W = self.head_width
        wide = lambda t: t if t.shape[-1] == W else _widen(t, t.shape[-1])
        self.length, self.cursor, self.init_len = T, cursor, init_len
        if init_len:
            self.init_kv[:, 0, :, :init_len] = wide(state["init_k"])
            self.init_kv[:, 1, :, :init_len] = wide(state["init_v"])
        if n_units:
            self._grow_reps(n_units) if n_units > self.reps.shape[1] else None
            self.reps[:, :n_units] = wide(reps.view(B, n_units, H, D)).reshape(B, n_units, -1)
            if self._resident:
                for u in range(0, n_units, self._chunk_units):
                    n = min(self._chunk_units, n_units - u)
                    self._chunks[u // self._chunk_units][:n] = wide(state["units"][u:u + n])
            else:
                for u in range(n_units):
                    self._host_unit_addr(u)                        # allocates the pinned chunk
                    self._host_unit_rows(u).copy_(wide(state["units"][u] if unit_at is None else unit_at(u)))
            self.num_global_block = n_units
        # tail -> rings (RoPE at the absolute positions) in pieces of one execution block
        tail_k, tail_v = wide(tail_k), wide(tail_v)
        exc = self.exc_block_size
        zq = torch.zeros((B, H, exc, W), dtype=torch.bfloat16, device=self.device)
        for st in range(0, n_tail, exc):
            n = min(exc, n_tail - st)
            ops.ingest(zq[:, :, :n], tail_k[:, :, st:st + n], tail_v[:, :, st:st + n], cursor + st, self.n_local - 1,
                       self.inv_freq, float(self.position_embedding.distance_scale), self.ring_k_raw, self.ring_k_rot,
                       self.ring_v, self.ring_score, torch.empty_like(zq), torch.empty_like(zq))
        if state.get("tail_score") is not None:
            rows = torch.arange(cursor, T, device=self.device) % self.ring_cap
            self.ring_score[:, :, rows] = state["tail_score"].to(torch.float32)
        if self._resident:
            check(self._lib.infllm_resident_set_state(self._resident, T, cursor, init_len, n_units), "infllm_resident_set_state")
        torch.cuda.synchronize()
        return self

    # ----------------------------------------------------------------- tracing
    def trace_repr_indices(self):
        """{unit: int tensor [B, H, repr_topk]} of the keys chosen as representatives (needs record_trace)."""
        res = {}
        for first, count, idx in self.trace_units:
            host = idx.cpu()
            for i in range(count):
                res[first + i] = host[:, i]
        return res
