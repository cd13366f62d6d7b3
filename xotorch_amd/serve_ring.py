"""Single-node multi-GPU ring serving worker (launched via torchrun by
`xot serve --gpus N`).

The product serving path on MI355X: every rank holds one contiguous layer
shard (ring partitioning), activations hop rank→rank as resident bf16 over
RCCL/xGMI, and requests are served with SLOT-BASED CONTINUOUS BATCHING:

- the KV cache is allocated once with batch dim = SLOTS; each request is
  admitted into a free slot and decoded alongside the others (the reference
  serves one request at a time over per-request caches,
  /root/reference/xotorch/orchestration/node.py:145);
- one decode tick advances EVERY active slot by one token in a single
  hipGraph replay (per-slot positions / seq_lens are static device tensors
  the graph reads, so admission/release never re-captures);
- prompt prefill is CHUNKED through the ring (stage 0 forwards sequence
  chunks so later stages overlap instead of idling through the whole
  prompt — request-level TTFT); prompts that are equally far run as one
  padded batch where the model addresses slots by index;
- rank 0 hosts the FULL ChatGPT-compatible API (the same ChatGPTAPI as the
  elastic Node path — models/topology/tinychat/encode routes included) via
  a thin Node adapter.

Control plane per tick: rank 0 broadcasts a small header (op, slot or slot
bitmask, len or chunk start, milli-temperature); ADMIT is followed by the prompt tokens; the last stage
samples and broadcasts the per-slot tokens; rank 0 streams them to clients.
All collectives go through RingComm, so N ranks verify on fewer GPUs (gloo
staging) while the real deployment runs pure RCCL.
"""
from __future__ import annotations

import argparse
import asyncio
import os
import queue
import sys
import threading
import time
import uuid
from dataclasses import dataclass, field
from pathlib import Path
from typing import Dict, List, Optional

if __package__ in (None, ""):  # torchrun launches this file by path
  sys.path.insert(0, str(Path(__file__).resolve().parent.parent))

import torch
import torch.distributed as dist

from xotorch_amd import ops
from xotorch_amd.engine.kvcache import make_cache
from xotorch_amd.models.config import config_from_hf
from xotorch_amd.models.registry import builtin_config, get_repo, register_local_model
from xotorch_amd.models.weights import fast_random_init_gpu, load_shard_weights, random_init
from xotorch_amd.parallel.comm import RingComm, init_distributed
from xotorch_amd.parallel.ring import equal_ring_shards

OP_IDLE, OP_DECODE, OP_ADMIT, OP_RELEASE, OP_SHUTDOWN, OP_PREFILL = 0, 1, 2, 3, 4, 5

MAX_SEQ = int(os.getenv("XOT_SERVE_MAX_SEQ", "4096"))
SLOTS = int(os.getenv("XOT_SERVE_SLOTS", "8"))
PREFILL_CHUNK = int(os.getenv("XOT_SERVE_PREFILL_CHUNK", "256"))


@dataclass
class SlotState:
  request_id: Optional[str] = None
  prompt_len: int = 0
  generated: int = 0
  max_new: int = 0
  temp: float = 0.0
  done: bool = False  # finished but not yet released (release is its own tick)
  ttft_s: float = 0.0
  t_admit: float = 0.0


@dataclass
class AdmitMsg:
  request_id: str
  tokens: torch.Tensor  # [1, S] int64 cpu
  max_new: int
  temp: float
  t_submit: float = field(default_factory=time.perf_counter)


class RingSlotWorker:
  """One rank of the serving ring. Rank 0 drives the control loop."""

  def __init__(self, model_id: str, rank: int, world: int, device="cuda",
               dtype=torch.bfloat16, model_dir: Optional[str] = None,
               slots: int = SLOTS, max_seq: int = MAX_SEQ, use_graphs: bool = True):
    self.model_id = model_id
    self.rank, self.world = rank, world
    self.device, self.dtype = device, dtype
    if not 1 <= slots <= 63:
      raise ValueError(f"slots must be in [1, 63] (release op is an int64 bitmask), got {slots}")
    self.slots, self.max_seq = slots, max_seq
    self.use_graphs = use_graphs and device == "cuda"
    own = Path(model_dir) / "config.json" if model_dir else None
    self.cfg = config_from_hf(own if own is not None and own.exists() else builtin_config(model_id) or {}, model_id)
    self.max_seq = min(self.max_seq, self.cfg.max_seq_len)
    self.shard = equal_ring_shards(model_id, self.cfg.n_layers, world)[rank]
    from xotorch_amd.models import model_class_for
    model_cls = model_class_for(self.cfg)
    prev_dtype = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
      with torch.device("meta"):
        model = model_cls(self.cfg, self.shard)
    finally:
      torch.set_default_dtype(prev_dtype)
    model = model.to_empty(device=device).to(dtype)
    if model_dir:
      load_shard_weights(model, model_dir, device="cpu")
      model = model.to(device)
    elif device == "cuda" and self.cfg.dim >= 2048:
      fast_random_init_gpu(model)
    else:
      random_init(model)
    model.reset_rope()
    model.eval()
    self.model = model
    self.cache = make_cache(self.cfg, self.shard, slots, self.max_seq, dtype, device)
    # slot-indexed models address any set of slots in one step: their prompts
    # prefill in batches of unequal length and parked slots are skipped;
    # the others get views of one slot's cache rows
    self.slot_indexed = getattr(model, "slot_indexed", False)
    self.hid_dtype = getattr(model, "hidden_dtype", dtype)
    if device == "cuda":
      torch.cuda.empty_cache()
      model.pack_decode_weights(reserve_bytes=8 << 30)
    self.comm = RingComm(device)
    self.next_rank = (rank + 1) % world
    self.prev_rank = (rank - 1) % world
    self.is_first = self.shard.is_first_layer
    self.is_last = self.shard.is_last_layer

    D = self.cfg.hidden_dim
    dev = device
    # static per-slot state (graph-visible)
    self.positions = torch.zeros(slots, dtype=torch.int32, device=dev)
    self.seq_lens = torch.ones(slots, dtype=torch.int32, device=dev)
    self.tok_buf = torch.zeros(slots, 1, dtype=torch.int64, device=dev)
    self.hid_buf = torch.zeros(slots, 1, D, dtype=self.hid_dtype, device=dev)
    self.slot_map = torch.full((slots,), -1, dtype=torch.int32, device=dev)  # -1: parked
    self._mapped = [-1] * slots  # what slot_map holds
    self.logits_buf: Optional[torch.Tensor] = None
    self.hid_out: Optional[torch.Tensor] = None
    # control/broadcast buffers
    self.hdr = torch.zeros(4, dtype=torch.int64, device=dev)
    self.tok_bcast = torch.zeros(slots, dtype=torch.int64, device=dev)
    self.active = [False] * slots
    self.slot_state: List[SlotState] = [SlotState() for _ in range(slots)]
    self._graph: Optional[torch.cuda.CUDAGraph] = None
    self._pf: Dict[int, dict] = {}  # slot -> in-progress chunked prefill (every rank)
    self._pf_turn = False
    self.eos_token_id = self.cfg.eos_token_id

  # ---------------- decode tick ----------------

  def _decode_forward(self):
    x = self.tok_buf if self.is_first else self.hid_buf
    kw = {"slots": self.slot_map} if self.slot_indexed else {}
    out = self.model(x, caches=self.cache.caches, positions=self.positions,
                     start_pos=-1, is_decode=True, seq_lens=self.seq_lens, **kw)
    if self.is_last:
      if self.logits_buf is None:
        self.logits_buf = torch.empty_like(out)
      self.logits_buf.copy_(out)
    else:
      self.hid_out = out
    self.positions.add_(1)
    self.seq_lens.add_(1)

  def _build_graph(self):
    if not self.use_graphs:
      return
    self.positions.fill_(1)
    self.seq_lens.fill_(2)
    self.tok_buf.random_(0, self.cfg.vocab_size)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
      with torch.inference_mode():
        ops.load_library(self.device, self.dtype)
        for _ in range(2):
          self._decode_forward()
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.inference_mode():
      with torch.cuda.graph(g):
        self._decode_forward()
    self._graph = g
    self._reset_inactive()

  def _reset_inactive(self):
    """Park inactive slots on their own LAST cache row (max_seq-1): the
    decode graph appends garbage KV for every slot each tick, and the
    admission clamp (max_new <= max_seq - plen - 1) guarantees an active
    slot's attention never reads past row max_seq-2 — so the scratch row
    can take garbage writes without ever clobbering real prefill data
    (prerequisite for interleaving chunked prefill with decode ticks)."""
    idle = [i for i in range(self.slots) if not self.active[i]]
    if self.slot_indexed:
      mapped = [i if on else -1 for i, on in enumerate(self.active)]
      if mapped != self._mapped:
        self.slot_map.copy_(torch.tensor(mapped, dtype=torch.int32))
        self._mapped = mapped
    if idle:
      idx = torch.tensor(idle, dtype=torch.int64, device=self.positions.device)
      self.positions[idx] = self.max_seq - 1
      self.seq_lens[idx] = 1

  def run_decode(self):
    """This rank's part of a decode tick: every active slot one token on
    (tokens in tok_buf, logits to logits_buf), nothing sampled."""
    if self._graph is not None:
      self._graph.replay()
    else:
      self._decode_forward()

  def decode_tick(self):
    with torch.inference_mode():
      if not self.is_first and self.world > 1:
        self.comm.recv(self.hid_buf, self.prev_rank)
      self.run_decode()
      if not self.is_last and self.world > 1:
        self.comm.send(self.hid_out, self.next_rank)
      if self.is_last:
        self._sample_all()
      if self.world > 1:
        self.comm.broadcast(self.tok_bcast, self.world - 1)
      if self.is_first:
        self.tok_buf.copy_(self.tok_bcast.view(self.slots, 1))
      self._reset_inactive()

  def _sample_all(self):
    from xotorch_amd import ops
    logits = self.logits_buf  # [slots, V]
    greedy = logits.argmax(dim=-1)
    toks = greedy
    temps = [self.slot_state[i].temp for i in range(self.slots)]
    if any(t > 0 for t in temps):
      toks = greedy.clone()
      for i, t in enumerate(temps):
        if t > 0 and self.active[i]:
          toks[i] = ops.softmax_sample(logits[i:i + 1], temperature=t, top_k=35)[0]
    self.tok_bcast.copy_(toks)

  # ---------------- prefill (chunked through the ring) ----------------

  def _slot_caches(self, slot: int):
    out = []
    for layer in self.cache.caches:
      sl = tuple(t[slot:slot + 1] if t is not None else None for t in layer)
      out.append(type(layer)(*sl) if hasattr(layer, "_fields") else sl)
    return out

  def _prefill_hidden(self, group: List[int], c0: int, last_only: bool = True) -> torch.Tensor:
    """The chunk that starts at c0 of the prompts in `group` through this
    rank's layers, as one batch (slot-indexed models; else one prompt).
    Shorter rows are padded at the end. Returns logits on the last stage."""
    dev = self.device
    pfs = [self._pf[i] for i in group]
    lens = [min(PREFILL_CHUNK, pf["plen"] - c0) for pf in pfs]
    S = max(lens)
    kw = {}
    if self.slot_indexed:
      caches = self.cache.caches
      kw["slots"] = torch.tensor(group, dtype=torch.int32, device=dev)
      if min(lens) < S:
        kw["lens"] = torch.tensor(lens, dtype=torch.int32, device=dev)
    else:
      (slot,) = group
      caches = self._pf[slot]["caches"]
    pos = torch.arange(c0, c0 + S, dtype=torch.int32, device=dev)
    if self.is_first:
      x = torch.zeros(len(group), S, dtype=torch.int64, device=dev)
      for row, (pf, n) in enumerate(zip(pfs, lens)):
        x[row, :n] = pf["toks"][0, c0:c0 + n]
    else:
      x = torch.empty(len(group), S, self.cfg.hidden_dim, dtype=self.hid_dtype, device=dev)
      self.comm.recv(x, self.prev_rank)
    return self.model(x, caches=caches, positions=pos, start_pos=c0, last_only=last_only, **kw)

  def _prefill_group(self, group: List[int], c0: int) -> Dict[int, int]:
    """One chunk of the prompts in `group`; returns the first sampled token of
    every prompt that ends with it (last stage only)."""
    with torch.inference_mode():
      h = self._prefill_hidden(group, c0)
      if not self.is_last:
        if self.world > 1:
          self.comm.send(h.contiguous(), self.next_rank)
        return {}
      first = {}
      for row, slot in enumerate(group):
        if c0 + PREFILL_CHUNK < self._pf[slot]["plen"]:
          continue
        logits = h[row:row + 1, -1] if h.dim() == 3 else h[row:row + 1]
        st = self.slot_state[slot]
        if st.temp > 0:
          from xotorch_amd import ops
          first[slot] = int(ops.softmax_sample(logits, temperature=st.temp, top_k=35)[0])
        else:
          first[slot] = int(logits.argmax(dim=-1)[0])
      return first

  def _begin_prefill(self, slot: int, toks: torch.Tensor):
    """Hand a prompt [1, S] to a free slot; its chunks run in later ticks."""
    self._pf[slot] = {"toks": toks, "c0": 0, "plen": toks.shape[1],
                      "caches": None if self.slot_indexed else self._slot_caches(slot)}

  def _activate(self, slot: int):
    """A slot whose prompt is in the cache joins the decode ticks."""
    plen = self._pf.pop(slot)["plen"]
    self.positions[slot] = plen
    self.seq_lens[slot] = plen + 1
    self.slot_map[slot] = slot
    self._mapped[slot] = slot
    self.active[slot] = True

  def _release(self, slots: List[int]):
    """Give slots back; they are parked until their next prompt."""
    for i in slots:
      self.active[i] = False
      self.slot_state[i] = SlotState()
      self._pf.pop(i, None)
    self._reset_inactive()

  def _log_done(self, st: SlotState):
    dt = max(1e-9, time.perf_counter() - st.t_admit)
    print(f"[serve] {str(st.request_id)[:8]} done: prompt {st.prompt_len}, "
          f"{st.generated} tokens, TTFT {st.ttft_s * 1000:.0f} ms, "
          f"{st.generated / dt:.1f} tok/s", flush=True)

  # ---------------- control loop ----------------

  def _bcast_hdr(self, op=OP_IDLE, slot=0, plen=0, extra=0):
    if self.rank == 0:
      self.hdr[0], self.hdr[1], self.hdr[2], self.hdr[3] = op, slot, plen, extra
    if self.world > 1:
      self.comm.broadcast(self.hdr, 0)
    return [int(v) for v in self.hdr.cpu()]

  def cancel(self, request_id: str):
    """Mark a request for release (client went away). Thread-safe; consumed
    by the rank-0 control loop on its next tick."""
    self._cancelled.add(request_id)

  _cancelled: set = None  # set in serve_forever (rank 0)

  def serve_forever(self, admit_q: Optional["queue.Queue"] = None, emit=None,
                    idle_sleep: float = 0.002, max_ticks: Optional[int] = None):
    """Run the ring loop. On rank 0, `admit_q` provides AdmitMsg and `emit`
    receives (request_id, token, is_finished, meta). Followers pass None."""
    self._cancelled = set()
    self._pf.clear()
    self._pf_turn = False
    idle_ticks = 0
    pending_release: List[int] = []
    inflight: Dict[int, AdmitMsg] = {}
    ticks = 0
    while max_ticks is None or ticks < max_ticks:
      ticks += 1
      op, slot, plen, extra = OP_IDLE, 0, 0, 0
      if self.rank == 0:
        if self._cancelled:
          for i in range(self.slots):
            st = self.slot_state[i]
            if (self.active[i] or i in self._pf) and st.request_id in self._cancelled and not st.done:
              st.done = True
              if emit:
                emit(st.request_id, 0, True, {"cancelled": True})
              pending_release.append(i)
          self._cancelled.clear()
        if pending_release:
          # one RELEASE tick drains the whole backlog (slot = bitmask), so a
          # finished slot never sees another decode tick's KV advance
          op, slot = OP_RELEASE, sum(1 << i for i in set(pending_release))
          pending_release.clear()
        else:
          msg = None
          free = next((i for i in range(self.slots)
                       if not self.active[i] and i not in self._pf), None)
          if admit_q is not None and free is not None:
            try:
              msg = admit_q.get_nowait()
            except queue.Empty:
              msg = None
          if msg is not None and msg.tokens is None:  # shutdown sentinel
            op = OP_SHUTDOWN
          elif msg is not None:
            op, slot, plen = OP_ADMIT, free, msg.tokens.shape[1]
            extra = int(msg.temp * 1000)
            inflight[free] = msg
          elif self._pf and (self._pf_turn or not any(self.active)):
            # alternate one prompt chunk with one decode tick so slots that
            # are already generating keep emitting during long prefills
            lead = max(self._pf, key=lambda i: self._pf[i]["c0"])  # finish-first
            op, plen = OP_PREFILL, self._pf[lead]["c0"]
            # prompts that are equally far go together where the model can
            group = [i for i in self._pf if self._pf[i]["c0"] == plen] if self.slot_indexed else [lead]
            slot = sum(1 << i for i in group)
            self._pf_turn = False
          elif any(self.active):
            op = OP_DECODE
            self._pf_turn = True
          else:
            op = OP_IDLE
      op, slot, plen, extra = self._bcast_hdr(op, slot, plen, extra)

      if op != OP_IDLE:
        idle_ticks = 0
      if op == OP_SHUTDOWN:
        break
      if op == OP_IDLE:
        if self.rank == 0:
          # adaptive backoff: a long-idle ring stops burning control-plane
          # broadcasts (each idle tick is an NCCL op on every rank)
          idle_ticks += 1
          time.sleep(min(idle_sleep * (1 + idle_ticks // 50), 0.05))
        continue
      if op == OP_RELEASE:
        self._release([i for i in range(self.slots) if slot & (1 << i)])
        continue
      if op == OP_ADMIT:
        if self.rank == 0:
          msg = inflight[slot]
          toks = msg.tokens.to(self.device)
        else:
          toks = torch.zeros(1, plen, dtype=torch.int64, device=self.device)
        if self.world > 1:
          self.comm.broadcast(toks, 0)
        st = SlotState(prompt_len=plen, temp=extra / 1000.0)
        self.slot_state[slot] = st
        self._begin_prefill(slot, toks)
        if self.rank == 0:
          msg = inflight.pop(slot)
          st.request_id = msg.request_id
          st.max_new = min(msg.max_new, self.max_seq - plen - 1)
          st.t_admit = msg.t_submit
        continue
      if op == OP_PREFILL:
        group = [i for i in range(self.slots) if slot & (1 << i)]
        first = self._prefill_group(group, plen)
        done = []
        for i in group:
          self._pf[i]["c0"] = plen + PREFILL_CHUNK
          if self._pf[i]["c0"] >= self._pf[i]["plen"]:
            done.append(i)
        if not done:
          continue
        # last chunk: activate the slots and ship the first tokens to rank 0
        self.tok_bcast.zero_()
        for i, tok in first.items():
          self.tok_bcast[i] = tok
        if self.world > 1:
          self.comm.broadcast(self.tok_bcast, self.world - 1)
        for i in done:
          self._activate(i)
          if self.is_first:
            self.tok_buf[i, 0] = self.tok_bcast[i]
          if self.rank != 0:
            continue
          st = self.slot_state[i]
          st.generated = 1
          st.ttft_s = time.perf_counter() - st.t_admit
          tok = int(self.tok_bcast[i])
          fin = (self.eos_token_id is not None and tok == self.eos_token_id) or st.generated >= st.max_new
          if emit:
            emit(st.request_id, tok, fin, {"ttft_s": st.ttft_s})
          if fin:
            st.done = True
            self._log_done(st)
            pending_release.append(i)
        continue
      # OP_DECODE
      self.decode_tick()
      if self.rank == 0:
        toks = self.tok_bcast.cpu()
        for i in range(self.slots):
          st = self.slot_state[i]
          if not self.active[i] or st.request_id is None or st.done:
            continue
          tok = int(toks[i])
          st.generated += 1
          fin = (self.eos_token_id is not None and tok == self.eos_token_id) or st.generated >= st.max_new
          if emit:
            emit(st.request_id, tok, fin, {})
          if fin:
            st.done = True
            self._log_done(st)
            pending_release.append(i)
    return ticks


# ---------------- rank 0: asyncio API adapter ----------------

class _CallbackSystem:
  """Duck-typed AsyncCallbackSystem surface the API uses."""

  def __init__(self):
    from xotorch_amd.helpers import AsyncCallbackSystem
    self._cbs = AsyncCallbackSystem()

  def register(self, name):
    return self._cbs.register(name)

  def trigger_all(self, *a):
    self._cbs.trigger_all(*a)


class RingAPINode:
  """Node-shaped adapter over the ring worker: gives ChatGPTAPI the surface
  it needs (process_prompt / on_token / inference_engine / topology) while
  the actual decode runs in the ring thread."""

  def __init__(self, worker: RingSlotWorker, tokenizer, loop):
    self.worker = worker
    self.tokenizer = tokenizer
    self.loop = loop
    self.on_token = _CallbackSystem()
    self.admit_q: queue.Queue = queue.Queue()
    self.request_meta: Dict[str, dict] = {}
    # the API looks at node.inference_engine.{tokenizer, shard}
    self.inference_engine = type("E", (), {})()
    self.inference_engine.tokenizer = tokenizer
    self.inference_engine.shard = worker.shard
    self.server = None

  @property
  def current_topology(self):
    from xotorch_amd.parallel.topology import Topology, DeviceCapabilities, DeviceFlops
    topo = Topology()
    for r in range(self.worker.world):
      topo.update_node(f"rank{r}", DeviceCapabilities(
        model="MI355X ring stage", chip="gfx950", memory=288 * 1024,
        flops=DeviceFlops(fp32=0, fp16=2500.0, int8=0)))
      topo.add_edge(f"rank{r}", f"rank{(r + 1) % self.worker.world}", "xgmi")
    topo.active_node_id = "rank0"
    return topo

  def emit(self, request_id: str, token: int, finished: bool, meta: dict):
    if meta.get("ttft_s") is not None:
      self.request_meta[request_id] = meta
    self.loop.call_soon_threadsafe(self.on_token.trigger_all, request_id, [token], finished)

  def cancel_request(self, request_id: str):
    self.worker.cancel(request_id)

  async def process_prompt(self, shard, prompt: str, request_id=None, inference_state=None):
    request_id = request_id or str(uuid.uuid4())
    state = inference_state or {}
    if shard is not None and shard.model_id != self.worker.model_id:
      raise ValueError(
        f"this ring serves {self.worker.model_id}; requested {shard.model_id} "
        f"(restart `xot serve {shard.model_id}` to switch)")
    ids = self.tokenizer.encode(prompt) or [self.tokenizer.eos_token_id or 0]
    if len(ids) >= self.worker.max_seq:
      raise ValueError(f"prompt length {len(ids)} exceeds context {self.worker.max_seq}")
    tokens = torch.tensor([ids], dtype=torch.int64)
    max_new = int(state.get("max_tokens") or 256)
    temp = float(state.get("temperature") or 0.0)
    self.admit_q.put(AdmitMsg(request_id, tokens, max_new, temp))
    return request_id


def main():
  p = argparse.ArgumentParser()
  p.add_argument("--model", type=str, default="llama-3-8b")
  p.add_argument("--port", type=int, default=52415)
  p.add_argument("--model-dir", type=str, default=None)
  p.add_argument("--slots", type=int, default=SLOTS)
  p.add_argument("--no-graphs", action="store_true")
  args = p.parse_args()
  if args.model_dir:
    register_local_model(args.model, args.model_dir)  # the API resolves models by card
  rank, world = init_distributed()
  device = "cuda" if torch.cuda.is_available() else "cpu"
  dtype = torch.bfloat16 if device == "cuda" else torch.float32
  worker = RingSlotWorker(args.model, rank, world, device, dtype, args.model_dir,
                          slots=args.slots, use_graphs=not args.no_graphs)
  if device == "cuda":
    worker._build_graph()

  if rank != 0:
    worker.serve_forever()
    return

  from xotorch_amd.api.chatgpt import ChatGPTAPI
  from xotorch_amd.engine.tokenizers import DummyTokenizer, resolve_tokenizer

  loop = asyncio.new_event_loop()
  asyncio.set_event_loop(loop)
  try:
    tokenizer = loop.run_until_complete(
      resolve_tokenizer(args.model_dir or get_repo(args.model, "HIPEngine")))
  except Exception:
    tokenizer = DummyTokenizer()
  node = RingAPINode(worker, tokenizer, loop)
  ring_thread = threading.Thread(
    target=worker.serve_forever, args=(node.admit_q, node.emit), daemon=True)
  ring_thread.start()
  api = ChatGPTAPI(node, "TorchEngine", default_model=args.model)

  async def start():
    await api.run("0.0.0.0", args.port)
    print(f"ring server ({world} ranks, {args.slots} slots, graphs="
          f"{worker._graph is not None}) on :{args.port}", flush=True)
    await asyncio.Event().wait()

  loop.run_until_complete(start())


if __name__ == "__main__":
  main()
