"""Inter-stage transport for the layer-sharded pipeline.

The reference has NO inter-shard data plane (its "sharded" path runs shard 0 alone,
``worker/app.py:334-336``). Here a pipeline step moves over two planes:

* control plane (host): the head's packed ``StepMeta`` for every tick is written ONCE into a
  shared-memory broadcast ring (``csrc/runtime/shm_ring.cpp``, all stages of a pipeline
  live on one 8-GPU node) the moment the head schedules it; every stage reads it from the
  same pages, so a stage's host stages the metadata upload and enqueues its graph replay
  long before the activations arrive — no stage ever waits on its GPU to learn what to do
  next, and the head's cost per tick is one memcpy + one release store whatever N is.
  (Carrying the metadata inside the activation message instead would make every stage's
  host wait for its receive to land before it could even launch: a host<->GPU round trip
  per hop per tick.) A gloo fallback (``DLI_PP_CTRL=gloo``) serves ranks on different
  hosts;
* data plane (device): hidden states stage r -> r+1 and sampled token ids tail -> head go by
  RCCL point-to-point over xGMI (``torch.distributed`` backend "nccl" == RCCL on ROCm), one
  grouped send/recv per rank per tick, ordered on the GPU streams: the receive is a stream
  dependency of the consumer's graph replay, never a host wait. Receives land in buffers
  allocated once per engine (a decode step's hidden state goes straight into the stage
  runner's static graph input); sends read the producer's output in place (the next replay
  that would overwrite it is stream-ordered behind the send). On CPU (tests) the data plane
  is gloo as well.

Every stage learns the activation shape of tick k from tick k's metadata (rows = tokens of
the step, cols = hidden size), so the data plane carries no headers at all.
"""
from __future__ import annotations

import itertools
import logging
import os
import socket
import threading
import time
from datetime import timedelta
from typing import List, Optional, Sequence, Tuple

import numpy as np
import torch
import torch.distributed as dist

from ..engine.batch import HEADER_LEN
from ..utils import faults
from ..utils.tracing import trace_range

# header word indices (int64 units) beyond StepMeta's own first 9
H_TICK = 12
_HDR_BYTES = HEADER_LEN * 8
_ring_ids = itertools.count()
_log = logging.getLogger("dli.transport")


def data_plane_name(comm: str, nccl: bool) -> str:
    """The resolved data plane as records report it: ``ipc`` (device mailboxes; on a CPU
    rank their shared-memory host model, ``ipc-host``), ``rccl`` (comm.cpp's own
    communicator), ``torch-rccl`` / ``torch-gloo`` (torch.distributed point-to-point)."""
    if comm == "ipc":
        return "ipc" if nccl else "ipc-host"
    if comm == "rccl":
        return "rccl"
    return "torch-rccl" if nccl else "torch-gloo"


def ctrl_slot_bytes(max_seqs: int, max_tokens: int, table_width: int) -> int:
    """Upper bound of one packed StepMeta message (header + int32 payload, see
    ``StepMeta.pack``): seq ids, 3 per-token arrays, 2 per-seq lengths, the block table,
    3 sampling words and a 2-word seed per sequence."""
    S, T = int(max_seqs), int(max(max_tokens, max_seqs))
    words = S + 3 * T + 2 * S + S * int(table_width) + 3 * S + 2 * S
    return _HDR_BYTES + 4 * words + 64


class PipeChannel:
    """Control + data planes of one pipeline rank (default process group = the stages).

    Data plane: ONE grouped ``batch_isend_irecv`` per rank per tick on the default
    communicator — {send my output of tick k-1 -> next, receive my input of tick k <- prev}
    (the tail's output is the sampled ids, sent to the head). Rank r's group at tick k pairs
    with rank r+1's and rank r-1's groups of the same tick (anti-diagonal schedule), so all
    ranks exchange together and nothing can wait on a later tick: deadlock-free. One
    communicator = one RCCL stream per rank: separate per-edge communicators would add
    streams that HIP may alias onto the same hardware queue (GPU_MAX_HW_QUEUES=4), putting
    a spinning receive in front of a send."""

    def __init__(self, device: torch.device, dtype=torch.bfloat16,
                 ctrl_bytes: int = 1 << 20, ctrl: Optional[str] = None,
                 msg_bytes: Tuple[int, int] = (64 << 20, 8 << 20),
                 comm: Optional[str] = None):
        self.rank = dist.get_rank()
        self.world = dist.get_world_size()
        self.device = torch.device(device)
        self.dtype = dtype
        # data plane: "torch" (torch.distributed p2p), "rccl" (comm.cpp on the compute
        # stream) or "ipc" (device mailboxes, ipc.cpp; on CPU its host model, fifo.py);
        # "auto" (default) = ipc when every rank is a GPU process on this host and the
        # mailboxes pass their self-test, torch otherwise (resolve_comm)
        # collective over all ranks (called once per engine). Idle serving ranks block on
        # the control plane between sessions: no timeout that could fire while idle.
        self.ctrl_group = dist.new_group(backend="gloo", timeout=timedelta(days=365))
        requested = comm or os.environ.get("DLI_PP_COMM", "auto")
        self.comm = resolve_comm(requested, self.device, self.ctrl_group)
        if self.comm not in ("torch", "rccl", "ipc"):
            raise ValueError(f"DLI_PP_COMM={self.comm}: expected auto | torch | rccl | ipc")
        self.nccl = dist.get_backend() == "nccl" or (self.comm == "ipc"
                                                     and self.device.type == "cuda")
        self.data_device = self.device if self.nccl else torch.device("cpu")
        self._ctrl_sends: List = []
        self.ring = None
        self.ctrl_kind = "none"
        self.ctrl_bytes = int(ctrl_bytes)
        self._msg = np.zeros(self.ctrl_bytes, dtype=np.uint8)       # head's staging buffer
        self._hdr_rx = torch.empty(HEADER_LEN, dtype=torch.int64)    # gloo fallback
        self._pay_rx = torch.empty(self.ctrl_bytes // 4, dtype=torch.int32)
        self.exchanges = 0
        self.fallback: Optional[str] = None      # why the requested plane was not used
        if self.world > 1:
            self._init_ctrl(ctrl or os.environ.get("DLI_PP_CTRL", "auto"))
            # every rank joins one grouped ring exchange up front, so whatever point-to-point
            # communicator state RCCL builds lazily is built with all ranks present (the
            # session's first exchanges involve only some ranks)
            ck = self.device if dist.get_backend() == "nccl" else torch.device("cpu")
            t = torch.full((1,), float(self.rank), device=ck)
            r = torch.empty(1, device=ck)
            for w in dist.batch_isend_irecv([dist.P2POp(dist.isend, t, self.next),
                                             dist.P2POp(dist.irecv, r, self.prev)]):
                w.wait()
            if int(r.item()) != self.prev:
                raise RuntimeError(f"pipeline ring check failed on rank {self.rank}")
        # DLI_PP_COMM=rccl: the data plane on this module's own RCCL communicator
        # (csrc/runtime/comm.cpp), enqueued on the compute stream; DLI_PP_COMM=ipc: device
        # mailboxes (csrc/runtime/ipc.cpp), also on the compute stream, or on CPU the same
        # protocol on shared-memory mailboxes (fifo.py); default: torch.distributed
        self.rccl = None
        self.ipc = None
        self.dead_peer: Optional[str] = None    # set by the watchdog: who died
        self._wd_stop = threading.Event()
        self._wd = None
        if self.world > 1 and self.comm == "rccl" and dist.get_backend() == "nccl":
            self._init_rccl()
        if self.world > 1 and self.comm == "ipc":
            self._init_ipc(*msg_bytes)
            ok = ipc_selftest(self.ipc, self.ctrl_group)
            if not ok:
                if requested == "ipc":
                    raise RuntimeError("IPC data plane failed its self-test")
                self._close_ipc()
                self.comm = "torch"
                self.nccl = dist.get_backend() == "nccl"
                self.data_device = self.device if self.nccl else torch.device("cpu")
                self.fallback = "ipc self-test failed"
                _log.warning("pipeline rank %d: IPC mailboxes failed their self-test; the "
                             "data plane falls back to torch.distributed (%s)", self.rank,
                             dist.get_backend())
        self.data_plane = data_plane_name(self.comm, self.nccl) if self.world > 1 else "none"

    # ------------------------------------------------------------------ setup
    def _init_rccl(self) -> None:
        from ..runtime import RcclComm
        box = [RcclComm.unique_id() if self.rank == 0 else None]
        dist.broadcast_object_list(box, src=0, group=self.ctrl_group)
        self.rccl = RcclComm(box[0], self.world, self.rank)
        t = torch.full((1,), float(self.rank), device=self.device)
        r = torch.empty(1, device=self.device)
        self.rccl.exchange([(t, self.next)], [(r, self.prev)],
                           torch.cuda.current_stream(self.device).cuda_stream)
        if int(r.item()) != self.prev:
            raise RuntimeError(f"RCCL ring check failed on rank {self.rank}")

    def _init_ipc(self, big: int, small: int) -> None:
        """Mailboxes: ``big`` bytes on the activation edges r -> r + 1, ``small`` on the rest
        (tail -> every rank: final hidden / tokens, every rank -> 0: candidates)."""
        from .fifo import mailbox_caps
        cap = mailbox_caps(self.world, big, small)
        box = [f"/dli_pp_{os.environ.get('MASTER_PORT', '0')}_{os.getpid()}_{next(_ring_ids)}"
               if self.rank == 0 else None]
        dist.broadcast_object_list(box, src=0, group=self.ctrl_group)
        prefix = box[0]
        if self.device.type == "cuda":
            from ..runtime import IpcEndpoint
            host = os.environ.get("DLI_IPC_FLAGS", "device") == "host"
            ep = IpcEndpoint(self.world, self.rank, cap, host_prefix=prefix if host else "")
            hs = [None] * self.world
            dist.all_gather_object(hs, ep.handles(), group=self.ctrl_group)
            dist.barrier(group=self.ctrl_group)
            ep.connect(hs)
        else:
            from .fifo import ShmMailboxTransport
            ep = ShmMailboxTransport(self.world, self.rank, cap, prefix)
            dist.barrier(group=self.ctrl_group)
            ep.connect()
        dist.barrier(group=self.ctrl_group)
        self.ipc = ep
        self.data_device = self.device

    def _close_ipc(self) -> None:
        if self.ipc is not None:
            if self.device.type == "cuda" and not self.drain():
                # a queue still blocked after the bounded drain: leak the endpoint rather
                # than free mailboxes a kernel may still touch
                self.ipc = None
                return
            self.ipc.close()
            self.ipc = None

    def check(self) -> None:
        """Raise if a ring process died (watchdog) or the device data plane flagged an error
        (a peer stopped signalling, a stale or mis-ordered message, an abort): one load of
        a pinned host word, called every tick by the head and by every stage, so a broken
        ring fails its session instead of serving tokens computed from stale activations."""
        if self.dead_peer is not None:
            raise PeerDied(self.dead_peer)
        if self.ipc is not None:
            bits = self.ipc.error()
            if bits:
                raise DataPlaneError(bits)

    # ------------------------------------------------------------------ failure detection
    def start_watchdog(self, period_s: float = 0.2) -> None:
        """Poll the liveness of every process on the ring (the shared-memory control ring
        records each one's pid) and the RCCL communicator's async error every ``period_s``;
        on a death abort the data plane AT ONCE (every wait this rank's queue holds on the
        dead peer is released, the device plane turns sticky-failed) so the next ``check``
        of the tick loop raises. Detection within ~``period_s`` instead of a wait budget or
        the RCCL watchdog's ``DLI_PP_TIMEOUT_S``."""
        if self.world == 1 or self._wd is not None:
            return
        if self.ring is None and self.rccl is None:
            return                      # gloo control plane across hosts: sockets tell
        self._wd = threading.Thread(target=self._watch, args=(float(period_s),), daemon=True,
                                    name=f"dli-pp-watchdog-{self.rank}")
        self._wd.start()

    def _watch(self, period: float) -> None:
        from ..runtime import RcclComm
        busy_since = None
        # an exchange enqueue holds the RCCL handle for microseconds (a lazy P2P connect for
        # well under a second); held longer it is blocked on a peer that will never answer
        busy_limit = float(os.environ.get("DLI_PP_TIMEOUT_S", "30"))
        while not self._wd_stop.wait(period):
            ring = self.ring
            d = ring.dead() if ring is not None else -1
            err = self.rccl.async_error() if self.rccl is not None else 0
            if err == RcclComm.BUSY:
                now = time.monotonic()
                busy_since = busy_since or now
                err = 0 if now - busy_since < busy_limit else err
            else:
                busy_since = None
            if d == -1 and err == 0:
                continue
            if d == 1000:
                self.dead_peer = "pipeline head (rank 0) exited"
            elif d >= 0:
                self.dead_peer = f"pipeline stage {d + 1} exited"
            elif err == RcclComm.BUSY:
                self.dead_peer = f"RCCL exchange blocked for over {busy_limit:.0f} s"
            else:
                self.dead_peer = f"RCCL communicator error {err}"
            self.abort_data_plane()
            return

    def abort_data_plane(self, timeout_s: float = 5.0) -> None:
        """Release this rank's queue from a dead peer: IPC mailboxes aborted (sticky
        error, every flag set), the direct RCCL communicator aborted (ncclCommAbort)."""
        if self.ipc is not None and hasattr(self.ipc, "abort"):
            try:
                self.ipc.abort(timeout_s)
            except Exception:  # noqa: BLE001
                pass
        if self.rccl is not None:
            try:
                self.rccl.abort()
            except Exception:  # noqa: BLE001
                pass

    def drain(self, timeout_s: float = 10.0) -> bool:
        """Wait (bounded) until this rank's compute stream has finished everything queued,
        re-aborting the mailboxes meanwhile (a stream-op wait, DLI_IPC_SYNC=stream, takes
        one release per queued wait). True when the stream drained."""
        if self.device.type != "cuda":
            return True
        import time as _t
        ev = torch.cuda.Event()
        ev.record(torch.cuda.current_stream(self.device))
        t0 = _t.monotonic()
        while not ev.query():
            if self.dead_peer is not None or (self.ipc is not None and self.ipc.error()):
                self.abort_data_plane(1.0)
            if _t.monotonic() - t0 > timeout_s:
                return False
            _t.sleep(0.005)
        return True

    def _stream(self) -> int:
        return (torch.cuda.current_stream(self.device).cuda_stream
                if self.device.type == "cuda" else 0)

    def _init_ctrl(self, mode: str) -> None:
        hosts = [None] * self.world
        dist.all_gather_object(hosts, socket.gethostname(), group=self.ctrl_group)
        use_shm = mode == "shm" or (mode == "auto" and len(set(hosts)) == 1)
        name = None
        if use_shm and self.rank == 0:
            from ..runtime import ShmRing
            name = (f"/dli_pp_{os.environ.get('MASTER_PORT', '0')}_{os.getpid()}_"
                    f"{next(_ring_ids)}")
            try:
                # 4N + 16 slots: the head runs at most ~N + 3 ticks ahead of the tail
                self.ring = ShmRing.create(name, 4 * self.world + 16, self.ctrl_bytes,
                                           self.world - 1)
            except OSError:
                name = None
        box = [name if self.rank == 0 else None]
        dist.broadcast_object_list(box, src=0, group=self.ctrl_group)
        name = box[0]
        if name is not None and self.rank > 0:
            from ..runtime import ShmRing
            self.ring = ShmRing.open(name, self.rank - 1)
        dist.barrier(group=self.ctrl_group)
        if name is not None and self.rank == 0:
            self.ring.unlink()           # mapped by every rank now: nothing left in /dev/shm
        self.ctrl_kind = "shm" if name is not None else "gloo"

    @property
    def next(self) -> int:
        return (self.rank + 1) % self.world

    @property
    def prev(self) -> int:
        return (self.rank - 1) % self.world

    # ------------------------------------------------------------------ control plane
    def broadcast_ctrl(self, header: np.ndarray, payload: np.ndarray) -> None:
        """Head -> every other stage; never waits for a consumer unless the ring is full."""
        if faults.active():
            faults.check("transport.exchange", tick=int(header[H_TICK]))
        header[4] = int(payload.shape[0])
        with trace_range("pp.ctrl"):
            if self.ring is not None:
                nb = _HDR_BYTES + 4 * int(payload.shape[0])
                if nb > self.ctrl_bytes:
                    raise ValueError(f"step metadata of {nb} B exceeds the control slot "
                                     f"({self.ctrl_bytes} B)")
                m = self._msg
                m[:_HDR_BYTES].view(np.int64)[:] = header
                m[_HDR_BYTES:nb].view(np.int32)[:] = payload
                self.ring.publish(m[:nb])
                return
            h = torch.from_numpy(np.ascontiguousarray(header, dtype=np.int64).copy())
            p = torch.from_numpy(np.ascontiguousarray(payload, dtype=np.int32).copy())
            for r in range(1, self.world):
                self._ctrl_sends.append((dist.isend(h, r, group=self.ctrl_group), h))
                if p.numel():
                    self._ctrl_sends.append((dist.isend(p, r, group=self.ctrl_group), p))
            # never block here: stage r consumes the message of tick j only after the head
            # has posted its data exchange of tick j, so a blocking drain BEFORE this tick's
            # exchange can deadlock a deep ring. The head drains in reap_ctrl().
            self._reap(blocking_above=None)

    def _reap(self, blocking_above):
        q = self._ctrl_sends
        i = 0
        while i < len(q) and q[i][0].is_completed():
            q[i][0].wait()
            i += 1
        del q[:i]
        if blocking_above is not None:
            while len(q) > blocking_above:
                q.pop(0)[0].wait()

    def reap_ctrl(self) -> None:
        """Head (gloo control plane), after posting this tick's data exchange: release
        delivered messages and bound the backlog."""
        if self._ctrl_sends:
            self._reap(blocking_above=64 * self.world)

    def recv_ctrl(self) -> Tuple[np.ndarray, np.ndarray]:
        """Next control message: (header int64[16], payload int32[n]). The arrays are views
        of a reused buffer, valid until the next call."""
        if self.ring is not None:
            m = self.ring.consume()
            return m[:_HDR_BYTES].view(np.int64), m[_HDR_BYTES:].view(np.int32)
        h = self._hdr_rx
        dist.recv(h, 0, group=self.ctrl_group)
        n = int(h[4])
        p = self._pay_rx[:n]
        if n:
            dist.recv(p, 0, group=self.ctrl_group)
        return h.numpy(), p.numpy()

    # ------------------------------------------------------------------ data plane
    def recv_buffer(self, shape: Sequence[int], dtype=None) -> torch.Tensor:
        """A receive buffer allocated ONCE (engine setup) on the data-plane device."""
        return torch.empty(tuple(shape), dtype=dtype or self.dtype, device=self.data_device)

    def exchange(self, sends, recvs) -> None:
        """This tick's grouped exchange, completed before anything later on this rank reads
        a receive buffer or overwrites a sent tensor.

        ``sends`` = [(tensor, peer, tag)] sent in place; ``recvs`` = [(buffer, peer, tag)]
        with buffers from ``recv_buffer`` (views allowed). Tags keep several messages between
        one pair apart (gloo matches per (peer, tag); RCCL ignores them).

        RCCL: every Work is waited on the CURRENT stream — a stream dependency, not a host
        wait — so the next kernels on this stream (the consumer replay, or the replay that
        rewrites a sent static output) run after the transfer. gloo: a host wait."""
        if self.ipc is not None:             # stream-ordered mailboxes, FIFO per edge
            with trace_range("pp.exchange"):
                self.ipc.exchange(
                    [(t.contiguous(), peer) for t, peer, _ in sends
                     if t is not None and t.numel()],
                    [(b, peer) for b, peer, _ in recvs if b.numel()], self._stream())
            self.exchanges += 1
            return
        if self.rccl is not None:            # stream-ordered, no waits (comm.cpp)
            with trace_range("pp.exchange"):
                self.rccl.exchange(
                    [(t.contiguous(), peer) for t, peer, _ in sends
                     if t is not None and t.numel()],
                    [(b, peer) for b, peer, _ in recvs if b.numel()],
                    torch.cuda.current_stream(self.device).cuda_stream)
            self.exchanges += 1
            return
        ops = []
        with trace_range("pp.exchange"):
            for t, peer, tag in sends:
                if t is None or t.numel() == 0:
                    continue
                if not self.nccl and t.device.type != "cpu":
                    t = t.to("cpu")          # same-device gloo rehearsal only
                ops.append(dist.P2POp(dist.isend, t.contiguous(), peer, tag=tag))
            for buf, peer, tag in recvs:
                if buf.numel() == 0:
                    continue
                ops.append(dist.P2POp(dist.irecv, buf, peer, tag=tag))
            if not ops:
                return
            works = dist.batch_isend_irecv(ops)
            for w in works:
                w.wait()
        self.exchanges += 1

    def to_compute(self, buf: torch.Tensor) -> torch.Tensor:
        """A received buffer as the compute device sees it (a copy only when gloo carries
        the data plane of a GPU rank: the same-device rehearsal)."""
        return buf if buf.device == self.device else buf.to(self.device, non_blocking=True)

    def flush(self) -> None:
        while self._ctrl_sends:
            w, _ = self._ctrl_sends.pop(0)
            w.wait()

    def close(self) -> None:
        self._wd_stop.set()
        if getattr(self, "rccl", None) is not None:
            if self.dead_peer is not None:
                self.rccl.abort()
            else:
                self.rccl.close()
            self.rccl = None
        if getattr(self, "ipc", None) is not None:
            self._close_ipc()
        if self.ring is not None:
            if self.rank == 0:
                self.ring.close()
            self.ring.destroy()
            self.ring = None


class PeerDied(RuntimeError):
    """The pipeline watchdog saw a ring process exit (or RCCL report an async error)."""


class DataPlaneError(RuntimeError):
    """The device mailbox data plane raised error bits (csrc/runtime/ipc.cpp)."""

    def __init__(self, bits: int):
        what = [n for b, n in ((1, "a peer stopped signalling (wait budget exceeded)"),
                               (2, "stale / lost / mis-ordered message (sequence check)"),
                               (4, "ring aborted")) if bits & b]
        super().__init__(f"IPC data plane error {bits}: " + "; ".join(what))
        self.bits = bits


def resolve_comm(requested: str, device: torch.device, group) -> str:
    """``auto`` -> ``ipc`` when this is a GPU rank and every rank of ``group`` runs on this
    host (the hipIpc mailboxes need one node), else ``torch``. Explicit values pass through.
    A collective over ``group`` (gloo) when ``auto``."""
    requested = (requested or "auto").lower()
    if requested != "auto":
        return requested
    hosts = [None] * dist.get_world_size(group)
    dist.all_gather_object(hosts, (socket.gethostname(), device.type == "cuda"), group=group)
    same_host = len({h for h, _ in hosts}) == 1
    return "ipc" if same_host and all(g for _, g in hosts) else "torch"


def ipc_selftest(ep, group, wait_s: float = 10.0) -> bool:
    """One message over EVERY edge of the endpoint (all sends, then all receives: the
    mailboxes start empty, so this order cannot block), each a rank/peer-specific pattern
    checked on arrival, under a short wait budget; then the error word. Every rank learns
    every rank's verdict (``group``, gloo), so all of them keep or drop the data plane
    together. On a GPU this is the first end-to-end use of the mapped peer memory: a node
    whose peer writes never land fails here and the caller falls back to torch/RCCL."""
    cap = np.asarray(ep.cap)
    W, me = cap.shape[0], dist.get_rank(group)
    dev = torch.device("cuda", torch.cuda.current_device()) if _is_gpu_ep(ep) else \
        torch.device("cpu")
    n = 256
    ok = True
    try:
        ep.set_wait(wait_s)
        sends = [(torch.arange(n, dtype=torch.int32, device=dev) + (me * W + p) * 1000, p)
                 for p in range(W) if p != me and cap[me, p] >= 4 * n]
        recvs = [(torch.empty(n, dtype=torch.int32, device=dev), q)
                 for q in range(W) if q != me and cap[q, me] >= 4 * n]
        st = torch.cuda.current_stream(dev).cuda_stream if dev.type == "cuda" else 0
        ep.exchange(sends, recvs, st)
        if dev.type == "cuda":
            torch.cuda.synchronize(dev)
        for buf, q in recvs:
            want = torch.arange(n, dtype=torch.int32, device=dev) + (q * W + me) * 1000
            ok = ok and bool(torch.equal(buf, want))
        ok = ok and ep.error() == 0
    except Exception:  # noqa: BLE001 — a failing endpoint is reported, not raised
        ok = False
    finally:
        try:
            ep.set_wait(float(os.environ.get("DLI_IPC_WAIT_S", "120")))
        except Exception:  # noqa: BLE001
            pass
    verdicts = [None] * dist.get_world_size(group)
    dist.all_gather_object(verdicts, ok, group=group)
    return all(verdicts)


def _is_gpu_ep(ep) -> bool:
    return type(ep).__name__ == "IpcEndpoint"


def rank_info(device: torch.device) -> dict:
    """Where this rank runs: host, process, device ordinal, the physical GPU behind it
    (PCI bus id when the runtime reports one) and the visibility mask it was started with.
    A multi-rank record carries every rank's entry, so a reader can tell N GPUs from N
    ranks sharing one."""
    dev = torch.device(device)
    info = {"rank": dist.get_rank() if dist.is_initialized() else 0,
            "host": socket.gethostname(), "pid": os.getpid(), "device": str(dev)}
    if dev.type == "cuda":
        idx = dev.index if dev.index is not None else torch.cuda.current_device()
        p = torch.cuda.get_device_properties(idx)
        bus = [getattr(p, k, None) for k in ("pci_domain_id", "pci_bus_id", "pci_device_id")]
        if all(b is not None for b in bus):
            info["pci"] = "%04x:%02x:%02x" % tuple(int(b) for b in bus)
        info["name"] = p.name
        for k in ("HIP_VISIBLE_DEVICES", "ROCR_VISIBLE_DEVICES", "CUDA_VISIBLE_DEVICES"):
            if os.environ.get(k):
                info[k] = os.environ[k]
    return info


def gather_rank_info(device: torch.device, group=None) -> List[dict]:
    """``rank_info`` of every rank of ``group`` (an object all-gather: every rank calls)."""
    out = [None] * dist.get_world_size(group)
    dist.all_gather_object(out, rank_info(device), group=group)
    return out


def distinct_gpus(infos: Sequence[dict]) -> int:
    """Physical GPUs behind a list of ``rank_info`` entries (by PCI id, else by ordinal)."""
    keys = {(i.get("host"), i.get("pci") or (i.get("HIP_VISIBLE_DEVICES"), i.get("device")))
            for i in infos if str(i.get("device", "")).startswith("cuda")}
    return len(keys)


def init_distributed(backend: Optional[str] = None, device: Optional[torch.device] = None,
                     init_method: Optional[str] = None, world_size: Optional[int] = None,
                     rank: Optional[int] = None):
    """Initialise torch.distributed from torchrun env vars (127.0.0.1 rendezvous), or from an
    explicit ``init_method`` (``tcp://host:port``) + ``world_size`` + ``rank``: a worker that
    joins a pipeline when the master assigns it a shard (``/load_shard`` with a "pipeline"
    spec, ``worker/server.py``).

    Failure detection: data-plane operations get a bounded timeout
    (``DLI_PP_TIMEOUT_S``, default 600 s), so a stage that dies mid-session turns a blocked
    exchange into an error: RCCL's watchdog aborts the communicator when the timeout fires
    (torch's ``TORCH_NCCL_ASYNC_ERROR_HANDLING`` default), gloo raises as soon as the dead
    peer's sockets close; the shared-memory control ring notices a dead producer / consumer
    process. The head then fails its pending requests and reports unhealthy
    (``worker/service.PipelineService``); the master's failure detector routes new requests
    to the remaining replicas."""
    if dist.is_initialized():
        r, w = dist.get_rank(), dist.get_world_size()
        if (rank is not None and int(rank) != r) or (world_size is not None
                                                     and int(world_size) != w):
            raise RuntimeError(f"a process group (rank {r} of {w}) already exists; asked for "
                               f"rank {rank} of {world_size}: destroy it first")
        return r, w
    os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
    os.environ.setdefault("MASTER_PORT", "29511")
    if backend is None:
        # ranks sharing one GPU (DLI_SAME_DEVICE=1 rehearsals) cannot form an RCCL
        # communicator (one rank per device): their process group is gloo, the data plane
        # is still the device mailboxes
        same = os.environ.get("DLI_SAME_DEVICE", "0") == "1"
        backend = os.environ.get("DLI_DIST_BACKEND") or (
            "nccl" if torch.cuda.is_available() and not same else "gloo")
    kw = {"timeout": timedelta(seconds=float(os.environ.get("DLI_PP_TIMEOUT_S", "600")))}
    if backend == "nccl" and device is not None:
        kw["device_id"] = device
    if init_method is not None:
        kw.update(init_method=init_method, world_size=int(world_size), rank=int(rank))
    dist.init_process_group(backend=backend, **kw)
    return dist.get_rank(), dist.get_world_size()
