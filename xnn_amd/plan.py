"""Edge plans: the int32 edge streams and CSR orderings the HIP kernels walk.

An :class:`EdgePlan` is built once per edge list (on the device, by
``xnn_graph_plan``) and cached on the graph. It holds

* ``src``, ``dst`` (int32) and ``shift`` (three signed 10-bit fields in one
  int32) for every edge, in the edge list's own order;
* the receiver CSR ``ptr_dst`` with ``perm_dst`` (``None`` when the edges are
  already grouped by receiver, as :func:`~xnn_amd.data.build_neighbor_list`
  returns them), and the sender CSR ``ptr_src`` / ``perm_src``;
* the structure of every atom (``batch32``) and the structures' atom ranges
  (``node_ptr``, int64).

This mirrors the orderings of the reference's no-atomics kernels
(``common/models/csr.py:20-51``): every per-atom sum walks one CSR row in a
fixed order, so results are bitwise reproducible.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import torch
from torch import Tensor

from . import _lib


@dataclass
class EdgePlan:
    n_nodes: int
    n_edges: int
    n_graphs: int
    src: Tensor
    dst: Tensor
    shift: Tensor
    ptr_dst: Tensor
    perm_dst: Optional[Tensor]
    ptr_src: Tensor
    perm_src: Tensor
    batch32: Tensor
    node_ptr: Tensor
    # a space-filling-curve order of the atoms (structure by structure), the order in
    # which the force reductions take them; None: index order
    visit: Optional[Tensor] = None

    @property
    def device(self) -> torch.device:
        return self.ptr_dst.device


class ShiftRangeError(ValueError):
    """Image shifts that the packed int32 of a plan cannot hold (10 bits an axis)."""


def _int64(t: Tensor, device) -> Tensor:
    return t.to(device=device, dtype=torch.int64).contiguous()


def build_plan(edge_index: Tensor, cell_shifts: Optional[Tensor], n_nodes: int,
               batch: Optional[Tensor] = None, n_atoms: Optional[Tensor] = None,
               pos: Optional[Tensor] = None, cell: Optional[Tensor] = None) -> EdgePlan:
    """Build the plan of an edge list on its (GPU) device, in one call of the library and
    one host read (of the checks). With ``pos`` (N, 3) the plan also orders the atoms along
    a space-filling curve (:attr:`EdgePlan.visit`; ``cell`` (B, 3, 3) or None).

    Raises ``ValueError`` for edge indices outside ``[0, n_nodes)``, image
    shifts outside ``[-512, 511]`` (:class:`ShiftRangeError`), atoms not grouped by structure
    and a ``batch`` or ``pos`` that does not cover the atoms.
    """
    device = edge_index.device
    if device.type != "cuda":
        raise ValueError("edge plans live on the GPU; move the graph to the device first")
    n_edges = int(edge_index.shape[1])
    edge_index = _int64(edge_index, device)
    shifts = None
    if cell_shifts is not None and cell_shifts.numel() > 0:
        shifts = _int64(cell_shifts, device)
    batch = None if batch is None else _int64(batch, device)
    if batch is not None and batch.shape[0] < n_nodes:
        raise ValueError(f"batch holds {batch.shape[0]} of the graph's {n_nodes} atoms")
    n_atoms = None if n_atoms is None else _int64(n_atoms, device)
    n_graphs = 1 if n_atoms is None else int(n_atoms.shape[0])
    if pos is not None and n_nodes > 0 and n_graphs > 0:
        if tuple(pos.shape) != (n_nodes, 3):
            raise ValueError(f"positions {tuple(pos.shape)} of a graph of {n_nodes} atoms")
        pos = pos.detach().to(device).contiguous()
        if pos.dtype not in (torch.float32, torch.float64):
            pos = pos.double()
        geom = _lib.dtype_code(pos.dtype)
        if cell is not None:
            cell = cell.detach().reshape(-1, 3, 3).to(device=device, dtype=pos.dtype).contiguous()
            cell = cell if cell.shape[0] == n_graphs else None
    else:
        geom, pos, cell = _lib.XNN_F64, None, None
    want_visit = pos is not None
    # the int32 arrays of the plan, one allocation (each view keeps it alive)
    sizes = [n_edges] * 5 + [n_nodes + 1] * 2 + [n_nodes] * (2 if want_visit else 1) + [1]
    views = torch.empty(sum(sizes), dtype=torch.int32, device=device).split(sizes)
    src, dst, shift, perm_dst, perm_src, ptr_dst, ptr_src, batch32 = views[:8]
    visit = views[8] if want_visit else None
    flags = views[-1]
    node_ptr = torch.empty(n_graphs + 1, dtype=torch.int64, device=device)
    ws_bytes = int(_lib.load().xnn_graph_plan_workspace_bytes(n_edges, n_nodes, n_graphs,
                                                              int(want_visit)))
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=device)
    _lib.call("xnn_graph_plan", _lib.ptr(edge_index), _lib.ptr(shifts), n_edges, n_nodes,
              _lib.ptr(batch), _lib.ptr(n_atoms), n_graphs, _lib.ptr(batch32), _lib.ptr(node_ptr),
              geom, _lib.ptr(pos), _lib.ptr(cell), _lib.ptr(visit), _lib.ptr(src), _lib.ptr(dst),
              _lib.ptr(shift), _lib.ptr(ptr_dst), _lib.ptr(perm_dst), _lib.ptr(ptr_src),
              _lib.ptr(perm_src), _lib.ptr(flags), _lib.ptr(ws), ws_bytes, _lib.stream(device))
    bits = int(flags.item())
    if bits & 2:
        raise ValueError(f"edge_index holds atom indices outside [0, {n_nodes})")
    if bits & 1:
        raise ShiftRangeError("cell_shifts outside [-512, 511]: the packed int32 shifts cannot "
                              "hold them (wrap the positions into the cell first)")
    if bits & 16:
        raise ValueError("batch holds structure indices outside [0, B)")
    if bits & 8:
        raise ValueError("the atoms of a batch must be grouped by structure (as collate does)")
    if bits & 32:
        raise ValueError(f"n_atoms sums to {int(node_ptr[-1])}, the graph has {n_nodes} atoms")
    return EdgePlan(n_nodes=n_nodes, n_edges=n_edges, n_graphs=n_graphs, src=src, dst=dst,
                    shift=shift, ptr_dst=ptr_dst, perm_dst=perm_dst if bits & 4 else None,
                    ptr_src=ptr_src, perm_src=perm_src, batch32=batch32, node_ptr=node_ptr,
                    visit=visit)


def plan_for(graph) -> EdgePlan:
    """The cached plan of an :class:`~xnn_amd.data.AtomicGraph` (rebuilt when its edge
    list, shifts or atom count change identity)."""
    cached = getattr(graph, "_xnn_plan", None)
    # identity of the (held) tensors, as the reference's orderings cache (csr.py:35-51)
    if (cached is not None and cached[0] is graph.edge_index and cached[1] is graph.cell_shifts
            and cached[2] == graph.num_nodes):
        return cached[3]
    plan = build_plan(graph.edge_index, graph.cell_shifts, graph.num_nodes, graph.batch,
                      graph.n_atoms, graph.pos, graph.cell)
    object.__setattr__(graph, "_xnn_plan",
                       (graph.edge_index, graph.cell_shifts, graph.num_nodes, plan))
    return plan
