"""E(n)-equivariant layers and stack on the fused HIP layer.

Same classes, constructor signatures and module structure as
models/EGNN/egnn_clean.py of the reference (``E_GCL`` :5-103, ``EGNN``
:106-146, ``unsorted_segment_sum/mean`` :149-164, ``get_edges(_batch)``
:167-191), so state dicts are interchangeable.  The per-edge work of
``E_GCL.forward`` -- edge_model (:49-58), the coordinate update of
coord_model (:72-82) and the message sum of node_model (:62) -- runs as one
fused HIP op (:class:`pymolecular_amd.fused.EGNNFusedFn`) that never
materialises the E x (2H+1+F_E) concatenation or the E x H messages; the
per-node part (node_mlp on cat([h, agg]) and the residual, :60-70) is the
fused node update (:func:`pymolecular_amd.node_update.node_update`), with the
same nn.Linear parameters.

Supported options of the fused path: act_fn = SiLU, attention = False,
normalize = False, tanh = False (the reference's defaults and the only
configuration any workload uses); other settings raise NotImplementedError.
"""
from __future__ import annotations

import torch
from torch import nn

from ...fused import TensorCache, coo_to_csr, egnn_fused
from ...layer_fn import gcl_layer
from ...node_update import dense, node_update

__all__ = ["E_GCL", "EGNN", "unsorted_segment_sum", "unsorted_segment_mean", "get_edges", "get_edges_batch"]


class _CSRCache:
    """dst-sorted CSR of an edge_index, cached per edge tensor by :class:`~pymolecular_amd.fused.TensorCache`
    (identity of the live tensors, not their addresses, so a new graph at a reused address is rebuilt)."""

    def __init__(self):
        self._cache = TensorCache(maxsize=8)

    def get(self, row: torch.Tensor, col: torch.Tensor, n: int):
        return self._cache.get((row, col), int(n), lambda: coo_to_csr(row, col, n))


_csr_cache = _CSRCache()


class E_GCL(nn.Module):
    """E(n) Equivariant Convolutional Layer (egnn_clean.py:5-103)."""

    def __init__(self, input_nf, output_nf, hidden_nf, edges_in_d=0, act_fn=nn.SiLU(), residual=True,
                 attention=False, normalize=False, coords_agg='mean', tanh=False):
        super().__init__()
        input_edge = input_nf * 2
        self.residual = residual
        self.attention = attention
        self.normalize = normalize
        self.coords_agg = coords_agg
        self.tanh = tanh
        self.epsilon = 1e-8
        edge_coords_nf = 1
        self.edges_in_d = edges_in_d
        self.act_is_silu = isinstance(act_fn, nn.SiLU)

        self.edge_mlp = nn.Sequential(
            nn.Linear(input_edge + edge_coords_nf + edges_in_d, hidden_nf),
            act_fn,
            nn.Linear(hidden_nf, hidden_nf),
            act_fn)

        self.node_mlp = nn.Sequential(
            nn.Linear(hidden_nf + input_nf, hidden_nf),
            act_fn,
            nn.Linear(hidden_nf, output_nf))

        layer = nn.Linear(hidden_nf, 1, bias=False)
        torch.nn.init.xavier_uniform_(layer.weight, gain=0.001)

        coord_mlp = [nn.Linear(hidden_nf, hidden_nf), act_fn, layer]
        if self.tanh:
            coord_mlp.append(nn.Tanh())
        self.coord_mlp = nn.Sequential(*coord_mlp)

        if self.attention:
            self.att_mlp = nn.Sequential(nn.Linear(hidden_nf, 1), nn.Sigmoid())

    def _check_supported(self):
        if self.attention or self.normalize or self.tanh or not self.act_is_silu:
            raise NotImplementedError("the fused EGNN layer implements act_fn=SiLU without attention, "
                                      "normalize or tanh (egnn_clean.py defaults)")
        if self.coords_agg not in ("mean", "sum"):
            raise Exception('Wrong coords_agg parameter' % self.coords_agg)

    def fused_messages(self, h, edge_index, coord, edge_attr=None, csr=None):
        """Returns (agg_msg = sum_j m_ij, agg_x = mean/sum_j (x_i - x_j) phi_ij) via the fused op."""
        self._check_supported()
        row, col = edge_index
        n = h.shape[0]
        row_ptrs, col_s, perm = csr if csr is not None else _csr_cache.get(row, col, n)
        e0, e2 = self.edge_mlp[0], self.edge_mlp[2]
        c0, c2 = self.coord_mlp[0], self.coord_mlp[2]
        ef = edge_attr if (edge_attr is not None and self.edges_in_d > 0) else None
        agg, agg_x = egnn_fused(h, coord, ef, row_ptrs, col_s, perm, e0.weight, e2.weight, c0.weight,
                                c2.weight.reshape(-1), e0.bias, e2.bias, c0.bias,
                                mean_agg=self.coords_agg == "mean", equivariant=True, linear_weights=True)
        return agg, agg_x

    def forward(self, h, edge_index, coord, edge_attr=None, node_attr=None, csr=None):
        if node_attr is None:   # the whole layer as one autograd node (layer_fn.gcl_layer)
            self._check_supported()
            row, col = edge_index
            row_ptrs, col_s, perm = csr if csr is not None else _csr_cache.get(row, col, h.shape[0])
            e0, e2, c0, c2 = self.edge_mlp[0], self.edge_mlp[2], self.coord_mlp[0], self.coord_mlp[2]
            n0, n2 = self.node_mlp[0], self.node_mlp[2]
            ef = edge_attr if (edge_attr is not None and self.edges_in_d > 0) else None
            h_out, coord = gcl_layer(h, coord, ef, row_ptrs, col_s, perm, e0.weight, e0.bias, e2.weight,
                                            e2.bias, c0.weight, c0.bias, c2.weight, n0.weight, n0.bias, n2.weight,
                                            n2.bias, self.coords_agg == "mean", self.residual, True)
            return h_out, coord, edge_attr
        agg, agg_x = self.fused_messages(h, edge_index, coord, edge_attr, csr)
        coord = coord + agg_x.to(coord.dtype)
        # node_model (:60-70): node_mlp(cat([h, agg(, node_attr)])) (+ h), as one fused node update
        x2 = agg if node_attr is None else torch.cat([agg, node_attr.to(agg.dtype)], dim=1)
        out = node_update(h, x2, self.node_mlp[0], self.node_mlp[2], residual=self.residual)
        return out, coord, edge_attr


class EGNN(nn.Module):
    """Stack of E_GCL layers between input/output embeddings (egnn_clean.py:106-146)."""

    def __init__(self, in_node_nf, hidden_nf, out_node_nf, in_edge_nf=0, device='cpu', act_fn=nn.SiLU(),
                 n_layers=4, residual=True, attention=False, normalize=False, tanh=False):
        super().__init__()
        self.hidden_nf = hidden_nf
        self.device = device
        self.n_layers = n_layers
        self.embedding_in = nn.Linear(in_node_nf, self.hidden_nf)
        self.embedding_out = nn.Linear(self.hidden_nf, out_node_nf)
        for i in range(0, n_layers):
            self.add_module("gcl_%d" % i, E_GCL(self.hidden_nf, self.hidden_nf, self.hidden_nf,
                                                edges_in_d=in_edge_nf, act_fn=act_fn, residual=residual,
                                                attention=attention, normalize=normalize, tanh=tanh))
        self.to(self.device)

    def forward(self, h, x, edges, edge_attr):
        h = dense(h, self.embedding_in)
        row, col = edges
        csr = _csr_cache.get(row, col, h.shape[0])   # one CSR for all layers, cached per edge tensor
        for i in range(0, self.n_layers):
            h, x, _ = self._modules["gcl_%d" % i](h, edges, x, edge_attr=edge_attr, csr=csr)
        h = dense(h, self.embedding_out)
        return h, x


def unsorted_segment_sum(data, segment_ids, num_segments):
    """Sum of ``data`` rows per segment id (egnn_clean.py:149-154)."""
    result = data.new_full((num_segments, data.size(1)), 0)
    result.index_add_(0, segment_ids, data)
    return result


def unsorted_segment_mean(data, segment_ids, num_segments):
    """Mean of ``data`` rows per segment id, empty segments give 0 (egnn_clean.py:157-164)."""
    result = unsorted_segment_sum(data, segment_ids, num_segments)
    count = torch.bincount(segment_ids, minlength=num_segments).to(data.dtype)
    return result / count.clamp(min=1)[:, None]


def get_edges(n_nodes):
    """Fully connected edges without self loops, i outer, j inner (egnn_clean.py:167-176)."""
    rows, cols = [], []
    for i in range(n_nodes):
        for j in range(n_nodes):
            if i != j:
                rows.append(i)
                cols.append(j)
    return [rows, cols]


def get_edges_batch(n_nodes, batch_size):
    """``batch_size`` copies of get_edges offset by n_nodes (egnn_clean.py:179-191)."""
    edges = get_edges(n_nodes)
    edge_attr = torch.ones(len(edges[0]) * batch_size, 1)
    edges = [torch.LongTensor(edges[0]), torch.LongTensor(edges[1])]
    if batch_size == 1:
        return edges, edge_attr
    rows, cols = [], []
    for i in range(batch_size):
        rows.append(edges[0] + n_nodes * i)
        cols.append(edges[1] + n_nodes * i)
    return [torch.cat(rows), torch.cat(cols)], edge_attr
