"""torch.autograd wiring of the Hermite forward and its closed-form VJP.

Counterpart of the reference's ``jax.custom_vjp`` pair
(math/jax_vjps/hermite.py:47-102 unbatched, :113-175 batched): the forward
keeps (G, c) and the backward calls the VJP kernel, whatever ``stable`` was,
exactly as ``hermite_renormalized_jax_bwd`` always calls ``vanilla_vjp_numba``.

Convention.  The reference VJP is holomorphic: it returns sum_k g_k dG_k/dtheta
for the cotangent g, unconjugated.  torch hands a backward function
grad = dL/d(conj G) and expects dL/d(conj theta), which for a holomorphic map
is conj( sum_k conj(grad_k) dG_k/dtheta ).  The stored-lattice VJP reads the
gradient and writes its results conjugated; the VJPs that recompute the
forward run it at (conj A, conj b, conj c) with the gradient as it is, which is
the same number: no conjugated copy of a lattice-sized gradient is made.
"""

from __future__ import annotations

import torch

from ..lattice import strategies as st
from ..settings import settings


class HermiteRenormalized(torch.autograd.Function):
    """G = hermite_renormalized(A, b, c, shape, stable) with a custom VJP."""

    @staticmethod
    def forward(ctx, A, b, c, shape, stable):
        G = st.stable_hip(shape, A, b, c) if stable else st.vanilla_hip(shape, A, b, c)
        ctx.save_for_backward(G, c)
        ctx.a_shape, ctx.b_shape, ctx.c_shape = A.shape, b.shape, c.shape
        return G

    @staticmethod
    def backward(ctx, grad):
        G, c = ctx.saved_tensors
        dA, db, dc = st.vanilla_vjp_grad_hip(G, c, grad)
        return dA.reshape(ctx.a_shape), db.reshape(ctx.b_shape), dc.reshape(ctx.c_shape), None, None


class HermiteRenormalizedBatched(torch.autograd.Function):
    """Batched G[k] = hermite_renormalized(A[k], b[k], c[k], shape, stable)."""

    @staticmethod
    def forward(ctx, A, b, c, shape, stable):
        G = st.vanilla_batch_hip(shape, A, b, c, stable=stable)
        ctx.save_for_backward(G, c)
        ctx.a_shape, ctx.b_shape, ctx.c_shape = A.shape, b.shape, c.shape
        return G

    @staticmethod
    def backward(ctx, grad):
        G, c = ctx.saved_tensors
        dA, db, dc = st.vanilla_vjp_grad_hip(G, c, grad, batched=True)
        return dA.reshape(ctx.a_shape), db.reshape(ctx.b_shape), dc.reshape(ctx.c_shape), None, None


class HermiteRenormalizedRecompute(torch.autograd.Function):
    """As HermiteRenormalized, but autograd keeps only (A, b, c): the backward
    recomputes the lattice slab by slab in a three-slab window
    (``vanilla_vjp_recompute_hip``), so G need not stay resident between the
    forward and the backward.  The VJP applies to the forward's own lattice,
    as the reference's backward does (jax_vjps/hermite.py:78-101): for the
    all-pivot average the backward recomputes that lattice whole with
    ``stable_hip`` (the windowed sweep runs the first-pivot recurrence only)
    and frees it once the VJP is taken."""

    @staticmethod
    def forward(ctx, A, b, c, shape, stable):
        G = st.stable_hip(shape, A, b, c) if stable else st.vanilla_hip(shape, A, b, c)
        ctx.save_for_backward(A, b, c)
        ctx.shape = tuple(shape)
        ctx.stable = bool(stable)
        return G

    @staticmethod
    def backward(ctx, grad):
        A, b, c = ctx.saved_tensors
        if ctx.stable:
            G = st.stable_hip(ctx.shape, A, b, c)
            dA, db, dc = st.vanilla_vjp_grad_hip(G, c, grad)
            del G
        else:
            dA, db, dc = st.vanilla_vjp_recompute_hip(ctx.shape, *st.conj_triple(A, b, c), grad)
        return dA.reshape(A.shape), db.reshape(b.shape), dc.reshape(c.shape), None, None


class HermiteDiagonal(torch.autograd.Function):
    """G = hermite_renormalized_diagonal(A, B, c, cutoffs, reorderedAB) with the
    reverse-sweep VJP (the reference's jax custom VJP pair,
    jax_vjps/hermite.py:248-336).  The backward recomputes the forward together
    with the VJP (``diagonal_vjp_hip``), so only (A, B, c) are kept."""

    @staticmethod
    def forward(ctx, A, B, c, cutoffs, reordered):
        from ..lattice import compact_fock as cf

        G = cf.diagonal_hip(A, B, c, cutoffs, reordered=reordered)
        ctx.save_for_backward(A, B, c)
        ctx.cutoffs, ctx.reordered = tuple(cutoffs), bool(reordered)
        return G

    @staticmethod
    def backward(ctx, grad):
        from ..lattice import compact_fock as cf

        A, B, c = ctx.saved_tensors
        _, dA, dB, dc = cf.diagonal_vjp_hip(*st.conj_triple(A, B, c), ctx.cutoffs, grad, reordered=ctx.reordered)
        return dA.reshape(A.shape), dB.reshape(B.shape), dc.reshape(c.shape), None, None


class HermiteLeftover(torch.autograd.Function):
    """out = hermite_renormalized_1leftoverMode(A, b, c, output_cutoff,
    pnr_cutoffs) with the reverse-sweep VJP (the reference's jax custom VJP
    pair, jax_vjps/hermite.py:343-445).  The forward's intermediate blocks are
    kept for the backward up to ``LEFTOVER_KEEP_BYTES`` (a (20, 20, 15, 15)
    output: 16 MB; its second forward took a quarter of a training step);
    beyond that, or with ``settings.HERMITE_RECOMPUTE_VJP``, only (A, b, c) are
    kept and the backward recomputes them (``leftover_vjp_hip``)."""

    @staticmethod
    def forward(ctx, A, b, c, output_cutoff, pnr_cutoffs, reordered):
        from ..lattice import compact_fock as cf

        out, ws = cf._leftover(A, b, c, output_cutoff, pnr_cutoffs, reordered)
        if ws.numel() <= cf.LEFTOVER_KEEP_BYTES and not settings.HERMITE_RECOMPUTE_VJP:
            ctx.save_for_backward(A, b, c, ws)
        else:
            ctx.save_for_backward(A, b, c)
        ctx.args = (int(output_cutoff), tuple(int(k) for k in pnr_cutoffs), bool(reordered))
        return out

    @staticmethod
    def backward(ctx, grad):
        from ..lattice import compact_fock as cf

        A, b, c, *kept = ctx.saved_tensors
        o, pnr, reordered = ctx.args
        if kept:
            dA, db, dc = cf.leftover_grad_hip(A, b, c, o, pnr, kept[0], grad, reordered=reordered)
        else:
            _, dA, db, dc = cf.leftover_vjp_hip(*st.conj_triple(A, b, c), o, pnr, grad, reordered=reordered)
        return dA.reshape(A.shape), db.reshape(b.shape), dc.reshape(c.shape), None, None, None
