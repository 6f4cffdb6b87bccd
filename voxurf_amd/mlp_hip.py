"""Host side of the rgbnet MLP on the matrix-core kernels (csrc/mlp.hip).

mlp_forward(x, linears, compute_dtype) -> logits [M, 3], differentiable w.r.t. x and
every Linear's weight and bias.  Shapes: width 192, at least one hidden layer of
192 x 192, input width <= 96 (the plain fine step's rgbnet takes 42 inputs, the
reference's fine rgbnet 79).

Precision (`prec` of the kernels):
  PREC_F32_SPLIT (float32, the default): float32 activations, weights and gradients;
      every product is formed from three-way BF16 splits of both operands (six BF16
      MFMA products per pair, FP32 accumulation), within 2^-23 relative of the exact
      product, so the results carry FP32 accuracy (the weight gradients too, from
      operands split once as they are staged in LDS); where no gradient follows, all layers
      in one launch with the same bits (net_logits);
  PREC_F32: the same on FP32 MFMAs (v_mfma_f32_32x32x2f32);
  PREC_BF16 (compute_dtype bfloat16): forward and data-gradient GEMMs as single BF16
      MFMAs with FP32 accumulation, activations stored in BF16; weights, biases,
      gradients and the optimiser stay FP32.

The pieces are also exposed without autograd (Packed, forward_rows, backward_rows)
for callers that keep the gradients in their own buffers (the fused training step).
"""
import torch

from ._lib import call, lib, on_stream, ptr, stream_of

WIDTH = 192
PREC_F32, PREC_BF16, PREC_F32_SPLIT = 0, 1, 2


def prec_of(compute_dtype, f32_split=True):
    """Kernel precision for an rgbnet compute dtype (float32 or bfloat16)."""
    if compute_dtype == torch.bfloat16:
        return PREC_BF16
    if compute_dtype == torch.float32:
        return PREC_F32_SPLIT if f32_split else PREC_F32
    raise RuntimeError("the rgbnet kernels compute in float32 or bfloat16")


def act_dtype(prec):
    """Element type of the stored activations."""
    return torch.bfloat16 if prec == PREC_BF16 else torch.float32


def _pad_width(d):
    for w in (64, 96):
        if d <= w:
            return w
    raise RuntimeError(f"rgbnet input width {d} > 96 is not supported by the MFMA kernels")


def _packed_buffer(Ws, prec, st):
    """Every MFMA operand of one set of weights in one buffer (one vx_mlp_pack_net launch)."""
    n_hidden = len(Ws) - 1
    k_in0 = Ws[0].shape[1]
    total = lib().vx_mlp_pack_net_elems(n_hidden, k_in0)
    if total < 0:
        raise RuntimeError("rgbnet shape not supported by the MFMA kernels")
    parts = 3 if prec == PREC_F32_SPLIT else 1
    buf = torch.empty(parts * total, dtype=torch.float32 if prec == PREC_F32 else torch.bfloat16,
                      device=Ws[0].device)
    w_ptrs = torch.tensor([W.data_ptr() for W in Ws[:-1]], dtype=torch.int64)
    call("vx_mlp_pack_net", prec, n_hidden, w_ptrs.data_ptr(), k_in0, ptr(buf), st)
    return buf


class Packed:
    """The MFMA operands of one set of weights: fwd[li] (layer li, forward) and bwd[li] (layer
    li transposed, backward)."""

    def __init__(self, Ws, prec, st):
        n_hidden = len(Ws) - 1
        self.buf = _packed_buffer(Ws, prec, st)
        parts = 3 if prec == PREC_F32_SPLIT else 1
        kt0 = _pad_width(Ws[0].shape[1]) // 32
        self.fwd, self.bwd = [], []
        off = 0
        for li in range(n_hidden):
            kt = kt0 if li == 0 else 6
            n = parts * lib().vx_mlp_pack_elems(kt, 6)
            self.fwd.append(self.buf[off:off + n])
            off += n
            self.bwd.append(self.buf[off:off + n])
            off += n
        self.kt0 = kt0
        self.prec = prec


def net_logits(X, Ws, bs, st, M_dev=None):
    """The logits [M, 3] of forward_rows at split precision (the same bits) without the hidden
    activations: all layers in one launch, which never writes them (vx_mlp_net_fwd)."""
    M = X.shape[0]
    logits = torch.empty((M, 3), dtype=torch.float32, device=X.device)
    packed = _packed_buffer(Ws, PREC_F32_SPLIT, st)
    b_a = torch.tensor([b.data_ptr() for b in bs[:-1]], dtype=torch.int64)
    call("vx_mlp_net_fwd", len(Ws) - 1, Ws[0].shape[1], ptr(X), X.shape[1], M, ptr(packed),
         b_a.data_ptr(), ptr(Ws[-1]), ptr(bs[-1]), ptr(logits), ptr(M_dev), st)
    return logits


def forward_rows(X, Ws, bs, prec, packed, st, M_dev=None, timing=None, bits=None):
    """logits [M, 3] and the hidden activations of X [M, 32*kt0] (padded rows in the
    activation element type).  M_dev: optional device int64 row count (at most M rows of
    the buffers are then used), so the launches need not wait for it on the host.
    timing: a list that receives (start, end, launches): events around the run of
    192 x 192 layers (back to back on the stream) and their number.  bits: a list that
    receives each hidden layer's ReLU mask as bits [M, 6] int32 (split precision only;
    backward_rows reads them instead of the activations' signs)."""
    M = X.shape[0]
    dev = X.device
    adt = act_dtype(prec)
    logits = torch.empty((M, 3), dtype=torch.float32, device=dev)
    hs = []
    h_in, kt = X, packed.kt0
    nlin = len(Ws)
    for li in range(nlin - 1):
        last = li == nlin - 2
        H = torch.empty((M, WIDTH), dtype=adt, device=dev)
        if timing is not None and li == 1:
            e0 = torch.cuda.Event(enable_timing=True)
            e0.record()
        mb = None
        if bits is not None and prec == PREC_F32_SPLIT:
            mb = torch.empty((M, WIDTH // 32), dtype=torch.int32, device=dev)
            bits.append(mb)
        # the first layer's real input width: its weights are packed with zeros past it
        k_in = Ws[0].shape[1] if li == 0 else 0
        call("vx_mlp_layer_fwd", prec, kt, k_in, 0, ptr(h_in), h_in.shape[1], M,
             ptr(packed.fwd[li]), ptr(bs[li]), ptr(H), WIDTH, None, None, None, ptr(M_dev),
             ptr(mb), st)
        if timing is not None and li == nlin - 2 and li >= 1:
            e1 = torch.cuda.Event(enable_timing=True)
            e1.record()
            timing.append((e0, e1, nlin - 2))
        if last:
            call("vx_mlp_logits", prec, ptr(H), WIDTH, M, ptr(Ws[-1]), ptr(bs[-1]), ptr(logits),
                 ptr(M_dev), st)
        hs.append(H)
        h_in, kt = H, 6
    return logits, hs


def backward_rows(X, hs, Ws, prec, packed, g, st, grads, M_dev=None, bits=None,
                  wstream=None, inputs_free=None, wblocks=0, timing=None, dx_cols=None):
    """Gradients of every weight and bias into the tensors of `grads` ([W0, b0, W1, ...],
    overwritten) and the gradient of X [M, 32*kt0] (returned, float32); M_dev and bits
    as filled by forward_rows.

    wstream: optional torch stream for the weight gradients (the output layer's too when
    `bits` holds the mask bits: its data gradient then comes from them).  The data
    gradients then run back to back on `st` (torch's current stream) and the weight
    gradients are queued on wstream behind them, so the MFMA-bound weight-gradient
    passes can run beside whatever the caller queues next on `st`; the entries of
    `grads` computed there are final once wstream reaches the point this returns at.  The
    first of them is the input layer's, and the row count is copied on wstream before
    it: X and M_dev may be rewritten once wstream has passed that pass, which
    `inputs_free` (an optional torch.cuda.Event) records.  The activations passed in and
    the tensors this function allocates are marked as used on wstream.  wblocks: row
    blocks of the hidden layers' weight-gradient passes there (0: one per CU; fewer
    leave CUs to the kernels beside them).  timing: a list that receives (start, end, 1)
    per 192 x 192 hidden layer: HIP events, on the stream it runs on, around that layer's
    weight-gradient row-block pass alone (its reduction is launched after the end
    event).  dx_cols: the caller reads only the gradient of X's first dx_cols columns
    (<= 32 with prec 2 and a 64-wide X: the input layer's data gradient then writes those
    32 columns only)."""
    M = X.shape[0]
    dev = X.device
    nlin = len(Ws)
    part = torch.empty(lib().vx_mlp_wgrad_part_elems(M), dtype=torch.float32, device=dev)
    partb = torch.empty(lib().vx_mlp_wgrad_partb_elems(M), dtype=torch.float32, device=dev)
    # output layer (K = 3) and the gradient of the last hidden activations
    dH = torch.empty((M, WIDTH), dtype=torch.float32, device=dev)
    wjobs = []
    if wstream is not None and bits:
        # data gradient from the mask bits on `st`; dW3, db3 (a pass over H) on wstream
        call("vx_mlp_last_dgrad", ptr(g), ptr(bits[-1]), M, ptr(Ws[-1]), ptr(dH), WIDTH,
             ptr(M_dev), st)
        wjobs.append((nlin - 1, 0, g, hs[-1]))
    else:
        if wstream is None:
            part_last, partb_last = part, partb
        else:
            # the output layer's partial sums on `st`, beside the weight-gradient passes
            part_last = torch.empty(lib().vx_mlp_wgrad_part_elems(M), dtype=torch.float32,
                                    device=dev)
            partb_last = torch.empty(lib().vx_mlp_wgrad_partb_elems(M), dtype=torch.float32,
                                     device=dev)
        call("vx_mlp_last_bwd", prec, ptr(g), ptr(hs[-1]), WIDTH, M, ptr(Ws[-1]), ptr(dH),
             WIDTH, ptr(part_last), ptr(partb_last), ptr(grads[2 * (nlin - 1)]),
             ptr(grads[2 * nlin - 1]), ptr(M_dev), st)
    dX = None
    for li in range(nlin - 2, -1, -1):
        h_prev = hs[li - 1] if li > 0 else X
        kt = 6 if li > 0 else packed.kt0
        # weight gradient of layer li: dY = dH (its output grad), X = its input
        if wstream is None:
            _wgrad(prec, kt, Ws[li].shape[1], dH, h_prev, M, part, partb, grads[2 * li],
                   grads[2 * li + 1], M_dev, 0, st, timing if li >= 1 else None, None)
        else:
            wjobs.append((li, kt, dH, h_prev))
        # data gradient through layer li
        if li > 0:
            dprev = torch.empty((M, WIDTH), dtype=torch.float32, device=dev)
            call("vx_mlp_layer_bwd", prec, kt, ptr(dH), WIDTH, M, ptr(packed.bwd[li]),
                 ptr(h_prev), WIDTH, ptr(dprev), WIDTH, ptr(M_dev),
                 ptr(bits[li - 1]) if bits else None, st)
            dH = dprev
        else:
            dX = torch.empty((M, 32 * kt), dtype=torch.float32, device=dev)
            nto = 1 if dx_cols is not None and dx_cols <= 32 and prec == 2 and kt == 2 else kt
            call("vx_mlp_layer_bwd", prec, nto, ptr(dH), WIDTH, M, ptr(packed.bwd[0]), None,
                 0, ptr(dX), 32 * kt, ptr(M_dev), None, st)
    if wjobs:
        ready = torch.cuda.Event()
        ready.record(torch.cuda.current_stream(dev))
        wstream.wait_event(ready)
        ws = wstream.cuda_stream
        with on_stream(wstream):
            Mw = M_dev.clone() if M_dev is not None else None
        for i, (li, kt, dY, h_prev) in enumerate(sorted(wjobs, key=lambda j: j[0])):
            if li == nlin - 1:
                call("vx_mlp_last_wgrad", prec, ptr(dY), ptr(h_prev), WIDTH, M, ptr(part),
                     ptr(partb), ptr(grads[2 * li]), ptr(grads[2 * li + 1]), ptr(Mw), ws)
            else:
                _wgrad(prec, kt, Ws[li].shape[1], dY, h_prev, M, part, partb, grads[2 * li],
                       grads[2 * li + 1], Mw, wblocks, ws, timing if li >= 1 else None,
                       wstream)
            dY.record_stream(wstream)
            h_prev.record_stream(wstream)
            if i == 0 and inputs_free is not None:
                inputs_free.record(wstream)
        part.record_stream(wstream)
        partb.record_stream(wstream)
    return dX


class LaunchTiming(list):
    """A timing list (see backward_rows) that also holds device wall-clock stamp pairs
    for up to `capacity` launches of the split weight-gradient pass: stamps[i] =
    (first workgroup start, last workgroup end), preset here so that no launch in the
    timed region clears them.  durations_us() gives each stamped launch's duration."""

    def __init__(self, device, capacity=256):
        super().__init__()
        self.stamps = torch.empty((capacity, 2), dtype=torch.int64, device=device)
        self.stamps[:, 0] = torch.iinfo(torch.int64).max
        self.stamps[:, 1] = 0
        self.used = 0

    def next_stamp(self):
        if self.used >= self.stamps.shape[0]:
            return None
        self.used += 1
        return self.stamps[self.used - 1]

    def durations_us(self):
        khz = lib().vx_wall_clock_khz()
        if khz <= 0 or self.used == 0:
            return []
        s = self.stamps[:self.used].cpu()
        return [float(e - b) * 1e3 / khz for b, e in s.tolist()]


def _wgrad(prec, kt, k_real, dY, X, M, part, partb, dW, db, M_dev, wblocks, st, timing,
           tstream):
    """One layer's weight and bias gradients (vx_mlp_wgrad).  With `timing` (a list), the
    row-block pass is launched on its own between two events on the stream it runs on
    (tstream; None: the current stream), appended as (start, end, 1), then reduced; a
    LaunchTiming also receives the pass's device wall-clock stamps."""
    if timing is None:
        call("vx_mlp_wgrad", prec, kt, k_real, ptr(dY), WIDTH, ptr(X), X.shape[1], M,
             ptr(part), ptr(partb), ptr(dW), ptr(db), ptr(M_dev), wblocks, st)
        return
    stamp = timing.next_stamp() if prec == PREC_F32_SPLIT and hasattr(timing, "next_stamp") \
        else None
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record(tstream)
    call("vx_mlp_wgrad_partials", prec, kt, ptr(dY), WIDTH, ptr(X), X.shape[1], M, ptr(part),
         ptr(partb), ptr(M_dev), wblocks, ptr(stamp), st)
    e1.record(tstream)
    call("vx_mlp_wgrad_reduce", kt, k_real, M, ptr(part), ptr(partb), ptr(dW), ptr(db),
         wblocks, st)
    timing.append((e0, e1, 1))


def padded_rows(x, k_in, prec):
    """x [M, d] -> contiguous [M, 32*kt0] rows in the activation element type (x is used
    in place when it already has that width; columns past k_in meet zero weights)."""
    kin = _pad_width(k_in)
    adt = act_dtype(prec)
    if x.shape[1] == kin and x.is_contiguous():
        return x.detach().to(adt)
    return torch.nn.functional.pad(x.detach(), (0, kin - x.shape[1])).to(adt).contiguous()


class _MlpFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, prec, keep, *params):
        Ws = [p.detach().contiguous() for p in params[0::2]]
        bs = [p.detach().contiguous() for p in params[1::2]]
        if any(w.dtype != torch.float32 for w in Ws):
            raise RuntimeError("rgbnet parameters must be float32")
        st = stream_of(x)
        X = padded_rows(x, Ws[0].shape[1], prec)
        if prec == PREC_F32_SPLIT and not keep:
            return net_logits(X, Ws, bs, st)
        packed = Packed(Ws, prec, st)
        bits = []
        logits, hs = forward_rows(X, Ws, bs, prec, packed, st, bits=bits)
        ctx.save_for_backward(X, *hs)
        ctx.bits = bits
        ctx.Ws, ctx.bs, ctx.packed, ctx.prec, ctx.din = Ws, bs, packed, prec, x.shape[1]
        return logits

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, glogits):
        X, *hs = ctx.saved_tensors
        Ws, bs = ctx.Ws, ctx.bs
        grads = []
        for W, b in zip(Ws, bs):
            grads += [torch.empty_like(W), torch.empty_like(b)]
        dX = backward_rows(X, hs, Ws, ctx.prec, ctx.packed, glogits.contiguous().float(),
                           stream_of(X), grads, bits=ctx.bits)
        return (dX[:, :ctx.din], None, None, *grads)


def check_shapes(linears):
    if len(linears) < 3 or any(l.out_features != WIDTH for l in linears[:-1]) or \
            linears[-1].out_features != 3 or any(l.in_features != WIDTH for l in linears[1:]):
        raise RuntimeError("rgbnet kernels support width 192, depth >= 3, 3 outputs")


def mlp_forward(x, linears, compute_dtype=torch.float32, padded=False, f32_split=True):
    """logits = rgbnet(x) on the MFMA kernels (float32 or bfloat16 compute; float32 by
    BF16 splits unless f32_split is False).

    padded=True: x [M, W] float32 rows already padded to the kernels' tile width W
    (64 or 96, the smallest >= in_features) with finite values past in_features; they
    are read in place and the gradient has the same [M, W] shape."""
    if not x.is_cuda:
        raise RuntimeError("the rgbnet kernels need CUDA (HIP) tensors")
    check_shapes(linears)
    prec = prec_of(compute_dtype, f32_split)
    params = []
    for l in linears:
        params += [l.weight, l.bias]
    if padded:
        kin = _pad_width(linears[0].in_features)
        if x.dim() != 2 or x.shape[1] != kin or x.dtype != torch.float32 or not x.is_contiguous():
            raise RuntimeError(f"padded rgbnet input must be contiguous float32 [M, {kin}]")
        x2 = x
    else:
        if x.shape[-1] != linears[0].in_features:
            raise RuntimeError(f"rgbnet input width {x.shape[-1]} != {linears[0].in_features}")
        x2 = x.reshape(-1, x.shape[-1]).float()
    # the activations are kept only for a gradient to come
    keep = torch.is_grad_enabled() and (x2.requires_grad or any(p.requires_grad for p in params))
    out = _MlpFn.apply(x2, prec, keep, *params)
    return out.reshape(*x.shape[:-1], 3)
