"""Learned GWB surrogate: an MLP from model parameters to log10 h_c percentile spectra.

Sits beside the reference's Gaussian-process emulator (holodeck/gps/gp_utils.py),
trained on libraries made by :mod:`holodeck_amd.librarian`.  Targets follow the
GP's convention on the library's ``gwb`` array (gp_utils.py:254-349: log10 of
statistics over realizations, with a 1e-40 floor): per frequency the log10 of
the median, 5th and 95th percentile of h_c, i.e. 3 F outputs.

Network: inputs rescaled to [0, 1] over the training box, hidden layers with
SiLU, linear output on standardised targets.  Training and inference run in
the library's HIP kernels (hd_mlp_*): BF16 operands on the matrix cores, FP32
accumulation, FP32 master weights and Adam moments.  PyTorch tensors are the
buffers only.

Outside the training box, or when asked to judge, the plain GPU SAM computes
the spectrum (:class:`SurrogateWithFallback`).
"""
import ctypes as C

import numpy as np
import torch

from . import _lib
from . import device as D

PERCENTILES = (50.0, 5.0, 95.0)
FLOOR = 1e-40


def targets_from_gwb(gwb):
    """(S, F, R) library h_c -> (S, 3F) log10 [median | 5th | 95th] per frequency."""
    gwb = np.asarray(gwb, dtype=float)
    q = np.percentile(gwb, PERCENTILES, axis=-1)            # (3, S, F)
    return np.log10(np.maximum(q, FLOOR)).transpose(1, 0, 2).reshape(gwb.shape[0], -1)


def _bf16(n_or_shape):
    return torch.empty(n_or_shape, dtype=torch.bfloat16, device=D.require_device())


def _f32(n_or_shape):
    return torch.empty(n_or_shape, dtype=torch.float32, device=D.require_device())


class MLPSurrogate:
    """n_in -> hidden... (SiLU) -> n_out, trained with Adam on mean squared error."""

    def __init__(self, n_in=6, hidden=(256, 256, 256, 256), n_out=90, seed=0):
        D.require_device()
        self.sizes = [int(n_in)] + [int(h) for h in hidden] + [int(n_out)]
        rng = np.random.default_rng(seed)
        self.W, self.b, self.Wb, self.mW, self.vW, self.mb, self.vb = [], [], [], [], [], [], []
        for fan_in, fan_out in zip(self.sizes[:-1], self.sizes[1:]):
            lim = np.sqrt(6.0 / fan_in) if fan_out != self.sizes[-1] else np.sqrt(1.0 / fan_in)
            w = rng.uniform(-lim, lim, size=(fan_out, fan_in)).astype(np.float32)   # (out, in)
            self.W.append(torch.as_tensor(w).to(D.require_device()))
            self.b.append(torch.zeros(fan_out, dtype=torch.float32, device=D.require_device()))
            self.Wb.append(self.W[-1].to(torch.bfloat16))
            self.mW.append(torch.zeros_like(self.W[-1]))
            self.vW.append(torch.zeros_like(self.W[-1]))
            self.mb.append(torch.zeros_like(self.b[-1]))
            self.vb.append(torch.zeros_like(self.b[-1]))
        self.step = 0
        self.x_lo = np.zeros(n_in)
        self.x_hi = np.ones(n_in)
        self.y_mean = np.zeros(n_out)
        self.y_std = np.ones(n_out)

    @property
    def nlayers(self):
        return len(self.sizes) - 1

    # ---- scaling ----
    def _x01(self, X):
        return (np.asarray(X, dtype=float) - self.x_lo) / (self.x_hi - self.x_lo)

    def in_box(self, X):
        x = self._x01(X)
        return np.all((x >= 0.0) & (x <= 1.0), axis=-1)

    # ---- device passes ----
    def _net(self):
        """This network for the whole-pass kernels, or None where they do not take its shape (then the
        layers run one by one)."""
        if self.nlayers > _lib.MLP_MAX_LAYERS:
            return None
        net = _lib.MlpNet(n_layers=self.nlayers)
        net.sizes[:self.nlayers + 1] = self.sizes
        for l in range(self.nlayers):
            net.w[l], net.b[l] = D.ptr(self.Wb[l]), D.ptr(self.b[l])
        return net if _lib.size("hd_mlp_fused", C.addressof(net)) else None

    def _forward(self, xb, keep):
        """xb: (M, n_in) bf16 device.  Returns output f32 (M, n_out) and, if keep, per-layer (z f32, h bf16)."""
        st = D.stream_ptr()
        M = xb.shape[0]
        h = xb
        cache = [(None, xb)]
        for l in range(self.nlayers):
            fin, fout = self.sizes[l], self.sizes[l + 1]
            if l < self.nlayers - 1:
                z = _f32((M, fout)) if keep else None
                hn = _bf16((M, fout))
                _lib.call("hd_mlp_gemm_bf16", D.ptr(h), fin, 1, D.ptr(self.Wb[l]), fin, 1, M, fout, fin,
                          _lib.HD_MLP_EPI_BIAS_SILU, D.ptr(self.b[l]), None, D.ptr(z), D.ptr(hn), fout, st)
                if keep:
                    cache.append((z, hn))
                h = hn
            else:
                y = _f32((M, fout))
                _lib.call("hd_mlp_gemm_bf16", D.ptr(h), fin, 1, D.ptr(self.Wb[l]), fin, 1, M, fout, fin,
                          _lib.HD_MLP_EPI_STORE, D.ptr(self.b[l]), None, D.ptr(y), None, fout, st)
        return y, cache

    def _backward(self, cache, dy):
        """dy: (M, n_out) bf16 gradient of the loss w.r.t. the output.  Returns [(dW f32, db f32)] per layer."""
        st = D.stream_ptr()
        M = dy.shape[0]
        grads = [None] * self.nlayers
        dz = dy
        for l in range(self.nlayers - 1, -1, -1):
            fin, fout = self.sizes[l], self.sizes[l + 1]
            h_in = cache[l][1]                       # (M, fin) bf16
            dW = _f32((fout, fin))
            # dW[o, i] = sum_m dz[m, o] h_in[m, i]
            _lib.call("hd_mlp_gemm_bf16", D.ptr(dz), 1, fout, D.ptr(h_in), 1, fin, fout, fin, M,
                      _lib.HD_MLP_EPI_STORE, None, None, D.ptr(dW), None, fin, st)
            db = _f32(fout)
            _lib.call("hd_mlp_colsum_bf16", D.ptr(dz), M, fout, D.ptr(db), st)
            grads[l] = (dW, db)
            if l > 0:
                # dh[m, i] = sum_o dz[m, o] W[o, i];  dz_prev = dh * silu'(z_prev)
                z_prev = cache[l][0]
                dzp = _bf16((M, fin))
                _lib.call("hd_mlp_gemm_bf16", D.ptr(dz), fout, 1, D.ptr(self.Wb[l]), 1, fin, M, fin, fout,
                          _lib.HD_MLP_EPI_SILU_BWD, None, D.ptr(z_prev), None, D.ptr(dzp), fin, st)
                dz = dzp
        return grads

    def _adam(self, grads, lr, b1=0.9, b2=0.999, eps=1e-8):
        st = D.stream_ptr()
        self.step += 1
        for l, (dW, db) in enumerate(grads):
            _lib.call("hd_mlp_adam", self.W[l].numel(), D.ptr(self.W[l]), D.ptr(dW), D.ptr(self.mW[l]),
                      D.ptr(self.vW[l]), lr, b1, b2, eps, self.step, D.ptr(self.Wb[l]), st)
            _lib.call("hd_mlp_adam", self.b[l].numel(), D.ptr(self.b[l]), D.ptr(db), D.ptr(self.mb[l]),
                      D.ptr(self.vb[l]), lr, b1, b2, eps, self.step, None, st)

    def loss_and_grads(self, X01, Yn):
        """Device loss (MSE on standardised targets) and gradients for one batch; X01, Yn numpy or tensors."""
        x = D.to_dev(np.asarray(X01, dtype=np.float32), dtype=torch.float32, slots=True)
        t = D.to_dev(np.asarray(Yn, dtype=np.float32), dtype=torch.float32, slots=True)
        step = _TrainStep.of(self, x, t, x.shape[0])
        if step is not None:
            loss = torch.zeros(1, dtype=torch.float32, device=x.device)
            y = _f32((x.shape[0], self.sizes[-1]))
            grads = [(torch.empty_like(W), torch.empty_like(b)) for W, b in zip(self.W, self.b)]
            step(None, x.shape[0], loss, y=y, grads=grads)
            return loss, grads, y
        xb = x.to(torch.bfloat16).contiguous()
        y, cache = self._forward(xb, keep=True)
        dy = _bf16(y.shape)
        loss = torch.zeros(1, dtype=torch.float32, device=y.device)
        _lib.call("hd_mlp_mse", D.ptr(y), D.ptr(t), y.numel(), D.ptr(dy), D.ptr(loss), D.stream_ptr())
        return loss, self._backward(cache, dy), y

    # ---- public API ----
    def fit(self, X, Y, epochs=200, batch=1024, lr=1e-3, seed=0, x_lo=None, x_hi=None, verbose=0, lr_min=None,
            rescale=True):
        """Train on parameters X (S, n_in) and targets Y (S, n_out); returns the per-epoch mean loss.

        Adam at ``lr``; with ``lr_min`` the step size follows a cosine from ``lr`` down to ``lr_min``
        over the epochs.  ``rescale=False`` keeps the input box and target scaling of an earlier fit
        (continued training).
        """
        X = np.asarray(X, dtype=float)
        Yn = D.to_dev(np.asarray(Y, dtype=float), slots=True)
        if rescale:
            self.x_lo = X.min(axis=0) if x_lo is None else np.asarray(x_lo, float)
            self.x_hi = X.max(axis=0) if x_hi is None else np.asarray(x_hi, float)
            mean, std = Yn.mean(dim=0), Yn.std(dim=0, unbiased=False).clamp(min=1e-6)
            self.y_mean, self.y_std = D.to_host(mean), D.to_host(std)
        else:
            mean, std = D.to_dev(self.y_mean), D.to_dev(self.y_std)
        X01 = torch.as_tensor(self._x01(X), dtype=torch.float32).to(D.require_device()).contiguous()
        Yn = ((Yn - mean) / std).to(torch.float32)
        S = X.shape[0]
        gen = torch.Generator(device="cpu").manual_seed(seed)
        hist = []
        step = _TrainStep.of(self, X01, Yn, min(batch, S))
        for ep in range(epochs):
            lr_ep = lr if lr_min is None else lr_min + 0.5 * (lr - lr_min) * (1.0 + np.cos(np.pi * ep / epochs))
            perm = torch.randperm(S, generator=gen).to(X01.device)
            tot = torch.zeros(1, dtype=torch.float32, device=X01.device)
            nb = 0
            for s0 in range(0, S - batch + 1 if S >= batch else 1, batch):
                idx = perm[s0:s0 + batch]
                if step is not None:
                    step(idx, idx.numel(), tot, lr=lr_ep)
                    nb += 1
                    continue
                xb = X01[idx].to(torch.bfloat16).contiguous()
                t = Yn[idx].contiguous()
                y, cache = self._forward(xb, keep=True)
                dy = _bf16(y.shape)
                _lib.call("hd_mlp_mse", D.ptr(y), D.ptr(t), y.numel(), D.ptr(dy), D.ptr(tot), D.stream_ptr())
                self._adam(self._backward(cache, dy), lr_ep)
                nb += 1
            hist.append(float(tot.item()) / max(nb, 1))
            if verbose and (ep + 1) % verbose == 0:
                print(f"surrogate: epoch {ep + 1}/{epochs} loss {hist[-1]:.4e}", flush=True)
        return np.array(hist)

    def predict_device(self, X01_bf16):
        """Standardised outputs (M, n_out) f32 for device inputs already in [0, 1] (bf16)."""
        net = self._net()
        if net is not None and X01_bf16.dtype == torch.bfloat16 and X01_bf16.dim() == 2 and X01_bf16.shape[0] > 0 \
                and X01_bf16.shape[1] == self.sizes[0]:
            y = _f32((X01_bf16.shape[0], self.sizes[-1]))
            _lib.call("hd_mlp_forward", C.addressof(net), D.ptr(X01_bf16), None, None, y.shape[0], D.ptr(y), None,
                      D.stream_ptr())
            return y
        y, _ = self._forward(X01_bf16, keep=False)
        return y

    # ---- persistence ----
    def save(self, path, **meta):
        """Weights (FP32 masters), scaling and optional metadata arrays to an ``.npz`` file."""
        arrs = {f"W{l}": self.W[l].cpu().numpy() for l in range(self.nlayers)}
        arrs.update({f"b{l}": self.b[l].cpu().numpy() for l in range(self.nlayers)})
        arrs.update(sizes=np.array(self.sizes), x_lo=self.x_lo, x_hi=self.x_hi, y_mean=self.y_mean,
                    y_std=self.y_std, step=np.array(self.step))
        for k, v in meta.items():
            arrs["meta_" + k] = np.asarray(v)
        np.savez(path, **arrs)

    @classmethod
    def load(cls, path):
        """Model saved by :meth:`save` (no pickled objects); metadata in ``.meta``."""
        with np.load(path, allow_pickle=False) as fh:
            sizes = [int(v) for v in fh["sizes"]]
            net = cls(n_in=sizes[0], hidden=sizes[1:-1], n_out=sizes[-1])
            dev = D.require_device()
            for l in range(net.nlayers):
                net.W[l] = torch.as_tensor(fh[f"W{l}"]).to(dev).contiguous()
                net.b[l] = torch.as_tensor(fh[f"b{l}"]).to(dev).contiguous()
                net.Wb[l] = net.W[l].to(torch.bfloat16)
            net.x_lo, net.x_hi = fh["x_lo"], fh["x_hi"]
            net.y_mean, net.y_std = fh["y_mean"], fh["y_std"]
            net.step = int(fh["step"])
            net.meta = {k[5:]: fh[k] for k in fh.files if k.startswith("meta_")}
        return net

    def predict(self, X, chunk=1 << 17):
        """log10 h_c percentile spectra (M, n_out) for parameters X (M, n_in)."""
        X = np.asarray(X, dtype=float)
        if chunk < 1:
            raise ValueError(f"chunk={chunk}: at least one row")
        net = self._net()
        if net is not None and X.ndim == 2 and X.shape[0] > 0 and X.shape[1] == self.sizes[0]:
            # scaling to and from the training box on the device: the same double operations
            n_in, n_out = self.sizes[0], self.sizes[-1]
            scale = np.empty(2 * (n_in + n_out))
            scale[:n_in], scale[n_in:2 * n_in] = self.x_lo, np.subtract(self.x_hi, self.x_lo)
            scale[2 * n_in:-n_out], scale[-n_out:] = self.y_std, self.y_mean
            out = np.empty((X.shape[0], n_out))
            one = X.nbytes <= D.STAGE_MAX_BYTES // 2 and X.shape[0] <= chunk
            if one:      # a small call: the scaling and the rows in one upload
                up = D.to_dev(np.concatenate([scale, X.ravel()]))
                scale, X = up[:scale.size], up[scale.size:].view(X.shape)
            else:
                scale = D.to_dev(scale)
            for s0 in range(0, X.shape[0], chunk):
                raw = X if one else D.to_dev(X[s0:s0 + chunk], slots=True)
                y = D.empty((raw.shape[0], n_out))
                _lib.call("hd_mlp_forward", C.addressof(net), None, D.ptr(raw), D.ptr(scale), y.shape[0], None,
                          D.ptr(y), D.stream_ptr())
                D.to_host(y, out=out[s0:s0 + chunk])
            return out
        X01 = np.asarray(self._x01(X), dtype=np.float32)
        out = []
        for s0 in range(0, X01.shape[0], chunk):
            xb = D.to_dev(X01[s0:s0 + chunk], dtype=torch.float32).to(torch.bfloat16).contiguous()
            out.append(D.to_host(self.predict_device(xb)).astype(float))
        return np.concatenate(out) * self.y_std + self.y_mean


class _TrainStep:
    """Batches of a network's training on the whole-pass kernels (hd_mlp_train_step), with the
    workspace of one batch."""

    @classmethod
    def of(cls, model, X, T, rows):
        """For device inputs X (S, n_in) and targets T (S, n_out) f32, batches of at most ``rows``; None
        where the kernels do not take the network or the arrays do not fit it."""
        net = model._net()
        if (net is None or model.sizes[-1] > 256 or rows < 1 or X.shape[1:] != (model.sizes[0],)
                or T.shape != (X.shape[0], model.sizes[-1])):
            return None
        return cls(model, net, X, T, rows)

    def __init__(self, model, net, X, T, rows):
        self.model, self.net, self.X, self.T, self.rows = model, net, X, T, rows
        self.ws = D.workspace(_lib.size("hd_mlp_train_workspace_size", C.addressof(net), rows))
        self.par = _lib.MlpParams()
        for l in range(model.nlayers):
            for name, ts in (("w", model.W), ("b", model.b), ("wb", model.Wb), ("mw", model.mW), ("vw", model.vW),
                             ("mb", model.mb), ("vb", model.vb)):
                getattr(self.par, name)[l] = D.ptr(ts[l])
        self.fresh = True

    def __call__(self, idx, rows, loss, lr=0.0, y=None, grads=None, b1=0.9, b2=0.999, eps=1e-8):
        """One batch: rows ``idx`` (device int64; None: the first ``rows``) with an Adam step, or, with
        ``grads``, the gradients alone; adds the mean squared error to ``loss``."""
        par = self.par
        if grads is None:
            self.model.step += 1
        else:
            par = _lib.MlpParams()
            for l, (dW, db) in enumerate(grads):
                par.dw[l], par.db[l] = D.ptr(dW), D.ptr(db)
        _lib.call("hd_mlp_train_step", C.addressof(self.net), C.addressof(par), D.ptr(self.X), D.ptr(self.T),
                  D.ptr(idx), rows, D.ptr(loss), D.ptr(y), int(self.fresh), lr, b1, b2, eps, max(self.model.step, 1),
                  D.ptr(self.ws), self.ws.numel(), D.stream_ptr())
        self.fresh = False


class SurrogateWithFallback:
    """Surrogate inside the training box; the plain GPU SAM outside it and on a judged fraction.

    The plain SAM answer for parameter rows is the library's: ``gwb_for_params`` over ``pspace``
    with ``nfreqs`` frequencies of a ``pta_dur`` [yr] PTA and ``nreals`` realizations, reduced by
    :func:`targets_from_gwb`.
    """

    def __init__(self, model, pspace, nfreqs=30, nreals=500, pta_dur=None, streams=3):
        from . import librarian
        self.model = model
        self.pspace = pspace
        self.nfreqs = int(nfreqs)
        self.nreals = int(nreals)
        self.pta_dur = librarian.DEF_PTA_DUR if pta_dur is None else pta_dur
        self.streams = streams

    def sam_targets(self, X, seed=0):
        """(n, 3F) log10 percentile spectra of the plain GPU SAM for parameter rows X (n, D)."""
        from . import librarian, utils
        from .constants import YR
        X = np.atleast_2d(np.asarray(X, dtype=float))
        if X.shape[0] == 0:
            return np.zeros((0, self.model.sizes[-1]))
        fe = utils.pta_freqs(dur=self.pta_dur * YR, num=self.nfreqs)[1]
        return librarian.gwb_for_params(self.pspace, X, fobs_edges=fe, nreals=self.nreals, seeds=seed,
                                        streams=self.streams, reduce=targets_from_gwb)

    def predict(self, X, judge_frac=0.01, seed=0):
        """(Y (n, 3F), report).  Report: counts, the judged rows' median / 95th-percentile absolute
        error [dex] over all outputs, and wall-clock seconds of each part."""
        import time
        X = np.asarray(X, dtype=float)
        t0 = time.perf_counter()
        inside = self.model.in_box(X)
        Y = np.empty((X.shape[0], self.model.sizes[-1]))
        if inside.any():
            Y[inside] = self.model.predict(X[inside])
        t1 = time.perf_counter()
        out_idx = np.flatnonzero(~inside)
        if out_idx.size:
            Y[out_idx] = self.sam_targets(X[out_idx], seed=seed)
        t2 = time.perf_counter()
        rng = np.random.default_rng(seed)
        cand = np.flatnonzero(inside)
        nj = int(np.ceil(judge_frac * cand.size)) if cand.size else 0
        judged = np.sort(rng.choice(cand, size=nj, replace=False)) if nj else np.array([], dtype=int)
        err = np.abs(Y[judged] - self.sam_targets(X[judged], seed=seed + 1_000_003)) if nj else None
        t3 = time.perf_counter()
        report = {"n": int(X.shape[0]), "n_fallback": int(out_idx.size), "n_judged": int(nj),
                  "median_dex_error": float(np.median(err)) if nj else None,
                  "p95_dex_error": float(np.percentile(err, 95)) if nj else None,
                  "t_surrogate_s": t1 - t0, "t_fallback_s": t2 - t1, "t_judge_s": t3 - t2, "t_total_s": t3 - t0}
        return Y, report
