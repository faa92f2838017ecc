"""Differentiable recurrent LIF network: device forward, exact adjoint backward.

The network: `n_in` Poisson sources -> `N` LIF neurons with an exponential
current (dv/dt = (I + bias - v)/tau_m, dI/dt = -I/tau_s, threshold v > theta,
reset v = 0, exact integration, no refractoriness), sparse input and recurrent
weights (`on_pre: I += w`), many independent trials (one workgroup each).  The
neuron update is Brian's own optimised statements for this model
(brian2_amd/specs/lif.json); the pathways run in Brian's schedule order (by
name: syn_in_pre, then syn_rec_pre), each a left fold in (source, synapse)
order, so a trial's forward pass is bit-identical to the cython runtime.

Loss per run (mean over trials b):
    L = 1/B sum_b [ sum_r ((t_br - target_r) / t_ref)^2
                    + c_v / (N T) sum_k sum_j (v_bkj / theta)^2 ]
t_br is the first spike time of readout neuron r (the first `n_readout`
neurons), linearly interpolated inside the step of the threshold crossing
between the state before the step and the updated state; v_bkj the membrane
potential after step k (after reset).  A readout that never spikes
contributes (T dt - target)^2 and no gradient.

Backward: the exact adjoint of the discrete forward map.  Per step
    u  = C + B I + A v          (the statements are linear in v, I: A, B, C and
    I' = beta I + sum_i s_i w     beta are read off them with autograd)
    v' = (1 - s) u,   s = [u > theta]
run in reverse time: lam_u = (1 - s)(lam_v' + dL/dv') (the reset is the jump
term: nothing flows back through a reset), plus the first-spike terms
dt*dt/du, dt*dt/dv at the crossing step; lam_v = A lam_u, lam_I = B lam_u +
beta lam_I'; weight gradients are event-based: dL/dw_ij += lam_I'_j at every
step where source i spiked.  Spikes themselves carry no gradient (a
perturbation that creates or deletes no spike leaves them unchanged).  The
state is kept at the start of every block of a few steps (or, where that is
too much memory, of every `ckpt_every` steps or not at all: LIFNetwork._form);
the backward pass recomputes a block forward from there, then walks it in
reverse.  Weight
gradients accumulate per trial (no atomics) and are summed over trials in a
fixed order.
"""
import ctypes
import os
import weakref

import numpy as np

from . import _lib
from .codegen import ParamStruct, filled, source_header, translate_block
from .kernels import LDS_BYTES, _rename, scalar_values
from .runtime import Device, Model

L = _lib.lib
SEED = 1234
S_RATE, S_POISSON, S_CONN_IN, S_CONN_REC, S_W_IN, S_W_REC, S_V0_LIF, S_TARGET = 9, 10, 11, 12, 13, 14, 15, 16
LIF = dict(N=1000, NE=800, n_in=200, tau_m=0.02, tau_s=0.005, theta=0.01, bias=0.0105, p=0.1,
           rate_lo=5.0, rate_hi=50.0, w_scale=0.5e-3, n_steps=2000, n_readout=10, t_ref=0.01, c_v=0.1)
BLOCK = 1024
KEEP_BYTES = 4 << 30  # that a network's losses hold for their backward passes at most, all together


def _torch():
    import torch

    return torch


def _rng_header():
    here = os.path.dirname(os.path.abspath(__file__))
    with open(os.path.join(here, "csrc", "hb_rng.h")) as f:
        return f.read()


def lif_inputs(trials, seed=SEED, c=LIF):
    """Inputs from the shared generator (csrc/hb_rng.h streams 9-16): input
    rates r_i = 5 + 45 U Hz; Bernoulli(0.1) input and recurrent connectivity
    (CSR by source, targets ascending); weights sigma * z (z standard normal,
    polar method; sigma = 0.5 mV / sqrt(expected fan-in)); v0 = theta * U per
    (trial, neuron); readout targets 20 + 160 U ms.  The Poisson trains are
    drawn on the device: input i spikes at step k of trial b iff
    U(S_POISSON, (b n_in + i) T + k) < r_i dt."""
    from .synth import bernoulli_host, polar_normal, uniform

    n_in, N = c["n_in"], c["N"]
    rates = c["rate_lo"] + (c["rate_hi"] - c["rate_lo"]) * uniform(seed, S_RATE, np.arange(n_in, dtype=np.uint64))
    pre_in, post_in = bernoulli_host(seed, 0, n_in, N, c["p"], stream=S_CONN_IN)
    pre_rec, post_rec = bernoulli_host(seed, 0, N, N, c["p"], stream=S_CONN_REC)
    sigma = c["w_scale"] / np.sqrt(c["p"] * (n_in + N))
    w_in = sigma * polar_normal(seed, len(pre_in), S_W_IN)
    w_rec = sigma * polar_normal(seed, len(pre_rec), S_W_REC)
    v0 = c["theta"] * uniform(seed, S_V0_LIF, np.arange(trials * N, dtype=np.uint64)).reshape(trials, N)
    targets = 0.02 + 0.16 * uniform(seed, S_TARGET, np.arange(c["n_readout"], dtype=np.uint64))
    return dict(rates=rates, pre_in=pre_in, post_in=post_in, pre_rec=pre_rec, post_rec=post_rec,
                w_in=w_in, w_rec=w_rec, v0=v0, targets=targets, sigma=sigma)


def linear_map(spec, consts, dt, float_t="double"):
    """The update statements of a two-variable linear model as v' = C + B I + A v,
    I' = beta I, with the coefficients and their derivatives with respect to
    tau_m and tau_s (autograd through the scalar block on the host)."""
    torch = _torch()
    with torch.enable_grad():  # also when called from an autograd backward pass
        return _linear_map(torch, spec, consts, dt)


def _linear_map(torch, spec, consts, dt):
    import math

    tau = {n: torch.tensor(float(consts[n]), dtype=torch.float64, requires_grad=True) for n in ("tau_m", "tau_s")}
    env = {k: torch.tensor(float(v), dtype=torch.float64) for k, v in consts.items() if k not in tau}
    env.update(tau)
    env["dt"] = torch.tensor(dt, dtype=torch.float64)
    fns = {"exp": torch.exp, "expm1": torch.expm1, "log": torch.log, "sqrt": torch.sqrt}
    for st in spec.scalar:
        env[st["var"]] = eval(st["expr"], {"__builtins__": {}}, {**fns, **env})
    v = torch.tensor(0.0, dtype=torch.float64, requires_grad=True)
    I_ = torch.tensor(0.0, dtype=torch.float64, requires_grad=True)
    env.update(v=v, I=I_)
    loc = dict(env)
    for st in spec.vector:
        loc[st["var"]] = eval(st["expr"], {"__builtins__": {}}, {**fns, **loc})
    vn, In = loc["v"], loc["I"]
    (A, B) = torch.autograd.grad(vn, (v, I_), create_graph=True)
    (beta_v, beta) = torch.autograd.grad(In, (v, I_), create_graph=True, allow_unused=True)
    if beta_v is not None and float(beta_v) != 0.0:
        raise NotImplementedError("the synaptic current's update depends on v")
    C = vn - (A * v + B * I_)
    coef = {"A": A, "B": B, "C": C, "beta": beta}
    out = {k: float(x.detach()) for k, x in coef.items()}
    for k, x in coef.items():
        g = torch.autograd.grad(x, (tau["tau_m"], tau["tau_s"]), retain_graph=True, allow_unused=True)
        out[f"d{k}"] = tuple(0.0 if gi is None else float(gi) for gi in g)
    # linearity check: the update at (1, 1) must equal C + B + A
    loc2 = dict(env)
    loc2.update(v=torch.tensor(1.0, dtype=torch.float64), I=torch.tensor(1.0, dtype=torch.float64))
    for st in spec.vector:
        loc2[st["var"]] = eval(st["expr"], {"__builtins__": {}}, {**fns, **loc2})
    if not math.isclose(float(loc2["v"].detach()), out["C"] + out["B"] + out["A"], rel_tol=1e-12, abs_tol=1e-15):
        raise NotImplementedError("the neuron update is not linear in (v, I)")
    return out


class LIFNetwork:
    """Trials of the differentiable LIF network on the device (see module doc).

    keep_bytes: device memory that the network's losses may hold for their backward passes,
    all together (default KEEP_BYTES); a loss beyond that is simulated again by its backward
    pass (_form)."""

    def __init__(self, trials=256, seed=SEED, config=None, weight_dtype="float", ckpt_every=100, keep_bytes=None):
        torch = _torch()
        self.c = dict(LIF if config is None else config)
        c = self.c
        self.B, self.N, self.n_in, self.T = int(trials), c["N"], c["n_in"], c["n_steps"]
        self.R = c["n_readout"]
        if self.N > BLOCK or self.n_in > BLOCK:
            raise NotImplementedError(f"groups of more than {BLOCK} neurons")
        if self.T % ckpt_every:
            raise ValueError("n_steps must be a multiple of ckpt_every")
        self.C = int(ckpt_every)
        self.S = self.T // self.C
        self.seed = int(seed)
        self.dt = 1e-4
        self.wt = weight_dtype
        self.keep_bytes = KEEP_BYTES if keep_bytes is None else int(keep_bytes)
        self._held = []  # weak references to the tensors held for backward passes
        self._shape()
        self._kernels()
        inp = lif_inputs(self.B, seed, c)
        self.inp = inp
        self.D = Device.get()
        dev = lambda a, dt: torch.from_numpy(np.ascontiguousarray(a).astype(dt)).to("cuda")  # noqa: E731
        # U < rate dt for a U of 53 bits over 2^53: the bits below ceil(rate dt 2^53), exactly
        # (never for a rate below 0 or without a value, always from 1 / dt on)
        bound = np.ceil(np.ldexp(inp["rates"] * self.dt, 53))
        self.r_dt = dev(np.where(bound > 0.0, np.minimum(bound, 2.0 ** 53), 0.0), np.int64)
        self.n_syn_in, self.n_syn_rec = len(inp["pre_in"]), len(inp["pre_rec"])
        # places of the synapses in the dense matrix; first synapse and synapses of each row
        niw, nsw = self._words()
        width = self.block * self.per_thread
        self.dense_size = (niw + nsw) * 64 * width
        self.in_at = dev(inp["pre_in"].astype(np.int64) * width + inp["post_in"], np.int64)
        self.rec_at = dev((inp["pre_rec"].astype(np.int64) + niw * 64) * width + inp["post_rec"], np.int64)
        rows = np.zeros(((niw + nsw) * 64, 2), np.int32)
        for pre, first in ((inp["pre_in"], 0), (inp["pre_rec"], niw * 64)):
            n = np.bincount(pre, minlength=1) if len(pre) else np.zeros(1, np.int64)
            rows[first:first + len(n), 0], rows[first:first + len(n), 1] = np.where(n > 0, np.cumsum(n) - n, 0), n
        self.row_at = dev(rows, np.int32)
        self.post_in = dev(inp["post_in"] if len(inp["post_in"]) else [0], np.int32)
        self.post_rec = dev(inp["post_rec"] if len(inp["post_rec"]) else [0], np.int32)
        npw = np.float32 if weight_dtype == "float" else np.float64
        self.w_in0 = dev(inp["w_in"].astype(npw), npw)
        self.w_rec0 = dev(inp["w_rec"].astype(npw), npw)
        self.v0 = dev(inp["v0"], np.float64)
        self.targets = dev(inp["targets"], np.float64)
        self._inp_fn = self.D.function(self.fwd_source, "lif_inputs")
        self._fwd_fn = self.D.function(self.fwd_source, "lif_forward")
        self._bwd_fns = {self.keep: self.D.function(self.bwd_source, "lif_backward")}

    # ------------------------------------------------------------------ kernels
    def _shape(self):
        """Threads of a trial's workgroup and neurons per thread: eight waves at most with float
        weights, sixteen with double ones, whose rows are twice the loads of a thread.  500
        steps forward and backward with 4 / 8 / 16 waves, ms: float weights, 9 trials of 1000
        neurons 1.53 / 1.39 / 1.40, 256 trials 1.53 / 1.41 / 1.44; double weights, 9 trials of
        777 neurons 1.65 / 1.48 / 1.37, 256 trials of 1000 1.82 / 1.66 / 1.56."""
        self.block = 64 * min(8 if self.wt == "float" else 16, -(-self.N // 64))
        self.per_thread = -(-self.N // self.block)
        # steps of a block of the backward pass: what its LDS holds (16 bytes per neuron and step,
        # 2 per possible event), a raster word per thread, at most 8
        words = sum(self._words())
        step = 16 * self.block * self.per_thread + 2 * 64 * words
        self.sub = max(1, min(8, self.block // words, (LDS_BYTES - 4096) // step))
        self.n_sub = -(-self.C // self.sub)
        # whether the states at the blocks' starts are kept, if there is room (_form)
        self.keep = self._bytes(self.sub) <= self.keep_bytes

    def _bytes(self, every):
        """What a loss holds with the state kept at every so many steps of an interval: the
        states, and every spike."""
        return self.B * (16 * self.S * -(-self.C // every) * self.N + 8 * self.T * sum(self._words()))

    def _form(self, held=True):
        """Steps of an interval from one kept state to the next: of a block (`sub`), of the
        whole interval (`C`), or 0, no state.

        The blocks' states (256 trials of 1000 neurons and 2000 steps: 1.11 GB with the spikes)
        are for a few losses at a time: together with those of other losses alive they stay
        within keep_bytes, and take a quarter of the device's free memory at most (asked for
        from 64 MB on).  A loss beyond that holds the intervals' states (0.16 GB), then
        nothing but its weights; the only loss alive always holds the intervals'.  held: whether
        the states are held from the forward pass to the backward pass."""
        self._held = [r for r in self._held if r() is not None]
        alive = [t for t in (r() for r in self._held) if t is not None] if held else []
        now, need = sum(t.numel() * t.element_size() for t in alive), self._bytes(self.sub)
        if now + need <= self.keep_bytes and (need < 64 << 20 or 4 * need <= _torch().cuda.mem_get_info()[0]):
            return self.sub
        return self.C if now == 0 or now + self._bytes(self.C) <= self.keep_bytes else 0

    def _kernels(self):
        """Loads the model's statements and generates both kernel sources."""
        self.model = Model.load("lif")
        self.su, self.th, self.rs = (self.model.group[k] for k in ("stateupdate", "threshold", "reset"))
        th = [(st["var"], st["expr"]) for st in self.th.vector]
        rs = [(st["var"], st["op"], st["expr"]) for st in self.rs.vector]
        if th != [("_cond", "v > theta")] or rs != [("v", "=", "0.0")]:
            raise NotImplementedError("threshold 'v > theta' and reset 'v = 0' expected")
        self.su_code = self._su_lines()
        self.fwd_source = self._fwd_source()
        self.bwd_source = self._bwd_source(self.keep)

    @classmethod
    def sources(cls, config=None, weight_dtype="float", trials=256, ckpt_every=100):
        """The generated kernel sources (no device needed)."""
        self = cls.__new__(cls)
        self.c = dict(LIF if config is None else config)
        self.N, self.dt, self.wt = self.c["N"], 1e-4, weight_dtype
        self.B, self.C, self.T, self.S = trials, ckpt_every, self.c["n_steps"], self.c["n_steps"] // ckpt_every
        self.keep_bytes = KEEP_BYTES
        self._shape()
        self._kernels()
        return self.fwd_source, self.bwd_source

    def _su_lines(self):
        types = {"v": "double", "I": "double", "t": "double", "dt": "double", "N": "int", "i": "int", "_idx": "int"}
        names = {}
        for n in ("_lio_1", "_lio_2", "_lio_3", "_lio_4"):
            types[n] = "double"
        sc = scalar_values(self.su, {"dt": self.dt, "N": self.N, **{k: self.c[k] for k in ("tau_m", "tau_s", "bias")}},
                           "double")
        self.su_scalars = sorted(sc)
        for n in self.su_scalars:
            types[n] = sc[n][1]
            names[n] = f"p.su_{n}"
        lines = translate_block(self.su.vector, self.su.conditional_write, types, set(), "double")
        return _rename(lines, names)

    def _struct(self, name, backward):
        WT = self.wt
        ps = ParamStruct(name)
        ps.val("n_seg", "int")    # checkpoint intervals of a run
        ps.val("n_steps", "int")  # steps of an interval
        ps.val("T_total", "int")
        ps.val("seed", "unsigned long long")
        ps.val("n_in", "int")
        ps.val("N", "int")
        ps.val("R", "int")
        ps.val("trial0", "int")
        ps.val("n_trials", "int")
        ps.val("theta", "double")
        ps.val("dt", "double")
        for n in self.su_scalars:
            ps.val(f"su_{n}", "double")
        ps.ptr("dense", WT, const=True)  # weights by (source, target), 0 where there is no synapse
        ps.ptr("raster", "unsigned long long", const=backward)  # [trial][step][words]
        ps.ptr("ckpt_v", "double", const=backward)
        ps.ptr("ckpt_I", "double", const=backward)
        ps.ptr("fs_step", "int", const=backward)
        if not backward:
            ps.val("every", "int")    # steps from one kept state to the next, in an interval (0: none)
            ps.val("n_keep", "int")   # kept states of an interval
            ps.ptr("r_dt", "unsigned long long", const=True)
            ps.ptr("v", "double")
            ps.ptr("I", "double")
            ps.ptr("fs_vprev", "double")
            ps.ptr("fs_u", "double")
            ps.ptr("l2", "double")
            ps.ptr("spk_i", "int")
            ps.ptr("spk_step", "int")
            ps.ptr("spk_n", "long long")
            ps.val("spk_cap", "long long")
        else:
            ps.val("A", "double")
            ps.val("B", "double")
            ps.val("beta", "double")
            ps.val("coef_fs", "double")
            ps.val("coef_v", "double")
            ps.ptr("targets", "double", const=True)
            ps.ptr("row_at", "int", const=True)  # first synapse and synapses of each row
            ps.ptr("post_in", "int", const=True)
            ps.ptr("post_rec", "int", const=True)
            ps.ptr("sub_v", "double")
            ps.ptr("sub_I", "double")
            ps.val("n_syn_in", "long long")
            ps.val("n_syn_rec", "long long")
            ps.ptr("g_in", "double")
            ps.ptr("g_rec", "double")
            ps.ptr("gacc", "double")
        return ps

    def _words(self):
        """64-bit words of a step's spikes: the inputs', then the neurons'."""
        return max(1, -(-self.c["n_in"] // 64)), -(-self.N // 64)

    def _head(self, ps, name):
        """What both kernels begin with.

        Thread x of the trial's workgroup has the neurons q*T + x, q < Q (few waves, so
        that what every wave does alike is done few times).  Rows of the dense matrices
        are numbered by the raster's bits (inputs, then neurons, in schedule order), with
        a column per neuron: every thread reads its own columns of each spiking source's
        row and adds them up itself, in (pathway, source) order, without a barrier
        between the rows."""
        NIW, NSW = self._words()
        T, Q = self.block, self.per_thread
        return [source_header(T), _rng_header(), ps.c_decl(), f"""
#define HB_NIW {NIW}          // words of a step's input spikes
#define HB_NW {NIW + NSW}           // words of a step
#define HB_Q {Q}             // neurons per thread
#define HB_ROWS 4            // rows in flight
// a step's rows, loaded at once: {Q} columns of each
template <typename V> struct hb_rows {{
    V x[HB_ROWS][HB_Q];
    __device__ __forceinline__ void load(const int u, const int row, const V* col) {{
        #pragma unroll
        for (int q = 0; q < HB_Q; q++) x[u][q] = col[(size_t)row * {T * Q} + q * {T}];
    }}
    __device__ __forceinline__ void add(double (&I)[HB_Q], const int m) const {{
        #pragma unroll
        for (int u = 0; u < HB_ROWS; u++)
            if (u < m)
                #pragma unroll
                for (int q = 0; q < HB_Q; q++) I[q] += (double)x[u][q];
    }}
}};
""", f'extern "C" __global__ void __launch_bounds__({T}) {name}(const {ps.name} p) {{',
            "    const int b = blockIdx.x;",
            "    const int lane = threadIdx.x & 63;",
            "    const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);",
            "    const int N = p.N;",
            "    const double dt = p.dt;",
            "    const size_t bo = (size_t)b * N;",
            f"    const {self.wt}* const col = p.dense + threadIdx.x;",
            f"#define HB_EACH_Q _Pragma(\"unroll\") for (int q = 0; q < HB_Q; q++)",
            f"#define HB_J (q * {T} + (int)threadIdx.x)  // neuron q of the thread",
            "    // stateupdate of neuron j at step k (Brian's statements)",
            "    auto hb_update = [&](const int j, const int k, double& v, double& I) __attribute__((always_inline)) {",
            "        const double t = (double)k * dt;",
            "        const int i = j, _idx = j;",
            "        (void)t; (void)i; (void)_idx;",
            ] + ["        " + x for x in self.su_code] + ["    };"]

    def _sum_lines(self, what, into, n):
        """Lines that add up a value per neuron: wave shuffles over 64 neurons, then the groups
        of 64 in order (n values side by side)."""
        NSW = self._words()[1]
        W = self.block // 64
        return [
            "            HB_EACH_Q {",
            f"                double x[{n}] = {{{', '.join(f'HB_J < N ? {w} : 0.0' for w in what)}}};",
            "                #pragma unroll",
            f"                for (int c = 0; c < {n}; c++) {{",
            "                    for (int o = 32; o > 0; o >>= 1) x[c] += __shfl_down(x[c], o, 64);",
            f"                    if (lane == 0 && q * {W} + wid < {NSW}) s_red[q * {W} + wid][c] = x[c];",
            "                }",
            "            }",
            "            __syncthreads();",
            f"            if ((int)threadIdx.x < {n}) {{",
            "                double acc = 0.0;",
            f"                for (int w = 0; w < {NSW}; w++) acc += s_red[w][threadIdx.x];",
            f"                {into} += acc;",
            "            }",
            "            __syncthreads();",
        ]

    def _fwd_source(self):
        """Forward pass of a trial per workgroup, all steps in one launch.

        A step is one barrier: every wave puts its neurons' spikes as words into LDS (two
        buffers in turn), and behind the barrier reads all words and adds its columns of
        the spiking sources' rows.  The inputs' spikes are drawn by a kernel of its own
        before (lif_inputs), which the whole chip shares; both end up in the raster, from
        which the backward pass knows every spike.  Bound by the chain of a step: update,
        barrier, words, one row fetch (L2).  256 trials of 1000 neurons (fp32 weights):
        2.05 us per step with ordered compactions and a barrier per row (ten barriers a
        step), 1.05 now and 0.05 for the draws."""
        ps = self._struct("hba_fwd", False)
        self.fwd_struct = ps
        NIW, NSW = self._words()
        T, Q = self.block, self.per_thread
        W = T // 64
        k = self._head(ps, "lif_forward")
        k += [
            f"    __shared__ unsigned long long s_ras[64][HB_NW];  // words of the last steps, and the inputs' ahead",
            f"    __shared__ double s_red[{NSW}][1];",
            "    double v[HB_Q], I[HB_Q], l2[HB_Q];",
            "    bool fs_open[HB_Q];",
            "    HB_EACH_Q {",
            "        v[q] = HB_J < N ? p.v[bo + HB_J] : 0.0;",
            "        I[q] = HB_J < N ? p.I[bo + HB_J] : 0.0;",
            "        fs_open[q] = HB_J < p.R && p.fs_step[b * p.R + (HB_J < p.R ? HB_J : 0)] < 0;",
            "        l2[q] = 0.0;",
            "        // waited for here: a wait inside the loop would be for the checkpoints' stores as well",
            "        asm volatile(\"\" : \"+v\"(v[q]), \"+v\"(I[q]));",
            "    }",
            "    double l2_all = p.l2[b];",
            "    long long n_spk = p.spk_i ? p.spk_n[b] : 0;",
            "    const int T = p.n_seg * p.n_steps;",
            "    unsigned long long* const ras = p.raster + (size_t)b * T * HB_NW;",
            "    // the spikes of n steps from k to the raster",
            "    auto hb_flush = [&](const int k, const int n) {",
            f"        for (int x = threadIdx.x; x < n * {NSW}; x += {T})",
            f"            ras[(size_t)(k + x / {NSW}) * HB_NW + HB_NIW + x % {NSW}] = s_ras[(k + x / {NSW}) & 63][HB_NIW + x % {NSW}];",
            "    };",
            "    // the inputs' words of the next 32 steps, read 32 steps ahead (every memory access in",
            "    // flight is waited for with a step's rows)",
            f"    constexpr int AHEAD = (32 * HB_NIW + {T - 1}) / {T};",
            "    unsigned long long ahead[AHEAD];",
            "    auto hb_ahead = [&](const int k) {",
            "        #pragma unroll",
            "        for (int a = 0; a < AHEAD; a++) {",
            f"            const int x = a * {T} + (int)threadIdx.x, s = k + x / HB_NIW;",
            "            ahead[a] = ras[s < T && x < 32 * HB_NIW ? (size_t)s * HB_NW + x % HB_NIW : 0];",
            "        }",
            "    };",
            "    hb_ahead(0);",
            "    size_t kept = (size_t)b * p.n_seg * p.n_keep * N;  // place of the next kept state",
            "    for (int k = 0, c = 0, left = 0; k < T; k++, left--) {  // left: steps to it",
            "        if ((k & 31) == 0) {",
            "            #pragma unroll",
            "            for (int a = 0; a < AHEAD; a++) {",
            f"                const int x = a * {T} + (int)threadIdx.x;",
            "                if (x < 32 * HB_NIW) s_ras[(k + x / HB_NIW) & 63][x % HB_NIW] = ahead[a];",
            "            }",
            "            hb_ahead(k + 32);",
            "            if (k > 0) hb_flush(k - 32, 32);",
            "        }",
            "        if (left == 0 && p.every > 0) {",
            "            HB_EACH_Q if (HB_J < N) { p.ckpt_v[kept + HB_J] = v[q]; p.ckpt_I[kept + HB_J] = I[q]; }",
            "            kept += N;",
            "            left = p.every;",
            "        }",
            "        bool cond[HB_Q], fs_any = false;",
            "        double v_prev[HB_Q];",
            "        unsigned long long mine[HB_Q], word = 0ull;",
            "        HB_EACH_Q {",
            "            v_prev[q] = v[q];",
            "            hb_update(HB_J, k, v[q], I[q]);",
            "            cond[q] = HB_J < N && v[q] > p.theta;",
            "            mine[q] = __builtin_amdgcn_ballot_w64(cond[q]);",
            "            fs_any = fs_any || (cond[q] && fs_open[q]);",
            "            word = lane == q ? mine[q] : word;",
            "        }",
            f"        if (lane < HB_Q && lane * {W} + wid < {NSW}) s_ras[k & 63][HB_NIW + lane * {W} + wid] = word;",
            "        if (__builtin_amdgcn_ballot_w64(fs_any) != 0ull)",
            "            HB_EACH_Q if (cond[q] && fs_open[q]) { // first spike of a readout",
            "                fs_open[q] = false;",
            "                p.fs_step[b * p.R + HB_J] = k; p.fs_vprev[b * p.R + HB_J] = v_prev[q]; p.fs_u[b * p.R + HB_J] = v[q];",
            "            }",
            "        __syncthreads();",
            "        const unsigned long long rd = s_ras[k & 63][lane < HB_NW ? lane : 0];",
            "        const unsigned long long rw = lane < HB_NW ? rd : 0ull;",
            "        // propagation, in schedule order: syn_in_pre, then syn_rec_pre; each a left fold in",
            "        // (source, synapse) order.  Everything about the sources is the same for the wave",
            "        unsigned long long nz = __builtin_amdgcn_ballot_w64(rw != 0ull);",
            "        if (nz != 0ull) {",
            f"            hb_rows<{self.wt}> r;",
            "            const int one = (lane << 6) + __builtin_ctzll(rw | 1ull << 63);  // the word's first source",
            "            const int n_nz = __popcll(nz);",
            "            if (n_nz <= HB_ROWS && __builtin_amdgcn_ballot_w64((rw & (rw - 1ull)) != 0ull && rw != 0ull) == 0ull) {",
            "                // few words of one source each (most steps); a missing one repeats the last:",
            "                // loads without a branch stay in flight",
            "                int l = 0;",
            "                #pragma unroll",
            "                for (int u = 0; u < HB_ROWS; u++) {",
            "                    l = nz != 0ull ? __builtin_ctzll(nz) : l;",
            "                    nz &= nz - 1ull;",
            "                    r.load(u, __builtin_amdgcn_readlane(one, l), col);",
            "                }",
            "                r.add(I, n_nz);",
            "            } else {  // word by word, bit by bit",
            "                for (; nz; nz &= nz - 1ull) {",
            "                    const int l = __builtin_ctzll(nz);",
            "                    unsigned long long bits = ((unsigned long long)(unsigned int)",
            "                        __builtin_amdgcn_readlane((int)(rw >> 32), l) << 32) | (unsigned int)__builtin_amdgcn_readlane((int)rw, l);",
            "                    while (bits) {",
            "                        int m = 0, row = 0;",
            "                        #pragma unroll",
            "                        for (int u = 0; u < HB_ROWS; u++) {",
            "                            m += bits != 0ull ? 1 : 0;",
            "                            row = bits != 0ull ? (l << 6) + __builtin_ctzll(bits) : row;",
            "                            bits &= bits - 1ull;",
            "                            r.load(u, row, col);",
            "                        }",
            "                        r.add(I, m);",
            "                    }",
            "                }",
            "            }",
            "        }",
            "        HB_EACH_Q {",
            "            if (cond[q]) v[q] = 0.0; // reset",
            "            l2[q] += v[q] * v[q];",
            "        }",
            "        if (p.spk_i) { // the step's spikes in ascending order",
            "            const int n_ = lane >= HB_NIW && lane < HB_NW ? __popcll(rw) : 0;",
            "            const int x_ = hb_wave_incl_scan(n_);",
            f"            HB_EACH_Q if (q * {W} + wid < {NSW}) {{",
            f"                const long long at = n_spk + __builtin_amdgcn_readlane(x_ - n_, HB_NIW + q * {W} + wid) "
            "+ __popcll(mine[q] & ((1ull << lane) - 1ull));",
            "                if (cond[q] && at < p.spk_cap) { p.spk_i[(size_t)b * p.spk_cap + at] = HB_J; "
            "p.spk_step[(size_t)b * p.spk_cap + at] = k; }",
            "            }",
            "            n_spk += __builtin_amdgcn_readlane(x_, 63);",
            "        }",
            "        if (++c == p.n_steps) { // an interval's sum",
            "            c = 0; left = 1;",
        ]
        k += self._sum_lines(["l2[q]"], "l2_all", 1)
        k += [
            "            HB_EACH_Q l2[q] = 0.0;",
            "        }",
            "    }",
            "    hb_flush((T - 1) & ~31, T - ((T - 1) & ~31));  // (behind the last interval's barriers)",
            "    HB_EACH_Q if (HB_J < N) { p.v[bo + HB_J] = v[q]; p.I[bo + HB_J] = I[q]; }",
            "    if (threadIdx.x == 0) { p.l2[b] = l2_all; if (p.spk_i) p.spk_n[b] = n_spk; }",
            "}",
            "// input spikes of every trial and step: input i of trial b spikes at step k iff",
            "// U(seed, stream, ((trial0 + b) n_in + i) T_total + k) < rate dt, compared as integers",
            "// (U is 53 bits over 2^53; r_dt: the bound ceil(rate dt 2^53)).  A wave draws a word of",
            "// DRAWS steps one after the other",
            "#define DRAWS 16",
            f'extern "C" __global__ void __launch_bounds__({T}) lif_inputs(const {ps.name} p) {{',
            "    const int lane = threadIdx.x & 63, T = p.n_seg * p.n_steps;",
            f"    const long long u = (long long)blockIdx.x * {W} + (threadIdx.x >> 6);",
            "    const int nk = (T + DRAWS - 1) / DRAWS;",
            "    const int b = (int)(u / (nk * HB_NIW)), w = (int)(u % HB_NIW), k0 = (int)(u / HB_NIW % nk) * DRAWS;",
            "    if (b >= p.n_trials) return;",
            "    const int i = w * 64 + lane;",
            "    const unsigned long long bound = i < p.n_in ? p.r_dt[i] : 0ull;",
            f"    const unsigned long long key = hb_mix64(p.seed ^ hb_mix64({S_POISSON}ull + 0x9e3779b97f4a7c15ULL));",
            "    unsigned long long z = key + (((unsigned long long)(p.trial0 + b) * p.n_in + i) * (unsigned long long)p.T_total"
            " + (unsigned long long)k0 + 1ull) * 0x9e3779b97f4a7c15ULL;",
            "    unsigned long long* const ras = p.raster + ((size_t)b * T + k0) * HB_NW + w;",
            "    for (int s = 0; s < DRAWS && k0 + s < T; s++, z += 0x9e3779b97f4a7c15ULL) {",
            "        const unsigned long long m = __builtin_amdgcn_ballot_w64((hb_mix64(z) >> 11) < bound);",
            "        if (lane == 0) ras[(size_t)s * HB_NW] = m;",
            "    }",
            "}",
        ]
        return "\n".join(k) + "\n"

    def _bwd_source(self, keep):
        """Backward pass of a trial per workgroup, all intervals in one launch.

        With the raster the recomputation of an interval is each thread's own: no spike has
        to be exchanged, and the rows of a step are fetched while the step before it is
        computed.  The steps are taken in blocks of SUB: a block's raster words become a
        list of its events in LDS (step and source, in order; a word per thread).  The states
        at every block's start come from the forward pass (keep) or from a first run through
        the interval from its checkpoint (sub_v, sub_I); from the last block to the first, its steps' states are
        recomputed into LDS (a column per neuron) and walked in reverse.  The adjoint of I is kept in the
        state's place, and the block's weight gradients follow: a wave adds it to the
        synapses of its sources that spiked, in descending step order.
        Bound by the latency of the rows and of the gradients.  256 trials: 5.05 us per
        step with the recomputation through a history of 16 bytes per neuron and step in
        memory, 2.02 with the first run through the interval, 1.36 with the states kept (the
        forward pass 1.00 to 1.05)."""
        ps = self._struct("hba_bwd", True)
        self.bwd_struct = ps
        NIW, NSW = self._words()
        NW = NIW + NSW
        T, Q, SB = self.block, self.per_thread, self.sub
        W = T // 64
        # events of a batch of weight gradients and pieces of 64 synapses of each (longer rows in
        # a loop behind it)
        GP = max(1, min(4, -(-int(1.1 * self.c["p"] * self.N) // 64)))
        GB = max(2, 12 // GP)
        k = self._head(ps, "lif_backward")
        k += [
            f"    __shared__ double s_hv[{SB}][{T * Q}], s_hi[{SB}][{T * Q}];",
            f"    __shared__ unsigned short s_ev[{SB * NW * 64}];  // events of a block: step << 11 | row",
            f"    __shared__ int s_of[{SB + 1}], s_sh[{max(1, T // 64)}];",
            f"    __shared__ double s_red[{NSW}][4];",
            "    double lam_v[HB_Q], lam_I[HB_Q], gA[HB_Q], gB[HB_Q], gC[HB_Q], gbeta[HB_Q], v[HB_Q], I[HB_Q];",
            "    int fs_k[HB_Q];",
            "    HB_EACH_Q {",
            "        lam_v[q] = lam_I[q] = gA[q] = gB[q] = gC[q] = gbeta[q] = 0.0;",
            "        fs_k[q] = HB_J < p.R ? p.fs_step[b * p.R + (HB_J < p.R ? HB_J : 0)] : -1;",
            "    }",
            "    double g_all = threadIdx.x < 4 ? p.gacc[b * 4 + (threadIdx.x & 3)] : 0.0;",
            "    const int C = p.n_steps, T = p.n_seg * C;",
            f"    const int n_sub = (C + {SB - 1}) / {SB};",
            "    const unsigned long long* const ras = p.raster + (size_t)b * T * HB_NW;",
            "    double* const g_in = p.g_in + (size_t)b * p.n_syn_in;",
            "    double* const g_rec = p.g_rec + (size_t)b * p.n_syn_rec;",
            f"    auto hb_len = [&](const int sb) {{ return C - sb * {SB} < {SB} ? C - sb * {SB} : {SB}; }};",
            "    // this thread's word of block sb of interval sg",
            "    const int ws = (int)threadIdx.x / HB_NW;  // its step",
            "    auto hb_word = [&](const int sg, const int sb) {",
            "        const bool in = sg >= 0 && ws < hb_len(sb);",
            f"        const unsigned long long w = ras[in ? (size_t)(sg * C + sb * {SB}) * HB_NW + threadIdx.x : 0];",
            "        return in ? w : 0ull;",
            "    };",
            "    // a block's list of events from the threads' words; returns their number",
            "    auto hb_list = [&](unsigned long long w) {",
            "        int n;",
            "        int x = hb_block_exscan(__popcll(w), s_sh, &n);",
            f"        if (threadIdx.x % HB_NW == 0 && ws < {SB}) s_of[ws] = x;",
            f"        if (threadIdx.x == 0) s_of[{SB}] = n;",
            "        for (; w; w &= w - 1ull) s_ev[x++] = (unsigned short)(ws << 11 | ((int)threadIdx.x % HB_NW * 64 + __builtin_ctzll(w)));",
            "        __syncthreads();",
            "        return n;",
            "    };",
            "    // the first n steps (from step k0) of the block in the list of n_ev events; before step",
            "    // s, keep(s).  Lane l holds event l and the events before step l; the rows of a step are",
            "    // loaded two steps ahead",
            "    auto hb_steps = [&](const int k0, const int n, const int n_ev, auto keep) __attribute__((always_inline)) {",
            "        const int ev = (int)s_ev[lane < n_ev ? lane : 0];",
            f"        const int of = s_of[lane < {SB} ? lane : {SB}];",
            "        auto event = [&](const int x) {",
            "            return (x < 64 ? __builtin_amdgcn_readlane(ev, x) : __builtin_amdgcn_readfirstlane((int)s_ev[x])) & 2047;",
            "        };",
            f"        hb_rows<{self.wt}> r[{SB + 2}];",
            f"        int x[{SB + 2}], m[{SB + 2}];",
            "        auto first = [&](const int s) {  // a step's events and its first rows (a missing one repeats",
            "            x[s] = __builtin_amdgcn_readlane(of, s);  // the last, or row 0: no branch around a load)",
            "            m[s] = __builtin_amdgcn_readlane(of, s + 1) - x[s];",
            "            #pragma unroll",
            "            for (int u = 0; u < HB_ROWS; u++) r[s].load(u, m[s] > 0 ? event(x[s] + (u < m[s] ? u : m[s] - 1)) : 0, col);",
            "        };",
            "        first(0);",
            f"        if ({SB} > 1) first({1 if SB > 1 else 0});",
            "        #pragma unroll",
            f"        for (int s = 0; s < {SB}; s++)",
            "            if (s < n) {",
            "                const int k = k0 + s;",
            "                keep(s);",
            f"                if (s + 2 < {SB}) first(s + 2);",
            "                bool cond[HB_Q];",
            "                HB_EACH_Q { hb_update(HB_J, k, v[q], I[q]); cond[q] = v[q] > p.theta; }",
            "                r[s].add(I, m[s]);",
            "                for (int u = HB_ROWS; u < m[s]; u++) {",
            f"                    hb_rows<{self.wt}> g;",
            "                    g.load(0, event(x[s] + u), col);",
            "                    g.add(I, 1);",
            "                }",
            "                HB_EACH_Q if (cond[q]) v[q] = 0.0;",
            "            }",
            "    };",
            "    // weight gradients.  A wave has the rows whose number is its own modulo the waves (so that",
            "    // a synapse is always added to by the same lane); its events of a block, the latest first,",
            f"    // in batches of {GB}: their synapses' gradients and targets are loaded (hb_take) before the",
            "    // adjoint of the block is known, and added to and stored behind it (hb_give)",
            f"    double gy[{GB}][{GP}];",
            f"    int gt[{GB}][{GP}], ge[{GB}], gn[{GB}], gs[{GB}], g_m = 0, g_c = 0;",
            "    unsigned long long g_left = 0ull;  // the wave's events of the 64 from g_c on still to come",
            "    auto hb_mine = [&](const int n_ev) {",
            "        const int ev = (int)s_ev[g_c + lane < n_ev ? g_c + lane : 0];",
            f"        return __builtin_amdgcn_ballot_w64(g_c + lane < n_ev && (ev & 2047) % {W} == wid);",
            "    };",
            "    auto hb_take = [&](const int n_ev) __attribute__((always_inline)) {",
            "        g_m = 0;",
            "        while (g_left == 0ull && g_c > 0) { g_c -= 64; g_left = hb_mine(n_ev); }",
            f"        int row[{GB}];",
            "        bool again = false;  // a row's second event waits for the next batch",
            "        #pragma unroll",
            f"        for (int u = 0; u < {GB}; u++) {{",
            "            const bool more = g_left != 0ull && !again;",
            "            const int x = more ? 63 - __builtin_clzll(g_left) : 0;",
            "            const int ev = __builtin_amdgcn_readfirstlane((int)s_ev[g_c + x]);",
            "            row[u] = ev & 2047;",
            "            #pragma unroll",
            "            for (int w = 0; w < u; w++) again = again || (more && row[w] == row[u]);",
            "            const bool ok = more && !again;",
            "            g_left = ok ? g_left & ~(1ull << x) : g_left;",
            "            g_m += ok ? 1 : 0;",
            "            gs[u] = ev >> 11;",
            "            ge[u] = ok ? p.row_at[2 * row[u]] : 0;",
            "            gn[u] = ok ? p.row_at[2 * row[u] + 1] : 0;",
            "        }",
            "        #pragma unroll",
            f"        for (int u = 0; u < {GB}; u++) {{",
            "            const bool in = row[u] < HB_NIW * 64;",
            "            double* const g = in ? g_in : g_rec;",
            "            const int* const post = in ? p.post_in : p.post_rec;",
            "            #pragma unroll",
            f"            for (int c = 0; c < {GP}; c++) {{",
            "                const int e = ge[u] + (c * 64 + lane < gn[u] ? c * 64 + lane : 0);",
            "                gy[u][c] = g[e];",
            "                gt[u][c] = post[e];",
            "            }",
            "            ge[u] = in ? ge[u] : ~ge[u];",
            "        }",
            "    };",
            "    auto hb_give = [&]() __attribute__((always_inline)) {",
            "        #pragma unroll",
            f"        for (int u = 0; u < {GB}; u++)",
            "            if (u < g_m) {",
            "                double* const g = ge[u] >= 0 ? g_in : g_rec;",
            "                const int* const post = ge[u] >= 0 ? p.post_in : p.post_rec;",
            "                const int e = (ge[u] >= 0 ? ge[u] : ~ge[u]) + lane;",
            "                #pragma unroll",
            f"                for (int c = 0; c < {GP}; c++)",
            "                    if (c * 64 + lane < gn[u]) g[e + c * 64] = gy[u][c] + s_hi[gs[u]][gt[u][c]];",
            f"                for (int y = {GP} * 64 + lane; y < gn[u]; y += 64) g[e - lane + y] += s_hi[gs[u]][post[e - lane + y]];",
            "            }",
            "    };",
        ]
        if keep:
            k += [
                "    unsigned long long w_next = hb_word(p.n_seg - 1, n_sub - 1);  // of the block to come (read ahead)",
                "    // the states at the start of the block to come, read a block ahead",
                "    double v_next[HB_Q], I_next[HB_Q];",
                "    auto hb_state = [&](const int sg, const int sb) __attribute__((always_inline)) {",
                "        const size_t so = (((size_t)b * p.n_seg + (sg > 0 ? sg : 0)) * n_sub + sb) * N;",
                "        HB_EACH_Q {",
                "            const int j = HB_J < N ? HB_J : N - 1;",
                "            v_next[q] = p.ckpt_v[so + j]; I_next[q] = p.ckpt_I[so + j];",
                "        }",
                "    };",
                "    hb_state(p.n_seg - 1, n_sub - 1);",
                "    for (int sg = p.n_seg - 1; sg >= 0; sg--) {",
                "        for (int sb = n_sub - 1; sb >= 0; sb--) {",
                f"            const int k0 = sg * C + sb * {SB}, n = hb_len(sb);",
                "            const int n_ev = hb_list(w_next);",
                "            w_next = sb > 0 ? hb_word(sg, sb - 1) : hb_word(sg - 1, n_sub - 1);",
                "            HB_EACH_Q { v[q] = HB_J < N ? v_next[q] : 0.0; I[q] = HB_J < N ? I_next[q] : 0.0; }",
                "            hb_state(sb > 0 ? sg : sg - 1, sb > 0 ? sb - 1 : n_sub - 1);",
            ]
        else:
            k += [
                "    unsigned long long w_next = hb_word(p.n_seg - 1, 0);  // of the block to come (read ahead)",
                "    for (int sg = p.n_seg - 1; sg >= 0; sg--) {",
                "        const size_t co = ((size_t)b * p.n_seg + sg) * N + threadIdx.x;",
                f"        HB_EACH_Q {{ v[q] = HB_J < N ? p.ckpt_v[co + q * {T}] : 0.0; I[q] = HB_J < N ? p.ckpt_I[co + q * {T}] : 0.0; }}",
                "        const size_t so = (size_t)b * n_sub * N + threadIdx.x;",
                "        for (int sb = 0; sb < n_sub - 1; sb++) {",
                "            const int n_ev = hb_list(w_next);",
                "            w_next = hb_word(sg, sb + 1);",
                "            HB_EACH_Q if (HB_J < N) {",
                f"                p.sub_v[so + (size_t)sb * N + q * {T}] = v[q]; p.sub_I[so + (size_t)sb * N + q * {T}] = I[q];",
                "            }",
                f"            hb_steps(sg * C + sb * {SB}, {SB}, n_ev, [](const int) {{}});",
                "        }",
                "        for (int sb = n_sub - 1; sb >= 0; sb--) {",
                f"            const int k0 = sg * C + sb * {SB}, n = hb_len(sb);",
                "            const int n_ev = hb_list(w_next);",
                "            w_next = sb > 0 ? hb_word(sg, sb - 1) : hb_word(sg - 1, 0);",
                "            if (sb < n_sub - 1)",
                "                HB_EACH_Q {",
                f"                    v[q] = HB_J < N ? p.sub_v[so + (size_t)sb * N + q * {T}] : 0.0;",
                f"                    I[q] = HB_J < N ? p.sub_I[so + (size_t)sb * N + q * {T}] : 0.0;",
                "                }",
            ]
        k += [
            "            hb_steps(k0, n - 1, n_ev, [&](const int s) { HB_EACH_Q { s_hv[s][HB_J] = v[q]; s_hi[s][HB_J] = I[q]; } });",
            "            HB_EACH_Q { s_hv[n - 1][HB_J] = v[q]; s_hi[n - 1][HB_J] = I[q]; }",
            "            g_c = n_ev > 0 ? (n_ev - 1) & ~63 : 0;",
            "            g_left = hb_mine(n_ev);",
            "            hb_take(n_ev);",
            "            for (int s = n - 1; s >= 0; s--) {",
            "                const int k = k0 + s;",
            "                HB_EACH_Q {",
            "                    const double v_prev = s_hv[s][HB_J], I_prev = s_hi[s][HB_J];",
            "                    double u = v_prev, In = I_prev;",
            "                    hb_update(HB_J, k, u, In);  // the step's update again (identical statements and values)",
            "                    const bool cond = HB_J < N && u > p.theta;",
            "                    const double v_post = cond ? 0.0 : u;",
            "                    double dLdu = cond ? 0.0 : __builtin_fma(p.coef_v * 2.0, v_post, lam_v[q]);",
            "                    double extra = 0.0;",
            "                    if (fs_k[q] == k) { // first spike of a readout: interpolated crossing time",
            "                        const double d = u - v_prev;",
            "                        const double tc = dt * ((double)k + (p.theta - v_prev) / d);",
            "                        const double dLdt = p.coef_fs * 2.0 * (tc - p.targets[HB_J]);",
            "                        dLdu += dLdt * (-dt * (p.theta - v_prev) / (d * d));",
            "                        extra = dLdt * (dt * (p.theta - u) / (d * d));",
            "                    }",
            "                    const double lamJ = lam_I[q];",
            "                    s_hi[s][HB_J] = lamJ;  // for the weight gradients below",
            "                    gA[q] = __builtin_fma(dLdu, v_prev, gA[q]);",
            "                    gB[q] = __builtin_fma(dLdu, I_prev, gB[q]);",
            "                    gC[q] += dLdu;",
            "                    gbeta[q] = __builtin_fma(lamJ, I_prev, gbeta[q]);",
            "                    lam_v[q] = __builtin_fma(p.A, dLdu, extra);",
            "                    lam_I[q] = __builtin_fma(p.B, dLdu, p.beta * lamJ);",
            "                }",
            "            }",
            "            // event-based weight gradients: lam of I after a step at the targets of a source that",
            "            // spiked in it",
            "            __syncthreads();",
            "            hb_give();",
            "            while (g_left != 0ull || g_c > 0) { hb_take(n_ev); hb_give(); }",
            "        }",
            "        {  // the interval's sums",
        ]
        k += self._sum_lines(["gA[q]", "gB[q]", "gC[q]", "gbeta[q]"], "g_all", 4)
        k += [
            "            HB_EACH_Q gA[q] = gB[q] = gC[q] = gbeta[q] = 0.0;",
            "        }",
            "    }",
            "    if (threadIdx.x < 4) p.gacc[b * 4 + threadIdx.x] = g_all;",
            "}",
        ]
        return "\n".join(k) + "\n"

    # ------------------------------------------------------------------ host side
    def _scalars(self, tau_m, tau_s):
        consts = {"tau_m": tau_m, "tau_s": tau_s, "bias": self.c["bias"], "theta": self.c["theta"]}
        sc = scalar_values(self.su, {"dt": self.dt, "N": self.N, **consts}, "double")
        return {n: sc[n][0] for n in self.su_scalars}, consts

    def _launch(self, fn, cls, vals, grid=None):
        buf = bytes(filled(cls, vals))
        stream = ctypes.c_void_p(_torch().cuda.current_stream().cuda_stream)
        _lib.check(L.hb_launch(fn, self.B if grid is None else grid, self.block, 0, stream, buf, len(buf)), "lif launch")

    def _base_vals(self, sc):
        v = dict(n_seg=self.S, n_steps=self.C, T_total=self.T, seed=self.seed, n_in=self.n_in, N=self.N, R=self.R,
                 trial0=0, n_trials=self.B, theta=self.c["theta"], dt=self.dt)
        for n, x in sc.items():
            v[f"su_{n}"] = x
        return v

    def forward(self, w_in, w_rec, tau_m, tau_s, record_spikes=False, spike_cap=200000, linearise=False, keep=True):
        """Runs all trials; returns (loss, saved) where saved holds what the backward
        pass needs (states, spikes, first-spike records).  linearise: with the neurons' linear
        map, which the host then forms while the device runs the steps.  With that, the
        scalars formed once and fewer copies back, 9 trials took 2.24 ms forward and
        backward instead of 2.74 (1.84 with what came since).  keep: whether a backward pass will follow (without states
        and spikes it simulates again)."""
        torch = _torch()
        w_in = w_in.detach().to(self.w_in0.dtype).contiguous()
        w_rec = w_rec.detach().to(self.w_rec0.dtype).contiguous()
        sc, consts = self._scalars(tau_m, tau_s)
        dense = torch.zeros(self.dense_size, dtype=w_in.dtype, device="cuda")
        dense[self.in_at] = w_in
        dense[self.rec_at] = w_rec
        saved = dict(w_in=w_in, w_rec=w_rec, dense=dense, tau_m=tau_m, tau_s=tau_s, scalars=(sc, consts))
        spk = None
        if record_spikes:
            spk_i = torch.zeros((self.B, spike_cap), dtype=torch.int32, device="cuda")
            spk = (spk_i, torch.zeros_like(spk_i), torch.zeros(self.B, dtype=torch.int64, device="cuda"), spike_cap)
        sim = self._simulate(dense, sc, self._form() if keep else 0, spk)
        saved.update(sim)
        if sim["every"]:
            self._held += [weakref.ref(sim[n]) for n in ("ckpt_v", "ckpt_I", "raster")]
        else:
            saved["raster"] = None
        saved["lin"] = linear_map(self.su, consts, self.dt) if linearise else None
        loss, saved["parts"] = self._loss(*(sim[n] for n in ("fs_step", "fs_vprev", "fs_u", "l2")))
        if record_spikes:
            si, ss, n = (x.cpu().numpy() for x in spk[:3])
            if (n > spike_cap).any():
                raise _lib.HipBrianError("spike record buffer overflow")
            saved["spikes"] = [(si[b, :n[b]].copy(), ss[b, :n[b]].astype(np.int64)) for b in range(self.B)]
        return loss, saved

    def _simulate(self, dense, sc, every, spk=None):
        """Runs all trials with the states kept as `every` says (_form); spk: (indices, steps,
        numbers, room) of the spike records.  Returns what the steps leave."""
        torch = _torch()
        B, N, R = self.B, self.N, self.R
        v = self.v0.clone()
        n_keep = -(-self.C // every) if every else 0
        ckpt_v = torch.empty((B, self.S, n_keep, N), dtype=torch.float64, device="cuda")
        fs_vprev = torch.zeros((B, R), dtype=torch.float64, device="cuda")
        out = dict(v=v, I=torch.zeros_like(v), ckpt_v=ckpt_v, ckpt_I=torch.empty_like(ckpt_v),
                   fs_step=torch.full((B, R), -1, dtype=torch.int32, device="cuda"), fs_vprev=fs_vprev,
                   fs_u=torch.zeros_like(fs_vprev), l2=torch.zeros(B, dtype=torch.float64, device="cuda"),
                   raster=torch.empty((B, self.T, sum(self._words())), dtype=torch.int64, device="cuda"))
        vals = self._base_vals(sc)
        vals.update(every=every, n_keep=n_keep, dense=dense.data_ptr(), r_dt=self.r_dt.data_ptr(),
                    **{n: t.data_ptr() for n, t in out.items()})
        if spk is not None:
            vals.update(spk_i=spk[0].data_ptr(), spk_step=spk[1].data_ptr(), spk_n=spk[2].data_ptr(), spk_cap=spk[3])
        cls = self.fwd_struct.ctypes_struct()
        waves = B * -(-self.T // 16) * self._words()[0]  # of lif_inputs
        self._launch(self._inp_fn, cls, vals, -(-waves // (self.block // 64)))
        self._launch(self._fwd_fn, cls, vals)
        return dict(out, every=every)

    def _loss(self, fs_step, fs_vprev, fs_u, l2):
        c, B, N, T = self.c, self.B, self.N, self.T
        k, fv, fu = _torch().stack([fs_step.double(), fs_vprev, fs_u]).cpu().numpy()
        spiked = k >= 0
        with np.errstate(divide="ignore", invalid="ignore"):
            tc = np.where(spiked, self.dt * (k + (c["theta"] - fv) / (fu - fv)), T * self.dt)
        tgt = np.asarray(self.inp["targets"], np.float64)
        fs_term = (((tc - tgt[None, :]) / c["t_ref"]) ** 2).sum() / B
        v_term = c["c_v"] / (N * T * c["theta"] ** 2) * float(l2.sum().item()) / B
        return fs_term + v_term, dict(first_spike=tc, fs_term=fs_term, v_term=v_term)

    def backward(self, saved, grad_out=1.0):
        """Gradients of the loss with respect to (w_in, w_rec, tau_m, tau_s)."""
        torch = _torch()
        c, B, N = self.c, self.B, self.N
        sc, consts = saved["scalars"]
        lin = saved["lin"] or linear_map(self.su, consts, self.dt)
        sim = saved if saved["every"] else self._simulate(saved["dense"], sc, self._form(held=False))
        keep = sim["every"] == self.sub
        if keep not in self._bwd_fns:
            self._bwd_fns[keep] = self.D.function(self._bwd_source(keep), "lif_backward")
        sub_v = torch.empty((1,) if keep else (B, self.n_sub, N), dtype=torch.float64, device="cuda")
        sub_I = torch.empty_like(sub_v)
        # (a pathway without synapses keeps a place to read)
        g_in = torch.zeros((B, max(1, self.n_syn_in)), dtype=torch.float64, device="cuda")
        g_rec = torch.zeros((B, max(1, self.n_syn_rec)), dtype=torch.float64, device="cuda")
        gacc = torch.zeros((B, 4), dtype=torch.float64, device="cuda")
        vals = self._base_vals(sc)
        vals.update(dense=saved["dense"].data_ptr(), raster=sim["raster"].data_ptr(),
                    ckpt_v=sim["ckpt_v"].data_ptr(), ckpt_I=sim["ckpt_I"].data_ptr(),
                    fs_step=saved["fs_step"].data_ptr(), A=lin["A"], B=lin["B"], beta=lin["beta"],
                    coef_fs=grad_out / (B * c["t_ref"] ** 2),
                    coef_v=grad_out * c["c_v"] / (N * self.T * c["theta"] ** 2) / B,
                    targets=self.targets.data_ptr(), row_at=self.row_at.data_ptr(), post_in=self.post_in.data_ptr(),
                    post_rec=self.post_rec.data_ptr(), sub_v=sub_v.data_ptr(),
                    sub_I=sub_I.data_ptr(), n_syn_in=g_in.shape[1], n_syn_rec=g_rec.shape[1], g_in=g_in.data_ptr(),
                    g_rec=g_rec.data_ptr(), gacc=gacc.data_ptr())
        self._launch(self._bwd_fns[keep], self.bwd_struct.ctypes_struct(), vals)
        gw_in = g_in.sum(0)[:self.n_syn_in]
        gw_rec = g_rec.sum(0)[:self.n_syn_rec]
        ga = gacc.sum(0).cpu().numpy()
        g_coef = {"A": ga[0], "B": ga[1], "C": ga[2], "beta": ga[3]}
        g_tau_m = sum(g_coef[k] * lin[f"d{k}"][0] for k in g_coef)
        g_tau_s = sum(g_coef[k] * lin[f"d{k}"][1] for k in g_coef)
        return gw_in, gw_rec, g_tau_m, g_tau_s


def _make_function():
    torch = _torch()

    class LIFLoss(torch.autograd.Function):
        """loss = LIFLoss.apply(net, w_in, w_rec, tau_m, tau_s): forward on the device,
        backward by the exact adjoint (weights and time constants).  recording: whether
        autograd records operations around the call (inside it, it never does)."""

        @staticmethod
        def forward(ctx, net, w_in, w_rec, tau_m, tau_s, recording=True):
            grad = recording and any(ctx.needs_input_grad)
            loss, saved = net.forward(w_in, w_rec, float(tau_m), float(tau_s), linearise=grad, keep=grad)
            ctx.net, ctx.saved = net, saved
            ctx.dtypes = (w_in.dtype, w_rec.dtype, tau_m.dtype, tau_s.dtype)
            return torch.tensor(loss, dtype=torch.float64, device=w_in.device)

        @staticmethod
        def backward(ctx, grad):
            g_in, g_rec, g_m, g_s = ctx.net.backward(ctx.saved, float(grad))
            d = ctx.dtypes
            return (None, g_in.to(d[0]), g_rec.to(d[1]), torch.tensor(g_m, dtype=d[2], device=grad.device),
                    torch.tensor(g_s, dtype=d[3], device=grad.device), None)[:len(ctx.needs_input_grad)]

    return LIFLoss


_FN = None


def lif_loss(net, w_in, w_rec, tau_m, tau_s):
    """Differentiable loss of the LIF network (see module doc)."""
    global _FN
    if _FN is None:
        _FN = _make_function()
    return _FN.apply(net, w_in, w_rec, tau_m, tau_s, _torch().is_grad_enabled())
