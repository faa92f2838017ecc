"""Batched parameter sweeps: many independent networks in one persistent kernel.

A sweep (e.g. 1024 CUBA networks of uneven size, each with its own
connectivity and parameters) is advanced by launches in which every workgroup
owns one network and steps it through ``steps_per_launch`` time steps without
any grid-wide synchronisation: its state in registers, its spikes and the
events of its targets in LDS (resident.ResidentKernel).  A pathway's events
carry one constant per network, so counting them per target gives the sums of
the cython runtime's left fold over the spike queue
(brian2/synapses/spikequeue.h:151-191 with delay 0) bit for bit.  Networks are
launched by size, so that small ones share a compute unit; the launches of the
sizes run side by side.

Launches are replayed from a hipGraph.  The largest block size and the number
of steps per launch are chosen by a small autotuner that times the candidates
on the real networks (results do not depend on either).
"""
import ctypes
import time

import numpy as np

from . import _lib
from .codegen import HostEval, ParamStruct, Renderer, cast_value, ctype_of, filled, translate_block
from .kernels import _rename, identifiers
from .resident import (
    MAX_NEURONS,
    ResidentKernel,
    lds_plan,
    neurons_in_registers,
    refractory_form,
    releasable,
    timestep_bound,
)
from .runtime import Device, Model, dev, ptr, zeros

L = _lib.lib


class SweepNetwork:
    """One network of the sweep: size, exc/inh split, seed, constant overrides."""

    def __init__(self, N, NE, seed, namespace):
        self.N, self.NE, self.seed, self.namespace = int(N), int(NE), int(seed), dict(namespace)


class BatchedCUBA:
    """Sweep of independent networks of one neuron model with two constant-weight
    pathways (exc: sources [0, NE) -> `exc_var`, inh: [NE, N) -> `inh_var`)."""

    def __init__(self, nets, model="cuba", p=0.02, dt=1e-4, float_t="double", record_spikes=True,
                 spike_capacity_hz=200.0, horizon_steps=10000):
        if isinstance(model, str):
            model = Model.load(model)
        self.model = model
        self.nets = list(nets)
        self.p = float(p)
        self.dt = float(dt)
        self.float_t = float_t
        self.record = record_spikes
        self.su = model.group.get("stateupdate")
        self.th = model.group.get("threshold")
        self.rs = model.group.get("reset")
        ex, ih = model.pathways["exc"], model.pathways["inh"]
        self.exc_var, self.inh_var = ex.vector[-1]["var"], ih.vector[-1]["var"]
        self.exc_expr, self.inh_expr = ex.vector[-1]["expr"], ih.vector[-1]["expr"]
        self.exc_spec, self.inh_spec = ex, ih
        if len(ex.vector) != 1 or len(ih.vector) != 1 or ex.vector[0]["op"] != "+=" or ih.vector[0]["op"] != "+=":
            raise NotImplementedError("batched sweeps support on_pre = '<var> += <constant expression>'")
        # state variables of the group (as in NeuronGroup)
        from .runtime import NeuronGroup

        proto = NeuronGroup(1, model, float_t=float_t)
        self.vars = proto.vars
        self.uses_refractory = proto.uses_refractory
        self.t_step = 0
        self.spike_capacity_hz = spike_capacity_hz
        self.horizon_steps = horizon_steps
        self._built = False
        self.counts = None  # events per neuron, where they do not fit a workgroup's LDS
        self.block = 256
        self.steps_per_launch = 100

    # ------------------------------------------------------------------ build
    def _scalars(self):
        """Per-network values of every scalar the vector code needs (loop
        invariants of each code object evaluated on the host, and constants)."""
        names = []
        table = []
        for k, net in enumerate(self.nets):
            row = {}
            host = {"dt": self.dt, "N": net.N}
            host.update(net.namespace)
            for tag, spec in (("su", self.su), ("th", self.th), ("rs", self.rs), ("pe", self.exc_spec),
                              ("pi", self.inh_spec)):
                if spec is None:
                    continue
                vals = dict(host)
                for n, v in spec.variables.items():
                    if v["kind"] == "Constant" and n not in vals:
                        vals[n] = v["value"]
                ev = HostEval(vals)
                types = {}
                for st in spec.scalar:
                    ct = ctype_of(st["dtype"], self.float_t, st["var"])
                    ev.values[st["var"]] = cast_value(ev.eval(st["expr"]), ct)
                    types[st["var"]] = ct
                for n in sorted(identifiers(spec.vector)):
                    if n in types or (n in spec.variables and spec.variables[n]["kind"] == "Constant"):
                        ct = types.get(n)
                        v = ev.values[n]
                        if ct is None:
                            ct = "bool" if isinstance(v, bool) else ("long long" if isinstance(v, int) else "double")
                        row[(tag, n)] = (v, ct)
            if k == 0:
                names = sorted(row)
                self.scalar_types = {key: row[key][1] for key in names}
            table.append([float(row[key][0]) for key in names])
        self.scalar_names = names
        table = np.array(table, np.float64)
        # refractory periods in steps: compared through their bound (resident.timestep_bound)
        self.bounds = {}
        for k, (tg, n) in enumerate(names):
            steps = table[:, k]
            if self.scalar_types[(tg, n)] == "long long" and tg == "su" and np.all(releasable(steps)):
                self.bounds[f"{tg}_{n}"] = f"tb_{n}"
                of = {int(x): timestep_bound(int(x), self.dt) for x in np.unique(steps)}
                table = np.column_stack([table, [of[int(x)] for x in steps]])
        return table

    def _struct(self):
        ps = ParamStruct("hbb_params")
        ps.ptr("clock", "long long", const=True)
        ps.val("step_off", "long long")
        ps.val("dt", "double")
        ps.val("n_steps", "int")
        ps.val("first", "int")  # the launch's networks: order[first + workgroup]
        ps.ptr("order", "int", const=True)
        ps.ptr("n_off", "int", const=True)
        ps.ptr("ne", "int", const=True)
        ps.ptr("row_ptr", "unsigned int", const=True)
        ps.ptr("post", "int", const=True)
        ps.ptr("scal", "double", const=True)
        for v, ct in self.vars.items():
            ps.ptr(f"a_{v}", "unsigned char" if ct == "bool" else ct)
        ps.ptr("counts", "unsigned int")
        ps.ptr("spk_i", "int")
        ps.ptr("spk_step", "int")
        ps.ptr("spk_off", "long long", const=True)
        ps.ptr("spk_cap", "long long", const=True)
        ps.ptr("spk_n", "long long")
        ps.ptr("status", "int")
        return ps

    def _kernel(self, rows_in_lds, counts_in_lds):
        """The step kernel (resident.ResidentKernel): the networks' scalars are read per
        workgroup, the pathway of an event is that of its source (exc below NE)."""
        names = {}
        for (tg, n) in self.scalar_types:
            names.setdefault(tg, {})[n] = f"{tg}_{n}"

        def block(tag, spec, extra=None):
            types = dict(self.vars)
            types.update({"t": "double", "dt": "double", "N": "int", "i": "int", "_idx": "int"})
            types.update(extra or {})
            types.update({n: ct for (tg, n), ct in self.scalar_types.items() if tg == tag})
            return _rename(translate_block(spec.vector, spec.conditional_write, types, set(), self.float_t, select=True),
                           names.get(tag, {}))

        def operand(tag, spec, var):
            types = {n: ct for (tg, n), ct in self.scalar_types.items() if tg == tag}
            c, _ = Renderer(types).render(spec.vector[-1]["expr"])
            ct = self.vars[var]
            return f"const {ct} {tag}_val = ({ct})({_rename([c], names.get(tag, {}))[0]});"

        update, spike = [], []
        if self.su is not None:
            update += ["{"] + block("su", self.su) + ["}"]
        if self.th is not None:
            update += ["{"] + block("th", self.th, {"_cond": "bool"}) + ["hb_cond = _cond;", "}"]
        if self.rs is not None:
            if {st["var"] for st in self.rs.vector} & {self.exc_var, self.inh_var}:
                raise NotImplementedError("reset writes a synaptic target variable")
            spike = block("rs", self.rs)
        test = refractory_form(update, spike, self.vars)
        prologue = [
            "const int net = p.order[p.first + (int)blockIdx.x];",
            "const int hb_off = p.n_off[net];",
            "const int N = p.n_off[net + 1] - hb_off;",
            "const int NE = p.ne[net];",
            "const unsigned int* hb_rp = p.row_ptr + hb_off + net;  // N + 1 entries per network",
            "// the plan's clock counts launches of n_steps steps each",
            "const long long hb_step0 = (p.clock[0] + p.step_off) * p.n_steps;",
            "const long long hb_so = p.spk_off[net], hb_sc = p.spk_cap[net];",
            "long long hb_sn = p.spk_n[net];",
        ]
        row = len(self.scalar_names) + len(self.bounds)
        for idx, (tg, n) in enumerate(self.scalar_names):
            ct = self.scalar_types[(tg, n)]
            prologue.append(f"const {ct} {tg}_{n} = ({ct})p.scal[(size_t)net * {row} + {idx}];")
        for idx, b in enumerate(self.bounds.values()):
            prologue.append(f"const double {b} = p.scal[(size_t)net * {row} + {len(self.scalar_names) + idx}];")
        prologue += [operand("pe", self.exc_spec, self.exc_var), operand("pi", self.inh_spec, self.inh_var)]
        shared = [
            "// spikes as bits by neuron and the spikes before each word (steps of many spikes)",
            "unsigned long long* const s_bit = (unsigned long long*)(hb_lds + (((unsigned char*)(s_spk + N) - hb_lds + 7) & ~7));",
            "int* const s_pre = (int*)(s_bit + (N + 63) / 64);",
        ]
        store = ("if (hb_sn + {r} < hb_sc) {{ p.spk_i[hb_so + hb_sn + {r}] = {i}; "
                 "p.spk_step[hb_so + hb_sn + {r}] = (int)hb_step; }}")
        record = [
            "// the record keeps a step's spikes in ascending order",
            "if (hb_nsp <= 64) {",
            "    if (wid == NW - 1) {  // rank by counting the smaller ones",
            "        const int id_ = lane < hb_nsp ? (int)s_spk[lane] : 0;",
            "        int r_ = 0;",
            "        for (int j = 0; j < hb_nsp; j++) r_ += (int)s_spk[j] < id_ ? 1 : 0;",
            "        if (lane < hb_nsp) { " + store.format(r="r_", i="id_") + " }",
            "    }",
            "} else {  // rank by the set bits below",
            "    const int nw_ = (N + 63) / 64;",
            "    for (int w = threadIdx.x; w < nw_; w += T) s_bit[w] = 0ull;",
            "    __syncthreads();",
            "    for (int j = threadIdx.x; j < hb_nsp; j += T)",
            "        atomicOr((unsigned int*)s_bit + (s_spk[j] >> 5), 1u << (s_spk[j] & 31));",
            "    __syncthreads();",
            "    if (wid == 0) {",
            "        int c_ = 0;",
            "        for (int w0 = 0; w0 < nw_; w0 += 64) {",
            "            const int n_ = w0 + lane < nw_ ? __popcll(s_bit[w0 + lane]) : 0;",
            "            const int x_ = hb_wave_incl_scan(n_);",
            "            if (w0 + lane < nw_) s_pre[w0 + lane] = c_ + x_ - n_;",
            "            c_ += __builtin_amdgcn_readlane(x_, 63);",
            "        }",
            "    }",
            "    __syncthreads();",
            "    for (int j = threadIdx.x; j < hb_nsp; j += T) {",
            "        const int id_ = (int)s_spk[j];",
            "        const int r_ = s_pre[id_ >> 6] + __popcll(s_bit[id_ >> 6] & ((1ull << (id_ & 63)) - 1ull));",
            "        " + store.format(r="r_", i="id_"),
            "    }",
            "}",
            "hb_sn += hb_nsp;",
        ]
        finish = ["if (threadIdx.x == 0) { p.spk_n[net] = hb_sn; if (hb_sc && hb_sn > hb_sc) atomicOr(p.status, 2); }"]
        return ResidentKernel(
            "batched_step", self._struct(), self.vars, update,
            [(self.exc_var, "+=", "pe_val"), (self.inh_var, "+=", "pi_val")], prologue,
            ["const int hb_tgt = (int)hb_syn;", "const int hb_path = hb_src < NE ? 0 : 1;"], spike=spike,
            refractory=self.uses_refractory and self.th is not None, record=record, finish=finish, rows_in_lds=rows_in_lds, counts_in_lds=counts_in_lds, shared=shared,
            bound=self.bounds.get(test))

    def _classes(self):
        """The networks by workgroup size, largest first: [(threads, first, networks)].

        A thread holds up to `resident` neurons, so a network takes the fewest threads (a
        power of two from 128 to `block`) that hold it, and small networks share a compute
        unit.  The launches of the sizes run side by side, so there are at most four."""
        R = neurons_in_registers(self.vars)
        out = []
        for k, n in enumerate(sorted((n.N for n in self.nets), reverse=True)):
            t = 128
            while t < self.block and t * R < n:
                t *= 2
            t = min(t, self.block)
            if not out or out[-1][0] != t:
                out.append([t, k, 0, n])
            out[-1][2] += 1
        return out

    def build(self):
        import torch

        from .synth import S_CONN, cuba_v0

        self.device = D = Device.get()
        sizes = np.array([n.N for n in self.nets], np.int64)
        self.n_off = np.zeros(len(sizes) + 1, np.int64)
        np.cumsum(sizes, out=self.n_off[1:])
        Ntot = int(self.n_off[-1])
        self.state = {}
        host = {}
        for v, ct in self.vars.items():
            if v == "lastspike":
                host[v] = np.full(Ntot, -1e4)
            elif v == "not_refractory":
                host[v] = np.ones(Ntot, np.uint8)
            else:
                host[v] = np.zeros(Ntot)
        for k, net in enumerate(self.nets):
            host["v"][self.n_off[k]:self.n_off[k + 1]] = cuba_v0(net.seed, net.N)
        for v, ct in self.vars.items():
            self.state[v] = dev(host[v], ct)
        # connectivity: per network Bernoulli(p) over all pairs, CSR by source
        s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        row_ptr = zeros(Ntot + len(sizes), "int")
        counts = []
        for k, net in enumerate(self.nets):
            base = int(self.n_off[k]) + k
            view = row_ptr[base: base + net.N + 1]
            _lib.check(L.hb_gen_bernoulli_rows(net.seed, S_CONN, 0, net.N, net.N, self.p, ptr(view), None, s))
            _lib.check(L.hb_scan_u32(ptr(view), net.N, s))
            counts.append(view[net.N: net.N + 1])
        totals = torch.cat(counts).cpu().numpy().astype(np.int64)
        syn_off = np.zeros(len(sizes) + 1, np.int64)
        np.cumsum(totals, out=syn_off[1:])
        if syn_off[-1] >= 2**32:
            raise NotImplementedError("more than 2^32 synapses in one sweep")
        self.n_syn = int(syn_off[-1])
        self.post = zeros(self.n_syn, "int")
        for k, net in enumerate(self.nets):
            base = int(self.n_off[k]) + k
            view = row_ptr[base: base + net.N + 1]
            pv = self.post[int(syn_off[k]):]
            _lib.check(L.hb_gen_bernoulli_rows(net.seed, S_CONN, 0, net.N, net.N, self.p, ptr(view), ptr(pv), s))
            view += int(syn_off[k])  # absolute positions into the concatenated post array
        self.row_ptr = row_ptr
        self.scal = dev(self._scalars(), "double")
        self.order = dev(np.argsort(-sizes, kind="stable").astype(np.int32), "int")
        self.n_off_d = dev(self.n_off.astype(np.int32), "int")
        self.ne_d = dev(np.array([n.NE for n in self.nets], np.int32), "int")
        cap = np.maximum(1024, (sizes * self.spike_capacity_hz * self.horizon_steps * self.dt).astype(np.int64))
        if not self.record:
            cap = np.zeros_like(cap)
        off = np.zeros(len(sizes), np.int64)
        off[1:] = np.cumsum(cap)[:-1]
        self.spk_cap = dev(cap, "long long")
        self.spk_off = dev(off, "long long")
        self._spk_off_h = off
        self.spk_n = zeros(len(sizes), "long long")
        tot = max(int(cap.sum()), 1)
        self.spk_i = zeros(tot, "int")
        self.spk_step = zeros(tot, "int")
        self.status = zeros(1, "int")
        self._compile()
        self._built = True

    def _compile(self):
        """Generates and compiles the step kernel for the current block size and
        steps per launch, and records it in a one-launch plan."""
        import torch

        D = self.device
        if self.t_step % self.steps_per_launch:
            raise ValueError("the current step is not a multiple of steps_per_launch")
        self.launch_clock = torch.full((1,), self.t_step // self.steps_per_launch, dtype=torch.int64, device="cuda")
        v = dict(clock=self.launch_clock.data_ptr(), step_off=0, dt=self.dt, n_steps=self.steps_per_launch,
                 order=self.order.data_ptr(), n_off=self.n_off_d.data_ptr(),
                 ne=self.ne_d.data_ptr(), row_ptr=self.row_ptr.data_ptr(), post=self.post.data_ptr(),
                 scal=self.scal.data_ptr(), spk_i=self.spk_i.data_ptr(), spk_step=self.spk_step.data_ptr(),
                 spk_off=self.spk_off.data_ptr(), spk_cap=self.spk_cap.data_ptr(), spk_n=self.spk_n.data_ptr(),
                 status=self.status.data_ptr())
        for n in self.vars:
            v[f"a_{n}"] = self.state[n].data_ptr()
        self.plan = ctypes.c_void_p()
        _lib.check(L.hb_plan_create(D.ctx, ptr(self.launch_clock), ctypes.byref(self.plan)))
        # one launch per workgroup size, side by side
        for k, (threads, first, count, nmax) in enumerate(self._classes()):
            extra = 8 + 12 * ((nmax + 63) // 64)
            if nmax > MAX_NEURONS:
                raise NotImplementedError(f"networks of more than {MAX_NEURONS} neurons")
            K = self._kernel(*lds_plan(nmax, 1, extra))
            fn = D.function(K.source, K.kernel_name)
            if not K.counts_in_lds and self.counts is None:
                self.counts = zeros(int(self.n_off[-1]), "int")
            cls = K.struct.ctypes_struct()
            v.update(first=first, counts=0 if self.counts is None else self.counts.data_ptr())
            a = filled(cls, v)
            buf = bytes(a)
            _lib.check(L.hb_plan_add(self.plan, fn, count, threads, K.lds_bytes(nmax, threads, extra), buf, len(buf),
                                     cls.step_off.offset))
            if k:
                _lib.check(L.hb_plan_set_lane(self.plan, k, 1 + (k - 1) % 3))

    # ------------------------------------------------------------------ run
    def run(self, n_steps, graph_launches=10):
        """Advances every network by n_steps (a multiple of steps_per_launch)."""
        if not self._built:
            self.build()
        S = self.steps_per_launch
        if n_steps % S:
            raise ValueError(f"n_steps must be a multiple of steps_per_launch={S}")
        self._run_launches(n_steps // S, graph_launches)
        self.t_step += n_steps
        st = int(self.status.item())
        if st:
            raise _lib.HipBrianError("spike record buffer overflow in the batched sweep" if st & 2 else f"status {st}")

    def _run_launches(self, launches, graph_launches):
        g = max(1, min(graph_launches, launches))
        _lib.check(L.hb_plan_run(self.plan, self.device.stream, launches, g if launches >= g else 1))

    def spikes(self, k):
        n = int(self.spk_n[k].item())
        o = int(self._spk_off_h[k])
        i = self.spk_i[o:o + n].cpu().numpy()
        s = self.spk_step[o:o + n].cpu().numpy().astype(np.int64)
        return i, s

    def get(self, var, k):
        a, b = int(self.n_off[k]), int(self.n_off[k + 1])
        return self.state[var][a:b].cpu().numpy()

    # ------------------------------------------------------------------ autotuner
    def snapshot(self):
        return ({v: t.clone() for v, t in self.state.items()}, self.spk_n.clone(), self.t_step)

    def restore(self, snap):
        st, n, t = snap
        for v, tt in st.items():
            self.state[v].copy_(tt)
        self.spk_n.copy_(n)
        self.t_step = t
        self.launch_clock.fill_(t // self.steps_per_launch)

    def autotune(self, blocks=(128, 256, 512, 1024), steps=(10, 50, 100), trial_steps=200):
        """Times each (block size, steps per launch) on the real networks from the
        current state, restores the state, and keeps the fastest."""
        import torch

        if not self._built:
            self.build()
        snap = self.snapshot()
        results = {}
        for T in blocks:
            for S in steps:
                if trial_steps % S:
                    continue
                self.block, self.steps_per_launch = T, S
                self.t_step = snap[2]
                self._compile()
                self.restore(snap)
                self._run_launches(trial_steps // S, max(1, (trial_steps // S)))  # warm (compile + capture)
                torch.cuda.synchronize()
                self.restore(snap)
                t0 = time.perf_counter()
                self._run_launches(trial_steps // S, max(1, (trial_steps // S)))
                torch.cuda.synchronize()
                results[(T, S)] = time.perf_counter() - t0
        best = min(results, key=results.get)
        self.block, self.steps_per_launch = best
        self.t_step = snap[2]
        self._compile()
        self.restore(snap)
        self.autotune_results = results
        return best, results
