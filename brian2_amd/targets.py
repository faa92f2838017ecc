"""Targets of a spike generator through plastic synapses, each stepped by a wave of its own.

A group whose only input is a SpikeGeneratorGroup through one pathway with on_post code
(brian2/synapses/synapses.py:205-216), and which drives nothing, is a set of neurons that
know nothing of each other: a neuron, its synapses and the generator's list are all that a
step needs.  So a wave takes one target through all the steps of a launch, with the
synapses' variables in LDS.
"""
from .chip import monitor_fields
from .codegen import ParamStruct, source_header, translate_block
from .kernels import LDS_BYTES, _rename, group_block, onpre_lines

SIZES = {"double": 8, "float": 4, "long long": 8, "int": 4}


class TargetSteps:
    """Source of the kernel (one workgroup of a wave per target).

    The wave's lanes hold the next 64 entries of the generator's list, the following 64 being
    on their way.  A step: the neuron's update (all lanes alike), the entries of this step, a
    lane each, with the on_pre statements on that source's synapse (hb_map: its place in LDS),
    their values added up in the entries' order, the on_post statements on all synapses if
    the neuron spikes, its reset.  No lane waits for memory but at the start, the end and for
    a spike's record.

    What bounds it: the chain of a step, two exponentials where a source spikes.  20 targets
    of 1000 sources at 15 Hz: 19.0 us per step as four launches (generator, update, gather,
    on_post), 1.0 now."""

    def __init__(self, group, scalars, syn_arrays, plastic, on_pre, target_index, pre_scalars, on_post, post_scalars,
                 target_var, op, val_t):
        g = self.group = group
        self.scalars, self.pre_scalars, self.post_scalars = scalars, pre_scalars, post_scalars
        self.syn_arrays = syn_arrays
        ps = ParamStruct(f"hbt_{g.name}")
        ps.val("step0", "long long")
        ps.val("dt", "double")
        ps.val("n_steps", "int")
        ps.val("N", "int")
        for v, ct in g.vars.items():
            ps.ptr(f"a_{v}", "unsigned char" if ct == "bool" else ct)
        for (tg, n), (_, ct) in sorted(scalars.items()):
            ps.val(f"{tg}_{n}", ct)
        for x, sc in (("c", pre_scalars), ("q", post_scalars)):
            for n, (_, ct) in sorted(sc.items()):
                ps.val(f"{x}_{n}", ct)
        for v, ct in syn_arrays.items():
            ps.ptr(f"s_{v}", ct)
        ps.ptr("post_ptr", "unsigned int", const=True)
        ps.ptr("post_syn", "unsigned int", const=True)
        ps.ptr("post_pre", "int", const=True)
        ps.ptr("gen_tb", "int", const=True)
        ps.ptr("gen_idx", "int", const=True)
        ps.val("gen_at", "long long")
        ps.val("gen_n", "long long")
        ps.val("src0", "int")
        ps.val("n_src", "int")
        ps.val("deg", "int")
        ps.val("pad", "int")
        ps.ptr("events", "unsigned long long")
        ps.ptr("status", "int")
        monitor_fields(ps, g)  # (a spike monitor's, if any)
        self.struct = ps
        self.kernel_name = f"targets_{g.name}"

        def block(tag, spec, extra=()):
            return group_block(tag, spec, g.vars, scalars, g.float_t, extra)

        types = dict(syn_arrays)
        types.update({"_idx": "int", "t": "double"})
        types.update({n: ct for n, (_, ct) in post_scalars.items()})
        post = _rename(translate_block(on_post, {}, types, set(), g.float_t), {n: f"p.q_{n}" for n in post_scalars})
        pre = onpre_lines(on_pre, target_index, syn_arrays, pre_scalars, g.float_t, f"hb_gv = ({val_t})", val_t)
        load = [f"{ct} {v} = s_{v}[hb_k];" for v, ct in syn_arrays.items()]
        save = [f"s_{v}[hb_k] = {v};" for v in syn_arrays if v in plastic]

        k = [source_header(64), ps.c_decl()]
        k.append(f'extern "C" __global__ void __launch_bounds__(64) {self.kernel_name}(const {ps.name} p) {{')
        k += [
            "    const int hb_lane = threadIdx.x, i = blockIdx.x, N = p.N, _idx = i;",
            "    const double dt = p.dt;",
            "    (void)dt; (void)N; (void)_idx;",
            "    extern __shared__ __align__(16) unsigned char hb_lds[];",
        ]
        at = "hb_lds"
        for v, ct in sorted(syn_arrays.items(), key=lambda x: -SIZES[x[1]]):
            k.append(f"    {ct}* const s_{v} = ({ct}*)({at});")
            at = f"s_{v} + p.deg"
        k += [
            f"    unsigned short* const hb_map = (unsigned short*)({at});  // a source's synapse, or 0xffff",
            "    const unsigned int hb_first = p.post_ptr[i];",
            "    const int hb_deg = (int)(p.post_ptr[i + 1] - hb_first);",
            "    for (int x = hb_lane; x < p.n_src; x += 64) hb_map[x] = 0xffff;",
            "    __syncthreads();",
            "    for (int hb_k = hb_lane; hb_k < hb_deg; hb_k += 64) {",
            "        const unsigned int e = p.post_syn[hb_first + hb_k];",
        ] + [f"        s_{v}[hb_k] = p.s_{v}[e];" for v in syn_arrays] + [
            "        hb_map[p.post_pre[hb_first + hb_k] - p.src0] = (unsigned short)hb_k;",
            "    }",
            "    __syncthreads();",
        ]
        for v, ct in g.vars.items():
            k.append(f"    {ct} {v} = p.a_{v}[i]{' != 0' if ct == 'bool' else ''};")
        k += [
            "    auto hb_entries = [&](const long long x0, int& hb_tb, int& hb_id) {",
            "        const long long x = x0 + hb_lane < p.gen_n ? x0 + hb_lane : p.gen_n - 1;",
            "        hb_tb = x >= 0 ? p.gen_tb[x] : 0; hb_id = x >= 0 ? p.gen_idx[x] : 0;",
            "        if (x0 + hb_lane >= p.gen_n) hb_tb = 0x7fffffff;",
            "    };",
            f"    auto hb_from = [](const {val_t} x, const int l) {{  // lane l's value",
        ] + (["        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));"]
             if val_t == "float" else [
            "        const long long b = __builtin_bit_cast(long long, x);",
            "        const unsigned int lo = (unsigned int)__builtin_amdgcn_readlane((int)b, l);",
            "        const unsigned int hi = (unsigned int)__builtin_amdgcn_readlane((int)(b >> 32), l);",
            "        return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);"]) + [
            "    };",
            "    long long hb_at = p.gen_at;",
            "    int hb_tb, hb_id, hb_tb2, hb_id2;",
            "    hb_entries(hb_at, hb_tb, hb_id);",
            "    hb_entries(hb_at + 64, hb_tb2, hb_id2);",
            "    unsigned long long hb_ev = 0ull;",
            "    for (int hb_s = 0; hb_s < p.n_steps; hb_s++) {",
            "        const long long hb_step = p.step0 + hb_s;",
            "        const double t = (double)hb_step * dt;",
            "        (void)t;",
            "        bool hb_cond = false;",
        ]
        if g.su is not None:
            k += ["        {"] + ["            " + x for x in block("su", g.su)] + ["        }"]
        if g.th is not None:
            k += ["        {"] + ["            " + x for x in block("th", g.th, {"_cond": "bool"})]
            k += ["            hb_cond = _cond;", "        }"]
            if g.uses_refractory:
                k.append("        if (hb_cond) { not_refractory = false; lastspike = t; }")
        k += [
            "        const bool hb_spiked = __builtin_amdgcn_ballot_w64(hb_cond) != 0ull;",
            "        for (;;) {  // this step's entries",
            "            const bool hb_on = hb_tb == (int)hb_step;",
            "            if (__builtin_amdgcn_ballot_w64(hb_on) != 0ull) {",
            "                const int hb_k = hb_on && hb_id >= p.src0 && hb_id < p.src0 + p.n_src ? (int)hb_map[hb_id - p.src0] : 0xffff;",
            f"                {val_t} hb_gv = 0;",
            "                if (hb_k != 0xffff) {",
            "                    const int _idx = hb_k;",
            "                    (void)_idx;",
        ]
        k += ["                    " + x for x in load + pre + save]
        k += [
            "                }",
            "                unsigned long long hb_m = __builtin_amdgcn_ballot_w64(hb_k != 0xffff);",
            "                hb_ev += (unsigned long long)__popcll(hb_m);",
            f"                for (; hb_m; hb_m &= hb_m - 1ull) {{ const {val_t} hb_v = hb_from(hb_gv, __builtin_ctzll(hb_m)); "
            f"{target_var} {op} hb_v; }}",
            "                __syncthreads();",
            "            }",
            "            if (__builtin_amdgcn_readlane(hb_tb, 63) > (int)hb_step) break;",
            "            hb_tb = hb_tb2; hb_id = hb_id2; hb_at += 64;",
            "            hb_entries(hb_at + 64, hb_tb2, hb_id2);",
            "        }",
            "        if (hb_spiked) {",
        ]
        if g.smon:
            k += [
                "            if (hb_lane == 0 && i >= p.mon_start && i < p.mon_stop) {",
                "                const unsigned long long o = atomicAdd(p.mon_n, 1ull);",
                "                if (o < (unsigned long long)p.mon_cap) { p.mon_i[o] = i; p.mon_step[o] = (int)hb_step; }",
                "                else atomicOr(p.status, 2);",
                "                p.mon_count[i - p.mon_start] += 1;",
                "            }",
            ]
        k += ["            for (int hb_k = hb_lane; hb_k < hb_deg; hb_k += 64) {", "                const int _idx = hb_k;", "                (void)_idx;"]
        k += ["                " + x for x in load + post + save]
        k += ["            }", "            __syncthreads();"]
        if g.rs is not None:
            k += ["            {"] + ["                " + x for x in block("rs", g.rs)] + ["            }"]
        k += ["        }", "    }", "    for (int hb_k = hb_lane; hb_k < hb_deg; hb_k += 64) {",
              "        const unsigned int e = p.post_syn[hb_first + hb_k];"]
        k += [f"        p.s_{v}[e] = s_{v}[hb_k];" for v in syn_arrays if v in plastic] + ["    }", "    if (hb_lane == 0) {"]
        for v, ct in g.vars.items():
            k.append(f"        p.a_{v}[i] = {v}{' ? 1 : 0' if ct == 'bool' else ''};")
        k += ["        p.events[i] += hb_ev;", "    }", "}"]
        self.source = "\n".join(k) + "\n"

    @staticmethod
    def lds_bytes(syn_arrays, deg, n_src):
        return (sum(SIZES[ct] for ct in syn_arrays.values()) * deg + 2 * n_src + 15) // 16 * 16

    @classmethod
    def takes(cls, net, source, g, s):
        """Whether pathway s from the spike generator onto group g, the network's only groups,
        is stepped this way: no delays, default launch shapes, no pair with two synapses, a
        target's synapses within a compute unit's LDS.

        Measured on MI355X, us per step, sources x targets (15 Hz), this against the staged
        launches: 200 x 5 0.57 / 13.6, 1000 x 20 1.0 / 19.1, 4000 x 100 1.6 / 38.1,
        1000 x 1000 1.1 / 32.3, 4000 x 600 4.3 / 69.9, 1000 x 12000 17.8 / 234.5; runs of a
        single step, 1000 x 20, 78.9 / 120.7: no size at which the launches win."""
        import torch

        if any(x is not None for x in (net.tile, net.npt, net.gather_pairs, net.bucket_cap)):
            return False
        if s.source is not source or s.target is not g or s.post_spec is None or s.count_events or s.carry is not None:
            return False
        if s.csr["dmin"] != 0 or s.csr["n_seg"] != 1 or s.post_delay_steps != 0 or int(s.csr["n_syn"]) == 0:
            return False
        if source.period_bins or len(source.timebins) == 0 or g.vars[s.target_var] not in ("double", "float"):
            return False
        tb, idx = source.timebins, source.indices
        if bool(((tb[1:] == tb[:-1]) & (idx[1:] == idx[:-1])).any()):
            return False
        ptr = s.csr["post_ptr"].long()
        deg = int((ptr[1:] - ptr[:-1]).max())
        n_src = s.src_range[1] - s.src_range[0]
        if deg >= 65535 or cls.lds_bytes(s.syn_ctypes(), deg, n_src) > LDS_BYTES - 64:
            return False
        tgt = torch.repeat_interleave(torch.arange(g.N, device="cuda"), ptr[1:] - ptr[:-1])
        pair = tgt * n_src + s.csr["post_pre"].long()[:len(tgt)] - s.src_range[0]
        return len(torch.unique(pair)) == len(tgt)
