# CedarHIP.jl — CedarSim's Newton-transient path on an MI355X through
# libcedarhip.so (include/cedarhip.h).
#
# What this module adds to CedarSim, leaving its netlist import, DAE
# interface and analysis entry points unchanged:
#   * lower(circuit): a walker over the circuit function make_spectre_circuit
#     returns (src/spectre.jl:1656-1697), in the style of AliasInterp
#     (src/aliasextract.jl:10-39): it runs the function under a CassetteOverlay
#     pass that records every Named device call into the flat arrays of
#     cs_netlist instead of tracing it into DAECompiler;
#   * hip_daefunction: the DAE contract f!(out,du,u,p,t) / jac!(J,du,u,p,γ,t)
#     (benchmarks/benchmark_common.jl:138,155) with jac_prototype, for any
#     SciML DAE solver;
#   * tran!(circ, tspan, HIPBackend()) and dc!(circ, HIPBackend()): the
#     whole step loop (src/sweeps.jl:437-465) on the GPU;
#   * tran_batch: the tran!. broadcast over a CircuitSweep in one launch;
#   * supply_energy with a ChainRulesCore.rrule whose pullback is the
#     library's checkpointed adjoint (the role of ODEForwardSensitivityProblem
#     in test/sensitivity.jl:29-41).
# Julia is not installed where this package was written; the module follows
# the header field by field and the SciMLBase / CassetteOverlay interfaces
# CedarSim itself uses.
module CedarHIP

using CedarSim
using CedarSim: Named, Net, AbstractNet, DScope, debug_scope, Gnd, SimpleResistor, SimpleCapacitor,
                SimpleInductor, VoltageSource, CurrentSource, vcvs, vccs, ParallelInstances
using CassetteOverlay
using ChainRulesCore
using SciMLBase
using SparseArrays

const lib = joinpath(@__DIR__, "..", "lib", "libcedarhip.so")

# ---- structs: field order and types exactly as include/cedarhip.h (ABI 2) --------------
struct CsNetlist
    n_nodes::Int32
    n_res::Int32;  res_nodes::Ptr{Int32};  res_r::Ptr{Float64}
    n_cap::Int32;  cap_nodes::Ptr{Int32};  cap_c::Ptr{Float64}
    n_ind::Int32;  ind_nodes::Ptr{Int32};  ind_l::Ptr{Float64}
    n_vsrc::Int32; vsrc_nodes::Ptr{Int32}; vsrc_wave::Ptr{Int32}
    n_isrc::Int32; isrc_nodes::Ptr{Int32}; isrc_wave::Ptr{Int32}
    n_vccs::Int32; vccs_nodes::Ptr{Int32}; vccs_gain::Ptr{Float64}
    n_vcvs::Int32; vcvs_nodes::Ptr{Int32}; vcvs_gain::Ptr{Float64}
    n_mos::Int32;  mos_nodes::Ptr{Int32};  mos_type::Ptr{Int32}
    mos_vth::Ptr{Float64}; mos_kp::Ptr{Float64}; mos_w::Ptr{Float64}; mos_l::Ptr{Float64}
    n_wave::Int32; wave_kind::Ptr{Int32}; wave_off::Ptr{Int32}; wave_len::Ptr{Int32}
    wave_dc::Ptr{Float64}
    n_wave_data::Int32; wave_data::Ptr{Float64}
    gmin::Float64
    dev_m::Ptr{Float64}
    n_va::Int32; va_model::Ptr{Int32}; va_node_ptr::Ptr{Int32}; va_nodes::Ptr{Int32}
    va_prm_ptr::Ptr{Int32}; n_va_prm::Int32; va_prm::Ptr{Float64}
end

mutable struct CsTranOpts
    t_start::Float64; t_stop::Float64; reltol::Float64; abstol::Float64
    dt_init::Float64; dt_min::Float64; dt_max::Float64; newton_tol::Float64
    dt_out::Float64; dc_abstol::Float64
    n_out::Int32; max_order::Int32; newton_maxit::Int32; init::Int32
    max_steps::Int64; batch_kernel::Int32; record_steps::Int32; jac_reuse::Int32; reserved::Int32
end
function CsTranOpts()
    o = CsTranOpts(zeros(10)..., zeros(Int32, 4)..., Int64(0), Int32(0), Int32(0), Int32(0), Int32(0))
    ccall((:cs_tran_opts_default, lib), Cvoid, (Ref{CsTranOpts},), o)
    o
end

mutable struct CsTranStats
    steps::Int64; rejected::Int64; newton_iters::Int64; t_end::Float64
    retcode::Int32; pad::Int32; busy_s::Float64
end
CsTranStats() = CsTranStats(0, 0, 0, 0.0, 0, 0, 0.0)
# the same record, immutable, so that a Vector of it has the C layout (arrays of
# per-instance statistics)
struct CsTranStatsRec
    steps::Int64; rejected::Int64; newton_iters::Int64; t_end::Float64
    retcode::Int32; pad::Int32; busy_s::Float64
end
CsTranStats(r::CsTranStatsRec) = CsTranStats(r.steps, r.rejected, r.newton_iters, r.t_end, r.retcode, r.pad, r.busy_s)

struct CsAdjointOpts
    vsrc::Int32; ckpt_every::Int32; max_steps::Int64
end

const CS_WAVE_DC, CS_WAVE_PULSE, CS_WAVE_PWL, CS_WAVE_SIN = 0, 1, 2, 3
const CS_INIT_DCOP, CS_INIT_UIC = 0, 1
const CS_BATCH_KERNEL_AUTO, CS_BATCH_KERNEL_LDS, CS_BATCH_KERNEL_GLOBAL = 0, 1, 2

# ---- errors: CedarException style (src/util.jl:3-21), retcodes as SciMLBase's ---------
struct CedarHIPException <: CedarSim.CedarException
    code::Int32
    msg::String
end
Base.showerror(io::IO, e::CedarHIPException) = print(io, "CedarHIP error ", e.code, ": ", e.msg)

check(ctx, rc) = rc == 0 ? nothing :
    throw(CedarHIPException(rc, unsafe_string(ccall((:cs_last_error, lib), Cstring, (Ptr{Cvoid},), ctx))))

retcode(rc) = rc == 0 ? SciMLBase.ReturnCode.Success :
              rc == -5 ? SciMLBase.ReturnCode.InitialFailure :
              rc == -6 ? SciMLBase.ReturnCode.DtLessThanMin :
              rc == -9 ? SciMLBase.ReturnCode.MaxIters : SciMLBase.ReturnCode.Failure

mutable struct Context
    ptr::Ptr{Cvoid}
end
const ABI = 3
function Context(device::Integer=0)
    abi = ccall((:cs_abi_version, lib), Int32, ())
    abi == ABI || throw(CedarHIPException(-1, "libcedarhip ABI $abi, this binding is ABI $ABI"))
    r = Ref{Ptr{Cvoid}}(C_NULL)
    rc = ccall((:cs_create, lib), Int32, (Int32, Ref{Ptr{Cvoid}}), device, r)
    rc == 0 || throw(CedarHIPException(rc, "cs_create failed (no HIP device?)"))
    ctx = Context(r[])
    finalizer(c -> ccall((:cs_destroy, lib), Int32, (Ptr{Cvoid},), c.ptr), ctx)
    ctx
end
Base.unsafe_convert(::Type{Ptr{Cvoid}}, c::Context) = c.ptr

# ---- the walker: a circuit function -> cs_netlist arrays -------------------------------
# Nets become integers (ground -1); each device call is recorded with the
# multiplier its nets carry (ParallelInstances, src/simulate_ir.jl:56-75).
struct LowerNet <: AbstractNet
    id::Int
    multiplier::Float64
end

Base.@kwdef mutable struct Flat
    n_nets::Int = 0
    ground::Set{Int} = Set{Int}()
    names::Dict{Int, String} = Dict{Int, String}()
    res::Vector{Tuple{Int, Int, Float64, Float64}} = []           # a, b, r, m
    cap::Vector{Tuple{Int, Int, Float64, Float64}} = []
    ind::Vector{Tuple{Int, Int, Float64, Float64, String}} = []   # ..., branch name
    vsrc::Vector{Tuple{Int, Int, Any, Float64, String}} = []      # a, b, source, m, name
    isrc::Vector{Tuple{Int, Int, Any, Float64}} = []
    vccs::Vector{Tuple{NTuple{4, Int}, Float64, Float64}} = []
    vcvs::Vector{Tuple{NTuple{4, Int}, Float64, Float64, String}} = []
    va::Vector{Tuple{Int, Vector{Int}, Vector{Float64}}} = []     # model index, terminals, flat params
    devices::Dict{String, Tuple{Symbol, Int}} = Dict{String, Tuple{Symbol, Int}}()   # name -> (kind, 1-based index)
end

struct LowerInterp <: CassetteOverlay.AbstractBindingOverlay{nothing, nothing}
    flat::Flat
end

function (self::LowerInterp)(::Type{Net}, name::Union{DScope, Nothing}=nothing, multiplier::Float64=1.0)
    self.flat.n_nets += 1
    id = self.flat.n_nets
    name === nothing || (self.flat.names[id] = string(name))
    LowerNet(id, multiplier)
end
(self::LowerInterp)(::Type{Net}, net::LowerNet, multiplier::Float64) =
    LowerNet(net.id, net.multiplier * multiplier)

(self::LowerInterp)(::Gnd, n::LowerNet; kwargs...) = (push!(self.flat.ground, n.id); nothing)

mult(nets...) = nets[1].multiplier
scoped(name) = string(DScope(debug_scope[], name))

function (self::LowerInterp)(n::Named, args...)
    e, f = n.element, self.flat
    named(kind, list) = (f.devices[scoped(n.name)] = (kind, length(list)))
    if e isa SimpleResistor
        push!(f.res, (args[1].id, args[2].id, CedarSim.undefault(e.r), mult(args...))); named(:res, f.res)
    elseif e isa SimpleCapacitor
        push!(f.cap, (args[1].id, args[2].id, CedarSim.undefault(e.capacitance), mult(args...))); named(:cap, f.cap)
    elseif e isa SimpleInductor
        push!(f.ind, (args[1].id, args[2].id, CedarSim.undefault(e.inductance), mult(args...), scoped(n.name)))
        named(:ind, f.ind)
    elseif e isa VoltageSource
        push!(f.vsrc, (args[1].id, args[2].id, e, mult(args...), scoped(n.name))); named(:vsrc, f.vsrc)
    elseif e isa CurrentSource
        push!(f.isrc, (args[1].id, args[2].id, e, mult(args...))); named(:isrc, f.isrc)
    elseif e isa typeof(vccs) || e isa CedarSim.vccs
        push!(f.vccs, (Tuple(a.id for a in args[1:4]), CedarSim.undefault(e.gain), mult(args...))); named(:vccs, f.vccs)
    elseif e isa CedarSim.vcvs
        push!(f.vcvs, (Tuple(a.id for a in args[1:4]), CedarSim.undefault(e.gain), mult(args...), scoped(n.name)))
        named(:vcvs, f.vcvs)
    elseif e isa CedarSim.VAModel
        push!(f.va, va_record(e, args))
    else
        # a subcircuit: walk into it under its own debug scope
        CedarSim.with(debug_scope => DScope(debug_scope[], n.name)) do
            self(e, args...)
        end
    end
    nothing
end

# A Verilog-A device: the compiled model of the same module name; its fields
# are DefaultOr parameters (src/vasim.jl:702-733), a default one is NaN.
function va_record(e, args)
    name = lowercase(string(nameof(typeof(e))))
    idx = findfirst(==(name), first.(va_models()))
    idx === nothing && throw(CedarHIPException(-1, "Verilog-A module $name is not compiled into libcedarhip"))
    pnames = va_models()[idx][3]
    prm = [let v = getfield(e, Symbol(p)); CedarSim.isdefault(v) ? NaN : Float64(CedarSim.undefault(v)) end
           for p in pnames]
    (idx - 1, [a.id for a in args], prm)
end

function va_models()
    out = Tuple{String, Int, Vector{String}}[]
    for i in 0:ccall((:cs_va_model_count, lib), Int32, ()) - 1
        buf = Vector{UInt8}(undef, 128); npt = Ref{Int32}(); npr = Ref{Int32}(); hc = Ref{Int32}()
        ccall((:cs_va_model_info, lib), Int32, (Int32, Ptr{UInt8}, Int32, Ref{Int32}, Ref{Int32}, Ref{Int32}),
              i, buf, 128, npt, npr, hc)
        names = String[]
        for k in 0:npr[] - 1
            b2 = Vector{UInt8}(undef, 128)
            ccall((:cs_va_model_param, lib), Int32, (Int32, Int32, Ptr{UInt8}, Int32), i, k, b2, 128)
            push!(names, unsafe_string(pointer(b2)))
        end
        push!(out, (unsafe_string(pointer(buf)), Int(npt[]), names))
    end
    out
end

"""
    lower(circuit) -> (arrays, unknown names)

Run the circuit function under the walker and return the flat netlist
arrays in the layout of `cs_netlist` plus the name of every unknown (nets,
then the branch currents of voltage sources, inductors and VCVS).
"""
function lower(circuit)
    interp = LowerInterp(Flat())
    interp(circuit)
    flat(interp.flat)
end

# waveform of a source: (kind, data, dc value or NaN)
function wave(src)
    t = src.tran
    dc = src.dc === nothing ? NaN : Float64(CedarSim.undefault(src.dc))
    t isa Number && return (CS_WAVE_DC, [Float64(t)], dc)
    t isa CedarSim.SpectreEnvironment.Pulse && return (CS_WAVE_PULSE, collect(Float64, t.params), dc)
    t isa CedarSim.SpectreEnvironment.PWL && return (CS_WAVE_PWL, collect(Float64, t.wave), dc)
    t isa CedarSim.SpectreEnvironment.Sin && return (CS_WAVE_SIN, collect(Float64, t.params), dc)
    (CS_WAVE_DC, [dc], dc)
end

function flat(f::Flat)
    node = Dict{Int, Int32}()
    names = String[]
    for id in 1:f.n_nets
        if id in f.ground
            node[id] = -1
        else
            node[id] = length(names)
            push!(names, get(f.names, id, "net$id"))
        end
    end
    N(i) = node[i]
    wk, wo, wl, wd, wdata = Int32[], Int32[], Int32[], Float64[], Float64[]
    function addwave(src)
        k, d, dc = wave(src)
        push!(wk, k); push!(wo, length(wdata)); push!(wl, length(d)); push!(wd, dc); append!(wdata, d)
        Int32(length(wk) - 1)
    end
    a = Dict{Symbol, Any}()
    a[:res_nodes] = Int32[x for r in f.res for x in (N(r[1]), N(r[2]))]; a[:res_r] = [r[3] for r in f.res]
    a[:cap_nodes] = Int32[x for r in f.cap for x in (N(r[1]), N(r[2]))]; a[:cap_c] = [r[3] for r in f.cap]
    a[:ind_nodes] = Int32[x for r in f.ind for x in (N(r[1]), N(r[2]))]; a[:ind_l] = [r[3] for r in f.ind]
    a[:vsrc_nodes] = Int32[x for r in f.vsrc for x in (N(r[1]), N(r[2]))]; a[:vsrc_wave] = Int32[addwave(r[3]) for r in f.vsrc]
    a[:isrc_nodes] = Int32[x for r in f.isrc for x in (N(r[1]), N(r[2]))]; a[:isrc_wave] = Int32[addwave(r[3]) for r in f.isrc]
    # AC magnitudes |ac| of the sources, V then I (src/simpledevices.jl:291,332)
    a[:src_ac] = Float64[[abs(r[3].ac) for r in f.vsrc]; [abs(r[3].ac) for r in f.isrc]]
    a[:vccs_nodes] = Int32[N(x) for r in f.vccs for x in r[1]]; a[:vccs_gain] = [r[2] for r in f.vccs]
    a[:vcvs_nodes] = Int32[N(x) for r in f.vcvs for x in r[1]]; a[:vcvs_gain] = [r[2] for r in f.vcvs]
    a[:wave_kind], a[:wave_off], a[:wave_len], a[:wave_dc], a[:wave_data] = wk, wo, wl, wd, wdata
    m = [r[4] for r in f.res]; append!(m, [r[4] for r in f.cap]); append!(m, [r[4] for r in f.ind])
    append!(m, [r[4] for r in f.vsrc]); append!(m, [r[4] for r in f.isrc]); append!(m, [r[3] for r in f.vccs])
    append!(m, [r[3] for r in f.vcvs])
    a[:dev_m] = all(==(1.0), m) ? nothing : m
    a[:va_model] = Int32[v[1] for v in f.va]
    a[:va_node_ptr] = Int32[0; cumsum([length(v[2]) for v in f.va])]
    a[:va_nodes] = Int32[N(x) for v in f.va for x in v[2]]
    a[:va_prm_ptr] = Int32[0; cumsum([length(v[3]) for v in f.va])]
    a[:va_prm] = Float64[x for v in f.va for x in v[3]]
    a[:n_nodes] = length(names)
    a[:devices] = f.devices
    unknowns = vcat(names, [r[5] * ".I" for r in f.vsrc], [r[5] * ".I" for r in f.ind], [r[4] * ".I" for r in f.vcvs])
    a, unknowns
end

P(v) = isempty(v) ? Ptr{Float64}(C_NULL) : pointer(v)
PI(v) = isempty(v) ? Ptr{Int32}(C_NULL) : pointer(v)

# the cs_netlist of lowered arrays; keep `a` alive (GC.@preserve) while it is used
function netlist(a; gmin=1e-12)
    e64, e32 = Float64[], Int32[]
    CsNetlist(a[:n_nodes],
        length(a[:res_r]), PI(a[:res_nodes]), P(a[:res_r]),
        length(a[:cap_c]), PI(a[:cap_nodes]), P(a[:cap_c]),
        length(a[:ind_l]), PI(a[:ind_nodes]), P(a[:ind_l]),
        length(a[:vsrc_wave]), PI(a[:vsrc_nodes]), PI(a[:vsrc_wave]),
        length(a[:isrc_wave]), PI(a[:isrc_nodes]), PI(a[:isrc_wave]),
        length(a[:vccs_gain]), PI(a[:vccs_nodes]), P(a[:vccs_gain]),
        length(a[:vcvs_gain]), PI(a[:vcvs_nodes]), P(a[:vcvs_gain]),
        0, PI(e32), PI(e32), P(e64), P(e64), P(e64), P(e64),
        length(a[:wave_kind]), PI(a[:wave_kind]), PI(a[:wave_off]), PI(a[:wave_len]), P(a[:wave_dc]),
        length(a[:wave_data]), P(a[:wave_data]),
        gmin,
        a[:dev_m] === nothing ? Ptr{Float64}(C_NULL) : pointer(a[:dev_m]),
        length(a[:va_model]), PI(a[:va_model]), PI(a[:va_node_ptr]), PI(a[:va_nodes]),
        PI(a[:va_prm_ptr]), length(a[:va_prm]), P(a[:va_prm]))
end

# ---- a compiled circuit --------------------------------------------------------------
struct HIPSystem
    ctx::Context
    cid::Int32
    n::Int
    nnz::Int
    n_params::Int
    unknowns::Vector{String}
    src_ac::Vector{Float64}
    pindex::Dict{String, Int}       # "R1", "C2", "L1", "G1", "E1", "V1.dc" -> 0-based index into p
end

struct CsParamLayout
    res_r::Int32; cap_c::Int32; ind_l::Int32; vccs_gain::Int32; vcvs_gain::Int32
    mos_vth::Int32; mos_kp::Int32; mos_w::Int32; mos_l::Int32
    wave_dc::Int32; wave_data::Int32; gmin::Int32; va_prm::Int32
    n_params::Int32
end

# the parameter vector's index of every named device value, from the
# library's layout of p; a source's value is "name.dc" (its wave_dc entry)
function param_indices(ctx::Context, cid, a)
    lay = Ref{CsParamLayout}()
    check(ctx, ccall((:cs_circuit_layout, lib), Int32, (Ptr{Cvoid}, Int32, Ref{CsParamLayout}), ctx, cid, lay))
    L = lay[]
    base = Dict(:res => L.res_r, :cap => L.cap_c, :ind => L.ind_l, :vccs => L.vccs_gain, :vcvs => L.vcvs_gain)
    d = Dict{String, Int}()
    for (name, (kind, k)) in a[:devices]
        if kind === :vsrc || kind === :isrc
            d[name * ".dc"] = L.wave_dc + a[kind === :vsrc ? :vsrc_wave : :isrc_wave][k]
        else
            d[name] = base[kind] + k - 1
        end
    end
    d
end

function HIPSystem(ctx::Context, circuit; gmin=1e-12)
    a, unknowns = lower(circuit)
    cid = Ref{Int32}(0)
    GC.@preserve a begin
        nl = netlist(a; gmin)
        check(ctx, ccall((:cs_circuit_load, lib), Int32, (Ptr{Cvoid}, Ref{CsNetlist}, Ref{Int32}), ctx, nl, cid))
    end
    info = zeros(Int32, 16)
    check(ctx, ccall((:cs_circuit_info_get, lib), Int32, (Ptr{Cvoid}, Int32, Ptr{Int32}), ctx, cid[], info))
    HIPSystem(ctx, cid[], info[1], info[3], info[5], unknowns, a[:src_ac], param_indices(ctx, cid[], a))
end

function default_params(s::HIPSystem)
    p = zeros(s.n_params)
    check(s.ctx, ccall((:cs_circuit_default_params, lib), Int32, (Ptr{Cvoid}, Int32, Ptr{Float64}), s.ctx, s.cid, p))
    p
end

# jac_prototype: the library's CSR pattern as a SparseMatrixCSC
function jac_prototype(s::HIPSystem)
    rp = zeros(Int32, s.n + 1); ci = zeros(Int32, s.nnz)
    check(s.ctx, ccall((:cs_circuit_pattern, lib), Int32, (Ptr{Cvoid}, Int32, Ptr{Int32}, Ptr{Int32}),
                       s.ctx, s.cid, rp, ci))
    rows = [r for r in 1:s.n for _ in rp[r]+1:rp[r+1]]
    sparse(rows, ci .+ 1, ones(s.nnz), s.n, s.n)
end

# f!(out, du, u, p, t) and jac!(J, du, u, p, γ, t) of the DAE contract
function hip_daefunction(s::HIPSystem)
    proto = jac_prototype(s)
    # CSR value k lands at the CSC position of the same (row, col)
    rp = zeros(Int32, s.n + 1); ci = zeros(Int32, s.nnz)
    check(s.ctx, ccall((:cs_circuit_pattern, lib), Int32, (Ptr{Cvoid}, Int32, Ptr{Int32}, Ptr{Int32}),
                       s.ctx, s.cid, rp, ci))
    pos = [findfirst(==(r), rowvals(proto)[nzrange(proto, ci[k] + 1)]) + first(nzrange(proto, ci[k] + 1)) - 1
           for r in 1:s.n for k in rp[r]+1:rp[r+1]]
    vals = zeros(s.nnz)
    f! = (out, du, u, p, t) -> check(s.ctx, ccall((:cs_residual, lib), Int32,
        (Ptr{Cvoid}, Int32, Ptr{Float64}, Ptr{Float64}, Ptr{Float64}, Ptr{Float64}, Float64, Int32),
        s.ctx, s.cid, out, du, u, p, t, 0))
    jac! = function (J, du, u, p, γ, t)
        check(s.ctx, ccall((:cs_jacobian, lib), Int32,
            (Ptr{Cvoid}, Int32, Ptr{Float64}, Ptr{Float64}, Ptr{Float64}, Ptr{Float64}, Float64, Float64, Int32),
            s.ctx, s.cid, vals, du, u, p, γ, t, 0))
        nonzeros(J)[pos] .= vals
        J
    end
    SciMLBase.DAEFunction{true}(f!; jac=jac!, jac_prototype=proto)
end

# ---- analyses: the plain path and the batch ---------------------------------------------
struct HIPBackend
    device::Int
end
HIPBackend() = HIPBackend(0)

struct HIPSolution
    t::Vector{Float64}
    u::Matrix{Float64}          # n x n_out
    unknowns::Vector{String}
    retcode::SciMLBase.ReturnCode.T
    stats::CsTranStats
end
Base.getindex(s::HIPSolution, name::AbstractString) = s.u[findfirst(==(name), s.unknowns), :]

"""
    tran!(circ, tspan, ::HIPBackend; reltol=1e-6, abstol=1e-9, n_out=201, u0=nothing, jac_reuse=true,
          kernel=:plain)

`tran!(circ, tspan)` (src/sweeps.jl:450-465) with the whole step loop on the
GPU: CedarDCOp's initialisation unless u0 is given, BDF, Newton (modified
Newton, the step's first factors reused by its later iterations, as IDA
does, unless jac_reuse=false) and the sparse LU on the device.
kernel=:lds runs the circuit as a batch of one in the LDS-resident kernel,
the whole transient in one launch (several times faster for a circuit that
fits; full Newton, so jac_reuse does not apply).
"""
function CedarSim.tran!(circ, tspan, be::HIPBackend; reltol=1e-6, abstol=1e-9, n_out=201, u0=nothing,
                       jac_reuse=true, kernel::Symbol=:plain)
    kernel in (:plain, :lds) || throw(ArgumentError("kernel is :plain or :lds"))
    ctx = Context(be.device)
    s = HIPSystem(ctx, circ)
    o = CsTranOpts()
    o.t_start, o.t_stop = tspan
    o.reltol, o.abstol = reltol, abstol
    o.n_out = n_out
    o.dt_out = (tspan[2] - tspan[1]) / (n_out - 1)
    o.init = u0 === nothing ? CS_INIT_DCOP : CS_INIT_UIC
    o.jac_reuse = jac_reuse && kernel == :plain ? 1 : 0   # IDA's Jacobian reuse within a step
    o.batch_kernel = kernel == :lds ? CS_BATCH_KERNEL_LDS : CS_BATCH_KERNEL_GLOBAL
    wave = zeros(s.n, n_out)                         # column k = sample k
    uf = zeros(s.n)
    st = CsTranStats()
    p = default_params(s)
    rc = ccall((:cs_tran, lib), Int32,
        (Ptr{Cvoid}, Int32, Ptr{Float64}, Ptr{Float64}, Ref{CsTranOpts}, Ptr{Float64}, Ptr{Float64}, Ref{CsTranStats}),
        ctx, s.cid, p, u0 === nothing ? Ptr{Float64}(C_NULL) : u0, o, wave, uf, st)
    rc in (-1, -2, -3, -7, -8) && check(ctx, rc)
    HIPSolution(collect(range(tspan[1], tspan[2]; length=n_out)), wave, s.unknowns, retcode(rc), st)
end

"""
    tran_sens(circ, tspan, params, ::HIPBackend; reltol=1e-6, abstol=1e-9, n_out=201, u0=nothing)
        -> (sol::HIPSolution, sens::Array{Float64,3})

ODEForwardSensitivityProblem + extract_local_sensitivities
(test/sensitivity.jl:29-41,55-66) on the GPU (cs_tran_sens): `params` names
device values ("R1", "C2", "L1", "G1", "E1", "V1.dc"); sens[i, j, k] is
d u_i / d params[j] at output sample k, the sensitivity of the discrete
solution on its own step sequence.
"""
function tran_sens(circ, tspan, params::Vector{String}, be::HIPBackend; reltol=1e-6, abstol=1e-9, n_out=201,
                   u0=nothing)
    ctx = Context(be.device)
    s = HIPSystem(ctx, circ)
    o = CsTranOpts()
    o.t_start, o.t_stop = tspan
    o.reltol, o.abstol = reltol, abstol
    o.n_out = n_out
    o.dt_out = (tspan[2] - tspan[1]) / (n_out - 1)
    o.init = u0 === nothing ? CS_INIT_DCOP : CS_INIT_UIC
    sp = Int32[get(() -> error("no sensitivity parameter $nm"), s.pindex, nm) for nm in params]
    wave = zeros(s.n, n_out)
    sens = zeros(s.n, length(sp), n_out)             # the C layout n_out x n_sp x n, column-major
    uf = zeros(s.n)
    st = CsTranStats()
    rc = ccall((:cs_tran_sens, lib), Int32,
        (Ptr{Cvoid}, Int32, Ptr{Float64}, Ptr{Float64}, Ref{CsTranOpts}, Int32, Ptr{Int32}, Ptr{Float64},
         Ptr{Float64}, Ptr{Float64}, Ref{CsTranStats}),
        ctx, s.cid, default_params(s), u0 === nothing ? Ptr{Float64}(C_NULL) : u0, o, length(sp), sp, wave,
        sens, uf, st)
    rc in (-1, -2, -3, -7, -8) && check(ctx, rc)
    HIPSolution(collect(range(tspan[1], tspan[2]; length=n_out)), wave, s.unknowns, retcode(rc), st), sens
end

# the parameter vector of lowered arrays, in the library's layout (include/cedarhip.h:
# res_r cap_c ind_l vccs_gain vcvs_gain, no square-law MOSFETs from the walker,
# wave_dc wave_data gmin va_prm)
param_vector(a; gmin=1e-12) = vcat(a[:res_r], a[:cap_c], a[:ind_l], a[:vccs_gain], a[:vcvs_gain],
                                   a[:wave_dc], a[:wave_data], [gmin], a[:va_prm])

"""
    tran!(cs::CircuitSweep, tspan, ::HIPBackend; reltol=1e-6, abstol=1e-9, n_out=201, u0=nothing)
        -> Vector{HIPSolution}

tran!.(cs) (src/sweeps.jl:489-501) as one batched launch: every sweep point is
lowered on the host, the points share the first point's compiled topology
and each runs as one instance with its own parameter vector (cs_batch_*).
"""
function CedarSim.tran!(cs::CedarSim.CircuitSweep, tspan, be::HIPBackend; reltol=1e-6, abstol=1e-9,
                        n_out=201, u0=nothing)
    ctx = Context(be.device)
    points = collect(cs)
    isempty(points) && return HIPSolution[]
    s = HIPSystem(ctx, first(points))
    params = Vector{Float64}[]
    for pt in points
        a, unknowns = lower(pt)
        unknowns == s.unknowns || error("tran! over a CircuitSweep: the sweep changes the circuit's topology")
        p = param_vector(a)
        length(p) == s.n_params || error("tran! over a CircuitSweep: the sweep changes the parameter layout")
        push!(params, p)
    end
    o = CsTranOpts()
    o.t_start, o.t_stop = tspan
    o.reltol, o.abstol = reltol, abstol
    o.n_out = n_out
    o.dt_out = (tspan[2] - tspan[1]) / (n_out - 1)
    o.init = u0 === nothing ? CS_INIT_DCOP : CS_INIT_UIC
    ni = length(points)
    cids = fill(s.cid, ni)
    bid = Ref{Int32}(0)
    check(ctx, ccall((:cs_batch_create, lib), Int32,
        (Ptr{Cvoid}, Int32, Ptr{Int32}, Ptr{Float64}, Ptr{Float64}, Ref{CsTranOpts}, Ref{Int32}),
        ctx, ni, cids, reduce(vcat, params), u0 === nothing ? Ptr{Float64}(C_NULL) : repeat(u0, ni), o, bid))
    try
        ms = Ref{Float64}(0)
        check(ctx, ccall((:cs_batch_run, lib), Int32, (Ptr{Cvoid}, Int32, Ref{Float64}), ctx, bid[], ms))
        wave = zeros(s.n, n_out, ni)                 # per instance n_out x n samples (C order)
        uf = zeros(s.n * ni)
        stv = Vector{CsTranStatsRec}(undef, ni)
        check(ctx, ccall((:cs_batch_results, lib), Int32,
            (Ptr{Cvoid}, Int32, Ptr{Float64}, Ptr{Float64}, Ptr{CsTranStatsRec}), ctx, bid[], wave, uf, stv))
        t = collect(range(tspan[1], tspan[2]; length=n_out))
        [HIPSolution(t, wave[:, :, i], s.unknowns, retcode(stv[i].retcode), CsTranStats(stv[i])) for i in 1:ni]
    finally
        ccall((:cs_batch_destroy, lib), Int32, (Ptr{Cvoid}, Int32), ctx, bid[])
    end
end

"""dc!(circ, ::HIPBackend) — dc!(circ) (src/sweeps.jl:437-448) on the GPU."""
function CedarSim.dc!(circ, be::HIPBackend)
    ctx = Context(be.device)
    s = HIPSystem(ctx, circ)
    u = zeros(s.n); st = CsTranStats()
    rc = ccall((:cs_dcop, lib), Int32,
        (Ptr{Cvoid}, Int32, Ptr{Float64}, Ref{CsTranOpts}, Ptr{Float64}, Ref{CsTranStats}),
        ctx, s.cid, default_params(s), CsTranOpts(), u, st)
    rc in (-1, -2, -3, -7, -8) && check(ctx, rc)
    Dict(zip(s.unknowns, u)), retcode(rc)
end

# ---- small-signal AC and noise (src/ac.jl:75-284) ------------------------------------
"""
    ac!(circ, ::HIPBackend) -> (ωs, names) -> Matrix{ComplexF64}

ac!(circ) on the GPU: the DC operating point (cs_dcop), then the response
(G + jωC) x = b at the requested unknowns for the sources' |ac| magnitudes
(cs_ac); the returned closure plays freqresp(ac, sym, ωs)."""
function CedarSim.ac!(circ, be::HIPBackend)
    ctx = Context(be.device)
    s = HIPSystem(ctx, circ)
    p = default_params(s)
    u = zeros(s.n); st = CsTranStats()
    check(ctx, ccall((:cs_dcop, lib), Int32,
        (Ptr{Cvoid}, Int32, Ptr{Float64}, Ref{CsTranOpts}, Ptr{Float64}, Ref{CsTranStats}),
        ctx, s.cid, p, CsTranOpts(), u, st))
    src_ac = s.src_ac
    function freqresp(ωs::Vector{Float64}, names::Vector{String})
        obs = Int32[findfirst(==(nm), s.unknowns) - 1 for nm in names]
        out = zeros(Float64, 2 * length(names) * length(ωs))
        check(ctx, ccall((:cs_ac, lib), Int32,
            (Ptr{Cvoid}, Int32, Ptr{Float64}, Ptr{Float64}, Ptr{Float64}, Int32, Ptr{Float64}, Int32,
             Ptr{Int32}, Ptr{Float64}),
            ctx, s.cid, p, u, isempty(src_ac) ? [0.0] : src_ac, length(ωs), ωs, length(obs), obs, out))
        z = complex.(out[1:2:end], out[2:2:end])
        permutedims(reshape(z, length(names), length(ωs)))   # rows: frequencies
    end
    freqresp
end

"""
    noise!(circ, ::HIPBackend; temp=27) -> (ωs, name) -> Vector{Float64}

noise!(circ) on the GPU; the returned closure plays PSD(noise, sym, ωs):
the resistors' thermal noise 4kT/R at the node, one transposed solve per
frequency (cs_noise)."""
function CedarSim.noise!(circ, be::HIPBackend; temp=27.0)
    ctx = Context(be.device)
    s = HIPSystem(ctx, circ)
    p = default_params(s)
    u = zeros(s.n); st = CsTranStats()
    check(ctx, ccall((:cs_dcop, lib), Int32,
        (Ptr{Cvoid}, Int32, Ptr{Float64}, Ref{CsTranOpts}, Ptr{Float64}, Ref{CsTranStats}),
        ctx, s.cid, p, CsTranOpts(), u, st))
    function psd(ωs::Vector{Float64}, name::String)
        obs = Int32(findfirst(==(name), s.unknowns) - 1)
        out = zeros(Float64, length(ωs))
        check(ctx, ccall((:cs_noise, lib), Int32,
            (Ptr{Cvoid}, Int32, Ptr{Float64}, Ptr{Float64}, Float64, Int32, Ptr{Float64}, Int32, Ptr{Float64}),
            ctx, s.cid, p, u, Float64(temp), length(ωs), ωs, obs, out))
        out
    end
    psd
end

"""
    tran_batch(ctx, systems, params, o; u0=nothing)

The tran!. broadcast over a sweep (src/sweeps.jl:489-501) as one launch:
instance i runs systems[i] with parameter vector params[i].
"""
function tran_batch(ctx::Context, systems::Vector{HIPSystem}, params::Vector{Vector{Float64}}, o::CsTranOpts;
                    u0=nothing)
    cids = Int32[s.cid for s in systems]
    p = reduce(vcat, params)
    u = u0 === nothing ? Ptr{Float64}(C_NULL) : reduce(vcat, u0)
    bid = Ref{Int32}(0)
    check(ctx, ccall((:cs_batch_create, lib), Int32,
        (Ptr{Cvoid}, Int32, Ptr{Int32}, Ptr{Float64}, Ptr{Float64}, Ref{CsTranOpts}, Ref{Int32}),
        ctx, length(cids), cids, p, u, o, bid))
    ms = Ref{Float64}(0)
    check(ctx, ccall((:cs_batch_run, lib), Int32, (Ptr{Cvoid}, Int32, Ref{Float64}), ctx, bid[], ms))
    uf = zeros(sum(s.n for s in systems))
    stv = Vector{CsTranStatsRec}(undef, length(cids))
    check(ctx, ccall((:cs_batch_results, lib), Int32, (Ptr{Cvoid}, Int32, Ptr{Float64}, Ptr{Float64},
                     Ptr{CsTranStatsRec}), ctx, bid[], C_NULL, uf, stv))
    ccall((:cs_batch_destroy, lib), Int32, (Ptr{Cvoid}, Int32), ctx, bid[])
    uf, CsTranStats.(stv), ms[]
end

# ---- differentiation: the supply energy and its adjoint ---------------------------------
"""
    supply_energy(s, p, u0, o; vsrc=0)

Energy delivered by voltage source `vsrc` over the transient (trapezoid on
the accepted points).  Its rrule returns the library's discrete adjoint
dE/dW for every MOSFET width, placed at the widths' slots of p.
"""
function supply_energy(s::HIPSystem, p::Vector{Float64}, u0::Vector{Float64}, o::CsTranOpts; vsrc=0)
    E, _ = energy_and_gradient(s, p, u0, o; vsrc)
    E
end

function energy_and_gradient(s::HIPSystem, p, u0, o; vsrc=0, ckpt_every=64, max_steps=400_000)
    oo = deepcopy(o); oo.init = CS_INIT_UIC
    ao = CsAdjointOpts(vsrc, ckpt_every, max_steps)
    lay = zeros(Int32, 14)
    check(s.ctx, ccall((:cs_circuit_layout, lib), Int32, (Ptr{Cvoid}, Int32, Ptr{Int32}), s.ctx, s.cid, lay))
    n_mos = lay[8] - lay[7]                    # mos_w - mos_kp
    E = zeros(1); g = zeros(max(n_mos, 1)); ns = zeros(Int64, 1)
    st = Vector{CsTranStatsRec}(undef, 1); ms = Ref{Float64}(0)
    check(s.ctx, ccall((:cs_adjoint_batch, lib), Int32,
        (Ptr{Cvoid}, Int32, Ptr{Int32}, Ptr{Float64}, Ptr{Float64}, Ref{CsTranOpts}, Ref{CsAdjointOpts},
         Ptr{Float64}, Ptr{Float64}, Ptr{Int64}, Ptr{Float64}, Ptr{Int32}, Ptr{CsTranStatsRec}, Ref{Float64}),
        s.ctx, 1, Int32[s.cid], p, u0, oo, ao, E, g, ns, C_NULL, C_NULL, st, ms))
    dp = zeros(length(p))
    dp[lay[8]+1:lay[8]+n_mos] .= g[1:n_mos]    # dE/dW at the widths' slots
    E[1], dp
end

function ChainRulesCore.rrule(::typeof(supply_energy), s::HIPSystem, p, u0, o; vsrc=0)
    E, dp = energy_and_gradient(s, p, u0, o; vsrc)
    pullback(Ē) = (NoTangent(), NoTangent(), Ē .* dp, NoTangent(), NoTangent())
    E, pullback
end

export HIPBackend, HIPSystem, hip_daefunction, tran_batch, tran_sens, supply_energy, lower

end # module
