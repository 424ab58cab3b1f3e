// tran_lds.hip — the LDS-resident batched transient kernels.
//
// k_tran_pack (the batched transient): one launch for the whole batch.  A
// persistent grid of workgroups of up to kPackWaves wavefronts walks a queue of
// chunks.  A chunk is up to kPackSegs segments, each a run of instances of
// one circuit: the workgroup copies the segments' plan images into LDS and
// each wavefront runs one instance's whole transient (lds_core.h) in its own
// LDS region beside its circuit's image.  Mixing a large circuit's instances
// with a small circuit's fills both the wavefront slots and the LDS of a
// workgroup, so that every instance of a batch can be resident at once.
#include "lds_core.h"

namespace cedar {

namespace {

using namespace lds;

// Measured against the descriptor-driven form of this kernel (two-level index
// lists per row and task, plan header in scalar registers, eight instances
// per workgroup whatever the batch): 4096 rings of 11 to 101 stages over
// 0.5 ns 394 -> 218 ms; 60 of them 309 -> 116 ms; one 33-stage ring 229 ->
// 101 ms; 1001 inverters over 2 ns from their DC points 16.5 -> 11.0 ms.
//
// OCC wavefronts per SIMD.  OCC = 4 (128 VGPRs): two workgroups of eight per
// CU, so that every instance of a 4096-instance batch is resident at once; also
// where LDS holds few instances beside an image and only so many registers
// let a second workgroup in (2048 101-stage rings over 20 ps, five to a
// workgroup: 12.3 ms in two rounds, 7.9 in one).  OCC = 2 (256 VGPRs) for
// batches that fill no more, and for circuits of more than 128 rows (NR = 4,
// 196 VGPRs, of which LDS holds at most three beside an image: two workgroups
// of their own size fit; 1536 149-stage rings 15.0 ms when workgroups had eight
// wavefronts, 8.5 now).  DYN: some circuit has a source that is not DC.
template <int NR, bool DYN, int OCC>
__global__ __launch_bounds__(W* kPackWaves) __attribute__((amdgpu_waves_per_eu(OCC)))
void k_tran_pack(const LdsArgs* args) {
    constexpr bool ILP = NR <= 2 && OCC == 2;
    extern __shared__ double lds_mem[];
    __shared__ int s_chunk;
    ConstPtr<LdsArgs> A = as_const(args);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint16_t* blob = reinterpret_cast<uint16_t*>(lds_mem);
    for (;;) {
        A = fresh(A);
        if (threadIdx.x == 0) s_chunk = atomicAdd(A->queue, 1);
        __syncthreads();
        const int ch = __builtin_amdgcn_readfirstlane(s_chunk);
        __syncthreads();
        if (ch >= A->n_chunks) break;
        const int s0 = __builtin_amdgcn_readfirstlane(A->chunk_seg[ch]);
        const int s1 = __builtin_amdgcn_readfirstlane(A->chunk_seg[ch + 1]);
        // every segment's plan image, at its own offset (multiples of 8 words)
        int seg = -1;
        for (int j = s0; j < s1; j++) {
            const int4 sa = A->segs[2 * j], sb = A->segs[2 * j + 1];
            Hdr c = as_const(A->cplans + __builtin_amdgcn_readfirstlane(sa.x));
            copy_image(c->blob, c->words, blob + __builtin_amdgcn_readfirstlane(sb.x), (int)threadIdx.x,
                       (int)blockDim.x);
            const int w0 = __builtin_amdgcn_readfirstlane(sb.w), cnt = __builtin_amdgcn_readfirstlane(sa.z);
            if (wave >= w0 && wave < w0 + cnt) seg = j;
        }
        __syncthreads();
        if (seg >= 0) {
            const int4 sa = A->segs[2 * seg], sb = A->segs[2 * seg + 1];
            const int cid = __builtin_amdgcn_readfirstlane(sa.x);
            const int k = wave - __builtin_amdgcn_readfirstlane(sb.w);
            const int inst = __builtin_amdgcn_readfirstlane(A->order[__builtin_amdgcn_readfirstlane(sa.y) + k]);
            // the circuit's own rows per lane (at most NR)
            const int nr = __builtin_amdgcn_readfirstlane(sa.w);
            double* region = lds_mem + __builtin_amdgcn_readfirstlane(sb.y) +
                             (size_t)k * __builtin_amdgcn_readfirstlane(sb.z);
            const View v{reinterpret_cast<char*>(region), blob + __builtin_amdgcn_readfirstlane(sb.x)};
            Hdr c = as_const(A->cplans + cid);
            const DPlan* P = A->plans + cid;
            NoRec rec;
            if (NR > 1 && nr == 1) run_lds<1, DYN, ILP>(rec, c, A, P, inst, v);
            else if (NR > 2 && nr == 2) run_lds<(NR > 2 ? 2 : NR), DYN, ILP>(rec, c, A, P, inst, v);
            else run_lds<NR, DYN, ILP>(rec, c, A, P, inst, v);
        }
        __syncthreads();
    }
}

// DC operating point of one circuit: the instance code's initial point,
// without the transient's re-initialisation at t_start.  One wavefront and
// one launch where the iteration graph took a launch and a host round trip
// per Newton iteration (20 inverters in a row: 7.0 -> 0.65 ms).
template <int NR, bool DYN>
__global__ __launch_bounds__(W) void k_lds_dcop(const LdsArgs* args) {
    constexpr int NM = 2 * NR;
    extern __shared__ double lds_mem[];
    ConstPtr<LdsArgs> A = as_const(args);
    Hdr c = as_const(A->cplans);
    const DPlan* P = A->plans;
    uint16_t* blob = reinterpret_cast<uint16_t*>(lds_mem);
    const int words = c->words, n = c->n;
    copy_image(c->blob, words, blob, lane_id(), W);
    lds_sync();
    const View v{reinterpret_cast<char*>(lds_mem + words / 4), blob};
    DevRegs<NM> dr;
    setup_instance<NM>(c, P, A->params, v, dr);
    double pinv[NR];
    uint32_t flag[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        pinv[r] = 0.0;
        flag[r] = 0;
    }
    lds_sync();
    long long nit = 0;
    const bool ok = init_point<NR, NM, DYN, (NR <= 2)>(c, v, P, dr, A->params[P->p_gmin], false, pinv, flag,
                                                       A->o.t_start, A->o.dc_abstol, nit, true);
    lds_sync();
    for (int k = lane_id(); k < n; k += W) A->u_final[c->colnat[k]] = v.at(c->b_u + 8 * k);
    if (lane_id() == 0) {
        A->stats->newton_iters = nit;
        A->stats->retcode = ok ? CS_OK : CS_E_NOCONV;
    }
}

// One Newton iteration of the batched kernels' instance code, recorded: the
// circuit's plan image and one instance in LDS, exactly as k_tran_pack holds
// them; the state u, the charge terms qx (pivot order) and a0 come from the
// caller.  Writes the assembled Jacobian (F order), the residual (pivot
// rows), the LU factors (F order) and the Newton update (pivot columns).
template <int NR>
__global__ __launch_bounds__(W) void k_lds_probe(const CPlan* cp, const DPlan* P, const double* p,
                                                 const double* u_piv, const double* qx_piv, double a0,
                                                 double t, int mode, double* f_asm, double* res_piv,
                                                 double* f_lu, double* dx_piv) {
    constexpr int NM = 2 * NR;
    extern __shared__ double lds_mem[];
    uint16_t* blob = reinterpret_cast<uint16_t*>(lds_mem);
    Hdr c = as_const(cp);
    const int words = c->words, n = c->n, nnz = c->nnz;
    copy_image(c->blob, words, blob, lane_id(), W);
    lds_sync();
    const View v{reinterpret_cast<char*>(lds_mem + words / 4), blob};
    DevRegs<NM> dr;
    setup_instance<NM>(c, P, p, v, dr);
    double qx[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int k = row_of(lane_id(), r, n);
        qx[r] = qx_piv[k];
        v.at(c->b_u + 8 * k) = u_piv[k];
    }
    lds_sync();
    eval_sources<true>(c, v, t, mode);
    lds_sync();
    const Hot h = load_hot(c);
    eval_mos<NM, true>(h, v, dr, p[P->p_gmin]);
    lds_sync();
    assemble<NR, true>(h, v, a0, qx);
    lds_sync();
    for (int e = lane_id(); e < nnz; e += W) f_asm[e] = v.at(c->b_F + 8 * e);
    for (int k = lane_id(); k < n; k += W) res_piv[k] = -v.at(c->b_x + 8 * k);
    lds_sync();
    factor_solve<true>(h, v);
    lds_sync();
    for (int e = lane_id(); e < nnz; e += W) f_lu[e] = v.at(c->b_F + 8 * e);
    for (int k = lane_id(); k < n; k += W) dx_piv[k] = v.at(c->b_x + 8 * k);
}

}  // namespace

hipError_t launch_lds_probe(int nr, const CPlan* cp, const DPlan* P, const double* p, const double* u_piv,
                            const double* qx_piv, double a0, double t, int mode, double* f_asm,
                            double* res_piv, double* f_lu, double* dx_piv, size_t lds, hipStream_t s) {
    switch (nr) {
        case 1: hipLaunchKernelGGL(k_lds_probe<1>, dim3(1), dim3(W), lds, s, cp, P, p, u_piv, qx_piv, a0, t,
                                   mode, f_asm, res_piv, f_lu, dx_piv); break;
        case 2: hipLaunchKernelGGL(k_lds_probe<2>, dim3(1), dim3(W), lds, s, cp, P, p, u_piv, qx_piv, a0, t,
                                   mode, f_asm, res_piv, f_lu, dx_piv); break;
        case 4: hipLaunchKernelGGL(k_lds_probe<4>, dim3(1), dim3(W), lds, s, cp, P, p, u_piv, qx_piv, a0, t,
                                   mode, f_asm, res_piv, f_lu, dx_piv); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

namespace {
typedef void (*PackKernel)(const LdsArgs*);
PackKernel pack_kernel(const PackShape& k) {
    switch (k.nr) {
        case 1:
            if (k.occ == 4) return k.dyn ? k_tran_pack<1, true, 4> : k_tran_pack<1, false, 4>;
            return k.dyn ? k_tran_pack<1, true, 2> : k_tran_pack<1, false, 2>;
        case 2:
            if (k.occ == 4) return k.dyn ? k_tran_pack<2, true, 4> : k_tran_pack<2, false, 4>;
            return k.dyn ? k_tran_pack<2, true, 2> : k_tran_pack<2, false, 2>;
        case 4: return k.dyn ? k_tran_pack<4, true, 2> : k_tran_pack<4, false, 2>;
        default: return nullptr;
    }
}
}  // namespace

// A CU deals a workgroup's wavefronts to its four SIMDs from the first one on,
// so a workgroup of five takes two places on that one: of three per SIMD they
// leave no room for a second workgroup, which the occupancy query (twelve
// places, ten taken) admits.  2048 101-stage rings, five to a workgroup,
// went in two rounds that way.
int pack_max_blocks(const PackShape& k, size_t lds) {
    int nb = 0, per_simd = 0;
    const PackKernel f = pack_kernel(k);
    if (!f || hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, W * k.waves, lds) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_simd, f, W * 4, 0) != hipSuccess)
        return 0;
    const int by_simd = per_simd / ((k.waves + 3) / 4);
    return nb < by_simd ? nb : by_simd;
}

hipError_t launch_tran_pack(const PackShape& k, const LdsArgs* d_args, int nblocks, size_t lds, hipStream_t s) {
    const PackKernel f = pack_kernel(k);
    if (!f) return hipErrorInvalidValue;
    hipLaunchKernelGGL(f, dim3(nblocks), dim3(W * k.waves), lds, s, d_args);
    return hipGetLastError();
}

hipError_t launch_lds_dcop(int nr, bool dyn, const LdsArgs* d_args, size_t lds, hipStream_t s) {
    void (*f)(const LdsArgs*) = nullptr;
    switch (nr) {
        case 1: f = dyn ? k_lds_dcop<1, true> : k_lds_dcop<1, false>; break;
        case 2: f = dyn ? k_lds_dcop<2, true> : k_lds_dcop<2, false>; break;
        case 4: f = dyn ? k_lds_dcop<4, true> : k_lds_dcop<4, false>; break;
        default: return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(f, dim3(1), dim3(W), lds, s, d_args);
    return hipGetLastError();
}

size_t lds_kernel_bytes(int32_t dbl_max, int32_t words_max) {
    return 8 * (size_t)dbl_max + 2 * (size_t)words_max;
}

}  // namespace cedar
