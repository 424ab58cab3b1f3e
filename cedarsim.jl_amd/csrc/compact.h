// compact.h — the 16-bit plan image of the LDS-resident batched kernels.
//
// Everything one Newton iteration reads is packed into one uint16 "blob"
// that a workgroup copies into LDS when it starts an instance, so the Newton
// loop issues no global loads at all.  State vectors live in pivot order:
// index k is both permuted row k and permuted column k (the static pivot
// sits on the diagonal), so the solve's output x[k] updates unknown k and the
// row-wise charge of row k belongs to the lane that owns k.
//
// An instance's numbers are one LDS region of doubles, and every operand in
// the blob is a byte offset from its start (a multiple of 8):
//
//   GC[2*(nlin+1)]  G and C of each linear entry side by side (one 16-byte
//                   read); the pair after the last is (0, 0)
//   F[nnz] x[n] inv[n] u[n]
//   zero, one, trash   constants 0.0 and 1.0; a slot nothing reads
//   st[3*n_mos + n_src]  stamps: id, dI/dVd, dI/dVg by device, then sources
//   wd[]            source data, each source's dc value after its data
//
// A stamp reference is the stamp's byte offset with the sign to apply in bit
// 0; dI/dVs = -(dI/dVd + dI/dVg) is expanded into two references.
//
// The iteration is straight streams of records, one record per lane and no
// index read that depends on another index, so the chain of one record is
// two LDS reads deep (the record, its operands):
//
//   ea[4*]  e r0 r1 -            F = r0 + r1        (entry without linear part)
//   eb[4*]  e l r0 r1            F = G + a0 C + r0 + r1
//   ec[8*]  e l r0..r5           the same with up to six references
//   ed[8*]  e l r0 r1 inv r2 r3  a diagonal the factorization never updates:
//                                also inv = 1/F
//   ez[]    e                    fill: F = 0
//   rr[8*n] l0 nl c0 r0..r4      residual of pivot row k: linear entries
//                                [l0, l0+nl), the byte offset of the first
//                                one's u, and references; nl = 0xFFFF: a long row
//                                (r0: its count of linear entries)
//   lcol[]                       byte offset of u[column] per linear entry
//   items[8*] dst q0 q1 l0 l1 k fl -   sums for the whole wavefront, in
//                                pairs: entries with many references (fl =
//                                0) and the residuals of long rows (fl = 1),
//                                references refs[q0..q1), linear entries [l0, l1)
//   src[4*] kind, offset in wd, length, byte offset of the stamp
//   steps[2*] the program of the solve: LU with the forward substitution
//                                folded in (Ly = b is the extra column of
//                                the factorization), then the backward
//                                substitution.  A step is up to 64 records
//                                of one kind, one per lane; a step reads what
//                                earlier steps wrote.  Low word: record
//                                number; high word: count - 1, kind << 6.
//                                One more descriptor follows the last, so
//                                that the next one can always be read ahead
//   rec[8*]                      the records: with V the region,
//     SP_SCALE  d0 s0 .. d3 s3      V[d] *= V[s], four times
//     SP_MUL1   d s a0 b0           V[d] = (V[d] - V[a0]V[b0]) V[s]
//     SP_MUL3   d s a0 b0 .. a2 b2  the same with three products
//     SP_DIA3   d i a0 b0 .. a2 b2  V[d] -= the products;  V[i] = 1/V[d]
//     SP_LMUL, SP_LDIA  d s ub ue   with the pairs upd[ub..ue), each record
//                                   by the whole wavefront
//   upd[2*] a b                  the pairs of the long tasks
//
// A task with more products than a record holds is continued in the next
// step (its partial result stays in V[d]); one with more than kLongTask is a
// long task.  Every class of records has at least one (on the trash slot), so
// that lanes past a class's end can read its last record.  The transposed
// program (adjoint: U^T, then L^T) and the linear entries by column (cdesc,
// lcl, lrow) follow after `words` and reach to `words_adj`; the transient
// copies only the first part.
#pragma once
#include <cstddef>
#include <cstdint>
#include <vector>

namespace cedar {

constexpr int32_t kLongRow = 16;     // linear entries of a residual beyond which the wavefront sums it
constexpr int32_t kEntRefs = 6;      // references an entry record holds
constexpr int32_t kRowRefs = 5;      // references a residual record holds
constexpr int32_t kLongTask = 12;    // products beyond which a task is a long one
constexpr uint32_t CP_GROUND = 0xFFFF;
// kinds of solve steps
enum : uint32_t { SP_MUL1 = 0, SP_MUL3 = 1, SP_SCALE = 2, SP_DIA3 = 3, SP_LMUL = 4, SP_LDIA = 5 };

struct CPlan {
    int32_t n, nnz, n_mos, n_src, nlin, stamp_n, nwd;
    int32_t words;        // transient image in uint16 (a multiple of 8)
    int32_t words_adj;    // with the adjoint's part
    int32_t dbl;          // LDS doubles of one instance
    // byte offsets into the region
    int32_t b_F, b_x, b_inv, b_u, b_zero, b_one, b_trash, b_st, b_wd;
    // uint16 offsets into the blob, and counts
    int32_t o_ea, n_ea, o_eb, n_eb, o_ec, n_ec, o_ed, n_ed, o_ez, n_ez;
    int32_t o_rr, o_lcol, o_items, n_items, o_refs, o_src;
    int32_t wide_rows;    // some residual record has more than two references or one linear entry
    int32_t wide_ed;      // some ed record has more than two references
    int32_t o_steps, n_lu, n_steps, o_rec, o_upd;   // steps [0, n_lu): LU + forward
    int32_t o_tsteps, n_tsteps, o_cdesc, o_lcl, o_lrow;
    // global arrays, read when an instance starts
    const uint16_t* blob;
    const int32_t* lpos;      // [nlin] F position of each linear entry
    const int32_t* colnat;    // [n] natural unknown of pivot column k
    const int32_t* diffrow;   // [n] pivot row k carries charge
    const int32_t* probe;     // [n] probe slot of pivot column k, or -1
    const int32_t* dev;       // [4*n_mos] byte offsets of u[d], u[g], u[s] (zero slot: ground), type
    const int32_t* devrow;    // [2*n_mos] pivot rows of d and s (0xFFFF ground)
    const double* mos_m;      // [n_mos] m-factors, or null (every m is 1)
    const double* src_m;      // [n_src] m-factors of the source values, or null
};

struct Plan;
// Build the blob and the side arrays.  Returns false (with a reason) when a
// 16-bit index would overflow; the caller then uses the global-plan kernel.
bool build_compact(const Plan& P, std::vector<uint16_t>& blob, CPlan& cp,
                   std::vector<int32_t>& lpos, std::vector<int32_t>& colnat, std::vector<int32_t>& diffrow,
                   std::vector<int32_t>& probe, std::vector<int32_t>& dev,
                   std::vector<int32_t>& devrow, const char** why);

// The packed launch's chunks.  A chunk fills one workgroup: at most `waves`
// instances in at most `segs` segments (runs of one circuit's instances),
// each circuit's image (img bytes) once plus dblb bytes per instance, within
// cap bytes.  Greedy, largest circuit first: a chunk takes as many instances
// of the largest circuit left as fit beside its image and fills its other
// slots and LDS from the smallest circuits left; of the counts of the large
// circuit that fit, it keeps the one that fills the most slots.  order lists
// the circuits, largest first; rem[c] the instances of circuit c to place.
// Returns the chunks in that order (each a list of (circuit, count)) and the
// largest chunk's bytes in need; empty when a circuit does not fit alone.
struct PackSeg { int32_t c, cnt; };
std::vector<std::vector<PackSeg>> pack_chunks(const std::vector<int32_t>& order, const std::vector<size_t>& img,
                                              const std::vector<size_t>& dblb, std::vector<size_t> rem,
                                              int waves, int segs, size_t cap, size_t* need);

}  // namespace cedar
