// gfx950 (CDNA4, wave64) kernels for the local SDDMM and SpMM.
//
//   sddmm: C[e] = S.vv[e] * <A[ii[e],:], B[jj[e],:]>      (reference: src/core_ops.cpp:5-22)
//   spmm : Y[ii[e],:] += A.vv[e] * X[jj[e],:]             (reference: src/core_ops.cpp:24-35)
//
// Both are gather-bound (about 0.25 flop per byte): no MFMA.  The unit of work
// is a row segment (plan_host.h): at most seg_max consecutive entries of one
// row.  A dense row of K reals is nvec 16-byte vectors, covered by LPR lanes
// holding VPL vectors each (nvec = LPR * VPL with the row stride a compile-time
// constant, or nvec < LPR * VPL given at run time in the "ragged" variants, whose
// spare lanes load a vector and count nothing, or a row that ends inside its last vector in the "odd"
// variants, or one shorter than a vector in the "thin" variant; rows over 4 KiB
// run as 4 KiB column slices, one launch each); one wavefront works on 64 / LPR
// segments at once and every global load instruction moves 64 x 16 B.  Segments
// arrive sorted longest first, so the lane groups of a wavefront run the same trip
// count.
//
// A segment is walked in batches of UB entries; what remains is one masked
// batch (the missing entries repeat the last one's loads and store nothing), or,
// in SpMM's short-segment launch, exact batches of UB/2, ..., 2, 1.  Every batch
// is straight-line code: within it all gathers are issued before any arithmetic
// (a scheduling barrier keeps the compiler from serialising them).
//
//   sddmm: the group keeps its A row slice in registers, gathers the B row
//          slices of a batch, and reduces the per-lane partial dot products
//          across the group with a halving exchange (NB-1 exchanges for NB
//          entries instead of NB*log2(LPR)); exchanges inside a 16-lane row
//          are DPP moves, those across rows the gfx950 row swaps
//          (v_permlane16_swap, v_permlane32_swap).  The lane that ends up
//          with entry u's dot product scales it by S.vv and stores it at the
//          caller's position: read per entry, or once per segment where a
//          segment's positions are consecutive; segments for which they are
//          not store in kernel order to a staging vector instead
//          (unstage_pairs_kernel brings those home), and for an arbitrary
//          entry order everything is stored in kernel order and brought home
//          by two tile-local passes through LDS (unpermute_pass1/2_kernel).
//   spmm : lane = slice of K, no cross-lane reduction; the group accumulates
//          a * X[c,:] in registers and does one read-modify-write of the Y
//          row slice.  Rows cut into several segments write partial sums that
//          spmm_fixup adds into Y in a fixed order (no atomics, results are
//          reproducible run to run).
//
// Streams that are read once (indices, sparse values, segment descriptors, A
// rows, Y rows) use non-temporal accesses so that the per-XCD L2 is left to
// the gathered B / X rows, the only operand with reuse.  The gathers themselves
// are plain loads: a non-temporal hint on the gathers of low-degree columns
// was measured to slow both kernels down by 15 to 40 %.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"

namespace spc3d {
namespace {

template <typename T> struct Vec;
template <> struct Vec<float> {
    typedef float type __attribute__((ext_vector_type(4)));
    typedef type loose __attribute__((aligned(4))); // same vector at element alignment
    static constexpr int N = 4;
};
template <> struct Vec<double> {
    typedef double type __attribute__((ext_vector_type(2)));
    typedef type loose __attribute__((aligned(8)));
    static constexpr int N = 2;
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBlock = 256; // 4 wavefronts

template <typename P> __device__ __forceinline__ P nt_load(const P *p)
{
    return __builtin_nontemporal_load(p);
}
template <typename P> __device__ __forceinline__ void nt_store(P v, P *p)
{
    __builtin_nontemporal_store(v, p);
}

__device__ __forceinline__ constexpr int ilog2(int x) { return x <= 1 ? 0 : 1 + ilog2(x >> 1); }

// ---- lane exchange ----------------------------------------------------------
// xchg<S>(v): the value lane (id ^ S) holds.  S < 16 (the only strides the kernels
// use it for; 16 and 32 go through swap_add below) stays inside a 16-lane DPP row: xor 1 and 2 are quad permutes, xor 8 is a rotation by 8, xor 4 is
// half-row mirror (i -> 7 - i = i ^ 7) after quad reverse (i ^ 3).
template <int CTRL> __device__ __forceinline__ int dpp_mov(int v)
{
    // every lane is written (all rows and banks enabled, the patterns used here have
    // no invalid source lane): no previous value to set up
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, false);
}
// Lane u of every 16-lane row to the whole row; u is a constant once the loop around it is unrolled.
__device__ __forceinline__ int row_bcast(int v, int u)
{
    switch (u) { // row_newbcast:u
    case 0: return dpp_mov<0x150>(v);
    case 1: return dpp_mov<0x151>(v);
    case 2: return dpp_mov<0x152>(v);
    case 3: return dpp_mov<0x153>(v);
    case 4: return dpp_mov<0x154>(v);
    case 5: return dpp_mov<0x155>(v);
    case 6: return dpp_mov<0x156>(v);
    case 7: return dpp_mov<0x157>(v);
    case 8: return dpp_mov<0x158>(v);
    case 9: return dpp_mov<0x159>(v);
    case 10: return dpp_mov<0x15A>(v);
    case 11: return dpp_mov<0x15B>(v);
    case 12: return dpp_mov<0x15C>(v);
    case 13: return dpp_mov<0x15D>(v);
    case 14: return dpp_mov<0x15E>(v);
    default: return dpp_mov<0x15F>(v);
    }
}
template <int S> __device__ __forceinline__ int xchg_i32(int v)
{
    if constexpr (S == 1)
        return dpp_mov<0xB1>(v); // quad_perm [1,0,3,2]
    else if constexpr (S == 2)
        return dpp_mov<0x4E>(v); // quad_perm [2,3,0,1]
    else if constexpr (S == 4)
        return dpp_mov<0x141>(dpp_mov<0x1B>(v)); // row_half_mirror o quad_perm [3,2,1,0]
    else if constexpr (S == 8)
        return dpp_mov<0x128>(v); // row_ror:8
    else
        return __shfl_xor(v, S, 64);
}
template <int S> __device__ __forceinline__ float xchg(float v)
{
    return __int_as_float(xchg_i32<S>(__float_as_int(v)));
}
template <int S> __device__ __forceinline__ double xchg(double v)
{
    const int lo = xchg_i32<S>(__double2loint(v));
    const int hi = xchg_i32<S>(__double2hiint(v));
    return __hiloint2double(hi, lo);
}

// Halving step across stride 16 or 32: a and b are two partial sums of which the
// lanes with bit S clear go on with a and those with bit S set with b.  One
// v_permlane16_swap / v_permlane32_swap (gfx950) exchanges the odd 16-lane rows of a
// with the even rows of b (the upper 32 lanes of a with the lower 32 of b): the two
// results, added, are a summed over the stride in the lanes with bit S clear and b
// in the others -- no selects and no second move, 2 instructions per 32-bit word
// where the DPP form takes 4.  With b == a it is the all-reduce across the stride.
template <int S> __device__ __forceinline__ void swap_rows(unsigned &a, unsigned &b)
{
    static_assert(S == 16 || S == 32, "row swaps exist for strides 16 and 32");
    if constexpr (S == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0], b = r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = r[0], b = r[1];
    }
}
template <int S> __device__ __forceinline__ float swap_add(float a, float b)
{
    unsigned x = __float_as_uint(a), y = __float_as_uint(b);
    swap_rows<S>(x, y);
    return __uint_as_float(x) + __uint_as_float(y);
}
template <int S> __device__ __forceinline__ double swap_add(double a, double b)
{
    unsigned xl = (unsigned)__double2loint(a), yl = (unsigned)__double2loint(b);
    unsigned xh = (unsigned)__double2hiint(a), yh = (unsigned)__double2hiint(b);
    swap_rows<S>(xl, yl);
    swap_rows<S>(xh, yh);
    return __hiloint2double((int)xh, (int)xl) + __hiloint2double((int)yh, (int)yl);
}

// Order in which the xor strides of an LPR-lane group are used: the steps that
// move the most values come first and get the cheapest exchanges: the row swaps
// of strides 32 and 16, then the single-instruction DPP moves.
template <int LPR> struct Strides;
template <> struct Strides<4> { static constexpr int s[2] = {2, 1}; };
template <> struct Strides<8> { static constexpr int s[3] = {2, 1, 4}; };
template <> struct Strides<16> { static constexpr int s[4] = {8, 2, 1, 4}; };
template <> struct Strides<32> { static constexpr int s[5] = {16, 8, 2, 1, 4}; };
template <> struct Strides<64> { static constexpr int s[6] = {32, 16, 8, 2, 1, 4}; };

// Halving exchange + finishing all-reduce over an LPR-lane group.
// In: part[u] = this lane's partial sum for entry u, u < NB.  Out: part[0] =
// the full sum of entry entry_of<LPR, NB>(sub), identical in every lane that
// maps to that entry.
template <typename T, int LPR, int NB, int STEP = 0, int N = NB>
__device__ __forceinline__ void group_reduce(T (&part)[NB], uint32_t sub)
{
    if constexpr (STEP < ilog2(LPR)) {
        constexpr int S = Strides<LPR>::s[STEP];
        if constexpr (N > 1) {
            const bool upper = (sub & S) != 0;
#pragma unroll
            for (int i = 0; i < N / 2; ++i) {
                if constexpr (S >= 16) {
                    part[i] = swap_add<S>(part[i], part[i + N / 2]);
                } else {
                    const T keep = upper ? part[i + N / 2] : part[i];
                    const T send = upper ? part[i] : part[i + N / 2];
                    part[i] = keep + xchg<S>(send);
                }
            }
            group_reduce<T, LPR, NB, STEP + 1, N / 2>(part, sub);
        } else {
            if constexpr (S >= 16)
                part[0] = swap_add<S>(part[0], part[0]);
            else
                part[0] += xchg<S>(part[0]);
            group_reduce<T, LPR, NB, STEP + 1, 1>(part, sub);
        }
    }
}

// Entry (0 .. NB-1) whose sum lane `sub` holds after group_reduce<LPR, NB>.
template <int LPR, int NB> __device__ __forceinline__ uint32_t entry_of(uint32_t sub)
{
    uint32_t u = 0;
#pragma unroll
    for (int t = 0; t < ilog2(NB); ++t)
        u |= ((sub & Strides<LPR>::s[t]) ? 1u : 0u) << (ilog2(NB) - 1 - t);
    return u;
}

// One lane per entry stores: the lane whose bits for the finishing strides are 0.
template <int LPR, int NB> __device__ __forceinline__ bool is_writer(uint32_t sub)
{
    uint32_t mask = 0;
#pragma unroll
    for (int t = ilog2(NB); t < ilog2(LPR); ++t)
        mask |= Strides<LPR>::s[t];
    return (sub & mask) == 0;
}

// Lane (within the group) that stores entry u after group_reduce<LPR, NB>.
template <int LPR, int NB> __device__ __forceinline__ constexpr int writer_lane(int u)
{
    int lane = 0;
    for (int t = 0; t < ilog2(NB); ++t)
        if ((u >> (ilog2(NB) - 1 - t)) & 1)
            lane |= Strides<LPR>::s[t];
    return lane;
}

// bcast(v, lane): v of lane `lane` of the group.  A group of 64 is the wavefront: the value goes to a
// scalar register, which spares the LDS permute, the address arithmetic of a gather (scalar base, the
// lane's offset) and the registers that hold a batch's weights (R-MAT 18, fp64 K = 128, on top of the copied
// hot rows: SDDMM 370 -> 357 us, SpMM 410 -> 369).  Smaller groups permute through LDS, the
// lane in the instruction's offset: `first` (the byte address of the group's first lane) is made per
// batch, or the compiler would add the lane to it outside the loop and keep all 16 sums in registers.
//
// entry(v, u): where every lane holds what its entry (lane % 16) of a batch of 16 has, a 16-lane DPP row
// holds the whole batch, and one move takes lane u of each row to all of the row: no LDS instruction, no
// wait (SpMM over row tiles, 560 M entries, fp32 K = 128, 19.25 -> 18.83 ms; SDDMM, which has vector
// instructions enough, 17.45 -> 17.75, and the segment kernels, level to 1 % slower, permute).
template <int LPR> struct Bcast {
    int first;
    __device__ __forceinline__ Bcast() : first(0)
    {
        if constexpr (LPR < 64) {
            first = (int)(threadIdx.x & 63u & ~(uint32_t)(LPR - 1)) * 4;
            asm volatile("" : "+v"(first));
        }
    }
    __device__ __forceinline__ uint32_t operator()(uint32_t v, int lane) const
    {
        if constexpr (LPR == 64)
            return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
        else
            return (uint32_t)__builtin_amdgcn_ds_bpermute(first + 4 * lane, (int)v);
    }
    __device__ __forceinline__ uint32_t entry(uint32_t v, int u) const
    {
        if constexpr (LPR == 16 || LPR == 32)
            return (uint32_t)row_bcast((int)v, u);
        else
            return (*this)(v, u);
    }
    __device__ __forceinline__ float entry(float v, int u) const
    {
        return __uint_as_float(entry(__float_as_uint(v), u));
    }
    __device__ __forceinline__ double entry(double v, int u) const
    {
        return __hiloint2double((int)entry((uint32_t)__double2hiint(v), u),
                                (int)entry((uint32_t)__double2loint(v), u));
    }
    __device__ __forceinline__ float operator()(float v, int lane) const
    {
        return __uint_as_float((*this)(__float_as_uint(v), lane));
    }
    __device__ __forceinline__ double operator()(double v, int lane) const
    {
        return __hiloint2double((int)(*this)((uint32_t)__double2hiint(v), lane),
                                (int)(*this)((uint32_t)__double2loint(v), lane));
    }
};

// A segment of the whole wavefront.
__device__ __forceinline__ void uniform(u32x4 &sg)
{
#pragma unroll
    for (int i = 0; i < 4; ++i)
        sg[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)sg[i]);
}

// Segment this lane group works on.  Segments are stored in chunks of kChunk;
// with nq == 8, chunk v belongs to queue v % 8.  The hardware deals the
// workgroups of a dispatch to the 8 XCDs round-robin by workgroup id, starting
// from an XCD that is fixed per hardware queue, so the workgroups b with equal
// (b + rot) % 8 all run on one XCD; they take the chunks of queue (b + rot) % 8
// and the dense rows of one column slice are then only ever gathered through
// one L2.  `rot` lines the queues of the auxiliary stream up with those of the
// main stream.  Any rot gives each segment to exactly one workgroup: if the
// hardware dealt workgroups differently the result would be the same, only
// slower.
template <int G> __device__ __forceinline__ uint64_t seg_index(uint32_t nq, uint32_t rot)
{
    constexpr uint32_t kSegPerBlock = (kBlock / 64) * G;
    constexpr uint32_t kBlocksPerChunk = kChunk / kSegPerBlock;
    static_assert(kChunk % kSegPerBlock == 0, "a chunk is a whole number of workgroups");
    const uint32_t b = blockIdx.x;
    uint64_t chunk;
    uint32_t inner;
    if (nq == 8) {
        const uint32_t j = b >> 3;
        chunk = (uint64_t)(j / kBlocksPerChunk) * 8 + ((b + rot) & 7u);
        inner = j % kBlocksPerChunk;
    } else {
        chunk = b / kBlocksPerChunk;
        inner = b % kBlocksPerChunk;
    }
    return chunk * kChunk + inner * kSegPerBlock + (threadIdx.x >> 6) * G +
           (threadIdx.x & 63u) / (64 / G);
}

// The short-segment launch walks a dependency chain per segment: descriptor, then
// column indices, then the gathers.  The plan keeps the first kFirstCols column indices
// of every short segment in a table addressed by the segment's position (past the
// segment's end they repeat its last column), so that they are fetched beside the
// descriptor instead of after it: two memory latencies per segment instead of three.
// Lane u of a group of LPR >= kFirstCols lanes gets the column of entry u % kFirstCols;
// a group of 4 lanes gets those of entries u and 4 + u.
// stream_c: SDDMM stores its results at permuted positions past the L2 (streaming)
// instead of with plain stores that the L2 can merge: for the blocks of a plan kept in
// column blocks, whose positions are long runs in a staging vector and whose block of
// dense rows is meant to stay in the L2s.
// stage / stage_from: SDDMM results whose position (perm) is stage_from or more go to
// place (position - stage_from) of the staging vector instead of into C (segments whose
// caller's positions are not consecutive; unstage_pairs_kernel brings them home).
// shift: added to the kernel position of an entry when no `perm` is read (a plan whose
// segments all have consecutive positions: perm[start] - start of the segment).
struct Ahead {
    uint32_t first[2] = {0, 0};
    bool stream_c = false;
    uint32_t stage_from = 0xFFFFFFFFu;
    void *stage = nullptr;
    uint32_t shift = 0;
};
constexpr uint32_t kStoreStream = 1u;  // sddmm_seg_kernel flags: Ahead::stream_c
constexpr uint32_t kStoreSegBase = 2u; // positions are perm[segment start] + offset
template <int LPR, bool WIDE>
__device__ __forceinline__ Ahead load_first_cols(const uint32_t *__restrict__ first_cols,
                                                 uint64_t sid, uint32_t sub)
{
    Ahead f;
    if constexpr (!WIDE) {
        constexpr uint32_t GL = (uint32_t)LPR < kFirstCols ? (uint32_t)LPR : kFirstCols;
        const uint32_t *at = first_cols + sid * kFirstCols + (sub & (GL - 1));
        f.first[0] = nt_load(at);
        if constexpr ((uint32_t)LPR < kFirstCols)
            f.first[1] = nt_load(at + LPR);
    }
    return f;
}

// Fills the table above for `n` short segments.
__global__ void __launch_bounds__(kBlock)
first_cols_kernel(const Seg *__restrict__ segs, uint32_t n, const uint32_t *__restrict__ col,
                  uint32_t *__restrict__ first_cols)
{
    const uint64_t t = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    const uint64_t s = t / kFirstCols;
    const uint32_t u = (uint32_t)(t % kFirstCols);
    if (s >= n)
        return;
    const Seg sg = segs[s];
    uint32_t c = 0;
    if (sg.len)
        c = col[sg.start + (u < sg.len ? u : sg.len - 1)];
    first_cols[t] = c;
}

// RG == 1 ("ragged"): a dense row is nvec 16-byte vectors with nvec < LPR * VPL,
// given at run time; lanes whose vector index is >= nvec load the last one and count nothing.  RG == 0: nvec ==
// LPR * VPL exactly and the row stride is a compile-time constant.  RG == 2, 3: below.
template <typename T, int LPR, int VPL, int RG>
__device__ __forceinline__ const typename Vec<T>::type *row_ptr(const T *base, uint32_t row,
                                                                uint32_t sub, uint32_t nvec)
{
    const uint64_t row_bytes = RG > 0 ? (uint64_t)nvec * 16 : (uint64_t)LPR * VPL * 16;
    return reinterpret_cast<const typename Vec<T>::type *>(
               reinterpret_cast<const char *>(base) + (uint64_t)row * row_bytes) +
           sub;
}

template <int LPR, int RG>
__device__ __forceinline__ bool lane_on(uint32_t sub, int v, uint32_t nvec)
{
    return RG <= 0 || sub + (uint32_t)v * LPR < nvec;
}

// 16-byte accesses at element alignment.  (Not through nt_load / nt_store: template
// argument deduction would drop the typedef's alignment.)
template <typename T> __device__ __forceinline__ typename Vec<T>::type loose_load(const char *p)
{
    return *reinterpret_cast<const typename Vec<T>::loose *>(p);
}
// The vector `off` bytes past `at`, the same in every lane of the wavefront.  (Left to itself the compiler
// adds the lane's offset to the loop-invariant base and does the rest in vector registers.)
template <typename T, bool LOOSE>
__device__ __forceinline__ typename Vec<T>::type load_beside(const char *at, uint32_t off)
{
    typedef __attribute__((address_space(1))) const char *Global;
    Global p = (Global)at;
    asm("" : "+s"(p));
    if constexpr (LOOSE)
        return *reinterpret_cast<__attribute__((address_space(1))) const typename Vec<T>::loose *>(p + off);
    else
        return *reinterpret_cast<__attribute__((address_space(1))) const typename Vec<T>::type *>(p + off);
}
template <typename T> __device__ __forceinline__ typename Vec<T>::type loose_load_nt(const char *p)
{
    return __builtin_nontemporal_load(reinterpret_cast<const typename Vec<T>::loose *>(p));
}
template <typename T>
__device__ __forceinline__ void loose_store(typename Vec<T>::type v, char *p)
{
    *reinterpret_cast<typename Vec<T>::loose *>(p) = v;
}
template <typename T>
__device__ __forceinline__ void loose_store_nt(typename Vec<T>::type v, char *p)
{
    __builtin_nontemporal_store(v, reinterpret_cast<typename Vec<T>::loose *>(p));
}

// RG == 2 ("odd"): a dense row of K reals is no whole number of 16-byte vectors
// (the kernels' `nvec` argument carries K).  Rows start at element alignment only,
// and the last vector of a row would reach past its end, so: the lane that holds the
// row's end loads the 16 bytes that END there (the leading elements of that vector
// belong to the lane before and are not counted), and lanes past the end load the
// same vector and count nothing.  Every load stays inside the row, without a
// branch.  Vector loads and stores at 4- or 8-byte alignment are what global memory
// accesses on this GPU allow.
//
// RG == 3 ("thin"): a dense row is shorter than 16 bytes (K < Vec<T>::N reals; `nvec`
// carries K again).  The row is the first K elements of one vector, loaded element by
// element (the elements past K repeat element K - 1: no branch, no access outside
// the row) and counted by the first lane of the group only; the group's other lanes
// load the same addresses and count nothing.  Runs the 4-lane shape.
template <typename T, int VPL> struct OddLanes {
    uint32_t off[VPL];             // byte offset within a row of this lane's vector v
    bool keep[VPL][Vec<T>::N];     // the elements of it that are this lane's
    bool all[VPL];                 // every element is
    uint32_t stride;               // reals from one dense row to the next (>= K: the kernel may
                                   // be working on a slice of K columns of wider rows)
    bool accum;                    // SDDMM adds to C instead of overwriting it (every slice of
                                   // wide rows but the first)
};
template <typename T, int VPL, int RG> struct Odd {};
// RG == -1 ("hot"): as RG == 0 but for what the gathers read: the lane that loads a column turns it
// into a distance in units of kHotUnit bytes from a base below both the dense operand and the buffer
// of its hot rows, so that a gather costs the same instructions.  (The base chosen per gather instead
// took three more, and 6 to 10 registers fewer: R-MAT 20, fp64 K = 64, scrambled column numbers, SpMM
// 807 -> 818 us against 806 -> 811 in this form.)
template <typename T, int VPL> struct Odd<T, VPL, -1> {
    uint32_t at, hot_at; // of row 0 of the operand; of "row kHotRow", the buffer's first
};
// RG == 1: where this lane's vectors lie in a row, and which of them are its own; a lane past the row's
// end loads the row's last vector and counts nothing: one select per dot product.  (Lanes switched off
// around each load were a branch and four moves per row: R-MAT 18, fp64 K = 100, SDDMM / SpMM 315 / 338
// -> 304 / 305 us with the scalar base of a 64-lane group; fp32 K = 96 150 / 141 -> 146 / 130; switched
// off once for a whole batch: level, rows of 75 vectors 4 % slower.)
template <typename T, int VPL> struct Odd<T, VPL, 1> {
    uint32_t off[VPL];
    bool on[VPL];
};
template <typename T, int VPL> struct Odd<T, VPL, 2> : OddLanes<T, VPL> {};
template <typename T, int VPL> struct Odd<T, VPL, 3> : OddLanes<T, VPL> {};

template <typename T, int LPR, int VPL, int RG>
__device__ __forceinline__ Odd<T, VPL, RG> odd_lanes(uint32_t sub, uint32_t K, uint32_t stride,
                                                     uint32_t accum)
{
    Odd<T, VPL, RG> o;
    if constexpr (RG >= 2) {
        o.stride = stride;
        o.accum = accum != 0;
    }
    if constexpr (RG == 1) { // `K` carries nvec
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            const uint32_t i = sub + (uint32_t)v * LPR;
            o.on[v] = i < K;
            o.off[v] = (i < K ? i : K - 1) * 16;
        }
    }
    if constexpr (RG == 2) {
        const uint32_t bytes = K * (uint32_t)sizeof(T); // >= 16: see pick_shape
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            const uint32_t first = (sub + (uint32_t)v * LPR) * 16;
            const uint32_t start = first < bytes - 16 ? first : bytes - 16;
            o.off[v] = start;
            o.all[v] = start == first;
#pragma unroll
            for (int i = 0; i < Vec<T>::N; ++i)
                o.keep[v][i] = start + (uint32_t)i * sizeof(T) >= first;
        }
    } else if constexpr (RG == 3) {
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            o.off[v] = 0;
            o.all[v] = false;
#pragma unroll
            for (int i = 0; i < Vec<T>::N; ++i)
                o.keep[v][i] = v == 0 && sub == 0 && (uint32_t)i < K;
        }
    }
    return o;
}

// What gather_row takes of a column.
template <typename T, int LPR, int VPL, int RG>
__device__ __forceinline__ uint32_t row_ref(uint32_t c, const Odd<T, VPL, RG> &odd)
{
    if constexpr (RG == -1)
        return c * (LPR * VPL * 16 / kHotUnit) + ((c & kHotRow) ? odd.hot_at : odd.at);
    else
        return c;
}

template <typename T, int RG>
__device__ __forceinline__ const char *odd_row(const T *base, uint32_t row, uint32_t stride)
{
    static_assert(RG >= 2, "rows at element alignment, `stride` reals apart");
    return reinterpret_cast<const char *>(base) + (uint64_t)row * ((uint64_t)stride * sizeof(T));
}

// Vector v of the row at r as this lane loads it in the RG >= 2 variants (NT: a
// row that is read once).
template <typename T, int RG, int VPL, bool NT = false>
__device__ __forceinline__ typename Vec<T>::type odd_load(const char *r, int v, uint32_t K,
                                                          const Odd<T, VPL, RG> &odd)
{
    if constexpr (RG == 3) {
        typename Vec<T>::type out{};
        const T *e = reinterpret_cast<const T *>(r);
#pragma unroll
        for (int i = 0; i + 1 < Vec<T>::N; ++i) // K <= N - 1
            out[i] = e[(uint32_t)i < K ? (uint32_t)i : K - 1];
        return out;
    } else if constexpr (NT) {
        return loose_load_nt<T>(r + odd.off[v]);
    } else {
        return loose_load<T>(r + odd.off[v]);
    }
}

// out[v] = this lane's vectors of dense row `row`.  RG >= 2 loads every element of
// them; what is not the lane's to count is left out by the caller (SDDMM: in the
// dot product; SpMM: at the store).
template <typename T, int LPR, int VPL, int RG>
__device__ __forceinline__ void gather_row(typename Vec<T>::type (&out)[VPL], const T *base,
                                           uint32_t row, uint32_t sub, uint32_t nvec,
                                           const Odd<T, VPL, RG> &odd)
{
    using V = typename Vec<T>::type;
    // where the row starts, and the lane's vector v in it
    const char *r = reinterpret_cast<const char *>(base);
    if constexpr (RG >= 2)
        r = odd_row<T, RG>(base, row, odd.stride);
    else if constexpr (RG == 1)
        r += (uint64_t)row * (nvec * 16);
    else
        r += (uint64_t)row * (RG == -1 ? kHotUnit : (uint32_t)(LPR * VPL * 16));
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
        // Rows of at most three vectors per lane: a fourth load of their last one would be a request more
        // (60 k rows of 3 to 14 over 600 k columns, fp64 K = 260: SDDMM 3 to 7 % slower).
        if (RG == 1 && VPL == 4 && v == 3 && nvec <= 3 * LPR) {
            out[v] = V{};
            continue;
        }
        if constexpr (RG == 3) {
            out[v] = odd_load<T, RG, VPL>(r, v, nvec, odd);
        } else {
            uint32_t off;
            if constexpr (RG >= 1)
                off = odd.off[v];
            else
                off = (sub + (uint32_t)v * LPR) * 16;
            if constexpr (LPR == 64) // row is uniform: a scalar base, the lane's offset beside it
                out[v] = load_beside<T, RG == 2>(r, off);
            else if constexpr (RG == 2)
                out[v] = loose_load<T>(r + off);
            else
                out[v] = *reinterpret_cast<const V *>(r + off);
        }
    }
}

// The lane's offsets in a row, made here and not outside the loop over batches, where the compiler would
// widen them to 64 bits and not find a gather's scalar base with a 32-bit offset any more.
template <typename T, int LPR, int VPL, int RG>
__device__ __forceinline__ void pin_offsets(uint32_t &sub, Odd<T, VPL, RG> &odd)
{
    if constexpr (LPR == 64) {
        if constexpr (RG == 1 || RG == 2) {
#pragma unroll
            for (int v = 0; v < VPL; ++v)
                asm volatile("" : "+v"(odd.off[v]));
        } else {
            asm volatile("" : "+v"(sub));
        }
    }
}

// a . b over the elements that are this lane's.
template <typename T, int VPL, int RG>
__device__ __forceinline__ T lane_dot(const typename Vec<T>::type (&a)[VPL],
                                      const typename Vec<T>::type (&b)[VPL],
                                      const Odd<T, VPL, RG> &odd)
{
    T dot = (T)0;
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
        const T before = dot;
#pragma unroll
        for (int i = 0; i < Vec<T>::N; ++i) {
            if constexpr (RG >= 2)
                dot += a[v][i] * (odd.keep[v][i] ? b[v][i] : (T)0);
            else
                dot += a[v][i] * b[v][i];
        }
        if constexpr (RG == 1)
            if (VPL == 1 || v > 0) // (rows of more than LPR vectors: every lane has its first)
                dot = odd.on[v] ? dot : before;
    }
    return dot;
}

// Writes y0 + acc (whole rows of Y) or acc (partial-sum slots, read back by
// spmm_fixup right after) to this lane's part of the row at drow: one vector store
// where the whole vector is the lane's, element stores for the lane at the row's end.
template <typename T, int VPL>
__device__ __forceinline__ void odd_store(char *drow, bool whole,
                                          const typename Vec<T>::type (&y0)[VPL],
                                          const typename Vec<T>::type (&acc)[VPL],
                                          const OddLanes<T, VPL> &odd)
{
    using V = typename Vec<T>::type;
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
        const V r = y0[v] + acc[v]; // y0 is zero for a slot
        if (odd.all[v]) {
            if (whole)
                loose_store_nt<T>(r, drow + odd.off[v]);
            else
                loose_store<T>(r, drow + odd.off[v]);
        } else {
            T *d = reinterpret_cast<T *>(drow + odd.off[v]);
#pragma unroll
            for (int i = 0; i < Vec<T>::N; ++i)
                if (odd.keep[v][i])
                    d[i] = r[i];
        }
    }
}

// ---------------------------------------------------------------- SDDMM ----
// One batch of NB entries from p0.  MK ("masked"): only the first n (1 <= n <= NB)
// exist; the others repeat entry n - 1 (loads without branches, from addresses
// that are being read anyway) and store nothing, so that a tail of any length
// costs one round of gathers.
//
// FZ ("fused"): the gathered B rows also feed the SpMM of the same pattern,
// acc += w_u * B[c_u,:] in kernel order, with w_u = S.vv (FZ == 1) or the SDDMM
// result just computed (FZ == 2); the weight of entry u is broadcast from the lane
// that stores it.
//
// PRE: the column indices of the batch were loaded ahead (lane u of the group holds that
// of entry u in ex.first[0], or, where the group has fewer lanes than the batch has entries,
// those of entries u and LPR + u in ex.first[0] and ex.first[1]); past the segment's end they
// repeat its last column.
//
// NG <= NB: every lane group of the wavefront has at most NG entries in this batch, so
// only the first NG gathers are issued.
template <typename T, int LPR, int VPL, int NB, int RG, bool MK, int FZ, bool PRE, int NG>
__device__ __forceinline__ void
sddmm_batch_one(const typename Vec<T>::type (&a)[VPL], typename Vec<T>::type (&acc)[VPL],
            const uint32_t *__restrict__ col, const uint32_t *__restrict__ perm,
            const T *__restrict__ sval, const T *__restrict__ B, T *__restrict__ C, uint32_t p0,
            uint32_t n, uint32_t sub, uint32_t nvec,
            const Odd<T, VPL, RG> &odd, const Ahead &ex)
{
    using V = typename Vec<T>::type;
    static_assert(NB <= LPR, "batch must fit the lane group");

    // Lane u of the group fetches the column of entry u; the writer lanes fetch
    // what they need for the store.  These head the dependency chain.
    uint32_t e = sub & (NB - 1);
    if (MK)
        e = e < n ? e : n - 1;
    const uint32_t cme = row_ref<T, LPR>(PRE ? ex.first[0] : nt_load(col + p0 + e), odd);
    const uint32_t uo = entry_of<LPR, NB>(sub);
    const bool writer = is_writer<LPR, NB>(sub) && (!MK || uo < n);
    T sv = (T)0;
    uint32_t dst = p0 + uo + ex.shift;
    if (writer) {
        sv = nt_load(sval + p0 + uo);
        if (perm)
            dst = nt_load(perm + p0 + uo);
    }

    static_assert(NG >= 1 && NG <= NB && (MK || NG == NB), "NG < NB only in a masked batch");
    V b[NG][VPL];
    uint32_t at = sub;
    Odd<T, VPL, RG> row = odd;
    pin_offsets<T, LPR, VPL, RG>(at, row);
    const Bcast<LPR> bcast;
    // The second half of a wide batch makes its addresses when the first half's loads are under way:
    // half the address registers (with the lane in the permutes' offset 100 -> 94 of them in SDDMM and
    // 138 -> 122 in the one-pass kernel at fp64 K = 64: a wavefront more per SIMD).
    uint32_t c[NG];
#pragma unroll
    for (int u = 0; u < NG; ++u)
        c[u] = bcast(cme, u);
#pragma unroll
    for (int u = 0; u < NG; ++u) {
        gather_row<T, LPR, VPL, RG>(b[u], B, c[u], at, nvec, row);
        if (LPR < 64 && NB >= 8 && u + 1 == NG / 2)
            __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0); // all gathers in flight before the first use

    T part[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        if (u < NG)
            part[u] = lane_dot<T, VPL, RG>(a, b[u], odd);
        else
            part[u] = (T)0;
    }
    group_reduce<T, LPR, NB>(part, sub);
    T result = part[0] * sv;
    // Results in the caller's order: when that is the kernel order the stores of a
    // batch fill whole lines and stream out; when it is not they are scattered, and
    // plain stores let the L2 merge neighbours into lines before writing back.
    if (writer) {
        const bool staged = dst >= ex.stage_from;
        T *out = staged ? static_cast<T *>(ex.stage) + (dst - ex.stage_from) : C + dst;
        if constexpr (RG >= 2) {
            if (odd.accum)
                result += *out;
        }
        if (perm && !ex.stream_c && !staged)
            *out = result;
        else
            nt_store(result, out);
    }
    if constexpr (FZ != 0) {
        const T mine = FZ == 2 ? result : sv; // valid on the writer lanes
#pragma unroll
        for (int u = 0; u < NG; ++u) {
            const bool on = !MK || (uint32_t)u < n;
            const T w = on ? bcast(mine, writer_lane<LPR, NB>(u)) : (T)0;
#pragma unroll
            for (int v = 0; v < VPL; ++v)
                acc[v] += (on ? b[u][v] : V{}) * w;
        }
    }
}

template <typename T, int LPR, int VPL, int NB, int RG, bool MK, int FZ, bool PRE>
__device__ __forceinline__ void
sddmm_batch_rounds(const typename Vec<T>::type (&a)[VPL], typename Vec<T>::type (&acc)[VPL],
            const uint32_t *__restrict__ col, const uint32_t *__restrict__ perm,
            const T *__restrict__ sval, const T *__restrict__ B, T *__restrict__ C, uint32_t p0,
            uint32_t n, uint32_t sub, uint32_t nvec,
            const Odd<T, VPL, RG> &odd, const Ahead &ex)
{
    using V = typename Vec<T>::type;
    // A group of LPR lanes reduces at most LPR entries at a time: the NB entries of
    // the batch are R rounds of G, all gathered before the first round is reduced, so
    // that narrow rows (LPR = 4, 8) keep as many gathers in flight as wide ones.
    constexpr int G = NB < LPR ? NB : LPR;
    constexpr int R = NB / G;
    static_assert(R * G == NB, "a batch is a whole number of rounds");
    static_assert(!PRE || R <= 2, "at most two rounds of columns are loaded ahead");

    // Lane u of the group fetches the column of entry u of each round; the writer
    // lanes fetch what they need for the store.  These head the dependency chain.
    const uint32_t uo = entry_of<LPR, G>(sub);
    const bool wlane = is_writer<LPR, G>(sub);
    uint32_t cme[R], dst[R];
    T sv[R];
    bool writer[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        uint32_t e = (uint32_t)r * G + (sub & (G - 1));
        if (MK)
            e = e < n ? e : n - 1;
        cme[r] = row_ref<T, LPR>(PRE ? ex.first[r & 1] : nt_load(col + p0 + e), odd);
        const uint32_t mine = (uint32_t)r * G + uo;
        writer[r] = wlane && (!MK || mine < n);
        sv[r] = (T)0;
        dst[r] = p0 + mine + ex.shift;
        if (writer[r]) {
            sv[r] = nt_load(sval + p0 + mine);
            if (perm)
                dst[r] = nt_load(perm + p0 + mine);
        }
    }

    V b[NB][VPL];
    const Bcast<LPR> bcast;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const uint32_t c = bcast(cme[j / G], j % G);
        gather_row<T, LPR, VPL, RG>(b[j], B, c, sub, nvec, odd);
    }
    __builtin_amdgcn_sched_barrier(0); // all gathers in flight before the first use

#pragma unroll
    for (int r = 0; r < R; ++r) {
        T part[G];
#pragma unroll
        for (int u = 0; u < G; ++u) {
            part[u] = lane_dot<T, VPL, RG>(a, b[r * G + u], odd);
        }
        group_reduce<T, LPR, G>(part, sub);
        T result = part[0] * sv[r];
        // Results in the caller's order: when that is the kernel order the stores of a
        // batch fill whole lines and stream out; when it is not they are scattered, and
        // plain stores let the L2 merge neighbours into lines before writing back.
        if (writer[r]) {
            const bool staged = dst[r] >= ex.stage_from;
            T *out = staged ? static_cast<T *>(ex.stage) + (dst[r] - ex.stage_from) : C + dst[r];
            if constexpr (RG >= 2) {
                if (odd.accum)
                    result += *out;
            }
            if (perm && !ex.stream_c && !staged)
                *out = result;
            else
                nt_store(result, out);
        }
        if constexpr (FZ != 0) {
            const T mine = FZ == 2 ? result : sv[r]; // valid on the writer lanes
#pragma unroll
            for (int u = 0; u < G; ++u) {
                const bool on = !MK || (uint32_t)(r * G + u) < n;
                const T w = on ? bcast(mine, writer_lane<LPR, G>(u)) : (T)0;
#pragma unroll
                for (int v = 0; v < VPL; ++v)
                    acc[v] += (on ? b[r * G + u][v] : V{}) * w;
            }
        }
    }
}

// A batch of NB entries: one round when the lane group can reduce them at once,
// several otherwise.  The two forms are kept apart on purpose: written as the
// R = 1 case of the rounds form, the single round compiles to 24 more VGPRs
// (100 -> 124 in the wide launch, 62 -> 74 and two wavefronts per SIMD fewer in
// the short one), which cost the 5-entry rows of a stencil 20 %.
template <typename T, int LPR, int VPL, int NB, int RG, bool MK, int FZ, bool PRE = false,
          int NG = NB>
__device__ __forceinline__ void
sddmm_batch(const typename Vec<T>::type (&a)[VPL], typename Vec<T>::type (&acc)[VPL],
            const uint32_t *__restrict__ col, const uint32_t *__restrict__ perm,
            const T *__restrict__ sval, const T *__restrict__ B, T *__restrict__ C, uint32_t p0,
            uint32_t n, uint32_t sub, uint32_t nvec,
            const Odd<T, VPL, RG> &odd, const Ahead &ex)
{
    if constexpr (NB <= LPR)
        sddmm_batch_one<T, LPR, VPL, NB, RG, MK, FZ, PRE, NG>(a, acc, col, perm, sval, B, C, p0, n,
                                                              sub, nvec, odd, ex);
    else
        sddmm_batch_rounds<T, LPR, VPL, NB, RG, MK, FZ, PRE>(a, acc, col, perm, sval, B, C, p0, n,
                                                             sub, nvec, odd, ex);
}

// n consecutive entries from p.  WIDE: full batches of UB, then one masked batch
// of the smallest size in {4, 8, 16} that holds the rest.  !WIDE (segments known
// to be short, run at twice the occupancy): masked batches of UB throughout, the
// first of them on the column indices in `ex.first` (loaded ahead, beside the segment's
// descriptor, from the plan's table of first columns: kFirstCols per short segment).
template <typename T, int LPR, int VPL, int UB, int RG, bool WIDE, int FZ>
__device__ __forceinline__ void
sddmm_walk(const typename Vec<T>::type (&a)[VPL], typename Vec<T>::type (&acc)[VPL],
           const uint32_t *__restrict__ col, const uint32_t *__restrict__ perm,
           const T *__restrict__ sval, const T *__restrict__ B, T *__restrict__ C, uint32_t p,
           uint32_t n, uint32_t sub, uint32_t nvec,
            const Odd<T, VPL, RG> &odd, const Ahead &ex)
{
    if constexpr (WIDE) {
        for (; n >= UB; n -= UB, p += UB)
            sddmm_batch<T, LPR, VPL, UB, RG, false, FZ>(a, acc, col, perm, sval, B, C, p, UB, sub, nvec, odd, ex);
        if (n == 0)
            return;
        if constexpr (UB > 8) {
            if (n > 8) {
                sddmm_batch<T, LPR, VPL, UB, RG, true, FZ>(a, acc, col, perm, sval, B, C, p, n, sub, nvec, odd, ex);
                return;
            }
        }
        if constexpr (UB > 4) {
            if (n > 4) {
                sddmm_batch<T, LPR, VPL, 8, RG, true, FZ>(a, acc, col, perm, sval, B, C, p, n, sub, nvec, odd, ex);
                return;
            }
        }
        sddmm_batch<T, LPR, VPL, (UB < 4 ? UB : 4), RG, true, FZ>(a, acc, col, perm, sval, B, C, p, n, sub, nvec, odd, ex);
    } else {
        static_assert(WIDE || UB <= (int)kFirstCols, "the first batch runs on the columns loaded ahead");
        {
            // Segments arrive sorted by length, so the groups of a wavefront mostly hold
            // the same number of entries: the batch is cut to what the longest of them
            // needs (a condition uniform over the wavefront), which spares the memory
            // pipeline the repeated gathers of a full masked batch.
            const uint32_t m = n < (uint32_t)UB ? n : (uint32_t)UB;
            if constexpr (UB == 8 && LPR >= 8) {
                if (__ballot(m > 2) == 0)
                    sddmm_batch<T, LPR, VPL, 2, RG, true, FZ, true>(a, acc, col, perm, sval, B, C, p, m, sub, nvec, odd, ex);
                else if (__ballot(m > 4) == 0)
                    sddmm_batch<T, LPR, VPL, 4, RG, true, FZ, true>(a, acc, col, perm, sval, B, C, p, m, sub, nvec, odd, ex);
                else if (__ballot(m > 5) == 0)
                    sddmm_batch<T, LPR, VPL, 8, RG, true, FZ, true, 5>(a, acc, col, perm, sval, B, C, p, m, sub, nvec, odd, ex);
                else
                    sddmm_batch<T, LPR, VPL, 8, RG, true, FZ, true>(a, acc, col, perm, sval, B, C, p, m, sub, nvec, odd, ex);
            } else {
                sddmm_batch<T, LPR, VPL, UB, RG, true, FZ, true>(a, acc, col, perm, sval, B, C, p, m, sub, nvec, odd, ex);
            }
            n -= m;
            p += m;
        }
#pragma nounroll
        while (n > 0) {
            const uint32_t m = n < (uint32_t)UB ? n : (uint32_t)UB;
            sddmm_batch<T, LPR, VPL, UB, RG, true, FZ>(a, acc, col, perm, sval, B, C, p, m, sub, nvec, odd, ex);
            n -= m;
            p += m;
        }
    }
}

// FZ != 0: also Y[row,:] += sum of the segment's w_u * B[c_u,:] (partial-sum slot for
// a cut row, as in spmm_seg_kernel); Y and partial are unused otherwise.
template <typename T, int LPR, int VPL, int UB, int RG, bool WIDE, int FZ>
__global__ void __launch_bounds__(kBlock, 1)
sddmm_seg_kernel(const Seg *__restrict__ segs, uint32_t nseg, uint32_t nq, uint32_t rot,
                 const uint32_t *__restrict__ col, const uint32_t *__restrict__ perm,
                 const T *__restrict__ sval, const T *__restrict__ A, const T *__restrict__ B,
                 T *__restrict__ C, T *__restrict__ Y, T *__restrict__ partial, uint32_t nvec,
                 uint32_t stride, uint32_t accum, const uint32_t *__restrict__ first_cols,
                 uint32_t flags, T *__restrict__ stage, uint32_t stage_from, uint32_t ref_at, uint32_t hot_at)
{
    static_assert(UB <= 16 && LPR <= 64, "at most 16 entries in flight per lane");
    using V = typename Vec<T>::type;
    const uint32_t sub = threadIdx.x & (LPR - 1);
    const uint64_t sid = seg_index<64 / LPR>(nq, rot);
    if (sid >= nseg)
        return;
    Ahead ex = load_first_cols<LPR, WIDE>(first_cols, sid, sub);
    ex.stream_c = (flags & kStoreStream) != 0;
    ex.stage = stage;
    ex.stage_from = stage_from;
    u32x4 sg = nt_load(reinterpret_cast<const u32x4 *>(segs) + sid); // row, start, len, slot
    if (sg[2] == 0)
        return;
    if constexpr (LPR == 64)
        uniform(sg);
    if (flags & kStoreSegBase) { // one position per segment instead of one per entry
        ex.shift = nt_load(perm + sg[1]) - sg[1];
        perm = nullptr;
    }

    Odd<T, VPL, RG> odd = odd_lanes<T, LPR, VPL, RG>(sub, nvec, stride, accum);
    if constexpr (RG == -1)
        odd.at = ref_at, odd.hot_at = hot_at;
    V a[VPL], acc[VPL];
    if constexpr (RG >= 2) {
        const char *arow = odd_row<T, RG>(A, sg[0], stride);
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            a[v] = odd_load<T, RG, VPL, true>(arow, v, nvec, odd);
#pragma unroll
            for (int i = 0; i < Vec<T>::N; ++i)
                a[v][i] = odd.keep[v][i] ? a[v][i] : (T)0;
            acc[v] = V{};
        }
    } else {
        const V *arow = row_ptr<T, LPR, VPL, RG>(A, sg[0], sub, nvec);
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            a[v] = lane_on<LPR, RG>(sub, v, nvec) ? nt_load(arow + v * LPR) : V{};
            acc[v] = V{};
        }
    }
    sddmm_walk<T, LPR, VPL, UB, RG, WIDE, FZ>(a, acc, col, perm, sval, B, C, sg[1], sg[2], sub,
                                              nvec, odd, ex);
    if constexpr (FZ != 0 && RG >= 2) {
        const bool whole = sg[3] == kWholeRow;
        char *drow = const_cast<char *>(whole ? odd_row<T, RG>(Y, sg[0], stride)
                                              : odd_row<T, RG>(partial, sg[3], stride));
        V y0[VPL];
#pragma unroll
        for (int v = 0; v < VPL; ++v)
            y0[v] = whole ? odd_load<T, RG, VPL, true>(drow, v, nvec, odd) : V{};
        odd_store<T, VPL>(drow, whole, y0, acc, odd);
    } else if constexpr (FZ != 0) {
        const bool whole = sg[3] == kWholeRow;
        V *dst = const_cast<V *>(whole ? row_ptr<T, LPR, VPL, RG>(Y, sg[0], sub, nvec)
                                       : row_ptr<T, LPR, VPL, RG>(partial, sg[3], sub, nvec));
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            if (!lane_on<LPR, RG>(sub, v, nvec))
                continue;
            if (whole)
                nt_store(nt_load(dst + v * LPR) + acc[v], dst + v * LPR);
            else
                dst[v * LPR] = acc[v]; // read back by spmm_fixup right after
        }
    }
}

// ----------------------------------------------------------------- SpMM ----
// Column of entry j < kFirstCols of a short segment out of the indices loaded ahead:
// lane u of the group holds that of entry u in FC[0] (groups of 4 lanes: of entries u
// and 4 + u in FC[0] and FC[1]).
template <int LPR>
__device__ __forceinline__ uint32_t first_col(const Bcast<LPR> &bcast, const uint32_t (&FC)[2], uint32_t j)
{
    if constexpr (LPR >= (int)kFirstCols)
        return bcast(FC[0], (int)j);
    else
    {
        // Values, not elements: a choice between two array elements is a choice of address, for
        // which the compiler moves the array to LDS and reads the dispatch packet to find the
        // thread's place in it (9 us per launch).
        const uint32_t a = FC[0], b = FC[1];
        return bcast((j & LPR) ? b : a, (int)(j & (LPR - 1)));
    }
}

// MK: only the first n of the NB entries exist; the others repeat the loads of
// entry n - 1 and add zero times zero.
// PRE: the batch is entries off .. off + NB - 1 of a short segment, off + NB <=
// kFirstCols, and takes its column indices from `ex.first` (first_col).
template <typename T, int LPR, int VPL, int NB, int RG, bool MK, bool PRE>
__device__ __forceinline__ void
spmm_batch_one(typename Vec<T>::type (&acc)[VPL], const uint32_t *__restrict__ col,
           const T *__restrict__ sval, const T *__restrict__ X, uint32_t p0, uint32_t n,
           uint32_t sub, uint32_t nvec,
            const Odd<T, VPL, RG> &odd, const Ahead &ex, uint32_t off)
{
    using V = typename Vec<T>::type;
    static_assert(NB <= LPR, "batch must fit the lane group");
    uint32_t e = sub & (NB - 1);
    if (MK)
        e = e < n ? e : n - 1;
    uint32_t cme = 0;
    if constexpr (!PRE)
        cme = row_ref<T, LPR>(nt_load(col + p0 + e), odd);
    const T vme = nt_load(sval + p0 + e);

    V x[NB][VPL];
    T av[NB];
    uint32_t at = sub;
    Odd<T, VPL, RG> row = odd;
    pin_offsets<T, LPR, VPL, RG>(at, row);
    const Bcast<LPR> bcast;
    uint32_t c[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u)
        c[u] = PRE ? first_col<LPR>(bcast, ex.first, off + u) : bcast(cme, u);
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        gather_row<T, LPR, VPL, RG>(x[u], X, c[u], at, nvec, row);
        if (LPR < 64 && NB >= 8 && u + 1 == NB / 2)
            __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0); // all gathers in flight before the first use
    // Entries are added in kernel order.
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        // The weights four entries ahead of their use, four at a time: all of them at once held 32
        // registers beside the gathers at fp64 (136 -> 98 with the rest: 4 wavefronts per SIMD, not 3;
        // R-MAT 18, K = 64: 188 -> 174 us).
        if (u % 4 == 0)
#pragma unroll
            for (int w = u ? u + 4 : 0; w < u + 8 && w < NB; ++w)
                av[w] = bcast(vme, w);
        const bool on = !MK || (uint32_t)u < n;
        const T a = on ? av[u] : (T)0;
#pragma unroll
        for (int v = 0; v < VPL; ++v)
            acc[v] += (on ? x[u][v] : V{}) * a;
    }
}

template <typename T, int LPR, int VPL, int NB, int RG, bool MK>
__device__ __forceinline__ void
spmm_batch_rounds(typename Vec<T>::type (&acc)[VPL], const uint32_t *__restrict__ col,
           const T *__restrict__ sval, const T *__restrict__ X, uint32_t p0, uint32_t n,
           uint32_t sub, uint32_t nvec,
            const Odd<T, VPL, RG> &odd)
{
    using V = typename Vec<T>::type;
    // Lane u of the group fetches column and value of entry u of each of the R rounds
    // of G <= LPR entries (see sddmm_batch).
    constexpr int G = NB < LPR ? NB : LPR;
    constexpr int R = NB / G;
    static_assert(R * G == NB, "a batch is a whole number of rounds");
    uint32_t cme[R];
    T vme[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        uint32_t e = (uint32_t)r * G + (sub & (G - 1));
        if (MK)
            e = e < n ? e : n - 1;
        cme[r] = row_ref<T, LPR>(nt_load(col + p0 + e), odd);
        vme[r] = nt_load(sval + p0 + e);
    }

    V x[NB][VPL];
    T av[NB];
    const Bcast<LPR> bcast;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const uint32_t c = bcast(cme[j / G], j % G);
        av[j] = bcast(vme[j / G], j % G);
        gather_row<T, LPR, VPL, RG>(x[j], X, c, sub, nvec, odd);
    }
    __builtin_amdgcn_sched_barrier(0); // all gathers in flight before the first use
    // Entries are added in kernel order.
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const bool on = !MK || (uint32_t)j < n;
        const T w = on ? av[j] : (T)0;
#pragma unroll
        for (int v = 0; v < VPL; ++v)
            acc[v] += (on ? x[j][v] : V{}) * w;
    }
}

template <typename T, int LPR, int VPL, int NB, int RG, bool MK>
__device__ __forceinline__ void
spmm_batch(typename Vec<T>::type (&acc)[VPL], const uint32_t *__restrict__ col,
           const T *__restrict__ sval, const T *__restrict__ X, uint32_t p0, uint32_t n,
           uint32_t sub, uint32_t nvec,
            const Odd<T, VPL, RG> &odd)
{
    const Ahead none{};
    if constexpr (NB <= LPR)
        spmm_batch_one<T, LPR, VPL, NB, RG, MK, false>(acc, col, sval, X, p0, n, sub, nvec, odd,
                                                       none, 0u);
    else
        spmm_batch_rounds<T, LPR, VPL, NB, RG, MK>(acc, col, sval, X, p0, n, sub, nvec, odd);
}

template <typename T, int LPR, int VPL, int UB, int RG, bool WIDE>
__device__ __forceinline__ void
spmm_walk(typename Vec<T>::type (&acc)[VPL], const uint32_t *__restrict__ col,
          const T *__restrict__ sval, const T *__restrict__ X, uint32_t p, uint32_t n,
          uint32_t sub, uint32_t nvec,
            const Odd<T, VPL, RG> &odd, const Ahead &ex)
{
    // Short segments: exact batches of UB, then UB/2 ... 1 as n requires.  Measured
    // against masked batches here (which cost registers, hence occupancy): 3 % faster
    // on 5-entry rows, level elsewhere.  SpMM's short rows are bound by the Y
    // read-modify-write stream, not by rounds of gathers.  The first kFirstCols
    // entries take their column indices from `ex.first`, which was loaded ahead, beside the
    // segment's descriptor.
    if constexpr (!WIDE) {
        static_assert(WIDE || (UB <= 4 && UB <= LPR), "short batches fit the lane group");
        {
            const uint32_t m = n < kFirstCols ? n : kFirstCols;
            uint32_t off = 0;
            for (; off + UB <= m; off += UB)
                spmm_batch_one<T, LPR, VPL, UB, RG, false, true>(acc, col, sval, X, p + off, UB,
                                                                 sub, nvec, odd, ex, off);
            if constexpr (UB > 2)
                if ((m - off) & 2) {
                    spmm_batch_one<T, LPR, VPL, 2, RG, false, true>(acc, col, sval, X, p + off, 2,
                                                                    sub, nvec, odd, ex, off);
                    off += 2;
                }
            if constexpr (UB > 1)
                if ((m - off) & 1)
                    spmm_batch_one<T, LPR, VPL, 1, RG, false, true>(acc, col, sval, X, p + off, 1,
                                                                    sub, nvec, odd, ex, off);
            n -= m;
            p += m;
        }
        for (; n >= UB; n -= UB, p += UB)
            spmm_batch<T, LPR, VPL, UB, RG, false>(acc, col, sval, X, p, UB, sub, nvec, odd);
        if constexpr (UB > 8)
            if (n & 8) {
                spmm_batch<T, LPR, VPL, 8, RG, false>(acc, col, sval, X, p, 8, sub, nvec, odd);
                p += 8;
            }
        if constexpr (UB > 4)
            if (n & 4) {
                spmm_batch<T, LPR, VPL, 4, RG, false>(acc, col, sval, X, p, 4, sub, nvec, odd);
                p += 4;
            }
        if constexpr (UB > 2)
            if (n & 2) {
                spmm_batch<T, LPR, VPL, 2, RG, false>(acc, col, sval, X, p, 2, sub, nvec, odd);
                p += 2;
            }
        if constexpr (UB > 1)
            if (n & 1)
                spmm_batch<T, LPR, VPL, 1, RG, false>(acc, col, sval, X, p, 1, sub, nvec, odd);
    } else {
        for (; n >= UB; n -= UB, p += UB)
            spmm_batch<T, LPR, VPL, UB, RG, false>(acc, col, sval, X, p, UB, sub, nvec, odd);
        if (n == 0)
            return;
        if constexpr (UB > 8) {
            if (n > 8) {
                spmm_batch<T, LPR, VPL, UB, RG, true>(acc, col, sval, X, p, n, sub, nvec, odd);
                return;
            }
        }
        if constexpr (UB > 4) {
            if (n > 4) {
                spmm_batch<T, LPR, VPL, 8, RG, true>(acc, col, sval, X, p, n, sub, nvec, odd);
                return;
            }
        }
        spmm_batch<T, LPR, VPL, (UB < 4 ? UB : 4), RG, true>(acc, col, sval, X, p, n, sub, nvec, odd);
    }
}

template <typename T, int LPR, int VPL, int UB, int RG, bool WIDE>
__global__ void __launch_bounds__(kBlock)
spmm_seg_kernel(const Seg *__restrict__ segs, uint32_t nseg, uint32_t nq, uint32_t rot,
                const uint32_t *__restrict__ col, const T *__restrict__ sval,
                const T *__restrict__ X, T *__restrict__ Y, T *__restrict__ partial,
                uint32_t nvec, uint32_t stride, uint32_t pstride,
                const uint32_t *__restrict__ first_cols, uint32_t ref_at, uint32_t hot_at)
{
    static_assert(UB <= 16 && LPR <= 64, "at most 16 entries in flight per lane");
    using V = typename Vec<T>::type;
    const uint32_t sub = threadIdx.x & (LPR - 1);
    const uint64_t sid = seg_index<64 / LPR>(nq, rot);
    if (sid >= nseg)
        return;
    Ahead ex = load_first_cols<LPR, WIDE>(first_cols, sid, sub);
    u32x4 sg = nt_load(reinterpret_cast<const u32x4 *>(segs) + sid); // row, start, len, slot
    if (sg[2] == 0)
        return;
    if constexpr (LPR == 64)
        uniform(sg);
    const bool whole = sg[3] == kWholeRow;
    Odd<T, VPL, RG> odd = odd_lanes<T, LPR, VPL, RG>(sub, nvec, stride, 0u);
    if constexpr (RG == -1)
        odd.at = ref_at, odd.hot_at = hot_at;
    if constexpr (!WIDE) {
        ex.first[0] = row_ref<T, LPR>(ex.first[0], odd);
        ex.first[1] = row_ref<T, LPR>(ex.first[1], odd);
    }

    V acc[VPL], y0[VPL];
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
        acc[v] = V{};
        y0[v] = V{};
    }
    if constexpr (RG >= 2) {
        char *drow = const_cast<char *>(whole ? odd_row<T, RG>(Y, sg[0], stride)
                                              : odd_row<T, RG>(partial, sg[3], pstride));
        if (whole) {
#pragma unroll
            for (int v = 0; v < VPL; ++v)
                y0[v] = odd_load<T, RG, VPL, true>(drow, v, nvec, odd);
        }
        spmm_walk<T, LPR, VPL, UB, RG, WIDE>(acc, col, sval, X, sg[1], sg[2], sub, nvec, odd, ex);
        odd_store<T, VPL>(drow, whole, y0, acc, odd);
    } else {
        V *dst = const_cast<V *>(whole ? row_ptr<T, LPR, VPL, RG>(Y, sg[0], sub, nvec)
                                       : row_ptr<T, LPR, VPL, RG>(partial, sg[3], sub, nvec));
        if (whole) {
#pragma unroll
            for (int v = 0; v < VPL; ++v)
                if (lane_on<LPR, RG>(sub, v, nvec))
                    y0[v] = nt_load(dst + v * LPR);
        }
        spmm_walk<T, LPR, VPL, UB, RG, WIDE>(acc, col, sval, X, sg[1], sg[2], sub, nvec, odd, ex);
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            if (!lane_on<LPR, RG>(sub, v, nvec))
                continue;
            if (whole)
                nt_store(y0[v] + acc[v], dst + v * LPR);
            else
                dst[v * LPR] = acc[v]; // read back by spmm_fixup right after
        }
    }
}

// Y[row,:] += the partial sums of a cut row.  A row's slots are cut into `parts` runs; `lanes`
// threads sum a run each (four loads in flight, in slot order, one 16-byte unit of the row per
// thread where rows are whole units, else one real), the runs are added in pairs through LDS.
// lanes and parts are powers of two, lanes * parts <= kBlock; the other threads of the block
// take further rows.  A row of Y is yunits units, of which `units` are summed from Y on.
// Few rows with many slots (the hubs of a small pattern) are a chain of loads each: R-MAT 13,
// 16-entry segments, fp32 K = 16: SpMM 11.1 us with one run per row, 7.4 with runs.  Rows that fill
// the chip are bound by the slots' bytes and take one run each, also where they have many: SpMM of
// 30,000 rows of 125 slots, fp32 K = 20, 431 us in runs and 422 without, 20,000 of 100, fp64 K = 100,
// 1941 and 1944, 4,500 of 250, fp32 K = 256, 2320 and 2340; R-MAT 18 and 20 are 0.2 % faster without.
template <typename T, typename U>
__global__ void __launch_bounds__(kBlock)
spmm_fixup_kernel(const SplitRow *__restrict__ splits, uint32_t nsplit, const U *__restrict__ partial,
                  U *__restrict__ Y, uint32_t units, uint32_t yunits, uint32_t lanes, uint32_t parts)
{
    __shared__ typename Vec<T>::type run[kBlock];
    U *sums = reinterpret_cast<U *>(run);
    const uint32_t per_row = lanes * parts;
    const uint32_t idx = blockIdx.x * (kBlock / per_row) + threadIdx.x / per_row;
    const uint32_t part = threadIdx.x % per_row / lanes;
    SplitRow sr{};
    if (idx < nsplit)
        sr = splits[idx];
    const uint32_t len = (sr.nslots + parts - 1) / parts;
    const uint32_t q0 = part * len < sr.nslots ? part * len : sr.nslots;
    const uint32_t q1 = q0 + len < sr.nslots ? q0 + len : sr.nslots;
    for (uint32_t j0 = 0; j0 < units; j0 += lanes) { // the same trips for every thread
        const uint32_t j = j0 + threadIdx.x % lanes;
        const bool on = j < units && idx < nsplit;
        U s{}, y{};
        if (on) {
            if (part == 0)
                y = Y[(size_t)sr.row * yunits + j];
            const U *p = partial + (size_t)sr.first_slot * units + j;
            uint32_t q = q0;
            for (; q + 4 <= q1; q += 4) {
                const U v0 = p[(size_t)(q + 0) * units], v1 = p[(size_t)(q + 1) * units];
                const U v2 = p[(size_t)(q + 2) * units], v3 = p[(size_t)(q + 3) * units];
                s = (((s + v0) + v1) + v2) + v3;
            }
            for (; q < q1; ++q)
                s += p[(size_t)q * units];
        }
        if (parts > 1) {
            sums[threadIdx.x] = s;
            __syncthreads();
            for (uint32_t step = parts / 2; step; step /= 2) { // runs i and i + step, in pairs
                if (part < step)
                    sums[threadIdx.x] = s += sums[threadIdx.x + step * lanes];
                __syncthreads();
            }
        }
        if (on && part == 0)
            Y[(size_t)sr.row * yunits + j] = y + s;
    }
}

// ------------------------------------------------- row tiles x column blocks ----
// Long rows over columns that are not skewed (a hypergraph's incidence matrix: 1024 entries
// per row, uniform over 500 k columns; 512-byte dense rows): every entry gathers a dense row
// that no cache holds unless the columns are visited block by block, and cutting a row at
// every block boundary costs its A row (SDDMM) or its Y row (SpMM) again per piece.  Here a
// workgroup keeps a TILE of rows in LDS for a whole sweep over the column blocks: kSweepRowBytes
// of A rows (SDDMM, read-only) or of Y accumulators (SpMM), one workgroup per CU, one launch
// per "generation" of as many tiles as the GPU has CUs.  The workgroups of a generation start
// together and meet the same amount of work in every block, so they walk the blocks in step,
// and barriers keep the wavefronts of one workgroup in step too (without them the oldest
// wavefronts run ahead by tens of blocks): at any time one block of dense rows is what an L2
// sees, and the gathers hit.
//
// The plan (build_sweep in plan_device.h) orders a tile's entries by block, inside a block by
// row; ptr[tile * nb + b] .. [.. + 1) is the range of block b.
// SDDMM, where any lane group can take any entry, takes the tile's entries as one stream: batch i of UB
// entries goes to lane group i % G, across the blocks' boundaries, with a barrier per round of G batches.
// (Dealt block by block a round was filled to 6.7 batches of 7 at best, 2.3 of 3 for shorter rows; and with a
// barrier per block instead of per round the wavefronts drift and gathers miss: 2 M rows over 500 k columns, 560 M
// entries, fp32 K = 128: block by block 19.7 ms for the call, as a stream with a barrier per block 19.2,
// per half block 18.3, per round 17.3.  Gathers as byte offsets in 32 bits, three instructions fewer each:
// between 6 % faster, 256- and 1024-byte rows, and 5 % slower here; not kept.)
// SpMM, with a barrier per block (one per batch measured 12 % slower), cuts every block's range into batches
// of its own: lane group g takes the contiguous batches [g per, (g + 1) per), per = ceil(nbat / G).  The sum
// of a row's run of entries is kept in registers and added to the row's sum in LDS, read when the run begins,
// when it ends (a run's sum of its own: carried on from the row's, fp32 rows of up to 1024 were three times as far
// from 64 bits, 4.8e-7 against 1.5e-7; the fp64 step of R-MAT 20 takes 1401 us for it and not 1365, others are level),
// and after every kRunBatches batches of a chunk: a tile may hold tens of thousands of a row's entries in one block.
// A row's entries are contiguous, so a row is shared between lane groups only
// where a boundary between two chunks falls inside it: its first part then ends a chunk (and
// goes to the row's sum by that lane group), the later parts each BEGIN a chunk.  The
// first run of every chunk therefore goes to an edge slot of its lane group instead, and
// after the block's barrier the edge slots are added to their rows in lane-group order, one
// lane group per row (the first of those that hold it); a second barrier ends the block.
// No atomics, one fixed order of additions: the same bits run to run.
// SpMM's loop is bound by the instructions of an entry (with every gather a hit it took 31 ps per entry where
// SDDMM took 23), so whatever an entry does not need is out of it: the edge slots lie behind the sums, where a
// run goes is one index, and entries past a chunk's end are cleared for the whole batch.  (Branches on
// "first run" and "no run yet" and four selects per entry before: 19.25 -> 17.75 ms for those 560 M entries;
// 200 k rows of 30 over 50 k columns 332 -> 274 us, fp64 107 over 40 k 1354 -> 1264.  Rows' sums asked for two
// entries ahead of a run: 17.95, 285 and 1315; a batch's gathers issued before the barriers of its block:
// rows of 30 7 % faster, longer ones 6 to 8 % slower, as are SDDMM's before its own, 2 %: the wavefronts drift.
// Every lane group with rows of its own, without edges or a barrier per block: a tenth faster with every
// gather a hit, and 9 % slower, at 65 % hits and not 88: chance makes the groups drift by half a block.)
constexpr int kSweepBlock = 1024;
constexpr uint32_t kRunBatches = 128; // of 16: no sum goes over more than 2048 terms, as in the segments
constexpr uint32_t kSweepRowBytes = 128u << 10; // of LDS for the tile's rows
constexpr uint32_t kSweepPtrWords = 1028;       // nb + 1 range bounds of a tile, in LDS too
// A lane's 16 bytes of a dense row.  ANY: rows of K reals, at least 16 bytes and at most LPR * 16,
// at element alignment; as in the "odd" variants above, the lane that holds the row's end takes
// the 16 bytes that END there and the lanes past it the same ones, and what is not a lane's to
// count is left out of dot products and stores.  A tile's rows stay LPR * 16 bytes apart in LDS.
// HOT: rows that fill the lanes, and gathers from the operand or from the copy of its hot rows (RG == -1 above:
// `ref` turns a column into a count of kHotUnit bytes from a base below both).
enum SweepRows { kExact, kAny, kHot };
struct HotAt {
    uint32_t at = 0, hot_at = 0;
};
template <typename T, int LPR, int ROWS> struct SweepLane {
    using V = typename Vec<T>::type;
    static constexpr bool ANY = ROWS == kAny;
    uint32_t sub, off = 0, bytes = LPR * 16;
    HotAt hot;
    bool keep[Vec<T>::N], all = true;
    __device__ __forceinline__ SweepLane(uint32_t lane, uint32_t K, HotAt h) : sub(lane), hot(h)
    {
        if constexpr (ANY) {
            bytes = K * (uint32_t)sizeof(T);
            const uint32_t first = sub * 16;
            off = first < bytes - 16 ? first : bytes - 16;
            all = off == first;
#pragma unroll
            for (int i = 0; i < Vec<T>::N; ++i)
                keep[i] = off + (uint32_t)i * sizeof(T) >= first;
        }
    }
    __device__ __forceinline__ const char *at(const T *base, uint32_t row) const
    {
        return reinterpret_cast<const char *>(base) + (uint64_t)row * bytes + off;
    }
    __device__ __forceinline__ V load(const T *base, uint32_t row) const
    {
        if constexpr (ANY)
            return loose_load<T>(at(base, row));
        else
            return reinterpret_cast<const V *>(base)[(uint64_t)row * LPR + sub];
    }
    // what `gather` takes of a column, and the lane's part of that dense row
    __device__ __forceinline__ uint32_t ref(uint32_t c) const
    {
        if constexpr (ROWS == kHot)
            return c * (LPR * 16 / kHotUnit) + ((c & kHotRow) ? hot.hot_at : hot.at);
        else
            return c;
    }
    __device__ __forceinline__ V gather(const T *base, uint32_t r) const
    {
        if constexpr (ROWS == kHot)
            return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(base) + (uint64_t)r * kHotUnit + sub * 16);
        else
            return load(base, r);
    }
    __device__ __forceinline__ V load_once(const T *base, uint32_t row) const
    {
        if constexpr (ANY)
            return loose_load_nt<T>(at(base, row));
        else
            return nt_load(reinterpret_cast<const V *>(base) + (uint64_t)row * LPR + sub);
    }
    __device__ __forceinline__ void store(V v, T *base, uint32_t row) const
    {
        char *to = const_cast<char *>(at(base, row));
        if (!ANY) {
            nt_store(v, reinterpret_cast<V *>(base) + (uint64_t)row * LPR + sub);
        } else if (all) {
            loose_store_nt<T>(v, to);
        } else {
#pragma unroll
            for (int i = 0; i < Vec<T>::N; ++i)
                if (keep[i])
                    reinterpret_cast<T *>(to)[i] = v[i];
        }
    }
    // a . b, a with zeros where nothing is kept
    __device__ __forceinline__ T dot(const V &a, const V &b) const
    {
        T d = a[0] * (ANY && !keep[0] ? (T)0 : b[0]);
#pragma unroll
        for (int i = 1; i < Vec<T>::N; ++i)
            d += a[i] * (ANY && !keep[i] ? (T)0 : b[i]);
        return d;
    }
};

// One batch of a lane group: its entries' columns, local rows and (for the lanes that need
// one) sparse values, asked for one batch ahead.
template <typename T> struct SweepIdx {
    uint32_t n = 0, col = 0, row = 0, pos = 0;
    T val = (T)0;
};

template <typename T, int LPR, int UB, int ROWS>
__global__ void __launch_bounds__(kSweepBlock)
sweep_sddmm_kernel(const uint32_t *__restrict__ ptr, const uint32_t *__restrict__ tile_rows,
                   const uint32_t *__restrict__ col, const uint16_t *__restrict__ lrow,
                   const T *__restrict__ sval, const uint32_t *__restrict__ pos,
                   const T *__restrict__ A, const T *__restrict__ B, T *__restrict__ C, uint32_t nb,
                   uint32_t R, uint32_t tile0, uint32_t K, HotAt hot)
{
    using V = typename Vec<T>::type;
    constexpr uint32_t G = kSweepBlock / LPR;
    static_assert(G * UB <= kSweepRound, "positions may pass the last entry by a round");
    __shared__ V tile_a[kSweepRowBytes / 16];
    const uint32_t tile = tile0 + blockIdx.x;
    const uint32_t grp = threadIdx.x / LPR, sub = threadIdx.x % LPR;
    const SweepLane<T, LPR, ROWS> lane(sub, K, hot);
    for (uint32_t i = threadIdx.x; i < R * LPR; i += kSweepBlock) { // i % LPR == sub
        const uint32_t g = tile_rows[(uint64_t)tile * R + i / LPR];
        V v{};
        if (g != 0xFFFFFFFFu)
            v = lane.load_once(A, g);
        if constexpr (ROWS == kAny) {
#pragma unroll
            for (int j = 0; j < Vec<T>::N; ++j)
                v[j] = lane.keep[j] ? v[j] : (T)0;
        }
        tile_a[i] = v;
    }
    const uint32_t lo = ptr[(uint64_t)tile * nb], hi = ptr[(uint64_t)tile * nb + nb];
    const uint32_t rounds = (hi - lo + G * UB - 1) / (G * UB); // of a batch per lane group
    __syncthreads();
    const uint32_t uo = entry_of<LPR, UB>(sub);
    const bool wlane = is_writer<LPR, UB>(sub);
    auto fetch = [&](uint32_t q) {
        SweepIdx<T> x;
        if (q >= hi)
            return x;
        x.n = hi - q < (uint32_t)UB ? hi - q : (uint32_t)UB;
        uint32_t e = sub & (UB - 1);
        e = e < x.n ? e : x.n - 1;
        x.col = lane.ref(nt_load(col + q + e));
        x.row = nt_load(lrow + q + e);
        x.val = (wlane && uo < x.n) ? nt_load(sval + q + uo) : (T)0;
        if (pos)
            x.pos = (wlane && uo < x.n) ? nt_load(pos + q + uo) : 0u;
        return x;
    };
    uint32_t p = lo + grp * UB;
    SweepIdx<T> cur = fetch(p);
    for (uint32_t r = 0; r < rounds; ++r, p += G * UB) {
        if (r)
            __syncthreads();
        if (p >= hi) // (the last round)
            continue;
        const SweepIdx<T> nxt = fetch(p + G * UB); // the next batch's indices before this one's gathers
        const Bcast<LPR> bcast;
        V bv[UB];
#pragma unroll
        for (int u = 0; u < UB; ++u)
            bv[u] = lane.gather(B, bcast(cur.col, u));
        __builtin_amdgcn_sched_barrier(0); // all gathers in flight before the first use
        T part[UB];
#pragma unroll
        for (int u = 0; u < UB; ++u)
            part[u] = lane.dot(tile_a[bcast(cur.row, u) * LPR + sub], bv[u]);
        group_reduce<T, LPR, UB>(part, sub);
        if (wlane && uo < cur.n) {
            if (pos) // the caller's positions: pieces of lines that this workgroup's next
                     // blocks complete, so plain stores, which the L2 merges
                C[cur.pos] = part[0] * cur.val;
            else
                nt_store(part[0] * cur.val, C + p + uo); // kernel order: whole lines, streaming
        }
        cur = nxt;
    }
}

template <typename T, int LPR, int UB, int ROWS>
__global__ void __launch_bounds__(kSweepBlock)
sweep_spmm_kernel(const uint32_t *__restrict__ ptr, const uint32_t *__restrict__ tile_rows,
                  const uint32_t *__restrict__ col, const uint16_t *__restrict__ lrow,
                  const T *__restrict__ sval, const uint32_t *__restrict__ vpos,
                  const T *__restrict__ X, T *__restrict__ Y, uint32_t nb, uint32_t R, uint32_t tile0,
                  uint32_t K, HotAt hot, const uint32_t *__restrict__ slot, T *__restrict__ partial)
{
    using V = typename Vec<T>::type;
    constexpr uint32_t G = kSweepBlock / LPR;
    constexpr uint32_t kNone = 0xFFFFFFFFu;
    // the tile's sums, and behind them an edge slot per lane group: the sum of its chunk's first run
    __shared__ V tile_y[kSweepRowBytes / 16 + kSweepBlock];
    __shared__ uint32_t edge_row[G];  // and its row (kNone: the chunk is empty)
    __shared__ uint32_t lptr[kSweepPtrWords];
    constexpr uint32_t kEdge = kSweepRowBytes / 16;
    const uint32_t tile = tile0 + blockIdx.x;
    for (uint32_t i = threadIdx.x; i < R * LPR; i += kSweepBlock)
        tile_y[i] = V{};
    for (uint32_t i = threadIdx.x; i < nb + 1; i += kSweepBlock)
        lptr[i] = ptr[(uint64_t)tile * nb + i];
    __syncthreads();
    const uint32_t grp = threadIdx.x / LPR, sub = threadIdx.x % LPR;
    const SweepLane<T, LPR, ROWS> lane(sub, K, hot);
    auto fetch = [&](uint32_t q, uint32_t qhi) {
        SweepIdx<T> x;
        x.n = qhi - q < (uint32_t)UB ? qhi - q : (uint32_t)UB;
        uint32_t e = sub & (UB - 1);
        e = e < x.n ? e : x.n - 1;
        x.col = lane.ref(nt_load(col + q + e));
        x.row = nt_load(lrow + q + e);
        x.val = vpos ? sval[nt_load(vpos + q + e)] : nt_load(sval + q + e);
        if ((sub & (UB - 1)) >= x.n)
            x.val = (T)0;
        return x;
    };
    // this lane group's chunk of block b: ceil(nbat / G) batches each, from lane group 0 on, so
    // that the lane groups with entries are the first ones and those that share a row are
    // neighbours
    auto chunk = [&](uint32_t b, uint32_t &lo, uint32_t &up) {
        const uint32_t s = lptr[b], e = lptr[b + 1];
        const uint32_t nbat = (e - s + UB - 1) / UB;
        const uint32_t per = (nbat + G - 1) / G;
        const uint64_t first = (uint64_t)grp * per, last = first + per;
        lo = first < nbat ? s + (uint32_t)first * UB : e;
        up = last < nbat ? s + (uint32_t)last * UB : e;
    };
    uint32_t p, hi;
    chunk(0, p, hi);
    SweepIdx<T> cur;
    if (p < hi)
        cur = fetch(p, hi);
    for (uint32_t b = 0; b < nb; ++b) {
        uint32_t p_nb = 0, hi_nb = 0;
        if (b + 1 < nb)
            chunk(b + 1, p_nb, hi_nb);
        const bool had = p < hi;
        const Bcast<LPR> head;
        uint32_t row = had ? head.entry(cur.row, 0) : kNone;
        if (sub == 0)
            edge_row[grp] = row;
        // the run that is being summed, and where its sum goes: the chunk's first to the edge slot
        V acc{}, base{};
        uint32_t to = kEdge + threadIdx.x, batch = 0;
        while (p < hi) {
            const uint32_t np = p + UB;
            SweepIdx<T> nxt;
            if (np < hi)
                nxt = fetch(np, hi);
            else if (p_nb < hi_nb)
                nxt = fetch(p_nb, hi_nb);
            const Bcast<LPR> bcast;
            V xv[UB];
#pragma unroll
            for (int u = 0; u < UB; ++u)
                xv[u] = lane.gather(X, bcast.entry(cur.col, u));
            __builtin_amdgcn_sched_barrier(0);
            // where a row begins: lane u of a group holds entry u and sees entry u - 1 (lane 0 the row
            // that is being summed); the wavefront steps aside only where one of its groups needs it.
            // (A broadcast of the row and a comparison per entry instead: 128 registers and spills of 20
            // bytes against 112 and none; 300 k x 100 k, fp64 K = 128 SpMM 2432 -> 2284 us, 512-byte rows
            // level.  A barrier per batch, as in SDDMM, cost 12 %: the groups' runs differ.)
            const uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp(
                (int)row, (int)cur.row, 0x111 /* row_shr:1 */, 0xF, 0xF, false);
            const uint64_t begins = __ballot(cur.row != before);
            const uint32_t mine = (uint32_t)(begins >> (threadIdx.x & 63u & ~(uint32_t)(LPR - 1)));
            uint32_t any = 0;
#pragma unroll
            for (int g = 0; g < 64 / LPR; ++g)
                any |= (uint32_t)(begins >> (g * LPR));
            if (__ballot(cur.n < (uint32_t)UB)) { // a chunk's last batch
#pragma unroll
                for (int u = 0; u < UB; ++u)
                    xv[u] = (uint32_t)u < cur.n ? xv[u] : V{};
            }
#pragma unroll
            for (int u = 0; u < UB; ++u) {
                if (any >> u & 1) {
                    const uint32_t l = bcast.entry(cur.row, u) * LPR + sub;
                    if (mine >> u & 1) {
                        tile_y[to] = base + acc;
                        base = tile_y[l];
                        acc = V{};
                        to = l;
                    }
                }
                acc += xv[u] * bcast.entry(cur.val, u);
            }
            if (++batch % kRunBatches == 0) {
                base += acc;
                acc = V{};
            }
            row = bcast.entry(cur.row, UB - 1);
            p = np;
            cur = nxt;
        }
        if (had)
            tile_y[to] = base + acc;
        p = p_nb;
        hi = hi_nb;
        if (!had && p < hi)
            cur = fetch(p, hi);
        __syncthreads(); // the edge slots of block b are written, its direct additions done
        // one lane group per row among the edge slots: the first that holds it adds them all,
        // in lane-group order
        const uint32_t er = edge_row[grp];
        if (er != kNone && (grp == 0 || edge_row[grp - 1] != er)) {
            V sum = tile_y[er * LPR + sub];
            for (uint32_t h = grp; h < G && edge_row[h] == er; ++h)
                sum += tile_y[kEdge + h * LPR + sub];
            tile_y[er * LPR + sub] = sum;
        }
        __syncthreads(); // before block b + 1 writes edge slots and accumulators again
    }
    for (uint32_t i = threadIdx.x; i < R * LPR; i += kSweepBlock) {
        const uint32_t g = tile_rows[(uint64_t)tile * R + i / LPR];
        if (g == 0xFFFFFFFFu)
            continue;
        const uint32_t part = slot ? slot[(uint64_t)tile * R + i / LPR] : kWholeRow;
        if (part == kWholeRow)
            lane.store(lane.load_once(Y, g) + tile_y[i], Y, g);
        else // a piece of a cut row
            lane.store(tile_y[i], partial, part);
    }
}

// The tiles' results to their places: out[dst[h]] = stage[src[h]], the h-th entry of a tile counted place after
// place.  What a tile's entries read lies anywhere in the tile's results (0.4 MB), so the workgroups of a tile
// run on one XCD, as its results were written, and meet them in its L2; what they write are whole rows.
// (13 M results beside the segments of the other rows: 117 us in fp64, 76 in fp32.)
constexpr uint32_t kHomePieces = 8; // workgroups of a tile
template <typename T>
__global__ void __launch_bounds__(kBlock)
hub_home_kernel(const uint32_t *__restrict__ ptr, uint32_t nb, uint32_t ntiles, const uint32_t *__restrict__ src,
                const uint32_t *__restrict__ dst, const T *__restrict__ stage, T *__restrict__ out)
{
    const uint32_t j = blockIdx.x >> 3, tile = j / kHomePieces * 8 + (blockIdx.x & 7u), piece = j % kHomePieces;
    if (tile >= ntiles)
        return;
    const uint32_t lo = ptr[(uint64_t)tile * nb], n = ptr[(uint64_t)(tile + 1) * nb] - lo;
    const uint32_t h0 = (uint32_t)((uint64_t)n * piece / kHomePieces);
    const uint32_t h1 = (uint32_t)((uint64_t)n * (piece + 1) / kHomePieces);
    constexpr uint32_t U = 8;
    for (uint32_t h = h0 + threadIdx.x; h < h1; h += U * kBlock) {
        uint32_t s[U], d[U];
        T v[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t at = lo + (h + u * kBlock < h1 ? h + u * kBlock : h);
            s[u] = nt_load(src + at);
            d[u] = nt_load(dst + at);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            v[u] = stage[s[u]];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (h + u * kBlock < h1)
                out[d[u]] = v[u];
    }
}

// ---------------------------------------------- row pack / unpack (comm buffers) ----
// The copies either side of the reference's sparse exchanges
// (SparseComm::copy_to_sendbuff / copy_from_recvbuff / SUM_from_recvbuff,
// src/comm.hpp:90-103,166-189): buffer slot i holds the dense row rows[i].
//
// LPR lanes (the power of two that covers a row, at most a wavefront) move one row, a unit
// of 16 bytes each, and several rows at a time, so that every index is asked for before the
// first row and every row before the first store (the copies are level from 4 rows in flight to 8; a
// sum takes one row at a time and several of its slots).  Bound by memory: nothing is
// computed.  UNIT: kVec - rows of whole 16-byte vectors; kLoose - rows that end inside one
// start at element alignment, and their last unit is the 16 bytes that END at the row's end
// (it overlaps the unit before: a copy writes the same bytes twice, a sum stores only the
// elements that are the unit's own); kElem - rows under 16 bytes, one real per lane.
// 500 k random rows of a 1 M-row panel, fp32 K = 50, pack / unpack / sum-unpack one after the other,
// each over its own panel: a real per lane with a division per real took 76 / 89 / 135 us, this
// 50 / 50 / 69 (a row of 200 bytes at any alignment touches 2.6 lines of 128; repeated alone, on a
// panel of which much stays in the Infinity Cache, 45 / 85 / 129 and 39 / 40 / 62).  Over panels that
// change from pass to pass the three took 298 and 202 us together.
// What is met again is cached and what is not streams: a panel's rows are read (by a sum) and written once, so they
// stream and leave the caches to the buffer, whose rows share lines with their neighbours, which other workgroups
// read, and which has just been written.  The other way round before; the three together, fp32 K = 50, 500 k slots of
// 1 M rows 202 -> 155 us, K = 64, 1 M slots 277 -> 244 (fp64 545 -> 494), fp64 K = 8 137 -> 104, fp32 K = 130, 1.5 M of
// 2 M 1100 -> 988, fp64 K = 256, 20 k of 60 k 54 -> 48.  (Streaming only the stores 157, 264, 527, 106, 986, 51; a
// pack that streams the rows it reads 160, 254, 517, 104, 1013, 48, one that caches what it writes 5 % slower.)
enum RowUnit { kVec, kLoose, kElem };
constexpr int kRowsAhead = 4;    // of a copy
// Fewer workgroups than this (8 per CU) do not fill the chip: one row at a time then, which
// makes more of them (50 k rows of 56 bytes: sum 6.8 against 4.8 us).
constexpr uint64_t kRowsMinBlocks = 2048;
// More than this are not launched, a workgroup goes on with a further share of the rows: a launch
// of 2^32 threads and more is refused, and 1.1 G rows of one real would ask for it.  (At 65,536
// workgroups rows that a fresh one would have taken wait for a second round: 2 M rows of 520 bytes,
// 1.5 M slots, the three copies 1097 -> 1132 us.)
constexpr uint64_t kRowsMaxBlocks = 1 << 20;
constexpr uint32_t row_unit_bytes(RowUnit u, size_t elem) { return u == kElem ? (uint32_t)elem : 16u; }

template <typename T, RowUnit UNIT> struct RowAccess {
    using V = typename Vec<T>::type;
    static __device__ __forceinline__ V load(const char *p)
    {
        if constexpr (UNIT == kVec)
            return *reinterpret_cast<const V *>(p);
        else
            return loose_load<T>(p);
    }
    static __device__ __forceinline__ V load_nt(const char *p)
    {
        if constexpr (UNIT == kVec)
            return nt_load(reinterpret_cast<const V *>(p));
        else
            return loose_load_nt<T>(p);
    }
    static __device__ __forceinline__ void store(V v, char *p)
    {
        if constexpr (UNIT == kVec)
            *reinterpret_cast<V *>(p) = v;
        else
            loose_store<T>(v, p);
    }
    static __device__ __forceinline__ void store_nt(V v, char *p)
    {
        if constexpr (UNIT == kVec)
            nt_store(v, reinterpret_cast<V *>(p));
        else
            loose_store_nt<T>(v, p);
    }
};
template <typename T> struct RowAccess<T, kElem> {
    using V = T;
    static __device__ __forceinline__ V load(const char *p) { return *reinterpret_cast<const T *>(p); }
    static __device__ __forceinline__ V load_nt(const char *p) { return nt_load(reinterpret_cast<const T *>(p)); }
    static __device__ __forceinline__ void store(V v, char *p) { *reinterpret_cast<T *>(p) = v; }
    static __device__ __forceinline__ void store_nt(V v, char *p) { *reinterpret_cast<T *>(p) = v; }
};

// Byte offset of unit v of a row of `bytes` bytes.
template <typename T, RowUnit UNIT> __device__ __forceinline__ uint64_t unit_off(uint32_t v, uint64_t bytes)
{
    const uint64_t at = (uint64_t)v * row_unit_bytes(UNIT, sizeof(T));
    return UNIT == kLoose && at + 16 > bytes ? bytes - 16 : at;
}

// buf[i, :] = panel[rows[i], :]
template <typename T, RowUnit UNIT, int LPR, int U>
__global__ void __launch_bounds__(kBlock)
rows_pack_kernel(const char *__restrict__ panel, const uint32_t *__restrict__ rows, uint32_t n,
                 uint32_t units, uint64_t bytes, char *__restrict__ buf)
{
    using A = RowAccess<T, UNIT>;
    constexpr uint32_t GPB = kBlock / LPR;
    const uint32_t sub = threadIdx.x % LPR;
    for (uint64_t share = (uint64_t)blockIdx.x * (GPB * U); share < n;
         share += (uint64_t)gridDim.x * (GPB * U)) {
        const uint64_t first = share + threadIdx.x / LPR;
        uint32_t row[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t i = first + u * GPB;
            row[u] = rows[i < n ? i : n - 1];
        }
        for (uint32_t v = sub; v < units; v += LPR) {
            const uint64_t off = unit_off<T, UNIT>(v, bytes);
            typename A::V x[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                x[u] = A::load(panel + (uint64_t)row[u] * bytes + off);
            __builtin_amdgcn_sched_barrier(0); // every row asked for before the first store
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint64_t i = first + u * GPB;
                if (i < n)
                    A::store_nt(x[u], buf + i * bytes + off);
            }
        }
    }
}

// For every distinct destination row (RowDest: the row, its first and last buffer slot, and
// where its slots start in `slots`, ascending): ADD = false: panel row = its last slot (what
// the reference's sequential copy leaves); ADD = true: panel row += each slot in order (the
// reference's sequential sum, bit for bit).
// ADD: one row per lane group (U == 1), D of its slots after the first in flight.
template <typename T, RowUnit UNIT, int LPR, int U, bool ADD, int D = 1>
__global__ void __launch_bounds__(kBlock)
rows_unpack_kernel(char *__restrict__ panel, const u32x4 *__restrict__ dests,
                   const uint32_t *__restrict__ slots, uint32_t n, uint32_t units, uint64_t bytes,
                   const char *__restrict__ buf)
{
    using A = RowAccess<T, UNIT>;
    constexpr uint32_t GPB = kBlock / LPR;
    static_assert(!ADD || U == 1, "sums go row by row");
    const uint32_t sub = threadIdx.x % LPR;
    for (uint64_t share = (uint64_t)blockIdx.x * (GPB * U); share < n;
         share += (uint64_t)gridDim.x * (GPB * U)) {
        const uint64_t first = share + threadIdx.x / LPR;
        u32x4 d[U]; // row, first slot, last slot, start in slots
        uint32_t left = 0; // slots of the row after its first
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t i = first + u * GPB;
            const uint64_t at = i < n ? i : n - 1;
            d[u] = nt_load(dests + at);
            if constexpr (ADD) {
                left = dests[at + 1][3] - d[u][3] - 1;
            }
        }
        for (uint32_t v = sub; v < units; v += LPR) {
            const uint64_t off = unit_off<T, UNIT>(v, bytes);
            typename A::V x[U], y[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                x[u] = A::load(buf + (uint64_t)d[u][ADD ? 1 : 2] * bytes + off);
                if constexpr (ADD)
                    y[u] = A::load_nt(panel + (uint64_t)d[u][0] * bytes + off);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (ADD) {
#pragma unroll
                for (int u = 0; u < U; ++u)
                    y[u] += x[u];
                for (uint32_t t = 1; t <= left; t += D) {
                    typename A::V z[D];
                    uint32_t slot[D];
#pragma unroll
                    for (int j = 0; j < D; ++j)
                        slot[j] = slots[d[0][3] + (t + j < left ? t + j : left)];
#pragma unroll
                    for (int j = 0; j < D; ++j)
                        z[j] = A::load(buf + (uint64_t)slot[j] * bytes + off);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < D; ++j)
                        if (t + j <= left)
                            y[0] += z[j];
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (first + u * GPB >= n)
                    continue;
                char *to = panel + (uint64_t)d[u][0] * bytes + off;
                if constexpr (!ADD) {
                    A::store_nt(x[u], to);
                } else {
                    if constexpr (UNIT == kLoose) {
                        const uint32_t skip = (uint32_t)((uint64_t)v * 16 - off) / (uint32_t)sizeof(T);
                        if (skip) { // the row's last unit: its leading elements are the unit's before
                            T *e = reinterpret_cast<T *>(to);
#pragma unroll
                            for (uint32_t j = 0; j < (uint32_t)Vec<T>::N; ++j)
                                if (j >= skip)
                                    e[j] = y[u][j];
                            continue;
                        }
                    }
                    A::store_nt(y[u], to);
                }
            }
        }
    }
}

// XCD on which each workgroup of a 1-D grid runs (hardware register XCC_ID).
__global__ void __launch_bounds__(64) xcc_probe_kernel(uint32_t *__restrict__ out)
{
    // s_getreg_b32 hwreg(HW_REG_XCC_ID = 20, offset 0, width 4)
    const uint32_t id = __builtin_amdgcn_s_getreg(20 | (0 << 6) | ((4 - 1) << 11));
    if (threadIdx.x == 0)
        out[blockIdx.x] = id;
}

// ------------------------------------------------------------- utilities ----
// Measurement aid (launch_probe_cols): the column of every kernel-order entry replaced so
// that the launches keep their instruction stream, segments and queues while every gather
// hits (mode 1: base + (c - base) % modulus, a table of `modulus` dense rows) or nearly
// every gather misses (mode 2: a hash of the entry's position, uniform over ncols).  hot (may be
// null): the columns that `col` names by rank.
__global__ void __launch_bounds__(kBlock)
probe_cols_kernel(uint32_t *__restrict__ col, uint64_t n, uint32_t mode, uint32_t base,
                  uint32_t modulus, uint32_t ncols, const uint32_t *__restrict__ hot)
{
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
        if (mode == 1) {
            const uint32_t c = hot && (col[i] & kHotRow) ? hot[col[i] & ~kHotRow] : col[i];
            col[i] = c >= base ? base + (c - base) % modulus : c % modulus;
        } else {
            uint64_t x = (i + 1) * 0x9E3779B97F4A7C15ull; // splitmix64 finaliser
            x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
            x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
            x ^= x >> 31;
            col[i] = (uint32_t)(x % ncols);
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(kBlock)
gather_kernel(const T *__restrict__ in, const uint32_t *__restrict__ perm, T *__restrict__ out,
              uint64_t n)
{
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride)
        out[i] = perm ? in[perm[i]] : in[i];
}

// out[perm[i]] = in[i] (perm null: out[i] = in[i])
template <typename T>
__global__ void __launch_bounds__(kBlock)
scatter_kernel(const T *__restrict__ in, const uint32_t *__restrict__ perm, T *__restrict__ out,
               uint64_t n)
{
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride)
        out[perm ? perm[i] : i] = in[i];
}

// out[i] = in[pos[i]], four results per lane and step, U steps in flight: positions and results move as
// 16-byte vectors, streaming; the reads in between are whatever `pos` makes them (runs, for the staged results
// of a plan kept in column blocks).  Where a row's columns are in no order they go to and fro among the row's
// runs (one per block of columns): a lane waits for them, and their lines are met again while the first level
// holds them, so a wavefront takes whole rows, one after the other, with many reads under way.  572 M results
// of rows of up to 1024, fp32, the whole SDDMM call: workgroups of 256 and one step 17.38 ms, two 17.03, four 16.86;
// of 64 and 4 steps 16.77, 8 16.70, 16 17.17; of 1024 and one 17.76.  Of 86 M: 3302 us -> 3258 (64 and 4), 3330 (8).
template <typename T, int BLOCK, int U>
__global__ void __launch_bounds__(BLOCK)
gather4_kernel(const T *__restrict__ in, const uint32_t *__restrict__ pos, T *__restrict__ out,
               uint64_t n)
{
    const uint64_t stride = (uint64_t)gridDim.x * BLOCK * 4 * U;
    const uint64_t nfull = n / 4 * 4;
    // Workgroups are dealt to the XCDs in turn: workgroup b takes the chunk that gives every
    // XCD a contiguous eighth of each round of chunks, so that neighbours in `out`, whose
    // reads tend to share lines of `in`, meet in one L2.
    uint32_t chunk = blockIdx.x;
    if (gridDim.x % 8 == 0)
        chunk = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    for (uint64_t i = ((uint64_t)chunk * BLOCK * U + threadIdx.x) * 4; i < nfull; i += stride) {
        u32x4 p[U];
#pragma unroll
        for (int k = 0; k < U; ++k) {
            const uint64_t at = i + (uint64_t)k * BLOCK * 4;
            p[k] = nt_load(reinterpret_cast<const u32x4 *>(pos + (at < nfull ? at : i)));
        }
        using V = typename Vec<T>::type; // 16 bytes: 4 floats or 2 doubles
        V v[U][4 / Vec<T>::N];
#pragma unroll
        for (int k = 0; k < U; ++k)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                v[k][u / Vec<T>::N][u % Vec<T>::N] = in[p[k][u]];
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (i + (uint64_t)k * BLOCK * 4 < nfull)
#pragma unroll
                for (int u = 0; u < 4 / Vec<T>::N; ++u)
                    nt_store(v[k][u], reinterpret_cast<V *>(out + i + (uint64_t)k * BLOCK * 4) + u);
    }
    const uint64_t t = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (t < n - nfull)
        out[nfull + t] = in[pos[nfull + t]];
}

// out[dst[h]] = stage[src[h]], h < n, dst ascending and mostly consecutive: four results in
// flight per lane, consecutive lanes on consecutive h.
template <typename T>
__global__ void __launch_bounds__(kBlock)
unstage_pairs_kernel(const T *__restrict__ stage, const uint32_t *__restrict__ src,
                     const uint32_t *__restrict__ dst, T *__restrict__ out, uint64_t n)
{
    constexpr uint64_t U = 4;
    const uint64_t span = (uint64_t)kBlock * U;
    uint64_t base = (uint64_t)blockIdx.x * span;
    for (; base + span <= n; base += (uint64_t)gridDim.x * span) {
        uint32_t s[U], d[U];
        T v[U];
#pragma unroll
        for (uint64_t u = 0; u < U; ++u) {
            s[u] = nt_load(src + base + u * kBlock + threadIdx.x);
            d[u] = nt_load(dst + base + u * kBlock + threadIdx.x);
        }
#pragma unroll
        for (uint64_t u = 0; u < U; ++u)
            v[u] = nt_load(stage + s[u]);
#pragma unroll
        for (uint64_t u = 0; u < U; ++u)
            nt_store(v[u], out + d[u]);
    }
    // what is left is less than one span, and one workgroup's `base` lies in it
    for (uint64_t h = base + threadIdx.x; h < n; h += kBlock)
        out[dst[h]] = stage[src[h]];
}

// ---- results of an arbitrary entry order to the caller's positions in two passes ------
// (see TwoPass in plan_device.h).  One workgroup per tile of kTwoPassBytes of results,
// held in LDS between its coalesced read and its grouped write.
constexpr uint32_t kTwoPassBytes = 160u << 10; // all of a CU's LDS
constexpr int kTwoPassBlock = 1024;
template <typename T> constexpr uint32_t two_pass_tile() { return kTwoPassBytes / sizeof(T); }

template <typename T>
__device__ __forceinline__ void tile_to_lds(T *buf, const T *__restrict__ src, uint32_t cnt)
{
    using V = typename Vec<T>::type;
    constexpr uint32_t VN = Vec<T>::N;
    constexpr uint32_t TILE = two_pass_tile<T>();
    constexpr uint32_t R = TILE / VN / kTwoPassBlock; // 16-byte loads per lane and tile: 10
    static_assert(R * VN * kTwoPassBlock == TILE, "a tile is a whole number of rounds");
    const V *in = reinterpret_cast<const V *>(src); // 16-byte aligned: a whole tile into a library buffer
    V *to = reinterpret_cast<V *>(buf);
    if (cnt == TILE) { // every load in flight before the first word is stored
        V v[R];
#pragma unroll
        for (uint32_t r = 0; r < R; ++r)
            v[r] = nt_load(in + threadIdx.x + r * kTwoPassBlock);
#pragma unroll
        for (uint32_t r = 0; r < R; ++r)
            to[threadIdx.x + r * kTwoPassBlock] = v[r];
        return;
    }
    const uint32_t nvec = cnt / VN;
    for (uint32_t i = threadIdx.x; i < nvec; i += kTwoPassBlock)
        to[i] = nt_load(in + i);
    for (uint32_t i = nvec * VN + threadIdx.x; i < cnt; i += kTwoPassBlock)
        buf[i] = src[i];
}

// Pass 1: tile blockIdx.x of `stage` (kernel order), out grouped by bucket of destination.
template <typename T>
__global__ void __launch_bounds__(kTwoPassBlock)
unpermute_pass1_kernel(const T *__restrict__ stage, const uint16_t *__restrict__ l1,
                       const uint32_t *__restrict__ dst1, T *__restrict__ mid, uint64_t n)
{
    constexpr uint32_t TILE = two_pass_tile<T>();
    __shared__ T buf[TILE];
    const uint64_t base = (uint64_t)blockIdx.x * TILE;
    if (base >= n)
        return;
    const uint32_t cnt = (uint32_t)(n - base < TILE ? n - base : TILE);
    constexpr uint32_t U = 10;
    // the first positions are asked for before the tile is: they do not depend on it
    uint32_t l[U], d[U];
    uint32_t s = threadIdx.x;
    const bool first_full = s + (U - 1) * kTwoPassBlock < cnt;
    if (first_full) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            l[u] = nt_load(l1 + base + s + u * kTwoPassBlock);
            d[u] = nt_load(dst1 + base + s + u * kTwoPassBlock);
        }
    }
    tile_to_lds(buf, stage + base, cnt);
    __syncthreads();
    if (first_full) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            nt_store(buf[l[u]], mid + d[u]);
        s += U * kTwoPassBlock;
    }
    for (; s + (U - 1) * kTwoPassBlock < cnt; s += U * kTwoPassBlock) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            l[u] = nt_load(l1 + base + s + u * kTwoPassBlock);
            d[u] = nt_load(dst1 + base + s + u * kTwoPassBlock);
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            nt_store(buf[l[u]], mid + d[u]);
    }
    for (; s < cnt; s += kTwoPassBlock)
        nt_store(buf[nt_load(l1 + base + s)], mid + nt_load(dst1 + base + s));
}

// Pass 2: bucket blockIdx.x of `mid`, out to the caller's positions [base, base + cnt) in order.
template <typename T>
__global__ void __launch_bounds__(kTwoPassBlock)
unpermute_pass2_kernel(const T *__restrict__ mid, const uint16_t *__restrict__ l2,
                       T *__restrict__ C, uint64_t n)
{
    using V = typename Vec<T>::type;
    constexpr uint32_t VN = Vec<T>::N;
    constexpr uint32_t TILE = two_pass_tile<T>();
    __shared__ T buf[TILE];
    const uint64_t base = (uint64_t)blockIdx.x * TILE;
    if (base >= n)
        return;
    const uint32_t cnt = (uint32_t)(n - base < TILE ? n - base : TILE);
    typedef uint16_t Idx __attribute__((ext_vector_type(VN)));
    constexpr uint32_t R = TILE / VN / kTwoPassBlock; // 16-byte stores per lane and tile: 10
    T *out = C + base;
    const bool fast = cnt == TILE && (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
    Idx li[R];
    if (fast) { // the positions do not depend on the tile: asked for first
#pragma unroll
        for (uint32_t r = 0; r < R; ++r)
            li[r] = nt_load(reinterpret_cast<const Idx *>(l2 + base) + threadIdx.x + r * kTwoPassBlock);
    }
    tile_to_lds(buf, mid + base, cnt);
    __syncthreads();
    if (fast) {
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) {
            V v;
#pragma unroll
            for (uint32_t e = 0; e < VN; ++e)
                v[e] = buf[li[r][e]];
            nt_store(v, reinterpret_cast<V *>(out) + threadIdx.x + r * kTwoPassBlock);
        }
        return;
    }
    uint32_t done = 0;
    if ((reinterpret_cast<uintptr_t>(out) & 15u) == 0) { // the caller's C may be a wrapped vector
        const uint32_t nvec = cnt / VN;
        for (uint32_t i = threadIdx.x; i < nvec; i += kTwoPassBlock) {
            const Idx l = nt_load(reinterpret_cast<const Idx *>(l2 + base) + i);
            V v;
#pragma unroll
            for (uint32_t e = 0; e < VN; ++e)
                v[e] = buf[l[e]];
            nt_store(v, reinterpret_cast<V *>(out) + i);
        }
        done = nvec * VN;
    }
    for (uint32_t j = done + threadIdx.x; j < cnt; j += kTwoPassBlock)
        out[j] = buf[l2[base + j]];
}

template <typename T>
__global__ void __launch_bounds__(kBlock) fill_kernel(T *__restrict__ p, uint64_t n, T value)
{
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride)
        p[i] = value;
}

// Plain streaming copy: four 16-byte non-temporal loads in flight per lane, then
// four non-temporal stores (5.8 TB/s read + written on this GPU; one load per
// iteration with plain accesses gives 4.6).  The last (< 4 * block) vectors go
// one by one, the tail (< 16 bytes) bytewise by the first lanes.
__global__ void __launch_bounds__(kBlock)
copy_kernel(u32x4 *__restrict__ dst, const u32x4 *__restrict__ src, uint64_t nvec,
            uint32_t tail_bytes)
{
    constexpr uint64_t U = 4;
    const uint64_t tid = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    const uint64_t span = (uint64_t)kBlock * U; // vectors one block moves per iteration
    const uint64_t nfull = nvec / span * span;
    for (uint64_t i = (uint64_t)blockIdx.x * span + threadIdx.x; i < nfull;
         i += (uint64_t)gridDim.x * span) {
        u32x4 v[U];
#pragma unroll
        for (uint64_t u = 0; u < U; ++u)
            v[u] = nt_load(src + i + u * kBlock);
#pragma unroll
        for (uint64_t u = 0; u < U; ++u)
            nt_store(v[u], dst + i + u * kBlock);
    }
    for (uint64_t i = nfull + tid; i < nvec; i += (uint64_t)gridDim.x * kBlock)
        dst[i] = src[i];
    if (tid < tail_bytes)
        reinterpret_cast<unsigned char *>(dst + nvec)[tid] =
            reinterpret_cast<const unsigned char *>(src + nvec)[tid];
}

// ------------------------------------------------------------- dispatch ----
struct Shape {
    int lpr, vpl;  // lpr == 0: rows over 4 KiB, run slice by slice
    int mode;      // the kernels' RG: 0 exact, 1 ragged, 2 odd, 3 thin
    uint32_t nvec; // 16-byte vectors per dense row; modes 2, 3: K, the reals per row
};

// A dense row of K reals of at most 4096 bytes runs in one launch (pair); longer ones
// go slice by slice, rows under 16 bytes take the "thin" variant of the 4-lane shape.  A whole number nvec of 16-byte
// vectors with nvec == LPR * VPL, LPR a power of two in [4, 64] and VPL in {1, 2, 4},
// runs a kernel with the row stride compiled in; other nvec run the "ragged" variant
// of the smallest shape that covers a row, in which the lanes past the row's end
// idle; rows that are no whole number of vectors, or of at most 16, run the "odd"
// variant of that shape.
Shape pick_shape(size_t elem, uint32_t K)
{
    const size_t bytes = (size_t)K * elem;
    if (K == 0 || bytes > 4096)
        return {0, 0, 0, 0};
    if (bytes < 16)
        return {4, 1, 3, K};
    const uint32_t nvec = (uint32_t)((bytes + 15) / 16);
    const bool odd = bytes % 16 != 0;
    for (int lpr = 64; lpr >= 4 && !odd; lpr >>= 1) {
        if (nvec % lpr)
            continue;
        const uint32_t vpl = nvec / lpr;
        if (vpl == 1 || vpl == 2 || vpl == 4)
            return {lpr, (int)vpl, 0, nvec};
        break;
    }
    // Narrow rows that leave lanes idle also run the odd variant, which loads whole vectors at
    // element alignment; from 17 vectors on its selects per element would cost SDDMM 2 to 4 %
    // over the ragged variant's one per dot product.
    const int mode = (odd || nvec <= 16) ? 2 : 1;
    const uint32_t arg = mode == 2 ? K : nvec;
    if (nvec > 128)
        return {64, 4, mode, arg};
    if (nvec > 64)
        return {64, 2, mode, arg};
    int lpr = 4;
    while ((uint32_t)lpr < nvec)
        lpr *= 2;
    return {lpr, 1, mode, arg};
}

// Workgroups needed to cover nseg segments (a whole number of chunks, and of
// rounds of 8 chunks when they are dealt to XCDs) with `groups_per_wave` segments
// per wavefront.
inline uint32_t blocks_for_groups(uint32_t nseg, uint32_t nq, int groups_per_wave)
{
    uint64_t chunks = ((uint64_t)nseg + kChunk - 1) / kChunk;
    if (nq == 8)
        chunks = (chunks + 7) / 8 * 8;
    return (uint32_t)(chunks * (kChunk / ((kBlock / 64) * groups_per_wave)));
}

// Two launches per call: the leading nseg_long segments (all at least
// kLongSegment entries long) run with UB gathers in flight per lane and
// 4 wavefronts per SIMD; the rest run the US-wide variant, whose register
// budget lets 8 wavefronts per SIMD hide the three dependent memory latencies
// of a short segment (descriptor -> indices -> gathers).  Measured: 5-entry
// rows of a stencil 1.6x faster with US = 4 than with 16, R-MAT hub segments
// 1.5x slower.  With an auxiliary stream the two run side by side.

// A pattern this small does not keep the chip busy for long enough to repay a
// second launch with its fork and join (about 20 us when the kernels are short):
// when it has segments of both kinds, all of them go to the wide launch (either
// kernel handles segments of any length; the long ones hold most of the entries).
// Measured on R-MAT 14 .. 19: one launch wins up to about 180 k segments (11 against
// 32 us at 12 k), two from 400 k on.
constexpr uint32_t kOneLaunchSegments = 196608;

// Segments for the wide launch (the first *nl) and for the short one.  Short segments that fill
// most of a wide batch, in a pattern that has no others, go to the wide launch too: one round of
// gathers instead of two to four.  Uniform rows of 12 to 15, fp32 K = 8: SDDMM 125 -> 116 us, SpMM 102
// -> 99; K = 64: 404 -> 388 and 442 -> 418; rows of 11 are level or better in the short one, and so are
// dense rows that leave lanes idle (15 entries, fp32 K = 134: 71 us together in the short one, 74).
// A few short ones left over from whole chunks of long ones go with those (500 k rows of 16, fp64 K = 64:
// the second launch and its fork cost 12 us of 608).
inline void split_launches(const DevPlanView &P, bool whole_lanes, uint32_t &nl, uint32_t &ns)
{
    nl = P.nseg_long, ns = P.nseg - P.nseg_long;
    if (nl ? P.nseg <= kOneLaunchSegments || ns <= nl / 64 : whole_lanes && P.nnz >= (uint64_t)12 * P.nseg)
        nl = P.nseg, ns = 0;
}

// Makes the auxiliary stream wait for everything queued on the main stream so
// far.  On failure nothing was queued on aux and the caller stays on main.
inline bool fork_aux(const Streams &S)
{
    return S.aux && hipEventRecord(S.fork, S.main) == hipSuccess &&
           hipStreamWaitEvent(S.aux, S.fork, 0) == hipSuccess;
}

// Makes the main stream wait for what was queued on the auxiliary stream; if the
// events fail, waits on the host instead, so the ordering holds either way.
inline hipError_t join_aux(const Streams &S)
{
    if (hipEventRecord(S.join, S.aux) == hipSuccess &&
        hipStreamWaitEvent(S.main, S.join, 0) == hipSuccess)
        return hipSuccess;
    (void)hipGetLastError();
    return hipStreamSynchronize(S.aux);
}

enum LaunchOf { kSddmm, kOnePass, kSpmm };

// Workgroups of a segment launch per CU, or 0: as many as its registers allow (4 to 8).  Where nearly every
// gather misses the L2s and a launch has more than enough of them in flight, fewer at once are served
// faster: unskewed columns (no slices), four rounds of wavefronts and more, mostly at least three lanes in four busy.
// `cached`: panels (of touched rows) that the Infinity Cache mostly holds.  Speed against as many as fit, median and
// range over uniform rows of 3 to 32 entries, 64 to 4096 bytes wide, over 2 k to 1 M columns:
//  - the wide launch, cached panels: 2 from 24 MiB and 16 entries on (rows that leave lanes of 64 idle from 24, of fewer
//    from 32; one-pass from 24 in groups of 64 without idle lanes or with longer rows, else from 32) 1.03 (0.99 .. 1.11); 3 from 16 MiB and 12
//    entries on (SpMM over mixed lengths from 8) 1.02 (0.97 .. 1.07).  Beyond 320 MiB SpMM over even rows alone: 3, 1.02
//    (0.99 .. 1.04); SDDMM and one-pass would lose up to 5 %.  Fewer than three lanes in four busy, cached panels, 16
//    entries on: 3, SpMM from 32 MiB 1.02 (0.98 .. 1.07), one-pass over longer rows from 16 MiB 1.02 (0.98 .. 1.04);
//  - the short launch, cached panels of 64 MiB and more, from 6 entries on: 4, SDDMM 1.03 (1.00 .. 1.11), SpMM 1.02 (1.00 ..
//    1.09; idle lanes of 64 and longer rows or 8 entries 1.04, 1.02 .. 1.07; idle lanes of 32 1.04, under 25 busy 5,
//    1.02); SDDMM with idle lanes 6, 1.01 (0.99 .. 1.05; under 25 of 32 busy 0.97, so none);
//  - SpMM whose rows leave lanes of 64 idle, otherwise: 6 from 32 MiB and 5 entries on, 1.01 (0.98 .. 1.05);
//  - one-pass in groups of 64 lanes, whose short launch holds up to 8 rows per wavefront: one vector per lane 4 (cached, 64
//    MiB, 6 entries) 1.05 (1.02 .. 1.08), else 5 (8 MiB, where they end inside a
//    vector 16, 5 entries) 1.02 (0.98 .. 1.07); with idle lanes 6 (cached, 32 MiB, 6
//    entries) 1.01 (0.98 .. 1.03), from 12 entries and 24 MiB on 5, 1.03; longer rows 4 (8 MiB, 3 entries) 1.03 (0.97 .. 1.08), where they
//    end inside a vector or lanes idle 5 (32 MiB, 3 entries; fewer than three lanes in four busy: cached, 7 entries) 1.03
//    (1.00 .. 1.06), over 2 KiB 4 (16 MiB and the same) 1.02 (0.99 .. 1.04);
//  - one-pass otherwise as the short launch, but 6: 1.00 (0.97 .. 1.01); from 12 entries over rows that end inside a vector
//    4, 1.04;
//  - SpMM's short launch at 4 and 5 entries, dense rows of 512 bytes and more, whatever the panel: 7, 1.01
//    .. 1.04 from 65,536 wavefronts on (half of them: 0.99).
// Rows of mixed lengths (Poisson), whose two launches are asked one by one: SpMM 0.99 .. 1.04, the others level.  Panels in
// the L2s want every wavefront (100 k rows of 20 over 2 k columns, fp64 K = 128: 0.87 / 0.92 / 0.91 at 3), and so do
// half-empty groups (400 k rows of 8, fp64 K = 65: 0.89 / 0.83 / 0.85 at 4).
template <int LPR, int VPL, int RG>
inline uint32_t workgroups_per_cu(const DevPlanView &P, bool wide, uint32_t nseg, LaunchOf what, uint64_t row_bytes)
{
    constexpr uint64_t kFull = (uint64_t)LPR * VPL * 16;
    const uint64_t panel = P.cols_touched * row_bytes, waves = (uint64_t)nseg * LPR / 64;
    if (P.nqueues != 1 || waves < 16384)
        return 0;
    const auto from = [&](uint64_t entries) { return P.nnz >= entries * P.nseg; }; // per segment, on average
    const auto holds = [&](uint64_t mib) { return panel >= mib << 20; };
    const bool cached = panel <= (uint64_t)320 << 20;
    const bool filled = row_bytes * 4 >= kFull * 3;
    if (wide) {
        const uint64_t least = what == kOnePass ? (LPR == 64 && (RG != 1 || VPL > 1) ? 24 : 32)
                                                : (RG == 1 ? (LPR == 64 ? 24 : 32) : 16);
        const bool even = nseg == P.nseg && (nseg - P.nseg_long <= nseg / 64 || !P.nseg_long);
        if (!filled)
            return cached && from(16) && (what == kSpmm ? holds(32) : what == kOnePass && VPL > 1 && holds(16)) ? 3 : 0;
        if (cached && holds(24) && even && from(least))
            return 2;
        if (LPR < 16 || !holds(16))
            return 0;
        if (what == kSpmm)
            return cached ? (from(8) ? 3 : 0) : (even && from(12) ? 3 : 0);
        return cached && from(12) ? 3 : 0;
    }
    // Beside a wide launch that takes every place (its rows are many, and short on average), a short one that is
    // held back ends last: 12 M entries in rows of 1 to 63, fp32 K = 128, SDDMM 1.03 -> 1.06 ms.
    if (nseg != P.nseg && P.nseg_long > P.nseg / 6 && !from(12))
        return 0;
    const bool near = cached && holds(64) && from(6);
    if (what == kOnePass && LPR == 64 && VPL > 1) {
        if (RG <= 0)
            return holds(8) && from(3) ? 4 : 0;
        if (VPL == 4)
            return holds(16) && (filled ? from(3) : cached && from(7)) ? 4 : 0;
        if (filled)
            return holds(32) && from(3) ? 5 : 0;
        return cached && holds(32) && from(7) ? 5 : 0;
    }
    if (!filled)
        return 0;
    if (what == kOnePass && LPR == 64) {
        if (RG == 1)
            return holds(24) && from(12) ? 5 : (cached && holds(32) && from(6) ? 6 : 0);
        return near ? 4 : (holds(RG == 2 ? 16 : 8) && from(5) ? 5 : 0);
    }
    if (what == kOnePass)
        return near ? (RG == 2 && from(12) ? 4 : 6) : 0;
    const bool idle = RG == 1 && LPR < 64 && row_bytes * 32 < kFull * 25; // fewer than 25 of 32 lanes busy
    if (what == kSddmm)
        return near && !idle ? (RG == 1 ? 6 : 4) : 0;
    if (RG == 1 && LPR < 64)
        return near ? (idle ? 5 : 4) : 0;
    if (RG == 1)
        return near && (VPL > 1 || from(8)) ? 4 : (holds(32) && from(5) ? 6 : 0);
    if (near)
        return 4;
    const bool few = RG <= 0 && kFull >= 512 && nseg == P.nseg && holds(64) && from(4) && !from(6);
    return few && waves >= 65536 ? 7 : 0;
}

// The least dynamic LDS with which no more of them fit a CU, whose 160 KiB are handed out in pieces of 1280
// bytes.
template <typename T, int LPR, int VPL, int RG>
inline uint32_t crowding_lds(const DevPlanView &P, bool wide, uint32_t nseg, LaunchOf what, uint32_t nvec)
{
    constexpr uint32_t kPiece = 1280, kPieces = (160u << 10) / kPiece;
    const uint64_t row_bytes = RG <= 0 ? (uint64_t)LPR * VPL * 16 : (uint64_t)nvec * (RG == 1 ? 16 : sizeof(T));
    const uint32_t n = workgroups_per_cu<LPR, VPL, RG>(P, wide, nseg, what, row_bytes);
    return n ? (kPieces / (n + 1) + 1) * kPiece : 0;
}

inline uint32_t store_flags(const DevPlanView &P)
{
    return (P.stream_c ? kStoreStream : 0u) | (P.perm && P.seg_base ? kStoreSegBase : 0u);
}

template <typename T, int LPR, int VPL, int UB, int US, int RG, int FZ>
hipError_t run_sddmm(const DevPlanView &P, const T *A, const T *B, T *C, T *Y, const Streams &S,
                     uint32_t nvec, uint32_t stride = 0, uint32_t accum = 0)
{
    uint32_t nl, ns;
    split_launches(P, RG <= 0, nl, ns);
    const bool both = nl && ns && fork_aux(S);
    constexpr LaunchOf kind = FZ ? kOnePass : kSddmm;
    if (nl)
        hipLaunchKernelGGL((sddmm_seg_kernel<T, LPR, VPL, UB, RG, true, FZ>),
                           dim3(blocks_for_groups(nl, P.nqueues, 64 / LPR)), dim3(kBlock),
                           (crowding_lds<T, LPR, VPL, RG>(P, true, nl, kind, nvec)),
                           S.main, P.segs, nl, P.nqueues, 0u, P.col, P.perm, (const T *)P.sval,
                           A, B, C, Y, (T *)P.partial, nvec, stride ? stride : nvec, accum,
                           (const uint32_t *)nullptr, store_flags(P), (T *)P.stage,
                           P.stage_from, P.ref_at, P.hot_at);
    if (ns)
        hipLaunchKernelGGL((sddmm_seg_kernel<T, LPR, VPL, US, RG, false, FZ>),
                           dim3(blocks_for_groups(ns, P.nqueues, 64 / LPR)), dim3(kBlock),
                           (crowding_lds<T, LPR, VPL, RG>(P, false, ns, kind, nvec)),
                           both ? S.aux : S.main, P.segs + nl, ns, P.nqueues,
                           both ? S.aux_rot : 0u, P.col, P.perm, (const T *)P.sval, A, B, C, Y,
                           (T *)P.partial, nvec, stride ? stride : nvec, accum, P.first_cols,
                           store_flags(P), (T *)P.stage, P.stage_from, P.ref_at, P.hot_at);
    const hipError_t launched = hipGetLastError();
    const hipError_t joined = both ? join_aux(S) : hipSuccess;
    return launched != hipSuccess ? launched : joined;
}

template <typename T, int LPR, int VPL, int UB, int US, int RG>
hipError_t run_spmm(const DevPlanView &P, const T *X, T *Y, const Streams &S, uint32_t nvec,
                    uint32_t stride = 0, size_t slice_off = 0, uint32_t pstride = 0)
{
    uint32_t nl, ns;
    split_launches(P, RG <= 0, nl, ns);
    const bool both = nl && ns && fork_aux(S);
    if (nl)
        hipLaunchKernelGGL((spmm_seg_kernel<T, LPR, VPL, UB, RG, true>),
                           dim3(blocks_for_groups(nl, P.nqueues, 64 / LPR)), dim3(kBlock),
                           (crowding_lds<T, LPR, VPL, RG>(P, true, nl, kSpmm, nvec)),
                           S.main, P.segs, nl, P.nqueues, 0u, P.col, (const T *)P.sval, X, Y,
                           (T *)P.partial + slice_off, nvec, stride ? stride : nvec, pstride,
                           (const uint32_t *)nullptr, P.ref_at, P.hot_at);
    if (ns)
        hipLaunchKernelGGL((spmm_seg_kernel<T, LPR, VPL, US, RG, false>),
                           dim3(blocks_for_groups(ns, P.nqueues, 64 / LPR)), dim3(kBlock),
                           (crowding_lds<T, LPR, VPL, RG>(P, false, ns, kSpmm, nvec)),
                           both ? S.aux : S.main, P.segs + nl, ns, P.nqueues,
                           both ? S.aux_rot : 0u, P.col, (const T *)P.sval, X, Y,
                           (T *)P.partial + slice_off, nvec, stride ? stride : nvec, pstride,
                           P.first_cols, P.ref_at, P.hot_at);
    const hipError_t launched = hipGetLastError();
    const hipError_t joined = both ? join_aux(S) : hipSuccess;
    return launched != hipSuccess ? launched : joined;
}

// (LPR, VPL, UB, US_SDDMM, US_SPMM): UB * VPL 16-byte gathers are in flight per
// lane in the long-segment launch, US * VPL in the short-segment one.
#define SPC3D_FOR_SHAPES(X)                                                                       \
    X(4, 1, 16, 8, 4) X(8, 1, 16, 8, 4) X(16, 1, 16, 8, 4) X(32, 1, 16, 8, 4) X(64, 1, 16, 8, 4)  \
    X(4, 2, 8, 4, 2) X(8, 2, 8, 4, 2) X(16, 2, 8, 4, 2) X(32, 2, 8, 4, 2) X(64, 2, 8, 4, 2)       \
    X(4, 4, 4, 2, 1) X(8, 4, 4, 2, 1) X(16, 4, 4, 2, 1) X(32, 4, 4, 2, 1) X(64, 4, 4, 2, 1)
// Rows that do not fill a shape: the smallest power-of-two LPR covering the row,
// then 64 lanes with 2 or 4 vectors each.  The ragged variants are only used from
// 17 vectors per row on.
#define SPC3D_FOR_ODD_SHAPES(X)                                                                   \
    X(4, 1, 16, 8, 4) X(8, 1, 16, 8, 4) X(16, 1, 16, 8, 4) X(32, 1, 16, 8, 4) X(64, 1, 16, 8, 4)  \
    X(64, 2, 8, 4, 2) X(64, 4, 4, 2, 1)
#define SPC3D_FOR_RAGGED_SHAPES(X) X(32, 1, 16, 8, 4) X(64, 1, 16, 8, 4) X(64, 2, 8, 4, 2) X(64, 4, 4, 2, 1)

// The exact shapes of the dense rows that hot_row_width admits.
#define SPC3D_FOR_HOT_SHAPES(X)                                                                   \
    X(16, 1, 16, 8, 4) X(32, 1, 16, 8, 4) X(64, 1, 16, 8, 4) X(64, 2, 8, 4, 2) X(64, 4, 4, 2, 1)

// Copies the hot rows of the operand `dense` (rows of row_bytes bytes) side by side; `out` and `base` are
// then the view and the operand's address for the launches that gather them from there (RG == -1).  False:
// the plan has none, its buffer is for narrower rows, it is out of reach of the operand, or the call gathers
// too little to repay the copy: a plan for wide rows may run narrow ones (400 k entries planned for 512 fp64
// columns and run at 32: SDDMM / SpMM / one-pass 30 / 26 / 37 us with the copy, 28 / 23 / 33 without).
inline bool hot_view(const DevPlanView &P, size_t elem, const void *dense, uint32_t row_bytes,
                     DevPlanView &out, const void **base, hipStream_t st, hipError_t *e)
{
    if (!P.nhot || row_bytes > P.hot_row_bytes || (!P.hot_copied && !hot_rows_pay(P.nnz, row_bytes)))
        return false;
    // the buffer has kHotUnit bytes to spare, so that both lie a whole number of units apart
    const uintptr_t d = reinterpret_cast<uintptr_t>(dense);
    uintptr_t h = reinterpret_cast<uintptr_t>(P.hot_rows);
    h += (d - h) % kHotUnit;
    const uintptr_t low = std::min(d, h);
    const uint64_t rows_bytes = (uint64_t)P.ncols * row_bytes, hot_bytes = (uint64_t)P.nhot * row_bytes;
    if (std::max(d + rows_bytes, h + hot_bytes) - low >= (uint64_t)kHotUnit << 32)
        return false;
    RowMapView rows;
    rows.rows = P.hot_cols;
    rows.nslots = P.nhot;
    *e = P.hot_copied ? hipSuccess
                      : launch_rows(0, elem == 8 ? 1 : 0, const_cast<void *>(dense), rows,
                                    row_bytes / (uint32_t)elem, reinterpret_cast<void *>(h), st);
    out = P;
    out.col = P.hot_col;
    out.first_cols = P.hot_first_cols;
    out.ref_at = (uint32_t)((d - low) / kHotUnit);
    out.hot_at = (uint32_t)((h - low) / kHotUnit) - kHotRow * (row_bytes / kHotUnit);
    *base = reinterpret_cast<const void *>(low);
    return *e == hipSuccess;
}

// Columns [at, at + w) of K (w == 0: all of them); the runs are those of the whole row either way.
template <typename T>
hipError_t launch_fixup(const DevPlanView &P, T *Y, uint32_t K, hipStream_t st, uint32_t at = 0,
                        uint32_t w = 0)
{
    if (!P.nsplit)
        return hipSuccess;
    using V = typename Vec<T>::type;
    const bool vec = K % Vec<T>::N == 0;
    const uint32_t units = vec ? K / Vec<T>::N : K;
    uint32_t lanes = 4;
    while (lanes < (uint32_t)kBlock && lanes < units)
        lanes *= 2;
    // Runs while the launch does not fill the chip anyway.
    uint32_t parts = 1;
    while (lanes * parts < (uint32_t)kBlock && parts * P.nsplit <= 2 * (uint64_t)P.nslots &&
           (uint64_t)P.nsplit * lanes * parts < (1u << 18))
        parts *= 2;
    const uint32_t rows = kBlock / (lanes * parts);
    const dim3 grid((P.nsplit + rows - 1) / rows);
    if (vec && w == 0)
        hipLaunchKernelGGL((spmm_fixup_kernel<T, V>), grid, dim3(kBlock), 0, st, P.splits, P.nsplit,
                           (const V *)P.partial, (V *)Y, units, units, lanes, parts);
    else
        hipLaunchKernelGGL((spmm_fixup_kernel<T, T>), grid, dim3(kBlock), 0, st, P.splits, P.nsplit,
                           (const T *)P.partial, Y + at, w ? w : K, K, lanes, parts);
    return hipGetLastError();
}

// The shape of rows that end inside a vector (mode 2) or are shorter than one (mode
// 3), for a slice of sh.nvec columns of rows `stride` reals apart.
Shape odd_shape(size_t elem, uint32_t K)
{
    const size_t bytes = (size_t)K * elem;
    if (bytes < 16)
        return {4, 1, 3, K};
    const uint32_t nvec = (uint32_t)((bytes + 15) / 16);
    if (nvec > 128)
        return {64, 4, 2, K};
    if (nvec > 64)
        return {64, 2, 2, K};
    int lpr = 4;
    while ((uint32_t)lpr < nvec)
        lpr *= 2;
    return {lpr, 1, 2, K};
}

template <typename T, int FZ>
hipError_t run_sddmm_odd(const Shape &sh, const DevPlanView &P, const T *A, const T *B, T *C,
                         T *Y, const Streams &SS, uint32_t stride, uint32_t accum)
{
#define X(L, V, U, S, S2)                                                                         \
    if (sh.mode == 2 && sh.lpr == L && sh.vpl == V)                                               \
        return run_sddmm<T, L, V, U, S, 2, FZ>(P, A, B, C, Y, SS, sh.nvec, stride, accum);
    SPC3D_FOR_ODD_SHAPES(X)
#undef X
    if (sh.mode == 3)
        return run_sddmm<T, 4, 1, 16, 8, 3, FZ>(P, A, B, C, Y, SS, sh.nvec, stride, accum);
    return hipErrorInvalidValue;
}

// Rows over 4 KiB go slice by slice: whole 4 KiB slices of columns first (all 256
// vector slots of the 64 x 4 shape busy), then what is left of the row, each slice a
// launch over the whole pattern that adds its part of the dot products to C.
constexpr uint32_t kSliceBytes = 4096;

// FZ == 0: SDDMM.  FZ == 1, 2: SDDMM fused with the SpMM of the same pattern over
// the same B (hipErrorNotSupported for rows over 4 KiB).
template <typename T, int FZ>
hipError_t sddmm_typed(const DevPlanView &P, const void *A, const void *B, void *C, void *Y,
                       uint32_t K, const Streams &SS)
{
    const hipStream_t st = SS.main;
    if (P.nseg == 0)
        return hipSuccess;
    const Shape sh = pick_shape(sizeof(T), K);
    bool done = false;
    hipError_t e = hipSuccess;
    DevPlanView H;
    const void *low = nullptr;
    if (sh.mode == 0 && hot_view(P, sizeof(T), B, sh.nvec * 16, H, &low, st, &e)) {
#define X(L, V, U, S, S2)                                                                         \
    if (!done && sh.lpr == L && sh.vpl == V) {                                                    \
        e = run_sddmm<T, L, V, U, S, -1, FZ>(H, (const T *)A, (const T *)low, (T *)C, (T *)Y, SS,   \
                                             sh.nvec);                                            \
        done = true;                                                                              \
    }
        SPC3D_FOR_HOT_SHAPES(X)
#undef X
    }
    if (e != hipSuccess)
        return e;
#define X(L, V, U, S, S2)                                                                         \
    if (!done && sh.mode == 0 && sh.lpr == L && sh.vpl == V) {                                    \
        e = run_sddmm<T, L, V, U, S, 0, FZ>(P, (const T *)A, (const T *)B, (T *)C, (T *)Y, SS,    \
                                            sh.nvec);                                             \
        done = true;                                                                              \
    }
    SPC3D_FOR_SHAPES(X)
#undef X
#define X(L, V, U, S, S2)                                                                         \
    if (!done && sh.mode == 1 && sh.lpr == L && sh.vpl == V) {                                    \
        e = run_sddmm<T, L, V, U, S, 1, FZ>(P, (const T *)A, (const T *)B, (T *)C, (T *)Y, SS,    \
                                            sh.nvec);                                             \
        done = true;                                                                              \
    }
    SPC3D_FOR_RAGGED_SHAPES(X)
#undef X
    if (!done && sh.mode >= 2) {
        e = run_sddmm_odd<T, FZ>(sh, P, (const T *)A, (const T *)B, (T *)C, (T *)Y, SS, K, 0u);
        done = true;
    }
    if (!done) {
        if constexpr (FZ != 0) {
            return hipErrorNotSupported;
        } else {
            const uint32_t per = kSliceBytes / (uint32_t)sizeof(T);
            for (uint32_t at = 0; at < K && e == hipSuccess; at += per) {
                const uint32_t w = K - at < per ? K - at : per;
                e = run_sddmm_odd<T, 0>(odd_shape(sizeof(T), w), P, (const T *)A + at,
                                        (const T *)B + at, (T *)C, nullptr, SS, K, at != 0);
            }
        }
    }
    const hipError_t last = hipGetLastError();
    if (e != hipSuccess || last != hipSuccess)
        return e != hipSuccess ? e : last;
    return FZ != 0 ? launch_fixup<T>(P, (T *)Y, K, st) : hipSuccess;
}

template <typename T>
hipError_t run_spmm_odd(const Shape &sh, const DevPlanView &P, const T *X, T *Y,
                        const Streams &SS, uint32_t stride, size_t slice_off, uint32_t pstride)
{
#define X(L, V, U, S, S2)                                                                         \
    if (sh.mode == 2 && sh.lpr == L && sh.vpl == V)                                               \
        return run_spmm<T, L, V, U, S2, 2>(P, X, Y, SS, sh.nvec, stride, slice_off, pstride);
    SPC3D_FOR_ODD_SHAPES(X)
#undef X
    if (sh.mode == 3)
        return run_spmm<T, 4, 1, 16, 4, 3>(P, X, Y, SS, sh.nvec, stride, slice_off, pstride);
    return hipErrorInvalidValue;
}

// The SpMM of a plan whose partial-sum rows hold fewer than K columns: so many columns at a time,
// each time the segments and the fix-up, which leaves the partial-sum rows to the next.  Every
// column is summed as in the whole call: the same bits.
template <typename T>
hipError_t spmm_by_columns(const DevPlanView &P, const T *X, T *Y, uint32_t K, const Streams &SS)
{
    const uint32_t per = std::min(P.partial_cols, kSliceBytes / (uint32_t)sizeof(T));
    for (uint32_t at = 0; at < K; at += per) {
        const uint32_t w = std::min(K - at, per);
        hipError_t e = run_spmm_odd<T>(odd_shape(sizeof(T), w), P, X + at, Y + at, SS, K, 0, w);
        if (e == hipSuccess)
            e = hipGetLastError();
        if (e == hipSuccess)
            e = launch_fixup<T>(P, Y, K, SS.main, at, w);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

template <typename T>
hipError_t spmm_typed(const DevPlanView &P, const void *X_, void *Y, uint32_t K,
                      const Streams &SS)
{
    const hipStream_t st = SS.main;
    if (P.nseg == 0)
        return hipSuccess;
    if (P.partial_cols && P.partial_cols < K && P.nsplit)
        return spmm_by_columns<T>(P, (const T *)X_, (T *)Y, K, SS);
    const Shape sh = pick_shape(sizeof(T), K);
    bool done = false;
    hipError_t e = hipSuccess;
    DevPlanView H;
    const void *low = nullptr;
    if (sh.mode == 0 && hot_view(P, sizeof(T), X_, sh.nvec * 16, H, &low, st, &e)) {
#define X(L, V, U, S, S2)                                                                         \
    if (!done && sh.lpr == L && sh.vpl == V) {                                                    \
        e = run_spmm<T, L, V, U, S2, -1>(H, (const T *)low, (T *)Y, SS, sh.nvec);                  \
        done = true;                                                                              \
    }
        SPC3D_FOR_HOT_SHAPES(X)
#undef X
    }
    if (e != hipSuccess)
        return e;
#define X(L, V, U, S, S2)                                                                         \
    if (!done && sh.mode == 0 && sh.lpr == L && sh.vpl == V) {                                    \
        e = run_spmm<T, L, V, U, S2, 0>(P, (const T *)X_, (T *)Y, SS, sh.nvec);                   \
        done = true;                                                                              \
    }
    SPC3D_FOR_SHAPES(X)
#undef X
#define X(L, V, U, S, S2)                                                                         \
    if (!done && sh.mode == 1 && sh.lpr == L && sh.vpl == V) {                                    \
        e = run_spmm<T, L, V, U, S2, 1>(P, (const T *)X_, (T *)Y, SS, sh.nvec);                   \
        done = true;                                                                              \
    }
    SPC3D_FOR_RAGGED_SHAPES(X)
#undef X
    if (!done && sh.mode >= 2) {
        e = run_spmm_odd<T>(sh, P, (const T *)X_, (T *)Y, SS, K, 0, K);
        done = true;
    }
    if (!done) {
        // rows over 4 KiB, slice by slice (see sddmm_typed); the slices of Y and of the
        // partial-sum rows are disjoint
        const uint32_t per = kSliceBytes / (uint32_t)sizeof(T);
        for (uint32_t at = 0; at < K && e == hipSuccess; at += per) {
            const uint32_t w = K - at < per ? K - at : per;
            e = run_spmm_odd<T>(odd_shape(sizeof(T), w), P, (const T *)X_ + at, (T *)Y + at, SS, K,
                                at, K);
        }
    }
    if (e == hipSuccess)
        e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    return launch_fixup<T>(P, (T *)Y, K, st);
}

inline uint32_t stream_grid(uint64_t n)
{
    const uint64_t want = (n + kBlock - 1) / kBlock;
    const uint64_t cap = 256 * 32; // 32 blocks per CU keeps a grid-stride loop busy
    return (uint32_t)(want < 1 ? 1 : (want > cap ? cap : want));
}

} // namespace

hipError_t launch_sddmm(int dtype, const DevPlanView &P, const void *A, const void *B, void *C,
                        uint32_t K, const Streams &stream)
{
    return dtype == 1 ? sddmm_typed<double, 0>(P, A, B, C, nullptr, K, stream)
                      : sddmm_typed<float, 0>(P, A, B, C, nullptr, K, stream);
}

hipError_t launch_sddmm_spmm(int dtype, int chained, const DevPlanView &P, const void *A,
                             const void *B, void *C, void *Y, uint32_t K, const Streams &stream)
{
    if (dtype == 1)
        return chained ? sddmm_typed<double, 2>(P, A, B, C, Y, K, stream)
                       : sddmm_typed<double, 1>(P, A, B, C, Y, K, stream);
    return chained ? sddmm_typed<float, 2>(P, A, B, C, Y, K, stream)
                   : sddmm_typed<float, 1>(P, A, B, C, Y, K, stream);
}

hipError_t launch_spmm(int dtype, const DevPlanView &P, const void *X, void *Y, uint32_t K,
                       const Streams &stream)
{
    return dtype == 1 ? spmm_typed<double>(P, X, Y, K, stream)
                      : spmm_typed<float>(P, X, Y, K, stream);
}

uint32_t sweep_lanes(int dtype, uint32_t K)
{
    const uint64_t bytes = (uint64_t)K * (dtype == 1 ? 8 : 4);
    return bytes == 256 ? 16u : (bytes == 512 ? 32u : (bytes == 1024 ? 64u : 0u));
}
uint32_t sweep_lanes_any(int dtype, uint32_t K)
{
    const uint64_t bytes = (uint64_t)K * (dtype == 1 ? 8 : 4);
    return bytes <= 128 || bytes > 1024 ? 0 : (bytes <= 256 ? 16u : (bytes <= 512 ? 32u : 64u));
}
uint32_t sweep_groups(uint32_t lanes) { return lanes ? kSweepBlock / lanes : 0; }
uint32_t sweep_rows_per_tile(uint32_t lanes) { return lanes ? kSweepRowBytes / (lanes * 16) : 0; }
uint32_t sweep_max_blocks(uint32_t lanes) { return lanes ? kSweepPtrWords - 1 : 0; }

namespace {
template <typename T, int LPR, int ROWS>
void sweep_launch(bool spmm, const SweepView &S, const T *A, const T *B, T *out, uint32_t tile0,
                  uint32_t ntiles, hipStream_t stream)
{
    const HotAt hot = {S.ref_at, S.hot_at};
    if (spmm)
        hipLaunchKernelGGL((sweep_spmm_kernel<T, LPR, 16, ROWS>), dim3(ntiles), dim3(kSweepBlock), 0,
                           stream, S.ptr, S.tile_rows, S.col, S.lrow, (const T *)S.sval, S.pos, B,
                           out, S.nblocks, S.rows_per_tile, tile0, S.K, hot, S.slot, (T *)S.partial);
    else
        hipLaunchKernelGGL((sweep_sddmm_kernel<T, LPR, 16, ROWS>), dim3(ntiles), dim3(kSweepBlock), 0,
                           stream, S.ptr, S.tile_rows, S.col, S.lrow, (const T *)S.sval, S.pos, A,
                           B, out, S.nblocks, S.rows_per_tile, tile0, S.K, hot);
}
template <typename T, int LPR>
void sweep_launch_rows(SweepRows rows, bool spmm, const SweepView &S, const T *A, const T *B, T *out,
                       uint32_t tile0, uint32_t ntiles, hipStream_t stream)
{
    if (rows == kExact)
        sweep_launch<T, LPR, kExact>(spmm, S, A, B, out, tile0, ntiles, stream);
    else if (rows == kAny)
        sweep_launch<T, LPR, kAny>(spmm, S, A, B, out, tile0, ntiles, stream);
    else
        sweep_launch<T, LPR, kHot>(spmm, S, A, B, out, tile0, ntiles, stream);
}
template <typename T>
hipError_t sweep_run(bool spmm, const SweepView &S, const T *A, const T *B, T *out, hipStream_t stream,
                     bool hot = false)
{
    if (S.ntiles == 0)
        return hipSuccess;
    // what the kernels assume of the plan: the tile's rows and range bounds fit their LDS
    if ((S.lanes != 16 && S.lanes != 32 && S.lanes != 64) || S.per_launch == 0 ||
        S.rows_per_tile * S.lanes * 16 > kSweepRowBytes ||
        (uint64_t)S.nblocks + 1 > kSweepPtrWords || S.K * sizeof(T) < 16 ||
        S.K * sizeof(T) > S.lanes * 16 || (hot && S.K * sizeof(T) != S.lanes * 16))
        return hipErrorInvalidValue;
    const SweepRows rows = S.K * sizeof(T) != S.lanes * 16 ? kAny : (hot ? kHot : kExact);
    for (uint32_t t0 = 0; t0 < S.ntiles; t0 += S.per_launch) { // one generation per launch
        const uint32_t n = S.ntiles - t0 < S.per_launch ? S.ntiles - t0 : S.per_launch;
        if (S.lanes == 16)
            sweep_launch_rows<T, 16>(rows, spmm, S, A, B, out, t0, n, stream);
        else if (S.lanes == 32)
            sweep_launch_rows<T, 32>(rows, spmm, S, A, B, out, t0, n, stream);
        else
            sweep_launch_rows<T, 64>(rows, spmm, S, A, B, out, t0, n, stream);
    }
    return hipGetLastError();
}
// The tiles of a sliced plan: their columns are named as the plan's hot form names them, where it has one.
// The other rows' segments run beside the tiles: the tiles wait for the L2s and leave the fabric idle,
// short rows are the other way round, and a tile's workgroup leaves each SIMD registers for a wavefront of the
// short-segment launch.  That starts a few microseconds after the tiles, which need a CU each.
template <typename T>
hipError_t hub_run(bool spmm, DevPlanView P, const SweepView &S, const T *A, const T *B, T *out, T *stage,
                   const Streams &streams)
{
    SweepView v = S;
    const void *base = B;
    const bool hot = P.nhot != 0;
    if (hot) {
        DevPlanView H;
        hipError_t e = hipSuccess;
        if (!hot_view(P, sizeof(T), B, S.K * (uint32_t)sizeof(T), H, &base, streams.main, &e))
            return e != hipSuccess ? e : hipErrorNotSupported;
        P.hot_copied = true;
        v.ref_at = H.ref_at;
        v.hot_at = H.hot_at;
    }
    P.nnz = S.rest_entries;
    const bool beside = P.nseg && fork_aux(streams);
    const bool staged = !spmm && !S.pos;
    hipError_t e = sweep_run<T>(spmm, v, A, static_cast<const T *>(base), staged ? stage : out, streams.main, hot);
    if (P.nseg) {
        Streams own = streams;
        if (beside) {
            own.main = streams.aux;
            own.aux = nullptr;
        }
        const hipError_t r = spmm ? spmm_typed<T>(P, B, out, S.K, own)
                                  : sddmm_typed<T, 0>(P, A, B, out, nullptr, S.K, own);
        e = e == hipSuccess ? r : e;
    }
    if (e == hipSuccess && staged)
        hipLaunchKernelGGL((hub_home_kernel<T>), dim3((S.ntiles + 7) / 8 * 8 * kHomePieces), dim3(kBlock), 0,
                           streams.main, S.ptr, S.nblocks, S.ntiles, S.src, S.dst, (const T *)stage, out);
    const hipError_t launched = hipGetLastError();
    const hipError_t joined = beside ? join_aux(streams) : hipSuccess;
    return e != hipSuccess ? e : (launched != hipSuccess ? launched : joined);
}
} // namespace

hipError_t launch_sweep_sddmm(int dtype, const SweepView &S, const void *A, const void *B, void *C,
                              hipStream_t stream)
{
    return dtype == 1 ? sweep_run<double>(false, S, (const double *)A, (const double *)B, (double *)C, stream)
                      : sweep_run<float>(false, S, (const float *)A, (const float *)B, (float *)C, stream);
}

hipError_t launch_sweep_spmm(int dtype, const SweepView &S, const void *X, void *Y, hipStream_t stream)
{
    return dtype == 1 ? sweep_run<double>(true, S, nullptr, (const double *)X, (double *)Y, stream)
                      : sweep_run<float>(true, S, nullptr, (const float *)X, (float *)Y, stream);
}

hipError_t launch_hub_sddmm(int dtype, const DevPlanView &P, const SweepView &S, const void *A, const void *B,
                            void *out, void *stage, const Streams &streams)
{
    return dtype == 1 ? hub_run<double>(false, P, S, (const double *)A, (const double *)B, (double *)out,
                                        (double *)stage, streams)
                      : hub_run<float>(false, P, S, (const float *)A, (const float *)B, (float *)out,
                                       (float *)stage, streams);
}

hipError_t launch_hub_spmm(int dtype, const DevPlanView &P, const SweepView &S, const void *X, void *Y,
                           const Streams &streams)
{
    return dtype == 1 ? hub_run<double>(true, P, S, nullptr, (const double *)X, (double *)Y, nullptr, streams)
                      : hub_run<float>(true, P, S, nullptr, (const float *)X, (float *)Y, nullptr, streams);
}

hipError_t launch_split_sums(int dtype, const DevPlanView &P, void *Y, uint32_t K, hipStream_t stream)
{
    return dtype == 1 ? launch_fixup<double>(P, (double *)Y, K, stream)
                      : launch_fixup<float>(P, (float *)Y, K, stream);
}

hipError_t launch_first_cols(const Seg *segs, uint32_t n, const uint32_t *col, uint32_t *first_cols,
                             hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    const uint64_t threads = (uint64_t)n * kFirstCols;
    hipLaunchKernelGGL(first_cols_kernel, dim3((uint32_t)((threads + kBlock - 1) / kBlock)),
                       dim3(kBlock), 0, stream, segs, n, col, first_cols);
    return hipGetLastError();
}

namespace {
// Fewer results than this do not fill the chip with wavefronts of 1024 of them (6 M: the call 214 -> 217 us;
// level at 8.6 M, 2 % faster at 28 M).
constexpr uint64_t kGatherDeep = (uint64_t)8 << 20;
template <typename T>
void gather4_run(const void *in, const uint32_t *pos, void *out, uint64_t n, hipStream_t st)
{
    constexpr uint64_t deep = 64 * 4 * 4; // results of a deep workgroup's step
    if (n >= kGatherDeep)
        hipLaunchKernelGGL((gather4_kernel<T, 64, 4>), dim3((uint32_t)std::min<uint64_t>((n + deep - 1) / deep, 32768)),
                           dim3(64), 0, st, (const T *)in, pos, (T *)out, n);
    else
        hipLaunchKernelGGL((gather4_kernel<T, kBlock, 1>), dim3(stream_grid((n + 3) / 4)), dim3(kBlock), 0, st,
                           (const T *)in, pos, (T *)out, n);
}
} // namespace

hipError_t launch_unstage(int dtype, const void *in, const uint32_t *pos, void *out, uint64_t n,
                          hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    if (dtype == 1)
        gather4_run<double>(in, pos, out, n, stream);
    else
        gather4_run<float>(in, pos, out, n, stream);
    return hipGetLastError();
}

hipError_t launch_unstage_pairs(int dtype, const void *stage, const uint32_t *src,
                                const uint32_t *dst, void *out, uint64_t n, hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    const uint64_t want = (n + (uint64_t)kBlock * 4 - 1) / ((uint64_t)kBlock * 4);
    const uint32_t grid = (uint32_t)(want > 65536 ? 65536 : want);
    if (dtype == 1)
        hipLaunchKernelGGL((unstage_pairs_kernel<double>), dim3(grid), dim3(kBlock), 0, stream,
                           (const double *)stage, src, dst, (double *)out, n);
    else
        hipLaunchKernelGGL((unstage_pairs_kernel<float>), dim3(grid), dim3(kBlock), 0, stream,
                           (const float *)stage, src, dst, (float *)out, n);
    return hipGetLastError();
}

uint32_t two_pass_lds_bytes() { return kTwoPassBytes; }

uint32_t two_pass_tile_elems(int dtype)
{
    return dtype == 1 ? two_pass_tile<double>() : two_pass_tile<float>();
}

hipError_t launch_unpermute_two_pass(int dtype, const void *stage, void *mid, const uint16_t *l1,
                                     const uint32_t *dst1, const uint16_t *l2, void *out, uint64_t n,
                                     hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    const uint64_t T = two_pass_tile_elems(dtype);
    const uint32_t grid = (uint32_t)((n + T - 1) / T);
    if (dtype == 1) {
        hipLaunchKernelGGL((unpermute_pass1_kernel<double>), dim3(grid), dim3(kTwoPassBlock), 0,
                           stream, (const double *)stage, l1, dst1, (double *)mid, n);
        hipLaunchKernelGGL((unpermute_pass2_kernel<double>), dim3(grid), dim3(kTwoPassBlock), 0,
                           stream, (const double *)mid, l2, (double *)out, n);
    } else {
        hipLaunchKernelGGL((unpermute_pass1_kernel<float>), dim3(grid), dim3(kTwoPassBlock), 0,
                           stream, (const float *)stage, l1, dst1, (float *)mid, n);
        hipLaunchKernelGGL((unpermute_pass2_kernel<float>), dim3(grid), dim3(kTwoPassBlock), 0,
                           stream, (const float *)mid, l2, (float *)out, n);
    }
    return hipGetLastError();
}

hipError_t launch_scatter_vals(int dtype, const void *in, const uint32_t *perm, void *out,
                               uint64_t n, hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    if (dtype == 1)
        hipLaunchKernelGGL((scatter_kernel<double>), dim3(stream_grid(n)), dim3(kBlock), 0, stream,
                           (const double *)in, perm, (double *)out, n);
    else
        hipLaunchKernelGGL((scatter_kernel<float>), dim3(stream_grid(n)), dim3(kBlock), 0, stream,
                           (const float *)in, perm, (float *)out, n);
    return hipGetLastError();
}

hipError_t launch_gather_vals(int dtype, const void *in, const uint32_t *perm, void *out,
                              uint64_t n, hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    if (dtype == 1)
        hipLaunchKernelGGL((gather_kernel<double>), dim3(stream_grid(n)), dim3(kBlock), 0, stream,
                           (const double *)in, perm, (double *)out, n);
    else
        hipLaunchKernelGGL((gather_kernel<float>), dim3(stream_grid(n)), dim3(kBlock), 0, stream,
                           (const float *)in, perm, (float *)out, n);
    return hipGetLastError();
}

namespace {
inline dim3 rows_grid(uint32_t n, uint32_t per)
{
    return dim3((uint32_t)std::min(((uint64_t)n + per - 1) / per, kRowsMaxBlocks));
}

template <typename T, RowUnit UNIT, int LPR, int U>
void rows_launch_ahead(int op, char *panel, const RowMapView &M, uint32_t n, uint32_t units,
                       uint64_t bytes, char *buf, hipStream_t st)
{
    const dim3 grid = rows_grid(n, kBlock / LPR * U), block(kBlock);
    if (op == 0)
        hipLaunchKernelGGL((rows_pack_kernel<T, UNIT, LPR, U>), grid, block, 0, st, panel, M.rows, n,
                           units, bytes, buf);
    else
        hipLaunchKernelGGL((rows_unpack_kernel<T, UNIT, LPR, U, false, 1>), grid, block, 0, st, panel,
                           (const u32x4 *)M.dests, M.slots, n, units, bytes, buf);
}

template <typename T, RowUnit UNIT, int LPR, int D>
void rows_launch_sum(char *panel, const RowMapView &M, uint32_t units, uint64_t bytes, char *buf,
                     hipStream_t st)
{
    hipLaunchKernelGGL((rows_unpack_kernel<T, UNIT, LPR, 1, true, D>),
                       rows_grid(M.nuniq, kBlock / LPR), dim3(kBlock), 0, st, panel,
                       (const u32x4 *)M.dests, M.slots, M.nuniq, units, bytes, buf);
}

template <typename T, RowUnit UNIT, int LPR>
void rows_launch(int op, char *panel, const RowMapView &M, uint32_t units, uint64_t bytes, char *buf,
                 hipStream_t st)
{
    // The slots of a row are a chain of two loads each, so as many of them go together as rows have
    // on average: 6,400 rows of 26 slots, fp32 K = 4, take 12 / 8.6 / 6.6 / 5.6 us by ones, twos,
    // fours and eights; 287 k rows of 2.7, K = 8, 24 / 21 / 22.5 / 28.
    if (op == 2) {
        if (M.nslots >= 8 * (uint64_t)M.nuniq)
            rows_launch_sum<T, UNIT, LPR, 8>(panel, M, units, bytes, buf, st);
        else if (M.nslots >= 3 * (uint64_t)M.nuniq)
            rows_launch_sum<T, UNIT, LPR, 4>(panel, M, units, bytes, buf, st);
        else
            rows_launch_sum<T, UNIT, LPR, 2>(panel, M, units, bytes, buf, st);
        return;
    }
    const uint32_t n = op == 0 ? M.nslots : M.nuniq;
    if (n / (kBlock / LPR * kRowsAhead) < kRowsMinBlocks)
        rows_launch_ahead<T, UNIT, LPR, 1>(op, panel, M, n, units, bytes, buf, st);
    else
        rows_launch_ahead<T, UNIT, LPR, kRowsAhead>(op, panel, M, n, units, bytes, buf, st);
}

template <typename T>
hipError_t rows_typed(int op, void *panel, const RowMapView &M, uint32_t K, void *buf, hipStream_t st)
{
    const uint64_t bytes = (uint64_t)K * sizeof(T);
    char *p = (char *)panel, *q = (char *)buf;
    if (bytes < 16) { // at most three reals
        rows_launch<T, kElem, 4>(op, p, M, K, bytes, q, st);
        return hipGetLastError();
    }
    const uint32_t units = (uint32_t)((bytes + 15) / 16);
#define SPC3D_ROWS(UNIT)                                                                          \
    do {                                                                                          \
        if (units == 1)                                                                           \
            rows_launch<T, UNIT, 1>(op, p, M, units, bytes, q, st);                               \
        else if (units == 2)                                                                      \
            rows_launch<T, UNIT, 2>(op, p, M, units, bytes, q, st);                               \
        else if (units <= 4)                                                                      \
            rows_launch<T, UNIT, 4>(op, p, M, units, bytes, q, st);                               \
        else if (units <= 8)                                                                      \
            rows_launch<T, UNIT, 8>(op, p, M, units, bytes, q, st);                               \
        else if (units <= 16)                                                                     \
            rows_launch<T, UNIT, 16>(op, p, M, units, bytes, q, st);                              \
        else if (units <= 32)                                                                     \
            rows_launch<T, UNIT, 32>(op, p, M, units, bytes, q, st);                              \
        else                                                                                      \
            rows_launch<T, UNIT, 64>(op, p, M, units, bytes, q, st);                              \
    } while (0)
    if (bytes % 16 == 0)
        SPC3D_ROWS(kVec);
    else
        SPC3D_ROWS(kLoose);
#undef SPC3D_ROWS
    return hipGetLastError();
}
} // namespace

hipError_t launch_rows(int op, int dtype, void *panel, const RowMapView &M, uint32_t K, void *buf,
                       hipStream_t stream)
{
    if (M.nslots == 0 || K == 0)
        return hipSuccess;
    return dtype == 1 ? rows_typed<double>(op, panel, M, K, buf, stream)
                      : rows_typed<float>(op, panel, M, K, buf, stream);
}

hipError_t launch_xcc_probe(uint32_t *out, uint32_t nblocks, hipStream_t stream)
{
    if (nblocks == 0)
        return hipSuccess;
    hipLaunchKernelGGL(xcc_probe_kernel, dim3(nblocks), dim3(64), 0, stream, out);
    return hipGetLastError();
}

hipError_t launch_probe_cols(uint32_t *col, uint64_t n, uint32_t mode, uint32_t base,
                             uint32_t modulus, uint32_t ncols, hipStream_t stream, const uint32_t *hot)
{
    if (n == 0)
        return hipSuccess;
    hipLaunchKernelGGL(probe_cols_kernel, dim3(stream_grid(n)), dim3(kBlock), 0, stream, col, n,
                       mode, base, modulus, ncols, hot);
    return hipGetLastError();
}

hipError_t launch_copy(void *dst, const void *src, uint64_t bytes, hipStream_t stream)
{
    if (bytes == 0)
        return hipSuccess;
    const uint64_t nvec = bytes / 16;
    hipLaunchKernelGGL(copy_kernel, dim3(stream_grid((nvec + 3) / 4 + 1)), dim3(kBlock), 0, stream,
                       (u32x4 *)dst, (const u32x4 *)src, nvec, (uint32_t)(bytes % 16));
    return hipGetLastError();
}

hipError_t launch_fill(int dtype, void *p, uint64_t n, double value, hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    if (dtype == 1)
        hipLaunchKernelGGL((fill_kernel<double>), dim3(stream_grid(n)), dim3(kBlock), 0, stream,
                           (double *)p, n, value);
    else
        hipLaunchKernelGGL((fill_kernel<float>), dim3(stream_grid(n)), dim3(kBlock), 0, stream,
                           (float *)p, n, (float)value);
    return hipGetLastError();
}

const char *kernel_variant(int dtype, uint32_t K)
{
    static thread_local char buf[64];
    const Shape sh = pick_shape(dtype == 1 ? 8 : 4, K);
    if (K == 0)
        snprintf(buf, sizeof buf, "none (no columns)");
    else if (sh.lpr == 0)
        snprintf(buf, sizeof buf, "seg<%s,LPR=64,VPL=4,odd> per 4 KiB slice",
                 dtype == 1 ? "f64" : "f32");
    else
        snprintf(buf, sizeof buf, "seg<%s,LPR=%d,VPL=%d%s>", dtype == 1 ? "f64" : "f32", sh.lpr,
                 sh.vpl, sh.mode == 1 ? ",ragged" : (sh.mode == 2 ? ",odd" : (sh.mode == 3 ? ",thin" : "")));
    return buf;
}

} // namespace spc3d
