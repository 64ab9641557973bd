// MFMA tile-GEMM kernel template for gfx950 (CDNA4, wave64).
//
// One source, instantiated by -D macros (one instance = one point of the tuner's search space):
//   HRN_DTYPE   0: fp16 x fp16 -> fp32 accumulate -> fp16 store      (ops/cuda/dense.py:4-54)
//               1: uint8 x int8 -> int32 accumulate -> int32 store   (ops/x86/dense.py:6-32)
//   HRN_OP      0: GEMM / batch_matmul   C[b,i,j] = sum_k A[b,i,k] * B[b,j,k]
//               1: conv2d NHWC x KRSC as implicit GEMM (M = n*ho*wo, N = co, K = kh*kw*ci)
//   HRN_BM/BN   workgroup tile, HRN_BKB bytes of K per LDS row, HRN_WM x HRN_WN wave grid,
//   HRN_MFMA    32 | 16 (MFMA tile edge), HRN_STAGES LDS stages, HRN_SWZ LDS chunk swizzle,
//   HRN_EPI     0 result of any alignment, staged where there is room, 1 LDS-staged epilogue with 16-byte coalesced
//               stores, 2 the same with half-width staging strips, HRN_WPE waves-per-SIMD hint, HRN_CONVWIN conv input window in LDS, HRN_PERSIST persistent
//               launch, HRN_SPLITK K split over several workgroups whose partial sums the last one adds up.
//
// Data movement: both operands are K-contiguous, so a tile is a set of rows of HRN_BKB bytes.
// Rows are cut into 16-byte chunks; every lane moves one chunk per load straight from HBM/L2
// into LDS (buffer_load_dwordx4 ... lds), one wave instruction filling 1 KiB of consecutive LDS.
// The chunk a lane fetches is XOR-swizzled so that the MFMA operand reads (ds_read_b128, one
// 16-byte chunk per lane) spread over all LDS banks.  A lane's byte offset inside its row never
// changes; the k-tile is selected by the scalar offset operand of the load, so the k-loop spends
// no vector instruction on addresses.  Out-of-range rows and conv halo taps are fetched with an
// out-of-range lane offset, the dummy tiles past the end of K through a zero-length buffer
// descriptor: the buffer unit turns both into zeros.
//
// Pipeline: HRN_STAGES tiles are in flight.  The barrier that publishes tile t+1 sits before the
// last k-step of tile t, so operand fragments of the next tile are already being read while the
// last MFMAs of the current tile run; fragments are double-buffered in registers and read in the
// order the MFMAs of the next step consume them (all of B, then A row-tile by row-tile).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "hrn_args.h"

#ifndef HRN_DTYPE
#error "instantiate with -DHRN_DTYPE=... (see hrn_api.cpp)"
#endif


namespace {

constexpr int DT = HRN_DTYPE;
constexpr int OP = HRN_OP;
constexpr int BM = HRN_BM, BN = HRN_BN, BKB = HRN_BKB;
constexpr int WM = HRN_WM, WN = HRN_WN, MT = HRN_MFMA, NS = HRN_STAGES, SWZ = HRN_SWZ;
// Conv window mode (HRN_OP=1, stride 1, dilation 1, 'same' padding): instead of fetching an im2col tile of A for every
// filter tap, the workgroup loads ONCE the window of input pixels its BM output pixels can reach (a contiguous range
// of BM + 2*(pad_h*W + pad_w) pixels, all channels) and every tap reads its operand fragments from that window at a row offset
// of r*W + s pixels; taps that fall into the padding are masked to zero in registers.  Only B (the filter) streams
// through the LDS stages.  The window lives in dynamic LDS; the staged epilogue reuses it once the last tap is read.
#ifndef HRN_CONVWIN
#define HRN_CONVWIN 0
#endif
constexpr bool CW = (HRN_CONVWIN != 0);
// Persistent mode: the launch has fewer workgroups than output tiles and every workgroup walks tiles
// blockIdx.x, blockIdx.x + gridDim.x, ...  The k-tiles of all its output tiles form ONE stream through the LDS
// stages, so the first k-tiles of the next output tile are already being fetched while the current tile's result is
// stored.  The stores are buffer stores issued unconditionally (masked lanes get an out-of-range offset), so every
// wave has a known number of them in the vector-memory counter and the waits on the following tile fetches can
// allow for them instead of draining them.
#ifndef HRN_PERSIST
#define HRN_PERSIST 0
#endif
constexpr bool PERS = (HRN_PERSIST != 0);
// Split-K: the grid holds `split` workgroups for every tile, side by side; number z of them multiplies k-tiles
// [z*kt_per_slice, (z+1)*kt_per_slice) and stores its raw fp32 / int32 partial sums in slice z of a workspace, tile by tile; the one that
// finishes a tile last adds them up (fold_slices).  Where the workspace has no room for the arrivals, slices are row-major and a second
// kernel (splitk_reduce_kernel) adds them up.
#ifndef HRN_SPLITK
#define HRN_SPLITK 0
#endif
constexpr bool SPLITK = (HRN_SPLITK != 0);
// uint8 path: 1 = the column sums of B (sum_k B[n,k], what the (u8 - 128) x s8 product is short of, times 128) come
// from the caller (HrnKArgs.bsum: one int32 per column and batch entry, a property of the weights alone) instead of
// being added up in the k-loop from the B fragments.
#ifndef HRN_COLSUM
#define HRN_COLSUM 0
#endif
constexpr bool COLSUM = (HRN_DTYPE == 1) && (HRN_COLSUM != 0);
// the results leave with the non-temporal hint: C is written once and not read by this kernel, and a round's 8 MiB of it
// per XCD would otherwise push the operand slabs of the next round out of the 4 MiB L2 (split-K partial sums go out at device scope
// instead, whoever adds them up: the other XCDs' slices are read from memory).  Staged results go without it where row_lines says so; those
// straight from the accumulators, which no strip gathers, keep it whatever their rows
#ifndef HRN_NTSTORE
#define HRN_NTSTORE 0
#endif
constexpr bool NTS = (HRN_NTSTORE != 0) && (HRN_SPLITK == 0);
// Issue order of a k-step: 1 = the source order of the row groups is pinned (a scheduling fence after every row of
// MFMAs), 0 = the compiler interleaves on its own, guided by group hints (one LDS read per few MFMAs).  Tiles that
// PHASED (below) takes run the phased schedule whatever this says.
#ifndef HRN_SCHED
#define HRN_SCHED 1
#endif
constexpr int SCHED = HRN_SCHED;
#ifndef HRN_LSPREAD
#define HRN_LSPREAD 2
#endif
constexpr int LSPREAD = HRN_LSPREAD;
static_assert(LSPREAD >= 0 && LSPREAD <= 3, "load spread");
constexpr int ES = (DT == 0) ? 2 : 1;                  // input element bytes
constexpr int OES = (DT == 0 && !SPLITK) ? 2 : 4;      // output element bytes
constexpr int NW = WM * WN, NT = NW * 64;
constexpr int CPR = BKB / 16;               // 16-byte chunks per tile row
constexpr int RPI = 64 / CPR;               // tile rows one wave load instruction covers
constexpr int A_LPW = CW ? 0 : (BM / RPI) / NW;   // load instructions per wave per tile
constexpr int B_LPW = (BN / RPI) / NW;
constexpr int LPT = A_LPW + B_LPW;          // vector memory ops per lane per tile
constexpr int KSB = (MT == 32) ? 32 : 64;   // bytes of K one MFMA consumes
constexpr int KS = BKB / KSB;               // MFMA k-steps per tile
constexpr int CPS = KSB / 16;               // chunks per k-step (= 64 / MT)
constexpr int WTM = BM / WM, WTN = BN / WN;
constexpr int TM = WTM / MT, TN = WTN / MT;
constexpr int A_BYTES = CW ? 0 : BM * BKB, B_BYTES = BN * BKB, STAGE_BYTES = A_BYTES + B_BYTES;
constexpr int ACC_N = (MT == 32) ? 16 : 4;
constexpr uint32_t OOB = 0x80000000u;

static_assert(BKB == 64 || BKB == 128 || BKB == 256, "BKB");
static_assert(MT == 32 || MT == 16, "MFMA");
static_assert(KS >= 1, "k-steps per tile");
static_assert((WM & (WM - 1)) == 0, "wave rows must be a power of two");
static_assert((CW || ((BM / RPI) % NW == 0 && A_LPW >= 1)) && (BN / RPI) % NW == 0 && B_LPW >= 1, "loads per wave");
static_assert(!CW || OP == 1, "window mode is a conv2d load path");
static_assert(BM % (WM * MT) == 0 && BN % (WN * MT) == 0, "wave tile");
static_assert(NS >= 2 && NS <= 5, "stages");
// HRN_EPI = 0 stages fp16 results as well, where the strips fit into the LDS of the stages: lanes that store what the MFMAs leave them
// with write 8 bytes here and there, 32 bytes of a row per instruction at best, and with the non-temporal hint each of them on
// its own.  (32-bit results go out 16 bytes at a time either way; staged, one wave's 64x64 tile of them takes 0.4 us longer.)  Unlike HRN_EPI = 1
// it takes rows of any alignment.  fp16, 128x128 tiles, stored non-temporally / not: 2000x2000x1024 25.4 / 16.4 -> 13.0 us, 3000x2304x512 34.5 / 15.6 -> 11.9, 4000x1024x512 19.7 / 13.1 -> 8.2.
constexpr bool STAGE_DIRECT = HRN_EPI == 0 && OES == 2 && !CW && !PERS && (MT * (WTN * OES / 16)) % 64 == 0 &&
                              NW * MT * (WTN * OES + 16) <= NS * STAGE_BYTES;
constexpr int EPI = STAGE_DIRECT ? 1 : HRN_EPI;
// LDS-staged epilogue: per wave a strip of MT rows x WTN outputs, rows padded by 16 bytes; in front of the strips the
// uint8 path keeps the column sums of B, one row of BN sums per wave row (each wave row sums its share of the k-steps)
// (HRN_EPI = 2: strips of half the wave tile's width, filled and written out twice per row-tile - half the LDS)
constexpr int ESPLIT = (EPI == 2) ? 2 : 1;
constexpr int SW = WTN / ESPLIT;            // outputs per strip row
constexpr int EPI_PITCH = SW * OES + 16;
constexpr int EPI_BASE = (DT == 1) ? ((WM * BN * 4 + 1023) / 1024) * 1024 : 0;
constexpr int EPI_BYTES = (EPI >= 1) ? EPI_BASE + NW * MT * EPI_PITCH : 0;
// the epilogue region (column sums + strips) reuses the stages (window mode: the window), except in persistent mode
// where the stages stay live
constexpr int EPI_OFF = PERS ? NS * STAGE_BYTES : 0;
constexpr int LDS_BYTES = PERS ? NS * STAGE_BYTES + EPI_BYTES
                               : ((CW || NS * STAGE_BYTES > EPI_BYTES) ? NS * STAGE_BYTES : EPI_BYTES);
constexpr int STORES_PER_TILE = (EPI >= 1) ? TM * ESPLIT * (MT * (SW * OES / 16) / 64) : 0;   // store instructions per wave per output tile
static_assert(EPI >= 0 && EPI <= 2 && TN % ESPLIT == 0, "epilogue kind");
// Channels-first epilogue (CHW kernels): strips of MT channels x CSW pixels (whole MFMA tiles, at most 64 pixels), as many as
// LDS holds beside what stays in it (window mode: the stages)
constexpr int chw_tiles() {
    for (int d = 64 / MT; d > 1; --d)
        if (TM % d == 0 && EPI_BASE + NW * MT * (d * MT * OES + 16) + (CW ? NS * STAGE_BYTES : 0) <= 163840) return d;
    return 1;
}
constexpr int CSW = chw_tiles() * MT;
constexpr int CHW_PITCH = CSW * OES + 16;
constexpr int CHW_BYTES = EPI_BASE + NW * MT * CHW_PITCH;
constexpr int CHW_LDS_BYTES = (CW || NS * STAGE_BYTES > CHW_BYTES) ? NS * STAGE_BYTES : CHW_BYTES;
constexpr bool HAS_CHW = OP == 1 && !PERS && !SPLITK && CHW_BYTES + (CW ? NS * STAGE_BYTES : 0) <= 163840;

static_assert(!PERS || (EPI >= 1 && !CW && !SPLITK && KS % 2 == 0), "persistent mode: staged epilogue, even k-steps");
static_assert(!PERS || (NS - 2) * LPT + STORES_PER_TILE <= 63, "persistent mode: vmcnt range");
static_assert(!SPLITK || !CW, "split-K uses the im2col load path");
static_assert(LDS_BYTES <= 163840, "LDS");
static_assert(EPI == 0 || (MT * (SW * OES / 16)) % 64 == 0, "staged epilogue: a strip must split into whole wave stores");
static_assert(SWZ == 0 || (CPR << (SWZ - 1)) <= MT, "swizzle period must fit in one MFMA tile");
static_assert((NS - 1) * LPT <= 63, "vmcnt range");
static_assert(NT <= 1024, "threads");
static_assert(DT == 0 || NS * STAGE_BYTES >= WM * BN * 4, "column sums must fit the stages");

// Phased schedule ("---- phased schedule" below) instead of the row-by-row one: 256x256 tiles of 128-byte rows in two
// stages on 8 waves in a 2x4 or 4x2 grid.  These are the tiles of the large products, where the matrix pipes decide;
// same card, 8192^3, row-by-row / phased: fp16 778 / 742 us (2x4, 16x16 MFMAs; 32x32: 884 / 842), u8 x s8 434 / 403 us
// (4x2), fp16 4096^3 101.5 / 97.5.  The grids 8x1 and 1x8 would need 152 fragment registers beside the 128 accumulators, and
// the uint8 path has no room for in-loop column sums, so both stay with the row-by-row schedule.
constexpr bool PHASED = OP == 0 && BM == 256 && BN == 256 && BKB == 128 && NS == 2 && NW == 8 && (WM == 2 || WM == 4) &&
                        !PERS && !SPLITK && (DT == 0 || COLSUM);

// Deep kernels: an instance of two stages with a third one, for launches that leave its LDS free anyway and whose operands do
// not come from a near L2 (hrn_api.cpp, deep_fits).
constexpr int DEEP_NS = 3;
constexpr bool HAS_DEEP = NS == 2 && !CW && !PERS && DEEP_NS * STAGE_BYTES <= 163840 && (DEEP_NS - 1) * LPT <= 63;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

template <int N> struct AccT;
template <> struct AccT<16> { using F = v16f; using I = v16i; };
template <> struct AccT<4> { using F = v4f; using I = v4i; };
using acc_t = typename std::conditional<DT == 0, typename AccT<ACC_N>::F, typename AccT<ACC_N>::I>::type;

__device__ __forceinline__ int div_by(int n, HrnDiv d) { return (int)d((uint32_t)n); }

__device__ __forceinline__ int swz_of_row(int row) {
    if (SWZ == 0) return 0;
    return (row >> (SWZ - 1)) & (CPR - 1);
}

// s_waitcnt encodings for gfx9: vmcnt[3:0]|[15:14], expcnt[6:4], lgkmcnt[11:8]
template <int VM, int LGKM>
__device__ __forceinline__ void wait_and_barrier() {
    constexpr int vm = VM > 63 ? 63 : VM;
    constexpr int imm = (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | ((LGKM & 15) << 8);
    asm volatile("s_waitcnt %0\n\ts_barrier" ::"n"(imm) : "memory");
}

template <int VM, int LGKM>
__device__ __forceinline__ void wait_only() {
    constexpr int vm = VM > 63 ? 63 : VM;
    constexpr int imm = (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | ((LGKM & 15) << 8);
    asm volatile("s_waitcnt %0" ::"n"(imm) : "memory");
}

typedef __amdgpu_buffer_rsrc_t rsrc_t;
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
constexpr int AGENT_SCOPE = 16;             // cache policy (sc1): a load or store that all XCDs of the device see
// pieces of a result in memory: rows and results start at any element with HRN_EPI = 0 and where split-K slices are added up.  (The
// attribute belongs to these names: template arguments and `auto` drop it, so stores name the type.)
typedef v4i out16_t __attribute__((aligned(HRN_EPI == 0 ? OES : 16)));
typedef long out8_t __attribute__((aligned(HRN_EPI == 0 ? OES : 8)));
typedef v4h sum8_t __attribute__((aligned(2)));
typedef v4i sum16_t __attribute__((aligned(4)));
static_assert(HRN_EPI != 0 || (alignof(out16_t) == OES && alignof(out8_t) == OES), "results of any alignment");

// raw buffer (stride 0): a lane offset >= `bytes` reads as zero instead of touching memory (the scalar offset of a
// load is not part of that check)
__device__ __forceinline__ rsrc_t make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ void load_chunk_to_lds(rsrc_t rsrc, char* lds_wave_base, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)lds_wave_base,
                                             16, (int)voff, (int)soff, 0, 0);
}

__device__ __forceinline__ v16f mfma(v4i x, v4i y, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, x), __builtin_bit_cast(v8h, y), c, 0, 0, 0);
}
__device__ __forceinline__ v4f mfma(v4i x, v4i y, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, x), __builtin_bit_cast(v8h, y), c, 0, 0, 0);
}
__device__ __forceinline__ v16i mfma(v4i x, v4i y, v16i c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(x, y, c, 0, 0, 0);
}
__device__ __forceinline__ v4i mfma(v4i x, v4i y, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(x, y, c, 0, 0, 0);
}

// Scheduling hints of one k-step (HRN_SCHED = 0): NR groups of {1 LDS read, NV/NR buffer loads, NMM/NR MFMAs}.
template <int R, int NR, int NMM, int NV>
__device__ __forceinline__ void sched_hint() {
    if constexpr (R < NR) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        constexpr int v = (NV * (R + 1)) / NR - (NV * R) / NR;
        if constexpr (v > 0) __builtin_amdgcn_sched_group_barrier(0x020, v, 0);
        constexpr int mm = (NMM * (R + 1)) / NR - (NMM * R) / NR;
        if constexpr (mm > 0) __builtin_amdgcn_sched_group_barrier(0x008, mm, 0);
        sched_hint<R + 1, NR, NMM, NV>();
    }
}

// The body of all kernels of an instance.
//   CHW (conv): the result is stored channels first, see HrnKArgs::out_plane.  Such a result used to be the row-major one,
// transposed by a pass of its own that read and wrote all of it once more.  The MFMAs are issued with their operands
// exchanged, so that a lane holds 4 consecutive pixels of one channel.
//   EXPAND (conv): the input of a transposed convolution, HrnKArgs::expand_shift; the zeros are not in memory.
//   NCHW transposed conv 16 x 56x56x64 -> 111x111x128, stride 2: 77 us with the passes around the kernel, 34 us without
// (50 MB of result).
//   DEEP: three stages instead of HRN_STAGES.
// How the arguments are handed in decides what the compiler does with the scalar registers.  Persistent instances take them by
// value (fp16 192 x 512x512x64: 4 spills and 24 idle instructions instead of 7 and 41, 21.3 us instead of 21.55), the others by
// reference (u8 x s8 8192^3: 418 us instead of 425; the rest of the cases within their spread either way).
using KArgs = typename std::conditional<OP == 1, HrnConvArgs, HrnKArgs>::type;
using BodyArgs = typename std::conditional<PERS, const KArgs, const KArgs&>::type;
template <bool CHW, bool EXPAND, bool DEEP, class Args>       // (Args: BodyArgs, a parameter so that a product need not have a conv's)
__device__ __forceinline__ void hrn_mfma_body(Args a) {
    constexpr int NS = DEEP ? DEEP_NS : HRN_STAGES;
    constexpr int OWN_LDS = CHW ? CHW_LDS_BYTES : LDS_BYTES;
    constexpr int KERNEL_LDS = (DEEP && NS * STAGE_BYTES > OWN_LDS) ? NS * STAGE_BYTES : OWN_LDS;
    constexpr bool DYN_LDS = DEEP && OP == 0;
    __shared__ __attribute__((aligned(1024))) char own_lds[DYN_LDS ? 1024 : KERNEL_LDS];
    extern __shared__ __attribute__((aligned(1024))) char win[];   // window mode: input window, later the epilogue region; DYN_LDS: all of it
    char* const lds = DYN_LDS ? win : own_lds;

    // every argument the start of the kernel needs, fetched at once: left to itself the compiler reads them where they are
    // used and waits for memory several times before the first load is out (1700 - 1900 cycles, 850 like this)
    if constexpr (TM * TN * ACC_N < 256) {      // (not where every register holds an accumulator)
        asm volatile("" ::"s"(a.A), "s"(a.B), "s"(a.C), "s"(a.M), "s"(a.N), "s"(a.K), "s"(a.ldb), "s"(a.ldc), "s"(a.tiles_m), "s"(a.tiles_n),
                     "s"(a.group_m), "s"(a.by_group.m), "s"(a.by_group.shift), "s"(a.by_gm.m), "s"(a.by_gm.shift), "s"(a.by_gm_last.m),
                     "s"(a.by_gm_last.shift));
        if constexpr (OP == 0) asm volatile("" ::"s"(a.lda), "s"(a.sA), "s"(a.sB), "s"(a.sC), "s"(a.batch), "s"(a.by_tiles.m), "s"(a.by_tiles.shift));
        if constexpr (OP == 1)
            asm volatile("" ::"s"(a.H), "s"(a.W), "s"(a.CI), "s"(a.HO), "s"(a.WO), "s"(a.KH), "s"(a.KW), "s"(a.cstride), "s"(a.cpad), "s"(a.cdil),
                         "s"(a.cstride_w), "s"(a.cpad_w), "s"(a.cdil_w), "s"(a.by_hw.m), "s"(a.by_hw.shift), "s"(a.by_wo.m), "s"(a.by_wo.shift));
        if constexpr (OP == 1 && !CW)
            asm volatile("" ::"s"(a.by_kwci.m), "s"(a.by_kwci.shift), "s"(a.by_ci.m), "s"(a.by_ci.shift), "s"(a.px), "s"(a.kw_end), "s"(a.tap_bytes),
                         "s"(a.taprow_bytes), "s"(a.carry_ci), "s"(a.d_ox), "s"(a.d_oy), "s"(a.x_step), "s"(a.y_step), "s"(a.off_step), "s"(a.x_row), "s"(a.row_bytes),
                         "s"(a.y_img), "s"(a.img_bytes));
        if constexpr (CW) asm volatile("" ::"s"(a.by_cpp.m), "s"(a.by_cpp.shift));
        if constexpr (SPLITK) asm volatile("" ::"s"(a.split), "s"(a.kt_per_slice), "s"(a.by_split.m), "s"(a.by_split.shift));
        if constexpr (COLSUM) asm volatile("" ::"s"(a.bsum));
    }
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm_idx = wave / WN, wn_idx = wave % WN;

    const int tiles_mn = a.tiles_m * a.tiles_n;
    const int batch = OP == 1 ? 1 : a.batch;          // (the images of a conv are rows of one product)
    const int total = tiles_mn * batch;               // output tiles (of one K slice)
    const uint32_t Kb = (uint32_t)a.K * ES;           // bytes of K
    const int KT_all = (Kb + BKB - 1) / BKB;
    int first_pid = blockIdx.x, slice = 0;
    if constexpr (SPLITK) {
        // Eighths of the (tile, slice) pairs, one per XCD: the slices of a tile count and fold where most of their partial sums were
        // written, and tiles side by side, which read the same rows of B, come into one L2.
        // Before, tiles went round the XCDs within each slice (eighths where 8 divides them).  Before / now, us: u8 x s8 149x1776x5056 in 3
        // slices 11.5 / 10.0, fp16 300x900x1592 in 3 9.8 / 8.7, 540x784x864 in 2 8.0 / 7.4, 97x840x7192 in 9 12.7 / 12.3, conv 3x3
        // 4x14x14x256 -> 256 in 4 10.3 / 9.8; where 8 divides the tiles as before.  Eighths of the slices instead: 500x500x1000 8.0 / 9.6,
        // conv u8 3x3 8x9x9x512 -> 512 10.6 / 12.4.
        const int pair = hrn_pair_of((int)blockIdx.x, total * a.split);
        first_pid = div_by(pair, a.by_split);
        slice = pair - first_pid * a.split;
    }
    const int kt0 = SPLITK ? slice * a.kt_per_slice : 0;                                   // first k-tile of this workgroup
    const int KT = SPLITK ? min(a.kt_per_slice, KT_all - kt0) : KT_all;                    // k-tiles of this workgroup

    // ---- tile raster: spread over the 8 XCDs so that each XCD's L2 sees a compact block ----
    auto tile_coords = [&](int pid, int& bz, int& tile_m, int& tile_n) {
        if (!SPLITK && (total & 7) == 0) pid = (pid & 7) * (total >> 3) + (pid >> 3);
        bz = OP == 1 ? 0 : div_by(pid, a.by_tiles);
        const int t = pid - bz * tiles_mn;
        const int group_sz = a.group_m * a.tiles_n;
        const int gid = div_by(t, a.by_group);
        const int first_m = gid * a.group_m;
        const int gsz = min(a.tiles_m - first_m, a.group_m);
        const int tin = t - gid * group_sz;
        const int col = div_by(tin, gsz == a.group_m ? a.by_gm : a.by_gm_last);
        // (everything here is wave-uniform, and saying so keeps what is derived from it - descriptors, scalar offsets - in
        // scalar registers)
        tile_m = __builtin_amdgcn_readfirstlane(first_m + tin - col * gsz);
        tile_n = __builtin_amdgcn_readfirstlane(col);
        bz = __builtin_amdgcn_readfirstlane(bz);
    };

    // ---- compute side: the output tile whose accumulators this workgroup holds ----
    int c_bz, c_tile_m, c_tile_n;
    tile_coords(first_pid, c_bz, c_tile_m, c_tile_n);
    int m0 = c_tile_m * BM, n0 = c_tile_n * BN;

    // conv: the input that is in memory, and the way from a position of the expanded one to it
    [[maybe_unused]] int in_h = 0, in_w = 0;
    if constexpr (OP == 1) { in_h = EXPAND ? a.in_h : a.H; in_w = EXPAND ? a.in_w : a.W; }
    [[maybe_unused]] auto unexpand = [&](int& y, int& x) {
        if constexpr (!EXPAND) return true;
        else {
            y -= a.top;
            x -= a.left;
            const bool hit = ((y | x) & ((1 << a.expand_shift) - 1)) == 0;
            y >>= a.expand_shift;                                  // (a negative position stays negative)
            x >>= a.expand_shift;
            return hit && (unsigned)y < (unsigned)in_h && (unsigned)x < (unsigned)in_w;
        }
    };

    // ---- issue side: the tile whose k-tiles are being fetched (the same tile unless the launch is persistent) ----
    uint32_t a_bytes;
    const uint32_t b_bytes = (uint32_t)a.N * (uint32_t)a.ldb * ES;
    if constexpr (OP == 0) a_bytes = (uint32_t)a.M * (uint32_t)a.lda * ES;
    else a_bytes = (uint32_t)div_by(a.M, a.by_hw) * (uint32_t)(in_h * in_w * a.CI) * ES;
    const char* baseA = (const char*)a.A;
    const char* baseB = (const char*)a.B;
    bool issue_alive = true;

    const int lrow = lane / CPR, lpos = lane % CPR;
    // Rows past the end of the matrix read as zeros.  Two ways to say which rows a load covers:
    //   one vector register per load with the lane's byte offset (out of range for such rows), against one descriptor per
    // operand - a load is then two instructions;
    //   where accumulators and fragments leave no room for that, or a persistent launch would make the offsets again for
    // every output tile (UNI), and the rows that successive loads of a wave cover
    // (NW*RPI apart) share their swizzle phase: a lane's offset inside "its" row block is the same for every load, and the
    // block - tile origin, wave, load index - goes into a descriptor per load, base advanced and size reduced by it.  That
    // costs some ten scalar instructions a load, about 65 cycles of the issuing wave: a 64x64 tile of one wave needed
    // 3050 cycles to issue the loads of its three stages, 2050 with the offsets in registers, and a k-tile of it 1390 instead
    // of 860.
    constexpr bool SAME_CHUNK = (SWZ == 0) || ((NW * RPI) % (CPR << (SWZ > 0 ? SWZ - 1 : 0))) == 0;
    constexpr int WPS = (163840 / (DEEP ? KERNEL_LDS : LDS_BYTES)) * NW / 4;                     // waves per SIMD that LDS lets in: registers must not
    constexpr int VGPRS = WPS >= 4 ? 128 : (WPS == 3 ? 168 : 256);         // keep any of them out
    constexpr bool UNI = SAME_CHUNK && (PERS || TM * TN * ACC_N + 8 * (TM + TN) + LPT + 56 > VGPRS);
    constexpr bool UNI_A = UNI && OP == 0;
    const uint32_t lane_chunk = (uint32_t)((lpos ^ swz_of_row(wave * RPI + lrow)) * 16);
    auto chunk_of = [&](int i) {                 // byte offset inside a row of the lane's chunk of load i
        return SAME_CHUNK ? lane_chunk : (uint32_t)((lpos ^ swz_of_row((i * NW + wave) * RPI + lrow)) * 16);
    };
    const uint32_t lane_offB = (uint32_t)lrow * (uint32_t)a.ldb * ES + lane_chunk;
    const uint32_t lane_offA = (uint32_t)lrow * (uint32_t)a.lda * ES + lane_chunk;
    uint32_t blkA = 0, blkB = 0;                 // byte offset of the wave's first row block of the issue-side tile
    uint32_t voffB[B_LPW];
    // GEMM: byte offset of the lane's chunk in k-tile 0.  Conv: pixel bookkeeping.
    uint32_t voffA[(A_LPW > 0 ? A_LPW : 1)];
    int iy0[OP == 1 ? (A_LPW > 0 ? A_LPW : 1) : 1], ix0[OP == 1 ? (A_LPW > 0 ? A_LPW : 1) : 1];
    HrnTap tap = {};             // conv: where the lane's chunk is in K
    int itile = first_pid;
    int issue_kt = 0;            // next k-tile (relative to kt0) of tile `itile` to fetch

    auto setup_issue = [&](int t) {
        issue_alive = !PERS || t < total;             // past the last tile every fetch reads zeros
        int bz = c_bz, tile_m = c_tile_m, tile_n = c_tile_n;
        if constexpr (PERS) tile_coords(issue_alive ? t : 0, bz, tile_m, tile_n);
        const int im0 = tile_m * BM, in0 = tile_n * BN;
        baseA = (const char*)a.A + (int64_t)bz * a.sA * ES;
        baseB = (const char*)a.B + (int64_t)bz * a.sB * ES;
        if constexpr (UNI) {
            blkB = (uint32_t)(in0 + wave * RPI) * (uint32_t)a.ldb * ES;
        } else {
#pragma unroll
            for (int i = 0; i < B_LPW; ++i) {
                const int n = in0 + (i * NW + wave) * RPI + lrow;
                voffB[i] = (n < a.N) ? (uint32_t)n * (uint32_t)a.ldb * ES + chunk_of(i) : OOB;
            }
        }
        if constexpr (UNI_A) {
            blkA = (uint32_t)(im0 + wave * RPI) * (uint32_t)a.lda * ES;
        } else if constexpr (OP == 0) {
#pragma unroll
            for (int i = 0; i < A_LPW; ++i) {
                const int m = im0 + (i * NW + wave) * RPI + lrow;
                voffA[i] = (m < a.M) ? (uint32_t)m * (uint32_t)a.lda * ES + chunk_of(i) : OOB;
            }
        } else if constexpr (!CW) {
            static_assert(OP == 0 || CW || SWZ == 0 || ((NW * RPI) % (CPR << (SWZ > 0 ? SWZ - 1 : 0))) == 0,
                          "conv: the lane's chunk column must not depend on the load index");
            const int chunk = lpos ^ swz_of_row(wave * RPI + lrow);
            tap = hrn_tap_at(a, chunk * (16 / ES) + kt0 * (BKB / ES), in_w, ES);      // of this workgroup's first k-tile
            // the lane's first row by division, the following ones (NW*RPI output pixels further each) by carry
            int m = im0 + wave * RPI + lrow;
            HrnRow row = hrn_row_at<EXPAND>(a, m);
#pragma unroll
            for (int i = 0; i < A_LPW; ++i) {
                iy0[i] = (m < a.M) ? row.y : -(1 << 28);
                ix0[i] = row.x;
                voffA[i] = row.off;
                m += NW * RPI;
                if (i + 1 < A_LPW) hrn_next_row<EXPAND>(a, row);
            }
        }
    };
    setup_issue(itile);

    // the stream moves on: next k-tile of this tile, or (persistent) k-tile 0 of the workgroup's next tile
    auto advance_issue = [&]() {
        ++issue_kt;
        if constexpr (PERS) {
            if (issue_kt == KT) { issue_kt = 0; itile += gridDim.x; setup_issue(itile); }
        }
    };

    // Fetch k-tile `issue_kt` of the issue-side tile straight into LDS stage `stage`: begin_issue() fixes the tile's
    // descriptors and scalar offset, issue_loads(first, count) emits a part of its LPT wave loads (A first, then B), so
    // that the caller can spread them between MFMAs, end_issue() moves the stream on.  RAG = the tile may be the last,
    // partly filled one (its chunks past the end of K are masked per lane); the plain form spends no vector ALU work.
    rsrc_t rA_cur, rB_cur;
    uint32_t ks_cur = 0, koff_cur = 0;
    bool live_cur = false;
    // descriptor of row block `i` of an operand: base advanced by the block's offset, size reduced by it
    auto block_rsrc = [&](const char* base, uint32_t bytes, uint32_t blk0, uint32_t ld_bytes, int i) {
        // (wave-uniform by construction; said explicitly, or the descriptor is treated as a per-lane value)
        const uint32_t off = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blk0 + (uint32_t)(i * NW * RPI) * ld_bytes));
        const uint32_t left = (uint32_t)__builtin_amdgcn_readfirstlane((int)((live_cur && bytes > off) ? bytes - off : 0u));
        return make_rsrc(base + off, left);
    };
    auto begin_issue = [&]() {
        const bool live = issue_alive && issue_kt < KT;                          // wave-uniform
        live_cur = live;
        koff_cur = (uint32_t)(kt0 + issue_kt) * BKB;                             // byte offset of the k-tile in a row
        // a dead tile (past the end of K, or past the workgroup's last output tile) reads zeros through empty descriptors
        rB_cur = make_rsrc(baseB, live ? b_bytes : 0u);
        rA_cur = make_rsrc(baseA, live ? a_bytes : 0u);
        ks_cur = live ? koff_cur : 0u;
        return live && koff_cur + BKB > Kb;                                      // ragged: the last tile is not full
    };
    // conv: the byte offset of load i of the next k-tile of A
    [[maybe_unused]] auto conv_address = [&](int i) __attribute__((always_inline)) {
        if constexpr (OP == 1) {
            int iy = iy0[i] + tap.dy, ix = ix0[i] + tap.dx;
            if constexpr (EXPAND) {
                return unexpand(iy, ix) ? voffA[i] + (uint32_t)((iy * in_w + ix) * a.CI + tap.c) * ES : OOB;
            } else {
                const bool ok = (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
                return ok ? voffA[i] + tap.off : OOB;
            }
        } else {
            return 0u;
        }
    };
    // They are made in front of the barrier that lets the loads go; left to itself the compiler makes all but the first between the loads.
    // Between / in front, us: fp16 3x3 in 2 slices 16x7x7x512 -> 512 15.8 / 14.9, 9x46x49x240 -> 64 18.1 / 17.9, u8 3x3 4x30x30x448 -> 320 19.7 / 18.6,
    // 5x5 16x21x24x176 -> 288 26.9 / 26.5.  Not with one MFMA tile a wave and one wave a SIMD, whose barrier then comes later: fp16 64x64 tiles, 3x3
    // 32x7x7x512 -> 512 25.5 / 26.3, 5x5 12x19x18x96 -> 80 15.3 / 16.0, stride 2, 2x54x54x352 -> 368 46.2 / 48.2 (u8 in slices 4x14x14x512 -> 256 11.1 /
    // 11.0).  Of 128x128 tiles on four waves one call was better off between its loads, stride 2 17x35x38x288 -> 272 25.7 / 27.0.
    constexpr bool ADDR_FIRST = OP == 1 && !CW && !(DT == 0 && TM * TN == 1 && NW <= 4);
    [[maybe_unused]] uint32_t addr[(A_LPW > 0 ? A_LPW : 1)];
    auto conv_addresses = [&]() __attribute__((always_inline)) {
        if constexpr (ADDR_FIRST) {
#pragma unroll
            for (int i = 0; i < A_LPW; ++i) {
                addr[i] = conv_address(i);
                asm volatile("" : "+v"(addr[i]));
            }
        }
    };
    auto issue_loads = [&](auto ragc, int stage, auto firstc, auto countc) {
        constexpr bool RAG = decltype(ragc)::value;
        constexpr int FIRST = decltype(firstc)::value, COUNT = decltype(countc)::value;
        char* sbase = lds + stage * STAGE_BYTES;
        [[maybe_unused]] uint32_t koff_rag = koff_cur;
        // the masks of the ragged form are computed inside its (rarely taken) branch, not hoisted in front of it
        if constexpr (RAG) asm volatile("" : "+v"(koff_rag));
#pragma unroll
        for (int q = FIRST; q < FIRST + COUNT; ++q) {
            if (q < A_LPW) {
                const int i = q;
                if constexpr (UNI_A) {
                    uint32_t v = lane_offA;
                    if constexpr (RAG) { if (koff_rag + lane_chunk >= Kb) v = OOB; }
                    load_chunk_to_lds(block_rsrc(baseA, a_bytes, blkA, (uint32_t)a.lda * ES, i), sbase + (i * NW + wave) * 1024, v, ks_cur);
                } else if constexpr (OP == 0) {
                    uint32_t v = voffA[i];
                    if constexpr (RAG) { if (koff_rag + chunk_of(i) >= Kb) v = OOB; }
                    load_chunk_to_lds(rA_cur, sbase + (i * NW + wave) * 1024, v, ks_cur);
                } else if constexpr (!CW) {
                    uint32_t v = ADDR_FIRST ? addr[i] : conv_address(i);
                    if constexpr (RAG) { if (koff_rag + lane_chunk >= Kb) v = OOB; }      // (past the last tap)
                    load_chunk_to_lds(rA_cur, sbase + (i * NW + wave) * 1024, v, 0u);
                }
            } else {
                const int i = q - A_LPW;
                if constexpr (UNI) {
                    uint32_t v = lane_offB;
                    if constexpr (RAG) { if (koff_rag + lane_chunk >= Kb) v = OOB; }
                    load_chunk_to_lds(block_rsrc(baseB, b_bytes, blkB, (uint32_t)a.ldb * ES, i), sbase + A_BYTES + (i * NW + wave) * 1024, v, ks_cur);
                } else {
                    uint32_t v = voffB[i];
                    if constexpr (RAG) { if (koff_rag + chunk_of(i) >= Kb) v = OOB; }
                    load_chunk_to_lds(rB_cur, sbase + A_BYTES + (i * NW + wave) * 1024, v, ks_cur);
                }
            }
        }
    };
    auto end_issue = [&]() {
        if constexpr (OP == 1 && !CW) {
            // advance the lane's (kh, kw, ci) position by one k-tile.  A load's address is then its row's plus the tap's; resolved anew for
            // every load it took some twelve vector instructions, two of them quarter-rate multiplications, now six.
            hrn_next_tap<BKB / ES, ES>(a, tap, (int)(koff_cur + BKB + lane_chunk) / ES, in_w);
        }
        advance_issue();
    };
    using TrueC = std::integral_constant<bool, true>;
    using FalseC = std::integral_constant<bool, false>;
    auto issue_tile = [&](int stage) {          // the whole tile at once (prologue)
        const bool rag = begin_issue();
        conv_addresses();
        if (rag) issue_loads(TrueC{}, stage, std::integral_constant<int, 0>{}, std::integral_constant<int, LPT>{});
        else issue_loads(FalseC{}, stage, std::integral_constant<int, 0>{}, std::integral_constant<int, LPT>{});
        end_issue();
    };

    // ---- per-lane MFMA operand addresses ----
    const int lr = lane % MT, lq = lane / MT;

    // ---- conv window mode: the window itself (dynamic LDS) and the per-row tap masks ----
    int w_pitch = 0;                                     // bytes of one pixel (all channels)
    if constexpr (CW) w_pitch = a.CI * ES;
    const int w_cch = CW ? w_pitch / BKB : 1;            // k-tiles per tap
    uint32_t tapmask[CW ? TM : 1];                       // bit t: tap t of this lane's pixel i is inside the image
    if constexpr (CW) {
        const rsrc_t rA = make_rsrc(baseA, a_bytes);
        const int w_rows = BM + 2 * (a.cpad * a.W + a.cpad_w);  // pixels the BM outputs can reach
        const int cpp = w_pitch / 16;                    // 16-byte chunks per pixel
        const int n_instr = (w_rows * cpp + 63) / 64;    // 1 KiB wave loads that cover the window
        const int gp0 = m0 - (a.cpad * a.W + a.cpad_w);  // input pixel index of window row 0
        // A lane's chunk moves on by NW * 64 chunks from load to load.  Its window row and its position in the row (EXPAND:
        // and the row's pixel) are divided out once and then carried: a division is some 40 instructions, and with three of
        // them per load (and one per stored piece, see HOIST below) the transposed conv below took 38.0 us instead of 33.8.
        const int d_row = div_by(NW * 64, a.by_cpp), d_pos = NW * 64 - d_row * cpp;
        int wrow = div_by(wave * 64 + lane, a.by_cpp), pos = wave * 64 + lane - wrow * cpp;
        [[maybe_unused]] int w_img = 0, w_y = 0, w_x = 0, d_img = 0, d_y = 0, d_x = 0;
        if constexpr (EXPAND) {
            const int gp = gp0 + wrow;
            w_img = gp / (a.H * a.W);
            int rem = gp - w_img * (a.H * a.W);
            if (rem < 0) { rem += a.H * a.W; --w_img; }
            w_y = rem / a.W; w_x = rem - w_y * a.W;
            d_img = d_row / (a.H * a.W);
            const int d_rem = d_row - d_img * (a.H * a.W);
            d_y = d_rem / a.W; d_x = d_rem - d_y * a.W;
        }
        for (int q = wave; q < n_instr; q += NW) {
            const int src = (pos & ~(CPR - 1)) | ((pos & (CPR - 1)) ^ swz_of_row(wrow));
            const int gp = gp0 + wrow;
            int px = gp;                                     // pixel in memory
            bool ok = wrow < w_rows && gp >= 0;
            if constexpr (EXPAND) {
                int iy = w_y, ix = w_x;
                ok = ok && unexpand(iy, ix);
                px = (w_img * in_h + iy) * in_w + ix;
            }
            const uint32_t v = ok ? (uint32_t)px * (uint32_t)w_pitch + src * 16 : OOB;
            load_chunk_to_lds(rA, win + q * 1024, v, 0u);
            pos += d_pos;
            const int carry = pos >= cpp ? 1 : 0;
            pos -= carry ? cpp : 0;
            wrow += d_row + carry;
            if constexpr (EXPAND) {                          // (each sum is less than twice its modulus)
                w_x += d_x + carry;
                w_y += d_y;
                w_img += d_img;
                if (w_x >= a.W) { w_x -= a.W; ++w_y; }
                if (w_y >= a.H) { w_y -= a.H; ++w_img; }
            }
        }
        // masks: pixel of fragment row i by one division, the following rows (MT further each) by carry
        const int hw = a.H * a.W;
        int m = m0 + wm_idx * WTM + lr;
        int img = div_by(m, a.by_hw);          // ('same' padding: the image and its result are of one size)
        int rem = m - img * hw;
        int oy = div_by(rem, a.by_wo), ox = rem - oy * a.W;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            uint32_t bits = 0;
            if (m < a.M) {
                for (int r = 0; r < a.KH; ++r)
                    for (int s2 = 0; s2 < a.KW; ++s2) {
                        const int iy = oy + r - a.cpad, ix = ox + s2 - a.cpad_w;
                        if ((unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W) bits |= 1u << (r * a.KW + s2);
                    }
            }
            tapmask[i] = bits;
            m += MT;
            ox += MT;
            while (ox >= a.W) { ox -= a.W; if (++oy == a.H) { oy = 0; ++img; } }
        }
    }
    const int w_lane = (wm_idx * WTM + lr);              // window mode: tile row of fragment 0
    int rd_tap = 0, rd_cch = 0, rd_r = 0, rd_s = 0;      // window mode: tap / channel chunk of the k-tile being READ
    const int g16 = (lq ^ swz_of_row(lr)) << 4;      // swizzle period <= MT, so only lr matters
    const int a_lane = (wm_idx * WTM + lr) * BKB;
    const int b_lane = A_BYTES + (wn_idx * WTN + lr) * BKB;

    acc_t acc[TM][TN];
    int bsum[TN];
    auto clear_acc = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < ACC_N; ++r) acc[i][j][r] = 0;
#pragma unroll
        for (int j = 0; j < TN; ++j) bsum[j] = 0;
    };
    clear_acc();

    // Operand fragments, double-buffered in registers.  Read slot r of a step: r < TN is B fragment r, the others are
    // the A fragments in row-tile order - the order in which the MFMAs of the step consume them (the first row of
    // MFMAs needs every B fragment).
    v4i fa[2][TM], fb[2][TN];
    constexpr int NRD = TM + TN;
    auto read_slot = [&](int buf, int stage_off, int kk, int r) {
        if (r < TN) {
            fb[buf][r] = *(const v4i*)(lds + stage_off + b_lane + r * MT * BKB + (g16 ^ (kk * KSB)));
        } else {
            const int i = r - TN;
            if constexpr (CW) {
                const int tapoff = (rd_r < a.KH) ? rd_r * a.W + rd_s : 0;    // r*W + s pixels; 0 past the last tap
                const int wrow = w_lane + i * MT + tapoff;
                const int kc = (kk * CPS + lq) ^ swz_of_row(wrow);
                fa[buf][i] = *(const v4i*)(win + wrow * w_pitch + rd_cch * BKB + kc * 16);
            } else {
                fa[buf][i] = *(const v4i*)(lds + stage_off + a_lane + i * MT * BKB + (g16 ^ (kk * KSB)));
            }
        }
    };
    auto read_frags = [&](int buf, int stage_off, int kk) {
#pragma unroll
        for (int r = 0; r < NRD; ++r) read_slot(buf, stage_off, kk, r);
    };
    // window mode: move the reader to the next k-tile (channel chunks inside a tap first, then kw, then kh)
    auto advance_reader = [&]() {
        if constexpr (CW) {
            if (++rd_cch == w_cch) { rd_cch = 0; ++rd_tap; if (++rd_s == a.KW) { rd_s = 0; ++rd_r; } }
        }
    };
    int mm_tap = 0, mm_cch = 0;                           // window mode: tap of the k-tile being MULTIPLIED
    uint32_t tap_bit = 0;
    auto set_masks = [&]() {
        if constexpr (CW) {
            tap_bit = mm_tap;
            if (++mm_cch == w_cch) { mm_cch = 0; ++mm_tap; }
        }
    };
    // the A fragment of row-tile i as the MFMA takes it: window taps in the padding contribute zero, uint8 becomes
    // int8 by subtracting 128 (the sign-bit flip; the epilogue adds 128 * sum_k B back)
    auto a_operand = [&](int buf, int i) {
        v4i av = fa[buf][i];
        if constexpr (CW) {
            const int on = -(int)((tapmask[i] >> tap_bit) & 1u);
            av = av & (v4i){on, on, on, on};
        }
        if constexpr (DT == 1) av = av ^ (int)0x80808080;
        return av;
    };
    // uint8 path: sum_k B[n,k] of the step's B fragments.  The WM waves of one column hold the same fragments, so
    // they take turns: wave row w sums the steps with step % WM == w, the epilogue adds the WM partial sums.
    auto bsum_step = [&](int buf, int step) {
        if constexpr (DT == 1 && !COLSUM) {
            if (WM == 1 || (step & (WM - 1)) == wm_idx) {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    int s = bsum[j];
                    s = __builtin_amdgcn_sdot4(fb[buf][j].x, 0x01010101, s, false);
                    s = __builtin_amdgcn_sdot4(fb[buf][j].y, 0x01010101, s, false);
                    s = __builtin_amdgcn_sdot4(fb[buf][j].z, 0x01010101, s, false);
                    s = __builtin_amdgcn_sdot4(fb[buf][j].w, 0x01010101, s, false);
                    bsum[j] = s;
                }
            }
        }
    };

    // ---- epilogue of the compute-side tile (c_bz, m0, n0) ----
    // MFMA was issued as (B fragment, A fragment), so a lane holds 4 consecutive n for one m:
    //   m = lr, n = (r/4)*8 + lq*4 + r%4   (32x32)     m = lr, n = lq*4 + r   (16x16)
    // (CHW: m and n exchanged)
    auto store_tile = [&]() __attribute__((always_inline)) {
        // the lane's coordinates, re-derived from values the compiler cannot trace back past this point: otherwise it
        // computes the epilogue's addresses in front of the k-loop and keeps them in registers all the way through it
        int lane_e = lane, lr_e, lq_e;
        asm volatile("" : "+v"(lane_e));
        lr_e = lane_e % MT; lq_e = lane_e / MT;
        char* const epi = CW ? win : lds + EPI_OFF;
        int* bs_lds = (int*)epi;
        if constexpr (DT == 1) {
            // 128 * sum_k B[n,k] completes the u8 x s8 product computed as (u8-128) x s8
            if constexpr (PERS) wait_and_barrier<63, 0>();     // the stages stay live: LDS traffic only, no drain
            else wait_and_barrier<0, 0>();
            if constexpr (COLSUM) {
                // the caller's sums of this tile's BN columns, 16 bytes per lane (N is a multiple of 4); a split-K
                // slice other than the first adds nothing (the sums cover all of K)
                for (int q = tid; q < BN / 4; q += NT) {
                    const int n = n0 + q * 4;
                    v4i v = {0, 0, 0, 0};
                    if (slice == 0 && n + 4 <= a.N) v = *(const v4i*)((const int*)a.bsum + (int64_t)c_bz * a.N + n);
                    *(v4i*)(bs_lds + q * 4) = v;
                }
            } else {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    int s = bsum[j];
#pragma unroll
                    for (int d = MT; d < 64; d <<= 1) s += __shfl_xor(s, d, 64);
                    if (lq_e == 0) bs_lds[wm_idx * BN + wn_idx * WTN + j * MT + lr_e] = s;
                }
            }
            if constexpr (PERS) wait_and_barrier<63, 0>();
            else __syncthreads();
        }
        // column sums of the 4 consecutive outputs a lane_e holds, all wave rows added
        auto colsum4 = [&](int nl) {
            v4i bs = *(const v4i*)(bs_lds + nl);
            if constexpr (!COLSUM) {
#pragma unroll
                for (int w = 1; w < WM; ++w) bs += *(const v4i*)(bs_lds + w * BN + nl);
            }
            return bs;
        };

        char* Cb = (char*)a.C + ((int64_t)slice * batch + c_bz) * a.sC * OES;
        using NtC = std::integral_constant<bool, NTS>;
        // Staged results: the non-temporal hint for rows of whole lines, and for rows of whole half lines up to 64 MiB of result, a limit between
        // the 57 MB and the 107 MB below.  Elsewhere the L2 joins the pieces that tiles side by side and the strips of a tile
        // leave of a line.  Hint / no hint, us: rows at 16 or 32 bytes u8 x s8 4653x3384x208 34.0 / 24.5, 8190x4040x128 47.9 / 27.3, fp16
        // 8190x8184x128 59.0 / 37.3, batch_matmul 192x512x520x64 55.2 / 25.4; half lines fp16 8190x8160x128 (134 MB) 58.5 / 43.0, batch_matmul
        // 192x512x544x64 (107 MB) 29.5 / 27.4, 4330x6624x1120 (57 MB) 63.4 / 63.3, 3000x2336x512 15.1 / 15.7, 100x300x352x64 10.8 / 12.7, u8 conv
        // 1x1 16x56x56x64 -> 112 7.4 / 8.3.  Long products hide the pieces: fp16 4330x6616x2048 102.8 / 98.9, x4096 186.1 / 188.7, x8192 364.5 / 363.3,
        // 2308x6904x5560 240.8 / 244.0, u8 4653x3384x4096 100.3 / 90.8.
        [[maybe_unused]] const uint32_t row_ends = (uint32_t)a.ldc * OES | (uint32_t)(uintptr_t)Cb;
        [[maybe_unused]] const bool row_lines =
            (row_ends & 127) == 0 || ((row_ends & 63) == 0 && (uint64_t)batch * (uint32_t)a.M * (uint32_t)a.ldc <= (64u << 20) / OES);
        [[maybe_unused]] const rsrc_t rsrcC = make_rsrc(Cb, (uint32_t)a.M * (uint32_t)a.ldc * OES);
        // (ntc: with the hint.  Staged results ask row_lines, the others take NtC)
        [[maybe_unused]] auto put16 = [&](auto ntc, char* dst, v4i val) __attribute__((always_inline)) {
            if constexpr (decltype(ntc)::value) __builtin_nontemporal_store(val, (out16_t*)dst);
            else *(out16_t*)dst = val;
        };
        [[maybe_unused]] auto put8 = [&](auto ntc, char* dst, long val) __attribute__((always_inline)) {
            if constexpr (decltype(ntc)::value) __builtin_nontemporal_store(val, (out8_t*)dst);
            else *(out8_t*)dst = val;
        };
        // partial sums that this kernel adds up lie tile by tile (the rows of tiles one behind the other), so that a tile's are stored and
        // read in one piece: as rows of the result, which rarely are whole lines, fp16 500x500x1000 in 4 slices took 7.8 us (7.2 like this),
        // 97x840x7192 in 9 12.2 (11.9), 40x864x560 in 2 5.9 (5.8); where N is whole lines nothing changes.  Those for splitk_reduce_kernel are row-major.
        [[maybe_unused]] const bool by_tile = SPLITK && a.arrivals;
        [[maybe_unused]] const int part_ld = by_tile ? min(BN, a.N - n0) : a.ldc;
        [[maybe_unused]] const int part_base = m0 * a.ldc + n0 * (by_tile ? min(BM, a.M - m0) : 1);
        [[maybe_unused]] auto put_partial = [&](int m, int n, auto val) __attribute__((always_inline)) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, val), rsrcC, (part_base + (m - m0) * part_ld + (n - n0)) * 4, 0, AGENT_SCOPE);
        };
        if constexpr (CHW) {
            // A wave parks MT channels x CSW pixels of its result in a private LDS strip and streams them out 16 bytes per
            // lane along the pixels.  A piece starts at any element (a plane may be odd); the few that reach past the end of
            // a plane or of the result go element by element.
            if constexpr (DT == 0) wait_and_barrier<0, 0>();          // (the int8 path has synchronised above) stages are dead now
            using oel_t = typename std::conditional<OES == 2, _Float16, int>::type;
            typedef v4i piece_t __attribute__((aligned(2)));
            char* strip = epi + EPI_BASE + wave * (MT * CHW_PITCH);
            constexpr int CPRW = CSW * OES / 16, EPC = 16 / OES, IT = CSW / MT;
            // where pixel m of the result lies: its image and its place in the plane.  Where a lane's pieces of a strip are the
            // same pixels of other channels (HOIST), the division is made once per strip of pixels, not per piece
            // (NCW conv1d 16 x 892 x 512 -> 512: 40.2 -> 38.2 us).
            const unsigned plane = (unsigned)a.out_plane;
            // Planes that are no whole lines begin and end strips inside them: such stores go through the L2, which joins the pieces
            // (transposed conv with planes of 111x111, 256x64 tiles: 31.0 us with the non-temporal hint, 25.5 without).
            [[maybe_unused]] const bool whole_lines = plane * OES % 128 == 0;
            constexpr bool HOIST = 64 % CPRW == 0;
            constexpr int NIB = HOIST ? TM / IT : 1;
            unsigned h_img[NIB], h_px[NIB];
            if constexpr (HOIST) {
#pragma unroll
                for (int b = 0; b < NIB; ++b) {
                    const unsigned m = (unsigned)(m0 + wm_idx * WTM + b * CSW + (lane_e % CPRW) * EPC);
                    h_img[b] = (unsigned)div_by((int)m, a.by_plane);
                    h_px[b] = m - h_img[b] * plane;
                }
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int nl = wn_idx * WTN + j * MT;
                [[maybe_unused]] int bs = 0;
                if constexpr (DT == 1) {
                    bs = bs_lds[nl + lr_e];
                    if constexpr (!COLSUM) {
#pragma unroll
                        for (int w = 1; w < WM; ++w) bs += bs_lds[w * BN + nl + lr_e];
                    }
                    bs *= 128;
                }
#pragma unroll
                for (int ib = 0; ib < TM; ib += IT) {
#pragma unroll
                    for (int i = 0; i < IT; ++i)
#pragma unroll
                        for (int g = 0; g < ACC_N / 4; ++g) {
                            char* dst = strip + lr_e * CHW_PITCH + (i * MT + g * 8 + lq_e * 4) * OES;
                            if constexpr (DT == 0) {
                                v4h o;
#pragma unroll
                                for (int r = 0; r < 4; ++r) o[r] = (_Float16)acc[ib + i][j][g * 4 + r];
                                *(v4h*)dst = o;
                            } else {
                                v4i o;
#pragma unroll
                                for (int r = 0; r < 4; ++r) o[r] = acc[ib + i][j][g * 4 + r] + bs;
                                *(v4i*)dst = o;
                            }
                        }
                    asm volatile("" ::: "memory");     // LDS serves one wave's requests in order: the reads below see the writes
#pragma unroll
                    for (int it = 0; it < (MT * CPRW + 63) / 64; ++it) {
                        const int c = it * 64 + lane_e;
                        const int row = c / CPRW, cc2 = c % CPRW;
                        const int n = n0 + nl + row;
                        const int m = m0 + wm_idx * WTM + ib * MT + cc2 * EPC;
                        if (c < MT * CPRW && n < a.N && m < a.M) {
                            const v4i val = *(const v4i*)(strip + row * CHW_PITCH + cc2 * 16);
                            const unsigned img = HOIST ? h_img[HOIST ? ib / IT : 0] : (unsigned)div_by(m, a.by_plane);
                            const unsigned px = HOIST ? h_px[HOIST ? ib / IT : 0] : (unsigned)m - img * plane;
                            oel_t* dst = (oel_t*)a.C + ((int64_t)img * a.N + n) * plane + px;
                            if (px + EPC <= plane && m + EPC <= a.M) {
                                if (NTS && whole_lines) __builtin_nontemporal_store(val, (piece_t*)dst);
                                else *(piece_t*)dst = val;
                            } else {
                                const oel_t* ve = (const oel_t*)&val;
                                unsigned p = px;
#pragma unroll
                                for (int e = 0; e < EPC; ++e) {
                                    if (m + e < a.M) *dst = ve[e];
                                    ++dst;
                                    if (++p == plane) { p = 0; dst += (int64_t)(a.N - 1) * plane; }
                                }
                            }
                        }
                    }
                    asm volatile("" ::: "memory");
                }
            }
        } else if constexpr (EPI >= 1) {
            // LDS-staged epilogue: a wave parks one MFMA row-tile (MT rows x SW columns) of its result in a private,
            // padded LDS strip, then streams it out with 16 bytes per lane_e, whole row segments per store instruction.
            if constexpr (DT == 0 && !PERS) wait_and_barrier<0, 0>();   // (the int8 path has synchronised above) stages are dead now
            char* strip = epi + EPI_BASE + wave * (MT * EPI_PITCH);
            constexpr int CPRW = SW * OES / 16;                // 16-byte chunks per strip row
            constexpr int EPC = 16 / OES;                      // output elements per chunk
            constexpr int TNS = TN / ESPLIT;                   // MFMA column tiles per strip
            // (two copies of the loop and one branch: a branch per strip costs u8 x s8 1205x1392x656 6.4 -> 6.95 us)
            auto staged = [&](auto ntc) __attribute__((always_inline)) {
                constexpr bool NT_HINT = decltype(ntc)::value;
#pragma unroll
                for (int i = 0; i < TM; ++i) {
#pragma unroll
                    for (int h = 0; h < ESPLIT; ++h) {
#pragma unroll
                        for (int js = 0; js < TNS; ++js) {
                            const int j = h * TNS + js;
#pragma unroll
                            for (int g = 0; g < ACC_N / 4; ++g) {
                                const int cl = js * MT + g * 8 + lq_e * 4;         // column inside the strip
                                char* dst = strip + lr_e * EPI_PITCH + cl * OES;
                                if constexpr (DT == 0 && !SPLITK) {
                                    v4h o;
#pragma unroll
                                    for (int r = 0; r < 4; ++r) o[r] = (_Float16)acc[i][j][g * 4 + r];
                                    *(v4h*)dst = o;
                                } else if constexpr (DT == 0) {
                                    v4f o;
#pragma unroll
                                    for (int r = 0; r < 4; ++r) o[r] = acc[i][j][g * 4 + r];
                                    *(v4f*)dst = o;
                                } else {
                                    const v4i bs = colsum4(wn_idx * WTN + h * SW + cl);
                                    v4i o;
#pragma unroll
                                    for (int r = 0; r < 4; ++r) o[r] = acc[i][j][g * 4 + r] + 128 * bs[r];
                                    *(v4i*)dst = o;
                                }
                            }
                        }
                        asm volatile("" ::: "memory");     // LDS serves one wave's requests in order: the reads below see the writes
#pragma unroll
                        for (int it = 0; it < MT * CPRW / 64; ++it) {
                            const int c = it * 64 + lane_e;
                            const int row = c / CPRW, cc2 = c % CPRW;
                            const v4i val = *(const v4i*)(strip + row * EPI_PITCH + cc2 * 16);
                            const int m = m0 + wm_idx * WTM + i * MT + row;
                            const int n = n0 + wn_idx * WTN + h * SW + cc2 * EPC;
                            if constexpr (PERS) {
                                // always issued, so that every wave has exactly STORES_PER_TILE stores per tile in flight
                                const uint32_t off = (m < a.M && n + EPC <= a.N) ? (uint32_t)(m * a.ldc + n) * OES : OOB;
                                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, val), rsrcC, (int)off, 0, NT_HINT ? 2 : 0);
                            } else if constexpr (SPLITK) {
                                if (m < a.M && n < a.N) put_partial(m, n, val);
                            } else {
                                char* dst = Cb + ((int64_t)m * a.ldc + n) * OES;
                                if (m < a.M) {
                                    if (n + EPC <= a.N) put16(ntc, dst, val);
                                    else if (OES == 2 && n + 4 <= a.N) put8(ntc, dst, (long)(((long)(uint32_t)val.y << 32) | (uint32_t)val.x));
                                }
                            }
                        }
                        asm volatile("" ::: "memory");
                    }
                }
            };
            if constexpr (NTS) {
                if (row_lines) staged(TrueC{});
                else staged(FalseC{});
            } else {
                staged(FalseC{});
            }
        } else {
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int m = m0 + wm_idx * WTM + i * MT + lr_e;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
#pragma unroll
                    for (int g = 0; g < ACC_N / 4; ++g) {
                        const int nl = wn_idx * WTN + j * MT + g * 8 + lq_e * 4;
                        const int n = n0 + nl;
                        if (m < a.M && n < a.N) {
                            char* dst = Cb + ((int64_t)m * a.ldc + n) * OES;
                            if constexpr (DT == 0 && !SPLITK) {
                                v4h o;
#pragma unroll
                                for (int r = 0; r < 4; ++r) o[r] = (_Float16)acc[i][j][g * 4 + r];
                                put8(NtC{}, dst, __builtin_bit_cast(long, o));
                            } else if constexpr (DT == 0) {
                                v4f o;
#pragma unroll
                                for (int r = 0; r < 4; ++r) o[r] = acc[i][j][g * 4 + r];
                                put_partial(m, n, o);
                            } else {
                                const v4i bs = colsum4(nl);
                                v4i o;
#pragma unroll
                                for (int r = 0; r < 4; ++r) o[r] = acc[i][j][g * 4 + r] + 128 * bs[r];
                                if constexpr (SPLITK) put_partial(m, n, o);
                                else put16(NtC{}, dst, o);
                            }
                        }
                    }
                }
            }
        }
    };

    // ---- split-K: the last slice of an output tile adds all of them up ----
    // Every slice stores its partial sums so that all XCDs see them, waits for the stores and counts itself in at the tile's
    // word.  Nobody waits for anybody: whoever counts last reads the slices (its own among them) and writes the result.  The
    // word may hold anything before: greet() raises it to this launch's ticket with no arrivals (tickets grow and are high numbers),
    // while the partial sums are on their way; only where it was higher does arrive() find something else, and installs the ticket
    // itself.  The last slice takes the arrivals back, for a replay of the launch from a graph.  Slices are
    // added in their order, as by splitk_reduce_kernel, the launch behind this one that workspaces without the words get.
    //   What it costs is three trips to memory, one of them the stores' that a kernel's end waits for anyway; a launch of its own cost
    // the call 3.5 us of host time and the device 2.7 - 4.6 us.  Loads and stores carry their scope themselves: fences instead
    // empty the L2s (1.3 - 5.4 us more).  fp16, per call: 32x4096x4096 in 4 slices 10.8 -> 10.4 us (7.7 without any sum),
    // 86x2648x576 in 2 9.0 -> 7.3, 540x784x864 in 2 8.8 -> 8.2, variance of 15x128x36x36 in 76 32.1 -> 19.1.
    [[maybe_unused]] auto greet = [&]() __attribute__((always_inline)) {
        if (tid == 0) (void)__hip_atomic_fetch_max(a.arrivals + first_pid, a.ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    [[maybe_unused]] auto arrive = [&]() __attribute__((always_inline)) {      // (one lane)
        uint64_t* const word = a.arrivals + first_pid;
        uint64_t n = __hip_atomic_fetch_add(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - a.ticket;
        if (n >= 0x10000) {                                           // not of this launch (compare-and-swap alone: 0.7 us per slice)
            uint64_t seen = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), next;
            do {
                n = seen - a.ticket < 0x10000 ? seen - a.ticket : 0;
                next = a.ticket + n + 1;
            } while (!__hip_atomic_compare_exchange_strong(word, &seen, next, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        }
        const bool last = n + 1 == (uint64_t)a.split;
        if (last) __hip_atomic_store(word, a.ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return last;
    };
    [[maybe_unused]] auto fold_slices = [&]() __attribute__((always_inline)) {
        using sum_t = typename std::conditional<DT == 0, v4f, v4i>::type;
        wait_only<0, 0>();                                            // the stores of this wave have arrived
        __syncthreads();
        int* const flag = (int*)lds;
        if (tid == 0) *flag = arrive();
        __syncthreads();
        const bool last = *flag != 0;
        if (!last) return;
        asm volatile("" ::: "memory");
        const int cpr = min(BN, a.N - n0) / 4, count = min(BM, a.M - m0) * cpr;   // 16-byte pieces of the tile
        const float inv = 1.0f / (float)cpr;
        const uint32_t slice_bytes = (uint32_t)a.M * (uint32_t)a.N * 4;
        const uint32_t tile_off = (uint32_t)(m0 * a.N + n0 * min(BM, a.M - m0)) * 4;
        const int64_t step = (int64_t)batch * a.sC * 4;
        // U pieces of a lane at a time, Z slices of each on the way
        auto fold = [&](auto uc, auto zc) __attribute__((always_inline)) {
            constexpr int U = decltype(uc)::value, Z = decltype(zc)::value;
#pragma unroll 1
            for (int v0 = tid; v0 < count; v0 += U * NT) {
                int m[U], n[U];
                uint32_t off[U];
                sum_t sum[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int v = v0 + u * NT, row = (int)(((float)v + 0.5f) * inv);      // v / cpr (v is below 2^16, so the quotient is exact)
                    m[u] = m0 + row;
                    n[u] = n0 + (v - row * cpr) * 4;
                    off[u] = v < count ? tile_off + (uint32_t)v * 16 : OOB;
                    sum[u] = sum_t{0, 0, 0, 0};
                }
                const char* part = (const char*)a.C + (int64_t)c_bz * a.sC * 4;
#pragma unroll 1
                for (int z0 = 0; z0 < a.split; z0 += Z, part += Z * step) {
                    sum_t t[Z][U];
#pragma unroll
                    for (int z = 0; z < Z; ++z)
                        if (z0 + z < a.split) {
                            const rsrc_t r = make_rsrc(part + z * step, slice_bytes);
#pragma unroll
                            for (int u = 0; u < U; ++u) t[z][u] = __builtin_bit_cast(sum_t, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off[u], 0, AGENT_SCOPE));
                        }
#pragma unroll
                    for (int z = 0; z < Z; ++z)
                        if (z0 + z < a.split) {
#pragma unroll
                            for (int u = 0; u < U; ++u) sum[u] += t[z][u];
                        }
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (v0 + u * NT < count) {
                        const int64_t at = (int64_t)c_bz * a.out_stride + (int64_t)m[u] * a.out_ld + n[u];
                        if constexpr (DT == 0) {
                            v4h o;
#pragma unroll
                            for (int r = 0; r < 4; ++r) o[r] = (_Float16)sum[u][r];
                            *(sum8_t*)((_Float16*)a.out + at) = o;
                        } else {
                            *(sum16_t*)((int*)a.out + at) = __builtin_bit_cast(v4i, sum[u]);
                        }
                    }
                }
            }
        };
        if (count > NT) fold(std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{});
        else fold(std::integral_constant<int, 1>{}, std::integral_constant<int, 16>{});
    };

    // ---- prologue: fill all stages, wait for tile 0 ----
    if constexpr (!PHASED) {
#pragma unroll 1
        for (int s = 0; s < NS; ++s) issue_tile(s);           // (rolled: most of a short kernel is straight-line code run once)
        wait_and_barrier<(NS - 1) * LPT, 0>();
        read_frags(0, 0, 0);
    }

    int stage = 0;
    // One k-step: the MFMAs of register buffer `cur`, row-tile by row-tile, with the fragment reads of the next step
    // (into the other buffer) and - in the last step of a k-tile - the wave loads of the tile that recycles this stage
    // issued between the rows.  The source order IS the issue order: every row ends in a scheduling fence.  Loads
    // come first (the next tile's fragment reads may not pass them: both touch LDS), over the first rows of the last
    // step; reads fill the remaining rows but leave the final row free, so that the barrier of the next tile does
    // not wait for a read that was just issued.
    auto kstep = [&](auto lastc, auto mayragc, const bool rag, const int cur, const int rd_stage_off, const int rd_kk,
                     const int kt, const int step) __attribute__((always_inline)) {
        constexpr bool LAST = decltype(lastc)::value;
        constexpr bool MAYRAG = decltype(mayragc)::value;
        constexpr int NLD = LAST ? LPT : 0;
        // rows of the last step that carry the tile's loads: HRN_LSPREAD 0 = none (all loads right behind the barrier),
        // 1 = the first quarter of the rows, 2 = half, 3 = all but the last two; spreading the requests smooths the
        // demand on the L2 (every workgroup of an XCD reaches its barrier at about the same time), at the price of a
        // later arrival of the tile.  The reads of the next step follow, the final row stays free (so that the barrier
        // of the next tile does not wait for a read that was just issued).
        constexpr int LWANT = LSPREAD == 0 ? 0 : (LSPREAD == 1 ? TM / 4 : (LSPREAD == 2 ? TM / 2 : TM - 2));
        constexpr int LROWS = NLD == 0 ? 0 : (LWANT < 1 ? ((LSPREAD > 0 && TM >= 2) ? 1 : 0) : (LWANT > TM - 1 ? TM - 1 : LWANT));
        constexpr int LFIRST = 0;                                                     // first load row
        constexpr int RFIRST_ROW = LROWS;                                             // first read row
        constexpr int RROWS_ALL = TM - LROWS;                                         // rows left for the reads
        constexpr int RROWS = RROWS_ALL >= 2 ? RROWS_ALL - 1 : RROWS_ALL;             // ... minus the free final row
        // the ragged form differs in the loads only, so the branch (wave-uniform) goes around just these
        auto loads = [&](auto firstc, auto countc) {
            if constexpr (MAYRAG) {
                if (rag) issue_loads(TrueC{}, stage, firstc, countc);
                else issue_loads(FalseC{}, stage, firstc, countc);
            } else {
                issue_loads(FalseC{}, stage, firstc, countc);
            }
        };
        if constexpr (LROWS == 0 && NLD > 0) loads(std::integral_constant<int, 0>{}, std::integral_constant<int, NLD>{});
        // uint8 products whose reads of the next step all go out in front of the first MFMAs (at most two rows): the fragments of this one, which go
        // through the vector ALU first, are waited for before, in a form that the compiler counts.  Without / with, us: 250x2500x8192 23.1 / 22.6,
        // 291x2704x4352 14.2 / 14.0, 150x3000x4096 12.9 / 12.7.  fp16 loses: 250x2500x8192 32.2 / 32.8, conv 3x3 32x56x56x64 -> 64 13.4 / 13.6; u8
        // convs are equal.
        if constexpr (DT == 1 && OP == 0 && !LAST && RROWS == 1) __builtin_amdgcn_s_waitcnt(0xC07F);        // lgkmcnt(0)
        v4i av = a_operand(cur, 0);
        auto row = [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i >= RFIRST_ROW && i - RFIRST_ROW < RROWS) {
                constexpr int f = NRD * (i - RFIRST_ROW) / RROWS, n = NRD * (i - RFIRST_ROW + 1) / RROWS - f;
#pragma unroll
                for (int r = f; r < f + n; ++r) read_slot(cur ^ 1, rd_stage_off, rd_kk, r);
            }
            if constexpr (LROWS > 0 && i >= LFIRST && i - LFIRST < LROWS) {
                constexpr int f = NLD * (i - LFIRST) / LROWS, n = NLD * (i - LFIRST + 1) / LROWS - f;
                loads(std::integral_constant<int, f>{}, std::integral_constant<int, n>{});
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = CHW ? mfma(av, fb[cur][j], acc[i][j]) : mfma(fb[cur][j], av, acc[i][j]);
            if constexpr (i + 1 < TM) av = a_operand(cur, i + 1);      // ready before the next row's MFMAs ask for it
            if constexpr (SCHED >= 1) __builtin_amdgcn_sched_barrier(0);
        };
        auto rows = [&](auto self, auto ic) -> void {
            row(ic);
            if constexpr (decltype(ic)::value + 1 < TM) self(self, std::integral_constant<int, decltype(ic)::value + 1>{});
        };
        rows(rows, std::integral_constant<int, 0>{});
        if constexpr (SCHED == 0) sched_hint<0, TM + TN, TM * TN, NLD>();
        bsum_step(cur, step);
    };
    // One k-tile.  P = register buffer that holds the fragments of its first k-step (the buffers alternate per
    // k-step, so with an odd number of k-steps per tile P alternates per tile).
    // MAYRAG: the k-tile this iteration fetches may be the partly filled last one of K (only then is the per-lane
    // masking of the loads compiled in; every other iteration runs the branch-free form).
    auto tile_body = [&](auto pc, auto mayragc, const int kt, const bool stores_between) __attribute__((always_inline)) {
        constexpr int P = decltype(pc)::value;
        const int stage_off = stage * STAGE_BYTES;
        const int next_stage = (stage + 1 == NS) ? 0 : stage + 1;
        set_masks();
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            const int cur = (kk + P) & 1;
            if (kk == KS - 1) {
                conv_addresses();
                // every fragment of tile kt is in registers: publish tile kt+1, recycle this stage
                if constexpr (PERS) {
                    if (stores_between && kt <= NS - 2) wait_and_barrier<(NS - 2) * LPT + STORES_PER_TILE, 0>();
                    else wait_and_barrier<(NS - 2) * LPT, 0>();
                } else {
                    wait_and_barrier<(NS - 2) * LPT, 0>();
                }
                const bool rag = begin_issue();
                        advance_reader();
                kstep(TrueC{}, mayragc, rag, cur, next_stage * STAGE_BYTES, 0, kt, kt * KS + kk);
                end_issue();
            } else {
                kstep(FalseC{}, FalseC{}, false, cur, stage_off, kk + 1, kt, kt * KS + kk);
            }
        }
        stage = next_stage;
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    // Iteration kt fetches k-tile kt + NS of the stream, so only iteration KT - 1 - NS can meet the partly filled last
    // k-tile (a persistent stream shorter than NS + 1 k-tiles wraps more than once: every iteration may then).
    const bool k_ragged = (Kb % BKB) != 0;
    const int kt_rag = k_ragged ? KT - 1 - NS : -1;
    const bool rag_any = k_ragged && PERS && kt_rag < 0;
    // the k-tiles [from, to) of the compute-side tile; P0/P1 alternate when a k-tile holds an odd number of k-steps
    auto tiles = [&](auto mayragc, const int from, const int to, const bool stores_between) __attribute__((always_inline)) {
        if constexpr (KS % 2 == 0) {
            for (int kt = from; kt < to; ++kt) tile_body(P0{}, mayragc, kt, stores_between);
        } else {
            int kt = from;
            if (kt < to && (kt & 1)) { tile_body(P1{}, mayragc, kt, stores_between); ++kt; }
            for (; kt < to; kt += 2) {
                tile_body(P0{}, mayragc, kt, stores_between);
                if (kt + 1 < to) tile_body(P1{}, mayragc, kt + 1, stores_between);
            }
        }
    };
    auto run_tile = [&](const bool stores_between) __attribute__((always_inline)) {
        if (rag_any) {
            tiles(TrueC{}, 0, KT, stores_between);
        } else {
            // three loops in a row instead of a test inside one: the hot loops carry no ragged-tile code at all
            const int cut = min(max(kt_rag, 0), KT);
            tiles(FalseC{}, 0, cut, stores_between);
            if (kt_rag >= 0) tiles(TrueC{}, cut, min(cut + 1, KT), stores_between);
            tiles(FalseC{}, kt_rag >= 0 ? min(cut + 1, KT) : cut, KT, stores_between);
        }
        if constexpr (SPLITK) {
            if (a.arrivals) greet();
        }
        store_tile();
    };
    // ---- phased schedule (PHASED) ----
    // Waves w and w + 4 share a SIMD.  Every wave alternates between a memory phase (fragment reads, tile fetches, waits)
    // and a matrix phase (16 or 8 MFMAs, nothing else but the sign flips in their shadow), a barrier after each, and waves
    // 4-7 enter the stream one barrier later: while one wave of a SIMD multiplies, the other moves data.
    //   A wave tile is cut into 2x2 quadrants; one of them, over the whole k-tile, is a step.  X is the operand with more
    // fragments, the steps of k-tile T are (X0,Y0) (X0,Y1) (X1,Y0) (X1,Y1).  Reads run one step ahead of their MFMAs and
    // are spread evenly over the steps:
    //   step 0: Y1 and a part of X1     step 1: the rest of X1     (of T)
    //   step 2: a part of X0            step 3: Y0 and the rest of X0     (of T + 1)
    // A half that has been read by everybody (it was read in step i, waited for in step i + 1) is refilled in step i + 2 or
    // later: step 1 fetches X0 and Y0, step 2 Y1, step 3 X1 of T + 2.  So every fetch has four to five steps (about 1.2 us)
    // to arrive, and a wait allows for the fetches that were issued after the half it is about.
    //   8192^3: matrix pipes busy in 81 % (fp16) and 73 % (u8 x s8) of the cycles, 73 - 76 and 60 % with the row-by-row
    // schedule; what bounds it then is power (the clock falls to 1.7 - 1.8 GHz): without the fetches in the loop the cycles fall
    // by 8.5 and 5 %, the time by 14 and 12 %.
    constexpr int HM = TM / 2, HN = TN / 2;                          // MFMA tiles of a half
    constexpr bool XA = TM >= TN;                                    // X is A
    constexpr int RA = HM * KS, RB = HN * KS;                        // fragments of a half
    constexpr int RX = XA ? RA : RB, RY = XA ? RB : RA, XP = (RX - RY) / 2;   // XP: the part of X read beside a half of Y
    v4i pa[2][PHASED ? HM : 1][KS], pb[2][PHASED ? HN : 1][KS];
    auto phased_run = [&]() __attribute__((always_inline)) {
        constexpr int LH = A_LPW / 2;                                // wave loads of a half (equal for A and B)
        // row of the tile at which load q of half h starts: half h is rows [h*wt/2, (h+1)*wt/2) of every wave row's wt rows
        auto row_of = [&](int wt, int h, int q) {
            const int u = q * NW + wave, per = wt / 2 / RPI;
            return (u / per) * wt + h * (wt / 2) + (u % per) * RPI;
        };
        // one descriptor per load, for the whole k-loop: its row block's base, and the bytes left from there
        rsrc_t dA[2][LH], dB[2][LH];
        int lA[2][LH], lB[2][LH];                                    // where the block goes in a stage
        live_cur = true;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < LH; ++q) {
                dA[h][q] = block_rsrc(baseA, a_bytes, (uint32_t)(m0 + row_of(WTM, h, q)) * (uint32_t)a.lda * ES, 0, 0);
                dB[h][q] = block_rsrc(baseB, b_bytes, (uint32_t)(n0 + row_of(WTN, h, q)) * (uint32_t)a.ldb * ES, 0, 0);
                lA[h][q] = __builtin_amdgcn_readfirstlane(row_of(WTM, h, q) * BKB);
                lB[h][q] = __builtin_amdgcn_readfirstlane(A_BYTES + row_of(WTN, h, q) * BKB);
            }
        const uint32_t chunkA = (uint32_t)((lpos ^ swz_of_row(row_of(WTM, 0, 0) + lrow)) * 16);
        const uint32_t chunkB = (uint32_t)((lpos ^ swz_of_row(row_of(WTN, 0, 0) + lrow)) * 16);
        const uint32_t offA = (uint32_t)lrow * (uint32_t)a.lda * ES + chunkA;
        const uint32_t offB = (uint32_t)lrow * (uint32_t)a.ldb * ES + chunkB;
        auto fetch = [&](auto isa, auto ragc, int h, int stg, int kt) __attribute__((always_inline)) {
            constexpr bool IA = decltype(isa)::value;
            const uint32_t ko = (uint32_t)kt * BKB;
            uint32_t v = IA ? offA : offB;
            if constexpr (decltype(ragc)::value) { if (ko + (IA ? chunkA : chunkB) >= Kb) v = OOB; }
#pragma unroll
            for (int q = 0; q < LH; ++q)
                load_chunk_to_lds(IA ? dA[h][q] : dB[h][q], lds + stg * STAGE_BYTES + (IA ? lA[h][q] : lB[h][q]), v, ko);
        };
        // fragments [from, to) of a half, in the order the MFMAs consume them (k-step outermost)
        auto read = [&](auto isa, int h, int stg, int from, int to) __attribute__((always_inline)) {
#pragma unroll
            for (int r = from; r < to; ++r) {
                if constexpr (decltype(isa)::value)
                    pa[h][r % HM][r / HM] = *(const v4i*)(lds + stg * STAGE_BYTES + a_lane + (h * HM + r % HM) * MT * BKB + (g16 ^ (r / HM * KSB)));
                else
                    pb[h][r % HN][r / HN] = *(const v4i*)(lds + stg * STAGE_BYTES + b_lane + (h * HN + r % HN) * MT * BKB + (g16 ^ (r / HN * KSB)));
            }
        };
        using X = std::integral_constant<bool, XA>;
        using Y = std::integral_constant<bool, !XA>;
        auto fence = [&]() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
        auto bar = [&]() __attribute__((always_inline)) { fence(); asm volatile("s_barrier" ::: "memory"); fence(); };
        // MFMAs of quadrant (A half h, B half g).  The uint8 sign flip of an A half happens at its first use (FLIP): the
        // first fragment in the memory phase before, each other one in the shadow of its predecessor's MFMAs (all of them
        // in the memory phases: 443 us instead of 413 for 8192^3).
        auto flip_first = [&](int h) __attribute__((always_inline)) { if constexpr (DT == 1) pa[h][0][0] ^= (int)0x80808080; };
        auto multiply = [&](auto flipc, int h, int g) __attribute__((always_inline)) {
            constexpr bool FLIP = DT == 1 && decltype(flipc)::value;
#pragma unroll
            for (int kk = 0; kk < KS; ++kk)
#pragma unroll
                for (int i = 0; i < HM; ++i)
#pragma unroll
                    for (int j = 0; j < HN; ++j) {
                        acc[h * HM + i][g * HN + j] = mfma(pb[g][j][kk], pa[h][i][kk], acc[h * HM + i][g * HN + j]);
                        if constexpr (FLIP) {
                            const int nr = kk * HM + i + 1;          // the next fragment, its registers spread over the HN MFMAs
                            if (nr < RA) {
#pragma unroll
                                for (int r = 4 * j / HN; r < 4 * (j + 1) / HN; ++r) pa[h][nr % HM][nr / HM][r] ^= (int)0x80808080;
                            }
                            fence();
                        }
                    }
        };
        using Yes = std::integral_constant<bool, true>;
        using No = std::integral_constant<bool, false>;
        // one k-tile; LOAD: tile T + 2 is fetched (ragc: it may be the partly filled last one)
        auto tile = [&](auto loadc, auto ragc, const int T) __attribute__((always_inline)) {
            constexpr bool LOAD = decltype(loadc)::value;
            const int stg = T & 1;
            auto landed = [&]() __attribute__((always_inline)) { wait_only<63, 0>(); fence(); };   // the reads of the step before
            landed();
            read(Y{}, 1, stg, 0, RY);
            read(X{}, 1, stg, 0, XP);
            flip_first(0);
            bar();
            multiply(Yes{}, 0, 0);
            bar();
            landed();
            read(X{}, 1, stg, XP, RX);
            if constexpr (LOAD) { fetch(X{}, ragc, 0, stg, T + 2); fetch(Y{}, ragc, 0, stg, T + 2); }
            if constexpr (!XA) flip_first(1);
            fence();
            wait_only<LOAD ? 5 * LH : 3 * LH, 15>();                 // X0 of T + 1
            bar();
            if constexpr (XA) multiply(No{}, 0, 1); else multiply(Yes{}, 1, 0);
            bar();
            landed();
            read(X{}, 0, stg ^ 1, 0, RX - XP);
            if constexpr (LOAD) fetch(Y{}, ragc, 1, stg, T + 2);
            if constexpr (XA) flip_first(1);
            fence();
            wait_only<LOAD ? 5 * LH : 2 * LH, 15>();                 // Y0 of T + 1
            bar();
            if constexpr (XA) multiply(Yes{}, 1, 0); else multiply(No{}, 0, 1);
            bar();
            landed();
            read(Y{}, 0, stg ^ 1, 0, RY);
            read(X{}, 0, stg ^ 1, RX - XP, RX);
            if constexpr (LOAD) fetch(X{}, ragc, 1, stg, T + 2);
            fence();
            wait_only<LOAD ? 4 * LH : 0, 15>();                      // Y1 and X1 of T + 1
            bar();
            multiply(No{}, 1, 1);
            bar();
        };
        auto whole = [&](int kt) __attribute__((always_inline)) {    // tile kt into stage kt, in the order of the loop
            auto all = [&](auto ragc) __attribute__((always_inline)) {
                fetch(X{}, ragc, 0, kt, kt); fetch(Y{}, ragc, 0, kt, kt); fetch(Y{}, ragc, 1, kt, kt); fetch(X{}, ragc, 1, kt, kt);
            };
            if ((uint32_t)(kt + 1) * BKB > Kb) all(Yes{}); else all(No{});
        };
        whole(0);
        if (KT > 1) { whole(1); wait_and_barrier<4 * LH, 0>(); }
        else wait_and_barrier<0, 0>();
        read(X{}, 0, 0, 0, RX);
        read(Y{}, 0, 0, 0, RY);
        if (wave >= NW / 2) bar();
        fence();
        int T = 0;
        for (const int full = KT - 2 - (Kb % BKB != 0 ? 1 : 0); T < full; ++T) tile(Yes{}, No{}, T);
        if (T + 2 < KT) { tile(Yes{}, Yes{}, T); ++T; }
        for (; T < KT; ++T) tile(No{}, No{}, T);                     // (reads one tile past the end, of either stage: never used)
        if (wave < NW / 2) bar();
    };
    if constexpr (PHASED) {
        phased_run();
        store_tile();
    } else if constexpr (PERS) {
        for (int ct = blockIdx.x; ct < total; ct += (int)gridDim.x) {
            tile_coords(ct, c_bz, c_tile_m, c_tile_n);
            m0 = c_tile_m * BM; n0 = c_tile_n * BN;
            // the stores of the previous tile's epilogue sit between the fetches that were issued before it and
            // the ones issued after it; while such a fetch is the one waited for, the wait allows for them
            run_tile(ct != (int)blockIdx.x && KT >= NS - 1);
            clear_acc();
        }
    } else {
        run_tile(false);
        if constexpr (SPLITK) {
            if (a.arrivals) fold_slices();
        }
    }
}

// a kernel that the instance has no room for is empty, and the host never launches it
// (all but the main kernel go through here, also where there is always room: called directly, the body of the channels-first
// kernel is scheduled 0.6 % slower, NCW conv1d 16 x 892 x 512 -> 512 30.56 -> 30.73 us)
template <bool ROOM, bool CHW, bool EXPAND, bool DEEP>
__device__ __forceinline__ void body_if(BodyArgs a) {
    if constexpr (ROOM) hrn_mfma_body<CHW, EXPAND, DEEP, BodyArgs>(a);
}

// Where 256 registers are enough for a wave, the compiler is told so.  Kernels of 16x16 MFMAs that are given 512 can get accumulators in the
// other half, copied through the lower one in the k-loop (60 and 100 moves in two u8 instances; those of 32x32 MFMAs that were looked
// at have none).  Given 512 / told, us: fp16 3x3 in 4 slices 2x20x20x432 -> 240 11.2 / 10.4, 3x3 32x7x7x512 -> 512 28.8 / 26.8, u8 3x3
// 15x34x33x384 -> 144 21.9 / 21.6.  Deep kernels fill the LDS with one workgroup, which would be reason enough for 512 registers, so those of
// products take their LDS dynamically: u8 x s8 1500x1536x4112 26.2 / 22.9, fp16 1500x1536x2048 17.25 / 17.2.  (Those of convs gain nothing by
// it: 5x5 10x30x30x208 -> 128 35.4 -> 36.6, 3x3 16x28x28x256 -> 160 23.9 -> 23.5.)
// The rule counts registers, not the waves that the LDS lets in.  Two instances whose LDS admits more end two registers above a wave's share and
// run with one wave less: u8 window conv 64x128x64, 4x1 waves, 4 stages (130), as fast with it (asked for four waves it spills 8 bytes:
// 28x28x128 -> 128 at batch 32 15.93 / 15.92, at 128 39.6 / 39.6), and u8 GEMM 128x128x64, 4x1 waves, 3 stages (170; asked for three, 16
// bytes spilled: 2048x2048x1024 14.5 / 14.1, 4096x4096x256 22.9 / 23.5, 3000x2504x720 17.5 / 17.7).  Others keep 512 registers as their
// static LDS admits one wave.
constexpr int MIN_WPE = NT > 256 ? (NT + 255) / 256 : (TM * TN * ACC_N + 8 * (TM + TN) <= 208 ? 2 : 1);      // (accumulators, two sets of fragments)

}  // namespace

#if HRN_WPE > 0
#define HRN_ENTRY extern "C" __global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(HRN_WPE, HRN_WPE)))
#else
#define HRN_ENTRY extern "C" __global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(MIN_WPE)))
#endif

// Which kernels this code object holds: those of the instance's own launches, the channels-first ones, or those that also
// expand their input.
#ifndef HRN_PART
#define HRN_PART 0
#endif

#if HRN_PART == 0
HRN_ENTRY hrn_mfma_kernel(const KArgs a) { hrn_mfma_body<false, false, false, BodyArgs>(a); }
HRN_ENTRY hrn_mfma_kernel_deep(const KArgs a) { body_if<HAS_DEEP, false, false, true>(a); }
#elif HRN_PART == 1
HRN_ENTRY hrn_mfma_kernel_chw(const KArgs a) { body_if<HAS_CHW, true, false, false>(a); }
HRN_ENTRY hrn_mfma_kernel_chw_deep(const KArgs a) { body_if<HAS_DEEP, true, false, true>(a); }
#else
HRN_ENTRY hrn_mfma_kernel_chw_expand(const KArgs a) { body_if<HAS_CHW, true, true, false>(a); }
HRN_ENTRY hrn_mfma_kernel_chw_expand_deep(const KArgs a) { body_if<HAS_DEEP, true, true, true>(a); }
#endif
