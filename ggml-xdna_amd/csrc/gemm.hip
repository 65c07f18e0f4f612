// The bfp16 GEMM: C[M][N] = A[M][K] . W[N][K]^T, A the expanded activation
// operand (the bfp16 pack stored decoded as bf16, zest_layout.h) and W a
// packed bfp16 weight from the resident cache.
//
// Per workgroup a BM x BN output tile, in K-steps of 64 (one tile-layout
// column chunk), by two kinds of waves:
//   * producer waves load the W slab (bfp16 units: 16 mantissas + their 2
//     exponent bytes) two steps ahead into registers, expand the units
//     losslessly to bf16 (zest::expand16) and store them into a ring of three
//     LDS stages; LDS rows are 64 bf16 with the 16-byte chunks XOR-swizzled by
//     row so the stores and the fragment reads are free of bank conflicts;
//   * consumer waves (CWM of them, each WM rows by all BN columns) load their
//     A fragments straight from memory into registers, two steps ahead (the
//     expanded layout holds each fragment as one contiguous 1 KB), read the W
//     fragments from LDS and run v_mfma_f32_32x32x16_bf16, each lane's eight
//     K values of an operand exactly one bfp16 block, accumulating in fp32.
// One consumer and one producer wave share each SIMD, so the producer's
// expansion and the consumer's MFMAs issue side by side. While the consumers
// work on step k, the producers fill step k+2, and step k+1 is complete, so
// the consumers read its first fragments before step k ends. One barrier per
// K-step. The store is fp32 row-major, as the reference's output mode 0
// (kernels/bfp16_gemm/aie_kernels/aie2p/mm_bfp_acc.cc:106-116, 258-278).
// A launch of several rounds of whole tiles runs as persistent workgroups,
// one a CU, each walking its XCD's tiles and fetching the next tile's first
// steps while it finishes the current one (gemm_kernel_tiles; mixed launches:
// gemm_kernel_mixed_tiles).
#include <algorithm>
#include <cmath>
#include <atomic>
#include <map>
#include <mutex>
#include <thread>
#include <type_traits>
#include <utility>
#include <vector>

#include "zest_common.h"
#include "zest_device.h"

#ifndef ZEST_GEMM_XCD
#define ZEST_GEMM_XCD 1  // XCD-aware workgroup -> tile order
#endif
#ifndef ZEST_GEMM_GROUP_M
#define ZEST_GEMM_GROUP_M 4  // tile rows per group of the tile order
#endif

// The split-K workspace of zest_gemm_group_noalloc: one static array per GPU
// (the code object's own copy on each device, held until the process ends),
// ZEST_NOALLOC_PARTIAL_BYTES of fp32 partial sums, then
// ZEST_NOALLOC_COUNTERS counters. Host code never passes `scratch` itself to
// a kernel (on the host it names a stand-in, not device memory): it uses the
// device address that scratch_address() looks up per device.
static __device__ __align__(256) uint8_t scratch[ZEST_NOALLOC_PARTIAL_BYTES + ZEST_NOALLOC_COUNTERS * 4];

namespace {

// Epilogues other than the GLU kinds (which are >= 0)
constexpr int EPI_PLAIN = -1, EPI_RESIDUAL = -2;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// BM x BN tile; CWM x CWN consumer waves, each a WM x WN block of 32x32 MFMA
// tiles (TI x TJ of them; consumer w takes row block w % CWM, column block
// w / CWM); NP/64 producer waves (as many as the consumers' row blocks by
// default). LDS holds the expanded W ring; after the K loop each consumer
// wave uses WM x WN floats of it for its epilogue. MINB workgroups a CU at
// least (the launch bound). KG K-groups: the workgroup holds KG copies of
// these waves, each with a ring of its own, and K-group g takes the g-th of
// KG equal runs of the tile's K-steps; the groups' sums are added in LDS,
// in group order (run_tile).
template <int BM_, int BN_, int CWM_, int NP_ = 64 * CWM_, int MINB_ = 1, int CWN_ = 1, int NP1_ = 0, int KG_ = 1>
struct gemm_cfg {
    static constexpr int BM = BM_, BN = BN_, CWM = CWM_, CWN = CWN_, MINB = MINB_, KG = KG_;
    static constexpr int NC = 64 * CWM * CWN;  // consumer threads
    static constexpr int NP = NP_;             // producer threads
    static constexpr int NP1 = NP1_;           // of them, the last NP1 take one W unit each, not two
    static constexpr int NW = (NC + NP) / 64;  // waves of a K-group
    static constexpr int NT = KG * (NC + NP);
    static constexpr int WM = BM / CWM, WN = BN / CWN;
    static constexpr int TI = WM / 32, TJ = WN / 32;
    static constexpr int NP2 = NP - NP1;    // producer threads of two W units (two blocks each) a K-step
    static constexpr int ROWB = 128;        // LDS bytes per row (64 bf16)
    static constexpr int STAGE = BN * ROWB;
    static constexpr int STAGES = 3;
    static constexpr size_t RING = (size_t) STAGES * STAGE;
    // K-group g's ring at g * RING; after the K loop, the epilogue regions
    // of group 0's waves in [0, BM*BN*4) and group g's sums at g * BM*BN*4
    static constexpr size_t LDS_BYTES = KG * (RING > (size_t) BM * BN * 4 ? RING : (size_t) BM * BN * 4);
    // a split-K launch: FIX partial tiles of the fixup at once, each
    // consumer wave's share of partial i at i * BM*BN*4 (as K-group i's sums)
    static constexpr size_t LDS_MAX = 163840 / MINB, TILE_BYTES = (size_t) BM * BN * 4;
    static constexpr int FIX = LDS_MAX / TILE_BYTES < 4 ? (int) (LDS_MAX / TILE_BYTES) : 4;
    static constexpr size_t LDS_SPLIT = LDS_BYTES > FIX * TILE_BYTES ? LDS_BYTES : FIX * TILE_BYTES;
    // a persistent launch: the GLU epilogue's staging (WM rows of 16 TJ + 4
    // floats a wave) above the ring
    static constexpr size_t LDS_APART = (size_t) STAGES * STAGE + (size_t) (NC / 64) * WM * (16 * TJ + 4) * 4;
    static constexpr size_t LDS_TILES = LDS_BYTES > LDS_APART ? LDS_BYTES : LDS_APART;
    static_assert(NP2 % 64 == 0 && NP1 % 64 == 0 && NP2 / 32 + NP1 / 64 == BN / 16,
                  "32 two-unit or 64 one-unit producer threads a 16-row W tile, whole waves of each");
    static_assert(WM % 32 == 0 && WN % 32 == 0, "wave tile must be whole 32x32 MFMA tiles");
};

// LDS rows are 128 bytes = 8 chunks of 16 bytes (one block as bf16 each);
// chunk c of row r is stored at position c ^ swz(r). swz is a linear map of
// the low four bits b of r, (b0^b1^b2, b1, b2^b3), for which no access has a
// bank conflict, whether 8 lanes meet in 128 bytes of banks or 16 in 256:
//   * a fragment read (one chunk of consecutive rows): swz takes 8 values
//     over 8 rows, and over the 8 even and the 8 odd rows of 16;
//   * a producer's store of two lanes a row (chunks c and c ^ 4): swz % 4
//     takes 4 values over 4 rows, and over the even and the odd rows of 8;
//   * a one-unit producer's, four lanes a row (chunks c, c ^ 2, c ^ 4, c ^ 6):
//     swz % 2 differs within two rows, and between rows r and r + 2.
// It depends only on r % 16, so the +32-row offsets of the MFMA tiles stay
// immediates.
__device__ inline int swz(int row) {
    return ((row ^ (row >> 1) ^ (row >> 2)) & 1) | (row & 2) | ((((row >> 2) ^ (row >> 3)) & 1) << 2);
}

__device__ inline void lds_put(uint8_t * smem, int off, uint4 v) { *reinterpret_cast<uint4 *>(smem + off) = v; }

__device__ inline bf16x8 lds_get(const uint8_t * smem, int off) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(smem + off));
}

__device__ inline uint4 load16(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
    return make_uint4(v[0], v[1], v[2], v[3]);
}

// A producer thread's registers for one K-step's U W units.
template <class C, int U = 2>
struct stage_regs {
    uint4 wm[U];
    uint32_t we;  // the units' exponent bytes: unit 0 in bits 0-15, unit 1 in bits 16-31
};

typedef __attribute__((address_space(3))) void * lds_ptr_t;

// The producer side. W loads go through a buffer resource: the slab's byte
// offset is wave-uniform (a scalar offset), the lane's place in it a fixed
// vector offset. The hardware range check covers the vector offset only, so
// every slab offset a load is given names a K-step of the operand (callers
// clamp the steps past the end to the last one). With U = 2, thread p takes
// two adjacent units of tile p/32 of the W slab: row p/2%16, column quarters
// 2h and 2h+1 with h = p%2, i.e. 32 contiguous mantissa bytes (two 16-byte
// loads) and 4 contiguous exponent bytes (one 4-byte load). With U = 1 (the
// slab's last tiles, after the NP2/32 of the two-unit threads), thread p
// takes one unit of tile NP2/32 + p/64: row p/4%16, quarter p%4 (16 mantissa
// bytes, 2 exponent bytes). Consecutive lanes so take consecutive bytes of a
// tile: the vector cache serves such loads at 64 B/clk a CU, and at 32 with
// consecutive lanes on consecutive rows, 64 bytes apart (2048 x 7168 x 2560 in
// one group 66 -> 64.8 us, 1024 x 2560 x 2560 alone 26 -> 25.3).
template <class C, int U = 2>
struct producer {
    static_assert(U == 1 || U == 2, "one or two W units a thread");
    __amdgpu_buffer_rsrc_t rw;
    int vwm, vwe;          // lane offsets: W mantissas, W exponents
    int stw[U][2];         // LDS offsets of the W units' two chunks each

    __device__ producer(const uint8_t * W, int64_t w_bytes, int p) {
        rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(W), (short) 0, (int) w_bytes, 0x00020000);
        const int t = U == 2 ? p >> 5 : C::NP2 / 32 + (p >> 6), row = (U == 2 ? p >> 1 : p >> 2) & 15;
        const int q0 = U == 2 ? 2 * (p & 1) : p & 3;  // the first unit's quarter
        vwm = t * ZEST_TILE_BYTES + row * ZEST_TILE_K + q0 * 16;
        vwe = t * ZEST_TILE_BYTES + ZEST_TILE_MANT + row * 8 + q0 * 2;
        const int wrow = t * 16 + row, sw = swz(wrow);
#pragma unroll
        for (int i = 0; i < U; i++) {
            stw[i][0] = wrow * C::ROWB + ((2 * (q0 + i)) ^ sw) * 16;
            stw[i][1] = wrow * C::ROWB + ((2 * (q0 + i) + 1) ^ sw) * 16;
        }
    }

    __device__ void load_w(stage_regs<C, U> & st, int w_off) const {
        st.wm[0] = load16(rw, vwm, w_off);
        if constexpr (U == 2) {
            st.wm[1] = load16(rw, vwm + 16, w_off);
            st.we = __builtin_amdgcn_raw_buffer_load_b32(rw, vwe, w_off, 0);
        } else {
            st.we = __builtin_amdgcn_raw_buffer_load_b16(rw, vwe, w_off, 0);
        }
    }

    // W unit i of a step by the branch-free fast expansion, stored.
    __device__ void store_w_unit(const stage_regs<C, U> & st, int i, zest::zest_u16x2 d, uint8_t * smem, int stage) const {
        uint32_t b[8];
        zest::expand16_by(st.wm[i], d, b);
        lds_put(smem, stw[i][0] + stage, make_uint4(b[0], b[1], b[2], b[3]));
        lds_put(smem, stw[i][1] + stage, make_uint4(b[4], b[5], b[6], b[7]));
    }

    // Every unit of the step by the general expansion, stored.
    __device__ void store_w_general(const stage_regs<C, U> & st, uint8_t * smem, int stage) const {
#pragma unroll
        for (int i = 0; i < U; i++) {
            uint32_t b[8];
            zest::expand16(st.wm[i], i ? st.we >> 16 : st.we & 0xffffu, b);
            lds_put(smem, stw[i][0] + stage, make_uint4(b[0], b[1], b[2], b[3]));
            lds_put(smem, stw[i][1] + stage, make_uint4(b[4], b[5], b[6], b[7]));
        }
    }

    // The units take the branch-free fast expansion; a step with a unit whose
    // exponent bytes need the general one is redone behind a single
    // wave-uniform branch, which real weights almost never take. Its condition
    // is made first, so it is there long before the branch. Zero blocks (byte
    // 0: the padding rows past N, the padding columns past K) come through it
    // too, but a zero mantissa is zero whatever its exponent, so only units
    // with a nonzero one are redone: else every step of the tiles that reach
    // past N would be, and a launch takes as long as its slowest tile (1884 x
    // 2316 x 11808 179 -> 106 us, 512 x 32001 x 4096 123 -> 108; 2304 and 32000
    // columns take 103 and 104).
    __device__ void store_w(const stage_regs<C, U> & st, uint8_t * smem, int stage) const {
        zest::zest_u16x2 d[U];
#pragma unroll
        for (int i = 0; i < U; i++) d[i] = zest::exp_offsets(st.we, i);
        const bool general = zest::exp_general(U == 2 ? __builtin_elementwise_max(d[0], d[U - 1]) : d[0]);
        const uint64_t any = __builtin_amdgcn_ballot_w64(general);
#pragma unroll
        for (int i = 0; i < U; i++) {
            store_w_unit(st, i, d[i], smem, stage);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (__builtin_expect(any != 0, 0)) {
            bool redo = false;
#pragma unroll
            for (int i = 0; i < U; i++)
                redo |= zest::exp_general(d[i]) && (st.wm[i].x | st.wm[i].y | st.wm[i].z | st.wm[i].w) != 0u;
            if (__builtin_amdgcn_ballot_w64(redo)) store_w_general(st, smem, stage);
        }
    }
};

// The consumers' A fragments come from memory straight into registers.
// Fragment i of sub-step s is sub-tile s of the 32-row group wm*WM/32 + i of
// the tile's K-step slab: lane l takes row l%32, chunk 2s + l/32 (one block
// as bf16, the MFMA's A operand), the 16 bytes at 32(l%32) + 16(l/32), so the
// wave's load covers one contiguous 1 KB. The K-step's offset is a scalar
// offset, which the range check does not cover: callers pass only steps of
// the operand.
template <class C>
struct a_loader {
    __amdgpu_buffer_rsrc_t ra;
    int va[C::TI];

    __device__ a_loader(const uint8_t * A, int64_t a_bytes, int wm, int lane) {
        ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(A), (short) 0, (int) a_bytes, 0x00020000);
#pragma unroll
        for (int i = 0; i < C::TI; i++)
            va[i] = (wm * C::WM / 32 + i) * ZEST_XGROUP_BYTES + (lane & 31) * 32 + (lane >> 5) * 16;
    }

    __device__ bf16x8 load(int i, int s, int a_off) const {
        return __builtin_bit_cast(bf16x8,
                                  __builtin_amdgcn_raw_buffer_load_b128(ra, va[i] + s * ZEST_XSUB_BYTES, a_off, 0));
    }

    // every fragment of a K-step
    __device__ void load_step(bf16x8 (&a)[4][C::TI], int a_off) const {
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < C::TI; i++) a[s][i] = load(i, s, a_off);
    }
};

// One K-step of a consumer wave: A from registers `a` (this step's,
// loaded two steps ago), W fragments from the stage at `cur`, read a
// sub-step ahead (sub-step 0 of stage `nxt` during the last). As each
// sub-step's MFMAs are issued, its A registers are reloaded with the same
// fragments of the step at a_next (LOAD), two steps ahead, so a load has two
// steps to land. The scheduling groups interleave the W reads and A loads
// with the MFMAs.
template <class C, bool LOAD>
__device__ inline void consume(f32x16 (&acc)[C::TI][C::TJ], bf16x8 (&a)[4][C::TI], bf16x8 (&bw)[2][C::TJ],
                               const uint8_t * smem, const int (&fw)[4], int cur, int nxt, const a_loader<C> & al,
                               int a_next) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int off = s < 3 ? fw[s + 1] + cur : fw[0] + nxt;
#pragma unroll
        for (int j = 0; j < C::TJ; j++) bw[(s + 1) & 1][j] = lds_get(smem, off + j * 32 * C::ROWB);
#pragma unroll
        for (int i = 0; i < C::TI; i++)
#pragma unroll
            for (int j = 0; j < C::TJ; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s][i], bw[s & 1][j], acc[i][j], 0, 0, 0);
        if (LOAD) {
#pragma unroll
            for (int i = 0; i < C::TI; i++) a[s][i] = al.load(i, s, a_next);
        }
#pragma unroll
        for (int q = 0; q < C::TI * C::TJ; q++) {
            if (q < C::TJ) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // a W fragment read
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                  // an MFMA
            if (LOAD && (q + 1) % C::TJ == 0) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // an A load
        }
    }
}

// The fp32 store. 32x32 accumulator layout: lane l, register v holds row
// (v/4)*8 + (l/32)*4 + v%4 and column l%32 of its MFMA tile. Stores go
// through a buffer resource covering rows [0, M) of C, so rows past M are
// dropped by the hardware range check on the vector offset (the whole byte
// offset is kept there); columns past N are masked per lane. Also ORs 1 into
// *nonfinite if any stored value is NaN or infinite.
// With `res` (RES), the consumer wave's WM x WN block of the residual comes
// into the wave's own LDS region first (LDS DMA, every load in flight at
// once: the ring is free after the K loop), and each output is acc + res
// (res may be Cout itself: every element is read before it is written, by
// the lane that writes it).
template <class C, bool RES = false>
__device__ inline void store_tile(const f32x16 (&acc)[C::TI][C::TJ], float * Cout, int64_t M, int64_t N, int64_t ldc,
                                  int64_t m0, int64_t n0, int wm, int wn, int lane, uint32_t * nonfinite,
                                  const float * res = nullptr, int64_t ldr = 0, uint8_t * smem = nullptr,
                                  int wave = 0) {
    const __amdgpu_buffer_rsrc_t rc =
        __builtin_amdgcn_make_buffer_rsrc(Cout, (short) 0, (int) (M * ldc * 4), 0x00020000);
    const int khalf = lane >> 5;
    const int row0 = (int) m0 + wm * C::WM;
    const float * rl = nullptr;  // the residual block in LDS: WM rows of WN floats
    if constexpr (RES) {
        // the block row-major in the region: instruction q fills bytes
        // [1024q, 1024q + 1024), lane l the 16 at 1024q + 16l, i.e. floats
        // f = 256q + 4l, row f / WN and column f % WN (a lane's 4 floats never
        // straddle rows: WN % 4 == 0); the whole byte offset is in the vector
        // offset, so the range check turns rows past M into zeros instead of
        // reads past the residual
        static_assert(C::WM * C::WN % 256 == 0 && C::WN % 4 == 0, "whole DMA instructions");
        uint8_t * region = smem + wave * (C::WM * C::WN * 4);
        const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(res), (short) 0, (int) (M * ldr * 4), 0x00020000);
#pragma unroll
        for (int q = 0; q < C::WM * C::WN / 256; q++) {
            const int f = 256 * q + 4 * lane, r = f / C::WN, c = f - r * C::WN;
            const int voff = (int) ((row0 + r) * ldr * 4 + (n0 + wn * C::WN + c) * 4);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rr, (lds_ptr_t) (region + q * 1024), 16, voff, 0, 0, 0);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        rl = reinterpret_cast<const float *>(region);
    }
    bool bad = false;
#pragma unroll
    for (int j = 0; j < C::TJ; j++) {
        const int64_t col = n0 + wn * C::WN + j * 32 + (lane & 31);
        if (col < N) {
            const int voff = (int) (col * 4 + (int64_t) khalf * 4 * ldc * 4);
#pragma unroll
            for (int i = 0; i < C::TI; i++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    float x = acc[i][j][v];
                    const int rt = i * 32 + (v >> 2) * 8 + khalf * 4 + (v & 3);  // row in the wave's block
                    if constexpr (RES) x += rl[rt * C::WN + j * 32 + (lane & 31)];
                    // only rows that are stored count
                    bad |= row0 + rt < M && !(__builtin_fabsf(x) <= 3.402823466e38f);
                    const int roff = (row0 + i * 32 + (v >> 2) * 8 + (v & 3)) * (int) ldc * 4;
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), rc, voff + roff, 0, 0);
                }
        }
    }
    if (nonfinite && __any(bad) && lane == 0) atomicOr(nonfinite, 1u);
}

// The fused gate/up epilogue: the weight is a gate/up pair interleaved by
// 32-row groups (zest_convert_weight_gu), so accumulator tiles 2p and 2p+1 of
// a wave hold the gate and the up values of the same 32 output columns, lane
// l%32 = column. Computes h = glu(g, u) in fp32 (the GLU kernel's arithmetic)
// and optionally stores it. For the down projection's operand the wave stages
// its WM x HW block of h in LDS (the K loop is over and every stage consumed),
// then reads it back by rows: lane l takes 16 consecutive columns of one row,
// i.e. two whole bfp16 blocks, which it encodes and stores decoded as the
// activation packer does (store_expanded16: two 16-byte stores). Each wave
// has its own LDS region, so no barrier is needed: a wave's LDS operations
// complete in order. Rows and columns past M and F come from zero padding and
// store zeros, as the packer's padding is. With APART the regions lie above
// the W ring (a persistent workgroup's producers fill the next tile's first
// stages meanwhile); else each is the wave's region of the split-K fixup.
template <class C, int KIND, bool APART = false>
__device__ inline void store_glu(const f32x16 (&acc)[C::TI][C::TJ], uint8_t * smem, uint8_t * xout, float * h,
                                 int64_t ldh, int64_t M, int64_t F, int64_t m0, int64_t n0, int wave, int wm, int wn,
                                 int lane, uint32_t * nonfinite) {
    constexpr int NPAIR = C::TJ / 2, HW = 32 * NPAIR;  // gate/up pairs; h columns of the wave
    static_assert(C::TJ % 2 == 0 && HW <= ZEST_TILE_K, "the fused GLU needs whole gate/up pairs in one K chunk");
    // staged rows of HW + 4 floats: the 16-lane groups of the row reads below
    // (rows r..r+15, one 16-byte column chunk) then hit distinct banks
    constexpr int P = HW + 4;
    static_assert(P <= C::WN && (size_t) C::BM * C::BN * 4 <= C::LDS_BYTES, "staging must fit the wave's region");
    static_assert(P == 16 * C::TJ + 4 && C::LDS_APART <= C::LDS_TILES, "staging above the ring must fit");
    float * st = reinterpret_cast<float *>(APART ? smem + C::STAGES * C::STAGE + wave * (C::WM * P * 4)
                                                 : smem + wave * (C::WM * C::WN * 4));
    const int64_t c0 = n0 / 2 + wn * HW;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < C::TI; i++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int rw = i * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);  // row in the wave tile
            const int64_t row = m0 + wm * C::WM + rw;
#pragma unroll
            for (int q = 0; q < NPAIR; q++) {
                const float g = acc[i][2 * q][v], u = acc[i][2 * q + 1][v];
                const float hv = zest::glu(KIND, g, u);
                const int64_t col = c0 + q * 32 + (lane & 31);
                bad |= !(__builtin_fabsf(g) <= 3.402823466e38f) || !(__builtin_fabsf(u) <= 3.402823466e38f) ||
                       !(__builtin_fabsf(hv) <= 3.402823466e38f);
                if (h && row < M && col < F) h[row * ldh + col] = hv;
                if (xout) st[rw * P + q * 32 + (lane & 31)] = hv;
            }
        }
    if (xout) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int64_t M_pad = zest_rows_padded(M);
        // a pass reads RPP rows, lane l taking row l%RPP and 16-column chunk l/RPP
        constexpr int QPR = HW / 16, RPP = 64 / QPR;
        const int q = lane / RPP;
#pragma unroll
        for (int j = 0; j < C::WM / RPP; j++) {
            const int rw = j * RPP + lane % RPP;
            const float4 * p = reinterpret_cast<const float4 *>(st + rw * P + q * 16);
            float v[16];
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const float4 f = p[x];
                v[4 * x] = f.x;
                v[4 * x + 1] = f.y;
                v[4 * x + 2] = f.z;
                v[4 * x + 3] = f.w;
            }
            zest::store_expanded16(xout, M_pad, m0 + wm * C::WM + rw, c0 + q * 16, v);
        }
        // The last tile row also zeroes the operand's rows that no tile
        // reaches, [m0 + BM, M_pad): a row's HW columns are Z lanes of 16
        // bytes, so a wave covers 64/Z rows at a time.
        constexpr int Z = HW / 8, RZ = 64 / Z;
        if (m0 + C::BM >= M)
            for (int64_t row = m0 + C::BM + wm * RZ + lane / Z; row < M_pad; row += RZ * C::CWM)
                *reinterpret_cast<uint4 *>(xout + zest_xoffset(row, c0 + (lane % Z) * 8, M_pad)) = make_uint4(0, 0, 0, 0);
    }
    if (nonfinite && __any(bad) && lane == 0) atomicOr(nonfinite, 1u);
}

// One weight of a launch. Weights that share the activation operand (a
// group: q, k and v) run as one launch; their column tiles follow each other.
struct gemm_weight {
    const uint8_t * w;  // packed bfp16
    float * c;          // fp32 output (plain epilogue)
    int64_t n, ldc;
    int w_kstride;      // bytes between K-steps of the packed weight
    int tile0;          // its first column tile in the launch
};

struct gemm_params {
    const uint8_t * a;  // expanded activations
    int64_t M;
    int a_kstride;      // bytes between K-steps of the activation operand
    int nk;             // K-steps
    int mt, nt;         // tile rows; column tiles of all weights
    int nw;             // weights
    gemm_weight wt[ZEST_GEMM_MAX_GROUP];
    uint8_t * xout;     // fused GLU outputs (one weight)
    float * h;
    int64_t ldh;
    const float * res;  // residual added by the EPI_RESIDUAL epilogue (one weight)
    int64_t ldr;
    uint32_t * nonfinite;
    // Split-K: with splits S > 1, workgroup v takes unit v of the sequence
    // (split 0 of every tile, split 1 of every tile, ...): split s of a tile is
    // its K-steps [s*nk/S, (s+1)*nk/S). The workgroups running one split walk
    // K side by side, as whole tiles do, so they keep sharing A and W slabs in
    // L2. The splits of a tile are summed through `partial` (BM*BN floats per
    // unit) and `counters` (one per tile and consumer wave, zero between
    // launches).
    int splits;
    float * partial;
    uint32_t * counters;
    // Mixed launches (gemm_kernel_mixed): the first nbig tiles (mt x nt
    // tiles of the big shape) run whole, each of the others as two tiles of
    // half its rows (the small shape).
    int nbig;
};

// Byte offset of a consumer wave's float4 (i, j, quad q) in a unit's partial
// sums: [unit][wave][i][j][quad][lane], so each store and load instruction
// covers 1 KB contiguous.
template <class C>
__device__ inline int partial_off(int unit, int wave, int i, int j, int q, int lane) {
    return (((((unit * (C::NC / 64) + wave) * (C::TI * C::TJ) + i * C::TJ + j) * 4 + q) * 64) + lane) * 16;
}

// Cache policy of the partial sums' loads and stores: sc1, coherent at device
// scope (the writer and the reader may sit on different XCDs, whose L2s are
// not coherent with each other). No fence is used: a device-scope fence
// writes back and invalidates the XCD's whole L2, which would take the A and
// W slabs the other workgroups there are sharing.
#define ZEST_SC1 16

// Split-K fixup of one consumer wave's block of tile t, split `split` of
// p.splits. Writes this wave's sums to its unit's partial (sc1 stores), waits
// for them to be acknowledged, and counts itself in. The wave that arrives
// last forms ((p[S-1] + p[S-2]) + p[S-3]) + ... + p[0] and resets the
// counter. The order is fixed, so the result does not depend on arrival
// order; since a + b == b + a exactly, a last wave of split S-1 or S-2 (the
// usual case: splits run in that order) starts from its own sums in acc and
// reads one partial fewer, others read their own back like the rest. Up to
// C::FIX partials at a time come into the wave's own LDS regions by LDS DMA
// (all of their loads in flight at once, no registers held; one round trip to
// the coherent level each cost 0.9 us a split), then are added from there. LDS is
// free: the K loop is over, and this workgroup has no other tile. Returns
// true for the last wave, whose acc then holds the tile's sums. No wave
// waits for another.
template <class C>
__device__ inline bool fixup(f32x16 (&acc)[C::TI][C::TJ], const gemm_params & p, uint8_t * smem, int t, int split,
                             int wave, int lane) {
    constexpr int PARTS = C::TI * C::TJ * 4;  // 1 KB pieces of a wave's share
    const int T = p.mt * p.nt, S = p.splits;
    const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(
        p.partial, (short) 0, (int) ((int64_t) T * S * C::BM * C::BN * 4), 0x00020000);
    const int me = split * T + t;
#pragma unroll
    for (int i = 0; i < C::TI; i++)
#pragma unroll
        for (int j = 0; j < C::TJ; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 x = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                                             acc[i][j][4 * q + 3]);
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), rp,
                                                       partial_off<C>(me, wave, i, j, q, lane), 0, ZEST_SC1);
            }
    // the stores have reached the coherent level before the count goes up
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t * counter = p.counters + (int64_t) t * (C::NC / 64) + wave;
    uint32_t old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    old = __shfl(old, 0);
    asm volatile("" ::: "memory");
    if (old != (uint32_t) (S - 1)) return false;
    constexpr int REGION = C::WM * C::WN * 4, TILE = C::BM * C::BN * 4;
    uint8_t * region = smem + wave * REGION;
    // acc already holds p[S-1] (split S-1) or its commuted first sum's other
    // operand (split S-2)
    const bool own = split >= S - 2;
    for (int v0 = own ? 1 : 0; v0 < S; v0 += C::FIX) {
        for (int v = v0; v < S && v < v0 + C::FIX; v++) {
            // operand v of the sum is p[S-1-v], except that a split-S-2 wave's
            // second operand is p[S-1] (its own sums stand in for p[S-2]). u is
            // uniform but derived from the split, which the tile arithmetic can
            // leave in a vector register, and a DMA's scalar offset taken from
            // one costs a loop per load
            const int u =
                __builtin_amdgcn_readfirstlane(own && v == 1 ? (split == S - 1 ? S - 2 : S - 1) : S - 1 - v);
            const int base = partial_off<C>(u * T + t, wave, 0, 0, 0, 0);
            uint8_t * to = region + (v - v0) * TILE;
#pragma unroll
            for (int x = 0; x < PARTS; x++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rp, (lds_ptr_t) (to + x * 1024), 16, lane * 16,
                                                         base + x * 1024, 0, ZEST_SC1);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        for (int v = v0; v < S && v < v0 + C::FIX; v++) {
            const uint8_t * from = region + (v - v0) * TILE;
#pragma unroll
            for (int i = 0; i < C::TI; i++)
#pragma unroll
                for (int j = 0; j < C::TJ; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float4 x =
                            *reinterpret_cast<const float4 *>(from + ((i * C::TJ + j) * 4 + q) * 1024 + lane * 16);
                        if (v == 0) {
                            acc[i][j][4 * q] = x.x;
                            acc[i][j][4 * q + 1] = x.y;
                            acc[i][j][4 * q + 2] = x.z;
                            acc[i][j][4 * q + 3] = x.w;
                        } else {
                            acc[i][j][4 * q] += x.x;
                            acc[i][j][4 * q + 1] += x.y;
                            acc[i][j][4 * q + 2] += x.z;
                            acc[i][j][4 * q + 3] += x.w;
                        }
                    }
        }
        // the reads are done before the next partials' DMA overwrites them
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if (lane == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// The workgroup barrier without a fence: no wave writes global memory in the
// K loop, and a fence would make the compiler wait for every load in flight;
// the LDS waits a barrier needs are explicit before it.
__device__ inline void bare_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// s_waitcnt lgkmcnt(0) alone: this wave's LDS stores done, loads left in flight
// (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
__device__ inline void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xC07F); }

// The producer's part of one tile over K-steps [k0, k0 + ns), with steps 0
// and 1 already requested into r0 and r1: step j's W units are loaded during
// step j-4 and stored into stage j%3 during step j-2 (the consumers read step
// j+1's first fragments before the barrier that ends step j, so a stage must
// be complete a step before it is consumed, and it is free only after the
// step that last read it). Every load goes into registers and every LDS store
// is the compiler's own, so the compiler counts the loads in flight and waits
// for exactly those whose registers a store reads; before a barrier only the
// LDS stores are waited for. Steps 2-3 are requested whether or not this tile
// has them (a step past this split's steps reads the next split's slab; one
// past the operand's last step, `last` steps after w0, reads that last step
// again; neither is stored), so the steady state starts with an exact count;
// it runs without conditions, and the last steps do their remaining stores
// one by one. With `next` (ns even), the two requests that follow the tile's
// last step fetch steps 0 and 1 of the workgroup's next tile (producer pn, at
// wn0) into r0 and r1 instead. The barriers match the consumers', step for
// step.
template <class C, int U = 2>
__device__ inline void produce_tile(const producer<C, U> & pr, uint8_t * smem, int w0, int w_kstride, int ns,
                                    int last, stage_regs<C, U> & r0, stage_regs<C, U> & r1, const producer<C, U> & pn,
                                    int wn0, int wn_kstride, bool next) {
    pr.store_w(r0, smem, 0);
    pr.load_w(r0, w0 + min(2, last) * w_kstride);
    if (ns > 1) pr.store_w(r1, smem, C::STAGE);
    pr.load_w(r1, w0 + min(3, last) * w_kstride);
    wait_lgkm0();
    bare_barrier();
    // during step k: step k+2 stored into stage (k+2)%3, step k+4 requested
    int stage = 2 * C::STAGE, k = 0;
    for (; k + 5 < ns; k += 2) {
        pr.store_w(r0, smem, stage);
        pr.load_w(r0, w0 + (k + 4) * w_kstride);
        stage = stage == 2 * C::STAGE ? 0 : stage + C::STAGE;
        wait_lgkm0();
        bare_barrier();
        pr.store_w(r1, smem, stage);
        pr.load_w(r1, w0 + (k + 5) * w_kstride);
        stage = stage == 2 * C::STAGE ? 0 : stage + C::STAGE;
        wait_lgkm0();
        bare_barrier();
    }
    for (; k < ns; k += 2) {
        if (k + 2 < ns) {
            pr.store_w(r0, smem, stage);
            if (k + 4 < ns)
                pr.load_w(r0, w0 + (k + 4) * w_kstride);
            else if (next && k + 4 == ns)
                pn.load_w(r0, wn0);
        }
        stage = stage == 2 * C::STAGE ? 0 : stage + C::STAGE;
        wait_lgkm0();
        bare_barrier();
        if (k + 1 < ns) {
            if (k + 3 < ns) {
                pr.store_w(r1, smem, stage);
                if (k + 5 < ns)
                    pr.load_w(r1, w0 + (k + 5) * w_kstride);
                else if (next && k + 5 == ns + 1)
                    pn.load_w(r1, wn0 + wn_kstride);
            }
            stage = stage == 2 * C::STAGE ? 0 : stage + C::STAGE;
            wait_lgkm0();
            bare_barrier();
        }
    }
}

// The producer's part of a workgroup's only tile.
template <class C, int U>
__device__ inline void produce(const producer<C, U> & pr, uint8_t * smem, int w0, int w_kstride, int ns, int last) {
    stage_regs<C, U> r0, r1;
    pr.load_w(r0, w0);
    pr.load_w(r1, w0 + min(1, last) * w_kstride);
    produce_tile<C, U>(pr, smem, w0, w_kstride, ns, last, r0, r1, pr, 0, 0, false);
}

// The consumer's K loop over a tile's steps [0, ns), its A fragments of
// steps 0 and 1 requested into a0s and a1s: starts with the barrier that
// completes the first two W stages. Past the tile's last step, a load of
// step j reads step min(j, last) (the next split's slab or the operand's
// last step again, never used). Pairs of steps run without conditions.
template <class C>
__device__ inline void consume_tile(f32x16 (&acc)[C::TI][C::TJ], bf16x8 (&a0s)[4][C::TI], bf16x8 (&a1s)[4][C::TI],
                                    const uint8_t * smem, const int (&fw)[4], const a_loader<C> & al, int a0, int ks,
                                    int ns, int last) {
    bf16x8 bw[2][C::TJ];
    bare_barrier();
#pragma unroll
    for (int j = 0; j < C::TJ; j++) bw[0][j] = lds_get(smem, fw[0] + j * 32 * C::ROWB);
    int cur = 0, k = 0;
    for (; k + 1 < ns; k += 2) {
        int nxt = cur == 2 * C::STAGE ? 0 : cur + C::STAGE;
        consume<C, true>(acc, a0s, bw, smem, fw, cur, nxt, al, a0 + min(k + 2, last) * ks);
        cur = nxt;
        bare_barrier();
        nxt = cur == 2 * C::STAGE ? 0 : cur + C::STAGE;
        consume<C, true>(acc, a1s, bw, smem, fw, cur, nxt, al, a0 + min(k + 3, last) * ks);
        cur = nxt;
        bare_barrier();
    }
    if (k < ns) {
        const int nxt = cur == 2 * C::STAGE ? 0 : cur + C::STAGE;
        consume<C, false>(acc, a0s, bw, smem, fw, cur, nxt, al, 0);
        bare_barrier();
    }
}

// The consumer's epilogue of one tile; APART as for store_glu (the plain
// store uses no LDS).
template <class C, int EPI, bool APART = false>
__device__ inline void epilogue(const f32x16 (&acc)[C::TI][C::TJ], const gemm_params & p, uint8_t * smem,
                                const gemm_weight & W, int64_t m0, int64_t n0, int wave, int wm, int wn, int lane) {
    if constexpr (EPI == EPI_RESIDUAL)
        store_tile<C, true>(acc, W.c, p.M, W.n, W.ldc, m0, n0, wm, wn, lane, p.nonfinite, p.res, p.ldr, smem, wave);
    else if constexpr (EPI < 0)
        store_tile<C>(acc, W.c, p.M, W.n, W.ldc, m0, n0, wm, wn, lane, p.nonfinite);
    else
        store_glu<C, EPI, APART>(acc, smem, p.xout, p.h, p.ldh, p.M, W.n / 2, m0, n0, wave, wm, wn, lane,
                                 p.nonfinite);
}

// Tile t of a launch in the tile order: tiles go in groups of GROUP_M tile
// rows, M-fastest inside a group, so the ~32 workgroups resident on one XCD
// cover a compact block of about 4 x 8 tiles and share their A and W slabs in
// its L2. Returns the tile's weight (of a group launch) and its first row and
// column.
template <class C>
__device__ inline gemm_weight tile_of(const gemm_params & p, int t, int64_t & m0, int64_t & n0) {
    const int per_group = ZEST_GEMM_GROUP_M * p.nt, first_m = t / per_group * ZEST_GEMM_GROUP_M;
    const int gm = min(p.mt - first_m, ZEST_GEMM_GROUP_M), in = t % per_group;
    const int tm = first_m + in % gm, tn = in / gm;
    int g = 0;
#pragma unroll
    for (int i = 1; i < ZEST_GEMM_MAX_GROUP; i++)
        if (i < p.nw && tn >= p.wt[i].tile0) g = i;
    g = __builtin_amdgcn_readfirstlane(g);
    m0 = (int64_t) tm * C::BM;
    n0 = (int64_t) (tn - p.wt[g].tile0) * C::BN;
    return p.wt[g];
}

// Workgroups go to the 8 XCDs round-robin by linear id b; the n workgroups
// numbered by this map hold a contiguous run of it on each XCD.
__device__ inline int xcd_order(int b, int n) {
#if ZEST_GEMM_XCD
    return (b % 8) * (n / 8) + min(b % 8, n % 8) + b / 8;
#else
    return b;
#endif
}

// One output tile (rows m0.., columns n0.. of weight W), over K-steps
// [k0, k0 + ns); with SPLIT, unit `split` of tile t. With K-groups (C::KG >
// 1; ns a multiple of KG), group g runs steps [k0 + g*ns/KG, k0 +
// (g+1)*ns/KG) on its own ring, the groups meet the same barriers step for
// step, and after the K loop every wave meets one more: groups 1.. have left
// their sums in LDS, and group 0 adds them in group order (((s0 + s1) + s2)
// + ...) before the split-K fixup and the epilogue. A group's waves take
// their roles rotated by g * NC/64, so that with waves placed on SIMDs in
// turn each SIMD holds consumers and producers alike.
template <class C, int EPI, bool SPLIT>
__device__ inline void run_tile(const gemm_params & p, uint8_t * smem, const gemm_weight & W, int64_t m0, int64_t n0,
                                int k0, int ns, int t, int split) {
    int grp = 0, wave, tid;
    if constexpr (C::KG > 1) {
        grp = __builtin_amdgcn_readfirstlane((int) threadIdx.x / (C::NC + C::NP));
        const int wig = __builtin_amdgcn_readfirstlane(((int) threadIdx.x % (C::NC + C::NP)) >> 6);
        wave = (wig + grp * (C::NC / 64)) % C::NW;
        tid = wave * 64 + ((int) threadIdx.x & 63);
    } else {
        tid = threadIdx.x;
        wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    }
    const int lane = tid & 63;
    const int nk = p.nk;
    uint8_t * const base = smem;
    if constexpr (C::KG > 1) {
        smem += grp * C::RING;
        ns /= C::KG;
        k0 += grp * ns;
    }
    if (wave >= C::NC / 64) {
        const int job = tid - C::NC;
        // uniform, but the tile arithmetic can leave it in a vector register,
        // and a load's scalar offset taken from one costs a loop per load
        const int w0 =
            __builtin_amdgcn_readfirstlane((int) ((n0 / ZEST_TILE_ROWS) * ZEST_TILE_BYTES) + k0 * W.w_kstride);
        if constexpr (C::NP1 > 0)
            if (job >= C::NP2) {  // whole waves: NP2 % 64 == 0
                const producer<C, 1> pr(W.w, (int64_t) W.w_kstride * nk, job - C::NP2);
                produce<C, 1>(pr, smem, w0, W.w_kstride, ns, nk - 1 - k0);
                if constexpr (C::KG > 1) bare_barrier();  // the K-groups' sums
                return;
            }
        const producer<C, 2> pr(W.w, (int64_t) W.w_kstride * nk, job);
        produce<C, 2>(pr, smem, w0, W.w_kstride, ns, nk - 1 - k0);
        if constexpr (C::KG > 1) bare_barrier();  // the K-groups' sums
        return;
    }

    // Consumer: rows wm*WM.. and columns wn*WN.. of the tile. swz depends
    // only on the row mod 16, so a column block's W rows keep rows wr's.
    const int wm = wave % C::CWM, wn = wave / C::CWM, khalf = lane >> 5, wr = lane & 31;
    int fw[4];
#pragma unroll
    for (int s = 0; s < 4; s++) fw[s] = (wn * C::WN + wr) * C::ROWB + ((2 * s + khalf) ^ swz(wr)) * 16;
    f32x16 acc[C::TI][C::TJ];
#pragma unroll
    for (int i = 0; i < C::TI; i++)
#pragma unroll
        for (int j = 0; j < C::TJ; j++) acc[i][j] = f32x16{};
    {
        // A two steps ahead in registers; no fence at the barriers, so the
        // loads stay in flight across them (consumers write no memory here)
        const a_loader<C> al(p.a, (int64_t) p.a_kstride * nk, wm, lane);
        const int ks = p.a_kstride;
        const int a0 =
            __builtin_amdgcn_readfirstlane((int) ((m0 / ZEST_XGROUP_ROWS) * ZEST_XGROUP_BYTES) + k0 * p.a_kstride);
        // the operand's last K-step, counted from a0: the steps loaded past
        // it load it again (the scalar offset is not range-checked)
        const int last = nk - 1 - k0;
        bf16x8 a0s[4][C::TI], a1s[4][C::TI];
        al.load_step(a0s, a0);
        al.load_step(a1s, a0 + min(1, last) * ks);
        consume_tile<C>(acc, a0s, a1s, smem, fw, al, a0, ks, ns, last);
        // the loads of steps past the end are still in flight
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }
    smem = base;
    if constexpr (C::KG > 1) {
        // every group is past its K loop's last barrier, so no ring is read
        // or written any more except by a consumer's unused read ahead
        if (grp > 0) {
            uint8_t * sums = smem + (size_t) grp * C::BM * C::BN * 4 + wave * (C::WM * C::WN * 4);
#pragma unroll
            for (int i = 0; i < C::TI; i++)
#pragma unroll
                for (int j = 0; j < C::TJ; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        *reinterpret_cast<float4 *>(sums + ((i * C::TJ + j) * 4 + q) * 1024 + lane * 16) =
                            make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                                        acc[i][j][4 * q + 3]);
            wait_lgkm0();
            bare_barrier();
            return;
        }
        bare_barrier();
#pragma unroll
        for (int g = 1; g < C::KG; g++) {
            const uint8_t * sums = smem + (size_t) g * C::BM * C::BN * 4 + wave * (C::WM * C::WN * 4);
#pragma unroll
            for (int i = 0; i < C::TI; i++)
#pragma unroll
                for (int j = 0; j < C::TJ; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float4 x =
                            *reinterpret_cast<const float4 *>(sums + ((i * C::TJ + j) * 4 + q) * 1024 + lane * 16);
                        acc[i][j][4 * q] += x.x;
                        acc[i][j][4 * q + 1] += x.y;
                        acc[i][j][4 * q + 2] += x.z;
                        acc[i][j][4 * q + 3] += x.w;
                    }
        }
    }
    if (SPLIT && !fixup<C>(acc, p, smem, t, split, wave, lane)) return;
    epilogue<C, EPI>(acc, p, smem, W, m0, n0, wave, wm, wn, lane);
}

// EPI: EPI_PLAIN the fp32 store, EPI_RESIDUAL the fp32 store of acc + res,
// >= 0 the fused GLU of that kind.
// SPLIT: split-K (p.splits > 1), else one whole tile per workgroup.
template <class C, int EPI, bool SPLIT>
__global__ __launch_bounds__(C::NT, C::MINB) void gemm_kernel(const gemm_params p) {
    extern __shared__ uint4 smem_u4[];
    uint8_t * smem = reinterpret_cast<uint8_t *>(smem_u4);
    const int v = xcd_order((int) blockIdx.x, (int) gridDim.x), nk = p.nk;
    const int T = p.mt * p.nt;
    const int split = SPLIT ? v / T : 0, t = SPLIT ? v - split * T : v;
    const int k0 = SPLIT ? split * nk / p.splits : 0, ns = SPLIT ? (split + 1) * nk / p.splits - k0 : nk;
    int64_t m0, n0;
    const gemm_weight W = tile_of<C>(p, t, m0, n0);
    run_tile<C, EPI, SPLIT>(p, smem, W, m0, n0, k0, ns, t, split);
}

// The mixed launch: CB tiles (p.mt x p.nt of them) whose count is a whole
// number of rounds of the GPU plus a part of one; that part runs as tiles of
// half the rows (CS), twice as many workgroups of about half the time, so the
// last round ends sooner. On each XCD the whole tiles come first (the first
// workgroups it is given), then the halves.
template <class CB, class CS, int EPI>
__global__ __launch_bounds__(CB::NT, 1) void gemm_kernel_mixed(const gemm_params p) {
    static_assert(CB::NT == CS::NT && CS::BM * 2 == CB::BM && CS::BN == CB::BN && CB::KG == 1 && CS::KG == 1,
                  "halves of the big tiles");
    extern __shared__ uint4 smem_u4[];
    uint8_t * smem = reinterpret_cast<uint8_t *>(smem_u4);
    const int b = (int) blockIdx.x, per_xcd = p.nbig / 8, i = b / 8;
    int64_t m0, n0;
    if (i < per_xcd) {
        const int t = (b % 8) * per_xcd + i;
        const gemm_weight W = tile_of<CB>(p, t, m0, n0);
        run_tile<CB, EPI, false>(p, smem, W, m0, n0, 0, p.nk, t, 0);
    } else {
        const int nhalf = (int) gridDim.x - p.nbig;
        const int u = xcd_order(b - p.nbig, nhalf);  // b - nbig keeps b's XCD: nbig % 8 == 0
        const int t = p.nbig + u / 2;
        const gemm_weight W = tile_of<CB>(p, t, m0, n0);
        run_tile<CS, EPI, false>(p, smem, W, m0 + (u % 2) * CS::BM, n0, 0, p.nk, t, 0);
    }
}

// Persistent workgroups for a launch of more than one round of whole tiles
// (ns = nk, even, at least 4; not the residual epilogue). Workgroup b works on
// XCD b % 8 and takes the tiles of that XCD's run (the contiguous run
// xcd_order gives it) in turn: start + b/8, start + b/8 + G/8, ... for G
// workgroups, a multiple of 8. The producers' last two requests of a tile
// fetch the next tile's first two W steps, and once past the tile's last
// barrier they expand and store them into the first two stages while the
// consumers run the epilogue (which uses no LDS, or the GLU's staging above
// the ring; the only LDS read a consumer still has in flight there is its
// unused read ahead of a next stage). The consumers request the next tile's
// first two A steps after the epilogue (held through it they would not fit
// the registers).
template <class C, int EPI>
__global__ __launch_bounds__(C::NT, 1) void gemm_kernel_tiles(const gemm_params p) {
    static_assert(C::KG == 1, "one K-group");
    extern __shared__ uint4 smem_u4[];
    uint8_t * smem = reinterpret_cast<uint8_t *>(smem_u4);
    const int b = (int) blockIdx.x, g = (int) gridDim.x / 8, T = p.mt * p.nt, nk = p.nk;
    const int x = b % 8, end = (x + 1) * (T / 8) + min(x + 1, T % 8);
    int t = x * (T / 8) + min(x, T % 8) + b / 8;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int64_t m0, n0;
    gemm_weight W = tile_of<C>(p, t, m0, n0);
    if (wave >= C::NC / 64) {
        const int job = tid - C::NC;
        producer<C> pr(W.w, (int64_t) W.w_kstride * nk, job);
        int w0 = __builtin_amdgcn_readfirstlane((int) ((n0 / ZEST_TILE_ROWS) * ZEST_TILE_BYTES));
        stage_regs<C> r0, r1;
        pr.load_w(r0, w0);
        pr.load_w(r1, w0 + W.w_kstride);
        for (;;) {
            const int tn = t + g;
            const bool next = tn < end;
            int64_t mn = m0, nn = n0;
            const gemm_weight Wn = next ? tile_of<C>(p, tn, mn, nn) : W;
            const producer<C> pn(Wn.w, (int64_t) Wn.w_kstride * nk, job);
            const int wn0 = __builtin_amdgcn_readfirstlane((int) ((nn / ZEST_TILE_ROWS) * ZEST_TILE_BYTES));
            produce_tile<C>(pr, smem, w0, W.w_kstride, nk, nk - 1, r0, r1, pn, wn0, Wn.w_kstride, next);
            if (!next) return;
            t = tn;
            W = Wn;
            pr = pn;
            w0 = wn0;
        }
    }
    const int wm = wave % C::CWM, wn = wave / C::CWM, khalf = lane >> 5, wr = lane & 31;
    int fw[4];
#pragma unroll
    for (int s = 0; s < 4; s++) fw[s] = (wn * C::WN + wr) * C::ROWB + ((2 * s + khalf) ^ swz(wr)) * 16;
    const a_loader<C> al(p.a, (int64_t) p.a_kstride * nk, wm, lane);
    const int ks = p.a_kstride;
    int a0 = __builtin_amdgcn_readfirstlane((int) ((m0 / ZEST_XGROUP_ROWS) * ZEST_XGROUP_BYTES));
    bf16x8 a0s[4][C::TI], a1s[4][C::TI];
    al.load_step(a0s, a0);
    al.load_step(a1s, a0 + ks);
    for (;;) {
        f32x16 acc[C::TI][C::TJ];
#pragma unroll
        for (int i = 0; i < C::TI; i++)
#pragma unroll
            for (int j = 0; j < C::TJ; j++) acc[i][j] = f32x16{};
        consume_tile<C>(acc, a0s, a1s, smem, fw, al, a0, ks, nk, nk - 1);
        // the loads of steps past the end are still in flight
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        epilogue<C, EPI, true>(acc, p, smem, W, m0, n0, wave, wm, wn, lane);
        t += g;
        if (t >= end) return;
        W = tile_of<C>(p, t, m0, n0);
        a0 = __builtin_amdgcn_readfirstlane((int) ((m0 / ZEST_XGROUP_ROWS) * ZEST_XGROUP_BYTES));
        al.load_step(a0s, a0);
        al.load_step(a1s, a0 + ks);
    }
}

// One item of a persistent mixed launch, a consumer wave's part: the K loop
// of a tile (its A fragments of steps 0 and 1 requested into a0s and a1s),
// then its epilogue (with no LDS of its own).
template <class C, int EPI>
__device__ inline void consume_item(const gemm_params & p, uint8_t * smem, const gemm_weight & W, int64_t m0,
                                    int64_t n0, int wave, int lane, bf16x8 (&a0s)[4][C::TI],
                                    bf16x8 (&a1s)[4][C::TI]) {
    const int wm = wave % C::CWM, wn = wave / C::CWM, khalf = lane >> 5, wr = lane & 31;
    int fw[4];
#pragma unroll
    for (int s = 0; s < 4; s++) fw[s] = (wn * C::WN + wr) * C::ROWB + ((2 * s + khalf) ^ swz(wr)) * 16;
    const a_loader<C> al(p.a, (int64_t) p.a_kstride * p.nk, wm, lane);
    const int a0 = __builtin_amdgcn_readfirstlane((int) ((m0 / ZEST_XGROUP_ROWS) * ZEST_XGROUP_BYTES));
    f32x16 acc[C::TI][C::TJ];
#pragma unroll
    for (int i = 0; i < C::TI; i++)
#pragma unroll
        for (int j = 0; j < C::TJ; j++) acc[i][j] = f32x16{};
    consume_tile<C>(acc, a0s, a1s, smem, fw, al, a0, p.a_kstride, p.nk, p.nk - 1);
    // the loads of steps past the end are still in flight
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    static_assert(EPI < 0 && EPI != EPI_RESIDUAL, "the plain store");
    epilogue<C, EPI>(acc, p, smem, W, m0, n0, wave, wm, wn, lane);
}

// A consumer wave's requests of a tile's first two A steps.
template <class C>
__device__ inline void load_item_a(const gemm_params & p, int64_t m0, int wave, int lane, bf16x8 (&a0s)[4][C::TI],
                                   bf16x8 (&a1s)[4][C::TI]) {
    const a_loader<C> al(p.a, (int64_t) p.a_kstride * p.nk, wave % C::CWM, lane);
    const int a0 = __builtin_amdgcn_readfirstlane((int) ((m0 / ZEST_XGROUP_ROWS) * ZEST_XGROUP_BYTES));
    al.load_step(a0s, a0);
    al.load_step(a1s, a0 + p.a_kstride);
}

// The mixed launch as persistent workgroups (nk even, at least 4), one a CU:
// workgroup b takes the whole tiles of XCD b % 8's run (the first nbig/8 of
// its tiles, as gemm_kernel_mixed's first nbig workgroups have them), then
// the half tiles of that XCD's run of halves, from b/8 in steps of G/8 (G
// workgroups, a multiple of 8, at most nbig). The producers request the next
// item's first two W steps during the current item's last ones (a half tile
// has its whole tile's W rows and the same producer layout) and store them
// into the first two stages while the consumers run the epilogue (the plain
// store, no LDS); the consumers request its first two A steps after it.
template <class CB, class CS, int EPI>
__global__ __launch_bounds__(CB::NT, 1) void gemm_kernel_mixed_tiles(const gemm_params p) {
    static_assert(CB::NT == CS::NT && CS::BM * 2 == CB::BM && CS::BN == CB::BN && CS::NP == CB::NP &&
                      CS::TI == CB::TI && CB::NP1 == 0 && CS::NP1 == 0 && CB::KG == 1 && CS::KG == 1,
                  "halves of the big tiles, with the same producers");
    extern __shared__ uint4 smem_u4[];
    uint8_t * smem = reinterpret_cast<uint8_t *>(smem_u4);
    const int b = (int) blockIdx.x, g = (int) gridDim.x / 8, x = b % 8, j = b / 8, nk = p.nk;
    const int T = p.mt * p.nt, per_xcd = p.nbig / 8, nhalf = 2 * (T - p.nbig);
    const int hs = x * (nhalf / 8) + min(x, nhalf % 8), he = (x + 1) * (nhalf / 8) + min(x + 1, nhalf % 8);
    const int n_whole = (per_xcd - j + g - 1) / g;
    const int n_items = n_whole + (hs + j < he ? (he - hs - j + g - 1) / g : 0);
    // item i: its tile, and the first row of its rows (a half's)
    auto item = [&](int i, int64_t & m0, int64_t & n0) {
        if (i < n_whole) return tile_of<CB>(p, x * per_xcd + j + i * g, m0, n0);
        const int u = hs + j + (i - n_whole) * g;
        const gemm_weight w = tile_of<CB>(p, p.nbig + u / 2, m0, n0);
        m0 += (u % 2) * CS::BM;
        return w;
    };
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int64_t m0, n0;
    gemm_weight W = item(0, m0, n0);
    if (wave >= CB::NC / 64) {
        const int job = tid - CB::NC;
        producer<CB> pr(W.w, (int64_t) W.w_kstride * nk, job);
        int w0 = __builtin_amdgcn_readfirstlane((int) ((n0 / ZEST_TILE_ROWS) * ZEST_TILE_BYTES));
        stage_regs<CB> r0, r1;
        pr.load_w(r0, w0);
        pr.load_w(r1, w0 + W.w_kstride);
        for (int i = 0;; i++) {
            const bool next = i + 1 < n_items;
            int64_t mn = m0, nn = n0;
            const gemm_weight Wn = next ? item(i + 1, mn, nn) : W;
            const producer<CB> pn(Wn.w, (int64_t) Wn.w_kstride * nk, job);
            const int wn0 = __builtin_amdgcn_readfirstlane((int) ((nn / ZEST_TILE_ROWS) * ZEST_TILE_BYTES));
            produce_tile<CB>(pr, smem, w0, W.w_kstride, nk, nk - 1, r0, r1, pn, wn0, Wn.w_kstride, next);
            if (!next) return;
            W = Wn;
            pr = pn;
            w0 = wn0;
        }
    }
    bf16x8 a0s[4][CB::TI], a1s[4][CB::TI];
    load_item_a<CB>(p, m0, wave, lane, a0s, a1s);
    for (int i = 0;; i++) {
        if (i < n_whole)
            consume_item<CB, EPI>(p, smem, W, m0, n0, wave, lane, a0s, a1s);
        else
            consume_item<CS, EPI>(p, smem, W, m0, n0, wave, lane, a0s, a1s);
        if (i + 1 >= n_items) return;
        W = item(i + 1, m0, n0);
        if (i + 1 < n_whole)
            load_item_a<CB>(p, m0, wave, lane, a0s, a1s);
        else
            load_item_a<CS>(p, m0, wave, lane, a0s, a1s);
    }
}

#ifndef ZEST_GEMM_PERSIST
#define ZEST_GEMM_PERSIST 1
#endif
#ifndef ZEST_GEMM_MAX_SPLIT
#define ZEST_GEMM_MAX_SPLIT 16
#endif
// The tile shapes. Which one a launch takes is the cost model's choice
// (plan_plain, launch_any).
//
// 256x128 tiles: 4 consumer waves of 64x128, or 8 of 32x128, two on each SIMD
// (the second hides latency that a CU with one tile in flight has nowhere else
// to hide, for twice the reads of W fragments from LDS).
using cfg_big = gemm_cfg<256, 128, 4>;
using cfg_glu = gemm_cfg<256, 128, 8, 256>;
// 128x160 tiles (4 consumer waves of 32x160) for weights of whole 160-row
// tiles (the tiles then read only rows each packed weight holds): where 256x128
// tiles leave CUs idle these may fill them (2048 x 2560 is 256 of them, one a CU, and
// 160 of the others). The producers are their critical path: four waves take
// two W units a thread (tiles 0-7) and two waves one (tiles 8-9), so the two
// SIMDs that hold a second producer wave carry one and a half waves'
// expansion, not two (five waves of two units: 52.5 -> 48.6 us).
using cfg_o = gemm_cfg<128, 160, 4, 384, 1, 1, 128>;
// The smaller tiles are bound by the chain of a producer's step (load, expand,
// store, wait, barrier), not by the matrix cores: at 16 workgroups on an idle
// GPU a K-step of a 128x128 tile took 0.38 us with producers of two units a
// thread, 0.36 of them the producers alone and 0.24 the consumers alone. So
// they have producers of one unit a thread, two waves on each SIMD whose
// steps overlap, and 8 consumers where 4 would leave a SIMD's other wave to
// wait for. 128x128 so: 0.36 us a step; the fastest for wide weights over up to
// 128 rows (98 x (8704 + 8704) x 2816 behind its norm 19.4 us, as 128x64 tiles
// 22.1; fused, 108 x 18432 x 3584, 26.7 and 30.4).
using cfg_small = gemm_cfg<128, 128, 4, 512, 1, 2, 512>;
// 128x64 tiles, two workgroups a CU (2048 x 1024 x 4096 31.6 -> 25.2 us, where
// 64x64 tiles were the best before), and as two K-groups, one workgroup a CU,
// for launches of up to one round of them: twice the loads in flight, and the
// groups' sums meet in LDS, not through a split-K fixup in memory (768 x 2560 x
// 4096 32.5 -> 22.4 us, 768 x 2560 x 2560 21.2 -> 15.0 us).
using cfg_mid = gemm_cfg<128, 64, 4, 256, 2, 1, 256>;
using cfg_mid2 = gemm_cfg<128, 64, 4, 256, 1, 1, 256, 2>;
// 64x64 tiles as two K-groups, for fewer rows or columns still: one workgroup
// a CU with producers of one unit a thread, or two with producers of two
// (48 x 2560 x 2560 10.3 us with the second alone, 8.9 with the first in
// two K splits; 48 x 19456 x 2560, 304 tiles, 20.9 with the first, 18.5 with the second).
using cfg_tiny2 = gemm_cfg<64, 64, 2, 256, 1, 1, 256, 2>;
using cfg_tiny2x2 = gemm_cfg<64, 64, 2, 128, 2, 1, 0, 2>;
// 64x64 tiles of one K-group: four waves of 96 registers and a 24 KB ring, so
// up to five workgroups a CU, for wide weights over few rows, where they are
// what keeps enough of W in flight (32 x (17408 + 17408) x 5120: 39.4 us, 5.1
// TB/s, against 44.5 as K-groups; 32 x 5945 x 6688 16.2 in five K splits against
// 20.7; 32 x 41572 x 1024 12.2 against 16.1), and for short K over many tiles (1833 x
// 2304 x 384 with the residual 11.0 against 12.3).
using cfg_tiny = gemm_cfg<64, 64, 2, 128, 5>;
// Mixed launches run their whole tiles as cfg_glu's (two consumers per SIMD)
// and the halves as 128x128 tiles of 8 consumer waves of 32x64 (4 row blocks
// x 2 column blocks) and 4 producers, the same threads (the q/k/v group at
// 2048 tokens: 66.8 -> 65.6 us against one consumer per SIMD in both).
using cfg_half8 = gemm_cfg<128, 128, 4, 256, 1, 2>;

// Per device and stream: the split-K workspace (grown as needed; counters
// zeroed when allocated, and zero again after every launch). Buffers that a
// captured graph names are not freed when they are outgrown, as the graph may
// be replayed: `held` keeps them until zest_release_stream.
struct sk_space {
    float * partial = nullptr;
    size_t partial_bytes = 0;
    uint32_t * counters = nullptr;
    size_t n_counters = 0;
    bool captured = false;
    std::vector<void *> held;
};

// Clears n counters (a kernel, not a memset, so a captured graph replays it).
__global__ void clear_counters(uint32_t * c, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) c[i] = 0;
}

// The device address of `scratch` on device `dev`, looked up once per device
// with that device current.
int scratch_address(int dev, uint8_t ** out) {
    static std::mutex mu;
    static uint8_t * addr[ZEST_MAX_DEVICES];  // no heap: the no-alloc entry point comes here on every call
    if (dev < 0 || dev >= ZEST_MAX_DEVICES) return zest::fail(ZEST_E_ARG, "device %d: at most %d", dev, ZEST_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void * p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return zest::fail(ZEST_E_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
        addr[dev] = (uint8_t *) p;
    }
    *out = addr[dev];
    return ZEST_OK;
}

int cu_count(int dev) {
    static std::mutex mu;
    static int cus[ZEST_MAX_DEVICES];
    if (dev < 0 || dev >= ZEST_MAX_DEVICES) return 256;
    std::lock_guard<std::mutex> lock(mu);
    if (cus[dev] > 0) return cus[dev];
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev] = n;
    return n;
}

// The split-K workspaces, by device and stream (until zest_release_stream).
// A stream as the workspaces are kept by: hipStreamPerThread is one handle for
// a stream of each thread, so there the thread is part of it.
using sk_stream = std::pair<hipStream_t, std::thread::id>;

sk_stream sk_stream_of(hipStream_t s) {
    return {s, s == hipStreamPerThread ? std::this_thread::get_id() : std::thread::id()};
}

std::mutex g_sk_mu;
std::map<std::pair<int, sk_stream>, sk_space> g_sk_spaces;

// A split-K workspace of at least these sizes, in `out`. The caller holds
// g_sk_mu until its launch is queued: until then another thread's launch on
// the stream could outgrow the workspace and free it, as its wait for the
// stream would not cover this launch. Nothing can be
// allocated while the stream is being captured: there `out.partial` is null
// where the stream's workspace is too small (the launch then runs unsplit).
int sk_reserve(hipStream_t s, size_t partial_bytes, size_t n_counters, sk_space & out, const char * name) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return zest::fail(ZEST_E_HIP, "%s: hipGetDevice failed", name);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (s && hipStreamIsCapturing(s, &capture) != hipSuccess)
        return zest::fail(ZEST_E_HIP, "%s: hipStreamIsCapturing failed", name);
    sk_space & sp = g_sk_spaces[{dev, sk_stream_of(s)}];
    const bool fits = sp.partial_bytes >= partial_bytes && sp.n_counters >= n_counters;
    out.partial = nullptr;
    if (capture != hipStreamCaptureStatusNone) {
        if (!fits) return ZEST_OK;
        sp.captured = true;
    }
    // a launch still running on the stream may use the buffers being replaced
    if (!fits && (sp.partial || sp.counters) && hipStreamSynchronize(s) != hipSuccess)
        return zest::fail(ZEST_E_HIP, "%s: stream synchronize", name);
    if (!fits && sp.captured) {
        for (void * b : {(void *) sp.partial, (void *) sp.counters})
            if (b) sp.held.push_back(b);
        // both anew, and at least twice the size, so few are ever held
        partial_bytes = std::max(partial_bytes, 2 * sp.partial_bytes);
        n_counters = std::max(n_counters, 2 * sp.n_counters);
        sp.partial = nullptr;
        sp.counters = nullptr;
        sp.partial_bytes = sp.n_counters = 0;
        sp.captured = false;
    }
    if (sp.partial_bytes < partial_bytes) {
        if (sp.partial) (void) hipFree(sp.partial);
        sp.partial = nullptr;
        sp.partial_bytes = 0;
        if (hipMalloc(&sp.partial, partial_bytes) != hipSuccess)
            return zest::fail(ZEST_E_HIP, "%s: split-K workspace of %zu bytes", name, partial_bytes);
        sp.partial_bytes = partial_bytes;
    }
    if (sp.n_counters < n_counters) {
        if (sp.counters) (void) hipFree(sp.counters);
        sp.counters = nullptr;
        sp.n_counters = 0;
        const size_t n = std::max(n_counters, (size_t) 4096);
        if (hipMalloc(&sp.counters, n * 4) != hipSuccess || hipMemsetAsync(sp.counters, 0, n * 4, s) != hipSuccess)
            return zest::fail(ZEST_E_HIP, "%s: split-K counters", name);
        sp.n_counters = n;
    }
    out.partial = sp.partial;
    out.partial_bytes = sp.partial_bytes;
    out.counters = sp.counters;
    out.n_counters = sp.n_counters;
    return ZEST_OK;
}

template <class C, int EPI, bool SPLIT>
int set_lds(const char * name) {
    // threads that launch a kernel for the first time at once may both set
    // the attribute: the same value, harmless
    static std::atomic<bool> attr_set{false};
    if (!attr_set.load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_kernel<C, EPI, SPLIT>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int) (SPLIT ? C::LDS_SPLIT : C::LDS_BYTES));
        if (e != hipSuccess) return zest::fail(ZEST_E_HIP, "%s: LDS attribute: %s", name, hipGetErrorString(e));
        attr_set.store(true, std::memory_order_release);
    }
    return ZEST_OK;
}

template <class C, int EPI>
int set_lds_tiles(const char * name) {
    static std::atomic<bool> attr_set{false};
    if (!attr_set.load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_kernel_tiles<C, EPI>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int) C::LDS_TILES);
        if (e != hipSuccess) return zest::fail(ZEST_E_HIP, "%s: LDS attribute: %s", name, hipGetErrorString(e));
        attr_set.store(true, std::memory_order_release);
    }
    return ZEST_OK;
}

template <class CB, class CS, int EPI>
int set_lds_mixed_tiles(const char * name) {
    static std::atomic<bool> attr_set{false};
    if (!attr_set.load(std::memory_order_acquire)) {
        const size_t bytes = std::max(CB::LDS_BYTES, CS::LDS_BYTES);
        const hipError_t e =
            hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_kernel_mixed_tiles<CB, CS, EPI>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int) bytes);
        if (e != hipSuccess) return zest::fail(ZEST_E_HIP, "%s: LDS attribute: %s", name, hipGetErrorString(e));
        attr_set.store(true, std::memory_order_release);
    }
    return ZEST_OK;
}

template <class CB, class CS, int EPI>
int set_lds_mixed(const char * name) {
    static std::atomic<bool> attr_set{false};
    if (!attr_set.load(std::memory_order_acquire)) {
        const size_t bytes = std::max(CB::LDS_BYTES, CS::LDS_BYTES);
        const hipError_t e =
            hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_kernel_mixed<CB, CS, EPI>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int) bytes);
        if (e != hipSuccess) return zest::fail(ZEST_E_HIP, "%s: LDS attribute: %s", name, hipGetErrorString(e));
        attr_set.store(true, std::memory_order_release);
    }
    return ZEST_OK;
}

// Launches one GEMM (a group of weights, or the fused GLU) as tiles of C in
// `splits` K splits, whose partial sums go through the workspace `sp`.
template <class C, int EPI>
int launch(gemm_params p, const int64_t * N, int splits, const sk_space & sp, hipStream_t s, const char * name) {
    p.mt = (int) ((p.M + C::BM - 1) / C::BM);
    int nt = 0;
    for (int i = 0; i < p.nw; i++) {
        p.wt[i].tile0 = nt;
        nt += (int) ((N[i] + C::BN - 1) / C::BN);
    }
    p.nt = nt;
    const int64_t T = (int64_t) p.mt * nt;
    p.splits = splits;
    if (C::KG > 1 && p.nk % (splits * C::KG))
        return zest::fail(ZEST_E_ARG, "%s: %d K-steps do not make %d splits of %d K-groups", name, p.nk, splits,
                          C::KG);
    const int64_t grid = T * p.splits;
    if (grid >= (1ll << 31) || (p.splits > 1 && grid * C::BM * C::BN * 4 >= (1ll << 31)))
        return zest::fail(ZEST_E_ARG, "%s: %lld tiles is too many", name, (long long) T);
    p.partial = sp.partial;
    p.counters = sp.counters;
#if ZEST_GEMM_PERSIST
    // more than one round: persistent workgroups, one a CU (not for the
    // residual epilogue, whose persistent form does not fit the registers)
    if constexpr (EPI != EPI_RESIDUAL && C::MINB == 1 && C::NP1 == 0 && C::KG == 1)
        if (p.splits == 1 && p.nk % 2 == 0 && p.nk >= 4) {
            int dev = 0;
            (void) hipGetDevice(&dev);
            const int64_t G = cu_count(dev) / 8 * 8;
            if (G >= 8 && T > G) {
                const int st = set_lds_tiles<C, EPI>(name);
                if (st != ZEST_OK) return st;
                hipLaunchKernelGGL((gemm_kernel_tiles<C, EPI>), dim3((unsigned) G), dim3(C::NT), C::LDS_TILES, s, p);
                return zest::check_launch(name);
            }
        }
#endif
    const int st = p.splits > 1 ? set_lds<C, EPI, true>(name) : set_lds<C, EPI, false>(name);
    if (st != ZEST_OK) return st;
    if (p.splits > 1)
        hipLaunchKernelGGL((gemm_kernel<C, EPI, true>), dim3((unsigned) grid), dim3(C::NT), C::LDS_SPLIT, s, p);
    else
        hipLaunchKernelGGL((gemm_kernel<C, EPI, false>), dim3((unsigned) grid), dim3(C::NT), C::LDS_BYTES, s, p);
    return zest::check_launch(name);
}

// A mixed launch: the first nbig big tiles whole, the rest as halves.
template <class CB, class CS, int EPI>
int launch_mixed(gemm_params p, const int64_t * N, int64_t nbig, hipStream_t s, const char * name) {
    p.mt = (int) ((p.M + CB::BM - 1) / CB::BM);
    int nt = 0;
    for (int i = 0; i < p.nw; i++) {
        p.wt[i].tile0 = nt;
        nt += (int) ((N[i] + CB::BN - 1) / CB::BN);
    }
    p.nt = nt;
    const int64_t T = (int64_t) p.mt * nt, grid = nbig + 2 * (T - nbig);
    if (grid >= (1ll << 31) || nbig % 8 || nbig >= T)
        return zest::fail(ZEST_E_ARG, "%s: mixed launch of %lld tiles", name, (long long) T);
    p.splits = 1;
    p.nbig = (int) nbig;
#if ZEST_GEMM_PERSIST
    // persistent workgroups, one a CU (not for the residual epilogue, whose
    // persistent form does not fit the registers)
    if constexpr (EPI != EPI_RESIDUAL)
        if (p.nk % 2 == 0 && p.nk >= 4) {
            int dev = 0;
            (void) hipGetDevice(&dev);
            const int64_t G = std::min<int64_t>(nbig, cu_count(dev) / 8 * 8);
            if (G >= 8) {
                const int st = set_lds_mixed_tiles<CB, CS, EPI>(name);
                if (st != ZEST_OK) return st;
                hipLaunchKernelGGL((gemm_kernel_mixed_tiles<CB, CS, EPI>), dim3((unsigned) G), dim3(CB::NT),
                                   std::max(CB::LDS_BYTES, CS::LDS_BYTES), s, p);
                return zest::check_launch(name);
            }
        }
#endif
    const int st = set_lds_mixed<CB, CS, EPI>(name);
    if (st != ZEST_OK) return st;
    hipLaunchKernelGGL((gemm_kernel_mixed<CB, CS, EPI>), dim3((unsigned) grid), dim3(CB::NT),
                       std::max(CB::LDS_BYTES, CS::LDS_BYTES), s, p);
    return zest::check_launch(name);
}

enum shape_kind {
    SHAPE_BIG, SHAPE_GLU, SHAPE_O, SHAPE_SMALL, SHAPE_MID, SHAPE_MID2, SHAPE_TINY2, SHAPE_TINY2X2, SHAPE_TINY, SHAPES,
    SHAPE_MIXED
};

struct tile_shape {
    int bm, bn, kg, per_cu, waves;  // waves: consumer waves, a counter each in a split launch
};

template <class C>
constexpr tile_shape shape_of() {
    return {C::BM, C::BN, C::KG, C::MINB, C::NC / 64};
}

constexpr tile_shape TILES[SHAPES] = {
    shape_of<cfg_big>(), shape_of<cfg_glu>(),   shape_of<cfg_o>(),       shape_of<cfg_small>(), shape_of<cfg_mid>(),
    shape_of<cfg_mid2>(), shape_of<cfg_tiny2>(), shape_of<cfg_tiny2x2>(), shape_of<cfg_tiny>(),
};

// The launch cost model, in microseconds. U = T * S units (T tiles in S K
// splits) on P CUs. A unit runs its K-steps (nk / (S * kg)) and `prologue` more
// (the pipeline's fill and the epilogue); a step takes `step` in a workgroup
// that has a nearly idle GPU for itself, and busy() times that in all the rounds
// of a launch: the clock falls under the power limit and the L2s fill up with
// the share of CUs at work, and workgroups that share a CU slow each other. A
// split launch pays for its partial sums: each unit writes its tile and the
// last ones read them back, 2 * U * BM*BN*4 bytes at 8 TB/s over `partial`, and
// `split` a split for their round trips. Where the weights and the output
// outgrow the 256 MB last-level cache, a launch takes up to 1 + `cold` times as
// long (from 200 to 400 MB). Each kind of launch has rates of its own: the
// epilogues cost differently, and a group's activations come from a norm where
// one weight's come from the packer, which stores past the caches. The mixed
// launch has too: its half tiles have another layout of waves than the 128x128
// tiles alone.
//
// The numbers are fits to 17000 launches timed plan after plan, each behind
// the kernel that makes its activations (a norm, a GLU or the packer), as the
// first reads of an operand that no L2 holds yet are a good part of a short
// launch: least squares, then a descent on the choice itself, after which two
// rates were moved by hand to where the choice lost least (128x128 tiles of one
// weight up by 5%, 256x128 tiles of 4 waves in a group down by 7%) and the rates
// of one weight's 256x128 tiles of 4 waves searched by themselves, the others
// held (4096x8192x5120 takes them: 262.6 us, 267.7 as 8 waves). The launches
// span single weights of any width, q/k/v and gate/up groups, heads of up to
// 151936 columns, residual and fused launches, 32 to 4096 rows, K 256 to 17408.
// Over them the choice takes 0.2 (fused) to 1.1% (one weight) longer than the
// fastest plan measured, the worst hundredth 3 to 13%.
enum launch_class { CLASS_SINGLE, CLASS_RESIDUAL, CLASS_GROUP, CLASS_FUSED, CLASSES };

struct launch_rate {
    double fixed, prologue, step;
    double load[6];  // busy()
    double split, partial, cold;
};

// {}: a shape that the kind does not take
constexpr launch_rate RATES[CLASSES][SHAPES] = {
    {   // one weight
     {2.4286, 8.5589, 0.5328, {0.2485}, 2.3683, 0.6743, 0.0976},
     {2.0349, 6.6824, 0.5278, {0.2952}, 2.4903, 0.5995, 0.1122},
     {1.7754, 14.2972, 0.3707, {0.4091}, 2.1513, 0.169, 0.0222},
     {1.9307, 3.4291, 0.4488, {0.1525}, 1.3371, 1.0892, 0.1335},
     {0, 3.0762, 0.3477, {0.1863, 1.4931, 1.3741}, 1.1467, 1.0997, 0.3409},
     {0.4572, 2.3648, 0.4867, {0.0891}, 1.1198, 1.8362, 0.2082},
     {1.3166, 1.1414, 0.349, {0.158}, 0.8535, 1.2643, 0.4217},
     {0.899, 2.84, 0.4333, {0.2195, 1.5544, 1.5184}, 0.7542, 0.6682, 0.4942},
     {0, 4.5243, 0.3027, {0.1582, 1.3153, 1.6153, 2.1583, 0.5474, 0.1096}, 0.8015, 0.7724, 0.6799},
    },
    {   // one weight, residual
     {4.6875, 13.8007, 0.4665, {0.659}, 0.861, 0.4655, 0},
     {4.7149, 9.1415, 0.461, {0.7206}, 0.7762, 0.4472, 0.0057},
     {1.6817, 15.8825, 0.3601, {0.4075}, 1.8692, 0.1466, 0.032},
     {2.5852, 13.9579, 0.3095, {0.5498}, 1.1535, 0.2057, 0.0697},
     {0.9722, 9.8312, 0.2547, {0.4533, 1.707, 1.9024}, 0.8829, 0.3954, 0.2392},
     {1.5205, 7.0075, 0.3579, {0.3598}, 0.7499, 1.7591, 0.0743},
     {2.0204, 4.8614, 0.2738, {0.2693}, 0.5265, 1.3108, 0.1},
     {1.6391, 4.7094, 0.3661, {0.3302, 1.6946, 1.6861}, 0.5636, 0.7032, 1.0184},
     {1.8307, 6.2391, 0.2095, {0.3796, 1.8189, 2.1157, 2.7646, 0.7054, 0.1742}, 0.5884, 0.4164, 0.6617},
    },
    {   // a group
     {4.632, 7.3286, 0.4373, {0.4991}, 3.0005, 0.1132, 0.0692},
     {3.4579, 7.0427, 0.4462, {0.5159}, 1.8586, 0.3202, 0.048},
     {2.0923, 7.5832, 0.3804, {0.3522}, 2.1902, 0.4381, 0.0116},
     {2.0139, 6.3952, 0.3075, {0.4969}, 1.7265, 0.4282, 0.058},
     {1.6618, 4.9488, 0.259, {0.2956, 1.6625, 1.841}, 1.0306, 0.8483, 0.0275},
     {1.964, 3.1205, 0.4234, {0.2743}, 0.8497, 0.9997, 0},
     {2.992, 1.814, 0.2916, {0.3084}, 0.8149, 0.0729, 0},
     {3.0795, 1.6498, 0.3942, {0.123, 1.6706, 1.6649}, 0.5748, 1.4268, 0},
     {1.9724, 3.8809, 0.2715, {0.1591, 1.4708, 1.6243, 2.234, 0.6013, 0.222}, 0.8035, 0.601, 0},
    },
    {   // fused GLU
     {},
     {2.1605, 8.4353, 0.4916, {0.3945}, 0.5585, 0.6701, 0.0555},
     {},
     {0.8151, 7.7693, 0.3619, {0.2423}, 1.8657, 0.4195, 0.0294},
     {2.1204, 4.8003, 0.2559, {0.1894, 1.8192, 1.8119}, 0, 1.5729, 0.0718},
     {1.9759, 3.2529, 0.4401, {0.1593}, 0.3617, 1.9569, 0},
     {2.266, 1.902, 0.3876, {0}, 0.805, 1.1022, 0},
     {1.326, 3.7091, 0.4531, {0.1083, 1.6447, 1.3917}, 0.2779, 2.9564, 0},
     {1.8356, 5.4968, 0.2744, {0.0615, 1.5575, 1.8098, 2.356, 0.5662, 0.1817}, 0, 1.6553, 0},
    },
};

// `whole`: a step in a whole round of 256x128 tiles; `half`, `half_prologue`
// and `half_load` as step, prologue and load[0] for the half tiles
struct mixed_rate {
    double fixed, prologue, whole, half, half_prologue, half_load, cold;
};

constexpr mixed_rate MIXED_RATES[CLASS_FUSED] = {
    {0, 13.1187, 0.5858, 0.5442, 0, 0.2438, 0.1086},
    {0, 14.8117, 0.7393, 0.3424, 18.3353, 0.6001, 0},
    {4.063, 6.9994, 0.6551, 0.3497, 5.0218, 0.3923, 0.0503},
};

// A step's time over a lone workgroup's, summed over the rounds of `units`
// units on P CUs. One workgroup a CU: whole rounds and a last, partly filled
// one, a round rising to 1 + load[0] with the square of the share of CUs. Two:
// to 1 + load[0] with one on each CU, then, once any CU has two, on a line from
// load[1] to load[2]. Up to five: a staircase by the CU with the most, 1 +
// load[0], load[1], load[2], load[3], then load[4] times their number, its
// steps sloped by load[5].
double busy(int per_cu, const double * load, double units, double P) {
    const double q = units / P;
    if (per_cu == 1) {
        const double n = std::floor(q), f = q - n;
        return n * (1 + load[0]) + (f > 0 ? 1 + load[0] * f * f : 0.0);
    }
    if (per_cu == 2) {
        const double n = std::floor(q / 2), f = q / 2 - n;
        if (f == 0) return n * load[2];
        return n * load[2] + (f <= 0.5 ? 1 + load[0] * 4 * f * f : load[1] + (load[2] - load[1]) * (2 * f - 1));
    }
    const double c = std::ceil(q);
    if (c <= 1) return 1 + load[0] * q * q;
    return (c <= 4 ? load[(int) c - 1] : load[4] * c) + load[5] * (q - (c - 1));
}

// What a plan is made from: a launch's sizes on P CUs.
struct launch_sizes {
    int64_t M;
    int nk, nw;
    int64_t N[ZEST_GEMM_MAX_GROUP];
    int64_t P;

    // tiles of one shape
    int64_t tiles(int bm, int bn) const {
        int64_t nt = 0;
        for (int i = 0; i < nw; i++) nt += (N[i] + bn - 1) / bn;
        return (M + bm - 1) / bm * nt;
    }

    // 0 with everything in the last-level cache, 1 with nothing
    double cold(int cls) const {
        double n = 0, k = (double) nk * ZEST_TILE_K;
        for (int i = 0; i < nw; i++) n += (double) N[i];
        const double out = cls == CLASS_RESIDUAL ? 8.0 : cls == CLASS_FUSED ? 1.0 : 4.0;  // bytes a column
        const double mb = (n * k * 1.125 + (double) M * (n * out + k * 2)) / 1e6;
        return std::min(1.0, std::max(0.0, (mb - 200) / 200));
    }
};

launch_sizes sizes_of(const gemm_params & p, const int64_t * N, int64_t P) {
    launch_sizes z{p.M, p.nk, p.nw, {}, P};
    for (int i = 0; i < p.nw; i++) z.N[i] = N[i];
    return z;
}

// What splitting K costs: grows with S.
double split_us(int cls, int k, int64_t T, int S) {
    if (S == 1) return 0.0;
    const launch_rate & r = RATES[cls][k];
    return r.split * S + r.partial * 2.0 * (double) (T * S) * TILES[k].bm * TILES[k].bn * 4 / 8e6;
}

double plan_us(int cls, int k, int64_t T, int S, const launch_sizes & z, double cold) {
    const launch_rate & r = RATES[cls][k];
    const tile_shape & t = TILES[k];
    const double steps = (double) z.nk / (S * t.kg) + r.prologue;
    const double us = r.fixed + steps * r.step * busy(t.per_cu, r.load, (double) (T * S), (double) z.P);
    return (us + split_us(cls, k, T, S)) * (1 + r.cold * cold);
}

// A launch's plan: its tile shape, K splits and, for a mixed launch, how many
// of its 256x128 tiles run whole.
struct gemm_plan {
    int kind = SHAPE_BIG;
    int splits = 1;
    int64_t nbig = 0;
    double us = 1e300;

    const tile_shape & tile() const { return TILES[kind == SHAPE_MIXED ? (int) SHAPE_GLU : kind]; }
};

// The split-K workspace of T tiles of shape k in S splits.
size_t partial_bytes_of(int k, int64_t T, int S) { return (size_t) (T * S) * TILES[k].bm * TILES[k].bn * 4; }
size_t counters_of(int k, int64_t T) { return (size_t) T * TILES[k].waves; }

// 128x160 tiles need weights of whole 160-row tiles
bool whole_o_tiles(const launch_sizes & z) {
    bool whole = true;
    for (int i = 0; i < z.nw; i++) whole &= z.N[i] % cfg_o::BN == 0;
    return whole;
}

// The mixed launch's plan: whole rounds of 256x128 tiles, the part-round left
// as half tiles. Its us stays 1e300 where there is none.
gemm_plan plan_mixed(int cls, const launch_sizes & z) {
    const int64_t T = z.tiles(cfg_glu::BM, cfg_glu::BN), R = T / z.P, rem = T % z.P;
    gemm_plan plan;
    if (R < 1 || rem == 0 || R * z.P % 8 != 0) return plan;
    const mixed_rate & m = MIXED_RATES[cls];
    const double whole = (double) R * (z.nk + m.prologue) * m.whole;
    const double half = (z.nk + m.half_prologue) * m.half * busy(1, &m.half_load, 2.0 * rem, (double) z.P);
    return {SHAPE_MIXED, 1, R * z.P, (m.fixed + whole + half) * (1 + m.cold * z.cold(cls))};
}

// The cheapest plan of a plain launch by the cost model: a tile shape with its
// K splits, or a mixed launch. A launch whose whole tiles give every CU one (two
// of the one-group 64x64 tiles) is not split: the largest gain of it measured
// there is 1%. A split keeps at least three K-steps a K-group, and the partial
// sums fit the static workspace of zest_gemm_group_noalloc, which runs the same
// plan. Only for K over 32768 may 256x128 tiles outgrow it, where that saves a
// twentieth of the time (2048 x 2816 x 65536 in four splits): that entry point
// refuses those. Weights of whole 160-row tiles stay inside it at any K, as it
// has accepted them since they ran as one unsplit round of 128x160 tiles.
gemm_plan plan_plain(const launch_sizes & z, int max_splits) {
    const int cls = z.nw > 1 ? CLASS_GROUP : CLASS_SINGLE;
    gemm_plan best = plan_mixed(cls, z), outgrown;
    const bool whole = whole_o_tiles(z);
    const double cold = z.cold(cls);
    for (int k = 0; k < SHAPES; k++) {
        const tile_shape & t = TILES[k];
        const launch_rate & r = RATES[cls][k];
        if (r.step == 0 || (k == SHAPE_O && !whole)) continue;
        const int64_t T = z.tiles(t.bm, t.bn), most = z.P * (t.per_cu > 2 ? 2 : 1);
        for (int S = 1; S <= max_splits; S++) {
            if (S > 1 && (T >= most || T * S > 4 * z.P * std::min(t.per_cu, 2) || z.nk < 3 * S * t.kg)) break;
            const bool fits = S == 1 || (partial_bytes_of(k, T, S) <= ZEST_NOALLOC_PARTIAL_BYTES &&
                                         counters_of(k, T) <= ZEST_NOALLOC_COUNTERS);
            if (!fits && (z.nk <= 512 || t.bm < 256 || whole)) break;
            // no more splits can win (the rest of this one's time is at least that of its first steps)
            if (S > 1 && r.fixed + r.prologue * r.step + split_us(cls, k, T, S) >= best.us) break;
            if (t.kg > 1 && (z.nk % (S * t.kg) || z.nk < 2 * S * t.kg)) continue;
            const double us = plan_us(cls, k, T, S, z, cold);
            gemm_plan & plan = fits ? best : outgrown;
            if (us < plan.us) plan = {k, S, 0, us};
        }
    }
    return outgrown.us * 1.05 < best.us ? outgrown : best;
}

// The columns that a fused GLU's tiles cover: the output operand's K padding
// too, the columns of 2F rounded up to 128 rows of the gate/up pair, whose
// rows past 2F are zero blocks, so the h columns past F store the packer's
// zeros (with 64-column tiles and F % 64 == 32 the last tile would end at F).
int64_t glu_columns(int64_t N) { return (N + 127) / 128 * 128; }

// The plan of a launch with epilogue `epi`. A residual launch and a fused GLU
// launch split K as the plain launch of their columns would, in as many
// K-groups (so their sums are that launch's, bit for bit: a sum depends on the
// K-steps' partition and order, not on the tile shape), and take the cheapest
// of their tile shapes for that partition.
gemm_plan plan_of(int epi, const launch_sizes & z, int max_splits) {
    const gemm_plan plain = plan_plain(z, max_splits);
    if (epi == EPI_PLAIN) return plain;
    const int cls = epi == EPI_RESIDUAL ? CLASS_RESIDUAL : CLASS_FUSED, S = plain.splits;
    const double cold = z.cold(cls);
    gemm_plan best;
    launch_sizes y = z;
    if (cls == CLASS_FUSED) y.N[0] = glu_columns(z.N[0]);
    else if (S == 1 && plain.tile().kg == 1) best = plan_mixed(cls, z);
    for (int k = 0; k < SHAPES; k++) {
        const tile_shape & t = TILES[k];
        if (RATES[cls][k].step == 0 || t.kg != plain.tile().kg || (k == SHAPE_O && !whole_o_tiles(z))) continue;
        const double us = plan_us(cls, k, y.tiles(t.bm, t.bn), S, y, cold);
        if (us < best.us) best = {k, S, 0, us};
    }
    return best;
}

// The tiles of a plan.
int64_t plan_tiles(int epi, const gemm_plan & plan, launch_sizes z) {
    if (epi >= 0) z.N[0] = glu_columns(z.N[0]);
    return z.tiles(plan.tile().bm, plan.tile().bn);
}

// Plans and launches a GEMM. A split-K plan takes its workspace from `fixed`
// when given (no allocation: a plan that does not fit is rejected, and the
// counters it uses are cleared first), else from the stream's, in use here
// until the launch is queued. Under capture on a stream whose workspace is
// too small it is the best unsplit plan instead.
template <int EPI>
int launch_any(const gemm_params & p, const int64_t * N, hipStream_t s, const char * name,
               const sk_space * fixed = nullptr) {
    int dev = 0;
    (void) hipGetDevice(&dev);
    const int64_t Nt = glu_columns(N[0]);
    const int64_t * cols = EPI >= 0 ? &Nt : N;
    const launch_sizes z = sizes_of(p, N, cu_count(dev));
    gemm_plan pp = plan_of(EPI, z, ZEST_GEMM_MAX_SPLIT);
    std::unique_lock<std::mutex> lock(g_sk_mu, std::defer_lock);
    sk_space sp;
    if (pp.splits > 1) {
        const int64_t T = plan_tiles(EPI, pp, z);
        const size_t partial_bytes = partial_bytes_of(pp.kind, T, pp.splits), n_counters = counters_of(pp.kind, T);
        if (fixed) {
            if (partial_bytes > fixed->partial_bytes || n_counters > fixed->n_counters)
                return zest::fail(ZEST_E_ARG,
                                  "%s: this shape's split-K plan needs %zu bytes of partial sums and %zu counters; "
                                  "the static workspace holds %zu bytes and %zu counters",
                                  name, partial_bytes, n_counters, fixed->partial_bytes, fixed->n_counters);
            sp = *fixed;
            hipLaunchKernelGGL(clear_counters, dim3((unsigned) ((n_counters + 255) / 256)), dim3(256), 0, s,
                               sp.counters, (int) n_counters);
        } else {
            lock.lock();
            const int st = sk_reserve(s, partial_bytes, n_counters, sp, name);
            if (st != ZEST_OK) return st;
            if (!sp.partial) pp = plan_of(EPI, z, 1);
        }
    }
    const int S = pp.splits;
    switch (pp.kind) {
        case SHAPE_GLU: return launch<cfg_glu, EPI>(p, cols, S, sp, s, name);
        case SHAPE_SMALL: return launch<cfg_small, EPI>(p, cols, S, sp, s, name);
        case SHAPE_MID: return launch<cfg_mid, EPI>(p, cols, S, sp, s, name);
        case SHAPE_MID2: return launch<cfg_mid2, EPI>(p, cols, S, sp, s, name);
        case SHAPE_TINY2: return launch<cfg_tiny2, EPI>(p, cols, S, sp, s, name);
        case SHAPE_TINY2X2: return launch<cfg_tiny2x2, EPI>(p, cols, S, sp, s, name);
        case SHAPE_TINY: return launch<cfg_tiny, EPI>(p, cols, S, sp, s, name);
        default: break;
    }
    if constexpr (EPI < 0) {
        if (pp.kind == SHAPE_BIG) return launch<cfg_big, EPI>(p, N, S, sp, s, name);
        if (pp.kind == SHAPE_O) return launch<cfg_o, EPI>(p, N, S, sp, s, name);
        if (pp.kind == SHAPE_MIXED) return launch_mixed<cfg_glu, cfg_half8, EPI>(p, N, pp.nbig, s, name);
    }
    return zest::fail(ZEST_E_ARG, "%s: no plan", name);
}

// The parts of a launch's parameters common to every kind.
gemm_params base_params(const void * a, int64_t M, int64_t K, uint32_t * nonfinite) {
    gemm_params p{};
    p.a = (const uint8_t *) a;
    p.M = M;
    p.a_kstride = (int) ((zest_rows_padded(M) / ZEST_XGROUP_ROWS) * ZEST_XGROUP_BYTES);
    p.nk = (int) (zest_k_padded(K) / ZEST_TILE_K);
    p.nonfinite = nonfinite;
    return p;
}

gemm_weight weight_of(const void * w, int64_t N, float * c, int64_t ldc) {
    gemm_weight g{};
    g.w = (const uint8_t *) w;
    g.c = c;
    g.n = N;
    g.ldc = ldc;
    g.w_kstride = (int) ((zest_rows_padded(N) / ZEST_TILE_ROWS) * ZEST_TILE_BYTES);
    return g;
}

// The rows of one launch's band. A launch reaches its output (and a
// residual) through buffer resources whose byte ranges are 32-bit, so an
// output of rows `ld` floats apart runs as bands of whole 256-row tiles, each
// under 2 GiB, one launch a band (the reference likewise cuts a claimed
// matmul into NPU calls of at most 1024 rows, src/xdna-npu.cpp:392-420).
// 0 when not even 256 rows fit.
int64_t band_rows(int64_t ld) {
    const int64_t rows = ((1ll << 31) - 1) / (ld * 4);
    return rows / ZEST_ROW_ALIGN * ZEST_ROW_ALIGN;
}

// The launch parameters of the band of rows [r0, r0 + rows): the activation
// operand from row r0 on (whole 32-row groups; the K-step stride stays the
// whole operand's) and each weight's output from its row r0.
gemm_params band_of(const gemm_params & p, int64_t r0, int64_t rows) {
    gemm_params q = p;
    q.M = rows;
    q.a = p.a + r0 / ZEST_XGROUP_ROWS * ZEST_XGROUP_BYTES;
    for (int i = 0; i < p.nw; i++)
        if (q.wt[i].c) q.wt[i].c += r0 * q.wt[i].ldc;
    if (q.res) q.res += r0 * q.ldr;
    return q;
}

bool aligned_to(const void * p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// zest_gemm_group's checks and launches. A no-alloc call takes its split-K
// workspace from the device's static array (looked up once the arguments
// pass), else from the per-stream workspace.
int gemm_group(const void * a, int64_t M, int64_t K, int n, const void * const * w, const int64_t * N,
               float * const * c, const int64_t * ldc, uint32_t * nonfinite, void * stream, const char * name,
               bool noalloc) {
    ZEST_REQUIRE(a && w && N && c && ldc, "%s: null pointer", name);
    ZEST_REQUIRE(n >= 1 && n <= ZEST_GEMM_MAX_GROUP, "%s: %d weights (1..%d)", name, n, ZEST_GEMM_MAX_GROUP);
    ZEST_REQUIRE(M > 0 && K > 0 && K % 8 == 0, "%s: M=%lld K=%lld", name, (long long) M, (long long) K);
    ZEST_REQUIRE(zest_act_bytes(M, K) < (1ull << 31), "%s: activations must be under 2 GiB", name);
    ZEST_REQUIRE(aligned_to(a, 16) && aligned_to(nonfinite, 4), "%s: a must be 16-byte aligned, nonfinite 4", name);
    gemm_params p = base_params(a, M, K, nonfinite);
    p.nw = n;
    int64_t ld_max = 0;
    for (int i = 0; i < n; i++) {
        ZEST_REQUIRE(w[i] && c[i], "%s: null weight or output %d", name, i);
        ZEST_REQUIRE(aligned_to(w[i], 16) && aligned_to(c[i], 4),
                     "%s: weight %d must be 16-byte aligned and its output 4", name, i);
        ZEST_REQUIRE(N[i] > 0 && ldc[i] >= N[i], "%s: weight %d: N=%lld ldc=%lld", name, i, (long long) N[i],
                     (long long) ldc[i]);
        ZEST_REQUIRE(zest_bfp16_bytes(N[i], K) < (1ull << 31), "%s: weight %d must be under 2 GiB (N=%lld K=%lld)",
                     name, i, (long long) N[i], (long long) K);
        p.wt[i] = weight_of(w[i], N[i], c[i], ldc[i]);
        ld_max = std::max(ld_max, ldc[i]);
    }
    const int64_t band = band_rows(ld_max);
    ZEST_REQUIRE(band > 0, "%s: 256 output rows of %lld floats must be under 2 GiB", name, (long long) ld_max);
    sk_space ws;
    const sk_space * fixed = nullptr;
    if (noalloc) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return zest::fail(ZEST_E_HIP, "%s: hipGetDevice failed", name);
        uint8_t * base = nullptr;
        const int st = scratch_address(dev, &base);
        if (st != ZEST_OK) return st;
        ws.partial = reinterpret_cast<float *>(base);
        ws.partial_bytes = ZEST_NOALLOC_PARTIAL_BYTES;
        ws.counters = reinterpret_cast<uint32_t *>(base + ZEST_NOALLOC_PARTIAL_BYTES);
        ws.n_counters = ZEST_NOALLOC_COUNTERS;
        fixed = &ws;
    }
    const hipStream_t s = zest::as_stream(stream);
    for (int64_t r0 = 0; r0 < M; r0 += band) {
        const int st = launch_any<EPI_PLAIN>(band_of(p, r0, std::min(band, M - r0)), N, s, name, fixed);
        if (st != ZEST_OK) return st;
    }
    return ZEST_OK;
}

} // namespace

namespace zest {

int scratch_setup(int dev) {
    uint8_t * p = nullptr;
    return scratch_address(dev, &p);
}

} // namespace zest

extern "C" int zest_gemm_group(const void * a, int64_t M, int64_t K, int n, const void * const * w, const int64_t * N,
                               float * const * c, const int64_t * ldc, uint32_t * nonfinite, void * stream) {
    return gemm_group(a, M, K, n, w, N, c, ldc, nonfinite, stream, "zest_gemm", false);
}

extern "C" int zest_gemm_group_noalloc(const void * a, int64_t M, int64_t K, int n, const void * const * w,
                                       const int64_t * N, float * const * c, const int64_t * ldc,
                                       uint32_t * nonfinite, void * stream) {
    return gemm_group(a, M, K, n, w, N, c, ldc, nonfinite, stream, "zest_gemm_group_noalloc", true);
}

extern "C" int zest_gemm_plan(int kind, int64_t M, int64_t K, int n, const int64_t * N, int cus, zest_plan * out) {
    ZEST_REQUIRE(N && out, "zest_gemm_plan: null pointer");
    ZEST_REQUIRE(kind >= ZEST_PLAN_RESIDUAL && kind <= ZEST_GLU_GEGLU_QUICK, "zest_gemm_plan: kind %d", kind);
    ZEST_REQUIRE(n >= 1 && n <= (kind == ZEST_PLAN_PLAIN ? ZEST_GEMM_MAX_GROUP : 1), "zest_gemm_plan: %d weights", n);
    ZEST_REQUIRE(M > 0 && K > 0 && K % 8 == 0 && cus > 0, "zest_gemm_plan: M=%lld K=%lld cus=%d", (long long) M,
                 (long long) K, cus);
    for (int i = 0; i < n; i++) ZEST_REQUIRE(N[i] > 0, "zest_gemm_plan: N[%d]=%lld", i, (long long) N[i]);
    static_assert(ZEST_PLAN_PLAIN == EPI_PLAIN && ZEST_PLAN_RESIDUAL == EPI_RESIDUAL, "a plan's kinds are the epilogues");
    gemm_params p = base_params(nullptr, M, K, nullptr);
    p.nw = n;
    const launch_sizes z = sizes_of(p, N, cus);
    const gemm_plan plan = plan_of(kind, z, ZEST_GEMM_MAX_SPLIT);
    const tile_shape & t = plan.tile();
    const int64_t T = plan_tiles(kind, plan, z);
    *out = {t.bm, t.bn, t.waves, t.kg, t.per_cu, plan.splits, T, plan.kind == SHAPE_MIXED ? plan.nbig : T,
            plan.splits > 1 ? (int64_t) partial_bytes_of(plan.kind, T, plan.splits) : 0};
    return ZEST_OK;
}

extern "C" int zest_release_stream(void * stream) {
    const hipStream_t s = zest::as_stream(stream);
    std::lock_guard<std::mutex> lock(g_sk_mu);
    bool synced = false;
    for (auto it = g_sk_spaces.begin(); it != g_sk_spaces.end();) {
        if (it->first.second != sk_stream_of(s)) {
            ++it;
            continue;
        }
        // launches still queued on the stream may use the workspace
        if (!synced && hipStreamSynchronize(s) != hipSuccess)
            return zest::fail(ZEST_E_HIP, "zest_release_stream: stream synchronize");
        synced = true;
        if (it->second.partial) (void) hipFree(it->second.partial);
        if (it->second.counters) (void) hipFree(it->second.counters);
        for (void * b : it->second.held) (void) hipFree(b);
        it = g_sk_spaces.erase(it);
    }
    return ZEST_OK;
}

extern "C" int zest_gemm(const void * a, int64_t M, const void * w, int64_t N, int64_t K, float * c, int64_t ldc,
                         uint32_t * nonfinite, void * stream) {
    return zest_gemm_group(a, M, K, 1, &w, &N, &c, &ldc, nonfinite, stream);
}

extern "C" int zest_gemm_residual(const void * a, int64_t M, const void * w, int64_t N, int64_t K, const float * res,
                                  int64_t ldr, float * c, int64_t ldc, uint32_t * nonfinite, void * stream) {
    ZEST_REQUIRE(a && w && c && res, "zest_gemm_residual: null pointer");
    ZEST_REQUIRE(M > 0 && N > 0 && K > 0 && K % 8 == 0, "zest_gemm_residual: M=%lld N=%lld K=%lld", (long long) M,
                 (long long) N, (long long) K);
    ZEST_REQUIRE(ldc >= N && ldr >= N, "zest_gemm_residual: ldc %lld / ldr %lld < N %lld", (long long) ldc,
                 (long long) ldr, (long long) N);
    ZEST_REQUIRE((reinterpret_cast<uintptr_t>(res) & 15) == 0 && ldr % 4 == 0,
                 "zest_gemm_residual: the residual's rows must be 16-byte aligned");
    ZEST_REQUIRE(aligned_to(a, 16) && aligned_to(w, 16) && aligned_to(c, 4) && aligned_to(nonfinite, 4),
                 "zest_gemm_residual: a and w must be 16-byte aligned, c and nonfinite 4");
    ZEST_REQUIRE(zest_act_bytes(M, K) < (1ull << 31) && zest_bfp16_bytes(N, K) < (1ull << 31),
                 "zest_gemm_residual: operands must be under 2 GiB");
    const int64_t band = band_rows(std::max(ldc, ldr));
    ZEST_REQUIRE(band > 0, "zest_gemm_residual: 256 rows of the output and residual must be under 2 GiB");
    gemm_params p = base_params(a, M, K, nonfinite);
    p.nw = 1;
    p.wt[0] = weight_of(w, N, c, ldc);
    p.res = res;
    p.ldr = ldr;
    const hipStream_t s = zest::as_stream(stream);
    for (int64_t r0 = 0; r0 < M; r0 += band) {
        const int st = launch_any<EPI_RESIDUAL>(band_of(p, r0, std::min(band, M - r0)), &N, s, "zest_gemm_residual");
        if (st != ZEST_OK) return st;
    }
    return ZEST_OK;
}

extern "C" int zest_gemm_glu(int kind, const void * a, int64_t M, const void * w_gu, int64_t F, int64_t K,
                             void * xout, float * h, int64_t ldh, uint32_t * nonfinite, void * stream) {
    ZEST_REQUIRE(a && w_gu && (xout || h), "zest_gemm_glu: null pointer");
    ZEST_REQUIRE(M > 0 && F > 0 && F % 32 == 0 && K > 0 && K % 8 == 0, "zest_gemm_glu: M=%lld F=%lld K=%lld",
                 (long long) M, (long long) F, (long long) K);
    ZEST_REQUIRE(!h || ldh >= F, "zest_gemm_glu: ldh %lld < F %lld", (long long) ldh, (long long) F);
    ZEST_REQUIRE(aligned_to(a, 16) && aligned_to(w_gu, 16) && aligned_to(xout, 16) && aligned_to(h, 4) &&
                     aligned_to(nonfinite, 4),
                 "zest_gemm_glu: a, w_gu and xout must be 16-byte aligned, h and nonfinite 4");
    ZEST_REQUIRE(zest_act_bytes(M, K) < (1ull << 31) && zest_bfp16_bytes(2 * F, K) < (1ull << 31) &&
                     zest_act_bytes(M, F) < (1ull << 31),
                 "zest_gemm_glu: operands must be under 2 GiB (M=%lld F=%lld K=%lld)", (long long) M, (long long) F,
                 (long long) K);
    gemm_params p = base_params(a, M, K, nonfinite);
    const int64_t N = 2 * F;
    p.nw = 1;
    p.wt[0] = weight_of(w_gu, N, nullptr, 0);
    p.xout = (uint8_t *) xout;
    p.h = h;
    p.ldh = ldh;
    hipStream_t s = zest::as_stream(stream);
    const char * name = "zest_gemm_glu";
    switch (kind) {
        case ZEST_GLU_SWIGLU: return launch_any<ZEST_GLU_SWIGLU>(p, &N, s, name);
        case ZEST_GLU_GEGLU: return launch_any<ZEST_GLU_GEGLU>(p, &N, s, name);
        case ZEST_GLU_GEGLU_ERF: return launch_any<ZEST_GLU_GEGLU_ERF>(p, &N, s, name);
        case ZEST_GLU_GEGLU_QUICK: return launch_any<ZEST_GLU_GEGLU_QUICK>(p, &N, s, name);
        case ZEST_GLU_REGLU: return launch_any<ZEST_GLU_REGLU>(p, &N, s, name);
        default: return zest::fail(ZEST_E_UNSUPPORTED, "zest_gemm_glu: GLU kind %d", kind);
    }
}
