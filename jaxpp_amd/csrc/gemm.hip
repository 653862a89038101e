// bf16 GEMM on gfx950 matrix cores (v_mfma_f32_16x16x32_bf16), operand tiles staged through
// LDS, with the epilogues a pipeline stage needs.
//
//   C[m,n] = epilogue( sum_k Aop[m,k] * Bop[n,k] )
//
// A workgroup of 4 or 8 waves owns a BM x BN output tile and walks K in steps
// of 64.  Operand tiles travel HBM -> LDS without passing through registers
// (global_load_lds_dwordx4), keeping the layout they have in HBM: an operand
// whose contraction index is contiguous in memory lands as swizzled [rows][64]
// slabs and is read back with 16-byte LDS reads; one whose contraction index
// is the slow one (the weights in a forward GEMM, both operands of a
// weight-gradient GEMM) lands as [64][rows] and is read back with the
// transposing 8-byte LDS reads (ds_read_b64_tr_b16).
//
// The weight operand is fed to the MFMA "A" port and the activation operand to
// the "B" port, so a lane ends up holding 4 consecutive n for one m; the
// epilogues regroup the tile through LDS and write whole rows.
//
// The 16x16x32 shape is chosen for what the device sustains, not for issue rate: on
// operands that change from one MFMA to the next it holds a higher clock than the
// 32x32x16 shape (2.03 against 1.82 PFLOP/s in a register-only loop; jpp_mfma_rate).
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <mutex>
#include <string>

#include "colsum.h"
#include "gemm_wave.h"

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

namespace {

// output tiles (jpp_gemm_args.tile)
enum { kTile128 = 1, kTile256x128 = 2, kTile128x256 = 3, kTile256 = 4, kTile64 = 5,
       kTile64x128 = 6 /* the library's own choice only */ };
constexpr long kCus = 256;
constexpr long kMostCus = 192;  // 256x256 tiles from which a forward grid of them is taken without asking

struct GemmParams {
  const bf16_t* a;
  const bf16_t* b;
  // a contraction spread over several operand pairs of k elements each (see k_parts in the
  // header): pair i > 0 is (a_more[i-1], b_more[i-1]); kt_part = K-steps per pair
  const bf16_t* a_more[3];
  const bf16_t* b_more[3];
  int k_parts, kt_part;
  // JPP_GROUP_K over several pairs: row groups of pair i > 0
  const int* seg_more[3];
  const int* seg_rows_more[3];
  void* c;
  void* c2;
  const bf16_t* bias;
  const bf16_t* resid;
  const bf16_t* aux;
  int m, n, k;
  long lda, ldb, ldc, ldc2, ldresid, ldaux;
  int gelu_tanh;
  int tiles_m, tiles_n;
  // grouped (mixture-of-experts) problems: seg[0..n_seg] are row offsets, multiples of 256
  const int* seg;
  const int* seg_rows;
  int n_seg, group_mode;
  int64_t group_rows;
  long stride_b, stride_c;
  // rotary embedding in the bf16 epilogue of the forward kernels (NULL: none): columns
  // [0, rope_cols) are heads of rope_hd elements, row r is position (rope_row0 + r) % rope_seq
  const float* rope_cos;
  const float* rope_sin;
  int rope_cols, rope_seq, rope_hd;
  long rope_row0;
  // JPP_GROUP_M with a bf16 epilogue as three launches (see group_head_rows): 1 = the 256x256
  // tiles of the rows before the split, 2 / 3 = 128x128 / 128x256 tiles over the rows behind
  // it (one of the two finds work), 0 = one launch for all rows
  int tail_split;
};

// One more problem of a launch that covers several independent products of one kind (same
// orientations, epilogue, contraction length and number of operand pairs): its operands and
// its place in the grid.  Workgroups first .. first + tiles_m tiles_n - 1 work on it.
struct GemmProblem {
  const bf16_t* a[4];
  const bf16_t* b[4];
  void* c;
  long lda, ldb, ldc;
  int tiles_m, tiles_n, first;
};
// kernel arguments: one problem, or (MP) up to four
template <bool MP>
struct GemmArgs {
  GemmParams p;
};
template <>
struct GemmArgs<true> {
  GemmParams p;          // problem 0 and everything the problems share
  GemmProblem more[3];   // problems 1..3; `first` past the grid for those not in use
  ColsumPanels cols;     // column sums that go along: the workgroups from col_first on
  int col_first;
  long col_rows;
};

// Whether a form of several problems takes column sums along: the small tiles, which a layer of few rows has.
constexpr bool takes_column_sums(int bm, int bn) { return bm * bn <= 128 * 128; }

// (sigmoid through the hardware reciprocal, 1 ulp: a correctly rounded division is ten
// instructions, and an epilogue evaluates 64 - 128 of these per lane)
__device__ __forceinline__ float swiglu_f(float g, float u) {
  return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
}
__device__ __forceinline__ void swiglu_grad_f(float g, float u, float d, float& dg, float& du) {
  const float sg = __builtin_amdgcn_rcpf(1.0f + __expf(-g));
  dg = d * u * sg * (1.0f + g * (1.0f - sg));
  du = d * g * sg;
}

// Output tile of a workgroup.  Consecutive workgroup ids land on different
// XCDs (8 of them, each with its own L2); give every XCD a contiguous range of
// tiles, and inside a range walk GROUP tile-rows at a time so the B panels in
// flight stay L2 resident.
constexpr int kColumnSplitRows = 16384;  // rows from which XCDs split by columns

template <bool WGRAD, int BM>
__device__ __forceinline__ void tile_of_block(int pid, int tiles_m, int tiles_n, bool front_only, int& tm, int& tn) {
  const int nwg = tiles_m * tiles_n;
  if ((tiles_n & 7) == 0 && tiles_m * BM >= kColumnSplitRows) {
    // Very tall outputs (the experts' row-grouped products: 16 384 token copies and more; not
    // by tile rows: 4096 rows of 64x64 tiles, N = 512, K = 7168 took 71 us this way, 43 the other):
    // every XCD owns an eighth of the tile columns and walks them 8 tile-rows at a time, so a
    // B panel - which changes from expert to expert - is fetched by one XCD only.  The split
    // below would hand whole row groups to single XCDs and have each of them stream every
    // column of B (+1.3 % on the Mixtral-shaped stage and, through the 112-tile-row weight
    // gradient of its down projection, +0.8 % on the 70B-shaped one; at 16 tile-rows it costs
    // 2.5 %, at 56 it changes nothing).
    const int x = pid & 7, l = pid >> 3, cols_per = tiles_n >> 3;
    const int group = l / (8 * cols_per), within = l - group * 8 * cols_per;
    const int gsize = min(tiles_m - group * 8, 8);
    tm = group * 8 + within % gsize;
    tn = x * cols_per + within / gsize;
    return;
  }
  // An XCD's range is an eighth of the tiles, the first tiles % 8 XCDs' one tile more.  (Left as
  // they come, the tiles of a column land on as many XCDs and each fetches the column's B panel:
  // 492 tiles of 64x64, K = 5696, 55 us instead of 34; 4148 of 128x128, K = 704, 147 instead of 101;
  // over 123 random products in 64x64 tiles 12 % on average.)  Row groups in a number of
  // tiles that is not a multiple of 8 are dealt out all the same: only the front of their grid
  // holds data, and the last XCDs would have none of it.
  if ((nwg & 7) == 0 || !front_only) {
    const int x = pid & 7;
    pid = x * (nwg >> 3) + min(x, nwg & 7) + (pid >> 3);
  }
  // Tile rows an XCD walks at a time.  Weight gradients (both operands activations, a panel
  // 8 MiB and more) whose output is at most 16 tiles high or wide take 4: measured, A/B on
  // one box, -0.7 % on the weight-gradient launches of the Llama-3-8B- and Mixtral-shaped
  // stages (-0.2 % step time); 4 for every weight gradient cost the 70B-shaped stage 0.6 %
  // (32 x 40 .. 32 x 224 tiles), 16 for every product cost 1.8 %.
  const int GROUP = WGRAD && (tiles_m <= 16 || tiles_n <= 16) ? 4 : 8;
  const int width = GROUP * tiles_n;
  const int group = pid / width;
  const int first = group * GROUP;
  const int gsize = min(tiles_m - first, GROUP);
  tm = first + (pid % width) % gsize;
  tn = (pid % width) / gsize;
}

// Operand tile of K-step kt when the contraction runs over up to four operand pairs: pair i
// starts at K-step c_i (c_0 = 0; c_1 <= c_2 <= c_3, equal where a pair has no steps).  All
// arguments are wave-uniform.
__device__ __forceinline__ const bf16_t* part_ptr(const bf16_t* p0, const bf16_t* p1,
                                                  const bf16_t* p2, const bf16_t* p3, int kt,
                                                  int c1, int c2, int c3, long step) {
  const int part = (kt >= c1) + (kt >= c2) + (kt >= c3);
  const bf16_t* base = part == 0 ? p0 : part == 1 ? p1 : part == 2 ? p2 : p3;
  const int start = part == 0 ? 0 : part == 1 ? c1 : part == 2 ? c2 : c3;
  return base + (long)(kt - start) * step;
}
// Row-grouped products know the number of rows in use (`rows`, a multiple of 256) on the
// device only; the grid covers the buffer's capacity.  When the 256x256 tiles of those rows
// end in a round that fills at most half of the 256 CUs, the tile rows of that round are
// left to a second launch of smaller tiles: 128x128 when the round holds at most 64 tiles
// (at most one round of the small tiles, about 0.43 of the time), 128x256 when it holds up to
// 128 (one round again, about 0.6).  Returns the first row of that part (`rows` when there
// is none) and which of the two launches it belongs to (tail_split values 2 and 3).
__device__ __forceinline__ long group_head_rows(int rows, int n, int& tail_kind) {
  const int tm = rows / 256, tn = n / 256, total = tm * tn, rest = total % 256;
  const bool split = total > 256 && rest > 0 && rest <= 128 && rest % tn == 0;
  tail_kind = rest <= 64 ? 2 : 3;
  return split ? (long)(tm - rest / tn) * 256 : (long)rows;
}
// K-steps that hold data of row group e of a grouped contraction
__device__ __forceinline__ int group_steps(const int* seg, const int* seg_rows, int e) {
  const int rows = seg_rows ? min(seg_rows[e], seg[e + 1] - seg[e]) : seg[e + 1] - seg[e];
  return (rows + 63) / 64;
}

// Whether a form streams the accumulator's rows through LDS beside its operand stages (C += A B): the
// large tiles, alone on their CU.  (A 128x128 tile with room for the rows would be alone on its CU too: the
// gradients of the epilogue's comment 115 us instead of 87.)
constexpr bool streams_accumulator(int bm, int bn) { return bm * bn > 128 * 128; }

template <int BM, int BN, bool TA, bool TB, int EPI, int NW, int NS, bool KP = false, bool MP = false,
          int KG = 1>
__global__ __launch_bounds__(NW * KG * 64) void gemm_kernel(GemmArgs<MP> args) {
  GemmParams p = args.p;
  int bid = blockIdx.x;  // this workgroup's tile within its problem
  if constexpr (MP && takes_column_sums(BM, BN)) {
    if (bid >= args.col_first) {
      extern __shared__ __align__(1024) uint8_t smem[];
      colsum_panel<NW * KG * 64>(args.cols, bid - args.col_first, args.col_rows, (float2(*)[64])smem);
      return;
    }
  }
  if constexpr (MP) {
    // which problem this workgroup belongs to (wave-uniform: scalar compares and selects,
    // field by field - never an index into the kernel arguments)
    const bool s1 = bid >= args.more[0].first, s2 = bid >= args.more[1].first,
               s3 = bid >= args.more[2].first;
#define JPP_PICK(own, field) \
  (s3 ? args.more[2].field : s2 ? args.more[1].field : s1 ? args.more[0].field : (own))
    p.a = JPP_PICK(p.a, a[0]);
    p.b = JPP_PICK(p.b, b[0]);
    p.a_more[0] = JPP_PICK(p.a_more[0], a[1]);
    p.a_more[1] = JPP_PICK(p.a_more[1], a[2]);
    p.a_more[2] = JPP_PICK(p.a_more[2], a[3]);
    p.b_more[0] = JPP_PICK(p.b_more[0], b[1]);
    p.b_more[1] = JPP_PICK(p.b_more[1], b[2]);
    p.b_more[2] = JPP_PICK(p.b_more[2], b[3]);
    p.c = JPP_PICK(p.c, c);
    p.lda = JPP_PICK(p.lda, lda);
    p.ldb = JPP_PICK(p.ldb, ldb);
    p.ldc = JPP_PICK(p.ldc, ldc);
    p.tiles_m = JPP_PICK(p.tiles_m, tiles_m);
    p.tiles_n = JPP_PICK(p.tiles_n, tiles_n);
    bid -= JPP_PICK(0, first);
#undef JPP_PICK
  }
  // Which waves issue the HBM -> LDS copies.  With two waves per SIMD the older one is served
  // first whenever it has an instruction ready, so it runs ahead and then waits at the
  // K-step's barrier for the younger one, whose K-step is therefore what a tile's time is made
  // of - and a wave issues in order: every copy it issues (16 cycles of the CU's path to
  // memory, longer when other waves' copies are queued) holds back its next MFMA.  So the four
  // older waves issue all copies (twice as many each) in the time they would wait anyway, and
  // the younger ones only read fragments and multiply: 2.4 - 3.3 % of the step on the Llama-
  // and Mixtral-shaped stages, 2 % on the BERT-large-shaped one (single GEMMs: TN -5 %,
  // NN / NT -2.5 % at 4096 x 28672 x 4096; two shapes of twelve +1 - 2 %).
  constexpr int DW = NW == 8 ? 4 : NW;
  using TileA = DmaTile<BM, TA, DW>;
  using TileB = DmaTile<BN, TB, DW>;
  constexpr int A_BYTES = TileA::BYTES, STAGE = TileA::BYTES + TileB::BYTES;
  constexpr int WN = NW / 2;                        // waves: 2 along m, NW/2 along n
  // 16x16 MFMA tiles per wave.  A K-step runs them in 2 HS blocks of TMH x TN (32 contraction
  // elements each); large wave tiles take the rows in two halves so that the fragments of
  // two blocks fit in registers beside the accumulators
  constexpr int TM = BM / 32, TN = BN / (16 * WN), HS = TM * TN >= 32 ? 2 : 1, TMH = TM / HS;
  constexpr int NB = 2 * HS;
  extern __shared__ __align__(1024) uint8_t smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  // (wave-uniform where the waves differ in what they do: a scalar branch around the copies)
  const int wave_all = DW == NW && KG == 1 ? tid >> 6 : __builtin_amdgcn_readfirstlane(tid >> 6);
  // KG > 1: the workgroup is KG groups of NW waves that share the output tile and take the
  // K-steps in turn (group g steps g, g + KG, ...), each with LDS stages of its own
  // - small tiles, whose K-step is a chain of latencies (barrier, fragment reads, copies) and
  // not work: at 512 x 1024 x 4096 (128 tiles of 64x64) one group takes 670 cycles a step with
  // eight stages, two groups 900 a pair of steps with four (22 -> 15.5 us; four groups with the
  // two stages that then fit 19 us: the copies land too late; five stages instead of four
  // change nothing).  Larger tiles gain nothing (128x128: 28 us one group, 35 us two).
  const int grp = KG == 1 ? 0 : wave_all / NW, wave = KG == 1 ? wave_all : wave_all % NW;
  const bool dma_wave = wave < DW;
  const int wm = wave / WN, wn = wave % WN;
  int tm, tn;
  const int tiles = p.tiles_m * p.tiles_n;
  tile_of_block<TA && TB, BM>(p.group_mode == JPP_GROUP_K ? bid % tiles : bid, p.tiles_m, p.tiles_n,
                          p.group_mode == JPP_GROUP_M, tm, tn);
  long m0 = (long)tm * BM;
  const long n0 = (long)tn * BN;
  if constexpr (EPI == JPP_EPI_BF16 && !KP && !MP) {   // (the launcher splits these only)
    if (p.group_mode == JPP_GROUP_M && p.tail_split) {
      int tail_kind;
      const long head = group_head_rows(p.seg[p.n_seg], p.n, tail_kind);
      if (p.tail_split == 1 ? m0 >= head : p.tail_split != tail_kind) return;
      if (p.tail_split != 1) m0 += head;
    }
  }

  const long a_off = TA ? m0 : m0 * p.lda, b_off = TB ? n0 : n0 * p.ldb;
  const bf16_t* a_src = p.a + a_off;
  const bf16_t* b_src = p.b + b_off;
  int kt_n = p.k / 64 * (KP ? p.k_parts : 1);
  // several operand pairs: first K-step of pairs 1..3 and their operands at this tile
  int c1 = p.kt_part, c2 = 2 * p.kt_part, c3 = 3 * p.kt_part;
  const bf16_t* a1 = KP ? p.a_more[0] + a_off : a_src;
  const bf16_t* a2 = KP ? p.a_more[1] + a_off : a_src;
  const bf16_t* a3 = KP ? p.a_more[2] + a_off : a_src;
  const bf16_t* b1 = KP ? p.b_more[0] + b_off : b_src;
  const bf16_t* b2 = KP ? p.b_more[1] + b_off : b_src;
  const bf16_t* b3 = KP ? p.b_more[2] + b_off : b_src;
  if (p.group_mode == JPP_GROUP_M) {
    // rows of A and C are grouped by expert; each group multiplies its own B
    if (m0 >= p.seg[p.n_seg]) return;
    int e = 0;
    while (p.seg[e + 1] <= m0) ++e;
    b_src += (long)e * p.stride_b;
  } else if (p.group_mode == JPP_GROUP_K) {
    // one output per expert; the contraction runs over the expert's rows
    const int e = bid / tiles;
    const long r0 = p.seg[e];
    // rows past the group's data are zero padding: steps made of nothing else are skipped
    kt_n = group_steps(p.seg, p.seg_rows, e);
    a_src += r0 * p.lda;
    b_src += r0 * p.ldb;
    if constexpr (KP) {
      // every further pair brings its own row groups (pair by pair, never an index into the
      // kernel arguments); a pair past k_parts starts where the contraction ends
      c1 = c2 = c3 = kt_n;
      if (p.k_parts > 1) {
        const long r = p.seg_more[0][e];
        a1 += r * p.lda; b1 += r * p.ldb;
        kt_n += group_steps(p.seg_more[0], p.seg_rows_more[0], e);
        c2 = c3 = kt_n;
      }
      if (p.k_parts > 2) {
        const long r = p.seg_more[1][e];
        a2 += r * p.lda; b2 += r * p.ldb;
        kt_n += group_steps(p.seg_more[1], p.seg_rows_more[1], e);
        c3 = kt_n;
      }
      if (p.k_parts > 3) {
        const long r = p.seg_more[2][e];
        a3 += r * p.lda; b3 += r * p.ldb;
        kt_n += group_steps(p.seg_more[2], p.seg_rows_more[2], e);
      }
    }
    p.c = EPI == JPP_EPI_BF16 ? (void*)((bf16_t*)p.c + (long)e * p.stride_c)
                              : (void*)((float*)p.c + (long)e * p.stride_c);
    if (kt_n == 0 && EPI == JPP_EPI_ACC_F32) return;
  }
  const long a_step = TA ? 64 * p.lda : 64;
  const long b_step = TB ? 64 * p.ldb : 64;
  // operand tiles of K-step kt: with several operand pairs the steps run through pair 0,
  // then pair 1, ... (kt and the pair index are wave-uniform: scalar arithmetic; the pair
  // pointers are picked by a chain of selects, never by indexing the kernel arguments)
  // (kernels built without KP take one pair and keep the plain address arithmetic)
#define a_at(kt) (KP ? part_ptr(a_src, a1, a2, a3, (kt), c1, c2, c3, a_step) : a_src + (long)(kt) * a_step)
#define b_at(kt) (KP ? part_ptr(b_src, b1, b2, b3, (kt), c1, c2, c3, b_step) : b_src + (long)(kt) * b_step)

  // of tile (i, j) a lane holds row wm BM/2 + 16 i + lane % 16 and the four columns
  // wn BN/WN + 16 j + 4 (lane / 16) + {0..3}
  f32x4 acc[TM][TN];
  // C += A B (EPI_ACC_F32): the epilogue only stores; the fp32 tile in memory is folded into
  // the accumulators during the first K-steps.  It travels HBM -> LDS like the operands, NW
  // whole rows (BN * 4 bytes each, one per wave) at a time, into one of NS+1 buffers behind
  // the operand stages: batch b is requested at the end of K-step b, after that K-step's
  // operand copies, and read out of LDS at the wait point of K-step b+NS.  The waits in
  // between leave the youngest requests in flight (vmcnt counts in order), so a batch has
  // NS K-steps to arrive and no K-step waits for HBM on its account; reading whole rows
  // keeps HBM on long bursts where a lane-per-row layout would touch 16 rows at once.  K
  // loops too short for that add the old values in the epilogue, where rows are whole too.
  static_assert(BN * 4 <= 1024, "a row of the fp32 tile is one 64-lane copy");
  constexpr int NBT = BM / NW, C_LDS = NS * (BM + BN) * 128, C_PITCH = 1024 + 16;  // a copy is 1 KB
  constexpr bool STREAM_C = EPI == JPP_EPI_ACC_F32 && streams_accumulator(BM, BN);
  const bool stream_c = STREAM_C && kt_n >= NBT + NS;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // byte offset, from the start of C, of this lane's 16 bytes of tile row `wave`
  // (lanes past the end of a narrow row repeat its last piece)
  const uint32_t c_off0 =
      (uint32_t)(((m0 + wave) * p.ldc + n0 + min(lane, BN / 4 - 1) * 4) * 4);
  uint8_t* const stages = smem + grp * (NS * STAGE);
  const uint32_t lds0 = lds_address(stages);
  // iteration t of a group is K-step t KG + grp of the contraction; the groups meet at every
  // iteration's barrier, so those that have run out of steps take part without multiplying
  const int it_n = KG == 1 ? kt_n : (kt_n + KG - 1) / KG;
  auto k_step = [&](int t) { return KG == 1 ? t : min(t * KG + grp, kt_n - 1); };
  typename TileA::Offsets offa;
  typename TileB::Offsets offb;
  TileA::offsets(offa, p.lda, wave, lane);
  TileB::offsets(offb, p.ldb, wave, lane);
  constexpr int IA = TileA::INSTS, IB = TileB::INSTS;
  const int row_w = wn * (BN / WN), row_x = wm * (BM / 2);

  // Software pipeline over K-steps of 64 with NS LDS stages:
  //   * the HBM -> LDS copy of K-step t+NS is issued inside K-step t, right after the
  //     barrier that retires stage t % NS's readers, so it has NS-1 K-steps to land;
  //   * that barrier sits in front of the last MFMA block of a K-step and the first
  //     fragments of K-step t+1 are read from LDS behind it, under those MFMAs.
  // Block q of a K-step multiplies contraction elements 32 (q / HS) .. + 31 of the stage: the
  // wave's TN fragments of B (read once per HS blocks) with part q % HS of its TM fragments
  // of A, each fragment read while the block before it computes.
  // Waits count requests from the youngest (vmcnt is in order): at the wait point of K-step
  // t the copies of K-steps t+2 .. t+NS-1 and the accumulator rows requested during the last
  // NS-1 K-steps may stay in flight (where a stage's refill is split over two K-steps, see
  // LATE below, its second half is the youngest request and everything is waited for).
  constexpr int OPB = IA + IB;  // operand copies per wave and K-step
  constexpr bool EXACT = NS == 2 && BM * BN <= 128 * 128;
  bf16x8 fw[2][TN], fx[2][TMH];
  if (kt_n > 0) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int k = k_step(min(s, it_n - 1));
      if (dma_wave && (!EXACT || s < it_n)) {
        TileA::template issue<0, IA>(uniform_ptr(a_at(k)), offa, lds0 + s * STAGE, wave);
        TileB::template issue<0, IB>(uniform_ptr(b_at(k)), offb, lds0 + s * STAGE + A_BYTES, wave);
      }
    }
    if constexpr (EXACT) dma_wait_groups<OPB, NS - 1>(it_n - 1);
    else dma_wait<(NS - 1) * OPB>();  // stage 0 has landed; the others may still be in flight
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < TN; ++j) fw[0][j] = TileB::frag16(stages + A_BYTES, row_w + j * 16, 0, lane);
#pragma unroll
  for (int i = 0; i < TMH; ++i) fx[0][i] = TileA::frag16(stages, row_x + i * 16, 0, lane);

  int st = 0;   // stage of K-step kt: kt % NS
  int cbi = 0;  // accumulator-row buffer of K-step kt: kt % (NS + 1)
  // The refill of a retired stage is 8 wave-level copies per wave, 64 per workgroup, and the
  // CU's path to memory takes one in 16 cycles: issued all behind the barrier, under the last
  // MFMA block, they kept that block waiting on the path (a wave issues in order) for twice
  // the time its MFMAs need.  With two stages the 256 x 256 tile therefore issues LATE of
  // its four parts under the first MFMA block of the next K-step instead (still three blocks
  // ahead of the wait for them): 4 - 6 % per K-step by timestamps inside the loop, 0.2 - 1 %
  // of the Llama-3-8B-shaped step depending on the device.  (3 or 4 parts late: slower again,
  // the copies land too late.)
  constexpr int LATE = (NS == 2 && BM == 256 && BN == 256 && NW == 8) ? 2 : 0;
  constexpr bool SPLIT = LATE > 0;
  // With two stages and two workgroups on a CU the last copies are not repeated: they would hold the
  // CU's path while the other workgroup's are due and this one's end would wait for them (512 x 4096
  // x 1024 with a GELU 15.1 -> 14.3 us, 512 x 3072 x 1024 12.5 -> 12.1).  Deep forms, alone on
  // their CU, and the 256 x 256 tile lose as much by the branches around their copies (0 - 2 %).
  const bf16_t* ga_late = nullptr;
  const bf16_t* gb_late = nullptr;
  int st_late = 0;
  for (int kt = 0; kt < it_n; ++kt) {
    const int nst = st + 1 == NS ? 0 : st + 1;
    const uint8_t* sa = stages + st * STAGE;
    const uint8_t* sb = sa + A_BYTES;
    const uint8_t* na = stages + nst * STAGE;
    const bool live = KG == 1 || kt * KG + grp < kt_n;
    // past the end the last K-step is fetched again, unused (EXACT: nothing is)
    const bool refill = dma_wave && (!EXACT || kt + NS < it_n);
    const int kn = k_step(min(kt + NS, it_n - 1));
    const bf16_t* ga = uniform_ptr(a_at(kn));
    const bf16_t* gb = uniform_ptr(b_at(kn));
#pragma unroll
    for (int ks = 0; ks < NB; ++ks) {
      const int cur = ks & 1, nxt = cur ^ 1, curw = ks / HS, part = ks % HS;
      if (ks < NB - 1) {
        if ((ks + 1) % HS == 0) {
#pragma unroll
          for (int j = 0; j < TN; ++j) fw[1][j] = TileB::frag16(sb, row_w + j * 16, 1, lane);
        }
#pragma unroll
        for (int i = 0; i < TMH; ++i)
          fx[nxt][i] = TileA::frag16(sa, row_x + ((ks + 1) % HS * TMH + i) * 16, (ks + 1) / HS, lane);
      } else {
        // every fragment of this stage is in registers: once all waves are here (and the
        // next stage has landed) this stage can be refilled
        {
          // accumulator rows requested during K-steps kt+1-NS .. kt-1 that may stay in flight
          int cin = 0;
          if (EPI == JPP_EPI_ACC_F32 && stream_c)
            cin = max(0, min(kt - 1, NBT - 1) - max(0, kt + 1 - NS) + 1);
          if (SPLIT || cin <= 0) dma_wait<(NS - 2) * OPB>();
          else if (cin == 1) dma_wait<(NS - 2) * OPB + 1>();
          else if (cin == 2) dma_wait<(NS - 2) * OPB + 2>();
          else dma_wait<(NS - 2) * OPB + 3>();
          static_assert(!STREAM_C || NS <= 4, "the wait above distinguishes up to three rows in flight");
        }
        lds_wait_all();
        __syncthreads();
        if constexpr (EPI == JPP_EPI_ACC_F32) {
          if (stream_c && kt >= NS && kt < NBT + NS) {
            // batch kt-NS (tile rows NW (kt-NS) .. + NW-1) is in LDS: the lanes that hold
            // those rows add them in.  Buffers are used round robin over NS+1, so the one
            // read here is written again only behind the next K-step's barrier.
            const int row0 = (kt - NS) * NW, rl = (lane & 15) - (row0 & 15);
            const int fold_buf = cbi + 1 == NS + 1 ? 0 : cbi + 1;  // (kt - NS) % (NS + 1)
            if (wm == row0 / (BM / 2) && rl >= 0 && rl < NW) {
              const uint8_t* src = smem + C_LDS + (fold_buf * NW + rl) * C_PITCH +
                                   (wn * (BN / WN) + (lane >> 4) * 4) * 4;
#pragma unroll
              for (int i = 0; i < TM; ++i)
                if (i == (row0 % (BM / 2)) / 16) {
#pragma unroll
                  for (int j = 0; j < TN; ++j) acc[i][j] += *(const f32x4*)(src + j * 64);
                }
            }
          }
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) fw[0][j] = TileB::frag16(na + A_BYTES, row_w + j * 16, 0, lane);
#pragma unroll
        for (int i = 0; i < TMH; ++i) fx[0][i] = TileA::frag16(na, row_x + i * 16, 0, lane);
      }
      // the refill of the retired stage is spread over this block's MFMAs: a wave that
      // issues its loads back to back waits on the memory pipeline with its MFMAs behind it
      constexpr int PARTS = TMH < IA && TMH < IB ? TMH : (IA < IB ? IA : IB);
      static_assert(IA % PARTS == 0 && IB % PARTS == 0 && TMH % PARTS == 0,
                    "loads per wave must split over the MFMA rows");
      // MFMAs go in 2x2 groups of tiles, walked so that from one MFMA to the next exactly one
      // operand changes: fewer operand bits toggle per issue than row by row, and the clock
      // under load follows the toggling (walks that change both operands at group borders,
      // whole rows, or columns first measured 0.5 - 1.2 % slower on the Llama-3-8B-shaped step)
      static_assert(TMH % 2 == 0 && TN % 2 == 0, "2x2 groups of MFMA tiles");
#pragma unroll
      for (int ib = 0; ib < TMH / 2; ++ib) {
        if (!SPLIT && ks == NB - 1) {
#pragma unroll
          for (int i = 2 * ib; i < 2 * ib + 2; ++i)
            if (i % (TMH / PARTS) == 0 && refill) {
              TileA::template issue_part<IA / PARTS>(i / (TMH / PARTS), ga, offa, lds0 + st * STAGE, wave);
              TileB::template issue_part<IB / PARTS>(i / (TMH / PARTS), gb, offb,
                                                     lds0 + st * STAGE + A_BYTES, wave);
            }
        }
        if constexpr (SPLIT) {
          static_assert(!SPLIT || (PARTS == 4 && TMH == 4 && LATE >= 2 && LATE <= 4),
                        "four parts, at most two of them in the last block (it has two slots)");
          // parts 0 .. 3 - LATE in the last block (spread from its end), the others one per
          // pair of MFMA rows from the start of the next K-step on
          const int slot = ks * 2 + ib;           // pair of MFMA rows within the K-step
          if (ks == NB - 1) {
            const int part = slot - (2 * NB - (4 - LATE));
            if (part >= 0 && refill) {
              TileA::template issue_part<IA / PARTS>(part, ga, offa, lds0 + st * STAGE, wave);
              TileB::template issue_part<IB / PARTS>(part, gb, offb, lds0 + st * STAGE + A_BYTES, wave);
            }
          } else if (slot < LATE && kt > 0 && dma_wave) {
            const int part = 4 - LATE + slot;
            TileA::template issue_part<IA / PARTS>(part, ga_late, offa, lds0 + st_late * STAGE, wave);
            TileB::template issue_part<IB / PARTS>(part, gb_late, offb,
                                                   lds0 + st_late * STAGE + A_BYTES, wave);
          }
        }
        if (KG > 1 && !live) continue;
        // a walk over the 2 x TN tiles of this pair of rows, the next pair taking the columns in
        // the opposite direction
#pragma unroll
        for (int q = 0; q < TN / 2; ++q) {
          const int jb = ib & 1 ? TN / 2 - 1 - q : q;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // (row, column) within the 2 x 2 group: 00 01 11 10, the next group 10 11 01 00
            const int ii = (q & 1) ? (e < 2 ? 1 : 0) : (e < 2 ? 0 : 1);
            const int jj = (e == 1 || e == 2) ? 1 : 0;
            const int i = 2 * ib + ii, j = 2 * jb + ((ib & 1) ? 1 - jj : jj);
            acc[part * TMH + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                fw[curw][j], fx[cur][i], acc[part * TMH + i][j], 0, 0, 0);
          }
        }
      }
    }
    if constexpr (EPI == JPP_EPI_ACC_F32) {
      if (stream_c && kt < NBT)
        dma_load16(uniform_ptr((const bf16_t*)p.c), c_off0 + (uint32_t)(kt * NW * p.ldc * 4),
                   lds0 + C_LDS + (cbi * NW + wave) * C_PITCH);
    }
    ga_late = ga; gb_late = gb; st_late = st;
    st = nst;
    cbi = cbi + 1 == NS + 1 ? 0 : cbi + 1;
  }
  dma_wait_all();

  // the groups' sums, in group order: wave w of every group holds the same elements, so they
  // change hands through LDS lane by lane, 16 bytes at a time
  if constexpr (KG > 1) {
    __syncthreads();
    uint8_t* const mine = smem + ((grp - 1) * NW + wave) * (TM * TN * 1024) + lane * 16;
    if (grp > 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) *(f32x4*)(mine + (i * TN + j) * 1024) = acc[i][j];
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
      for (int g = 1; g < KG; ++g)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] += *(const f32x4*)(mine + (g * NW * TM * TN + i * TN + j) * 1024);
    }
  }
  // tile rows that pass through LDS at a time in the epilogues below: of a tile shared by
  // several wave groups (a small one) all
  constexpr bool WHOLE = KG > 1;

  if constexpr (EPI == JPP_EPI_ACC_F32 || EPI == JPP_EPI_F32) {
    // fp32 outputs leave through LDS as well (see below), a quarter of the tile per pass:
    // 16-byte stores of contiguous rows instead of 32-byte pieces of 32 rows
    constexpr int IPP = WHOLE ? TM : TM / 2, RP = WHOLE ? BM : IPP * 16, PITCH = BN * 4 + 16,
                  NT = NW * KG * 64, PASSES = WHOLE ? 1 : 2 * (TM / IPP);
    constexpr int TPR = BN / 4, RPI = NT / TPR, PER = RP / RPI;
    static_assert(RP % RPI == 0, "rows of a pass split evenly over the threads");
    const int c4 = (tid % TPR) * 4;
    auto row_of = [&](int pass, int it) {
      return m0 + (pass / (TM / IPP)) * (BM / 2) + (pass % (TM / IPP)) * IPP * 16 + tid / TPR + it * RPI;
    };
    // Old values that did not stream in are read here, by rows and past the caches: a small tile's
    // all at once, a large one's (out of registers for that) a pass ahead, the next pass's while this
    // one's leave.  Through the caches, and each pass's behind the one before it, a layer's four gradients
    // of hidden 2048 and gated feed-forward 5632 on 512 tokens took 112 us as 256x256 tiles, now 95.5 as 128x128, again and
    // again by themselves; among the row's other kernels, under a profiler, 108 and 100 - 103.  Their accumulators' 361 MB
    // alone are 66 us at 5.5 TB/s: the old values are asked for behind the contraction.
    const bool add_here = EPI == JPP_EPI_ACC_F32 && !stream_c;
    constexpr int BUFS = PASSES * PER <= 8 ? PASSES : 1;
    f32x4 old[BUFS][PER];
    auto fetch = [&](int pass) {
#pragma unroll
      for (int it = 0; it < PER; ++it)
        old[pass % BUFS][it] =
            __builtin_nontemporal_load((const f32x4*)((const float*)p.c + row_of(pass, it) * p.ldc + n0 + c4));
    };
    if (add_here) {
#pragma unroll
      for (int pass = 0; pass < BUFS; ++pass) fetch(pass);
    }
#pragma unroll(BUFS)
    for (int pass = 0; pass < PASSES; ++pass) {
      const int half = pass / (TM / IPP), i0 = (pass % (TM / IPP)) * IPP;
      __syncthreads();
      if (WHOLE ? grp == 0 : wm == half) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          if (i >= i0 && i < i0 + IPP) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
              *(f32x4*)(smem + ((WHOLE ? row_x : 0) + (i - i0) * 16 + (lane & 15)) * PITCH +
                        (wn * (BN / WN) + j * 16 + (lane >> 4) * 4) * 4) = acc[i][j];
          }
      }
      __syncthreads();
      f32x4 v[PER];
#pragma unroll
      for (int it = 0; it < PER; ++it) v[it] = *(const f32x4*)(smem + (tid / TPR + it * RPI) * PITCH + c4 * 4);
      if (add_here) {
#pragma unroll
        for (int it = 0; it < PER; ++it) v[it] = old[pass % BUFS][it] + v[it];
        if (BUFS == 1 && pass + 1 < PASSES) fetch(pass + 1);
      }
#pragma unroll
      for (int it = 0; it < PER; ++it) {
        float* dst = (float*)p.c + row_of(pass, it) * p.ldc + n0 + c4;
        // the accumulators are not read again before the next microbatch: stored past the
        // caches they leave L2 to the operand panels (+0.4 % on the Llama-8B-shaped stage)
        if (EPI == JPP_EPI_ACC_F32) __builtin_nontemporal_store(v[it], (f32x4*)dst);
        else *(f32x4*)dst = v[it];
      }
    }
  } else {
    // bf16 outputs.  An accumulator lane holds one row and 4 consecutive columns, so storing
    // from that layout scatters 8-byte pieces over 32 rows per instruction.  Instead the tile
    // goes through LDS (free after the K loop) half at a time - fp32, [BM/2 rows][BN + 4]
    // - and is taken back out by rows: a thread owns 8 consecutive columns of a row, so
    // every global access of the epilogue (output, residual, pre-activation, gate/up) is a
    // 16-byte piece of a contiguous run, and the arithmetic runs in fp32 exactly as before.
    constexpr int HALF = WHOLE ? BM : BM / 2, PITCH = BN * 4 + 16, NT = NW * KG * 64;
    const bf16_t* bias = p.bias;
#pragma unroll 1
    for (int half = 0; half < BM / HALF; ++half) {
      __syncthreads();  // fragments of the last K-step / the previous half are out of LDS
      if (WHOLE ? grp == 0 : wm == half) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            *(f32x4*)(smem + ((WHOLE ? row_x : 0) + i * 16 + (lane & 15)) * PITCH +
                      (wn * (BN / WN) + j * 16 + (lane >> 4) * 4) * 4) = acc[i][j];
      }
      __syncthreads();
      const long mrow0 = m0 + half * HALF;
      if constexpr (EPI == JPP_EPI_SWIGLU) {
        // a thread owns 8 features of a row: gate at columns 64q + w, up at 64q + 32 + w
        constexpr int TPR = BN / 16, RPI = NT / TPR;  // threads per row, rows per sweep
        const int fc = tid % TPR, q = fc >> 2, w = (fc & 3) * 8;
        for (int r = tid / TPR; r < HALF; r += RPI) {
          const uint8_t* row = smem + r * PITCH + (q * 64 + w) * 4;
          const float4 g0 = *(const float4*)row, g1 = *(const float4*)(row + 16);
          const float4 u0 = *(const float4*)(row + 128), u1 = *(const float4*)(row + 144);
          const uint4 gp = make_uint4(pack_bf16x2(g0.x, g0.y), pack_bf16x2(g0.z, g0.w),
                                      pack_bf16x2(g1.x, g1.y), pack_bf16x2(g1.z, g1.w));
          const uint4 up = make_uint4(pack_bf16x2(u0.x, u0.y), pack_bf16x2(u0.z, u0.w),
                                      pack_bf16x2(u1.x, u1.y), pack_bf16x2(u1.z, u1.w));
          bf16_t* crow = (bf16_t*)p.c + (mrow0 + r) * p.ldc + n0 + q * 64 + w;
          // gate and up are next read by the backward pass, many tasks later: stored past the
          // caches (their product below is the next GEMM's operand and stays cached)
          __builtin_nontemporal_store(u32x4{gp.x, gp.y, gp.z, gp.w}, (u32x4*)crow);
          __builtin_nontemporal_store(u32x4{up.x, up.y, up.z, up.w}, (u32x4*)(crow + 32));
          // from the rounded values, as a separate kernel would read them back
          float gv[8], uv[8];
          unpack8(gp, gv);
          unpack8(up, uv);
#pragma unroll
          for (int e = 0; e < 8; ++e) gv[e] = swiglu_f(gv[e], uv[e]);
          *(uint4*)((bf16_t*)p.c2 + (mrow0 + r) * p.ldc2 + n0 / 2 + q * 32 + w) = pack8(gv);
        }
      } else if constexpr (EPI == JPP_EPI_DSWIGLU) {
        // the tile holds ds for BN features; gate / up of block q at columns 64q.., 64q+32..
        constexpr int TPR = BN / 8, RPI = NT / TPR;
        const int fc = tid % TPR, q = fc >> 2, w = (fc & 3) * 8;
        for (int r = tid / TPR; r < HALF; r += RPI) {
          const uint8_t* row = smem + r * PITCH + fc * 32;
          const float4 d0 = *(const float4*)row, d1 = *(const float4*)(row + 16);
          const long col = 2 * n0 + q * 64 + w;
          const bf16_t* arow = p.aux + (mrow0 + r) * p.ldaux + col;
          float gv[8], uv[8], dv[8];
          unpack8(*(const uint4*)arow, gv);
          unpack8(*(const uint4*)(arow + 32), uv);
          unpack8(make_uint4(pack_bf16x2(d0.x, d0.y), pack_bf16x2(d0.z, d0.w),
                             pack_bf16x2(d1.x, d1.y), pack_bf16x2(d1.z, d1.w)), dv);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            float dg, du;
            swiglu_grad_f(gv[e], uv[e], dv[e], dg, du);
            gv[e] = dg;
            uv[e] = du;
          }
          bf16_t* crow = (bf16_t*)p.c + (mrow0 + r) * p.ldc + col;
          *(uint4*)crow = pack8(gv);
          *(uint4*)(crow + 32) = pack8(uv);
        }
      } else {
        constexpr int TPR = BN / 8, RPI = NT / TPR;
        const int c8 = (tid % TPR) * 8;
        float bv[8];
        if (bias) unpack8(*(const uint4*)(bias + n0 + c8), bv);
        for (int r = tid / TPR; r < HALF; r += RPI) {
          const uint8_t* row = smem + r * PITCH + c8 * 4;
          const float4 a0 = *(const float4*)row, a1 = *(const float4*)(row + 16);
          float v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
          const long at = (mrow0 + r) * p.ldc + n0 + c8;
          if (bias) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += bv[e];
          }
          if constexpr (EPI == JPP_EPI_BF16) {
            if (p.resid) {
              float rv[8];
              unpack8(*(const uint4*)(p.resid + (mrow0 + r) * p.ldresid + n0 + c8), rv);
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] += rv[e];
            }
            if constexpr (!TA && TB) {
              // rotary embedding of the query / key heads (forward projection): the partner
              // of a column sits half a head away in the same staged row; both are rounded to
              // bf16 first, as a pass of its own would read them back
              if (p.rope_cos && n0 + c8 < p.rope_cols) {
                const int hh = p.rope_hd >> 1, cin = (n0 + c8) & (p.rope_hd - 1);
                const bool lo = cin < hh;
                const uint8_t* prow = row + (lo ? hh : -hh) * 4;
                const float4 b0 = *(const float4*)prow, b1 = *(const float4*)(prow + 16);
                const float w[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
                const long pos = (p.rope_row0 + mrow0 + r) % p.rope_seq;
                const float* ct = p.rope_cos + pos * hh + (cin & (hh - 1));
                const float* st = p.rope_sin + pos * hh + (cin & (hh - 1));
                const float4 c0 = *(const float4*)ct, c1 = *(const float4*)(ct + 4);
                const float4 s0 = *(const float4*)st, s1 = *(const float4*)(st + 4);
                const float cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
                const float sn[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                  const float own = (float)(__bf16)v[e], other = (float)(__bf16)w[e];
                  float o1, o2;
                  rope_rotate(lo ? own : other, lo ? other : own, cs[e], sn[e], o1, o2);
                  v[e] = lo ? o1 : o2;
                }
              }
            }
          } else if constexpr (EPI == JPP_EPI_GELU) {
            float gl[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) gl[e] = gelu_f(v[e], p.gelu_tanh);
            *(uint4*)((bf16_t*)p.c2 + (mrow0 + r) * p.ldc2 + n0 + c8) = pack8(gl);
          } else if constexpr (EPI == JPP_EPI_DGELU) {
            float uv[8];
            unpack8(*(const uint4*)(p.aux + (mrow0 + r) * p.ldaux + n0 + c8), uv);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] *= gelu_grad_f(uv[e], p.gelu_tanh);
          }
          *(uint4*)((bf16_t*)p.c + at) = pack8(v);
        }
      }
    }
  }
}

#undef a_at
#undef b_at

template <int BM, int BN, bool TA, bool TB, int EPI, int NW, int NS, int KG = 1>
const char* class_name() {
  // built once per instantiation; the initialisation of a function-local static is
  // thread-safe
  static const std::string name = [] {
    char buf[64];
    const char* lay = TA ? "tn" : (TB ? "nn" : "nt");
    const char* epi = EPI == JPP_EPI_BF16 ? "bf16" : EPI == JPP_EPI_GELU ? "gelu"
                    : EPI == JPP_EPI_DGELU ? "dgelu" : EPI == JPP_EPI_ACC_F32 ? "accf32"
                    : EPI == JPP_EPI_SWIGLU ? "swiglu" : EPI == JPP_EPI_DSWIGLU ? "dswiglu" : "f32";
    snprintf(buf, sizeof(buf), "gemm_%s_%s_%dx%d%s%s%s", lay, epi, BM, BN, NW == 8 ? "w8" : "",
             NS == 2 ? "" : NS == 3 ? "s3" : NS == 4 ? "s4" : "s5", KG == 1 ? "" : "k2");
    return std::string(buf);
  }();
  return name.c_str();
}

template <int BM, int BN, bool TA, bool TB, int EPI, int NW = 4, int NS = 2, bool KP = false, int KG = 1>
int launch(hipStream_t stream, GemmParams& p) {
  // two operand stages; the bf16 epilogues stage half a tile in fp32 with padded rows
  constexpr int SMEM_LOOP = KG * NS * (BM + BN) * 128,
                SMEM_EPI = (KG > 1 ? BM : BM / 2) * (BN * 4 + 16);
  // + NS+1 buffers of NW rows of the fp32 tile (padded) for C += A B
  constexpr int SMEM = EPI == JPP_EPI_ACC_F32 && streams_accumulator(BM, BN) ? SMEM_LOOP + (NS + 1) * NW * (1024 + 16)
                       : (EPI == JPP_EPI_F32 || SMEM_LOOP > SMEM_EPI) ? SMEM_LOOP : SMEM_EPI;
  if constexpr (!KP) {
    // several operand pairs: only the accumulating weight-gradient kernels are built for that
    if (p.k_parts > 1) {
      if constexpr (TA && TB && EPI == JPP_EPI_ACC_F32 && !(BM == 256 && BN == 128))
        return launch<BM, BN, TA, TB, EPI, NW, NS, true, KG>(stream, p);
      else
        return jpp_set_error(JPP_ERR_INVALID, "gemm: several operand pairs are supported for "
                             "accumulated weight gradients (tn, JPP_EPI_ACC_F32), not on 256x128 "
                             "tiles");
    }
  }
  // algorithmic extent: grouped launches count the non-padding rows when the caller gave them
  const double cb = EPI == JPP_EPI_ACC_F32 || EPI == JPP_EPI_DSWIGLU ? 8
                    : EPI == JPP_EPI_F32 ? 4 : EPI == JPP_EPI_SWIGLU ? 3 : 2;
  double am = p.m, ak = (double)p.k * (p.k_parts > 1 ? p.k_parts : 1), copies = 1;
  if (p.group_mode == JPP_GROUP_M && p.group_rows) am = p.group_rows;
  if (p.group_mode == JPP_GROUP_K) { ak = p.group_rows; copies = p.n_seg; }
  const double b_bytes = 2.0 * p.n * ak * (p.group_mode == JPP_GROUP_M ? p.n_seg : 1);
  // (the small-tile launches of a row-grouped product's last round add their time to the class
  // of its 256x256 launch, which declares the whole product's work)
  const bool tail = p.tail_split >= 2;
  ProbeScope probe(stream, tail ? class_name<256, 256, TA, TB, EPI, 8, 2>()
                                : class_name<BM, BN, TA, TB, EPI, NW, NS, KG>(),
                   tail ? 0.0 : 2.0 * am * p.n * ak,
                   tail ? 0.0 : 2.0 * am * ak + b_bytes + copies * am * p.n * cb);
  auto kern = gemm_kernel<BM, BN, TA, TB, EPI, NW, NS, KP, false, KG>;
  static_assert(SMEM <= 160 * 1024, "LDS of one CU");
  // the LDS limit of a kernel is sticky: set once per instantiation, by whichever host
  // thread launches it first (the others wait for that call and see its result)
  static std::once_flag configured;
  static hipError_t configure_rc = hipSuccess;
  std::call_once(configured, [&] {
    configure_rc = hipFuncSetAttribute((const void*)kern,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
  });
  JPP_CHECK_HIP(configure_rc);
  p.tiles_m = p.m / BM;
  p.tiles_n = p.n / BN;
  const int blocks = p.tiles_m * p.tiles_n * (p.group_mode == JPP_GROUP_K ? p.n_seg : 1);
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(NW * KG * 64), SMEM, stream, GemmArgs<false>{p});
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

// Several accumulated weight gradients (C_i += sum_j A_ij^T B_ij) as one grid of BM x BN
// tiles: problem i's tiles follow problem i-1's, so the half-filled last rounds of the single
// launches (384 or 896 tiles on 256 CUs) close up - the four weight gradients of a
// Llama-3-8B-shaped layer are 13 full rounds together - and small ones share the device.
template <int BM, int BN, int NW, int NS, int KG = 1>
int launch_multi(hipStream_t stream, GemmParams* ps, int n, const ColsumPanels& cols, int col_blocks, long col_rows) {
  constexpr int SMEM = KG * NS * (BM + BN) * 128 + (streams_accumulator(BM, BN) ? (NS + 1) * NW * (1024 + 16) : 0);
  static_assert(SMEM <= 160 * 1024, "LDS of one CU");
  GemmArgs<true> args;
  args.p = ps[0];
  int first = 0;
  double flops = 0, bytes = 0;
  for (int i = 0; i < n; ++i) {
    GemmParams& p = ps[i];
    p.tiles_m = p.m / BM;
    p.tiles_n = p.n / BN;
    const double ak = (double)p.k * p.k_parts;
    flops += 2.0 * p.m * p.n * ak;
    bytes += 2.0 * ak * (p.m + p.n) + 8.0 * p.m * p.n;
    if (i > 0) {
      GemmProblem& q = args.more[i - 1];
      q.a[0] = p.a; q.b[0] = p.b;
      for (int j = 0; j < 3; ++j) { q.a[j + 1] = p.a_more[j]; q.b[j + 1] = p.b_more[j]; }
      q.c = p.c; q.lda = p.lda; q.ldb = p.ldb; q.ldc = p.ldc;
      q.tiles_m = p.tiles_m; q.tiles_n = p.tiles_n; q.first = first;
    }
    first += p.tiles_m * p.tiles_n;
  }
  args.p.tiles_m = ps[0].tiles_m;
  args.p.tiles_n = ps[0].tiles_n;
  for (int i = n; i < 4; ++i) {
    memset(&args.more[i - 1], 0, sizeof(GemmProblem));
    args.more[i - 1].first = 0x7fffffff;
  }
  args.cols = cols;
  args.col_first = first;
  args.col_rows = col_rows;
  if (col_blocks)   // (the sums that go along count here, not in a class of their own)
    for (int i = 0; i < 4; ++i)
      if (cols.first[i] < col_blocks) bytes += 2.0 * col_rows * cols.cols[i];
  static const std::string cls =
      std::string(class_name<BM, BN, true, true, JPP_EPI_ACC_F32, NW, NS, KG>()) + "_multi";
  ProbeScope probe(stream, cls.c_str(), flops, bytes);
  auto kern = gemm_kernel<BM, BN, true, true, JPP_EPI_ACC_F32, NW, NS, true, true, KG>;
  static std::once_flag configured;
  static hipError_t configure_rc = hipSuccess;
  std::call_once(configured, [&] {
    configure_rc = hipFuncSetAttribute((const void*)kern,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
  });
  JPP_CHECK_HIP(configure_rc);
  hipLaunchKernelGGL(kern, dim3(first + col_blocks), dim3(NW * KG * 64), SMEM, stream, args);
  JPP_LAUNCH_CHECK();
  return JPP_OK;
}

// The 128x128 tile runs with five LDS stages (one workgroup per CU) when every CU has at most
// one tile, else with two (two workgroups per CU); the 64x64 tile, whose two wave groups share
// it, with four or two by the same rule - and if the contraction is long enough for the longer
// prologue.  Time of the deep form over that of two stages, 96 to 256 tiles, operands out of L2 as
// a layer finds them: 128x128 1.03 - 1.11 at 1 - 3 K-steps, 1.03 at 4, 0.96 at 6, 0.8 at 16;
// 64x64 1.05 at 1 - 4, 1.02 at 6, 0.99 at 8, 0.91 at 12, 0.84 at 20.
bool deep_stages(long tiles, long ksteps, int tile) {
  return tiles <= kCus && ksteps > (tile == kTile128 ? 4 : 8);
}

struct Extent { long m, n; };

// What the choice of a tile and of its form go by: the extent of the grid (of a grouped contraction
// an output per group), the part of it that holds data (of grouped rows, if the caller counted
// them) and the K-steps (of a grouped contraction the groups' average, 0 if not counted).
// The form follows the grid also where grouped rows fill only a part of it: consecutive tiles
// belong to one XCD, so the workgroups that find work lie on the first ones, more than one
// per CU there (top-2 of 8 experts, hidden 512, on 512 tokens: the row 5 % slower with the form
// by the rows that hold data).
Extent grid_extent(const jpp_gemm_args* a) {
  return {a->group_mode == JPP_GROUP_K ? a->m * a->n_seg : a->m, a->n};
}
Extent work_extent(const jpp_gemm_args* a) {
  Extent e = grid_extent(a);
  if (a->group_mode == JPP_GROUP_M && a->group_rows)   // half of a segment's last 256 rows are padding on average
    e.m = std::min<long>(e.m, (a->group_rows + 128L * a->n_seg + 255) / 256 * 256);
  return e;
}
long work_ksteps(const jpp_gemm_args* a) {
  if (a->group_mode == JPP_GROUP_K) return a->group_rows ? a->group_rows / (64L * a->n_seg) + 1 : 0;
  return a->k / 64 * (a->k_parts > 1 ? a->k_parts : 1);
}
// tiles of bm x bn in all of the extents, -1 if one does not divide into them
long count_tiles(const Extent* e, int n, int bm, int bn) {
  long tiles = 0;
  for (int i = 0; i < n; ++i) {
    if (e[i].m % bm || e[i].n % bn) return -1;
    tiles += (e[i].m / bm) * (e[i].n / bn);
  }
  return tiles;
}
bool deep_form(const jpp_gemm_args* a, int tile) {
  const Extent e = grid_extent(a);
  const int b = tile == kTile64 ? 64 : 128;
  return deep_stages(count_tiles(&e, 1, b, b), work_ksteps(a), tile);
}

// `deep`: which form of the 64x64 and 128x128 tiles
template <bool TA, bool TB, int EPI>
int launch_tiled(hipStream_t stream, GemmParams& p, int tile, bool deep) {
  switch (tile) {
    case kTile256x128:  // 8 waves of 128x32; three stages where the accumulator rows leave room
      return launch<256, 128, TA, TB, EPI, 8, EPI == JPP_EPI_ACC_F32 ? 2 : 3>(stream, p);
    case kTile128x256:  // 8 waves of 64x64
      return launch<128, 256, TA, TB, EPI, 8, EPI == JPP_EPI_ACC_F32 ? 2 : 3>(stream, p);
    case kTile256: return launch<256, 256, TA, TB, EPI, 8>(stream, p);
    case kTile64x128:
      // the 64x64 form for products that rotate heads of 128: the same sums in the same order
      // (two wave groups), so the rotated product is the plain one's bits rotated
      if constexpr (!TA && TB && EPI == JPP_EPI_BF16)
        return launch<64, 128, TA, TB, EPI, 4, 3, false, 2>(stream, p);
      else
        return jpp_set_error(JPP_ERR_INVALID, "gemm: unknown tile %d", tile);
    case kTile64:  // two groups of 4 waves (32x32 each) that take the K-steps in turn
      return deep ? launch<64, 64, TA, TB, EPI, 4, 4, false, 2>(stream, p)
                  : launch<64, 64, TA, TB, EPI, 4, 2, false, 2>(stream, p);
    default:  // 128x128: 8 waves (64x32 each)
      return deep ? launch<128, 128, TA, TB, EPI, 8, 5>(stream, p)
                  : launch<128, 128, TA, TB, EPI, 8, 2>(stream, p);
  }
}

// Expected time of a product of `tiles` tiles, `ksteps` K-steps of 64 each, in us, with w = tiles of the
// busiest of the 256 CUs and s = tiles / 256 (`gelu`: the arithmetic of a GELU epilogue):
//   w = 1:  start + tile_cost + gelu + s * share + ksteps * lone_step
//   w > 1:  start + w * (tile_cost + gelu) + s * share + ksteps * (w * step + s * share_step)
// (two workgroups of a two-stage form fit on a CU, their steps overlap; `share`: what the tiles wait for
// together, the fp32 tile that a weight gradient's workgroup reads, adds to and writes).  The constants are
// least-squares fits to random products in every form, with the operands out of L2, as a layer finds
// them, and accumulators out of every cache.
// Forward: 969 products (M, N 128 .. 16384, K 128 .. 16384, every orientation and epilogue), mean error 4
// - 10 %; the smallest estimate costs 0.1 % against the measured best.  128x256 stands 10 % above its
// fit: 128x128 is otherwise passed over where they are close.  Against the rule before (256x256 from 192
// tiles on, else 128x128: 36 % on average) it is slower by more than 2 % for 9 of the 969, all but one by
// 6 % at most (180 tiles of 256x256, 3 K-steps: 14 %): a 512 x 1024 x 4096 input gradient has 32 tiles of
// 128x128 for 256 CUs and took 28 us, 15 us as 128 tiles of 64x64 with two wave groups each.
// 200 weight gradients that are not added to anything (written as bf16 or f32) are priced alike: 0.1 % over the measured
// best, 10 % at worst; as accumulated ones 0.5 % and 22 % (2304 x 768 x 256: 7.0 us, 6.0 as 64x64).
// Accumulated weight gradients: 420 launches of 1 to 4 products (outputs 128 .. 8192 a side, 64 .. 8192 tokens), mean
// error 2 - 11 %; the smallest estimate costs 0.3 % against the measured best.  256x256 from 192 tiles on
// cost 9 % there and 36 % at worst (300 tiles, 2 K-steps: 44 us, 33 as 128x128; 1176 tiles, 4: 135 and 121): a
// 256x256 tile, alone on its CU, waits for its fp32 tile apart from its K-steps, of two 128x128 tiles one's
// wait falls on the other's steps.
struct TileForm {
  int tile, bm, bn;
  bool deep;              // which of the tile's two forms (kTile128, kTile64)
  float start, tile_cost, gelu, lone_step, step, share, share_step;
};
constexpr TileForm kForward[] = {
    {kTile64, 64, 64, true, 0.f, 4.8f, 0.5f, 0.18f, 0.18f, 0.f, 0.f},     {kTile64, 64, 64, false, 2.7f, 1.5f, 0.3f, 0.26f, 0.17f, 0.f, 0.f},
    {kTile128, 128, 128, true, 0.f, 6.3f, 2.1f, 0.39f, 0.39f, 0.f, 0.f},  {kTile128, 128, 128, false, 3.4f, 2.3f, 1.7f, 0.49f, 0.365f, 0.f, 0.f},
    {kTile128x256, 128, 256, true, 1.1f, 7.4f, 5.2f, 0.705f, 0.715f, 0.f, 0.f},
    {kTile256, 256, 256, true, 0.2f, 10.2f, 10.f, 1.05f, 1.08f, 0.f, 0.f}};
constexpr TileForm kWeightGrad[] = {
    {kTile64, 64, 64, true, 0.f, 3.8f, 0.f, 0.24f, 0.24f, 3.9f, 0.f},    {kTile64, 64, 64, false, 4.3f, 0.f, 0.f, 0.22f, 0.21f, 2.f, 0.f},
    {kTile128, 128, 128, true, 0.f, 5.7f, 0.f, 0.485f, 0.485f, 6.4f, 0.f},
    {kTile128, 128, 128, false, 5.1f, 0.45f, 0.f, 0.43f, 0.39f, 4.3f, 0.115f},
    {kTile128x256, 128, 256, true, 3.f, 4.4f, 0.f, 0.9f, 0.83f, 7.8f, 0.08f},
    {kTile256, 256, 256, true, 5.6f, 6.3f, 0.f, 1.28f, 1.08f, 16.f, 0.53f}};

// tile with the smallest estimate for products of these extents in one grid (`grid`: the extents
// that its form goes by)
int cheapest_tile(const Extent* e, const Extent* grid, int n, long ksteps, bool wgrad /* accumulated */, bool gelu,
                  bool may_128x256) {
  int best = kTile128;
  float best_us = 0.f;
  for (const TileForm& f : wgrad ? kWeightGrad : kForward) {
    if (f.tile == kTile128x256 && !may_128x256) continue;
    const long tiles = count_tiles(e, n, f.bm, f.bn);
    if (tiles < 0) continue;
    if ((f.tile == kTile64 || f.tile == kTile128) &&
        f.deep != deep_stages(count_tiles(grid, n, f.bm, f.bn), ksteps, f.tile)) continue;
    const long w = (tiles + kCus - 1) / kCus;
    const float share = (float)tiles / kCus;
    const float t = f.start + w * (f.tile_cost + (gelu ? f.gelu : 0.f)) + share * f.share +
                    ksteps * (w == 1 ? f.lone_step : w * f.step + share * f.share_step);
    if (best_us == 0.f || t < best_us) { best_us = t; best = f.tile; }
  }
  return best;
}

// The 256x256 tile run by 8 waves (two per SIMD, so one wave's LDS reads hide under the other's
// MFMAs) is the fastest whenever it gives most CUs a tile; smaller problems go by the estimate, and
// accumulated weight gradients all do.
int choose_tile(const jpp_gemm_args* a) {
  const Extent e = work_extent(a);
  if (a->group_mode != JPP_GROUP_NONE && !a->group_rows) return kTile256;
  const long t256 = e.m % 256 == 0 && e.n % 256 == 0 ? (e.m / 256) * (e.n / 256) : 0;
  const bool wgrad = a->trans_a && a->trans_b && a->epilogue == JPP_EPI_ACC_F32;
  if (t256 >= kMostCus && !wgrad) return kTile256;
  const Extent grid = grid_extent(a);
  const bool gelu = a->epilogue == JPP_EPI_GELU || a->epilogue == JPP_EPI_DGELU;
  const int tile = cheapest_tile(&e, &grid, 1, work_ksteps(a), wgrad, gelu, true);
  // A rotated head of 128 lies inside one tile: 64x128 at the price of 64x64, which it does not keep (512 x 3072 x 2048
  // 16.6 us, 20 measured).  With the rotation the 128x128 tile does not keep its own either: where 64x128 is taken it
  // needs 0.73 - 0.90 of that one's time (93 of 120 random products of 128 .. 2048 rows; in the others they are equal).
  return tile == kTile64 && a->rope_cos && a->rope_head_dim > 64 ? (int)kTile64x128 : tile;
}

// Products that run on waves of their own (gemm_wave.hip), by the rows of their tiles (0: they do
// not).  32 while those tiles are at most one per CU: over 65 random shapes (M, N, K 128 .. 8192; both
// orientations, plain and GELU epilogues) they take 0.99 to 0.70 of the time of the best tile
// here, 0.8 in the median; above that line, two rounds of them, 1.01 to 1.45.  From there 64 while `tile`,
// the choice among the tiles here, is the 64x64 one and those are at most one per CU, and with a GELU from
// 9 K-steps on (gemm_wave.hip has the figures).  A plain forward product without bias and
// residual stays: its bits are those a product with the rotary epilogue rotates.
int rows_on_waves(const jpp_gemm_args* a, int tile) {
  const bool kind = a->epilogue == JPP_EPI_BF16 ? !a->trans_b || a->bias || a->resid
                                                : a->epilogue == (a->trans_b ? JPP_EPI_GELU : JPP_EPI_DGELU);
  if (!kind || a->tile || a->trans_a || a->group_mode != JPP_GROUP_NONE || a->k_parts > 1 || a->rope_cos) return 0;
  if ((a->m / 32) * (a->n / 64) <= kCus) return 32;
  return tile == kTile64 && (a->m / 64) * (a->n / 64) <= kCus && (a->epilogue == JPP_EPI_BF16 || a->k > 8 * 64) ? 64 : 0;
}

// sub-problem whose first row / column is (m_off, n_off) of the full one
void shift_origin(GemmParams& p, bool ta, bool tb, int epi, long m_off, long n_off) {
  p.a += ta ? m_off : m_off * p.lda;
  p.b += tb ? n_off : n_off * p.ldb;
  for (int i = 0; i + 1 < p.k_parts; ++i) {
    p.a_more[i] += ta ? m_off : m_off * p.lda;
    p.b_more[i] += tb ? n_off : n_off * p.ldb;
  }
  const long c_cols = epi == JPP_EPI_DSWIGLU ? 2 * n_off : n_off;  // dSwiGLU writes d gate, d up
  const bool f32 = epi == JPP_EPI_ACC_F32 || epi == JPP_EPI_F32;
  p.c = f32 ? (void*)((float*)p.c + m_off * p.ldc + c_cols)
            : (void*)((bf16_t*)p.c + m_off * p.ldc + c_cols);
  if (p.c2)  // SwiGLU: s has one column per gate/up pair; GELU: as wide as C
    p.c2 = (bf16_t*)p.c2 + m_off * p.ldc2 + (epi == JPP_EPI_SWIGLU ? n_off / 2 : n_off);
  if (p.bias) p.bias += n_off;
  if (p.rope_cos) {  // (n_off is a multiple of 256: whole heads)
    p.rope_row0 += m_off;
    p.rope_cols = (int)(p.rope_cols > n_off ? p.rope_cols - n_off : 0);
  }
  if (p.resid) p.resid += m_off * p.ldresid + n_off;
  if (p.aux) p.aux += m_off * p.ldaux + c_cols;
}

int dispatch(hipStream_t stream, const jpp_gemm_args* a, GemmParams& p, int tile, bool deep = false) {
  const int ta = a->trans_a != 0, tb = a->trans_b != 0, e = a->epilogue;
#define JPP_GEMM_CASE(TA_, TB_, E_) \
  if (ta == TA_ && tb == TB_ && e == E_) return launch_tiled<TA_, TB_, E_>(stream, p, tile, deep)
  JPP_GEMM_CASE(0, 1, JPP_EPI_BF16);     // forward
  JPP_GEMM_CASE(0, 1, JPP_EPI_GELU);     // forward + GELU
  JPP_GEMM_CASE(0, 1, JPP_EPI_F32);      // forward, f32 out (router logits)
  JPP_GEMM_CASE(0, 1, JPP_EPI_SWIGLU);   // gate/up projection + SwiGLU
  JPP_GEMM_CASE(0, 1, JPP_EPI_ACC_F32);  // weight gradient from a transposed activation
  JPP_GEMM_CASE(0, 0, JPP_EPI_BF16);     // input gradient
  JPP_GEMM_CASE(0, 0, JPP_EPI_DGELU);    // input gradient through GELU
  JPP_GEMM_CASE(0, 0, JPP_EPI_DSWIGLU);  // input gradient through SwiGLU
  JPP_GEMM_CASE(1, 1, JPP_EPI_ACC_F32);  // weight gradient, accumulated
  JPP_GEMM_CASE(1, 1, JPP_EPI_BF16);     // weight gradient, bf16
  JPP_GEMM_CASE(1, 1, JPP_EPI_F32);      // weight gradient, f32
#undef JPP_GEMM_CASE
  return jpp_set_error(JPP_ERR_INVALID, "gemm: unsupported combination trans_a=%d trans_b=%d epilogue=%d",
                       ta, tb, e);
}

// checks one problem's arguments and fills the kernel's view of it
int prepare(const jpp_gemm_args* a, GemmParams& p) {
  JPP_REQUIRE(a && a->a && a->b && a->c, "gemm: null operand");
  const bool group_k = a->group_mode == JPP_GROUP_K;
  JPP_REQUIRE(a->m > 0 && a->n > 0 && (a->k > 0 || group_k), "gemm: empty problem %ldx%ldx%ld",
              (long)a->m, (long)a->n, (long)a->k);
  JPP_REQUIRE(a->m % 128 == 0 && a->n % 128 == 0 && (a->k % 64 == 0 || group_k),
              "gemm: M,N must be multiples of 128 and K of 64, got %ldx%ldx%ld", (long)a->m,
              (long)a->n, (long)a->k);
  JPP_REQUIRE(a->lda >= (a->trans_a ? a->m : (group_k ? 0 : a->k)) &&
                  a->ldb >= (a->trans_b ? a->n : (group_k ? 0 : a->k)) &&
                  a->ldc >= a->n,
              "gemm: leading dimension too small");
  JPP_REQUIRE(a->lda % 8 == 0 && a->ldb % 8 == 0 && a->ldc % 4 == 0,
              "gemm: leading dimensions must keep 16-byte alignment");
  JPP_REQUIRE(((uintptr_t)a->a | (uintptr_t)a->b | (uintptr_t)a->c) % 16 == 0,
              "gemm: operands must be 16-byte aligned");
  JPP_REQUIRE(a->m < (1L << 31) && a->n < (1L << 31) && a->k < (1L << 31), "gemm: too large");
  p.a = (const bf16_t*)a->a;
  p.b = (const bf16_t*)a->b;
  p.c = a->c;
  p.c2 = a->c2;
  p.bias = (const bf16_t*)a->bias;
  p.resid = (const bf16_t*)a->resid;
  p.aux = (const bf16_t*)a->aux;
  p.m = (int)a->m; p.n = (int)a->n; p.k = (int)a->k;
  p.lda = a->lda; p.ldb = a->ldb; p.ldc = a->ldc;
  p.ldc2 = a->ldc2; p.ldresid = a->ldresid; p.ldaux = a->ldaux;
  p.gelu_tanh = a->gelu_tanh;
  p.seg = a->seg; p.seg_rows = a->seg_rows; p.n_seg = a->n_seg; p.group_mode = a->group_mode;
  p.group_rows = a->group_rows;
  p.tail_split = 0;
  p.stride_b = a->stride_b; p.stride_c = a->stride_c;
  p.k_parts = a->k_parts > 1 ? a->k_parts : 1;
  p.kt_part = (int)(a->k / 64);
  for (int i = 0; i < 3; ++i) {
    p.a_more[i] = (const bf16_t*)a->a_more[i];
    p.b_more[i] = (const bf16_t*)a->b_more[i];
    p.seg_more[i] = a->seg_more[i];
    p.seg_rows_more[i] = a->seg_rows_more[i];
  }
  p.rope_cos = a->rope_cos; p.rope_sin = a->rope_sin;
  p.rope_cols = (int)a->rope_cols; p.rope_seq = a->rope_seq; p.rope_hd = a->rope_head_dim;
  p.rope_row0 = 0;
  if (a->rope_cos || a->rope_sin) {
    JPP_REQUIRE(a->rope_cos && a->rope_sin, "gemm: rope_cos and rope_sin go together");
    JPP_REQUIRE(a->epilogue == JPP_EPI_BF16 && !a->trans_a && a->trans_b && !a->bias &&
                    !a->resid && a->group_mode == JPP_GROUP_NONE,
                "gemm: the rotary epilogue goes with JPP_EPI_BF16, trans_a = 0, trans_b = 1 and "
                "no bias, residual or groups");
    JPP_REQUIRE((a->rope_head_dim == 64 || a->rope_head_dim == 128) && a->rope_seq > 0 &&
                    a->rope_cols >= 0 && a->rope_cols <= a->n &&
                    a->rope_cols % a->rope_head_dim == 0,
                "gemm: rotary epilogue: heads of 64 or 128 elements, rope_cols a multiple of the "
                "head size and at most N, rope_seq positive");
    JPP_REQUIRE(((uintptr_t)a->rope_cos | (uintptr_t)a->rope_sin) % 16 == 0,
                "gemm: rotary tables must be 16-byte aligned");
  }
  if (a->k_parts > 1) {
    JPP_REQUIRE(a->k_parts <= 4 && a->group_mode != JPP_GROUP_M,
                "gemm: at most 4 operand pairs, and not with grouped rows (JPP_GROUP_M)");
    for (int i = 0; i + 1 < a->k_parts; ++i) {
      JPP_REQUIRE(a->a_more[i] && a->b_more[i] &&
                      ((uintptr_t)a->a_more[i] | (uintptr_t)a->b_more[i]) % 16 == 0,
                  "gemm: operand pair %d is null or not 16-byte aligned", i + 1);
      if (group_k)
        JPP_REQUIRE(a->seg_more[i] && !a->seg_rows_more[i] == !a->seg_rows,
                    "gemm: operand pair %d of a grouped contraction needs its row groups "
                    "(seg_more, and seg_rows_more when seg_rows is given)", i + 1);
    }
  }
  if (a->group_mode != JPP_GROUP_NONE) {
    JPP_REQUIRE(a->group_mode == JPP_GROUP_M || a->group_mode == JPP_GROUP_K,
                "gemm: unknown group_mode %d", a->group_mode);
    JPP_REQUIRE(a->seg && a->n_seg > 0 && a->n_seg <= 256, "gemm: grouped problem needs seg[n_seg+1]");
    JPP_REQUIRE((a->m % 256 == 0 && a->n % 256 == 0) || (a->group_mode == JPP_GROUP_K && a->tile),
                "gemm: grouped problems need M, N multiples of 256 (a grouped contraction with "
                "a tile of the caller's choice: of that tile)");
    JPP_REQUIRE(!a->bias && !a->resid, "gemm: grouped problems take no bias / residual");
  }
  if (a->epilogue == JPP_EPI_GELU)
    JPP_REQUIRE(a->c2 && a->ldc2 >= a->n && a->ldc2 % 4 == 0, "gemm: GELU epilogue needs c2");
  if (a->epilogue == JPP_EPI_DGELU)
    JPP_REQUIRE(a->aux && a->ldaux >= a->n && a->ldaux % 4 == 0, "gemm: dGELU epilogue needs aux");
  if (a->epilogue == JPP_EPI_SWIGLU)
    JPP_REQUIRE(a->c2 && a->ldc2 >= a->n / 2 && a->ldc2 % 4 == 0 && !a->bias && !a->resid &&
                    a->group_mode != JPP_GROUP_K,
                "gemm: SwiGLU epilogue needs c2 [M, N/2] and takes no bias / residual");
  if (a->epilogue == JPP_EPI_DSWIGLU)
    JPP_REQUIRE(a->aux && a->ldaux >= 2 * a->n && a->ldaux % 4 == 0 && a->ldc >= 2 * a->n &&
                    !a->bias && !a->resid && a->group_mode != JPP_GROUP_K,
                "gemm: dSwiGLU epilogue needs aux and C of width 2N and takes no bias / residual");
  if (a->epilogue == JPP_EPI_ACC_F32)
    JPP_REQUIRE((double)a->m * a->ldc * 4 < 4294967296.0,
                "gemm: an accumulated output must span less than 4 GiB (32-bit offsets)");
  if (a->resid) JPP_REQUIRE(a->ldresid >= a->n && a->ldresid % 4 == 0, "gemm: bad ldresid");
  return JPP_OK;
}

}  // namespace

extern "C" int jpp_gemm_bf16(void* stream_, const jpp_gemm_args* a) {
  hipStream_t stream = (hipStream_t)stream_;
  GemmParams p;
  if (int rc = prepare(a, p)) return rc;
  int tile = a->tile ? a->tile : choose_tile(a);
  if (const int rows = rows_on_waves(a, tile)) {
    const GemmWave d = {p.a, p.b, (bf16_t*)p.c, (bf16_t*)p.c2, p.bias, p.resid, p.aux, p.m, p.n, p.k,
                        p.lda, p.ldb, p.ldc, p.ldc2, p.ldresid, p.ldaux, p.gelu_tanh};
    ProbeScope probe(stream, a->trans_b ? "gemm_nn_wave" : "gemm_nt_wave", 2.0 * a->m * a->n * a->k,
                     2.0 * (a->m * a->k + a->n * a->k + a->m * a->n));
    return launch_gemm_wave(stream, d, a->trans_b != 0, a->epilogue, rows);
  }
  // several operand pairs of an ungrouped product: the 256-wide tiles whatever its size
  // (jpp_gemm_bf16_multi is the way to run small ones)
  if (a->k_parts > 1 && !a->tile && a->group_mode == JPP_GROUP_NONE) tile = kTile256;
  JPP_REQUIRE(a->tile >= 0 && a->tile <= 5, "gemm: unknown tile %d", a->tile);
  // (the rotary epilogue finds a column's partner in the staged row of its own tile)
  JPP_REQUIRE(a->tile != kTile64 || !a->rope_cos || a->rope_head_dim <= 64,
              "gemm: the rotary epilogue's heads of %d elements do not lie inside a 64x64 tile (tile 5)",
              a->rope_head_dim);
  if ((tile == kTile256x128 || tile == kTile256) && a->m % 256) tile = a->n % 256 ? kTile128 : kTile128x256;
  if ((tile == kTile128x256 || tile == kTile256) && a->n % 256) tile = a->m % 256 ? kTile128 : kTile256x128;
  // (256x128 is the one tile not built for several pairs)
  if (a->k_parts > 1 && !a->tile && tile == kTile256x128) tile = kTile128;

  // A grid of 256x256 tiles whose last round fills at most half of the 256 CUs runs that
  // round as a separate launch of 128x256 tiles over the last rows or columns: a full round
  // of half-size tiles takes little more than half the time the half-empty round did.
  // (Only when the choice of tile was left to the library.)
  if (tile == 4 && a->tile == 0 && a->group_mode == JPP_GROUP_NONE) {
    const long tm = a->m / 256, tn = a->n / 256, rest = (tm * tn) % 256;
    if (tm * tn > 256 && rest > 0 && rest <= 128) {
      const long rows = rest % tn == 0 ? rest / tn * 256 : 0;             // split along M
      const long cols = !rows && rest % tm == 0 ? rest / tm * 256 : 0;    // split along N
      if (rows || cols) {
        GemmParams head = p, tail = p;
        if (rows) {
          head.m = p.m - (int)rows;
          tail.m = (int)rows;
          shift_origin(tail, a->trans_a != 0, a->trans_b != 0, a->epilogue, head.m, 0);
        } else {
          head.n = p.n - (int)cols;
          tail.n = (int)cols;
          shift_origin(tail, a->trans_a != 0, a->trans_b != 0, a->epilogue, 0, head.n);
        }
        const int rc = dispatch(stream, a, head, 4);
        return rc != JPP_OK ? rc : dispatch(stream, a, tail, 3);
      }
    }
  }
  // Row groups: how many rows are in use is known on the device only, so the same split is
  // made there (group_head_rows) - the launches of small tiles are always enqueued and the
  // workgroups of those that find no rows of theirs leave at once.
  if (tile == 4 && a->tile == 0 && a->group_mode == JPP_GROUP_M && a->epilogue == JPP_EPI_BF16) {
    const long tm = a->m / 256, tn = a->n / 256;
    if (tm * tn > 256 && tn <= 128) {
      GemmParams head = p, small = p, wide = p;
      head.tail_split = 1;
      small.tail_split = 2;
      small.m = (int)std::min<long>(a->m, 64 / tn * 256);    // at most 64 tiles of 256x256
      wide.tail_split = 3;
      wide.m = (int)std::min<long>(a->m, 128 / tn * 256);    // at most 128
      int rc = dispatch(stream, a, head, 4);
      if (rc == JPP_OK && small.m > 0) rc = dispatch(stream, a, small, kTile128, true);  // (at most 256 tiles)
      return rc != JPP_OK ? rc : dispatch(stream, a, wide, 3);
    }
  }
  return dispatch(stream, a, p, tile, deep_form(a, tile));
}

extern "C" int jpp_gemm_bf16_multi(void* stream, const jpp_gemm_args* problems, int n_problems) {
  return jpp_wgrads_bf16((hipStream_t)stream, n_problems, problems, 0, nullptr, 0, nullptr);
}

int jpp_wgrads_bf16(hipStream_t stream, int n_problems, const jpp_gemm_args* problems, int n_cols,
                    const jpp_colsum_item* items, int64_t rows, float* partial) {
  JPP_REQUIRE(problems && n_problems >= 1 && n_problems <= 4, "gemm_multi: 1 to 4 problems");
  if (n_problems == 1) {
    if (n_cols)
      if (int rc = jpp_colsum_accum_multi(stream, n_cols, items, rows, partial)) return rc;
    return jpp_gemm_bf16(stream, problems);
  }
  GemmParams ps[4];
  Extent e[4];
  long tiles = 0;
  for (int i = 0; i < n_problems; ++i) {
    const jpp_gemm_args* a = problems + i;
    if (int rc = prepare(a, ps[i])) return rc;
    JPP_REQUIRE(a->trans_a && a->trans_b && a->epilogue == JPP_EPI_ACC_F32 &&
                    a->group_mode == JPP_GROUP_NONE && !a->bias && !a->resid && !a->tile,
                "gemm_multi: problem %d is not a plain accumulated weight gradient (trans_a = "
                "trans_b = 1, JPP_EPI_ACC_F32, no groups, bias, residual or tile choice)", i);
    JPP_REQUIRE(a->k == problems[0].k && ps[i].k_parts == ps[0].k_parts,
                "gemm_multi: problem %d differs from problem 0 in k or k_parts", i);
    e[i] = {a->m, a->n};
    tiles += (a->m / 64) * (a->n / 64);
  }
  JPP_REQUIRE(tiles < (1L << 30), "gemm_multi: too many tiles");
  const long ksteps = (long)ps[0].k / 64 * ps[0].k_parts;
  const int tile = cheapest_tile(e, e, n_problems, ksteps, true, false, false);
  const bool deep = deep_stages(tile == kTile64 ? tiles : tiles / 4, ksteps, tile);
  // A layer's bias gradients beside its weight gradients: their workgroups run in the shadow of the tiles' (hidden
  // 768 on 1152 tokens: 31.0 us and a launch of 5.7, together 31.3), and there is one launch less to enqueue.
  ColsumPanels cols;
  memset(&cols, 0, sizeof(cols));
  int blocks = 0;
  if (n_cols && tile != kTile256)
    if (int rc = colsum_panels(n_cols, items, rows, &cols, &blocks)) return rc;
  if (n_cols && !blocks)
    if (int rc = jpp_colsum_accum_multi(stream, n_cols, items, rows, partial)) return rc;
  if (tile == kTile256) return launch_multi<256, 256, 8, 2>(stream, ps, n_problems, cols, 0, 0);
  if (tile == kTile64)
    return deep ? launch_multi<64, 64, 4, 4, 2>(stream, ps, n_problems, cols, blocks, rows)
                : launch_multi<64, 64, 4, 2, 2>(stream, ps, n_problems, cols, blocks, rows);
  return deep ? launch_multi<128, 128, 8, 5>(stream, ps, n_problems, cols, blocks, rows)
              : launch_multi<128, 128, 8, 2>(stream, ps, n_problems, cols, blocks, rows);
}
