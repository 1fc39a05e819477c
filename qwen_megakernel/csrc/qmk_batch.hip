// Batched forward of T tokens through Qwen3 on gfx950: prompt prefill (T
// tokens of one sequence at consecutive positions) and batched decode (one
// token of each of B sequences, each at its own position), or any mix.
// Unlike the per-token decode kernel, the work here has T rows per weight
// read, so the projections run as MFMA GEMMs (v_mfma_f32_16x16x32_bf16) and a
// layer is a short sequence of kernels on the caller's stream instead of one
// persistent launch.  Numerics follow HF Qwen3's bf16 eager path op for op, as
// the decode kernel does: every projection is an fp32 sum rounded once to
// bf16; norms, RoPE, softmax probabilities, residual adds and SiLU*up round
// where HF rounds.
//
// The reference prefills one token per step() (qwen_megakernel/model.py:210-211)
// and decodes one sequence; the batched forward is an addition.
//
// At most kRowsMax tokens take gemm_rows and its fused prologues and epilogues ("few tokens" below).
// Per layer above that (kernels in launch order):
//   gemm_tiled(qkv)    -> qkv_finish (split-K sum, q/k RMSNorm + RoPE, K/V append;
//                         in the GEMM's epilogue when K is not split)
//   attention          (one workgroup per (token, KV head) over short contexts; MFMA
//                       tiles of each prompt, over key chunks where they are few;
//                       128-position chunks per token for a batched step)
//   gemm_tiled(o)      -> residual_norm (residual add, post-attention RMSNorm)
//   gemm_tiled(g|u)    -> gate_up_finish (SiLU(g) * u; in the GEMM's epilogue when K
//                         is not split)
//   gemm_tiled(down)   -> residual_norm (residual add, next layer's input RMSNorm
//                                        or the final norm)
// then the LM head over the emitted rows (bf16 logits, argmax keys)
// -> keys_reduce (per-row argmax).

#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/qwen_megakernel.h"
#include "qmk_batch_decode.h"
#include "qmk_decode_kernel.h"

namespace qmk {
namespace batch {


constexpr int kD = 128, kNQ = 16, kNKV = 8, kQS = kNQ * kD, kNQKV = (kNQ + 2 * kNKV) * kD;
constexpr int kQT = 64;  // MFMA prefill attention: tokens per tile
constexpr int kKB = 64, kKPad = kD + 8, kVPad = kKB + 8;  // its split passes: keys per block, LDS rows
// Tokens of the smallest tile, and of the smallest that starts below kQT.  us per 4-layer forward, as tiles
// against left tokens: 8 runs of 5 after 2000 positions 392 / 476, 12 of 8 after 1500 476 / 546, 40 of 4
// after 1500 917 / 773, 100 of 12 from position 0 583 / 529.
constexpr int kMinTile = 5, kMinTileNear = 16;
constexpr int kLeftWave = 512;  // left tokens below this position may take a wave each
constexpr int kMfmaAttnTokens = 320;   // prompts of this many tokens run attention_mfma
constexpr int kMfmaAttnContext = 256;  // so do fewer tokens over this many positions of context; attention_rows below
constexpr int kMaxAttnChunks = 16;    // split attention_mfma passes: a tile's key chunks at most
constexpr int kSplitChunk = 128;  // split attention: positions per workgroup
constexpr int kSplitBelow = 32;   // fewer tokens than this use the split attention ...
constexpr int kSplitContext = 128;  // ... over more than this many positions of context
constexpr int kMaxSplit = 16;     // K splits of one GEMM (their partials are summed in a fixed order)
constexpr int kMaxEmit = 256;

static_assert(Qwen3_0_6B::D == kD && Qwen3_0_6B::NQ == kNQ && Qwen3_0_6B::NKV == kNKV, "head layout");
static_assert(Qwen3_1_7B::D == kD && Qwen3_1_7B::NQ == kNQ && Qwen3_1_7B::NKV == kNKV, "head layout");

// Per-token metadata, checked once (embed_tokens).  An invalid token (id outside
// the vocabulary, sequence or position out of range) reads embedding row 0,
// writes nothing into any cache and emits -1.
struct Tok {
  int token, seq, pos, valid;
};

struct Cache {
  uint16_t* k;
  uint16_t* v;
  long long seq_stride;  // elements from one sequence's [L][NKV][S][D] block to the next
  int max_seq_len;
};

__device__ __forceinline__ bf16x8 ld_bf16x8(const uint16_t* p) { return __builtin_bit_cast(bf16x8, ld16(p)); }
__device__ __forceinline__ bf16x8 ld_bf16x8_stream(const uint16_t* p) {
  return __builtin_bit_cast(bf16x8, ld_stream(p));
}

__device__ __forceinline__ size_t cache_base(const Cache& c, const Tok& tk, int L, int g) {
  return (size_t)tk.seq * c.seq_stride + ((size_t)L * kNKV + g) * c.max_seq_len * kD;
}

// Sum over the block (256 threads) of one value per head; `red` is [2][4].
__device__ __forceinline__ void block_sum2(float (&v)[2], float (*red)[4]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  v[0] = wave_sum(v[0]);
  v[1] = wave_sum(v[1]);
  __syncthreads();
  if (lane == 0) {
    red[0][wave] = v[0];
    red[1][wave] = v[1];
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; h++) v[h] = (red[h][0] + red[h][1]) + (red[h][2] + red[h][3]);
}

__device__ __forceinline__ void block_max2(float (&v)[2], float (*red)[4]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  v[0] = wave_max(v[0]);
  v[1] = wave_max(v[1]);
  __syncthreads();
  if (lane == 0) {
    red[0][wave] = v[0];
    red[1][wave] = v[1];
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; h++) v[h] = fmaxf(fmaxf(red[h][0], red[h][1]), fmaxf(red[h][2], red[h][3]));
}

// ---------------------------------------------------------------- tokens

// Tiles of the MFMA attention: up to kQT tokens of one sequence at consecutive positions, neighbours in
// the call.  A run of such tokens (a prompt) is cut into tiles from its own start, so the tiles of one
// prompt hold no token of the next.  What would be a tile of fewer than kMinTile tokens is left to the rows
// at the kernels' end (attention_left), as are tokens past `cap` tiles and invalid ones.  (With tiles cut every kQT tokens of the call, those that
// held two prompts went to attention_rows: four prompts of 411..613 tokens, Qwen3-1.7B, 56 us per
// layer beside 37 of attention_mfma, now 40 in all.)
// The split passes' key chunks are planned here too, from the tiles that there are, not from the sequences
// that the cache could hold (a turn of 100 tokens after 6000 positions in a cache of 8 sequences, 4 layers:
// 887 us with the chunks shared by the part tiles of all 8, 376 with those of its own two tiles).
struct AttnPlan {
  int* hdr;    // {tiles, left tokens, key chunks per tile, blocks per chunk, left tokens past kLeftWave}
  int4* tile;  // {first token, tokens, its position, sequence}, the ones with the most keys first
  int2* raw;   // {first token, tokens} in token order,
  int* rank;   // the places of those in `tile`,
  int* key;    // and their last positions
  int* where;  // per token: tile * kQT + row, or -1
  int* left;   // tokens in no tile: those of positions below kLeftWave from the front, others from the back
  int cap;     // tiles at most (0: no plan)
  int budget;  // split passes: tile chunks that the partials hold (0: whole tiles)
  int nkb;     // and blocks of kKB keys that the call's context may have
};

// Key chunks of each of `tiles` tiles in a call of nt = ceil(T / kQT): its share of the budget, of two
// blocks or more.  One chunk (more tiles than half the budget): the whole context.
__host__ __device__ __forceinline__ int2 attn_key_chunks(int budget, int nkb, int nt, int tiles) {
  int nch = budget / (tiles > nt ? tiles : nt);
  nch = nch < nkb / 2 ? nch : nkb / 2;
  nch = nch > 1 ? nch : 1;
  const int ck = (nkb + nch - 1) / nch;
  return make_int2((nkb + ck - 1) / ck, ck);
}

// One workgroup of 256 threads, each over T / 256 neighbouring tokens; info(t) = {sequence, position},
// sequence -1 for an invalid token.
template <class F>
__device__ __forceinline__ void plan_attention(int T, const AttnPlan& pl, F&& read) {
  // up to kHeld tokens, everything between the inputs and the plan stays in LDS (2048 tokens: 23 us in
  // global memory, 17 in LDS, 6 for one run; embedding alone takes 5)
  constexpr int kHeld = 2048, kTiles = 288;
  __shared__ int2 held[kHeld], lraw[kTiles];
  __shared__ int lwhere[kHeld], lrank[kTiles], lkey[kTiles], ws[4], ntiles, nleft[2];
  const bool in_lds = T <= kHeld && pl.cap <= kTiles;
  int2* const raw = in_lds ? lraw : pl.raw;
  int* const rank = in_lds ? lrank : pl.rank;
  int* const key = in_lds ? lkey : pl.key;
  int* const where = in_lds ? lwhere : pl.where;
  const int th = threadIdx.x, wave = th >> 6, lane = th & 63, per = (T + 255) / 256, a = min(T, th * per),
            b = min(T, a + per);
  {  // every load of the thread's tokens before the first use
    int2 x[kHeld / 256];
#pragma unroll
    for (int i = 0; i < kHeld / 256; i++) x[i] = read(min(th + 256 * i, T - 1));
#pragma unroll
    for (int i = 0; i < kHeld / 256; i++) held[th + 256 * i] = x[i];
  }
  if (th == 0) nleft[0] = nleft[1] = 0;
  auto header = [&](int tiles, int left, int far) {
    const int2 kc = attn_key_chunks(pl.budget, pl.nkb, (T + kQT - 1) / kQT, tiles);
    *reinterpret_cast<int4*>(pl.hdr) = make_int4(tiles, left, kc.x, kc.y);
    pl.hdr[4] = far;
  };
  __syncthreads();
  auto info = [&](int t) { return t < kHeld ? held[t] : read(t); };
  {  // one run (a single prompt): its tiles, the last one first
    const int2 x0 = info(0);
    int one = x0.x >= 0;
    for (int t = th; t < T; t += 256) {
      const int2 x = info(t);
      one &= (x.x == x0.x) & (x.y == x0.y + t);
    }
    const int nt = (T + kQT - 1) / kQT;
    if (__syncthreads_and(one) && nt <= pl.cap) {
      for (int i = th; i < nt; i += 256)
        pl.tile[nt - 1 - i] = make_int4(i * kQT, min(kQT, T - i * kQT), x0.y + i * kQT, x0.x);
      for (int t = th; t < T; t += 256) pl.where[t] = (nt - 1 - t / kQT) * kQT + t % kQT;
      if (th == 0) header(nt, 0, 0);
      return;
    }
  }
  auto starts = [&](int t, int2 x) {  // token t (x, valid) does not continue token t - 1's run
    if (t == 0) return true;
    const int2 y = info(t - 1);
    return y.x != x.x || y.y + 1 != x.y;
  };
  auto scan = [&](int v, bool sum) {  // exclusive over the threads: sum, or maximum from -1
    const int none = sum ? 0 : -1;
    auto op = [&](int x, int y) { return sum ? x + y : max(x, y); };
    int incl = v;
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(incl, o);
      if (lane >= o) incl = op(incl, x);
    }
    const int prev = __shfl_up(incl, 1);
    if (lane == 63) ws[wave] = incl;
    __syncthreads();
    int ex = lane ? prev : none;
    for (int q = 0; q < wave; q++) ex = op(ex, ws[q]);
    __syncthreads();
    return ex;
  };
  // each token's end of run: the next token that is invalid or starts a run
  {
    int next = -T;  // minus the first such token after the segment (the scans go forward over threads)
    int mine = -T;
    for (int t = b - 1; t >= a; t--) {
      const int2 x = info(t);
      if (x.x < 0 || starts(t, x)) mine = -t;
    }
    // exclusive maximum over the threads after this one
    int incl = mine;
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_down(incl, o);
      if (lane + o < 64) incl = max(incl, x);
    }
    const int after = __shfl_down(incl, 1);
    if (lane == 0) ws[wave] = incl;
    __syncthreads();
    if (lane < 63) next = after;
    for (int q = wave + 1; q < 4; q++) next = max(next, ws[q]);
    __syncthreads();
    int end = -next;
    for (int t = b - 1; t >= a; t--) {
      where[t] = end;
      const int2 x = info(t);
      if (x.x < 0 || starts(t, x)) end = t;
    }
  }
  // rows of the tile whose first token is t (0: left)
  auto tile_rows = [&](int t, int end) {
    const int n = min(kQT, end - t);
    return n < (info(t).y < kQT ? kMinTileNear : kMinTile) ? 0 : n;
  };
  int last = -1;  // the segment's last run start
  for (int t = a; t < b; t++) {
    const int2 x = info(t);
    if (x.x >= 0 && starts(t, x)) last = t;
  }
  const int rs0 = scan(last, false);
  int rs = rs0, cnt = 0;
  for (int t = a; t < b; t++) {
    const int2 x = info(t);
    if (x.x < 0) continue;
    if (starts(t, x)) rs = t;
    cnt += (t - rs) % kQT == 0 && tile_rows(t, where[t]) > 0;
  }
  int id = scan(cnt, true) - 1;
  rs = rs0;
  for (int t = a; t < b; t++) {
    const int2 x = info(t);
    int wh = -1;
    if (x.x >= 0) {
      if (starts(t, x)) rs = t;
      const int row = (t - rs) % kQT, rows = tile_rows(t - row, where[t]);
      if (rows) {
        id += row == 0;
        if (id < pl.cap) {
          wh = id * kQT + row;
          if (row == 0) {
            raw[id] = make_int2(t, rows);
            key[id] = x.y + rows - 1;  // the tile's last position
          }
        }
      }
    }
    where[t] = wh;
    if (wh < 0) {
      const bool far = x.x >= 0 && x.y >= kLeftWave;
      const int i = atomicAdd(&nleft[far], 1);
      pl.left[far ? T - 1 - i : i] = t;
    }
  }
  if (th == 255) ntiles = min(pl.cap, id + 1);  // the last thread's count of tiles is the call's
  __threadfence_block();
  __syncthreads();
  const int nt = ntiles;
  if (th == 0) header(nt, nleft[0] + nleft[1], nleft[1]);
  // the tiles by their last position (keys), largest first, and each token's place among them
  for (int i = th; i < nt; i += 256) {
    const int kx = key[i];
    int r = 0;
    for (int k = 0; k < nt; k++) {
      const int ky = key[k];
      r += ky > kx || (ky == kx && k < i);
    }
    const int2 tl = raw[i], x = info(tl.x);
    pl.tile[r] = make_int4(tl.x, tl.y, x.y, x.x);
    rank[i] = r;
  }
  __threadfence_block();
  __syncthreads();
  for (int t = th; t < T; t += 256) {
    const int wh = where[t];
    pl.where[t] = wh < 0 ? -1 : rank[wh / kQT] * kQT + wh % kQT;
  }
}

// One workgroup per token t: its checked record, X[t] = embed[token], and what the first layer's q/k/v
// projection needs of it: N[t] = RMSNorm(X[t]) (NORM), or the row's sum of squares for gemm_rows,
// ssq[t][0] (its other partials 0).  Token 0's also checks the emit rows.  With a plan, a
// workgroup before them all plans the attention tiles.  (Token records, embedding and norm as three launches took 4.5 us
// each.)
template <int H, bool NORM>
__global__ void __launch_bounds__(256) embed_tokens(const int* __restrict__ tokens, const int* __restrict__ seqs,
                                                    const int* __restrict__ pos, int T, const int* __restrict__ emit,
                                                    int R, int num_seqs, int max_context, int vocab,
                                                    const uint16_t* __restrict__ embed, Tok* __restrict__ tok,
                                                    int* __restrict__ erow, uint16_t* __restrict__ X,
                                                    const uint16_t* __restrict__ norm_w, float eps,
                                                    uint16_t* __restrict__ Nout, float* __restrict__ ssq, AttnPlan pl) {
  constexpr int J = H / 256, JW = J / 2;  // elements and bf16 pairs per thread
  typedef unsigned words_t __attribute__((ext_vector_type(JW)));
  __shared__ float red[4];
  const int t = (int)blockIdx.x - (pl.cap ? 1 : 0), i0 = J * threadIdx.x;
  auto valid = [&](int id, int sq, int p) {
    return (id >= 0) & (id < vocab) & (sq >= 0) & (sq < num_seqs) & (p >= 0) & (p < max_context);  // no branches
  };
  if (t < 0) {
    plan_attention(T, pl, [&](int u) {
      const int sq = seqs ? seqs[u] : u, p = pos[u];
      return make_int2(valid(tokens[u], sq, p) ? sq : -1, p);
    });
    return;
  }
  const int id = tokens[t], sq = seqs ? seqs[t] : t, p = pos[t];
  const bool ok = valid(id, sq, p);
  if (threadIdx.x == 0) tok[t] = Tok{ok ? id : 0, ok ? sq : 0, ok ? p : 0, ok ? 1 : 0};
  if (t == 0)
    for (int i = threadIdx.x; i < R; i += 256) {
      const int e = emit ? emit[i] : i;
      erow[i] = (e >= 0 && e < T) ? e : -1;
    }
  const words_t xw = *reinterpret_cast<const words_t*>(embed + (size_t)(ok ? id : 0) * H + i0);
  *reinterpret_cast<words_t*>(X + (size_t)t * H + i0) = xw;
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < JW; e++) ss += lo_bf16(xw[e]) * lo_bf16(xw[e]) + hi_bf16(xw[e]) * hi_bf16(xw[e]);
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  ss = (red[0] + red[1]) + (red[2] + red[3]);
  if constexpr (NORM) {
    const float rstd = rcp_sqrt_torch(__fdiv_rn(ss, (float)H) + eps);
    const words_t ww = *reinterpret_cast<const words_t*>(norm_w + i0);
    words_t out;
#pragma unroll
    for (int e = 0; e < JW; e++)
      out[e] = pack_bf16x2(bf16r(lo_bf16(ww[e]) * bf16r(lo_bf16(xw[e]) * rstd)),
                           bf16r(hi_bf16(ww[e]) * bf16r(hi_bf16(xw[e]) * rstd)));
    *reinterpret_cast<words_t*>(Nout + (size_t)t * H + i0) = out;
  } else {
    for (int i = threadIdx.x; i < H / 8; i += 256) ssq[(size_t)t * (H / 8) + i] = i == 0 ? ss : 0.f;
  }
}

// ---------------------------------------------------------------- GEMM
//
// W rows come from up to three row-major [rows][K] matrices laid end to end
// (q, k, v; or gate, up).  The GEMMs run on 16x16x32 bf16 MFMAs, whose
// operand layouts (checked by qmk_selftest_mfma) are: lane l supplies
// A[l%16][8*(l/16) .. +7] and B[8*(l/16) .. +7][l%16], i.e. 16 contiguous bytes
// of an X row and of a W row; it receives C[4*(l/16) + i][l%16], i = 0..3.
struct Seg {
  const uint16_t* w[3];
  int rows[3];
};

__device__ __forceinline__ const uint16_t* seg_row(const Seg& s, int n, int K) {
  if (n < s.rows[0]) return s.w[0] + (size_t)n * K;
  n -= s.rows[0];
  if (n < s.rows[1]) return s.w[1] + (size_t)n * K;
  n -= s.rows[1];
  return s.w[2] + (size_t)n * K;
}

// The work after the q/k/v projection for one (token, head) of the 32 q/k/v heads, one wave,
// lane l holding the head's bf16-rounded projections x0 = column l, x1 = column l + 64: q:
// RMSNorm over head_dim + RoPE -> Q;  k: the same -> K cache at the token's position;  v: -> V
// cache.  (modeling_qwen3.py:252-253, 168)
struct QkvOut {
  const Tok* tok;
  int L;
  const uint16_t* q_norm;
  const uint16_t* k_norm;
  const uint16_t* cos_t;
  const uint16_t* sin_t;
  Cache c;
  float eps;
  uint16_t* Q;
};

__device__ __forceinline__ void qkv_head(const QkvOut& o, int t, int h, int lane, float x0, float x1) {
  const Tok tk = o.tok[t];
  if (h >= kNQ + kNKV) {
    if (tk.valid) {
      uint16_t* dst = o.c.v + cache_base(o.c, tk, o.L, h - kNQ - kNKV) + (size_t)tk.pos * kD;
      dst[lane] = (uint16_t)f32_to_bf16(x0);
      dst[lane + 64] = (uint16_t)f32_to_bf16(x1);
    }
    return;
  }
  const bool is_q = h < kNQ;
  if (!is_q && !tk.valid) return;
  const uint16_t* nw = is_q ? o.q_norm : o.k_norm;
  const uint16_t* cr = o.cos_t + (size_t)tk.pos * kD;
  const uint16_t* sr = o.sin_t + (size_t)tk.pos * kD;
  const float ss = wave_sum(x0 * x0 + x1 * x1);
  const float rstd = rcp_sqrt_torch(__fdiv_rn(ss, (float)kD) + o.eps);
  const float n0 = bf16r(bf16_to_f32(ldu16(nw + lane)) * bf16r(x0 * rstd));
  const float n1 = bf16r(bf16_to_f32(ldu16(nw + lane + 64)) * bf16r(x1 * rstd));
  const float c0 = bf16_to_f32(ldu16(cr + lane)), c1 = bf16_to_f32(ldu16(cr + lane + 64));
  const float s0 = bf16_to_f32(ldu16(sr + lane)), s1 = bf16_to_f32(ldu16(sr + lane + 64));
  // x*cos + rotate_half(x)*sin, rotate_half(x) = (-x[64:], x[:64])
  const float y0 = bf16r(bf16r(n0 * c0) + bf16r(-n1 * s0));
  const float y1 = bf16r(bf16r(n1 * c1) + bf16r(n0 * s1));
  uint16_t* dst =
      is_q ? o.Q + (size_t)t * kQS + h * kD : o.c.k + cache_base(o.c, tk, o.L, h - kNQ) + (size_t)tk.pos * kD;
  dst[lane] = (uint16_t)f32_to_bf16(y0);
  dst[lane + 64] = (uint16_t)f32_to_bf16(y1);
}

// qkv_head for the 128 rows x 128 columns of one head held in LDS (bf16), rows t0.. (those
// below T): wave w takes rows 32w..32w+31, four at a time, 16 lanes per row; lane c of a row
// holds columns 4c..4c+3 and their RoPE partners 64+4c..64+4c+3.  The sum of squares runs over
// the row's 16 lanes.  Everything the rows read from global memory besides the tile (their token
// records, then their cos/sin entries, and the head-norm weights) is requested up front by
// qkv_rows_fetch, before the tile goes through LDS, so the eight row groups do not each wait for
// two dependent loads.
struct QkvRowsIn {
  Tok tk[8];
  uint2 cl[8], ch[8], sl[8], sh[8];
  float nw[8];
};

__device__ __forceinline__ void qkv_rows_fetch(const QkvOut& o, int t0, int T, int h, int w, int lane, QkvRowsIn& in) {
  const int c = lane & 15, sub = lane >> 4;
  const bool is_v = h >= kNQ + kNKV, is_q = h < kNQ;
#pragma unroll
  for (int it = 0; it < 8; it++) {
    const int t = t0 + 32 * w + 4 * it + sub;
    in.tk[it] = o.tok[t < T ? t : t0];
  }
  if (is_v) return;
  const uint16_t* wp = is_q ? o.q_norm : o.k_norm;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    in.nw[e] = bf16_to_f32(ldu16(wp + 4 * c + e));
    in.nw[4 + e] = bf16_to_f32(ldu16(wp + 64 + 4 * c + e));
  }
#pragma unroll
  for (int it = 0; it < 8; it++) {
    const size_t pb = (size_t)in.tk[it].pos * kD;
    in.cl[it] = *reinterpret_cast<const uint2*>(o.cos_t + pb + 4 * c);
    in.ch[it] = *reinterpret_cast<const uint2*>(o.cos_t + pb + 64 + 4 * c);
    in.sl[it] = *reinterpret_cast<const uint2*>(o.sin_t + pb + 4 * c);
    in.sh[it] = *reinterpret_cast<const uint2*>(o.sin_t + pb + 64 + 4 * c);
  }
}

__device__ __forceinline__ void qkv_tile_rows(const QkvOut& o, const uint16_t (*Xh)[128], int t0, int T, int h, int w,
                                              int lane, const QkvRowsIn& in) {
  const int c = lane & 15, sub = lane >> 4;
  const bool is_v = h >= kNQ + kNKV, is_q = h < kNQ;
#pragma unroll
  for (int it = 0; it < 8; it++) {
    const int row = 32 * w + 4 * it + sub, t = t0 + row;
    if (t0 + 32 * w + 4 * it >= T) break;  // uniform: no row of this group is below T
    const bool live = t < T;
    const Tok tk = in.tk[it];
    const uint2 lo = *reinterpret_cast<const uint2*>(&Xh[row][4 * c]);
    const uint2 hi = *reinterpret_cast<const uint2*>(&Xh[row][64 + 4 * c]);
    float x[8] = {lo_bf16(lo.x), hi_bf16(lo.x), lo_bf16(lo.y), hi_bf16(lo.y),
                  lo_bf16(hi.x), hi_bf16(hi.x), lo_bf16(hi.y), hi_bf16(hi.y)};
    if (is_v) {
      if (live && tk.valid) {
        uint16_t* dst = o.c.v + cache_base(o.c, tk, o.L, h - kNQ - kNKV) + (size_t)tk.pos * kD;
        *reinterpret_cast<uint2*>(dst + 4 * c) = lo;
        *reinterpret_cast<uint2*>(dst + 64 + 4 * c) = hi;
      }
      continue;
    }
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) ss += x[e] * x[e];
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) ss += __shfl_xor(ss, m);  // within the row's 16 lanes
    const float rstd = rcp_sqrt_torch(__fdiv_rn(ss, (float)kD) + o.eps);
    float n[8];
#pragma unroll
    for (int e = 0; e < 8; e++) n[e] = bf16r(in.nw[e] * bf16r(x[e] * rstd));
    const uint2 cl = in.cl[it], ch = in.ch[it], sl = in.sl[it], sh = in.sh[it];
    const float cs[8] = {lo_bf16(cl.x), hi_bf16(cl.x), lo_bf16(cl.y), hi_bf16(cl.y),
                         lo_bf16(ch.x), hi_bf16(ch.x), lo_bf16(ch.y), hi_bf16(ch.y)};
    const float sn[8] = {lo_bf16(sl.x), hi_bf16(sl.x), lo_bf16(sl.y), hi_bf16(sl.y),
                         lo_bf16(sh.x), hi_bf16(sh.x), lo_bf16(sh.y), hi_bf16(sh.y)};
    // x*cos + rotate_half(x)*sin, rotate_half(x) = (-x[64:], x[:64])
    float y[8];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      y[e] = bf16r(bf16r(n[e] * cs[e]) + bf16r(-n[4 + e] * sn[e]));
      y[4 + e] = bf16r(bf16r(n[4 + e] * cs[4 + e]) + bf16r(n[e] * sn[4 + e]));
    }
    if (!live || (!is_q && !tk.valid)) continue;
    uint16_t* dst =
        is_q ? o.Q + (size_t)t * kQS + h * kD : o.c.k + cache_base(o.c, tk, o.L, h - kNQ) + (size_t)tk.pos * kD;
    *reinterpret_cast<uint2*>(dst + 4 * c) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
    *reinterpret_cast<uint2*>(dst + 64 + 4 * c) = make_uint2(pack_bf16x2(y[4], y[5]), pack_bf16x2(y[6], y[7]));
  }
}

// SiLU(g) * u as HF rounds it: bf16(bf16(silu(g)) * u), g and u bf16 (modeling_qwen3.py:82)
__device__ __forceinline__ float silu_mul(float g, float u) {
  const float sg = bf16r(__fdiv_rn(g, 1.0f + expf(-g)));
  return bf16r(sg * u);
}

// What gemm_tiled does with its sums: kEpiPart writes them to part (any K split); with the K
// range unsplit, kEpiQkv (128-column tiles = one q/k/v head each) runs the head's norm, RoPE and
// K/V append (qkv_head) and kEpiGateUp (tile columns 0..63 the gate rows m0..m0+63, 64..127
// the up rows of the same m) writes bf16(bf16(silu(g)) * u) to M, so neither the fp32 sums nor
// a finishing kernel touch memory.
enum { kEpiPart = 0, kEpiQkv = 1, kEpiGateUp = 2 };

struct GateUpOut {
  uint16_t* M;
  int I;
};

// Large T (prompt prefill): an LDS-tiled MFMA GEMM, part[z][t][n] = the sum
// over K split z of X[t][k] W[n][k].  Workgroup tile 128 rows x TN columns
// (TN = 128, or 64 for narrow N so that more workgroups run), BK = 64; wave w
// computes rows 64*(w&1)..+63 x columns (TN/2)*(w>>1)..+TN/2-1 as 4 x TN/32
// MFMA tiles.  Both operands go from global memory straight into LDS (LDS DMA,
// 16 bytes per lane) through two stages: step s+1's requests are issued right
// after the barrier that opens step s, so they land during step s's MFMAs.
// A stage row is 64 bf16, eight 16-byte chunks; chunk c of row r sits at
// position c ^ (r & 7), so the lanes that read one chunk of 8 consecutive rows
// touch every LDS bank once.  Two workgroups per CU (64 KB of LDS each).
// Measured at 2048 tokens against the same tiles staged through registers
// with padded rows: q/k/v 27.5 -> 22.4 us, gate/up 41.3 -> 32.5, o 19.4 ->
// 17.4, down 24.7 -> 22.9 (bit-identical sums: the K order is unchanged).
constexpr int kTM = 128, kTK = 64;

// 16 bytes per lane from global memory straight into LDS: lane i's bytes land at lds + 16 i (lds
// is the same for every lane of the wave)
__device__ __forceinline__ void dma16(const void* src, void* lds) {
  __builtin_amdgcn_global_load_lds(as_global<void>(src), (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// Barrier of a ring of DMA stages: at most N of this wave's requests are still in flight, its LDS
// reads so far have returned, and every wave of the workgroup has come this far.  (__syncthreads
// would do for the order, but the count of requests left in flight has to be exact.)
template <int N>
__device__ __forceinline__ void ring_barrier() {
  wait_vmcnt_upto<N>();
  __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int TN, int EPI = kEpiPart>
__global__ void __launch_bounds__(256, 2) gemm_tiled(const uint16_t* __restrict__ X, int T, int K, Seg seg, int N,
                                                     int ksplit, float* __restrict__ part, QkvOut qo, GateUpOut go) {
  static_assert(TN == 64 || TN == 128, "tile width");
  static_assert(EPI == kEpiPart || TN == 128, "fused epilogues take 128-column tiles");
  constexpr int WJ = TN / 32;  // 16-column MFMA tiles per wave (a wave covers TN / 2 columns)
  constexpr int ABytes = kTM * kTK * 2, BBytes = TN * kTK * 2, StB = ABytes + BBytes;
  constexpr int NA = ABytes / 4096, NB = BBytes / 4096;  // 1 KB DMA blocks (8 rows) per wave and stage
  __shared__ __align__(1024) unsigned char sm[2 * StB];
  const int n0 = blockIdx.x * TN, t0 = blockIdx.y * kTM;
  // K split z of ksplit (blockIdx.z): columns [kz, kz + K / ksplit); partial sums to part[z]
  const int kz = blockIdx.z * (K / ksplit);
  part += (size_t)blockIdx.z * T * N;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = w & 1, wn = w >> 1;
  // DMA block q of wave w holds rows 8 (NA w + q) .. +7 of A (of B: NB); lane l fills position
  // l % 8 of row l / 8 of the block, i.e. it requests chunk (l % 8) ^ (row & 7) of that row
  const uint16_t* asrc[NA];
  const uint16_t* bsrc[NB];
#pragma unroll
  for (int q = 0; q < NA; q++) {
    const int row = 8 * (NA * w + q) + (lane >> 3), c = (lane & 7) ^ (row & 7);
    asrc[q] = X + (size_t)min(t0 + row, T - 1) * K + kz + 8 * c;
  }
#pragma unroll
  for (int q = 0; q < NB; q++) {
    const int row = 8 * (NB * w + q) + (lane >> 3), c = (lane & 7) ^ (row & 7);
    if constexpr (EPI == kEpiGateUp)  // tile columns 0..63: gate rows m0.., 64..127: up rows m0..
      bsrc[q] = seg.w[row >> 6] + (size_t)(n0 / 2 + (row & 63)) * K + kz + 8 * c;
    else
      bsrc[q] = seg_row(seg, n0 + row, K) + kz + 8 * c;
  }
  auto issue = [&](int st) {
    const int k = st * kTK;
    unsigned char* base = sm + (st & 1) * StB;
#pragma unroll
    for (int q = 0; q < NA; q++) dma16(asrc[q] + k, base + 1024 * (NA * w + q));
#pragma unroll
    for (int q = 0; q < NB; q++) dma16(bsrc[q] + k, base + ABytes + 1024 * (NB * w + q));
  };
  f32x4 acc[4][WJ];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < WJ; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int l16 = lane & 15, lq = lane >> 4;
  const int steps = K / ksplit / kTK;
  issue(0);
  for (int st = 0; st < steps; st++) {
    wait_vmcnt(0);    // this wave's requests of step st have landed
    __syncthreads();  // every wave's have, and step st - 1's stage is read
    if (st + 1 < steps) issue(st + 1);
    const unsigned char* base = sm + (st & 1) * StB;
#pragma unroll
    for (int kc = 0; kc < kTK / 8; kc += 4) {  // 32 K per MFMA: chunks kc..kc+3, lane chunk kc + lq
      bf16x8 a[4], b[WJ];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int row = 64 * wm + 16 * i + l16;
        a[i] = *reinterpret_cast<const bf16x8*>(base + row * (kTK * 2) + 16 * ((kc + lq) ^ (row & 7)));
      }
#pragma unroll
      for (int j = 0; j < WJ; j++) {
        const int row = (TN / 2) * wn + 16 * j + l16;
        b[j] = *reinterpret_cast<const bf16x8*>(base + ABytes + row * (kTK * 2) + 16 * ((kc + lq) ^ (row & 7)));
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < WJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }
  if constexpr (EPI == kEpiPart) {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < WJ; j++) {
        const int n = n0 + (TN / 2) * wn + 16 * j + l16;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int t = t0 + 64 * wm + 16 * i + 4 * (lane >> 4) + r;
          if (t < T) part[(size_t)t * N + n] = acc[i][j][r];
        }
      }
  } else if constexpr (EPI == kEpiQkv) {
    // the tile's 128 rows x 128 columns (one head), bf16-rounded, through LDS: then wave w takes
    // rows 32w..32w+31 one at a time, lane l columns l and l + 64
    static_assert(sizeof(sm) >= kTM * 128 * 2, "the head tile fits the operand stages");
    auto Xh = reinterpret_cast<uint16_t(*)[128]>(sm);
    QkvRowsIn in;
    qkv_rows_fetch(qo, t0, T, blockIdx.x, w, lane, in);
    __syncthreads();  // every wave's last operand reads are done
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < WJ; j++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          Xh[64 * wm + 16 * i + 4 * (lane >> 4) + r][64 * wn + 16 * j + l16] = (uint16_t)f32_to_bf16(acc[i][j][r]);
    __syncthreads();
    qkv_tile_rows(qo, Xh, t0, T, blockIdx.x, w, lane, in);
  } else {
    // the tile's gate and up projections, bf16-rounded, through LDS: G[row][c], U[row][c] for
    // m = m0 + c; then each thread takes 8 consecutive m of one row at a time and stores them
    // as one 16-byte chunk
    static_assert(sizeof(sm) >= 2 * kTM * 64 * 2, "the gate and up tiles fit the operand stages");
    auto G = reinterpret_cast<uint16_t(*)[64]>(sm);
    auto U = G + kTM;
    __syncthreads();  // every wave's last operand reads are done
    auto GU = wn == 0 ? G : U;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < WJ; j++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          GU[64 * wm + 16 * i + 4 * (lane >> 4) + r][16 * j + l16] = (uint16_t)f32_to_bf16(acc[i][j][r]);
    __syncthreads();
    const int m0 = n0 / 2, row = threadIdx.x >> 1, t = t0 + row;
    if (t < T) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int c0 = 32 * (threadIdx.x & 1) + 8 * q;
        const u32x4 g8 = *reinterpret_cast<const u32x4*>(&G[row][c0]);
        const u32x4 u8 = *reinterpret_cast<const u32x4*>(&U[row][c0]);
        const uint32_t gw[4] = {g8.x, g8.y, g8.z, g8.w}, uw[4] = {u8.x, u8.y, u8.z, u8.w};
        uint32_t mw[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
          mw[e] = pack_bf16x2(silu_mul(lo_bf16(gw[e]), lo_bf16(uw[e])), silu_mul(hi_bf16(gw[e]), hi_bf16(uw[e])));
        *reinterpret_cast<u32x4*>(go.M + (size_t)t * go.I + m0 + c0) = u32x4{mw[0], mw[1], mw[2], mw[3]};
      }
    }
  }
}

// Sum of the K-split partials of element (t, n), in split order.  All loads
// are issued before the first add.
__device__ __forceinline__ float sum_splits(const float* part, int ksplit, int T, int N, int t, int n) {
  const size_t stride = (size_t)T * N, idx = (size_t)t * N + n;
  float v[kMaxSplit];
#pragma unroll
  for (int s = 0; s < kMaxSplit; s++) v[s] = s < ksplit ? part[s * stride + idx] : 0.f;
  float y = v[0];
#pragma unroll
  for (int s = 1; s < kMaxSplit; s++)
    if (s < ksplit) y += v[s];
  return y;
}

// ---------------------------------------------------------------- row kernels

// One workgroup of 256 threads per token, J = H / 256 consecutive elements per
// thread (16-byte partial loads, 8- or 16-byte bf16 loads and stores).
// x = X[t] (+ bf16(sum of the split partials, in split order) when `part` is
// given, written back: HF's bf16 residual add);
// N[t] = bf16(w * bf16(x * rsqrt(mean(x^2) + eps))) (Qwen3RMSNorm).
// (At 2048 tokens, 4 splits: 12.2 us with one element per thread of 1024.)
template <int H>
__global__ void __launch_bounds__(256) residual_norm(const float* __restrict__ part, int ksplit, int T,
                                                     uint16_t* __restrict__ X, const uint16_t* __restrict__ w,
                                                     float eps, uint16_t* __restrict__ Nout) {
  constexpr int J = H / 256, JW = J / 2, JV = J / 4;  // elements, bf16 pairs, float4s per thread
  static_assert(J == 4 || J == 8, "four or eight elements per thread");
  typedef unsigned words_t __attribute__((ext_vector_type(JW)));
  __shared__ float red[4];
  const int t = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int i0 = J * threadIdx.x;
  words_t* const xp = reinterpret_cast<words_t*>(X + (size_t)t * H + i0);
  const words_t xw = *xp;
  float y[J];
#pragma unroll
  for (int e = 0; e < JW; e++) {
    y[2 * e] = lo_bf16(xw[e]);
    y[2 * e + 1] = hi_bf16(xw[e]);
  }
  if (part) {
    const size_t stride = (size_t)T * H;
    const float* p0 = part + (size_t)t * H + i0;
    float sum[J];
    // the splits in groups of G: every load of a group is issued before its adds.  Groups of
    // four for few splits (2048 tokens, 4 splits: 8.0 us, against 8.9 with groups of 16), of 16
    // float4 registers for many (128 tokens, 16 splits: 3.8 us, against 4.3 with groups of 4)
    auto add_splits = [&](auto g) {
      constexpr int G = decltype(g)::value;
      for (int s0 = 0; s0 < ksplit; s0 += G) {
        f32x4 v[G][JV];
#pragma unroll
        for (int q = 0; q < G; q++)
          if (s0 + q < ksplit) {
#pragma unroll
            for (int c = 0; c < JV; c++) v[q][c] = *reinterpret_cast<const f32x4*>(p0 + (s0 + q) * stride + 4 * c);
          }
#pragma unroll
        for (int q = 0; q < G; q++)
          if (s0 + q < ksplit) {
#pragma unroll
            for (int j = 0; j < J; j++) sum[j] = s0 + q == 0 ? v[q][j / 4][j % 4] : sum[j] + v[q][j / 4][j % 4];
          }
      }
    };
    if (ksplit <= 4) add_splits(std::integral_constant<int, 4>{});
    else add_splits(std::integral_constant<int, 16 / JV>{});
    words_t out;
#pragma unroll
    for (int e = 0; e < JW; e++) {
      y[2 * e] = bf16r(y[2 * e] + bf16r(sum[2 * e]));
      y[2 * e + 1] = bf16r(y[2 * e + 1] + bf16r(sum[2 * e + 1]));
      out[e] = pack_bf16x2(y[2 * e], y[2 * e + 1]);
    }
    *xp = out;
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < J; j++) ss += y[j] * y[j];
  ss = wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  ss = (red[0] + red[1]) + (red[2] + red[3]);
  const float rstd = rcp_sqrt_torch(__fdiv_rn(ss, (float)H) + eps);
  const words_t ww = *reinterpret_cast<const words_t*>(w + i0);
  words_t out;
#pragma unroll
  for (int e = 0; e < JW; e++)
    out[e] = pack_bf16x2(bf16r(lo_bf16(ww[e]) * bf16r(y[2 * e] * rstd)), bf16r(hi_bf16(ww[e]) * bf16r(y[2 * e + 1] * rstd)));
  *reinterpret_cast<words_t*>(Nout + (size_t)t * H + i0) = out;
}

// One wave per (token, head) of the 32 q/k/v heads.  Sums the split partials
// and rounds (the bf16 projections), then q: RMSNorm over head_dim + RoPE ->
// Q;  k: the same -> K cache at the token's position;  v: -> V cache.
// (modeling_qwen3.py:252-253, 168)
__global__ void __launch_bounds__(64) qkv_finish(const float* __restrict__ part, int ksplit, int T, QkvOut o) {
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const float x0 = bf16r(sum_splits(part, ksplit, T, kNQKV, t, h * kD + lane));
  const float x1 = bf16r(sum_splits(part, ksplit, T, kNQKV, t, h * kD + lane + 64));
  qkv_head(o, t, h, lane, x0, x1);
}

// M[t][n] = bf16(bf16(silu(g)) * u); g and u are columns n and I + n of the
// gate/up product (modeling_qwen3.py:82).
__global__ void __launch_bounds__(256) gate_up_finish(const float* __restrict__ part, int ksplit, int T, int I,
                                                      uint16_t* __restrict__ M) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)T * I) return;
  const int t = (int)(i / I), n = (int)(i % I);
  const float g = bf16r(sum_splits(part, ksplit, T, 2 * I, t, n));
  const float u = bf16r(sum_splits(part, ksplit, T, 2 * I, t, I + n));
  M[i] = (uint16_t)f32_to_bf16(silu_mul(g, u));
}

// ---------------------------------------------------------------- attention
//
// Eager GQA attention of token t over positions 0..pos of its sequence, for
// the two query heads of KV head g (modeling_qwen3.py:185-203): scores
// bf16(bf16(q.k) * scale), softmax in fp32 with the global max, probabilities
// rounded to bf16, P@V summed in fp32 and rounded to bf16.

// Scores of positions [0, n) into sc[h][p]; running max in m.
// Each 16-lane row takes one position (16 lanes x 8 dims); a wave four.
__device__ __forceinline__ void score_chunk(const uint16_t* kc, const u32x4 (&qv)[2], float scale, int n,
                                            float* sc0, float* sc1, float (&m)[2]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, slot = lane >> 4, t16 = lane & 15;
  for (int p = wave * 4 + slot; p < n; p += 16) {
    const u32x4 kx = ld16(kc + (size_t)p * kD + 8 * t16);
    const float s0 = bf16r(bf16r(row16_sum(dot8(kx, qv[0], 0.f))) * scale);
    const float s1 = bf16r(bf16r(row16_sum(dot8(kx, qv[1], 0.f))) * scale);
    if (t16 == 0) {
      sc0[p] = s0;
      sc1[p] = s1;
    }
    m[0] = fmaxf(m[0], s0);
    m[1] = fmaxf(m[1], s1);
  }
}

// Probability-weighted V rows [0, n), dims 2*lane..+1 of both
// heads, wave w taking rows w, w+4, ...
__device__ __forceinline__ void pv_chunk(const uint16_t* vc, const float* p0, const float* p1, int n,
                                         float (&acc)[2][2]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll 4
  for (int i = wave; i < n; i += 4) {
    const uint32_t v2 = ld32(vc + (size_t)i * kD + 2 * lane);
    const float va = lo_bf16(v2), vb = hi_bf16(v2);
    const float pa = p0[i], pb = p1[i];
    acc[0][0] += pa * va;
    acc[0][1] += pa * vb;
    acc[1][0] += pb * va;
    acc[1][1] += pb * vb;
  }
}

// Sum of the four waves' P@V partials (fixed order); thread (h = tid/128, d = tid%128).
__device__ __forceinline__ float pv_merge_waves(const float (&acc)[2][2], float (*pv)[2][kD]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; h++) {
    pv[wave][h][2 * lane] = acc[h][0];
    pv[wave][h][2 * lane + 1] = acc[h][1];
  }
  __syncthreads();
  const int h = threadIdx.x >> 7, d = threadIdx.x & 127;
  return ((pv[0][h][d] + pv[1][h][d]) + pv[2][h][d]) + pv[3][h][d];
}

// One workgroup per (token, KV head), both query heads, for contexts below kMfmaAttnContext.  It reserves LDS
// for more scores than those need, so that seven workgroups run on a CU: with eight, 255 tokens take 358 us per
// 4-layer forward, with seven 351 (100 and 200 tokens the same).
constexpr int kRowScores = 2048;
static_assert(kRowScores >= kMfmaAttnContext, "the scores of one context");
__global__ void __launch_bounds__(256) attention_rows(const uint16_t* __restrict__ Q, const Tok* __restrict__ tok,
                                                      int L, Cache c, float scale, uint16_t* __restrict__ out) {
  __shared__ float sc[2][kRowScores];
  __shared__ float red[2][4];
  __shared__ float pv[4][2][kD];
  const int t = blockIdx.x, g = blockIdx.y, t16 = threadIdx.x & 15;
  const Tok tk = tok[t];
  uint16_t* dst = out + (size_t)t * kQS + 2 * g * kD;  // both heads: 256 contiguous values
  if (!tk.valid) {
    dst[threadIdx.x] = 0;
    return;
  }
  const int C = tk.pos + 1;
  const size_t base = cache_base(c, tk, L, g);
  const uint16_t* kc = c.k + base;
  const uint16_t* vc = c.v + base;
  u32x4 qv[2];
#pragma unroll
  for (int h = 0; h < 2; h++) qv[h] = ld16(Q + (size_t)t * kQS + (2 * g + h) * kD + 8 * t16);
  float M[2] = {-INFINITY, -INFINITY};
  score_chunk(kc, qv, scale, C, sc[0], sc[1], M);
  block_max2(M, red);
  float S[2] = {0.f, 0.f};
  for (int i = threadIdx.x; i < C; i += 256) {
    S[0] += exp_acc(sc[0][i] - M[0]);
    S[1] += exp_acc(sc[1][i] - M[1]);
  }
  block_sum2(S, red);
  const float inv0 = __fdiv_rn(1.0f, S[0]), inv1 = __fdiv_rn(1.0f, S[1]);
  for (int i = threadIdx.x; i < C; i += 256) {
    sc[0][i] = bf16r(exp_acc(sc[0][i] - M[0]) * inv0);
    sc[1][i] = bf16r(exp_acc(sc[1][i] - M[1]) * inv1);
  }
  __syncthreads();
  float acc[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
  pv_chunk(vc, sc[0], sc[1], C, acc);
  dst[threadIdx.x] = (uint16_t)f32_to_bf16(pv_merge_waves(acc, pv));
}

// The attention of one token and KV head (both query heads) by NW waves: whole workgroups, or single waves
// (NW 1).  Both heads' scores of up to CAP positions are in LDS at once; a lane row of 16 takes a position
// (8 dims per lane), of K and of V, U of them in flight.  HF's two passes: with more than CAP
// positions the first keeps the running (max, sum) and the second forms the scores again.
template <int NW, int CAP>
struct LeftLds {
  float sc[2][CAP];
  float pv[NW > 1 ? NW : 0][2][kD];
  float2 ml[NW > 1 ? NW : 0][2];
};

template <int NW, int CAP>
__device__ __forceinline__ void left_row(const uint16_t* __restrict__ Q, const Tok* __restrict__ tok, int t, int g, int L,
                                         const Cache& c, float scale, uint16_t* __restrict__ out,
                                         LeftLds<NW, CAP>& lds) {
  constexpr int NT = 64 * NW, U = NW > 1 ? 4 : 8, R = 4 * NW;  // threads, rows in flight per lane row, rows per round
  const int lane = threadIdx.x & 63, slot = lane >> 4, t16 = lane & 15;
  const int w = NW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0, tid = NW > 1 ? (int)threadIdx.x : lane;
  // a wave's own LDS accesses are in order: only the compiler has to keep them so
  auto sync = [] {
    if constexpr (NW > 1) __syncthreads();
    else asm volatile("" ::: "memory");
  };
  const Tok tk = tok[t];
  const int pos = __builtin_amdgcn_readfirstlane(tk.pos);
  uint16_t* dst = out + (size_t)t * kQS + 2 * g * kD;  // both heads: 256 contiguous values
  if (!__builtin_amdgcn_readfirstlane(tk.valid)) {
    if (tid < 64) *reinterpret_cast<uint2*>(dst + 4 * tid) = make_uint2(0, 0);
    return;
  }
  const size_t base = cache_base(c, tk, L, g);
  const uint16_t* kc = c.k + base + 8 * t16;
  const uint16_t* vc = c.v + base + 8 * t16;
  u32x4 qv[2];
#pragma unroll
  for (int h = 0; h < 2; h++) qv[h] = ld16(Q + (size_t)t * kQS + (2 * g + h) * kD + 8 * t16);
  const int nch = pos / CAP + 1;
  // rows p + R j of the chunk from c0 (past the token's position: its own row)
  auto rows = [&](const uint16_t* x, int c0, int p, u32x4 (&r)[U]) {
#pragma unroll
    for (int j = 0; j < U; j++) r[j] = ld16(x + (size_t)min(c0 + p + R * j, pos) * kD);
  };
  auto scores = [&](int c0, int n) {
    for (int p = 4 * w + slot; p - slot < n; p += R * U) {
      u32x4 kx[U];
      rows(kc, c0, p, kx);
#pragma unroll
      for (int j = 0; j < U; j++) {
        const float s0 = row16_sum(dot8(kx[j], qv[0], 0.f)), s1 = row16_sum(dot8(kx[j], qv[1], 0.f));
        if (t16 < 2 && p + R * j < n) lds.sc[t16][p + R * j] = bf16r(bf16r(t16 ? s1 : s0) * scale);
      }
    }
  };
  float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};  // of this thread's positions
  for (int ch = 0; ch < nch; ch++) {
    const int c0 = ch * CAP, n = min(pos + 1 - c0, CAP);
    sync();  // what was in LDS before these scores is read
    scores(c0, n);
    sync();
#pragma unroll
    for (int h = 0; h < 2; h++) {
      float mx = m[h], e = 0.f;
      for (int k = tid; k < n; k += NT) mx = fmaxf(mx, lds.sc[h][k]);
      for (int k = tid; k < n; k += NT) {
        const float s = lds.sc[h][k];
        e += s == -INFINITY ? 0.f : exp_acc(s - mx);
      }
      l[h] = (m[h] == -INFINITY ? 0.f : l[h] * exp_acc(m[h] - mx)) + e;
      m[h] = mx;
    }
  }
  u32x4 vx[U];
  rows(vc, 0, 4 * w + slot, vx);  // the first rows of V, behind the reduction
  float M[2], inv[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    M[h] = wave_max_all(m[h]);
    inv[h] = wave_total(m[h] == -INFINITY ? 0.f : l[h] * exp_acc(m[h] - M[h]));
    if constexpr (NW > 1) {
      if (lane == 0) lds.ml[w][h] = make_float2(M[h], inv[h]);
    }
  }
  if constexpr (NW > 1) {
    sync();
#pragma unroll
    for (int h = 0; h < 2; h++) {
      M[h] = -INFINITY;
      for (int q = 0; q < NW; q++) M[h] = fmaxf(M[h], lds.ml[q][h].x);
      inv[h] = 0.f;
      for (int q = 0; q < NW; q++) {
        const float2 e = lds.ml[q][h];
        inv[h] += e.x == -INFINITY ? 0.f : e.y * exp_acc(e.x - M[h]);
      }
    }
  }
#pragma unroll
  for (int h = 0; h < 2; h++) inv[h] = __fdiv_rn(1.0f, inv[h]);
  float acc[2][8];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int e = 0; e < 8; e++) acc[h][e] = 0.f;
  for (int ch = 0; ch < nch; ch++) {
    const int c0 = ch * CAP, n = min(pos + 1 - c0, CAP);
    if (nch > 1) {
      sync();
      scores(c0, n);
      sync();
    }
    for (int k = tid; k < n; k += NT) {
      lds.sc[0][k] = bf16r(exp_acc(lds.sc[0][k] - M[0]) * inv[0]);
      lds.sc[1][k] = bf16r(exp_acc(lds.sc[1][k] - M[1]) * inv[1]);
    }
    sync();
    for (int p = 4 * w + slot; p - slot < n; p += R * U) {
      if (ch || p >= R) rows(vc, c0, p, vx);
#pragma unroll
      for (int j = 0; j < U; j++) {
        // rows past the chunk's positions count as zeros (their row repeats one that may hold an infinity)
        const bool live = p + R * j < n;
        const float p0 = live ? lds.sc[0][p + R * j] : 0.f, p1 = live ? lds.sc[1][p + R * j] : 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t v = live ? vx[j][e] : 0u;
          acc[0][2 * e] = __builtin_fmaf(p0, lo_bf16(v), acc[0][2 * e]);
          acc[0][2 * e + 1] = __builtin_fmaf(p0, hi_bf16(v), acc[0][2 * e + 1]);
          acc[1][2 * e] = __builtin_fmaf(p1, lo_bf16(v), acc[1][2 * e]);
          acc[1][2 * e + 1] = __builtin_fmaf(p1, hi_bf16(v), acc[1][2 * e + 1]);
        }
      }
    }
  }
  // the wave's four lane rows, then the waves in order
#pragma unroll
  for (int h = 0; h < 2; h++) {
#pragma unroll
    for (int e = 0; e < 8; e++) acc[h][e] = rows_sum4(acc[h][e]);
    if (lane < 16) {
      if constexpr (NW > 1) {
        *reinterpret_cast<f32x4*>(&lds.pv[w][h][8 * t16]) = f32x4{acc[h][0], acc[h][1], acc[h][2], acc[h][3]};
        *reinterpret_cast<f32x4*>(&lds.pv[w][h][8 * t16 + 4]) = f32x4{acc[h][4], acc[h][5], acc[h][6], acc[h][7]};
      } else {
        *reinterpret_cast<u32x4*>(dst + h * kD + 8 * t16) =
            u32x4{pack_bf16x2(acc[h][0], acc[h][1]), pack_bf16x2(acc[h][2], acc[h][3]),
                  pack_bf16x2(acc[h][4], acc[h][5]), pack_bf16x2(acc[h][6], acc[h][7])};
      }
    }
  }
  if constexpr (NW > 1) {
    sync();
    if (threadIdx.x < 2 * kD) {
      float y = 0.f;
#pragma unroll
      for (int q = 0; q < NW; q++) y += (&lds.pv[q][0][0])[threadIdx.x];
      dst[threadIdx.x] = (uint16_t)f32_to_bf16(y);
    }
  }
}

// The tokens that are in no tile (hdr[1] of them), shared by the NW-wave workgroups of the launch: a
// workgroup per (token, KV head), but a wave where more than kLeftFew of them lie below kLeftWave (a
// workgroup's barriers cost more than such a context: 130 runs of 3 tokens from position 0, 475 us by
// workgroups, 344 by waves; 256 tokens at 100..2000, 56 of them below 512, 1226 and 1303).  The workgroups that
// take KV head g sit on one XCD, so tokens of one sequence share its L2.
// Against one wave per (token, query head), four positions at a time, us per 4-layer forward, and against
// the separate launch of attention_rows that this replaces in turn: 256 sequences' tokens at 100..2000
// 4220, 1570, now 1226; 400 of a prompt with 100 sequences' tokens at 1000..3000 6030, 2685, 1138; 100 runs
// of 4 after 300 987, 735, 618; two prompts of 512 token by token 2110, 778, 900, of 200 after 2000 5410,
// 2590, 1510.
constexpr int kLeftFew = 128;
template <int NW, int CAP>
__device__ __forceinline__ void attention_left(const uint16_t* __restrict__ Q, const Tok* __restrict__ tok, int T, int L,
                                               const Cache& c, float scale, uint16_t* __restrict__ out,
                                               const AttnPlan& pl, unsigned char* smem) {
  const int nleft = pl.hdr[1], far = pl.hdr[4], near = nleft - far;
  if (nleft == 0) return;
  const int wg = blockIdx.x + gridDim.x * blockIdx.y, g = wg & 7, step = gridDim.x * gridDim.y / 8;
  auto at = [&](int i) { return __builtin_amdgcn_readfirstlane(pl.left[i]); };
  LeftLds<NW, CAP>& all = *reinterpret_cast<LeftLds<NW, CAP>*>(smem);
  for (int i = wg >> 3; i < far; i += step) left_row<NW, CAP>(Q, tok, at(T - 1 - i), g, L, c, scale, out, all);
  if (near <= kLeftFew) {
    // (from the workgroups that the far ones leave free)
    for (int i = (wg >> 3) + (step - far % step); i < near + step; i += step) {
      if (i >= step) left_row<NW, CAP>(Q, tok, at(i - step), g, L, c, scale, out, all);
    }
  } else if (near) {
    __syncthreads();
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    LeftLds<1, kLeftWave>& own = reinterpret_cast<LeftLds<1, kLeftWave>*>(smem)[w];
    for (int i = (wg >> 3) + step * w; i < near; i += step * NW)
      left_row<1, kLeftWave>(Q, tok, at(i), g, L, c, scale, out, own);
  }
}

// Prompt prefill attention on MFMA, over tiles of up to kQT consecutive tokens of a sequence (AttnPlan).
// A tile's query rows of one head share each block of cached keys and values, staged through LDS.  Two
// passes over the keys, as HF's eager softmax: pass 1 gives each row's max M and sum L of exp(s - M)
// (online per lane over the blocks, then across lanes and the waves of a row group); pass 2
// recomputes the scores, rounds the probabilities bf16(exp(s - M) / L) and multiplies them with V on
// MFMA.  Scores are bf16(bf16(q.k) * scale), as in attention_rows.  The tokens that are in no tile follow
// after the tiles (attention_left).
//
// MFMA 16x16x32 bf16 layout: lane l supplies A[l%16][8(l/16)..+7] and B[8(l/16)..+7][l%16] and receives
// C[4(l/16)+i][l%16].  A wave owns 16 query rows of the tile and 32 keys of every block.  Scores are
// computed transposed (A = 16 keys' K rows, B = the rows' q), so lane (l16, lg) holds row l16's scores
// of keys 16n + 4lg + i, i = 0..3: every lane carries one query row.  P@V takes A = those
// probabilities straight from the registers: the 8 k-slots 8lg..8lg+7 of a 32-key step are keys
// 4lg..4lg+3 and 16+4lg..16+4lg+3 of the wave's keys, and V's operand has to come in that order.  The
// waves of a row group add their P@V partials through LDS at the end (in a fixed order).
//
// The kernels share that plan.  attention_mfma walks each tile's whole context: 16 workgroups of 16 waves
// per head (one per CU) share the head's tiles, in order of their keys, so that each walks about as many
// (the last tile of a prompt alone has twice the average).  Where that leaves CUs idle, few tiles over
// a long context, the keys are split into chunks (attention_mfma_pass1, _pass2, _merge below).

// Transposed LDS read (gfx950): 16 lanes read four rows of 16 columns (bf16), 8 bytes each, and lane i
// receives the four rows' values of column i
__device__ __forceinline__ uint2 lds_read_tr4(const unsigned char* p) {
  typedef short short4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) short4_t* lds_t;
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)p));
}

// Blocks of 128 keys, four waves per row group, K and V straight from global memory into LDS: V stays
// row-major there and is transposed by the reads.  What bounds it is the latency of a block's chain
// (LDS reads, products, about 100 VALU instructions and 8 exponentials per wave and pass, barrier):
// VALU work fills 57 % of the cycles in which a CU has waves, the MFMAs 16 %.  Against blocks of 64 keys and 8
// waves (two per SIMD, staged through registers, V transposed on the way into LDS), per 4-layer
// forward, Qwen3-0.6B, us: 768 tokens 459 -> 448, 1024 529 -> 510, 2048 845 -> 805-821.  Measured on the
// way: 8 waves and two workgroups per CU 85 us per layer at 2048 tokens, 8 waves and four stages 92,
// this form with the heads in the grid's second dimension 80, as it is 76.
__global__ void __launch_bounds__(1024) attention_mfma(const uint16_t* __restrict__ Q, const Tok* __restrict__ tok, int T,
                                                       int L, Cache c, float scale, uint16_t* __restrict__ out, AttnPlan pl) {
  constexpr int KQ = 4, NW = 4 * KQ, KB = 32 * KQ;  // key parts of a block, waves, keys per block
  static_assert(kNQ == 16 && kNKV == 8, "two query heads per KV head and XCD");
  static_assert(kQT == 64, "4 row groups of 16 x KQ key parts of 32");
  // two stages of a K block and a V block, [KB][kD] each; after the passes the same bytes hold the P@V
  // partials of all key parts but the first [KQ - 1][4 row groups][16 rows][kD] fp32 for the first
  // part's waves to add
  constexpr int kBlk = KB * kD * 2, kStage = 2 * kBlk;
  static_assert(2 * kStage >= (KQ - 1) * 4 * 16 * kD * 4, "the partials fit in the stages");
  __shared__ __align__(1024) unsigned char smem[2 * kStage];
  __shared__ float s_ml[4][KQ][16][2];  // (max, sum) per row group, key part and row
  auto red = reinterpret_cast<float(*)[4][16][kD]>(smem);
  const int nt = pl.hdr[0];
  // workgroups go to the eight XCDs in turn, so those of KV head g (query heads 2g, 2g+1) share XCD g's
  // L2: its K and V, read by every tile, stay there (with the heads in the grid's second dimension each
  // XCD read all of them)
  const int h = (((int)blockIdx.x & 7) << 1) | ((int)blockIdx.x >> 3), g = h >> 1, by = blockIdx.y;
  // the wave index made uniform, so that branches on the wave's rows and keys are scalar
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15,
            lg = lane >> 4;
  const int rg = w / KQ, kh = w % KQ;  // rows 16rg..16rg+15, keys 32kh..32kh+31 of each block
  // of the tiles in order of their keys, workgroup by of S takes by, 2S - 1 - by, 2S + by, 4S - 1 - by, ..
  const int S = gridDim.y;
  for (int u = 0; u * S < nt; u++) {
    const int ti = u * S + (u & 1 ? S - 1 - by : by);
    if (ti >= nt) continue;  // uniform over the workgroup
    const int4 tl = pl.tile[ti];
    const int t0 = __builtin_amdgcn_readfirstlane(tl.x), nrows = __builtin_amdgcn_readfirstlane(tl.y);
    const int pos0 = __builtin_amdgcn_readfirstlane(tl.z), pmax = pos0 + nrows - 1;
    const Tok first{0, __builtin_amdgcn_readfirstlane(tl.w), pos0, 1};
    const size_t base = cache_base(c, first, L, g);
    const uint16_t* kc = c.k + base;
    const uint16_t* vc = c.v + base;
    const int rpos = pos0 + 16 * rg + l16;      // this lane's row position
    const int wave_first = pos0 + 16 * rg;      // the wave's smallest row position
    const int wave_last = pos0 + 16 * rg + 15;  // the wave's largest row position
    const int nkb = (pmax + KB) / KB;         // blocks covering positions 0..pmax
    // Block kb: positions kb*KB + r; rows past pmax repeat row pmax (masked below).  Wave w moves rows
    // 8w..8w+7 straight into LDS, four rows (1 KB) per instruction; lane l fills position l % 16 of
    // row l / 16.  K: 16-byte chunk c of row r at position c ^ (r & 7), so the lanes that read one chunk
    // of 8 consecutive rows meet every bank once.  V: the 32-byte pairs of chunks at pair ^ (r & 7),
    // for the transposed reads, which take 32 bytes of 8 consecutive rows per 32 lanes.
    const int drow = 8 * w + lg;  // and + 4
    auto issue = [&](int kb, int st, bool v) {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const int r = drow + 4 * q;
        const size_t row = (size_t)min(kb * KB + r, pmax) * kD;
        unsigned char* dst = smem + st * kStage + (8 * w + 4 * q) * (kD * 2);
        dma16(kc + row + 8 * (l16 ^ (r & 7)), dst);
        if (v) dma16(vc + row + 8 * ((((l16 >> 1) ^ (r & 7)) << 1) | (l16 & 1)), dst + kBlk);
      }
    };
    // the blocks in the order in which they are used, those of pass 1, then those of pass 2, each
    // requested while the one before it is at hand
    auto request = [&](int it) {
      if (it < 2 * nkb) issue(it < nkb ? it : it - nkb, it & 1, it >= nkb);
    };
    request(0);
    // B operands: this lane's query row (rows past the tile's tokens repeat its last one)
    const int tq = t0 + min(16 * rg + l16, nrows - 1);
    bf16x8 qb[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) qb[kk] = ld_bf16x8(Q + (size_t)tq * kQS + h * kD + 32 * kk + 8 * lg);
    // raw q.k of row l16 with keys kb*KB + 32kh + 16n + 4lg + i
    auto tile_scores = [&](int st, int n) {
      const unsigned char* kr = smem + st * kStage + (32 * kh + 16 * n + l16) * (kD * 2);
      f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 4; kk++)
        sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16x8*>(kr + 16 * ((4 * kk + lg) ^ (l16 & 7))), qb[kk], sc, 0, 0, 0);
      return sc;
    };
    // the four scores bf16(bf16(q.k) * scale), two roundings per conversion; no branch per
    // element (the callers mask by select), so the four chains interleave
    auto scaled = [&](const f32x4& sc, float (&x)[4]) {
      const uint32_t r01 = pack_bf16x2(sc[0], sc[1]), r23 = pack_bf16x2(sc[2], sc[3]);
      const uint32_t s01 = pack_bf16x2(lo_bf16(r01) * scale, hi_bf16(r01) * scale);
      const uint32_t s23 = pack_bf16x2(lo_bf16(r23) * scale, hi_bf16(r23) * scale);
      x[0] = lo_bf16(s01);
      x[1] = hi_bf16(s01);
      x[2] = lo_bf16(s23);
      x[3] = hi_bf16(s23);
    };
    int it = 0;  // the block at hand
    auto walk = [&](auto&& f) {  // f(block, stage) for each block of a pass
      for (int kb = 0; kb < nkb; kb++, it++) {
        ring_barrier<0>();  // the block has landed in every wave, and the other stage is read
        request(it + 1);
        f(kb, it & 1);
      }
    };
    // ---- pass 1: per lane, online max and sum of exp over its positions (one exp per score,
    // one rescale per block)
    float m = -INFINITY, ls = 0.f;
    walk([&](int kb, int stg) {
      const int kbase = kb * KB + 32 * kh;
      if (kbase > wave_last) return;  // every key of the wave's part follows its rows
      // MASKED: the part reaches the causal diagonal of the wave's rows (the last one or two
      // blocks of a tile); every earlier key precedes every row, so neither the mask nor the
      // clamp of exp_acc is needed (exp_finite gives the same values for finite arguments)
      auto block = [&](auto masked) {
        constexpr bool MASKED = decltype(masked)::value;
        float x[2][4];
        float mb = -INFINITY;
#pragma unroll
        for (int n = 0; n < 2; n++) {
          const f32x4 sc = !MASKED || kbase + 16 * n <= wave_last ? tile_scores(stg, n) : f32x4{0.f, 0.f, 0.f, 0.f};
          scaled(sc, x[n]);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            if constexpr (MASKED) x[n][i] = kbase + 16 * n + 4 * lg + i <= rpos ? x[n][i] : -INFINITY;
            mb = fmaxf(mb, x[n][i]);
          }
        }
        // no branch: while every key so far is masked for this lane's row (mn = -inf) the terms
        // are taken against 0, and exp_acc turns -inf into 0, so ls stays 0
        const float mn = fmaxf(m, mb);
        const float ref = MASKED && mn == -INFINITY ? 0.f : mn;
        float e = 0.f;
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
          for (int i = 0; i < 4; i++) e += MASKED ? exp_acc(x[n][i] - ref) : exp_finite(x[n][i] - ref);
        ls = ls * exp_acc(m - ref) + e;
        m = mn;
      };
      if (kbase + 31 <= wave_first) block(std::false_type{});
      else block(std::true_type{});
    });
    // row l16's (max, sum): over the 4 lanes of equal l16, then the row group's waves (in the
    // same order in each, so they hold the same M and 1/L)
    {
      float mx = m;
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      float sm = m == -INFINITY ? 0.f : ls * exp_acc(m - mx);
      sm += __shfl_xor(sm, 16);
      sm += __shfl_xor(sm, 32);
      if (lg == 0) {
        s_ml[rg][kh][l16][0] = mx;
        s_ml[rg][kh][l16][1] = sm;
      }
    }
    __syncthreads();
    float qm[KQ], ql[KQ];
#pragma unroll
    for (int q = 0; q < KQ; q++) {
      qm[q] = s_ml[rg][q][l16][0];
      ql[q] = s_ml[rg][q][l16][1];
    }
    float gm = qm[0];
#pragma unroll
    for (int q = 1; q < KQ; q++) gm = fmaxf(gm, qm[q]);
    float sm = 0.f;
#pragma unroll
    for (int q = 0; q < KQ; q++) sm += qm[q] == -INFINITY ? 0.f : ql[q] * exp_acc(qm[q] - gm);
    const float ginv = __fdiv_rn(1.0f, sm);
    // ---- pass 2: probabilities (bf16, as HF rounds them) times V
    f32x4 acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    walk([&](int kb, int stg) {
      const int kbase = kb * KB + 32 * kh;
      if (kbase > wave_last) return;
      // A operand: k-slot 4n + i of this lane is key kbase + 16n + 4lg + i of row l16
      uint32_t pw[4];
      auto probs = [&](auto masked) {  // MASKED as in pass 1
        constexpr bool MASKED = decltype(masked)::value;
#pragma unroll
        for (int n = 0; n < 2; n++) {
          // a 16-key tile wholly past the wave's rows is masked for every row: no MFMA for it
          const f32x4 sc = !MASKED || kbase + 16 * n <= wave_last ? tile_scores(stg, n) : f32x4{0.f, 0.f, 0.f, 0.f};
          float x[4], pr[4];
          scaled(sc, x);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            // the probability bf16(exp(s - M) / L) (rounded once, by the packing below); masked
            // keys, whose terms may be anything, take 0
            if constexpr (MASKED) pr[i] = kbase + 16 * n + 4 * lg + i <= rpos ? exp_acc(x[i] - gm) * ginv : 0.f;
            else pr[i] = exp_finite(x[i] - gm) * ginv;
          }
          pw[2 * n] = pack_bf16x2(pr[0], pr[1]);
          pw[2 * n + 1] = pack_bf16x2(pr[2], pr[3]);
        }
      };
      if (kbase + 31 <= wave_first) probs(std::false_type{});
      else probs(std::true_type{});
      const bf16x8 pa = __builtin_bit_cast(bf16x8, u32x4{pw[0], pw[1], pw[2], pw[3]});
      // B operand: dim 16j + l16 of those keys.  A transposed read gives each lane of a group of 16 four
      // consecutive rows' values of its own column; lane i of the group points at row i / 4, columns
      // 4 (i % 4)..+3
      const int vr = 32 * kh + 4 * lg + (l16 >> 2);
      const unsigned char* vrow = smem + stg * kStage + kBlk + vr * (kD * 2) + 8 * (l16 & 3);
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int o = 32 * (j ^ (vr & 7));  // rows vr and vr + 16 swizzle alike
        const uint2 lo = lds_read_tr4(vrow + o), hi = lds_read_tr4(vrow + o + 16 * kD * 2);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa, __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y}),
                                                         acc[j], 0, 0, 0);
      }
    });
    // the row group's partials: all but the first wave's through LDS (over the stages), added to the first
    // wave's in order
    ring_barrier<0>();
    if (kh != 0) {
#pragma unroll
      for (int j = 0; j < 8; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[kh - 1][rg][4 * lg + i][16 * j + l16] = acc[j][i];
    }
    __syncthreads();
    if (kh == 0) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int r = 16 * rg + 4 * lg + i;
        if (r < nrows) {
          uint16_t* dst = out + (size_t)(t0 + r) * kQS + h * kD;
#pragma unroll
          for (int j = 0; j < 8; j++) {
            const int d = 16 * j + l16;
            float y = acc[j][i];
#pragma unroll
            for (int q = 0; q < KQ - 1; q++) y += red[q][rg][4 * lg + i][d];
            dst[d] = (uint16_t)f32_to_bf16(y);
          }
        }
      }
    }
    __syncthreads();  // the partials are read before the next tile's first block
  }
  static_assert(sizeof(LeftLds<NW, 8192>) <= sizeof(smem) && NW * sizeof(LeftLds<1, kLeftWave>) <= sizeof(smem),
                "the left tokens' arrays fit in the stages");
  attention_left<NW, 8192>(Q, tok, T, L, c, scale, out, pl, smem);
}

// Blocks of kKB = 64 keys and workgroups of 8 waves, two per row group.  The split passes take the keys in
// chunks of ck blocks, one workgroup per (tile, chunk, query head): kAttnPass1 (attention_mfma_pass1)
// writes each row's (max, sum) of its chunk to ml; kAttnPass2 (attention_mfma_pass2) takes every chunk's
// (max, sum) of its rows (in chunk order) for the global max M and sum L, and writes its chunk's P@V
// partial (fp32) to part; attention_mfma_merge adds the partials in chunk order.  Workgroups of chunks
// past a tile's last key do nothing.  A call of many part tiles takes one chunk per tile: then the second
// pass writes the output and the merge does nothing.  kAttnFull (attention_mfma_short): both passes over a
// tile's whole context, shared as attention_mfma's, for short contexts.
// K and V go through two register sets, so that a request has two blocks of compute to land, and V is
// transposed on its way into LDS.  For few blocks after a cold start that is the better form:
// attention_mfma's LDS DMA measured, in us per layer, 100 tokens after 6000 positions, pass 1
// 17.0-19.4 against 14.8, pass 2 22.0-25.3 against 21.0 (two and four stages); four prompts of
// 411..613 tokens 46 against 40.
constexpr int kAttnWaves = 8;
enum AttnMode : int { kAttnFull = 0, kAttnPass1 = 1, kAttnPass2 = 2 };

// LDS slot of key q (0..kKB-1) of a block in the transposed V: the order in
// which a wave's P@V k-slots take its keys (see above)
__device__ __forceinline__ int attn_v_slot(int q) {
  const int half = q >> 5, r = q & 31;
  return 32 * half + 8 * ((r & 15) >> 2) + 4 * (r >> 4) + (r & 3);
}

// Index of (tile, head, chunk)'s row block in the split passes' ml and part buffers
__device__ __forceinline__ size_t attn_chunk_row(int tile, int h, int nch, int chunk, int row) {
  return (((size_t)tile * kNQ + h) * nch + chunk) * kQT + row;
}

template <int MODE>
__device__ __forceinline__ void attention_chunk_body(const uint16_t* __restrict__ Q, const Tok* __restrict__ tok, int T,
                                                    int L, Cache c, float scale, uint16_t* __restrict__ out,
                                                    const AttnPlan& pl, float2* __restrict__ ml,
                                                    float* __restrict__ part) {
  constexpr int NT = kAttnWaves * 64;
  static_assert(kQT == 64 && kKB == 64 && kAttnWaves == 8, "4 row groups of 16 x 2 key halves of 32");
  // K block [kKB][kKPad] and transposed V [kD][kVPad]; after the passes the same bytes hold the
  // odd waves' P@V partials [4 row groups][16 rows][kD] fp32 for the even waves to add
  constexpr int kKBytes = kKB * kKPad * 2, kVBytes = kD * kVPad * 2, kRedBytes = 4 * 16 * kD * 4;
  static_assert(kKBytes + kVBytes >= kRedBytes, "the partials fit in the K/V buffers");
  __shared__ __align__(16) unsigned char smem[kKBytes + kVBytes];
  auto Ks = reinterpret_cast<uint16_t(*)[kKPad]>(smem);
  auto Vt = reinterpret_cast<uint16_t(*)[kVPad]>(smem + kKBytes);
  auto Vw = reinterpret_cast<uint32_t(*)[kVPad / 2]>(smem + kKBytes);  // the same rows as 32-bit words
  auto red = reinterpret_cast<float(*)[16][kD]>(smem);
  __shared__ float s_ml[4][2][16][2];  // (max, sum) per row group, key half and row
  const int4 hdr = *reinterpret_cast<const int4*>(pl.hdr);
  const int nch = MODE == kAttnFull ? 1 : hdr.z, ck = hdr.w, items = hdr.x * nch;
  const int h = blockIdx.y, g = h >> 1;
  // the wave index made uniform, so that branches on the wave's rows and keys are scalar
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15,
            lg = lane >> 4;
  const int rg = w >> 1, kh = w & 1;  // rows 16rg..16rg+15, keys 32kh..32kh+31 of each block
  // the (tile, chunk) items are shared as attention_mfma's tiles; with several chunks there are no more
  // of them than workgroups
  const int S = gridDim.x;
  for (int u = 0; u * S < items; u++) {
    const int item = u * S + (u & 1 ? S - 1 - (int)blockIdx.x : (int)blockIdx.x);
    if (item >= items) continue;  // uniform over the workgroup
    const int ti = item / nch, chunk = item % nch;
    const int4 tl = pl.tile[ti];
    const int t0 = __builtin_amdgcn_readfirstlane(tl.x), nrows = __builtin_amdgcn_readfirstlane(tl.y);
    const int pos0 = __builtin_amdgcn_readfirstlane(tl.z), pmax = pos0 + nrows - 1;
    const Tok first{0, __builtin_amdgcn_readfirstlane(tl.w), pos0, 1};
    const size_t base = cache_base(c, first, L, g);
    const uint16_t* kc = c.k + base;
    const uint16_t* vc = c.v + base;
    // B operands: this lane's query row (rows past the tile's tokens repeat its last one)
    const int tq = t0 + min(16 * rg + l16, nrows - 1);
    bf16x8 qb[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) qb[kk] = ld_bf16x8(Q + (size_t)tq * kQS + h * kD + 32 * kk + 8 * lg);
    const int rpos = pos0 + 16 * rg + l16;      // this lane's row position
    const int wave_first = pos0 + 16 * rg;      // the wave's smallest row position
    const int wave_last = pos0 + 16 * rg + 15;  // the wave's largest row position
    const int nkb = (pmax + kKB) / kKB;         // blocks covering positions 0..pmax
    // this workgroup's blocks: all of them, or its chunk's (none past the tile's last key)
    const int kb0 = MODE == kAttnFull ? 0 : chunk * ck, kb1 = MODE == kAttnFull ? nkb : min(kb0 + ck, nkb);
    if (kb0 >= kb1) continue;  // uniform over the workgroup (a chunk past the tile's keys)
    // Block kb: positions kb*kKB + pr; rows past pmax load row pmax (masked below).  Each
    // thread carries kCh 16-byte chunks of K (and of V): block kb+1 is requested into registers
    // before block kb's MFMAs, so its memory latency overlaps them, and written to LDS after
    // the next barrier.
    constexpr int kCh = kKB * (kD / 8) / NT;
    // two register sets: block kb + 2 is requested right after block kb is written to LDS, so a
    // request has two blocks of compute to land
    u32x4 rk[2][kCh], rv[2][kCh];
    auto load_k = [&](int set, int kb) {
#pragma unroll
      for (int j = 0; j < kCh; j++) {
        const int ci = threadIdx.x + NT * j, pr = ci >> 4, col = (ci & 15) * 8;
        rk[set][j] = ld16(kc + (size_t)min(kb * kKB + pr, pmax) * kD + col);
      }
    };
    // V: this thread carries keys 2va and 2va+1 of the block, dims 8vc..8vc+7 (a wave's lanes
    // cover four dim chunks of 16 key pairs), so each transposed LDS word takes both keys' values
    static_assert(kCh == 2, "one key pair per thread");
    const int va = (lane >> 2) + 16 * (w & 1), vcol = 8 * ((lane & 3) + 4 * (w >> 1));
    auto load_v = [&](int set, int kb) {
#pragma unroll
      for (int j = 0; j < 2; j++) rv[set][j] = ld16(vc + (size_t)min(kb * kKB + 2 * va + j, pmax) * kD + vcol);
    };
    auto put_k = [&](int set) {
#pragma unroll
      for (int j = 0; j < kCh; j++) {
        const int ci = threadIdx.x + NT * j, pr = ci >> 4, col = (ci & 15) * 8;
        *reinterpret_cast<u32x4*>(&Ks[pr][col]) = rk[set][j];
      }
    };
    auto put_v = [&](int set) {  // transposed, keys in P@V slot order: Vt[dim][slot]; keys 2va, 2va+1
                                 // take adjacent slots, so each dim is one 32-bit word
      const int sw = attn_v_slot(2 * va) >> 1;
      const u32x4 a0 = rv[set][0], a1 = rv[set][1];
      const uint32_t k0[4] = {a0.x, a0.y, a0.z, a0.w}, k1[4] = {a1.x, a1.y, a1.z, a1.w};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        Vw[vcol + 2 * e][sw] = (k0[e] & 0xffffu) | (k1[e] << 16);
        Vw[vcol + 2 * e + 1][sw] = (k0[e] >> 16) | (k1[e] & 0xffff0000u);
      }
    };
    // raw q.k of row l16 with keys kb*kKB + 32kh + 16n + 4lg + i
    auto tile_scores = [&](int n) {
      f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 4; kk++)
        sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16x8*>(&Ks[32 * kh + 16 * n + l16][32 * kk + 8 * lg]), qb[kk], sc, 0, 0, 0);
      return sc;
    };
    // the four scores bf16(bf16(q.k) * scale), two roundings per conversion; no branch per
    // element (the callers mask by select), so the four chains interleave
    auto scaled = [&](const f32x4& sc, float (&x)[4]) {
      const uint32_t r01 = pack_bf16x2(sc[0], sc[1]), r23 = pack_bf16x2(sc[2], sc[3]);
      const uint32_t s01 = pack_bf16x2(lo_bf16(r01) * scale, hi_bf16(r01) * scale);
      const uint32_t s23 = pack_bf16x2(lo_bf16(r23) * scale, hi_bf16(r23) * scale);
      x[0] = lo_bf16(s01);
      x[1] = hi_bf16(s01);
      x[2] = lo_bf16(s23);
      x[3] = hi_bf16(s23);
    };
    // ---- pass 1: per lane, online max and sum of exp over its positions (one exp per score,
    // one rescale per block)
    float m = -INFINITY, ls = 0.f;
    auto pass1 = [&](int kb) {
      const int kbase = kb * kKB + 32 * kh;
      if (kbase > wave_last) return;  // every key of the wave's half block follows its rows
      // MASKED: the half block reaches the causal diagonal of the wave's rows (the last one or two
      // blocks of a tile); every earlier key precedes every row, so neither the mask nor the
      // clamp of exp_acc is needed (exp_finite gives the same values for finite arguments)
      auto block = [&](auto masked) {
        constexpr bool MASKED = decltype(masked)::value;
        float x[2][4];
        float mb = -INFINITY;
#pragma unroll
        for (int n = 0; n < 2; n++) {
          const f32x4 sc = !MASKED || kbase + 16 * n <= wave_last ? tile_scores(n) : f32x4{0.f, 0.f, 0.f, 0.f};
          scaled(sc, x[n]);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            if constexpr (MASKED) x[n][i] = kbase + 16 * n + 4 * lg + i <= rpos ? x[n][i] : -INFINITY;
            mb = fmaxf(mb, x[n][i]);
          }
        }
        // no branch: while every key so far is masked for this lane's row (mn = -inf) the terms
        // are taken against 0, and exp_acc turns -inf into 0, so ls stays 0
        const float mn = fmaxf(m, mb);
        const float ref = MASKED && mn == -INFINITY ? 0.f : mn;
        float e = 0.f;
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
          for (int i = 0; i < 4; i++) e += MASKED ? exp_acc(x[n][i] - ref) : exp_finite(x[n][i] - ref);
        ls = ls * exp_acc(m - ref) + e;
        m = mn;
      };
      if (kbase + 31 <= wave_first) block(std::false_type{});
      else block(std::true_type{});
    };
    float gm, ginv;
    if constexpr (MODE != kAttnPass2) {
      // blocks past the last one are requested too (clamped rows, never used), so that every path
      // issues the same loads and the compiler's counted waits stay exact
      load_k(0, kb0);
      load_k(1, kb0 + 1);
      for (int kb = kb0; kb < kb1; kb += 2) {
        __syncthreads();  // the previous block's reads are done
        put_k(0);
        __syncthreads();
        load_k(0, kb + 2);
        pass1(kb);
        if (kb + 1 >= kb1) break;
        __syncthreads();
        put_k(1);
        __syncthreads();
        load_k(1, kb + 3);
        pass1(kb + 1);
      }
      // row l16's (max, sum): over the 4 lanes of equal l16, then the row group's two waves (the
      // even wave's pair first in every wave, so both waves hold the same M and 1/L)
      {
        float mx = m;
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        float sm = m == -INFINITY ? 0.f : ls * exp_acc(m - mx);
        sm += __shfl_xor(sm, 16);
        sm += __shfl_xor(sm, 32);
        if (lg == 0) {
          s_ml[rg][kh][l16][0] = mx;
          s_ml[rg][kh][l16][1] = sm;
        }
      }
      __syncthreads();
      const float m0 = s_ml[rg][0][l16][0], l0 = s_ml[rg][0][l16][1];
      const float m1 = s_ml[rg][1][l16][0], l1 = s_ml[rg][1][l16][1];
      gm = fmaxf(m0, m1);
      const float sm = (m0 == -INFINITY ? 0.f : l0 * exp_acc(m0 - gm)) + (m1 == -INFINITY ? 0.f : l1 * exp_acc(m1 - gm));
      if constexpr (MODE == kAttnPass1) {
        // the chunk's (max, sum) of row 16rg + l16 (-inf, 0 when every key of the chunk follows it)
        if (kh == 0 && lg == 0) ml[attn_chunk_row(ti, h, nch, chunk, 16 * rg + l16)] = make_float2(gm, sm);
        continue;
      }
      ginv = __fdiv_rn(1.0f, sm);
    } else {
      // the row's global (max, sum) from its chunks' (chunk 0 holds key 0, so the sum is > 0), the
      // sum in chunk order.  Every chunk's pairs of the tile's rows go to LDS first (over the K/V
      // buffers, unused until the barrier that opens pass 2's first block), in one round of loads.
      const int nc = (nkb + ck - 1) / ck, row = 16 * rg + l16;
      float2* const s_cml = reinterpret_cast<float2*>(smem);  // [nc][kQT]
      static_assert(kMaxAttnChunks * kQT * sizeof(float2) <= kKBytes + kVBytes, "the chunks' pairs fit in LDS");
      for (int i = threadIdx.x; i < nc * kQT; i += NT) s_cml[i] = ml[attn_chunk_row(ti, h, nch, i / kQT, i % kQT)];
      __syncthreads();
      float mx = -INFINITY;
      for (int q = 0; q < nc; q++) mx = fmaxf(mx, s_cml[q * kQT + row].x);
      float sm = 0.f;
      for (int q = 0; q < nc; q++) {
        const float2 e = s_cml[q * kQT + row];
        sm += e.x == -INFINITY ? 0.f : e.y * exp_acc(e.x - mx);
      }
      gm = mx;
      ginv = __fdiv_rn(1.0f, sm);
    }
    // ---- pass 2: probabilities (bf16, as HF rounds them) times V
    f32x4 acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto pass2 = [&](int kb) {
      const int kbase = kb * kKB + 32 * kh;
      if (kbase > wave_last) return;
      // A operand: k-slot 4n + i of this lane is key kbase + 16n + 4lg + i of row l16
      uint32_t pw[4];
      auto probs = [&](auto masked) {  // MASKED as in pass 1
        constexpr bool MASKED = decltype(masked)::value;
#pragma unroll
        for (int n = 0; n < 2; n++) {
          // a 16-key tile wholly past the wave's rows is masked for every row: no MFMA for it
          const f32x4 sc = !MASKED || kbase + 16 * n <= wave_last ? tile_scores(n) : f32x4{0.f, 0.f, 0.f, 0.f};
          float x[4], pr[4];
          scaled(sc, x);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            // the probability bf16(exp(s - M) / L) (rounded once, by the packing below); masked
            // keys, whose terms may be anything, take 0
            if constexpr (MASKED) pr[i] = kbase + 16 * n + 4 * lg + i <= rpos ? exp_acc(x[i] - gm) * ginv : 0.f;
            else pr[i] = exp_finite(x[i] - gm) * ginv;
          }
          pw[2 * n] = pack_bf16x2(pr[0], pr[1]);
          pw[2 * n + 1] = pack_bf16x2(pr[2], pr[3]);
        }
      };
      if (kbase + 31 <= wave_first) probs(std::false_type{});
      else probs(std::true_type{});
      const bf16x8 pa = __builtin_bit_cast(bf16x8, u32x4{pw[0], pw[1], pw[2], pw[3]});
#pragma unroll
      for (int j = 0; j < 8; j++)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            pa, *reinterpret_cast<const bf16x8*>(&Vt[16 * j + l16][32 * kh + 8 * lg]), acc[j], 0, 0, 0);
    };
    load_k(0, kb0);
    load_v(0, kb0);
    load_k(1, kb0 + 1);
    load_v(1, kb0 + 1);
    for (int kb = kb0; kb < kb1; kb += 2) {
      __syncthreads();
      put_k(0);
      put_v(0);
      __syncthreads();
      load_k(0, kb + 2);
      load_v(0, kb + 2);
      pass2(kb);
      if (kb + 1 >= kb1) break;
      __syncthreads();
      put_k(1);
      put_v(1);
      __syncthreads();
      load_k(1, kb + 3);
      load_v(1, kb + 3);
      pass2(kb + 1);
    }
    // the row group's two partials: the odd wave's through LDS (over the K/V buffers), added to
    // the even wave's
    __syncthreads();
    if (kh == 1) {
#pragma unroll
      for (int j = 0; j < 8; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[rg][4 * lg + i][16 * j + l16] = acc[j][i];
    }
    __syncthreads();
    if (kh == 0) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int r = 16 * rg + 4 * lg + i;
        if (r < nrows) {
          if (MODE == kAttnFull || nch == 1) {
            uint16_t* dst = out + (size_t)(t0 + r) * kQS + h * kD;
#pragma unroll
            for (int j = 0; j < 8; j++)
              dst[16 * j + l16] = (uint16_t)f32_to_bf16(acc[j][i] + red[rg][4 * lg + i][16 * j + l16]);
          } else {  // this chunk's fp32 partial of the row
            float* dst = part + attn_chunk_row(ti, h, nch, chunk, r) * kD;
#pragma unroll
            for (int j = 0; j < 8; j++) dst[16 * j + l16] = acc[j][i] + red[rg][4 * lg + i][16 * j + l16];
          }
        }
      }
    }
    if constexpr (MODE == kAttnPass2) __syncthreads();  // the partials are read before the next item's pairs
  }
  if constexpr (MODE != kAttnPass1) {
    static_assert(sizeof(LeftLds<kAttnWaves, 3328>) <= sizeof(smem) &&
                      kAttnWaves * sizeof(LeftLds<1, kLeftWave>) <= sizeof(smem),
                  "the left tokens' arrays fit in the K/V buffers");
    attention_left<kAttnWaves, 3328>(Q, tok, T, L, c, scale, out, pl, smem);
  }
}

#define QMK_ATTN_ARGS                                                                                      \
  const uint16_t *__restrict__ Q, const Tok *__restrict__ tok, int T, int L, Cache c, float scale,                  \
      uint16_t *__restrict__ out, AttnPlan pl, float2 *__restrict__ ml, float *__restrict__ part
// (The second pass held to 128 registers, for two workgroups per CU, spilled 18 and ran slower: 32
// tokens after 7,000 positions 2.57-2.63 against 2.39-2.44 ms per prefill.)
__global__ void __launch_bounds__(kAttnWaves * 64) attention_mfma_short(QMK_ATTN_ARGS) {
  attention_chunk_body<kAttnFull>(Q, tok, T, L, c, scale, out, pl, ml, part);
}
// (six waves per SIMD, three workgroups per CU, for calls of more tile chunks than CUs)
__global__ void __launch_bounds__(kAttnWaves * 64, 6) attention_mfma_pass1(QMK_ATTN_ARGS) {
  attention_chunk_body<kAttnPass1>(Q, tok, T, L, c, scale, out, pl, ml, part);
}
__global__ void __launch_bounds__(kAttnWaves * 64) attention_mfma_pass2(QMK_ATTN_ARGS) {
  attention_chunk_body<kAttnPass2>(Q, tok, T, L, c, scale, out, pl, ml, part);
}
#undef QMK_ATTN_ARGS

// The split passes' output: each row of a tile is the sum of its chunks' partials in chunk order,
// rounded to bf16.  One workgroup of kD threads per (token, query head).
__global__ void __launch_bounds__(kD) attention_mfma_merge(const float* __restrict__ part, AttnPlan pl,
                                                          uint16_t* __restrict__ out) {
  const int t = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
  const int wh = pl.where[t], nch = pl.hdr[2], ck = pl.hdr[3];
  if (wh < 0 || nch == 1) return;  // written by the second pass
  const int tile = wh / kQT, row = wh % kQT;
  const int4 tl = pl.tile[tile];
  const int pmax = tl.z + tl.y - 1;
  const int nc = ((pmax + kKB) / kKB + ck - 1) / ck;
  // eight chunks' loads in flight at a time, added in chunk order
  float y = 0.f;
  for (int q0 = 0; q0 < nc; q0 += 8) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = q0 + j < nc ? part[attn_chunk_row(tile, h, nch, q0 + j, row) * kD + d] : 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (q0 + j < nc) y += v[j];
  }
  out[(size_t)t * kQS + h * kD + d] = (uint16_t)f32_to_bf16(y);
}

// Context-split attention: one token per row of the launch (a batched decode step; a few tokens of a
// prompt), its context in chunks of kSplitChunk positions, one workgroup of 4 waves per (chunk, KV
// head, token), or per every gridDim.x'th chunk (launch_attn_chunks), in HF's two passes over three
// launches:
// - attn_chunk_scores requests the chunk's K rows (a lane row of 16 takes one position, so one wave
//   instruction reads four whole rows), scores them as HF rounds them, stores the scores (fp32)
//   and the chunk's (max m, sum l of exp(s - m)) per head.  RAW: q, k, v come as the q/k/v
//   projection left them; each workgroup forms its q heads (head RMSNorm + RoPE) behind the K
//   requests, and the chunk that holds the token's position also forms its k row, appends K and V
//   and takes its own k from LDS, so no workgroup of the launch reads that cache row (valid only
//   when no other token of the launch is of this sequence).  Otherwise Q is finished and K/V
//   appended by an earlier launch;
// - attn_chunk_pv requests the chunk's V rows, takes the global (M, L) from the chunks' pairs (one
//   pair per lane, the same order in every workgroup of the token), forms the probabilities
//   bf16(exp(s - M) * (1 / L)) one position per lane, and leaves the chunk's P@V partial;
// - attn_chunk_merge adds the partials in a fixed order and rounds to bf16.
// K and V are read once each, so HBM bounds it; what it is held to is that every chunk's rows are
// requested at once (32 KB per workgroup) and that the work per position after the dot products
// (exponentials, rounding) is done by one lane and not by the 16 that share a row.  A fixed chunk
// rather than a fixed number of splits per token keeps the longest sequence of a ragged batch
// from setting the time.  Qwen3-0.6B, us per layer for the three launches, against the forms it
// replaced: 8 sequences of 5..1500 positions 32.3 -> 15.6, 3 of 5000..6100 74.7 -> 21.8, 48 of
// 100..1000 86 -> 35.
template <bool RAW, bool SEVERAL>
__global__ void __launch_bounds__(256) attn_chunk_scores(const uint16_t* __restrict__ src, const Tok* __restrict__ tok,
                                                         int L, const uint16_t* __restrict__ q_norm,
                                                         const uint16_t* __restrict__ k_norm,
                                                         const uint16_t* __restrict__ cos_t,
                                                         const uint16_t* __restrict__ sin_t, Cache c, float eps,
                                                         float scale, int nch, float* __restrict__ scores,
                                                         float2* __restrict__ ml) {
  constexpr int NR = kSplitChunk / 16;  // 16-position rounds, all in flight
  __shared__ float sc[2][kSplitChunk];
  __shared__ __align__(16) uint16_t qs[2][kD], kn[kD];
  __shared__ float wm[4], wl[4];
  const int g = blockIdx.y, t = blockIdx.z, step = gridDim.x;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, slot = lane >> 4,
            t16 = lane & 15;
  const Tok tk = tok[t];
  const int pos = __builtin_amdgcn_readfirstlane(tk.pos);
  int j = blockIdx.x;
  if (!tk.valid || j * kSplitChunk > pos) return;
  const size_t base = cache_base(c, tk, L, g);
  const uint16_t* kc = c.k + base;
  const bool own = RAW && (SEVERAL ? pos / kSplitChunk % step : pos / kSplitChunk) == j;  // this workgroup's chunks hold the token's own position
  u32x4 qv[2];
  // waves 0, 1: q heads 2g, 2g+1; wave 2: k head g; wave 3: v head g
  const int h = w < 2 ? 2 * g + w : (w == 2 ? kNQ + g : kNQ + kNKV + g);
  uint32_t x0b = 0, x1b = 0, w0b = 0, w1b = 0, c0b = 0, c1b = 0, s0b = 0, s1b = 0;
  if constexpr (RAW) {  // a CU returns loads in order, so these go out ahead of the K rows
    const uint16_t* xs = src + (size_t)t * kNQKV + h * kD;
    const uint16_t* nw = w < 2 ? q_norm : k_norm;
    const uint16_t* cr = cos_t + (size_t)pos * kD;
    const uint16_t* sr = sin_t + (size_t)pos * kD;
    x0b = ldu16(xs + lane), x1b = ldu16(xs + lane + 64);
    w0b = ldu16(nw + lane), w1b = ldu16(nw + lane + 64);
    c0b = ldu16(cr + lane), c1b = ldu16(cr + lane + 64);
    s0b = ldu16(sr + lane), s1b = ldu16(sr + lane + 64);
  } else {
#pragma unroll
    for (int hh = 0; hh < 2; hh++) qv[hh] = ld16(src + (size_t)t * kQS + (2 * g + hh) * kD + 8 * t16);
  }
  // positions past the token's own repeat the last one before it (masked below); its own row is not
  // in the cache yet (RAW)
  const int plast = RAW ? max(pos - 1, 0) : pos;
  u32x4 kx[NR];
  auto request = [&](int j) {
#pragma unroll
    for (int r = 0; r < NR; r++)
      kx[r] = ld16(kc + (uint32_t)(min(j * kSplitChunk + 16 * r + 4 * w + slot, plast) * kD + 8 * t16));
  };
  request(j);
  u32x4 k_now = u32x4{0, 0, 0, 0};
  if constexpr (RAW) {
    if (w == 3) {
      if (own) {
        c.v[base + (size_t)pos * kD + lane] = (uint16_t)x0b;
        c.v[base + (size_t)pos * kD + lane + 64] = (uint16_t)x1b;
      }
    } else {
      const float x0 = bf16_to_f32(x0b), x1 = bf16_to_f32(x1b);
      const float ss = wave_sum(x0 * x0 + x1 * x1);
      const float rstd = rcp_sqrt_torch(__fdiv_rn(ss, (float)kD) + eps);
      const float n0 = bf16r(bf16_to_f32(w0b) * bf16r(x0 * rstd));
      const float n1 = bf16r(bf16_to_f32(w1b) * bf16r(x1 * rstd));
      const float cc0 = bf16_to_f32(c0b), cc1 = bf16_to_f32(c1b), ss0 = bf16_to_f32(s0b), ss1 = bf16_to_f32(s1b);
      const uint16_t y0 = (uint16_t)f32_to_bf16(bf16r(bf16r(n0 * cc0) + bf16r(-n1 * ss0)));
      const uint16_t y1 = (uint16_t)f32_to_bf16(bf16r(bf16r(n1 * cc1) + bf16r(n0 * ss1)));
      uint16_t* dst = w < 2 ? qs[w] : kn;
      dst[lane] = y0;
      dst[lane + 64] = y1;
      if (w == 2 && own) {
        c.k[base + (size_t)pos * kD + lane] = y0;
        c.k[base + (size_t)pos * kD + lane + 64] = y1;
      }
    }
    __syncthreads();
#pragma unroll
    for (int hh = 0; hh < 2; hh++) qv[hh] = *reinterpret_cast<const u32x4*>(&qs[hh][8 * t16]);
    k_now = *reinterpret_cast<const u32x4*>(&kn[8 * t16]);
  }
  for (;;) {
    const int c0 = j * kSplitChunk, n = min(pos + 1 - c0, kSplitChunk);
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const int i = 16 * r + 4 * w + slot;
      const u32x4 kr = RAW && c0 + i == pos ? k_now : kx[r];
      const float s0 = row16_sum(dot8(kr, qv[0], 0.f)), s1 = row16_sum(dot8(kr, qv[1], 0.f));
      if (t16 < 2) sc[t16][i] = t16 ? s1 : s0;
    }
    __syncthreads();
    // one (head, position) per thread: the score as HF rounds it, the chunk's maximum and sum
    static_assert(kSplitChunk == 128, "256 threads: 2 heads x 128 positions, two waves per head");
    const int hh = w >> 1, i = threadIdx.x & (kSplitChunk - 1);
    const float s = bf16r(bf16r(sc[hh][i]) * scale);
    if (i < n) scores[((size_t)t * kNQ + 2 * g + hh) * ((size_t)nch * kSplitChunk) + c0 + i] = s;
    const float m = wave_max_all(i < n ? s : -INFINITY);
    const float l = wave_total(i < n && m > -INFINITY ? exp_acc(s - m) : 0.f);
    if (lane == 0) {
      wm[w] = m;
      wl[w] = l;
    }
    __syncthreads();  // (the next chunk's scores may be written; its pairs come after another barrier)
    if (threadIdx.x < 2) {
      const int q = 2 * threadIdx.x;
      const float ma = wm[q], mb = wm[q + 1], mx = fmaxf(ma, mb);
      const float la = ma == -INFINITY ? 0.f : wl[q] * exp_acc(ma - mx);
      const float lb = mb == -INFINITY ? 0.f : wl[q + 1] * exp_acc(mb - mx);
      ml[((size_t)t * kNQ + 2 * g + threadIdx.x) * nch + j] = make_float2(mx, la + lb);
    }
    j += step;
    if (!SEVERAL || j * kSplitChunk > pos) return;
    request(j);
  }
}

template <bool SEVERAL>
__global__ void __launch_bounds__(256) attn_chunk_pv(const Tok* __restrict__ tok, int L, Cache c, int nch,
                                                     const float* __restrict__ scores, const float2* __restrict__ ml,
                                                     float* __restrict__ pvp) {
  constexpr int NR = kSplitChunk / 16;
  __shared__ float pr[2][kSplitChunk];
  __shared__ float wacc[4][2][kD];
  const int g = blockIdx.y, t = blockIdx.z, step = gridDim.x;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, slot = lane >> 4,
            t16 = lane & 15;
  const Tok tk = tok[t];
  const int pos = __builtin_amdgcn_readfirstlane(tk.pos);
  int j = blockIdx.x;
  if (!tk.valid || j * kSplitChunk > pos) return;
  const uint16_t* vc = c.v + cache_base(c, tk, L, g);
  // this thread's score (head w / 2, position i of the chunk) and its head's pairs, then the V rows
  const int hh = w >> 1, i = threadIdx.x & (kSplitChunk - 1), used = pos / kSplitChunk + 1;
  const size_t row = (size_t)t * kNQ + 2 * g + hh;
  const float* sch = scores + row * ((size_t)nch * kSplitChunk);
  float s = sch[min(j * kSplitChunk + i, pos)];
  const float2* mlh = ml + row * nch;
  const float2 first = lane < used ? mlh[lane] : make_float2(-INFINITY, 0.f);
  u32x4 vx[NR];
  auto request = [&](int j) {
#pragma unroll
    for (int r = 0; r < NR; r++)
      vx[r] = ld16(vc + (uint32_t)(min(j * kSplitChunk + 16 * r + 4 * w + slot, pos) * kD + 8 * t16));
  };
  request(j);
  float mx = first.x;
  for (int q = 64 + lane; q < used; q += 64) mx = fmaxf(mx, mlh[q].x);
  mx = wave_max_all(mx);
  float ls = first.x == -INFINITY ? 0.f : first.y * exp_acc(first.x - mx);
  for (int q = 64 + lane; q < used; q += 64) {
    const float2 e = mlh[q];
    ls += e.x == -INFINITY ? 0.f : e.y * exp_acc(e.x - mx);
  }
  const float inv = __fdiv_rn(1.0f, wave_total(ls));
  for (;;) {
    const int n = min(pos + 1 - j * kSplitChunk, kSplitChunk);
    pr[hh][i] = i < n ? bf16r(exp_acc(s - mx) * inv) : 0.f;
    __syncthreads();
    float acc[2][8];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int e = 0; e < 8; e++) acc[q][e] = 0.f;
#pragma unroll
    for (int r = 0; r < NR; r++) {
      const int p = 16 * r + 4 * w + slot;
      // rows past the last position carry probability 0 and a repeated row; taken as zeros, so that
      // an infinity in that row is not counted twice (0 * inf)
      const bool live = p < n;
      const u32x4 vr = u32x4{live ? vx[r].x : 0u, live ? vx[r].y : 0u, live ? vx[r].z : 0u, live ? vx[r].w : 0u};
      const float vf[8] = {lo_bf16(vr.x), hi_bf16(vr.x), lo_bf16(vr.y), hi_bf16(vr.y),
                           lo_bf16(vr.z), hi_bf16(vr.z), lo_bf16(vr.w), hi_bf16(vr.w)};
      const float p0 = pr[0][p], p1 = pr[1][p];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        acc[0][e] = __builtin_fmaf(p0, vf[e], acc[0][e]);
        acc[1][e] = __builtin_fmaf(p1, vf[e], acc[1][e]);
      }
    }
    // the wave's four lane rows, then the four waves in order
#pragma unroll
    for (int q = 0; q < 2; q++) {
#pragma unroll
      for (int e = 0; e < 8; e++) acc[q][e] = rows_sum4(acc[q][e]);
      if (lane < 16) {
        *reinterpret_cast<f32x4*>(&wacc[w][q][8 * t16]) = f32x4{acc[q][0], acc[q][1], acc[q][2], acc[q][3]};
        *reinterpret_cast<f32x4*>(&wacc[w][q][8 * t16 + 4]) = f32x4{acc[q][4], acc[q][5], acc[q][6], acc[q][7]};
      }
    }
    __syncthreads();  // (the next chunk's probabilities may be written; its sums come after another barrier)
    const int d = threadIdx.x & 127, ho = threadIdx.x >> 7;  // 256 threads: both heads' dims
    pvp[(((size_t)t * nch + j) * kNQ + 2 * g) * kD + threadIdx.x] =
        ((wacc[0][ho][d] + wacc[1][ho][d]) + wacc[2][ho][d]) + wacc[3][ho][d];
    j += step;
    if (!SEVERAL || j * kSplitChunk > pos) return;
    s = sch[min(j * kSplitChunk + i, pos)];
    request(j);
  }
}

// The output of (token t, head): its used chunks' partials added, rounded to bf16 (zeros for an invalid
// token).  Thread (q, c4) adds every eighth chunk from q for dims 4c4..+3, then the eight sums in order.
__global__ void __launch_bounds__(256) attn_chunk_merge(const Tok* __restrict__ tok, int nch,
                                                        const float* __restrict__ pvp, uint16_t* __restrict__ out) {
  __shared__ f32x4 part[8][32];
  const int t = blockIdx.x, h = blockIdx.y, q = threadIdx.x >> 5, c4 = threadIdx.x & 31;
  const Tok tk = tok[t];
  const int used = tk.valid ? tk.pos / kSplitChunk + 1 : 0;
  const float* src = pvp + ((size_t)t * nch * kNQ + h) * kD + 4 * c4;
  f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int j = q; j < used; j += 8) y += *reinterpret_cast<const f32x4*>(src + (size_t)j * kQS);
  part[q][c4] = y;
  __syncthreads();
  if (q == 0) {
#pragma unroll
    for (int k = 1; k < 8; k++) y += part[k][c4];
    *reinterpret_cast<uint2*>(out + (size_t)t * kQS + h * kD + 4 * c4) =
        make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
  }
}

// ---------------------------------------------------------------- LM head
//
// The LM head kernels round each logit to bf16, optionally write its fp32 copy, and keep, per row
// and wave or workgroup, the largest key (orderable bf16 logit << 32 | ~index): the first index of
// the maximum, HF's greedy argmax.  keys_reduce then takes each row's largest key; no atomics, so
// the result is independent of scheduling.

__device__ __forceinline__ unsigned long long key_max(unsigned long long a, unsigned long long b) { return a > b ? a : b; }

// lm_head_tiled: the LM head of more than 16 emitted rows.  A persistent grid of two workgroups per
// CU; a workgroup of 4 waves takes the 64-row vocabulary tiles blockIdx.x, + gridDim.x, ... against
// 16 MT emitted rows (blockIdx.y the group of rows), walking them as one sequence of 64-K steps
// through a ring of four LDS stages: both operands go from global memory straight into LDS three
// steps ahead, across tile boundaries, so every weight row is read once per group of rows, in whole
// 128-byte lines, and 48 KB of weights per CU are in flight.  Wave w takes columns 16w..+15 of the
// tile.  Stage rows are swizzled as gemm_tiled's.  Each lane keeps its rows' best (logit, index)
// over its tiles (its columns come in increasing order, so the first of equal logits stays).
// HBM bounds it (311 MB of Qwen3-0.6B weights, plus the fp32 logits).  48 rows: one wave per 16-row
// tile, operands straight from global memory and weights re-read per 16 rows, 187 us -> 76.
constexpr int kLmTileWGs = 512, kLmStages = 4;

template <int MT, int K>
__global__ void __launch_bounds__(256, 2) lm_head_tiled(const uint16_t* __restrict__ X, const int* __restrict__ rows,
                                                        int R, const uint16_t* __restrict__ W, int V,
                                                        unsigned long long* __restrict__ keys_part,
                                                        float* __restrict__ logits) {
  constexpr int AR = MT <= 2 ? 32 : 64;               // emitted rows staged (clamped past R)
  constexpr int NA = AR / 32, NB = 2, KS = K / 64;    // 1 KB DMA blocks (8 rows) per wave and stage
  constexpr int StB = (AR + 64) * 128;
  static_assert(MT <= 4 && 16 * MT <= AR && K % 64 == 0, "row tiles");
  static_assert(kLmStages * StB >= 4 * 16 * MT * 8, "the keys' exchange fits the stages");
  __shared__ __align__(1024) unsigned char sm[kLmStages * StB];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int l16 = lane & 15, lq = lane >> 4;
  const int r0 = blockIdx.y * 16 * MT, ntiles = V / 64, step0 = gridDim.x;
  const int mine = (int)blockIdx.x < ntiles ? (ntiles - (int)blockIdx.x + step0 - 1) / step0 : 0;
  const int nsteps = mine * KS;
  const uint16_t* asrc[NA];
  const uint16_t* bsrc[NB];
#pragma unroll
  for (int q = 0; q < NA; q++) {
    const int row = 8 * (NA * w + q) + (lane >> 3), c = (lane & 7) ^ (row & 7);
    asrc[q] = X + (size_t)max(rows[min(r0 + row, R - 1)], 0) * K + 8 * c;
  }
#pragma unroll
  for (int q = 0; q < NB; q++) {
    const int row = 8 * (NB * w + q) + (lane >> 3), c = (lane & 7) ^ (row & 7);
    bsrc[q] = W + ((size_t)blockIdx.x * 64 + row) * K + 8 * c;
  }
  // steps past the last are requested too (the last one again, into stages no one reads), so that
  // the count of requests in flight is the same at every step
  auto issue = [&](int step) {
    const int sc = min(step, nsteps - 1), k = (sc % KS) * 64;
    const size_t tb = (size_t)(sc / KS) * step0 * 64 * K + k;
    unsigned char* base = sm + (step % kLmStages) * StB;
#pragma unroll
    for (int q = 0; q < NA; q++) dma16(asrc[q] + k, base + 1024 * (NA * w + q));
#pragma unroll
    for (int q = 0; q < NB; q++) dma16(bsrc[q] + tb, base + AR * 128 + 1024 * (NB * w + q));
  };
  f32x4 acc[MT];
  uint32_t bval[MT][4], bidx[MT][4];
#pragma unroll
  for (int i = 0; i < MT; i++) {
    acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; r++) bval[i][r] = 0, bidx[i][r] = 0xffffffffu;
  }
  if (nsteps > 0) {
#pragma unroll
    for (int u = 0; u < kLmStages - 1; u++) issue(u);
  }
  for (int st = 0; st < nsteps; st++) {
    // step st has landed (two younger steps may be in flight) in every wave, and its predecessor's
    // stage is read
    ring_barrier<(kLmStages - 2) * (NA + NB)>();
    issue(st + kLmStages - 1);
    const unsigned char* base = sm + (st % kLmStages) * StB;
#pragma unroll
    for (int kc = 0; kc < 8; kc += 4) {
      const int brow = 16 * w + l16;
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(base + AR * 128 + brow * 128 + 16 * ((kc + lq) ^ (brow & 7)));
#pragma unroll
      for (int i = 0; i < MT; i++) {
        const int row = 16 * i + l16;
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(base + row * 128 + 16 * ((kc + lq) ^ (row & 7)));
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[i], 0, 0, 0);
      }
    }
    if (st % KS == KS - 1) {  // the tile is complete
      const uint32_t n = (uint32_t)(((st / KS) * step0 + blockIdx.x) * 64 + 16 * w + l16);
#pragma unroll
      for (int i = 0; i < MT; i++) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int t = r0 + 16 * i + 4 * lq + r;
          const uint32_t hb = f32_to_bf16(acc[i][r]), o = orderable16(hb);
          if (logits && t < R) logits[(size_t)t * V + n] = bf16_to_f32(hb);
          if (o > bval[i][r] || bidx[i][r] == 0xffffffffu) {
            bval[i][r] = o;
            bidx[i][r] = n;
          }
        }
        acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  // each row's best over the 16 lanes that hold its columns, then over the waves
  ring_barrier<0>();  // the last requests have landed, the last stage is read
  auto red = reinterpret_cast<unsigned long long(*)[16 * MT]>(sm);
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      unsigned long long best = ((unsigned long long)bval[i][r] << 32) | (unsigned long long)(0xffffffffu - bidx[i][r]);
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) best = key_max(best, __shfl_xor(best, o));
      if (l16 == 0) red[w][16 * i + 4 * lq + r] = best;
    }
  __syncthreads();
  const int t = r0 + (int)threadIdx.x;
  if ((int)threadIdx.x < 16 * MT && t < R)
    keys_part[(size_t)t * gridDim.x + blockIdx.x] =
        key_max(key_max(red[0][threadIdx.x], red[1][threadIdx.x]), key_max(red[2][threadIdx.x], red[3][threadIdx.x]));
}

// LM head for at most 16 emitted rows, streamed by a persistent grid: 256
// workgroups of 8 waves; wave g takes the 16-column vocabulary tiles g, g+2048,
// ... (4 or 5 each, so every CU streams within 8% of the mean), walking them as
// one sequence of 64-K steps with kLmDepth steps of weights in flight across
// tile boundaries.  The emitted rows sit in LDS.  Each wave keeps its best key
// per row; keys_reduce takes the best over the 2048 waves.
constexpr int kLmWaves = 8, kLmBlocks = 256, kLmDepth = 4;

__global__ void __launch_bounds__(kLmWaves * 64) lm_head_stream(const uint16_t* __restrict__ X,
                                                                const int* __restrict__ rows, int R,
                                                                const uint16_t* __restrict__ W, int K, int V,
                                                                unsigned long long* __restrict__ keys_part,
                                                                float* __restrict__ logits) {
  extern __shared__ __align__(16) uint16_t xl[];  // [R][K]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int i = threadIdx.x; i < R * K / 8; i += kLmWaves * 64) {
    const int r = (i * 8) / K, k = (i * 8) % K;
    *reinterpret_cast<u32x4*>(xl + r * K + k) = ld16(X + (size_t)max(rows[r], 0) * K + k);
  }
  const int nw = gridDim.x * kLmWaves, gw = blockIdx.x * kLmWaves + wave;
  const int ntiles = V / 16, KS = K / 64;
  const int mine = gw < ntiles ? (ntiles - gw + nw - 1) / nw : 0;
  const int nsteps = mine * KS;
  const int kq = 8 * (lane >> 4);
  const int row = min(lane & 15, R - 1);
  auto wptr = [&](int step) {
    return W + (size_t)((gw + (step / KS) * nw) * 16 + (lane & 15)) * K + kq + (step % KS) * 64;
  };
  bf16x8 buf[kLmDepth][2];
#pragma unroll
  for (int u = 0; u < kLmDepth; u++)
    if (u < nsteps) {
      buf[u][0] = ld_bf16x8_stream(wptr(u));
      buf[u][1] = ld_bf16x8_stream(wptr(u) + 32);
    }
  __syncthreads();
  unsigned long long best[4] = {0, 0, 0, 0};
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < nsteps; s0 += kLmDepth) {
#pragma unroll
    for (int u = 0; u < kLmDepth; u++) {
      const int step = s0 + u;
      if (step < nsteps) {
        const int k = (step % KS) * 64;
        const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(xl + row * K + kq + k);
        const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(xl + row * K + kq + k + 32);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, buf[u][0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, buf[u][1], acc, 0, 0, 0);
        if (step + kLmDepth < nsteps) {
          buf[u][0] = ld_bf16x8_stream(wptr(step + kLmDepth));
          buf[u][1] = ld_bf16x8_stream(wptr(step + kLmDepth) + 32);
        }
        if (step % KS == KS - 1) {  // the tile is complete
          const int n = (gw + (step / KS) * nw) * 16 + (lane & 15);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int t = 4 * (lane >> 4) + i;
            const uint32_t hb = f32_to_bf16(acc[i]);
            if (logits && t < R) logits[(size_t)t * V + n] = bf16_to_f32(hb);
            best[i] = key_max(best[i], ((unsigned long long)orderable16(hb) << 32) |
                                           (unsigned long long)(0xffffffffu - (uint32_t)n));
          }
          acc = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    unsigned long long b = best[i];
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) b = key_max(b, __shfl_xor(b, o));
    const int t = 4 * (lane >> 4) + i;
    if ((lane & 15) == 0 && t < R) keys_part[(size_t)t * nw + gw] = b;
  }
}

// out[r] = token of row r's largest key over the LM head's tiles (-1 for an
// invalid emit row or token).  One workgroup per row.
__global__ void __launch_bounds__(256) keys_reduce(const unsigned long long* __restrict__ keys_part, int ntiles,
                                                   const int* __restrict__ erow, const Tok* __restrict__ tok,
                                                   int* __restrict__ out) {
  __shared__ unsigned long long red[4];
  const int r = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  unsigned long long best = 0;
  for (int i = threadIdx.x; i < ntiles; i += 256) best = key_max(best, keys_part[(size_t)r * ntiles + i]);
  best = wave_max_u64(best);
  if (lane == 0) red[wave] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    best = key_max(key_max(red[0], red[1]), key_max(red[2], red[3]));
    const int e = erow[r];
    out[r] = (e >= 0 && tok[e].valid) ? (int)(0xffffffffu - (uint32_t)best) : -1;
  }
}

// LM head for at most 4 emitted rows with each vocabulary row read whole: one wave instruction
// loads 1 KB of one row (lm_head_stream's MFMA operands take 64 bytes of each of 16 rows per
// instruction, which streams the head at about 5.3 TB/s against about 7 for whole rows).  The same
// persistent grid: wave gw takes vocabulary rows gw, gw + 2048, ..., four rows of weights in
// flight; each lane holds the emitted rows' matching 16-byte chunks in registers and adds its share
// of every dot product with v_dot2; wave_sum8 then finishes eight (vocabulary row, emitted row)
// sums at once, and the lanes that receive them round the logits and keep the best keys.  Keys
// per (emitted row, wave) as lm_head_stream's, for keys_reduce.
template <int R, int K>
__global__ void __launch_bounds__(kLmWaves * 64) lm_head_rows(const uint16_t* __restrict__ X,
                                                              const int* __restrict__ rows, int nrow,
                                                              const uint16_t* __restrict__ W, int V,
                                                              unsigned long long* __restrict__ keys_part,
                                                              float* __restrict__ logits) {
  static_assert(R >= 1 && R <= 4 && K % 512 == 0, "up to four rows, whole 512-element segments");
  constexpr int NS = K / 512;        // 16-byte chunks per lane of one vocabulary row
  constexpr int G = R == 3 ? 2 : 8 / R;  // vocabulary rows per eight-sum reduction
  constexpr int D = 4;               // vocabulary rows in flight (eight: 52.0 against 49.6 us, one 1024-wide row)
  const int lane = threadIdx.x & 63;
  const int nw = gridDim.x * kLmWaves, gw = blockIdx.x * kLmWaves + (threadIdx.x >> 6);
  const int mine = gw < V ? (V - gw + nw - 1) / nw : 0;  // this wave's vocabulary rows
  // the emitted rows' chunks (row r: elements 512 s + 8 lane .. +7 of segment s); rows past nrow
  // repeat the last one and are never written
  u32x4 x[R][NS];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const uint16_t* xr = X + (size_t)max(rows[min(r, nrow - 1)], 0) * K;
#pragma unroll
    for (int sg = 0; sg < NS; sg++) x[r][sg] = ld16(xr + 512 * sg + 8 * lane);
  }
  auto wrow = [&](int i) { return W + (size_t)(gw + nw * min(i, mine - 1)) * K + 8 * lane; };
  u32x4 buf[D][NS];
#pragma unroll
  for (int u = 0; u < D; u++)
#pragma unroll
    for (int sg = 0; sg < NS; sg++) buf[u][sg] = ld_stream(wrow(u) + 512 * sg);
  unsigned long long best = 0;  // lanes 8k: the best key of emitted row k % R
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; k++) v[k] = 0.f;
  // rows past `mine` read the wave's last row again (every path issues the same loads) and are
  // left out of the keys
  for (int i0 = 0; i0 < mine; i0 += 8) {
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = i0 + u, g = u % G;
#pragma unroll
      for (int r = 0; r < R; r++) {
        float acc = 0.f;
#pragma unroll
        for (int sg = 0; sg < NS; sg++) acc = dot8(buf[u % D][sg], x[r][sg], acc);
        v[g * R + r] = acc;
      }
#pragma unroll
      for (int sg = 0; sg < NS; sg++) buf[u % D][sg] = ld_stream(wrow(i + D) + 512 * sg);
      if (g == G - 1) {
        const float sum = wave_sum8(v, lane);  // lanes 8k..8k+7: slot k = (row g', emitted row r)
        const int k = lane >> 3, gk = k / R, rk = k % R;
        const int n = gw + nw * (i - (G - 1) + gk);
        if ((lane & 7) == 0 && k < G * R && i - (G - 1) + gk < mine && rk < nrow) {
          const uint32_t hb = f32_to_bf16(sum);
          if (logits) logits[(size_t)rk * V + n] = bf16_to_f32(hb);
          best = key_max(best, ((unsigned long long)orderable16(hb) << 32) | (unsigned long long)(0xffffffffu - (uint32_t)n));
        }
      }
    }
  }
  // each emitted row's best over its lanes (8k with k % R = r)
#pragma unroll
  for (int r = 0; r < R; r++) {
    unsigned long long b = ((lane & 7) == 0 && (lane >> 3) % R == r && (lane >> 3) < G * R) ? best : 0ull;
    b = wave_max_u64(b);
    if (lane == 0 && r < nrow) keys_part[(size_t)r * nw + gw] = b;
  }
}

// ---------------------------------------------------------------- few tokens
//
// At most kRowsMax tokens (a batched step, a short prompt): the projections run as gemm_rows, whole K
// in one workgroup, with the work between them in their prologues and epilogues.  Per layer:
//
//   gemm_rows<NORM>(q,k,v)   input RMSNorm on the operands, bf16 q|k|v out
//   attention                one token per sequence: attn_chunk_* straight from q|k|v; else
//                            qkv_rows_finish (q/k norm + RoPE, K/V append), then any form
//   gemm_rows(o)             epilogue: residual add into the hidden rows, their squares summed
//   gemm_rows<NORM>(g|u)     post-attention RMSNorm on the operands, SiLU(g)*u out
//   gemm_rows(down)          epilogue as o's
//
// gemm_rows: one workgroup of NW waves per tile of 16 NB output columns (8: HALF, whose MFMA columns
// 8-15 repeat rows 0-7, loads that the same instruction makes anyway: twice the workgroups for the
// narrow o and down) and all T rows (MT MFMA row tiles).  Wave w takes K / NW of the K range: its
// whole weight slice is requested at once, straight from the row-major rows in the MFMA operand
// layout, behind the small loads (vector memory returns in order), and the waves' partial tiles are
// summed in LDS in wave order, so every column is one fp32 sum rounded once.
// RMSNorm needs each row's sum of squares before the product: the kernels that write the hidden rows
// (embed_tokens, the residual epilogues) leave partial sums per 8 columns (ssq[t][H / 8]), a wave
// adds each row's, and every wave normalises its own operands in registers, bf16(w * bf16(x *
// rstd)) as HF; so no workgroup stages whole rows in LDS first.
// It is bound by latency (dispatch, one round trip for rows and weights, two barriers), not by its
// bytes: 4-6 us for the 4-13 MB of a Qwen3-0.6B projection.  Against
// split-K gemm_tiled with finishing kernels (us per forward of 4 layers from position 0): Qwen3-0.6B 8
// tokens 194 -> 175, 16 202 -> 187, 32 211 -> 203; Qwen3-1.7B 8 tokens 332 -> 279, 32 363 -> 339.
// Every workgroup of a NORM product normalises all T rows, so above 32 it loses (48 tokens 224 ->
// 236).
constexpr int kRowsMax = 32;

enum RowEpi : int { kEpiStore = 0, kEpiResidual = 1, kEpiSiluMul = 2 };

// Row of W feeding column `col` of tile `tile` (NC columns): kEpiSiluMul takes
// gate rows in columns 0..NC/2-1 and the up rows of the same NC/2 outputs in
// columns NC/2..NC-1; otherwise the seg rows in order.
template <int EPI, int NC>
__device__ __forceinline__ const uint16_t* tile_row(const Seg& seg, int tile, int col, int K) {
  if (EPI == kEpiSiluMul) {
    const uint16_t* base = col < NC / 2 ? seg.w[0] : seg.w[1];
    return base + (size_t)(tile * (NC / 2) + col % (NC / 2)) * K;
  }
  return seg_row(seg, tile * NC + col, K);
}

// LDS of gemm_rows: the waves' partial tiles of one row tile, and the rows' rstd
template <int MT, int NC, int NW>
constexpr size_t rows_lds() {
  return (size_t)NW * 16 * NC * 4 + 16 * MT * 4;
}

// (four waves per SIMD: one workgroup of 16 waves or two of 8 per CU.  Told no occupancy, the
// compiler splits the requests to fit eight.)
template <int MT, int NB, int EPI, bool NORM, int NW, int K, bool HALF>
__global__ void __launch_bounds__(NW * 64)
    __attribute__((amdgpu_waves_per_eu(4, 4)))
    gemm_rows(const uint16_t* __restrict__ X, const uint16_t* __restrict__ norm_w, const float* __restrict__ ssq_in,
              float eps, int T, Seg seg, uint16_t* __restrict__ Y, int ldy, float* __restrict__ ssq_out) {
  constexpr int ITERS = K / (64 * NW);  // 64-K steps per wave
  constexpr int NC = 16 * NB;
  constexpr int NO = HALF ? 8 : NC;  // product columns per tile
  static_assert(!HALF || (NB == 1 && EPI != kEpiSiluMul), "half tiles: one 16-column MFMA tile, plain rows");
  extern __shared__ __align__(16) unsigned char smem[];
  float (*red)[16][NO] = reinterpret_cast<float (*)[16][NO]>(smem);
  float* rstd_s = reinterpret_cast<float*>(smem + (size_t)NW * 16 * NO * 4);
  const int tile = blockIdx.x, tb = blockIdx.y * 16 * MT;  // rows tb .. tb + 16 MT - 1
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l16 = lane & 15;
  const int kq = 8 * (lane >> 4), k0 = w * (64 * ITERS);
  // the rows' partial sums of squares (row w, w + NW, ..), then this wave's operand rows
  constexpr int NR = NORM ? (16 * MT + NW - 1) / NW : 1;
  constexpr int nss = K / 8;  // partials per row: 128 or 256
  f32x4 sv[NR];
  if constexpr (NORM) {
#pragma unroll
    for (int q = 0; q < NR; q++) {
      const float* sp = ssq_in + (size_t)min(tb + w + NW * q, T - 1) * nss;
      sv[q] = 4 * lane < nss ? *reinterpret_cast<const f32x4*>(sp + 4 * lane) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  u32x4 a[MT][ITERS][2], wn[NORM ? ITERS : 1][2];
#pragma unroll
  for (int it = 0; it < ITERS; it++)
#pragma unroll
    for (int hf = 0; hf < 2; hf++) {
      const int k = k0 + 64 * it + 32 * hf + kq;
      if constexpr (NORM) wn[it][hf] = ld16(norm_w + k);
#pragma unroll
      for (int i = 0; i < MT; i++) a[i][it][hf] = ld16(X + (size_t)min(tb + 16 * i + l16, T - 1) * K + k);
    }
  // this thread's outputs of one row tile (16 rows x OC columns), and their elements of the hidden
  // rows (residual)
  constexpr int OC = EPI == kEpiSiluMul ? NC / 2 : NO;  // output columns per tile
  static_assert(16 * OC <= NW * 64, "one output per thread and row tile");
  const int rt = threadIdx.x / OC, rc = threadIdx.x % OC;
  uint32_t xold[MT];
  if constexpr (EPI == kEpiResidual) {
#pragma unroll
    for (int i = 0; i < MT; i++) xold[i] = ldu16(Y + (size_t)min(tb + 16 * i + rt, T - 1) * ldy + tile * OC + rc);
  }
  bf16x8 b[ITERS][2][NB];
#pragma unroll
  for (int j = 0; j < NB; j++) {
    const uint16_t* wrow = (HALF ? tile_row<EPI, NO>(seg, tile, lane & 7, K)
                                 : tile_row<EPI, NC>(seg, tile, 16 * j + l16, K)) + kq + k0;
#pragma unroll
    for (int it = 0; it < ITERS; it++) {
      b[it][0][j] = ld_bf16x8_stream(wrow + 64 * it);
      b[it][1][j] = ld_bf16x8_stream(wrow + 64 * it + 32);
    }
  }
  if constexpr (NORM) {
#pragma unroll
    for (int q = 0; q < NR; q++) {
      const float ss = wave_sum((sv[q][0] + sv[q][1]) + (sv[q][2] + sv[q][3]));
      if (lane == 0 && w + NW * q < 16 * MT) rstd_s[w + NW * q] = rcp_sqrt_torch(__fdiv_rn(ss, (float)K) + eps);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const float r = rstd_s[16 * i + l16];
#pragma unroll
      for (int it = 0; it < ITERS; it++)
#pragma unroll
        for (int hf = 0; hf < 2; hf++) {
          u32x4 v = a[i][it][hf];
          const u32x4 n = wn[it][hf];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const uint32_t y = pack_bf16x2(lo_bf16(v[e]) * r, hi_bf16(v[e]) * r);
            v[e] = pack_bf16x2(lo_bf16(n[e]) * lo_bf16(y), hi_bf16(n[e]) * hi_bf16(y));
          }
          a[i][it][hf] = v;
        }
    }
  }
  f32x4 acc[MT][NB];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NB; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int it = 0; it < ITERS; it++)
#pragma unroll
    for (int hf = 0; hf < 2; hf++)
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int i = 0; i < MT; i++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[i][it][hf]), b[it][hf][j],
                                                              acc[i][j], 0, 0, 0);
#pragma unroll
  for (int i = 0; i < MT; i++) {  // one row tile at a time through LDS
    if (i) __syncthreads();
    if (!HALF || l16 < 8) {
#pragma unroll
      for (int j = 0; j < NB; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) red[w][4 * (lane >> 4) + r][16 * j + l16] = acc[i][j][r];
    }
    __syncthreads();
    const int t = tb + 16 * i + rt;
    if (rt >= 16) continue;  // whole waves
    auto col_sum = [&](int cc) {
      float y = 0.f;
#pragma unroll
      for (int k = 0; k < NW; k++) y += red[k][rt][cc];  // wave order
      return y;
    };
    uint16_t* dst = Y + (size_t)t * ldy + tile * OC + rc;
    if constexpr (EPI == kEpiSiluMul) {
      const float g = bf16r(col_sum(rc)), u = bf16r(col_sum(rc + NC / 2));
      if (t < T) *dst = (uint16_t)f32_to_bf16(silu_mul(g, u));
    } else if constexpr (EPI == kEpiResidual) {
      const float x = bf16r(bf16_to_f32(xold[i]) + bf16r(col_sum(rc)));
      // 8 columns of row t are 8 neighbouring lanes: one partial sum of squares
      float ss = x * x;
      ss = dpp_add<0xB1>(ss);   // quad_perm [1,0,3,2]
      ss = dpp_add<0x4E>(ss);   // quad_perm [2,3,0,1]
      ss = dpp_add<0x141>(ss);  // row_half_mirror
      if (t < T) {
        *dst = (uint16_t)f32_to_bf16(x);
        if (rc % 8 == 0) ssq_out[(size_t)t * (ldy / 8) + (tile * OC + rc) / 8] = ss;
      }
    } else {
      const float y = col_sum(rc);
      if (t < T) *dst = (uint16_t)f32_to_bf16(y);
    }
  }
}

// q/k norm + RoPE and K/V append from gemm_rows' bf16 q|k|v rows: one wave per (token, head)
__global__ void __launch_bounds__(256) qkv_rows_finish(const uint16_t* __restrict__ QKV, QkvOut o) {
  const int t = blockIdx.x, h = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const uint16_t* x = QKV + (size_t)t * kNQKV + h * kD + lane;
  const uint32_t x0 = ldu16(x), x1 = ldu16(x + 64);
  qkv_head(o, t, h, lane, bf16_to_f32(x0), bf16_to_f32(x1));
}

// ---------------------------------------------------------------- self-test

// C[16][16] = A[16][32] . B[16][32]^T through one MFMA with the operand
// layouts the GEMMs assume.
__global__ void mfma_selftest(const uint16_t* A, const uint16_t* B, float* C) {
  const int lane = threadIdx.x, kq = 8 * (lane >> 4);
  const bf16x8 a = ld_bf16x8(A + (lane & 15) * 32 + kq);
  const bf16x8 b = ld_bf16x8(B + (lane & 15) * 32 + kq);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; i++) C[(4 * (lane >> 4) + i) * 16 + (lane & 15)] = acc[i];
}

// ---------------------------------------------------------------- host side

struct Gemm {
  int ksplit, tn;  // K splits, tile width (128 or 64 columns)
};

// Above kRowsMax tokens every projection of both models takes the LDS-tiled GEMM: N a multiple of the
// 128-column tile and K a multiple of four 64-wide steps.  (A register-staged MFMA GEMM, one wave
// per 16-row tile, ran below 96 tokens before; the tiled kernel on a 128-row tile whose rows past
// T repeat the last one was faster at every count measured: 64 tokens 2.09 -> 1.55 ms per 0.6B
// prefill, 80 tokens 2.43 -> 1.65.)
template <class M>
constexpr bool tiled_shapes() {
  using Dm = Dims<M>;
  constexpr int kStep4 = 4 * kTK;
  return kNQKV % 128 == 0 && Dm::H % 128 == 0 && (2 * Dm::I) % 128 == 0 && Dm::H % kStep4 == 0 &&
         kQS % kStep4 == 0 && Dm::I % kStep4 == 0;
}
static_assert(tiled_shapes<Qwen3_0_6B>() && tiled_shapes<Qwen3_1_7B>(), "projection shapes of the tiled GEMM");

// 128-column tiles: K split (at most 8 ways, >= 4 steps of 64 each) until about 512 workgroups
// run, two per CU.
int tiled_splits(int T, int N, int K) {
  const long long tiles = (long long)((T + kTM - 1) / kTM) * (N / 128);
  int ks = 1;
  while (tiles * ks < 512 && ks < 8 && K % (ks * 2 * 4 * kTK) == 0) ks *= 2;
  return ks;
}

// 64-column tiles, for problems whose 128-column plan leaves CUs idle (narrow N at a few hundred
// rows or fewer): K split (at most 16 ways, >= 2 steps of 64 each) until 256 workgroups run (at 64
// tokens 512 was slower, a prefill 1.535 -> 1.585 ms), while the fp32 partials
// (ksplit * T * N * 4 bytes) stay within twice the weight bytes (N * K * 2).
int narrow_splits(int T, int N, int K) {
  const long long tiles = (long long)((T + kTM - 1) / kTM) * (N / 64);
  int ks = 1;
  while (tiles * ks < 256 && ks * 2 <= kMaxSplit && K % (ks * 2 * kTK) == 0 && K / (ks * 2) >= 2 * kTK &&
         (long long)ks * 2 * T * 4 <= 2LL * K * 2)
    ks *= 2;
  return ks;
}

Gemm plan_gemm(int T, int N, int K) {
  const int ks = tiled_splits(T, N, K);
  const long long wgs = (long long)((T + kTM - 1) / kTM) * (N / 128) * ks;
  if (wgs >= 256) return {ks, 128};
  const int ks64 = narrow_splits(T, N, K);
  if ((long long)((T + kTM - 1) / kTM) * (N / 64) * ks64 > wgs) return {ks64, 64};
  return {ks, 128};
}

// The q/k/v and gate/up GEMMs with their finishing work in the epilogue (kEpiQkv, kEpiGateUp)
// when the plan can leave K unsplit: at least kFuseMinWG 128-column tiles (q/k/v: that many per
// 1024 of K).  Then no fp32 sums go to memory and no finishing kernel runs; *ks_out = 0 says so.
// Otherwise the sums go to part and *ks_out is the split count for the finishing kernel.  With
// half the CUs given a tile, the unsplit GEMM plus its epilogue still beats the split one plus the
// finishing kernel (prefill ms, against a bound of one tile per CU: 0.6B 384 tokens 2.84-2.90 ->
// 2.67-2.74, 512 3.25-3.34 -> 3.01-3.10, 640 3.80-3.88 -> 3.30-3.36, 896 4.08-4.19 -> 3.79-3.88;
// 1.7B 256 tokens 3.47-3.57 -> 3.31-3.38, gate/up on 192 tiles); with a quarter it loses (0.6B
// 256 tokens 2.39-2.45 -> 2.62-2.65, q/k/v on 64 tiles and gate/up on 96), and so does the 1.7B
// q/k/v, whose K of 2048 doubles each tile's work, on 128 and 160 tiles (512 tokens 4.06-4.15
// -> 4.38-4.49, 640 5.10-5.20 -> 5.27-5.37).
constexpr int kFuseMinWG = 128;

void launch_gemm(const uint16_t* X, int T, int K, const Seg& seg, int N, float* part, hipStream_t s, int* ks_out,
                 int epi = kEpiPart, const QkvOut* qo = nullptr, const GateUpOut* go = nullptr) {
  const QkvOut q0 = qo ? *qo : QkvOut{};
  const GateUpOut g0 = go ? *go : GateUpOut{};
  const long long fuse_min = epi == kEpiQkv ? (long long)kFuseMinWG * std::max(1, K / 1024) : kFuseMinWG;
  if (epi != kEpiPart && (long long)((T + kTM - 1) / kTM) * (N / 128) >= fuse_min) {
    const dim3 grid(N / 128, (T + kTM - 1) / kTM, 1);
    if (epi == kEpiQkv)
      hipLaunchKernelGGL((gemm_tiled<128, kEpiQkv>), grid, dim3(256), 0, s, X, T, K, seg, N, 1, part, q0, g0);
    else
      hipLaunchKernelGGL((gemm_tiled<128, kEpiGateUp>), grid, dim3(256), 0, s, X, T, K, seg, N, 1, part, q0, g0);
    *ks_out = 0;
    return;
  }
  const Gemm g = plan_gemm(T, N, K);
  const dim3 grid(N / g.tn, (T + kTM - 1) / kTM, g.ksplit);
  if (g.tn == 128)
    hipLaunchKernelGGL((gemm_tiled<128, kEpiPart>), grid, dim3(256), 0, s, X, T, K, seg, N, g.ksplit, part, q0, g0);
  else
    hipLaunchKernelGGL((gemm_tiled<64, kEpiPart>), grid, dim3(256), 0, s, X, T, K, seg, N, g.ksplit, part, q0, g0);
  *ks_out = g.ksplit;
}

size_t part_floats(int T, int N, int K) { return (size_t)plan_gemm(T, N, K).ksplit * T * N; }

int split_chunks(int max_context) { return (max_context + kSplitChunk - 1) / kSplitChunk; }

// The context-split attention (three launches, each token's context over workgroups of
// kSplitChunk positions) for a batched step and for few tokens over a longer context; the row kernel (one launch) for few tokens over
// a short one (Qwen3-0.6B, 31 tokens after 100 positions: 223 us split against 218 rows per 4-layer
// forward; after 250, 228 against 254).  Its work grows with tokens x context, attention_mfma's with
// the context alone (a 64-token tile costs the same for 1 token as for 64), so a prompt of one
// sequence takes attention_mfma from about 32768 tokens x positions (split against attention_mfma
// with its keys in chunks, us per 4-layer forward: after 700 positions 8 tokens 200 / 225 and 31
// tokens 244 / 251; after 2000, 4 tokens 199 / 228 and 16 tokens 241 / 243; after 6500, 1 token 202
// / 267 and 4 tokens 230 / 271).  A batched decode step (one token per sequence, whose tiles hold
// several sequences and would fall back to the row kernel) takes the split form at any batch: 48
// sequences of 100..1000 positions ran attention_mfma over no tile and then the row kernel, 86 us
// per layer against 35.
constexpr int kSplitWork = 32768;
bool split_attention(int T, int max_context, bool one_per_seq) {
  return max_context > kSplitContext && (one_per_seq || (T < kSplitBelow && (long long)T * max_context < kSplitWork));
}

// attention_mfma pays off from about 320 tokens or 256 positions of context (below that the row
// kernel's per-token reads are cheaper than its passes).  Measured 0.6B prefills, row kernel
// against attention_mfma: 256 tokens 2.55 / 2.62 ms, 384 tokens 3.37 / 3.18, 512 tokens 4.23 /
// 3.67, 768 tokens 5.85 / 4.45; with its keys in chunks (below), after 400 positions: 32 tokens
// 2.01 / 1.78, 256 tokens 3.57 / 2.45; after 950: 64 tokens 3.06 / 1.99.
bool mfma_attention(int T, int max_context, bool one_per_seq) {
  return !one_per_seq && !split_attention(T, max_context, false) &&
         (T >= kMfmaAttnTokens || max_context >= kMfmaAttnContext);
}

// Up to this context attention_mfma_short's smaller blocks win: a tile of five blocks of 128 keys or fewer has
// too little to hide the first one's arrival and the sum of the four key parts behind, and half of its last
// block is past the diagonal (us per 4-layer forward, short against
// the 128-key form: 640 tokens 418 / 416, 768 456 / 452, 1024 526 / 516; four prompts of 411..613 tokens
// 1283 / 1313).
constexpr int kShortAttn = 640;

// attention_mfma's keys in chunks (the split passes) when its tiles would
// leave CUs idle and either the context before the prompt is at least as long as the prompt (a
// prompt of few tiles over a long context, e.g. a new turn appended to a long conversation, where
// each tile's workgroup would walk the whole context alone: Qwen3-0.6B, whole tiles against chunks, 128
// tokens after 7000 positions 13.9 / 2.8 ms, 32 tokens after 4000 4.82 / 1.90) or the prompt has
// at most 8 tiles (from position 0: 384 tokens 2.87-2.90 / 2.82-2.83, 512 tokens 3.32-3.36 /
// 3.24; with more tiles from position 0 the whole tiles balance the causal work as well: 768 tokens
// 3.70-3.74 / 3.75-3.76, 1024 tokens 3.97-4.00 / 3.99).
// Up to 8 tiles, at most kMaxAttnChunks tile chunks, at least two blocks each: 256 workgroups, so
// the second pass (one workgroup per CU) runs in one round (at most 32: 32 tokens after 7,000
// positions 2.39-2.44 against 2.02-2.07 ms per prefill; at most 8: 2.34-2.38).  More tiles take up
// to 4 x kMaxAttnChunks tile chunks, two or more rounds, rather than one chunk each (1024 tokens
// after 4000 positions 10.76 -> 7.56 ms, after 6000 14.05 -> 9.17).  The fp32 partials (32 KB per
// tile chunk and head) stay within 32 MB.  The result is the call's budget of tile chunks (0: whole tiles);
// attn_key_chunks shares it among the tiles that the call turns out to have.
int attn_chunk_budget(int T, int max_context) {
  const int nt = (T + kQT - 1) / kQT, nkb = (max_context + kKB - 1) / kKB;
  if ((nt + 1) / 2 * kNQ >= kNumWG || (max_context < 2 * T && nt > 8)) return 0;
  const int most = nt <= 8 ? kMaxAttnChunks : 4 * kMaxAttnChunks, nch = attn_key_chunks(most, nkb, nt, nt).x;
  // as many as workgroups are launched per head.  Above 8 tiles, which run in several rounds, no more than a
  // single prompt takes: workgroups go to the shader engines in turn, and idle ones among them leave whole
  // engines with less (1500 tokens after 3000 positions, 48 of 64: 1615 us per 4-layer forward against 1370)
  return nch > 1 ? (nt <= 8 ? most : nch * nt) : 0;
}

// Tiles planned for a call: each sequence's run may end in a part tile, up to kMoreTiles of them.
constexpr int kMoreTiles = 255;
int attn_tiles(int T) { return std::min(T, (T + kQT - 1) / kQT + kMoreTiles); }

struct Layout {
  size_t tok, erow, keys, x, n, q, att, m, qkv, ssq, part, scores, ml, pv, plan, mml, mpart, total;
};

template <class M>
Layout layout(int T, int R, int max_context, bool one_per_seq) {
  using Dm = Dims<M>;
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  Layout l{};
  size_t off = 0;
  auto take = [&](size_t& field, size_t bytes) {
    field = off;
    off += al(bytes);
  };
  take(l.tok, (size_t)T * sizeof(Tok));
  take(l.erow, (size_t)R * 4);
  take(l.keys, (size_t)R * kLmBlocks * kLmWaves * 8);
  static_assert(kLmBlocks * kLmWaves >= kLmTileWGs && Dm::V % 64 == 0, "LM head keys and tiles");
  take(l.x, (size_t)T * Dm::H * 2);
  take(l.n, (size_t)T * Dm::H * 2);
  take(l.q, (size_t)T * kQS * 2);
  take(l.att, (size_t)T * kQS * 2);
  take(l.m, (size_t)T * Dm::I * 2);
  if (split_attention(T, max_context, one_per_seq) || (one_per_seq && T <= kRowsMax)) {
    const int nch = split_chunks(max_context);
    take(l.scores, (size_t)T * kNQ * nch * kSplitChunk * 4);
    take(l.ml, (size_t)T * kNQ * nch * 8);
    take(l.pv, (size_t)T * nch * kQS * 4);
  }
  if (T <= kRowsMax) {
    take(l.qkv, (size_t)T * kNQKV * 2);
    take(l.ssq, (size_t)T * (Dm::H / 8) * 4);
  } else {
    size_t pf = part_floats(T, kNQKV, Dm::H);
    pf = std::max(pf, part_floats(T, Dm::H, kQS));
    pf = std::max(pf, part_floats(T, 2 * Dm::I, Dm::H));
    pf = std::max(pf, part_floats(T, Dm::H, Dm::I));
    take(l.part, pf * 4);
  }
  if (mfma_attention(T, max_context, one_per_seq)) {
    // header, tiles twice with their ranks and keys, where, left; then the (max, sum) of the tile chunks or,
    // with one chunk each, of the tiles, and the tile chunks' partials
    take(l.plan, 32 + (size_t)attn_tiles(T) * 32 + (size_t)T * 8);
    if (const int budget = attn_chunk_budget(T, max_context)) {
      take(l.mml, (size_t)std::max(budget, attn_tiles(T)) * kNQ * kQT * sizeof(float2));
      take(l.mpart, (size_t)budget * kNQ * kQT * kD * 4);
    }
  }
  l.total = off;
  return l;
}

struct Args {
  int T, R, num_seqs, max_context;
  bool one_per_seq;  // token t is sequence t's only token (batched decode step)
  const int *tokens, *seqs, *pos, *emit;
  int* out_tokens;
  float* logits;
  const uint16_t *embed, *final_norm, *lm_head, *cos_t, *sin_t;
  const LDGLayerWeights* layers;  // host array
  Cache cache;
  int num_layers;
  float attn_scale;
  char* ws;
};

// LM head + argmax of R emitted rows: whole vocabulary rows for R <= 4, the streamed MFMA form up to
// 16, tiles through LDS above that.
template <class M>
void launch_lm_head(const uint16_t* N, const int* erow, int R, const uint16_t* W, unsigned long long* keys,
                    float* logits, const Tok* tok, int* out, hipStream_t s) {
  using Dm = Dims<M>;
  if (R <= 4) {
    const dim3 grid(kLmBlocks), block(kLmWaves * 64);
    switch (R) {
      case 1: hipLaunchKernelGGL((lm_head_rows<1, Dm::H>), grid, block, 0, s, N, erow, R, W, Dm::V, keys, logits); break;
      case 2: hipLaunchKernelGGL((lm_head_rows<2, Dm::H>), grid, block, 0, s, N, erow, R, W, Dm::V, keys, logits); break;
      case 3: hipLaunchKernelGGL((lm_head_rows<3, Dm::H>), grid, block, 0, s, N, erow, R, W, Dm::V, keys, logits); break;
      default: hipLaunchKernelGGL((lm_head_rows<4, Dm::H>), grid, block, 0, s, N, erow, R, W, Dm::V, keys, logits); break;
    }
    hipLaunchKernelGGL(keys_reduce, dim3(R), dim3(256), 0, s, keys, kLmBlocks * kLmWaves, erow, tok, out);
    return;
  }
  if (R <= 16) {
    const size_t lds = (size_t)R * Dm::H * 2;
    hipLaunchKernelGGL(lm_head_stream, dim3(kLmBlocks), dim3(kLmWaves * 64), lds, s, N, erow, R, W, Dm::H, Dm::V,
                       keys, logits);
    hipLaunchKernelGGL(keys_reduce, dim3(R), dim3(256), 0, s, keys, kLmBlocks * kLmWaves, erow, tok, out);
    return;
  }
  // two workgroups per CU, shared by the groups of up to 64 rows
  const int groups = (R + 63) / 64;
  const dim3 grid(kLmTileWGs / groups, groups);
  if (R <= 32)
    hipLaunchKernelGGL((lm_head_tiled<2, Dm::H>), grid, dim3(256), 0, s, N, erow, R, W, Dm::V, keys, logits);
  else
    hipLaunchKernelGGL((lm_head_tiled<4, Dm::H>), grid, dim3(256), 0, s, N, erow, R, W, Dm::V, keys, logits);
  hipLaunchKernelGGL(keys_reduce, dim3(R), dim3(256), 0, s, keys, (int)grid.x, erow, tok, out);
}

// gemm_rows with RMSNorm over `tiles` tiles of 16 NB product columns, 16 waves: all T rows in every
// workgroup, so the weights are read once
template <int K, int NB, int EPI>
void launch_rows_norm(int tiles, const uint16_t* X, const uint16_t* nw, const float* ssq, float eps, int T,
                      const Seg& seg, uint16_t* Y, int ldy, hipStream_t s) {
  constexpr int NW = 16;
  auto go = [&](auto mt) {
    constexpr int MT = decltype(mt)::value;
    constexpr size_t lds = rows_lds<MT, 16 * NB, NW>();
    static_assert(lds <= 64 * 1024, "the default dynamic LDS limit");
    hipLaunchKernelGGL((gemm_rows<MT, NB, EPI, true, NW, K, false>), dim3(tiles), dim3(NW * 64), lds, s, X, nw, ssq, eps,
                       T, seg, Y, ldy, nullptr);
  };
  if (T <= 16) go(std::integral_constant<int, 1>{});
  else go(std::integral_constant<int, 2>{});
}

// gemm_rows with the residual epilogue into the H columns of X: a workgroup per 16-row tile (a second
// one finds the weights in its XCD's L2) and 8 columns, or 16 where 8 would make more workgroups
// than CUs (one of 16 waves fits; H = 2048, 24 rows, 512 workgroups against 256: o 10.0 -> 6.4
// us, down 22.6 -> 15.2)
template <int K, int H>
void launch_rows_residual(const uint16_t* A, int T, const Seg& seg, uint16_t* X, float* ssq, hipStream_t s) {
  constexpr int NW = 16;
  const int rt = (T + 15) / 16;
  if (rt * (H / 8) <= kNumWG)
    hipLaunchKernelGGL((gemm_rows<1, 1, kEpiResidual, false, NW, K, true>), dim3(H / 8, rt), dim3(NW * 64),
                       (rows_lds<1, 8, NW>()), s, A, nullptr, nullptr, 0.f, T, seg, X, H, ssq);
  else
    hipLaunchKernelGGL((gemm_rows<1, 1, kEpiResidual, false, NW, K, false>), dim3(H / 16, rt), dim3(NW * 64),
                       (rows_lds<1, 16, NW>()), s, A, nullptr, nullptr, 0.f, T, seg, X, H, ssq);
}

// The context-split attention of one layer: RAW from the q/k/v projection's output, else from
// finished q rows.
struct AttnChunks {
  int nch;
  float* scores;
  float2* ml;
  float* pvp;
};
AttnChunks attn_chunks(const Args& a, const Layout& l) {
  return {split_chunks(a.max_context), reinterpret_cast<float*>(a.ws + l.scores),
          reinterpret_cast<float2*>(a.ws + l.ml), reinterpret_cast<float*>(a.ws + l.pv)};
}

// Workgroups of a launch at most: the call's context is a bound that its tokens may lie far below, and a
// workgroup without a chunk still costs 2 ns, so above this each takes several chunks (one step, 4 layers,
// us, one chunk each / several: 128 sequences at 100..200 with a bound of 4096 1010 / 423, of 201 430 both;
// where the bound is the context, 16 sequences at 3000..8000 475 / 500, 32 at 100..7000 563 / 585, 256 at
// 1000..1100 1276 / 1326: a chunk's rows are requested when the one before is done).
// An odd number per (token, head), since workgroups go to the eight XCDs in turn: with eight, every token's
// first chunk falls on the same one (48 sequences at 100..200, bound 4096: 354 us with 8, 300 with 10 and 9).
constexpr int kChunkWGs = 3072;

template <bool RAW>
void launch_attn_chunks(const Args& a, const AttnChunks& ac, const uint16_t* src, const Tok* tok, int L,
                        const LDGLayerWeights& w, float eps, uint16_t* out, hipStream_t s) {
  auto go = [&](auto several, int per_head) {
    constexpr bool SEVERAL = decltype(several)::value;
    const dim3 grid(per_head, kNKV, a.T);
    hipLaunchKernelGGL((attn_chunk_scores<RAW, SEVERAL>), grid, dim3(256), 0, s, src, tok, L,
                       static_cast<const uint16_t*>(w.q_norm_weight), static_cast<const uint16_t*>(w.k_norm_weight),
                       a.cos_t, a.sin_t, a.cache, eps, a.attn_scale, ac.nch, ac.scores, ac.ml);
    hipLaunchKernelGGL(attn_chunk_pv<SEVERAL>, grid, dim3(256), 0, s, tok, L, a.cache, ac.nch, ac.scores, ac.ml,
                       ac.pvp);
  };
  const int most = std::max(1, kChunkWGs / (kNKV * a.T));
  if (ac.nch <= most) go(std::false_type{}, ac.nch);
  else go(std::true_type{}, most - 1 + most % 2);
  hipLaunchKernelGGL(attn_chunk_merge, dim3(a.T, kNQ), dim3(256), 0, s, tok, ac.nch, ac.pvp, out);
}

// The attention plan of a call (cap 0 when its attention takes no tiles); embed_tokens fills it.
AttnPlan attn_plan(const Args& a, const Layout& l) {
  if (!mfma_attention(a.T, a.max_context, a.one_per_seq)) return AttnPlan{};
  const int cap = attn_tiles(a.T);
  int* hdr = reinterpret_cast<int*>(a.ws + l.plan);
  int4* tile = reinterpret_cast<int4*>(hdr + 8);
  int2* raw = reinterpret_cast<int2*>(tile + cap);
  int* rank = reinterpret_cast<int*>(raw + cap);
  int* where = rank + 2 * cap;
  return {hdr,   tile,        raw, rank, rank + cap,
          where, where + a.T, cap, attn_chunk_budget(a.T, a.max_context), (a.max_context + kKB - 1) / kKB};
}

// The attention of one layer whose q rows are finished and K/V appended: the context-split form, the
// MFMA form, or the row kernel.
void launch_attention(const Args& a, const Layout& l, const uint16_t* Q, const Tok* tok, int L,
                      const LDGLayerWeights& w, float eps, uint16_t* ATT, hipStream_t s) {
  const int T = a.T;
  if (split_attention(T, a.max_context, a.one_per_seq)) {
    launch_attn_chunks<false>(a, attn_chunks(a, l), Q, tok, L, w, eps, ATT, s);
    return;
  }
  if (!mfma_attention(T, a.max_context, a.one_per_seq)) {
    hipLaunchKernelGGL(attention_rows, dim3(T, kNKV), dim3(256), 0, s, Q, tok, L, a.cache, a.attn_scale, ATT);
    return;
  }
  const AttnPlan pl = attn_plan(a, l);
  if (pl.budget) {
    float2* aml = reinterpret_cast<float2*>(a.ws + l.mml);
    float* apart = reinterpret_cast<float*>(a.ws + l.mpart);
    const dim3 grid(pl.budget, kNQ);
    hipLaunchKernelGGL(attention_mfma_pass1, grid, dim3(kAttnWaves * 64), 0, s, Q, tok, T, L, a.cache, a.attn_scale,
                       ATT, pl, aml, apart);
    hipLaunchKernelGGL(attention_mfma_pass2, grid, dim3(kAttnWaves * 64), 0, s, Q, tok, T, L, a.cache, a.attn_scale,
                       ATT, pl, aml, apart);
    hipLaunchKernelGGL(attention_mfma_merge, dim3(T, kNQ), dim3(kD), 0, s, apart, pl, ATT);
  } else if (a.max_context <= kShortAttn) {
    hipLaunchKernelGGL(attention_mfma_short, dim3(kNumWG / kNQ, kNQ), dim3(kAttnWaves * 64), 0, s, Q,
                       tok, T, L, a.cache, a.attn_scale, ATT, pl, nullptr, nullptr);
  } else {
    hipLaunchKernelGGL(attention_mfma, dim3(kNQ, kNumWG / kNQ), dim3(1024), 0, s, Q, tok, T, L, a.cache, a.attn_scale,
                       ATT, pl);
  }
}

template <class M>
int forward_rows(const Args& a, hipStream_t s) {
  using Dm = Dims<M>;
  const int T = a.T, R = a.R;
  const Layout l = layout<M>(T, R, a.max_context, a.one_per_seq);
  Tok* tok = reinterpret_cast<Tok*>(a.ws + l.tok);
  int* erow = reinterpret_cast<int*>(a.ws + l.erow);
  auto* keys = reinterpret_cast<unsigned long long*>(a.ws + l.keys);
  uint16_t* X = reinterpret_cast<uint16_t*>(a.ws + l.x);
  uint16_t* N = reinterpret_cast<uint16_t*>(a.ws + l.n);
  uint16_t* Qb = reinterpret_cast<uint16_t*>(a.ws + l.q);
  uint16_t* ATT = reinterpret_cast<uint16_t*>(a.ws + l.att);
  uint16_t* MM = reinterpret_cast<uint16_t*>(a.ws + l.m);
  uint16_t* QKV = reinterpret_cast<uint16_t*>(a.ws + l.qkv);
  float* ssq = reinterpret_cast<float*>(a.ws + l.ssq);
  const float eps = 1e-6f;
  auto u16 = [](const void* p) { return static_cast<const uint16_t*>(p); };
  const AttnPlan pl = attn_plan(a, l);
  hipLaunchKernelGGL((embed_tokens<Dm::H, false>), dim3(T + (pl.cap ? 1 : 0)), dim3(256), 0, s, a.tokens, a.seqs, a.pos,
                     T, a.emit, R, a.num_seqs, a.max_context, Dm::V, a.embed, tok, erow, X, nullptr, eps, nullptr, ssq, pl);
  for (int L = 0; L < a.num_layers; L++) {
    const LDGLayerWeights& w = a.layers[L];
    const Seg qkv{{u16(w.q_proj_weight), u16(w.k_proj_weight), u16(w.v_proj_weight)}, {kQS, kNKV * kD, kNKV * kD}};
    launch_rows_norm<Dm::H, 1, kEpiStore>(kNQKV / 16, X, u16(w.input_layernorm_weight), ssq, eps, T, qkv, QKV, kNQKV, s);
    if (a.one_per_seq) {
      launch_attn_chunks<true>(a, attn_chunks(a, l), QKV, tok, L, w, eps, ATT, s);
    } else {
      const QkvOut qo{tok, L, u16(w.q_norm_weight), u16(w.k_norm_weight), a.cos_t, a.sin_t, a.cache, eps, Qb};
      hipLaunchKernelGGL(qkv_rows_finish, dim3(T, (kNQ + 2 * kNKV) / 4), dim3(256), 0, s, QKV, qo);
      launch_attention(a, l, Qb, tok, L, w, eps, ATT, s);
    }
    const Seg o{{u16(w.o_proj_weight), nullptr, nullptr}, {Dm::H, 0, 0}};
    launch_rows_residual<kQS, Dm::H>(ATT, T, o, X, ssq, s);
    const Seg gu{{u16(w.gate_proj_weight), u16(w.up_proj_weight), nullptr}, {Dm::I, Dm::I, 0}};
    constexpr int GB = Dm::I / 8 / kNumWG;  // 32 or 48 product columns per workgroup: at most one per CU
    launch_rows_norm<Dm::H, GB < 2 ? 2 : GB, kEpiSiluMul>(Dm::I / (8 * (GB < 2 ? 2 : GB)), X, u16(w.post_attn_layernorm_weight), ssq, eps, T,
                                                          gu, MM, Dm::I, s);
    const Seg dn{{u16(w.down_proj_weight), nullptr, nullptr}, {Dm::H, 0, 0}};
    launch_rows_residual<Dm::I, Dm::H>(MM, T, dn, X, ssq, s);
  }
  hipLaunchKernelGGL((residual_norm<Dm::H>), dim3(T), dim3(256), 0, s, nullptr, 0, T, X, a.final_norm, eps, N);
  launch_lm_head<M>(N, erow, R, a.lm_head, keys, a.logits, tok, a.out_tokens, s);
  return hipGetLastError() == hipSuccess ? QMK_OK : QMK_ERR_HIP;
}

template <class M>
int forward(const Args& a, hipStream_t s) {
  using Dm = Dims<M>;
  const int T = a.T, R = a.R;
  if (T <= kRowsMax) return forward_rows<M>(a, s);
  const Layout l = layout<M>(T, R, a.max_context, a.one_per_seq);
  Tok* tok = reinterpret_cast<Tok*>(a.ws + l.tok);
  int* erow = reinterpret_cast<int*>(a.ws + l.erow);
  auto* keys = reinterpret_cast<unsigned long long*>(a.ws + l.keys);
  uint16_t* X = reinterpret_cast<uint16_t*>(a.ws + l.x);
  uint16_t* N = reinterpret_cast<uint16_t*>(a.ws + l.n);
  uint16_t* Qb = reinterpret_cast<uint16_t*>(a.ws + l.q);
  uint16_t* ATT = reinterpret_cast<uint16_t*>(a.ws + l.att);
  uint16_t* MM = reinterpret_cast<uint16_t*>(a.ws + l.m);
  float* part = reinterpret_cast<float*>(a.ws + l.part);
  const float eps = 1e-6f;
  auto blocks = [](size_t n) { return dim3((unsigned)((n + 255) / 256)); };
  auto u16 = [](const void* p) { return static_cast<const uint16_t*>(p); };
  int ks = 1;

  const AttnPlan pl = attn_plan(a, l);
  hipLaunchKernelGGL((embed_tokens<Dm::H, true>), dim3(T + (pl.cap ? 1 : 0)), dim3(256), 0, s, a.tokens, a.seqs, a.pos,
                     T, a.emit, R, a.num_seqs, a.max_context, Dm::V, a.embed, tok, erow, X,
                     u16(a.layers[0].input_layernorm_weight), eps, N, nullptr, pl);
  for (int L = 0; L < a.num_layers; L++) {
    const LDGLayerWeights& w = a.layers[L];
    const Seg qkv{{u16(w.q_proj_weight), u16(w.k_proj_weight), u16(w.v_proj_weight)}, {kQS, kNKV * kD, kNKV * kD}};
    const QkvOut qo{tok, L, u16(w.q_norm_weight), u16(w.k_norm_weight), a.cos_t, a.sin_t, a.cache, eps, Qb};
    launch_gemm(N, T, Dm::H, qkv, kNQKV, part, s, &ks, kEpiQkv, &qo);
    if (ks) hipLaunchKernelGGL(qkv_finish, dim3(T, kNQ + 2 * kNKV), dim3(64), 0, s, part, ks, T, qo);
    launch_attention(a, l, Qb, tok, L, w, eps, ATT, s);
    const Seg o{{u16(w.o_proj_weight), nullptr, nullptr}, {Dm::H, 0, 0}};
    launch_gemm(ATT, T, kQS, o, Dm::H, part, s, &ks);
    hipLaunchKernelGGL((residual_norm<Dm::H>), dim3(T), dim3(256), 0, s, part, ks, T, X,
                       u16(w.post_attn_layernorm_weight), eps, N);
    const Seg gu{{u16(w.gate_proj_weight), u16(w.up_proj_weight), nullptr}, {Dm::I, Dm::I, 0}};
    const GateUpOut go{MM, Dm::I};
    launch_gemm(N, T, Dm::H, gu, 2 * Dm::I, part, s, &ks, kEpiGateUp, nullptr, &go);
    if (ks) hipLaunchKernelGGL(gate_up_finish, blocks((size_t)T * Dm::I), dim3(256), 0, s, part, ks, T, Dm::I, MM);
    const Seg dn{{u16(w.down_proj_weight), nullptr, nullptr}, {Dm::H, 0, 0}};
    launch_gemm(MM, T, Dm::I, dn, Dm::H, part, s, &ks);
    const uint16_t* next_norm = L + 1 < a.num_layers ? u16(a.layers[L + 1].input_layernorm_weight) : a.final_norm;
    hipLaunchKernelGGL((residual_norm<Dm::H>), dim3(T), dim3(256), 0, s, part, ks, T, X, next_norm, eps, N);
  }
  launch_lm_head<M>(N, erow, R, a.lm_head, keys, a.logits, tok, a.out_tokens, s);
  return hipGetLastError() == hipSuccess ? QMK_OK : QMK_ERR_HIP;
}

}  // namespace batch
}  // namespace qmk

using namespace qmk;

extern "C" {

size_t qmk_forward_workspace_bytes(int model, int num_tokens, int num_emit, int max_context) {
  if (num_tokens < 1 || num_emit < 1 || num_emit > batch::kMaxEmit || max_context < 1) return 0;
  if (model == QMK_MODEL_QWEN3_1_7B) return batch::layout<Qwen3_1_7B>(num_tokens, num_emit, max_context, false).total;
  if (model == QMK_MODEL_QWEN3_0_6B) return batch::layout<Qwen3_0_6B>(num_tokens, num_emit, max_context, false).total;
  return 0;
}

int qmk_forward_tokens(int model, int num_tokens, const int* tokens, const int* seq_ids, const int* positions,
                       int num_emit, const int* emit_rows, int* out_tokens, float* logits_out,
                       const void* embed_weight, const LDGLayerWeights* layer_weights_host,
                       const void* final_norm_weight, const void* lm_head_weight, const void* cos_table,
                       const void* sin_table, void* k_cache, void* v_cache, int num_seqs, long long seq_stride,
                       int num_layers, int max_seq_len, int max_context, float attn_scale, void* workspace,
                       size_t workspace_bytes, hipStream_t stream) {
  if (model != QMK_MODEL_QWEN3_0_6B && model != QMK_MODEL_QWEN3_1_7B) return QMK_ERR_ARG;
  if (num_tokens < 1 || num_emit < 1 || num_emit > batch::kMaxEmit || !tokens || !seq_ids || !positions ||
      !emit_rows || !out_tokens || !embed_weight || !layer_weights_host || !final_norm_weight || !lm_head_weight ||
      !cos_table || !sin_table || !k_cache || !v_cache || !workspace || num_seqs < 1 || num_layers < 1 ||
      num_layers > kMaxLayers || max_seq_len < 1 || max_context < 1 || max_context > max_seq_len ||
      !(attn_scale > 0.f))
    return QMK_ERR_ARG;
  const long long kv_per_seq = (long long)num_layers * batch::kNKV * max_seq_len * batch::kD;
  if (num_seqs > 1 && (seq_stride < kv_per_seq || seq_stride % 8 != 0)) return QMK_ERR_ARG;
  for (const void* q : {embed_weight, final_norm_weight, lm_head_weight, cos_table, sin_table, (const void*)k_cache,
                        (const void*)v_cache, (const void*)workspace})
    if (!aligned16(q)) return QMK_ERR_ARG;
  for (int L = 0; L < num_layers; L++) {
    const LDGLayerWeights& w = layer_weights_host[L];
    const void* p[11] = {w.input_layernorm_weight, w.q_proj_weight, w.k_proj_weight, w.v_proj_weight,
                         w.q_norm_weight, w.k_norm_weight, w.o_proj_weight, w.post_attn_layernorm_weight,
                         w.gate_proj_weight, w.up_proj_weight, w.down_proj_weight};
    for (const void* q : p)
      if (!q || !aligned16(q)) return QMK_ERR_ARG;
  }
  if (workspace_bytes < qmk_forward_workspace_bytes(model, num_tokens, num_emit, max_context)) return QMK_ERR_ARG;
  batch::Args a{};
  a.T = num_tokens;
  a.R = num_emit;
  a.num_seqs = num_seqs;
  a.max_context = max_context;
  a.tokens = tokens;
  a.seqs = seq_ids;
  a.pos = positions;
  a.emit = emit_rows;
  a.out_tokens = out_tokens;
  a.logits = logits_out;
  a.embed = static_cast<const uint16_t*>(embed_weight);
  a.final_norm = static_cast<const uint16_t*>(final_norm_weight);
  a.lm_head = static_cast<const uint16_t*>(lm_head_weight);
  a.cos_t = static_cast<const uint16_t*>(cos_table);
  a.sin_t = static_cast<const uint16_t*>(sin_table);
  a.layers = layer_weights_host;
  a.cache = batch::Cache{static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(v_cache),
                         num_seqs > 1 ? seq_stride : 0, max_seq_len};
  a.num_layers = num_layers;
  a.attn_scale = attn_scale;
  a.ws = static_cast<char*>(workspace);
  return model == QMK_MODEL_QWEN3_1_7B ? batch::forward<Qwen3_1_7B>(a, stream) : batch::forward<Qwen3_0_6B>(a, stream);
}

size_t qmk_decode_batch_workspace_bytes(int model, int batch, int max_context) {
  if (batch < 1 || batch > batch::kMaxEmit || max_context < 1) return 0;
  if (model == QMK_MODEL_QWEN3_1_7B) return batch::layout<Qwen3_1_7B>(batch, batch, max_context, true).total;
  if (model == QMK_MODEL_QWEN3_0_6B) return batch::layout<Qwen3_0_6B>(batch, batch, max_context, true).total;
  return 0;
}

int qmk_decode_batch(int model, int batch, const int* tokens, const int* positions, int* out_tokens,
                     float* logits_out, const void* embed_weight, const LDGLayerWeights* layer_weights_host,
                     const void* final_norm_weight, const void* lm_head_weight, const void* cos_table,
                     const void* sin_table, void* k_cache, void* v_cache, long long seq_stride, int num_layers,
                     int max_seq_len, int max_context, float attn_scale, void* workspace, size_t workspace_bytes,
                     hipStream_t stream) {
  if (model != QMK_MODEL_QWEN3_0_6B && model != QMK_MODEL_QWEN3_1_7B) return QMK_ERR_ARG;
  if (batch < 1 || batch > batch::kMaxEmit || !tokens || !positions || !out_tokens || !embed_weight ||
      !layer_weights_host || !final_norm_weight || !lm_head_weight || !cos_table || !sin_table || !k_cache ||
      !v_cache || !workspace || num_layers < 1 || num_layers > kMaxLayers || max_seq_len < 1 || max_context < 1 ||
      max_context > max_seq_len || !(attn_scale > 0.f))
    return QMK_ERR_ARG;
  const long long kv_per_seq = (long long)num_layers * batch::kNKV * max_seq_len * batch::kD;
  if (batch > 1 && (seq_stride < kv_per_seq || seq_stride % 8 != 0)) return QMK_ERR_ARG;
  for (const void* q : {embed_weight, final_norm_weight, lm_head_weight, cos_table, sin_table, (const void*)k_cache,
                        (const void*)v_cache, (const void*)workspace})
    if (!aligned16(q)) return QMK_ERR_ARG;
  for (int L = 0; L < num_layers; L++) {
    const LDGLayerWeights& w = layer_weights_host[L];
    const void* p[11] = {w.input_layernorm_weight, w.q_proj_weight, w.k_proj_weight, w.v_proj_weight,
                         w.q_norm_weight, w.k_norm_weight, w.o_proj_weight, w.post_attn_layernorm_weight,
                         w.gate_proj_weight, w.up_proj_weight, w.down_proj_weight};
    for (const void* q : p)
      if (!q || !aligned16(q)) return QMK_ERR_ARG;
  }
  // The persistent kernel writes out_tokens (-1) before every workgroup has read tokens and
  // positions, so a call whose out_tokens overlaps them takes the multi-launch path, which reads
  // them first.
  const auto overlaps = [&](const void* p) {
    const char* a = static_cast<const char*>(p);
    const char* o = reinterpret_cast<const char*>(out_tokens);
    return a < o + batch * sizeof(int) && o < a + batch * sizeof(int);
  };
  if (qmk_batch_persistent_enabled() && batch >= kBatchMin && batch <= kBatchMax && max_context <= kBatchMaxContext &&
      !overlaps(tokens) && !overlaps(positions)) {
    const int s = qmk_decode_batch_persistent(model, batch, tokens, positions, out_tokens, logits_out, embed_weight,
                                              layer_weights_host, final_norm_weight, lm_head_weight, cos_table,
                                              sin_table, k_cache, v_cache, seq_stride, num_layers, max_seq_len,
                                              max_context, attn_scale, stream);
    if (s != QMK_ERR_DEVICE) return s;
  }
  if (workspace_bytes < qmk_decode_batch_workspace_bytes(model, batch, max_context)) return QMK_ERR_ARG;
  batch::Args a{};
  a.T = batch;
  a.R = batch;
  a.num_seqs = batch;
  a.max_context = max_context;
  a.one_per_seq = true;
  a.tokens = tokens;
  a.seqs = nullptr;
  a.pos = positions;
  a.emit = nullptr;
  a.out_tokens = out_tokens;
  a.logits = logits_out;
  a.embed = static_cast<const uint16_t*>(embed_weight);
  a.final_norm = static_cast<const uint16_t*>(final_norm_weight);
  a.lm_head = static_cast<const uint16_t*>(lm_head_weight);
  a.cos_t = static_cast<const uint16_t*>(cos_table);
  a.sin_t = static_cast<const uint16_t*>(sin_table);
  a.layers = layer_weights_host;
  a.cache = batch::Cache{static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(v_cache), batch > 1 ? seq_stride : 0,
                         max_seq_len};
  a.num_layers = num_layers;
  a.attn_scale = attn_scale;
  a.ws = static_cast<char*>(workspace);
  return model == QMK_MODEL_QWEN3_1_7B ? batch::forward<Qwen3_1_7B>(a, stream) : batch::forward<Qwen3_0_6B>(a, stream);
}

int qmk_selftest_mfma(const void* a, const void* b, float* c, hipStream_t stream) {
  if (!a || !b || !c) return QMK_ERR_ARG;
  hipLaunchKernelGGL(batch::mfma_selftest, dim3(1), dim3(64), 0, stream, static_cast<const uint16_t*>(a),
                     static_cast<const uint16_t*>(b), c);
  return hipGetLastError() == hipSuccess ? QMK_OK : QMK_ERR_HIP;
}

}  // extern "C"
