// C ABI of libmi_moe: validation, workspace carving and the launch sequence of the block.
// Declarations and the reference interfaces they replace: include/mi_moe.h.
#include "../../include/mi_moe.h"

#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>

#include "common.hpp"

using namespace mi_moe;

// ------------------------------------------------------------------ errors
namespace {

thread_local char g_last_error[512] = "";

// The registered handler with its data.  A failing thread takes a reference under the lock and calls
// the handler outside it, so a handler swapped meanwhile stays alive (its dtor runs when the last
// reference goes) and a handler may itself register another one.
struct Handler {
  void (*fn)(const char *, void *);
  void *data;
  void (*dtor)(void *);
  ~Handler() {
    if (dtor && data) dtor(data);
  }
};
std::mutex g_handler_lock;
std::shared_ptr<Handler> g_handler;

int fail(const char *fmt, ...) __attribute__((format(printf, 1, 2)));
int fail(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof g_last_error, fmt, ap);
  va_end(ap);
  std::shared_ptr<Handler> h;
  {
    std::lock_guard<std::mutex> g(g_handler_lock);
    h = g_handler;
  }
  if (h && h->fn) h->fn(g_last_error, h->data);
  return 1;
}

// No exception leaves an entry point: every extern "C" body is a function-try-block that ends in this.
#define MI_CATCH(name)                                                                  \
  catch (const std::exception &ex_) { return fail(name ": %s", ex_.what()); }           \
  catch (...) { return fail(name ": unknown C++ exception"); }

int hip_fail(const char *what, hipError_t e) {
  return fail("%s: %s", what, hipGetErrorString(e));
}

#define MI_HIP(call)                                   \
  do {                                                 \
    hipError_t e_ = (call);                            \
    if (e_ != hipSuccess) return hip_fail(#call, e_);  \
  } while (0)

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

size_t align_up(size_t v, size_t a = 256) { return (v + a - 1) / a * a; }

// the block runs on the tuned kernels with 4- or 8-bit codes in groups of 64; other group sizes take the
// products on raw codes where those serve the shape (ForwardWs::raw), the rest and 2-bit codes the plain products
bool plain_config(const mi_moe_config &c) { return c.group_size != 64 || c.bits == 2; }

int check_config(const mi_moe_config *c) {
  if (!c) return fail("config is NULL");
  if (c->bits != 2 && c->bits != 4 && c->bits != 8) return fail("bits must be 2, 4 or 8, got %d", c->bits);
  if (c->group_size != 32 && c->group_size != 64 && c->group_size != 128)
    return fail("group_size must be 32, 64 or 128, got %d", c->group_size);
  if (c->hidden <= 0 || c->hidden % 64) return fail("hidden must be a positive multiple of 64, got %d", c->hidden);
  if (c->intermediate <= 0 || c->intermediate % 64)
    return fail("intermediate must be a positive multiple of 64, got %d", c->intermediate);
  if (c->hidden % c->group_size || c->intermediate % c->group_size)
    return fail("hidden and intermediate must be multiples of group_size (%d), got %d, %d", c->group_size, c->hidden,
                c->intermediate);
  if (c->n_experts < 1 || c->n_experts > 512) return fail("n_experts must be in [1, 512], got %d", c->n_experts);
  if (c->top_k < 1 || c->top_k > c->n_experts || c->top_k > 32)
    return fail("top_k must be in [1, min(n_experts, 32)], got %d", c->top_k);
  if (c->score_mode < 0 || c->score_mode > 2) return fail("unknown score_mode %d", c->score_mode);
  if (!plain_config(*c) && c->bits == 4 && (c->hidden % 128 || c->intermediate % 128))
    return fail("4-bit weights need hidden and intermediate to be multiples of 128 (got %d, %d)", c->hidden,
                c->intermediate);
  return 0;
}

int check_qmat(const mi_moe_qmat &m, const char *name) {
  if (!m.w || !m.scales || !m.biases) return fail("%s: weight, scales and biases must be non-NULL", name);
  if (!aligned16(m.w) || !aligned16(m.scales) || !aligned16(m.biases))
    return fail("%s: pointers must be 16-byte aligned", name);
  return 0;
}

// carve consecutive 256-byte aligned regions out of a workspace; the first one starts at the next
// 256-byte boundary (every *_workspace_size reserves 256 bytes for that)
struct Carver {
  char *base;
  size_t off = 0;
  explicit Carver(void *p)
      : base(reinterpret_cast<char *>((reinterpret_cast<uintptr_t>(p) + 255u) & ~(uintptr_t)255u)) {}
  template <typename T>
  T *take(size_t n) {
    T *p = reinterpret_cast<T *>(base + off);
    off += align_up(n * sizeof(T));
    return p;
  }
};

struct ForwardWs {
  uint16_t *logits;
  uint32_t *topk_idx;
  uint16_t *topk_w;
  uint32_t *counts, *offsets, *work, *mtiles, *perm, *inv_perm, *src_of;
  Records records;  // the streamed segments', in `work` or (split) in a place of their own
  int max_mtiles;
  bool tiled;  // tile lists are built
  bool heavy;  // most rows are tiled: see heavy_batch()
  int tmr;     // segments of at least this many rows are tiled
  void *disp_scratch;
  uint16_t *hh, *y, *xperm, *xnorm;
  uint16_t *gu;  // plain products only: the gate and the up product, [P, I] each
  bool mid;             // groups of 64: all segments in pieces on raw codes (see mid_batch)
  bool pieces;          // the same tiles for the segments of a heavy batch that are tiled, the others streamed
  bool raw_all;         // groups of 32 / 128: all segments in pieces (see raw_list_batch)
  bool raw;             // group sizes 32 / 128: the products on raw codes (qmm_rows, qmm_short)
  uint32_t *raw_tiles;  // the list of pieces, the copy of x in their order (4-bit) and the group sums of x and h, or nullptr:
  int raw_cap;          // (groups of 32 / 128) all segments go through the kernel of a few rows, in as many passes as they need
  int raw_from;         // segments of this many rows and more are cut into pieces
  int raw_piece;        // of this many rows
  uint16_t *raw_copy, *raw_xsums, *raw_hsums;
  size_t bytes_raw;     // up to the end of those
  void *router_scratch;  // byte planes of x and of the router matrix (logits on the int8 matrix cores), or nullptr
  size_t bytes_min;      // without the byte planes: a workspace of this size makes the forward take the fp64 logits (same bits)
  size_t bytes;
};

// The kernels that take a list of pieces: operands below 2 GiB, in multiples of 128 values.
bool codes_tiles_fit(const mi_moe_config &c, int64_t T) {
  const int64_t P = T * c.top_k, most = (int64_t)1 << 31;
  return c.hidden % 128 == 0 && c.intermediate % 128 == 0 && T * c.hidden * 2 < most &&
         P * c.intermediate * 2 < most && (int64_t)codes_sums_bytes(P, c.intermediate, c.group_size) < most &&
         (int64_t)codes_sums_bytes(T, c.hidden, c.group_size) < most &&
         (int64_t)c.hidden * c.intermediate * c.bits / 8 < most;
}
// Group sizes 32 and 128: batches whose segments all go in pieces (qmm_short_kernel), one launch a product; the others go through the kernel of a few rows, which a
// segment of at most T rows has to be more than one pass of.  Us of a forward, tiles of 32 x 32 results (qmm_tiles.hip; with 8-bit codes between twenty and forty rows
// an expert short segments on the kernel of a few rows beside them, on another stream) / pieces, (experts, k, hidden, intermediate, bits, group):
//   128, 8, 2048, 768, 4, 32   even at 100 / 160 / 256 / 400 / 512 tokens 147, 150, 152, 168, 175 / 122, 127, 134, 140, 149; Zipf-1.1 at 100 / 256 / 512 98, 116, 163 / 86, 100, 143
//   128, 8, 2048, 768, 4, 128  even at 100 / 256 / 512 113, 120, 138 / 93, 107, 118; Zipf-1.1 78, 91, 124 / 71, 83, 115
//   128, 8, 2048, 768, 8, 32   even at 100 / 330 / 512 199, 236, 248 / 187, 200, 208; Zipf-1.1 at 330 / 512 260, 213 / 234, 193; 1.3 at 500 189 / 180
//   128, 8, 2048, 768, 8, 128  even at 330 / 512 194, 198 / 160, 169; Zipf-1.1 at 330 / 512 229, 180 / 184, 151
//   64, 6, 2048, 1408, 4, 32   128 tokens, even and Zipf-1.1 139, 131 / 119, 105; 8, 2, 4096, 7168, 4, 32 at 256 tokens 346 / 280; 8, 2, 4096, 14336, 8, 32 at 100 645 / 515
// All segments on the kernel of a few rows (4-bit, 32): 512 tokens and even routing 328, Zipf-1.1 1017.
bool raw_list_batch(const mi_moe_config &c, int64_t T) {
  return T > kRowsMost && T * c.top_k >= (int64_t)4 * c.n_experts && codes_tiles_fit(c, T);
}
// Groups of 64, 8-bit codes: the same for batches of a few rows an expert, where a popular expert's segment is many passes of the streaming kernel and a tile of 256
// weight rows mostly padding.  Us of a forward, other route (streamed; pieces on dequantised weights from 17 rows an expert on) / this, (experts, k, hidden, intermediate):
//   128, 8, 2048, 768  even at 64 / 80 / 150 / 200 / 300 tokens 153, 164, 179, 213, 196 / 156, 157, 161, 165, 164; Zipf-1.1 at 64 / 100 / 200 160, 232, 443 / 90, 101, 113
//   64, 6, 2048, 1408  even at 60 / 100 / 200 148, 170, 191 / 139, 143, 151; 16, 4, 4096, 6400 at 30 / 50 / 100 415, 499, 375 / 345, 352, 367, Zipf-1.1 at 50 524 / 347
//   8, 2, 4096, 14336  even at 32 / 40 / 48 / 56 / 64 / 80 / 100 / 130 tokens 350, 378, 362 to 399, 474, 500, 538, 463, 436 / 400, 405, 404, 406, 409, 426, 427, 434; Zipf-1.1 at 40 / 64 / 100
//                      475, 615, 520 / 412, 420, 571
// With fewer blocks in the down product than CUs its blocks are what a forward waits for, whatever their rows, and streaming stays ahead up to some thirteen rows.  At 25 and 32 rows
// an expert 128 experts would still gain (400 / 512 tokens 206, 189 / 167, 174, skewed 163 / 153) and eight skewed ones lose (above); from 24 on the launch plan of 8-bit
// batches holds streamed segments beside tiles, as its callers know it.
bool few_rows_batch(const mi_moe_config &c, int64_t T) { return T * c.top_k < (int64_t)24 * c.n_experts; }
bool mid_bytes_batch(const mi_moe_config &c, int64_t T) {
  const int64_t P = T * c.top_k, E = c.n_experts, least = E * (c.hidden / 256) >= 256 ? 6 : 14;
  return c.bits == 8 && c.group_size == 64 && E >= 8 && P >= least * E && few_rows_batch(c, T) && codes_tiles_fit(c, T);
}
// Groups of 64, 4-bit codes: batches whose segments all go through pieces on raw codes, in one launch a product on the caller's
// stream (the others: streamed segments, and tiles of 256 weight rows on side streams).  From the batches on for which the tile lists
// are built and the router has kernels of its own, up to 96 rows per expert on average (beyond: piece_batch).  Measured when pieces had 64 rows, in the experts' order, us
// of a forward, other route / this one (now, same card as the first table of list_pieces: 117 at 203 tokens, 153 at 700, 182 at 1100, even routing):
//   128 experts, hidden 2048, even routing at 96 / 128 / 203 / 320 / 512 / 1024 / 2048 / 4096 tokens 145, 151, 176, 216, 218, 266, 360, 484 /
//   128, 124, 128, 134, 168, 221, 350, 566; Zipf-1.1 136, 139, 160, 173, 193, 237, 344, 490 / 92, 95, 114, 134, 157, 219, 341, 560;
//   hidden 4096, intermediate 1536, even at 128 / 256 / 512 / 1024 / 2048 tokens 536, 587, 665, 785, 1144 / 372, 375, 449, 649, 1101; Zipf-1.3
//   315, 442, 510, 698, 1079 / 271, 354, 477, 693, 1123.
// Longer segments in 256-row tiles beside this (a fork, six launches more): 203 for 169 at 512 tokens, 516 for 490 at 4096.
//   fewer experts, even and Zipf-1.1, (experts, k, hidden, intermediate): 64, 6, 2048, 1408 at 128, 300, 700, 1000 tokens 166, 200, 260, 265 and 139, 193, 249,
//   269 / 110, 135, 198, 238 and 113, 147, 202, 245; 32, 4, 2048, 1024 at 128, 300, 700 120, 109, 134 and 132, 159, 166 / 60, 75, 102 and 73, 87, 113;
//   16, 4, 4096, 6400 at 128, 256, 384 414, 531, 526 and 479, 521, 609 / 273, 374, 474 and 330, 366, 461; 16, 2, 2048, 2048 at 256, 512, 760 110, 161, 139 and
//   169, 173, 185 / 81, 98, 105 and 89, 99, 115; 8, 2, 4096, 14336 at 256, 300, 384 642, 723, 644 and 677, 719, 771 / 492, 499, 525 and 485, 481, 516.
// 8-bit codes (8 experts, 4096 x 14336, 256 / 512 tokens): 741, 737 / 835, 1107.  Fewer than 512 pairs, or than eight experts, keep the other route, though
// these tiles are faster there as well (144 to 504 pairs, 4 to 16 experts: 1.08 to 2.1 times).
bool mid_batch(const mi_moe_config &c, int64_t T, bool tiled) {
  const int64_t P = T * c.top_k;
  if (c.bits == 8) return mid_bytes_batch(c, T);
  return tiled && c.bits == 4 && T > kFusedRouterMaxTokens && P <= (int64_t)96 * c.n_experts && P >= 512 && c.n_experts >= 8 && codes_tiles_fit(c, T);
}

// Batches whose pieces go to qmm_short_kernel, 64 rows and less.  Us of a forward, qmm_pieces_kernel (64 rows up to 48 an expert on average, 96 from there) / this, one card:
//   128 experts, hidden 2048, even routing at 96 / 160 / 240 / 330 / 512 / 700 / 900 / 1024 / 1280 tokens 107, 111, 113, 121, 135, 151, 168, 170, 194 / 95, 99, 104, 113, 122,
//   137, 156, 179, 220; Zipf-1.1 at 512 / 700 / 1024 / 1500 tokens 159, 179, 197, 244 / 149, 169, 196, 242; 1.3 at 96 / 250 / 700 / 1500 tokens 99, 84, 181, 251 / 88, 81, 170, 248;
//   hidden 4096, intermediate 1536, even at 96 / 250 / 400 / 700 / 900 / 1024 tokens 343, 357, 370, 476, 507, 525 / 319, 340, 357, 443, 492, 604; Zipf-1.3 at 96 / 250 / 700
//   tokens 312, 299, 552 / 288, 284, 526;
//   64 experts, 6, hidden 2048, intermediate 1408, even at 100 / 165 / 600 / 900 tokens (56 and 84 rows) 99, 102, 148, 174 / 90, 95, 144, 192; 64, 4, 4096 x 2048, 200 tokens 244 / 230;
//   256 experts, 8, 2048 x 512, 200 / 500 tokens 145, 151 / 132, 145.
// With even routing most segments leave a second piece from about 60 rows on average on, and the line lies there.  From 48 rows on, where the others are pieces of 96, the two are near each
// other, and which is ahead goes by the routing, which the host does not see: 128 experts at 800 / 850 / 900 / 955 tokens, hidden 2048, even 163, 163, 166, 171 / 151, 157, 161, 167, Zipf-0.5 166, 168,
// 173, 176 / 171, 175, 176, 182, 1.1 147, 152, 162, 169 / 151, 156, 160, 169, 1.3 138, 141, 145, 150 / 145, 148, 150, 153; hidden 4096, even 482, 494, 514, 529 / 460, 481, 525, 553, Zipf-1.1 563, 587, 601,
// 627 / 559, 581, 588, 623; 256 experts, 2048 x 512, 1800 tokens, even and Zipf-1.1 226, 208 / 230, 210; 64 experts at 560 / 639 tokens 146, 152 / 140, 147 and 158, 167 / 154, 165; 16 experts,
// 2048 x 4096, 220 tokens 127, 144 / 108, 121.
bool short_pieces(int64_t pairs, int n_experts) { return pairs < (int64_t)60 * n_experts; }

// Rows of a piece beyond those.  Longer ones read a weight row for more token rows; but a block's time grows with its rows, and until the pieces are several times what
// the chip holds at once, the longest segments' blocks are what a launch waits for.  Gate/up and down kernels, us, pieces of 96 / 128 rows (128 experts,
// hidden 2048) at an average of 64, 94 rows: Zipf-1.1 164, 219 / 181, 224; even 147, 212 / 151, 183; at 256 rows, Zipf-1.1, 421 / 422.
int piece_rows(int64_t pairs, int n_experts) { return short_pieces(pairs, n_experts) ? kShortTileM : pairs < (int64_t)80 * n_experts ? 96 : kPieceM; }

// Larger batches: the same pieces for the segments of nine rows and more, the others streamed ahead of them.  Us of a forward, tiles of 256 weight rows in three
// classes on two streams / this: 128 experts, hidden 2048, 4096 tokens, Zipf-1.1 501 / 492; hidden 4096, 8192 tokens, Zipf-1.3 3052 / 2972; gate/up and down
// kernels of 8192 tokens, even routing, 840 / 800.  Nearer to float64 as well (3.87e-3 / 2.87e-3), since the weights are not rounded.  Streaming them
// beside the tiles on a side stream, or only those of one row, or of one to three: the same times, since each way keeps both launches.  Without them, every segment
// in pieces as in the middle range, streamed / not, even and Zipf-1.1 at 1600 / 2048 / 3000 / 4096 / 8192 tokens (hidden 2048): 232, 282, 371, 473, 860 and 281, 303,
// 400, 479, 851 / 227, 278, 367, 469, 855 and 261, 289, 377, 475, 842; hidden 4096, Zipf-1.3, 4096 and 8192 tokens 1635, 2923 / 1619, 2900.  So the line at 96 rows
// an expert is where the 256-column tiles used to begin, and no longer where either side is the faster one.
// 8-bit codes: pieces of up to 128 rows on dequantised weights (qmm_bytes.hip) for the segments of seventeen rows and more, the others streamed.  Us of a forward, the other
// route (tiles of 256 weight rows in three classes on two to four streams) / this, (experts, k, hidden, intermediate):
//   8, 2, 4096, 14336  even at 100 / 160 / 256 / 400 / 700 / 1400 / 2048 tokens 573, 591, 734, 696, 940, 1430, 1788 / 382 to 425, 400, 437, 497, 810, 1285, 1741;
//                      Zipf-1.1 at 100 / 300 / 1000 572, 810, 1161 / 544, 595, 988
//   128, 8, 2048, 768  even at 300 / 512 / 1024 / 2048 / 2500 / 3200 / 4096 tokens 259, 251, 299, 398, 457, 447, 534 / 207, 189, 226, 349, 419, 455, 541; Zipf-1.1 at 400 / 1024 /
//                      4096 209, 276, 549 / 163, 238, 529
//   64, 6, 2048, 1408  even at 400 / 1400 / 2000 232, 372, 381 / 181, 320, 398; Zipf-1.1 at 1400 / 2400 400, 486 / 326, 438
//   16, 4, 4096, 6400  even at 100 / 400 459, 565 / 374, 469
// Even routing from 170 to 255 rows an expert on average is where the other route is at its best, one tile of 256 rows for nearly every expert and two pieces here: 64, 6, 4096, 1408 at 1800 /
// 2200 / 2600 / 3000 tokens 679, 689, 793, 1000 / 688, 735, 818, 940; 128, 8, 4096, 1536 at 2500 / 3200 / 3600 / 4096 1429, 1456, 1525, 1852 / 1408, 1551, 1635, 1800; 32, 4, 4096, 2048 at 1300 /
// 1900 / 2100 490, 552, 667 / 507, 582, 625; 64, 8, 6144, 2048 at 1700 1373 / 1488.  Any skew turns it round, and the host does not see which it is: Zipf-0.5 and 1.1, 64, 6, 4096, 1408 at 2200 794,
// 813 / 712, 745, 128, 8, 4096, 1536 at 3200 1547, 1627 / 1425, 1517; Zipf-1.1, 32, 4, 4096, 2048 at 1900 661 / 542, 64, 8, 6144, 2048 at 1700 1567 / 1424.  Rows of 2048 values are short enough
// for a block's ends to weigh, and there the other route stays from 176 rows an expert on.
bool piece_batch(const mi_moe_config &c, int64_t T, bool heavy) {
  const int64_t P = T * c.top_k;
  if (!heavy || T <= kFusedRouterMaxTokens || c.n_experts < 8 || !codes_tiles_fit(c, T)) return false;
  return c.bits == 4 ? P >= 512 : c.hidden >= 4096 || P < (int64_t)176 * c.n_experts;
}

// norm: the normalised rows of the residual variant are kept as long as their segments stream.
ForwardWs carve_forward(const mi_moe_config &c, int64_t T, void *ws, bool norm) {
  const int64_t P = T * c.top_k;
  Carver cv(ws);
  ForwardWs f;
  f.logits = cv.take<uint16_t>((size_t)T * c.n_experts);
  f.topk_idx = cv.take<uint32_t>((size_t)P);
  f.topk_w = cv.take<uint16_t>((size_t)P);
  f.counts = cv.take<uint32_t>(c.n_experts);
  f.offsets = cv.take<uint32_t>(c.n_experts + 1);
  f.work = cv.take<uint32_t>((size_t)c.n_experts * 16);
  // M tiles of the tiled kernel: the 256-row list holds at most P / 256 full tiles plus one
  // remainder per tiled segment (a segment is at most T rows long: no token picks an expert twice)
  // (the tiled kernel reads scales in 8-byte pieces: rows of scales must be 4-byte aligned, i.e.
  // an even number of groups per row; other shapes stay on the streaming kernel)
  const bool tiled_ok = (c.hidden / 64) % 2 == 0 && (c.intermediate / 64) % 2 == 0;
  f.tiled = tiled_ok && !plain_config(c) && tiled_batch(P, c.n_experts, c.bits);
  f.heavy = f.tiled && heavy_batch(P, c.n_experts, c.bits);
  const int tmr = f.tmr = tile_min_rows(c.bits, f.heavy);
  f.max_mtiles = f.tiled ? (int)(P / kBigTileM + (P / tmr < c.n_experts ? P / tmr : c.n_experts)) : 0;
  f.mtiles = cv.take<uint32_t>(tile_list_words(f.max_mtiles, c.n_experts));
  f.perm = cv.take<uint32_t>((size_t)P);
  f.inv_perm = cv.take<uint32_t>((size_t)P);
  f.src_of = cv.take<uint32_t>((size_t)P);
  f.hh = cv.take<uint16_t>((size_t)P * c.intermediate);
  f.y = cv.take<uint16_t>((size_t)P * c.hidden);
  f.disp_scratch = f.y;  // (per-block histograms, read before the first product: at most 4 E bytes for 1024 pairs, and one block's)
  f.xperm = cv.take<uint16_t>(f.tiled && c.bits == 4 ? (size_t)T * c.hidden : 0);
  f.xnorm = cv.take<uint16_t>((size_t)T * c.hidden);  // rms_norm(x) of the residual variant
  RowsArgs up{}, down{};  // (the extents only)
  static const uint32_t records[1] = {};
  up.work = down.work = records;
  up.max_active = down.max_active = (int)(P < c.n_experts ? P : c.n_experts);
  up.max_rows = down.max_rows = T;
  up.N = down.K = c.intermediate;
  up.K = down.N = c.hidden;
  f.raw = plain_config(c) && qmm_rows_applies(up, c.group_size, c.bits, MI_MOE_DTYPE_BF16, true) &&
          qmm_rows_applies(down, c.group_size, c.bits, MI_MOE_DTYPE_BF16, false);
  f.gu = cv.take<uint16_t>(plain_config(c) && !f.raw ? 2 * (size_t)P * c.intermediate : 0);
  f.raw_tiles = nullptr;
  f.raw_cap = 0;
  f.raw_from = 1;
  f.raw_piece = kShortTileM;
  f.bytes_min = cv.off;
  f.mid = mid_batch(c, T, f.tiled);
  f.pieces = !f.mid && piece_batch(c, T, f.heavy);
  if (f.mid && c.bits == 8) {
    f.raw_cap = short_list_cap(P, c.n_experts, 1, f.raw_piece);
    f.raw_tiles = cv.take<uint32_t>(short_list_words(f.raw_cap));
    f.raw_xsums = cv.take<uint16_t>(codes_sums_bytes(T, c.hidden, c.group_size) / 2);
    f.raw_hsums = cv.take<uint16_t>(codes_sums_bytes(P, c.intermediate, c.group_size) / 2);
  } else if (f.mid) {
    // All of it lies in memory that is free at the time where it fits, so that batches which have to fit a scratch of a given size take
    // this route as well: the list in place of the work records (nothing is streamed), the group sums of x where the down product writes
    // its rows later, those of h in the normalised rows, which only the router and the copy of x read.
    f.raw_piece = piece_rows(P, c.n_experts);
    f.raw_cap = short_list_cap(P, c.n_experts, 1, f.raw_piece);
    const size_t list = short_list_words(f.raw_cap), xsums = codes_sums_bytes(T, c.hidden, c.group_size, true), hsums = codes_sums_bytes(P, c.intermediate, c.group_size, true);
    f.raw_tiles = list <= (size_t)c.n_experts * 16 ? f.work : cv.take<uint32_t>(list);
    f.raw_copy = f.xperm;
    const size_t hist = align_up(dispatch_workspace_bytes(c.n_experts, P));  // (which are read while the sums are made)
    f.raw_xsums = hist + xsums <= (size_t)P * c.hidden * 2 ? f.y + hist / 2 : cv.take<uint16_t>(xsums / 2);
    f.raw_hsums = hsums <= (size_t)T * c.hidden * 2 ? f.xnorm : cv.take<uint16_t>(hsums / 2);
  }
  if (f.pieces) {
    f.raw_from = f.tmr;
    f.raw_piece = kPieceM;  // (more rows an expert than the middle range has: piece_rows' last)
    f.raw_cap = short_list_cap(P, c.n_experts, f.raw_from, f.raw_piece);
    // (as above; nothing reads the 256-column tiles' lists, and where there is no norm the place of its rows is free)
    const size_t list = short_list_words(f.raw_cap);
    const size_t xsums = c.bits == 4 ? codes_sums_bytes(T, c.hidden, c.group_size, true) : 0, hsums = c.bits == 4 ? codes_sums_bytes(P, c.intermediate, c.group_size, true) : 0;
    const bool in_norm = !norm && xsums + hsums <= (size_t)T * c.hidden * 2;
    f.raw_tiles = list <= tile_list_words(f.max_mtiles, c.n_experts) ? f.mtiles : cv.take<uint32_t>(list);
    f.raw_copy = f.xperm;
    f.raw_xsums = in_norm ? f.xnorm : cv.take<uint16_t>(xsums / 2);
    f.raw_hsums = in_norm ? f.xnorm + xsums / 2 : cv.take<uint16_t>(hsums / 2);
  }
  f.raw_all = f.raw && raw_list_batch(c, T);
  // Where everything streams, or goes through the kernel of a few rows, a segment of several passes is as many records, whose blocks run beside each other: with skewed
  // routing one block would go over a popular expert's weights pass after pass, long after the others are done.  Us of a forward, a record a segment / a pass (same bits):
  //   128, 8, 2048, 768, 4 bits  Zipf-1.1 at 16 / 24 / 32 / 48 / 64 / 80 / 95 tokens 63, 81, 82, 116, 141, 176, 201 / 50, 57, 52, 68, 73, 88, 94; 1.3 at 32 / 95 82, 203 / 48, 89; even
  //                              at 16 / 32 / 64 / 95 65, 83, 97, 120 / 64, 83, 95, 114
  //   128, 8, 4096, 1536, 4 bits Zipf-1.3 at 24 / 64 / 95 221, 374, 527 / 155, 234, 303; 64, 6, 2048, 1408, 4 bits, Zipf-1.1 at 40 102 / 67
  //   128, 8, 2048, 768, 8 bits  Zipf-1.1 at 64 159 / 93; 8, 2, 4096, 14336, 8 bits at 32 / 48 416, 533 / 348, 457
  f.records = Records(f.work);
  const bool rows_kernel = f.raw && !f.raw_all, streams = !plain_config(c) && !f.tiled && !f.mid;
  if (int log2 = c.bits == 4 && streams ? 3 : 4; (streams || rows_kernel) && T > 1 << log2) {  // (rows of a pass)
    const int64_t most = P < c.n_experts ? P : c.n_experts;
    auto slots = [&]() { return most + ((P - most) >> log2); };
    uint32_t *const at = cv.take<uint32_t>((size_t)(slots() < kMostRecords ? slots() : kMostRecords) * 16);
    while (slots() > kMostRecords) ++log2;  // (from half a million pairs on: several passes)
    f.records = Records(at, log2, (int)slots());
  }
  if (f.raw_all) {
    f.raw_cap = short_list_cap(P, c.n_experts, f.raw_from, f.raw_piece);
    f.raw_tiles = cv.take<uint32_t>(short_list_words(f.raw_cap));
    f.raw_copy = cv.take<uint16_t>(codes_copy_bytes(c.bits, T, c.hidden) / 2);
    f.raw_xsums = cv.take<uint16_t>(codes_sums_bytes(T, c.hidden, c.group_size) / 2);
    f.raw_hsums = cv.take<uint16_t>(codes_sums_bytes(P, c.intermediate, c.group_size) / 2);
  }
  f.bytes_raw = cv.off;
  const bool i8_router = router_logits_i8_applies(T, c.hidden, c.n_experts);  // (the last region: optional, see bytes_min)
  f.router_scratch = cv.take<char>(i8_router ? router_logits_i8_bytes(T, c.hidden, c.n_experts) : 0);
  if (!i8_router) f.router_scratch = nullptr;
  f.bytes = cv.off;
  return f;
}

}  // namespace

// Scratch of mi_moe_forward_static: the workspace a forward needs, as one array that is part of the
// library's code object.  Every GPU that loads the library holds its own copy at its own address until
// the process ends.  In host code the name is only a handle for hipGetSymbolAddress: the address a
// kernel may use is looked up once per handle (mi_moe_create, on the handle's device) and kept there.
// A batch is taken whose least workspace (ForwardWs::bytes_min) is MI_MOE_STATIC_SCRATCH_BYTES or less.  The same again lies behind it for what the tiles on raw
// codes want beyond that (bytes_raw), so that such a batch takes the kernels that mi_moe_forward gives it.  That is never more: the copy of x has the size of the
// normalised rows, its group sums at most that of the down product's rows, those of h at most h's (K is a multiple of 128 there, and 16 groups of sums, to whole
// numbers of which they are padded, are no larger than 128 values), and a list of at least four rows a segment is smaller than two of the arrays of pairs.  Records of
// several a segment, where there are no tiles, are the experts' and 8 bytes a pair, less than the pairs' rows.
constexpr size_t kStaticScratch = (size_t)2 * MI_MOE_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratch];

// Prefill-sized batches: the tile classes and the streamed segments are independent chains (gate/up then
// down over the same rows); three of the four run on side streams, forked from and joined back into the
// caller's stream by events.  The streams and events belong to the GPU, not to a handle: one set per
// device for the whole process, created by the first mi_moe_create on that device and kept until the
// process ends (a model of 48 to 94 layers would otherwise hold 150 to 280 streams on a device with a
// handful of hardware queues).  The host-side fork ... join sequence of a forward runs under the set's
// lock: an event is recorded and waited for by the same forward, never by two at once.
struct DeviceStreams {
  std::mutex lock;
  bool ready = false;
  hipStream_t side[3] = {nullptr, nullptr, nullptr};
  hipEvent_t fork = nullptr, paired = nullptr, join[3] = {nullptr, nullptr, nullptr};
};
constexpr int kMaxStreamDevices = 64;
static DeviceStreams g_device_streams[kMaxStreamDevices];
static std::atomic<int> g_side_streams_created{0};

// the set of `dev` (the current device), created on first use (default priority)
static hipError_t device_streams(int dev, DeviceStreams **out) {
  if (dev < 0 || dev >= kMaxStreamDevices) return hipErrorInvalidDevice;
  DeviceStreams &d = g_device_streams[dev];
  std::lock_guard<std::mutex> g(d.lock);
  if (!d.ready) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < 3 && e == hipSuccess; ++i) {
      if (!d.side[i]) {
        e = hipStreamCreateWithFlags(&d.side[i], hipStreamNonBlocking);
        if (e == hipSuccess) g_side_streams_created.fetch_add(1);
      }
      if (e == hipSuccess && !d.join[i]) e = hipEventCreateWithFlags(&d.join[i], hipEventDisableTiming);
    }
    if (e == hipSuccess && !d.fork) e = hipEventCreateWithFlags(&d.fork, hipEventDisableTiming);
    if (e == hipSuccess && !d.paired) e = hipEventCreateWithFlags(&d.paired, hipEventDisableTiming);
    if (e != hipSuccess) return e;  // what exists is kept for the next attempt
    d.ready = true;
  }
  *out = &d;
  return hipSuccess;
}

// Whether work of `st` may be forked to `side`.  A stream that a capture has forked to stays in it until the capture ends, also
// where it has been joined back: work of another stream would be recorded in that graph instead of run, and its stream with it.
static bool may_fork(hipStream_t st, hipStream_t side) {
  hipStreamCaptureStatus of_side = hipStreamCaptureStatusNone, of_st = hipStreamCaptureStatusNone;
  unsigned long long id_side = 0, id_st = 0;
  if (hipStreamGetCaptureInfo(side, &of_side, &id_side) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  if (of_side == hipStreamCaptureStatusNone) return true;
  if (hipStreamGetCaptureInfo(st, &of_st, &id_st) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return of_side == hipStreamCaptureStatusActive && of_st == hipStreamCaptureStatusActive && id_side == id_st;
}
// The same for all of a device's side streams, whose lock the caller holds.
static bool may_fork(hipStream_t st, const DeviceStreams &ds) {
  for (hipStream_t s : ds.side)
    if (!may_fork(st, s)) return false;
  return true;
}

struct mi_moe_s {
  mi_moe_config cfg;
  mi_moe_weights w;
  int device = -1;                       // the GPU that was current in mi_moe_create: counters, streams, scratch live there
  unsigned char *scratch_dev = nullptr;  // device address of `scratch` on the handle's GPU
  uint32_t *counters = nullptr;  // device: arrival counters of the fused decode router, zero at rest
  DeviceStreams *streams = nullptr;      // the device's side streams and events (not owned)
};

void destroy_handle(mi_moe_s *h) {
  if (!h) return;
  if (h->counters) (void)hipFree(h->counters);
  delete h;
}

extern "C" {

const char *mi_moe_last_error(void) { return g_last_error; }

void mi_moe_set_error_handler(void (*handler)(const char *, void *), void *data,
                              void (*dtor)(void *)) try {
  std::shared_ptr<Handler> next, old;
  if (handler || data || dtor) next = std::make_shared<Handler>(Handler{handler, data, dtor});
  {
    std::lock_guard<std::mutex> g(g_handler_lock);
    old = std::move(g_handler);
    g_handler = std::move(next);
  }
  // `old` goes here, outside the lock: its dtor runs once no failing thread still uses it
} catch (...) {
  // out of host memory: the previous handler stays
}

const char *mi_moe_version(void) { return "mi_moe 0.1 gfx950"; }

int mi_moe_create(const mi_moe_config *cfg, const mi_moe_weights *weights, mi_moe_handle *out) try {
  if (!out) return fail("create: out handle is NULL");
  if (check_config(cfg)) return 1;
  if (!weights) return fail("create: weights is NULL");
  if (!weights->router_w || !aligned16(weights->router_w))
    return fail("create: router_w must be non-NULL and 16-byte aligned");
  if (check_qmat(weights->gate, "gate") || check_qmat(weights->up, "up") || check_qmat(weights->down, "down"))
    return 1;
  mi_moe_s *h = new (std::nothrow) mi_moe_s;
  if (!h) return fail("create: out of host memory");
  h->cfg = *cfg;
  h->w = *weights;
  // the only device memory the library owns: 260 bytes of counters per handle
  const size_t cbytes = (size_t)(1 + kFusedRouterMaxTokens) * sizeof(uint32_t);
  hipError_t e = hipGetDevice(&h->device);
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&h->counters), cbytes);
  if (e == hipSuccess) e = hipMemset(h->counters, 0, cbytes);
  // the device's streams and events for the independent chains of a prefill-sized forward
  if (e == hipSuccess) e = device_streams(h->device, &h->streams);
  // where the built-in scratch of mi_moe_forward_static lives on this GPU
  if (e == hipSuccess) e = hipGetSymbolAddress(reinterpret_cast<void **>(&h->scratch_dev), HIP_SYMBOL(scratch));
  if (e == hipSuccess && (!h->scratch_dev || (reinterpret_cast<uintptr_t>(h->scratch_dev) & 255u))) e = hipErrorInvalidSymbol;
  if (e != hipSuccess) {
    destroy_handle(h);
    return fail("create: device memory, streams and events of the handle: %s", hipGetErrorString(e));
  }
  *out = h;
  return 0;
} MI_CATCH("create")

int mi_moe_destroy(mi_moe_handle h) try {
  destroy_handle(h);
  return 0;
} MI_CATCH("destroy")

int mi_moe_workspace_size(const mi_moe_config *cfg, int64_t max_tokens, size_t *bytes) try {
  if (!bytes) return fail("workspace_size: bytes is NULL");
  if (check_config(cfg)) return 1;
  if (max_tokens < 0) return fail("workspace_size: negative token count");
  if (max_tokens * cfg->top_k > (int64_t)1 << 30) return fail("workspace_size: too many (token, expert) pairs");
  // A caller keeps one workspace for its largest batch: it has to hold what every smaller one takes.  That grows with the tokens except where a route ends whose regions
  // the next one does without: 8-bit batches of a few rows an expert, and operands that reach 2 GiB.
  const mi_moe_config &c = *cfg;
  auto last_of = [](int64_t most, auto takes) {  // up to `most` tokens, the largest batch of a route that takes all smaller ones
    int64_t lo = 0, hi = most;
    while (lo < hi) {
      const int64_t mid = lo + (hi - lo + 1) / 2;
      if (takes(mid)) lo = mid;
      else hi = mid - 1;
    }
    return lo;
  };
  const int64_t fits = last_of(max_tokens, [&](int64_t T) { return codes_tiles_fit(c, T); });
  const int64_t few = last_of(fits, [&](int64_t T) { return few_rows_batch(c, T); });
  size_t most = 0;
  for (const int64_t T : {max_tokens, fits, few}) {
    const size_t need = carve_forward(c, T, nullptr, true).bytes;
    most = need > most ? need : most;
  }
  *bytes = most + 256;
  return 0;
} MI_CATCH("workspace_size")

// The operands of the two grouped products of a forward: gate/up (rows gathered from x by token, written
// in sorted order, SwiGLU fused) and down (rows read in sorted order, written back in (token, slot) order).
static void grouped_args(const mi_moe_config &c, const mi_moe_weights &w, const ForwardWs &f, const uint16_t *x,
                         int64_t T, GroupedArgs &a, GroupedArgs &d) {
  const int64_t P = T * c.top_k;
  const bool paired = c.bits == 4;
  a = GroupedArgs{};
  a.work = f.records.at;
  a.max_active = (int)(P < c.n_experts ? P : c.n_experts);
  a.max_records = f.records.slots;
  const bool lists = f.tiled && !f.pieces;
  a.mtiles = lists ? f.mtiles : nullptr;
  a.max_mtiles = f.max_mtiles;
  a.tile_cap_e = lists ? c.n_experts : 0;
  a.bits = c.bits;
  a.total_rows = P;
  a.max_rows_per_expert = T;  // a token picks an expert at most once
  a.max_streamed_rows = f.tiled ? f.tmr - 1 : 0;
  a.x = x;
  a.x_perm = paired ? (f.tiled ? f.xperm : nullptr) : x;
  a.x_paired = false;
  a.y_paired = paired;
  a.src_rows = f.src_of;
  a.src_in_work = true;
  a.dst_rows = nullptr;
  a.w0 = w.gate.w; a.s0 = w.gate.scales; a.b0 = w.gate.biases;
  a.w1 = w.up.w;   a.s1 = w.up.scales;   a.b1 = w.up.biases;
  a.y = f.hh;
  a.N = c.intermediate;
  a.K = c.hidden;
  d = a;
  d.x = f.hh;
  d.x_perm = f.hh;
  d.x_paired = paired;
  d.y_paired = false;
  d.src_rows = nullptr;
  d.src_in_work = false;
  d.dst_rows = f.perm;
  d.w0 = w.down.w; d.s0 = w.down.scales; d.b0 = w.down.biases;
  d.w1 = nullptr; d.s1 = d.b1 = nullptr;
  d.y = f.y;
  d.N = c.hidden;
  d.K = c.intermediate;
}

// The launch sequence of one forward.  ev: nullptr, or kStages + 1 events recorded on the
// stream before the first launch and after each stage.
// kt: nullptr, or MI_MOE_N_KERNEL_TIMES timers for the grouped-product kernels (with ev).
static int forward_impl(mi_moe_handle h, const uint16_t *x_in, int64_t T, uint16_t *out, void *workspace,
                        size_t workspace_bytes, const mi_moe_debug_out *dbg, hipStream_t st,
                        hipEvent_t *ev, const uint16_t *norm_weight = nullptr, float eps = 0.f,
                        KernelTimer *kt = nullptr) {
  const uint16_t *x = x_in;
  if (!h) return fail("forward: handle is NULL");
  if (T < 0) return fail("forward: negative token count");
  if (T == 0) return 0;
  if (!x || !out) return fail("forward: x and out must be non-NULL");
  if (!aligned16(x) || !aligned16(out)) return fail("forward: x and out must be 16-byte aligned");
  int dev = -1;
  MI_HIP(hipGetDevice(&dev));
  if (dev != h->device)
    return fail("forward: the handle was created on GPU %d, the calling thread's current GPU is %d", h->device, dev);
  const mi_moe_config &c = h->cfg;
  const int64_t P = T * c.top_k;
  if (P > (int64_t)1 << 30) return fail("forward: too many (token, expert) pairs");
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255u))
    return fail("forward: workspace must be non-NULL and 256-byte aligned");
  ForwardWs f = carve_forward(c, T, workspace, norm_weight != nullptr);
  if (workspace_bytes < f.bytes_min)
    return fail("forward: workspace too small (%zu bytes, need %zu)", workspace_bytes, f.bytes);
  if (workspace_bytes < f.bytes_raw) {
    f.raw_tiles = nullptr;
    f.mid = f.pieces = f.raw_all = false;
    f.records = Records(f.work);
  }
  if (workspace_bytes < f.bytes) f.router_scratch = nullptr;  // room for everything but the byte planes: fp64 logits, same bits
  int stage = 0;
#define MI_STAGE_DONE()                                  \
  do {                                                   \
    if (ev) MI_HIP(hipEventRecord(ev[++stage], st));     \
  } while (0)
  if (ev) MI_HIP(hipEventRecord(ev[0], st));
  const bool fused_router = router_fused_applies(T, c.n_experts, c.top_k);
  const bool mid = f.mid, raw_codes = mid || f.pieces;
  uint32_t *const tile_lists = f.tiled && !raw_codes ? f.mtiles : nullptr;
  const int tile_cap = f.max_mtiles, tile_from = f.tmr;
  const ShortTiles shorts = {raw_codes || f.raw ? f.raw_tiles : nullptr, (uint32_t)f.raw_from, (uint32_t)f.raw_piece};
  const Records records = mid && !fused_router ? Records() : f.records;
  if (norm_weight) {  // the block's input is rms_norm(x); x itself is added back in the combine
    if (!fused_router) MI_HIP(launch_rms_norm(x_in, norm_weight, eps, T, c.hidden, f.xnorm, st));
    x = f.xnorm;      // decode: written by the router kernel below
  }

  // 4-bit: the tiled kernel reads activations with paired 8-blocks; h is produced that way, x is copied once
  // per forward (prefill-sized T only): by the router's logits kernel, which holds every piece of x in
  // registers anyway, or by a kernel of its own (light batches pair the rows beside their streamed segments)
  const bool paired = c.bits == 4;
  const bool streamed_first = f.tiled && !f.heavy && !ev && !mid;  // light batches start their streamed segments first
  const bool pair_in_router = f.tiled && paired && !raw_codes && !streamed_first && !fused_router && !plain_config(c) &&
                              router_logits_pairs_rows(T, c.hidden);
  if (fused_router) {
    // decode: one launch for the three stages (the stage times then all land in the first)
    MI_HIP(launch_router_fused(x_in, h->w.router_w, h->w.router_bias, norm_weight, eps, f.xnorm, T, c.hidden,
                               c.n_experts, c.top_k,
                               c.score_mode, f.logits, f.topk_idx, f.topk_w, h->counters, f.counts, f.offsets,
                               f.perm, f.inv_perm, f.src_of, records, tile_lists, tile_cap, tile_from, shorts, st));
    MI_STAGE_DONE();
    MI_STAGE_DONE();
    MI_STAGE_DONE();
  } else {
    // Which route the logits take (all three give the same bits).  Measured, 128 experts, hidden 2048, logits +
    // selection, us at 1024 / 2048 / 4096 / 8192 tokens: fp64 matrix cores 19.9 / 27.0 / 45.7 / 81.6; byte planes +
    // int8 product, selection apart 22.5 / 26.5 / 39.7 / 64.1; one kernel per 32 tokens (planes in LDS, selection
    // included; a block's phases follow each other, and there are T / 32 blocks) 41.3 / 41.9 / 45.2 / 49.5.
    const int64_t logit_work = T * (int64_t)c.hidden * ((c.n_experts + 127) / 128);
    const bool i8_pays = f.router_scratch && logit_work >= (int64_t)3 << 20;
    if (i8_pays && logit_work >= (int64_t)12 << 20 && router_tile_applies(T, c.hidden, c.n_experts, c.top_k)) {
      // logits and selection in one kernel (the stage times both land in the first)
      MI_HIP(launch_router_tile(x, h->w.router_w, h->w.router_bias, T, c.hidden, c.n_experts, c.top_k, c.score_mode,
                                f.logits, f.topk_idx, f.topk_w, f.router_scratch, st, pair_in_router ? f.xperm : nullptr));
      MI_STAGE_DONE();
      MI_STAGE_DONE();
    } else {
      if (i8_pays)
        MI_HIP(launch_router_logits_i8(x, h->w.router_w, h->w.router_bias, T, c.hidden, c.n_experts, f.logits,
                                       f.router_scratch, st, pair_in_router ? f.xperm : nullptr));
      else
        MI_HIP(launch_router_logits(x, h->w.router_w, h->w.router_bias, T, c.hidden, c.n_experts, f.logits, st,
                                    pair_in_router ? f.xperm : nullptr));
      MI_STAGE_DONE();
      MI_HIP(launch_router_select(f.logits, T, c.n_experts, c.top_k, c.score_mode, f.topk_idx, f.topk_w, st));
      MI_STAGE_DONE();
    }
    MI_HIP(launch_dispatch(f.topk_idx, P, c.n_experts, c.top_k, f.counts, f.offsets, f.perm, f.inv_perm,
                           f.src_of, records, tile_lists, tile_cap, tile_from, shorts,
                           mid || f.raw_all || (f.pieces && c.bits == 4)
                               ? prepare_args(x, T, c.hidden, c.group_size, codes_copy_bytes(c.bits, T, c.hidden) ? f.raw_copy : nullptr, f.raw_xsums, raw_codes && c.bits == 4)
                               : PrepareArgs{}, f.disp_scratch, st));
    MI_STAGE_DONE();
  }
  GroupedArgs a{}, d{};
  grouped_args(c, h->w, f, x, T, a, d);
  const int max_active = a.max_active;
  if (f.tiled && paired && !streamed_first && !pair_in_router && !raw_codes) MI_HIP(launch_pair_rows(x, T, c.hidden, f.xperm, st));
  // independent chains run beside each other where side streams are to be had, whose lock is held until they have been joined back
  std::unique_lock<std::mutex> streams_guard;
  const bool chains = !ev && !mid && !f.raw_all && !plain_config(c) && large_qmm_applies(a);
  if (chains) streams_guard = std::unique_lock<std::mutex>(h->streams->lock);
  const bool fork = chains && may_fork(st, *h->streams);
  if (!fork && streamed_first && paired && large_qmm_applies(a)) MI_HIP(launch_pair_rows(x, T, c.hidden, f.xperm, st));  // (a side stream's work)
  // the pieces
  CodesArgs ca{}, cd{};
  const bool copied = codes_copy_bytes(c.bits, T, c.hidden) > 0;
  ca.x = copied ? f.raw_copy : x;
  ca.x_rows = T;
  ca.sums = f.raw_xsums;
  ca.src_rows = f.src_of;
  ca.w0 = h->w.gate.w; ca.s0 = h->w.gate.scales; ca.b0 = h->w.gate.biases;
  ca.w1 = h->w.up.w; ca.s1 = h->w.up.scales; ca.b1 = h->w.up.biases;
  ca.y = f.hh;
  ca.y_order = copied ? RowOrder::kQuads : RowOrder::kPlain;
  ca.y_sums = f.raw_hsums;
  ca.N = c.intermediate; ca.K = c.hidden;
  cd.x = f.hh;
  cd.x_rows = P;
  cd.sums = f.raw_hsums;
  cd.dst_rows = f.perm;
  cd.w0 = h->w.down.w; cd.s0 = h->w.down.scales; cd.b0 = h->w.down.biases;
  cd.y = f.y;
  cd.N = c.hidden; cd.K = c.intermediate;
  auto tiles_up = [&](hipStream_t s) -> hipError_t {
    if (f.pieces && c.bits == 8) return launch_qmm_bytes(ca, f.raw_tiles, f.raw_cap, true, s);
    if (f.raw_piece > kShortTileM) return launch_qmm_pieces(ca, f.raw_tiles, f.raw_cap, true, s);
    return launch_qmm_short(ca, f.raw_tiles, f.raw_cap, c.group_size, c.bits, true, s);
  };
  auto tiles_down = [&](hipStream_t s) -> hipError_t {
    if (f.pieces && c.bits == 8) return launch_qmm_bytes(cd, f.raw_tiles, f.raw_cap, false, s);
    if (f.raw_piece > kShortTileM) return launch_qmm_pieces(cd, f.raw_tiles, f.raw_cap, false, s);
    return launch_qmm_short(cd, f.raw_tiles, f.raw_cap, c.group_size, c.bits, false, s);
  };
  struct TimerScope {  // a timer never outlives the launch it is meant for
    explicit TimerScope(KernelTimer *t) { g_kernel_timer = t; }
    ~TimerScope() { g_kernel_timer = nullptr; }
  };
  if (mid) {
    if (fused_router) MI_HIP(launch_prepare_rows(x, T, c.hidden, c.group_size, MI_MOE_DTYPE_BF16, true, nullptr, f.raw_xsums, st));  // (8-bit codes: no copy)
    {
      TimerScope scope(kt ? &kt[2] : nullptr);
      MI_HIP(tiles_up(st));
    }
    MI_STAGE_DONE();
    {
      TimerScope scope(kt ? &kt[4 + 2] : nullptr);
      MI_HIP(tiles_down(st));
    }
    MI_STAGE_DONE();
  } else if (f.pieces) {
    for (int half = 0; half < 2; ++half) {
      {
        TimerScope scope(kt ? &kt[4 * half + 3] : nullptr);
        MI_HIP(launch_small_qmm(half == 0 ? a : d, half == 0, st));
      }
      {
        TimerScope scope(kt ? &kt[4 * half + 2] : nullptr);
        MI_HIP(half == 0 ? tiles_up(st) : tiles_down(st));
      }
      MI_STAGE_DONE();
    }
  } else if (f.raw_all) {
    if (fused_router)
      MI_HIP(launch_prepare_rows(x, T, c.hidden, c.group_size, MI_MOE_DTYPE_BF16, true, copied ? f.raw_copy : nullptr, f.raw_xsums, st));
    MI_HIP(tiles_up(st));
    MI_STAGE_DONE();
    MI_HIP(tiles_down(st));
    MI_STAGE_DONE();
  } else if (f.raw) {
    // group sizes 32 / 128 without lists: the kernel of a few rows
    RowsArgs ra{}, rd{};
    ra.work = f.records.at;
    ra.max_active = max_active;
    ra.max_records = f.records.slots;
    ra.max_rows = T;
    rd = ra;
    ra.x = x;
    ra.src_rows = f.src_of;
    ra.src_in_work = true;
    ra.w0 = h->w.gate.w; ra.s0 = h->w.gate.scales; ra.b0 = h->w.gate.biases;
    ra.w1 = h->w.up.w; ra.s1 = h->w.up.scales; ra.b1 = h->w.up.biases;
    ra.y = f.hh;
    ra.N = c.intermediate; ra.K = c.hidden;
    rd.x = f.hh;
    rd.dst_rows = f.perm;
    rd.w0 = h->w.down.w; rd.s0 = h->w.down.scales; rd.b0 = h->w.down.biases;
    rd.y = f.y;
    rd.N = c.hidden; rd.K = c.intermediate;
    MI_HIP(launch_qmm_rows(ra, c.group_size, c.bits, MI_MOE_DTYPE_BF16, true, st));
    MI_STAGE_DONE();
    MI_HIP(launch_qmm_rows(rd, c.group_size, c.bits, MI_MOE_DTYPE_BF16, false, st));
    MI_STAGE_DONE();
  } else if (plain_config(c)) {
    // 2-bit codes, or rows the kernels on raw codes do not take: the plain products, one output row per sorted pair.  Row r of
    // the sorted order belongs to pair perm[r], token src_of[r], expert topk_idx[perm[r]].
    const size_t PI = (size_t)P * c.intermediate;
    MI_HIP(launch_qmm_plain(x, h->w.gate.w, h->w.gate.scales, h->w.gate.biases, f.src_of, f.topk_idx, f.perm, nullptr,
                            (uint32_t)T, (uint32_t)c.n_experts, P, 1, c.intermediate, c.hidden, c.group_size, c.bits, true, MI_MOE_DTYPE_BF16, f.gu, st));
    MI_HIP(launch_qmm_plain(x, h->w.up.w, h->w.up.scales, h->w.up.biases, f.src_of, f.topk_idx, f.perm, nullptr,
                            (uint32_t)T, (uint32_t)c.n_experts, P, 1, c.intermediate, c.hidden, c.group_size, c.bits, true, MI_MOE_DTYPE_BF16, f.gu + PI, st));
    MI_HIP(launch_swiglu(f.gu, f.gu + PI, (int64_t)PI, f.hh, st));
    MI_STAGE_DONE();
    MI_HIP(launch_qmm_plain(f.hh, h->w.down.w, h->w.down.scales, h->w.down.biases, nullptr, f.topk_idx, f.perm, f.perm,
                            0u, (uint32_t)c.n_experts, P, 1, c.hidden, c.intermediate, c.group_size, c.bits, true, MI_MOE_DTYPE_BF16, f.y, st));
    MI_STAGE_DONE();
  } else if (fork) {
    // Four chains that share no rows: the three tile classes and the streamed segments, each
    // gate/up then down.  The short classes leave most of the chip idle when they run alone
    // (a few dozen workgroups of 64 K steps each); side by side they fill it.  The chain that is
    // expected to be the longest stays on the caller's stream and is launched first (the others
    // start a cross-stream wait later, and the join waits for them): the tile class of the average
    // segment in a heavy batch, the streamed segments of a light one (whose tile lists are empty
    // unless the routing is uneven; the copy of x with paired rows, which only the tiles read,
    // then runs on a side stream as well).
    // A segment is at most T rows long: a class that cannot occur gets no stream (a fork and a
    // join cost a few microseconds each).
    const bool exists[4] = {T > 128, T > 64, true, true};
    int n_side = 0;
    DeviceStreams &ds = *h->streams;
    MI_HIP(hipEventRecord(ds.fork, st));
    // the launches, in a function of their own: whatever happens in it, the side streams it has
    // used are joined back below (a caller must never be left with work of ours running beside
    // its stream, or with a capture that has not been joined)
    auto launch_chains = [&]() -> int {
      if (streamed_first) {
        MI_HIP(launch_small_qmm(a, true, st));
        MI_HIP(launch_small_qmm(d, false, st));
        for (int cls = 0; cls < 3; ++cls) {
          if (!exists[cls]) continue;
          hipStream_t s = ds.side[n_side++];
          if (n_side == 1) {
            MI_HIP(hipStreamWaitEvent(s, ds.fork, 0));
            if (paired) {
              MI_HIP(launch_pair_rows(x, T, c.hidden, f.xperm, s));
              MI_HIP(hipEventRecord(ds.paired, s));
            }
          } else {
            MI_HIP(hipStreamWaitEvent(s, paired ? ds.paired : ds.fork, 0));
          }
          MI_HIP(launch_large_qmm_class(a, true, cls, s));
          MI_HIP(launch_large_qmm_class(d, false, cls, s));
        }
      } else {
        // which class is the longest depends on the routing, which the host does not see; it takes
        // the class of the average segment (even routing: 320 to 2048 tokens of the 128-expert shape
        // -9 % against always leading with the 256-row class; zipf-1.1 routing: +4 to +6 % there)
        const int64_t avg_rows = P / (max_active > 0 ? max_active : 1);
        const int lead = avg_rows <= 64 ? 2 : (avg_rows <= 128 ? 1 : 0);
        // With the 256-row class in the lead (more than 128 rows per expert on average) the other three chains
        // follow each other on ONE side stream: two kernels share the chip at a time instead of four, and the
        // 256-row launches are stretched less (128-expert shape, 2560 to 8192 tokens, Zipf and even routing:
        // -1.3 to -5.5 %; Mixtral shape: no change).  With a shorter class in the lead the side chains hold most
        // of the rows and need a stream each (one stream for them at 320 to 2048 tokens, Zipf routing: +10 to +36 %).
        const bool one_side = lead == 0;
        if (one_side) {
          hipStream_t s = ds.side[n_side++];
          MI_HIP(hipStreamWaitEvent(s, ds.fork, 0));
          MI_HIP(launch_large_qmm_class(a, true, 0, st));
          MI_HIP(launch_large_qmm_class(d, false, 0, st));
          // the side stream: every gate/up launch, then every down launch (against chain after chain: -0.6 %)
          for (int cls = 1; cls <= 2; ++cls) MI_HIP(launch_large_qmm_class(a, true, cls, s));
          MI_HIP(launch_small_qmm(a, true, s));
          for (int cls = 1; cls <= 2; ++cls) MI_HIP(launch_large_qmm_class(d, false, cls, s));
          MI_HIP(launch_small_qmm(d, false, s));
          return 0;
        }
        for (int i = 0; i < 4; ++i) {
          const int chain = i == 0 ? lead : (i <= lead ? i - 1 : i);
          if (!exists[chain]) continue;
          hipStream_t s = st;
          if (i > 0) {
            s = ds.side[n_side++];
            MI_HIP(hipStreamWaitEvent(s, ds.fork, 0));
          }
          if (chain < 3) {
            MI_HIP(launch_large_qmm_class(a, true, chain, s));
            MI_HIP(launch_large_qmm_class(d, false, chain, s));
          } else {
            MI_HIP(launch_small_qmm(a, true, s));
            MI_HIP(launch_small_qmm(d, false, s));
          }
        }
      }
      return 0;
    };
    const int rc = launch_chains();
    hipError_t je = hipSuccess;
    for (int i = 0; i < n_side; ++i) {
      hipError_t e = hipEventRecord(ds.join[i], ds.side[i]);
      if (e == hipSuccess) e = hipStreamWaitEvent(st, ds.join[i], 0);
      if (e != hipSuccess && je == hipSuccess) je = e;
    }
    if (rc) return rc;
    MI_HIP(je);
  } else if (kt) {
    // one kernel after the other, each dispatch with a timer of its own: tile classes 0, 1, 2 (the
    // 256-, 128- and 64-row lists), then the streamed segments; gate/up first, then down
    for (int half = 0; half < 2; ++half) {
      const GroupedArgs &g = half == 0 ? a : d;
      for (int cls = 0; cls < 3; ++cls) {
        TimerScope scope(&kt[4 * half + cls]);
        MI_HIP(launch_large_qmm_class(g, half == 0, cls, st));
      }
      {
        TimerScope scope(&kt[4 * half + 3]);
        MI_HIP(launch_small_qmm(g, half == 0, st));
      }
      MI_STAGE_DONE();
    }
  } else {
    MI_HIP(launch_grouped_qmm(a, true, st));
    MI_STAGE_DONE();
    MI_HIP(launch_grouped_qmm(d, false, st));
    MI_STAGE_DONE();
  }
  if (streams_guard.owns_lock()) streams_guard.unlock();
  MI_HIP(launch_combine(f.y, f.topk_w, nullptr, T, c.top_k, c.hidden, norm_weight ? x_in : nullptr, out, st));
  MI_STAGE_DONE();
#undef MI_STAGE_DONE

  if (dbg) {
    if (dbg->topk_idx) MI_HIP(hipMemcpyAsync(dbg->topk_idx, f.topk_idx, P * 4, hipMemcpyDeviceToDevice, st));
    if (dbg->topk_w) MI_HIP(hipMemcpyAsync(dbg->topk_w, f.topk_w, P * 2, hipMemcpyDeviceToDevice, st));
    if (dbg->counts) MI_HIP(hipMemcpyAsync(dbg->counts, f.counts, c.n_experts * 4, hipMemcpyDeviceToDevice, st));
    if (dbg->offsets) MI_HIP(hipMemcpyAsync(dbg->offsets, f.offsets, (c.n_experts + 1) * 4, hipMemcpyDeviceToDevice, st));
    if (dbg->perm) MI_HIP(hipMemcpyAsync(dbg->perm, f.perm, P * 4, hipMemcpyDeviceToDevice, st));
    if (dbg->inv_perm) MI_HIP(hipMemcpyAsync(dbg->inv_perm, f.inv_perm, P * 4, hipMemcpyDeviceToDevice, st));
  }
  return 0;
}

int mi_moe_forward(mi_moe_handle h, const uint16_t *x, int64_t T, uint16_t *out, void *workspace,
                   size_t workspace_bytes, const mi_moe_debug_out *dbg, void *stream) try {
  return forward_impl(h, x, T, out, workspace, workspace_bytes, dbg, static_cast<hipStream_t>(stream), nullptr);
} MI_CATCH("forward")

int mi_moe_forward_static(mi_moe_handle h, const uint16_t *x, int64_t T, uint16_t *out,
                          const mi_moe_debug_out *dbg, void *stream) try {
  if (!h) return fail("forward_static: handle is NULL");
  if (T < 0) return fail("forward_static: negative token count");
  if (T * (int64_t)h->cfg.top_k > (int64_t)1 << 30) return fail("forward_static: too many (token, expert) pairs");
  const ForwardWs f = carve_forward(h->cfg, T, nullptr, false);
  const size_t need = f.bytes_min;
  if (need > (size_t)MI_MOE_STATIC_SCRATCH_BYTES)
    return fail("forward_static: %lld tokens of this layer need %zu bytes of workspace, the built-in scratch holds %zu "
                "(use mi_moe_forward with a workspace of the caller's)",
                (long long)T, need, (size_t)MI_MOE_STATIC_SCRATCH_BYTES);
  // no allocation from here on: the kernels get the address looked up by mi_moe_create
  return forward_impl(h, x, T, out, h->scratch_dev, f.bytes_raw < kStaticScratch ? f.bytes_raw : kStaticScratch, dbg, static_cast<hipStream_t>(stream), nullptr);
} MI_CATCH("forward_static")

int mi_moe_forward_residual(mi_moe_handle h, const uint16_t *x, const uint16_t *norm_weight, float eps,
                            int64_t T, uint16_t *out, void *workspace, size_t workspace_bytes,
                            const mi_moe_debug_out *dbg, void *stream) try {
  if (!norm_weight || !aligned16(norm_weight)) return fail("forward_residual: norm_weight must be non-NULL and 16-byte aligned");
  if (!(eps >= 0.f)) return fail("forward_residual: eps must be non-negative");
  if (x == out) return fail("forward_residual: out must not alias x (x is read again at the end)");
  return forward_impl(h, x, T, out, workspace, workspace_bytes, dbg, static_cast<hipStream_t>(stream), nullptr,
                      norm_weight, eps);
} MI_CATCH("forward_residual")

int mi_moe_rms_norm(const uint16_t *x, const uint16_t *weight, float eps, int64_t T, int32_t hidden,
                    uint16_t *out, void *stream) try {
  if (T < 0) return fail("rms_norm: negative row count");
  if (hidden <= 0 || hidden % 8) return fail("rms_norm: hidden must be a positive multiple of 8, got %d", hidden);
  if (!(eps >= 0.f)) return fail("rms_norm: eps must be non-negative");
  if (T == 0) return 0;
  if (!x || !weight || !out) return fail("rms_norm: x, weight and out must be non-NULL");
  if (!aligned16(x) || !aligned16(weight) || !aligned16(out)) return fail("rms_norm: pointers must be 16-byte aligned");
  MI_HIP(launch_rms_norm(x, weight, eps, T, hidden, out, static_cast<hipStream_t>(stream)));
  return 0;
} MI_CATCH("rms_norm")

int mi_moe_forward_timed(mi_moe_handle h, const uint16_t *x, int64_t T, uint16_t *out, void *workspace,
                         size_t workspace_bytes, void *stream, float *stage_ms, float *kernel_ms) try {
  if (!stage_ms) return fail("forward_timed: stage_ms is NULL");
  for (int i = 0; i < MI_MOE_N_STAGES; ++i) stage_ms[i] = 0.f;  // what an empty batch or a failed call leaves
  hipStream_t st = static_cast<hipStream_t>(stream);
  constexpr int kEvents = MI_MOE_N_STAGES + 1 + 2 * MI_MOE_N_KERNEL_TIMES;
  hipEvent_t ev[kEvents];
  for (int i = 0; i < kEvents; ++i) {
    const hipError_t e = hipEventCreate(&ev[i]);
    if (e != hipSuccess) {
      while (--i >= 0) (void)hipEventDestroy(ev[i]);
      return hip_fail("hipEventCreate", e);
    }
  }
  KernelTimer kt[MI_MOE_N_KERNEL_TIMES];
  for (int i = 0; i < MI_MOE_N_KERNEL_TIMES; ++i) {
    kt[i].start = ev[MI_MOE_N_STAGES + 1 + 2 * i];
    kt[i].stop = ev[MI_MOE_N_STAGES + 2 + 2 * i];
  }
  int rc = forward_impl(h, x, T, out, workspace, workspace_bytes, nullptr, st, ev, nullptr, 0.f, kt);
  if (kernel_ms)
    for (int i = 0; i < MI_MOE_N_KERNEL_TIMES; ++i) kernel_ms[i] = 0.f;
  if (rc == 0 && T > 0) {
    hipError_t e = hipEventSynchronize(ev[MI_MOE_N_STAGES]);
    if (e != hipSuccess) rc = hip_fail("hipEventSynchronize", e);
    for (int i = 0; rc == 0 && i < MI_MOE_N_STAGES; ++i) {
      e = hipEventElapsedTime(&stage_ms[i], ev[i], ev[i + 1]);
      if (e != hipSuccess) rc = hip_fail("hipEventElapsedTime", e);
    }
    for (int i = 0; rc == 0 && kernel_ms && i < MI_MOE_N_KERNEL_TIMES; ++i) {
      if (!kt[i].used) continue;
      e = hipEventElapsedTime(&kernel_ms[i], kt[i].start, kt[i].stop);
      if (e != hipSuccess) rc = hip_fail("hipEventElapsedTime (kernel)", e);
    }
  }
  for (int i = 0; i < kEvents; ++i) (void)hipEventDestroy(ev[i]);
  return rc;
} MI_CATCH("forward_timed")

// ------------------------------------------------------------------ stage level

int mi_moe_route_workspace_size(int32_t n_experts, int64_t T, size_t *bytes) try {
  if (!bytes) return fail("route_workspace_size: bytes is NULL");
  if (n_experts < 1 || n_experts > 512 || T < 0) return fail("route_workspace_size: bad arguments");
  *bytes = align_up((size_t)T * n_experts * 2) + 256;
  return 0;
} MI_CATCH("route_workspace_size")

int mi_moe_route(const uint16_t *x, const uint16_t *router_w, const float *router_bias, int64_t T,
                 int32_t hidden, int32_t n_experts, int32_t top_k, int32_t score_mode,
                 uint32_t *topk_idx, uint16_t *topk_w, uint16_t *logits_out, void *workspace,
                 size_t workspace_bytes, void *stream) try {
  if (T < 0) return fail("route: negative token count");
  if (hidden <= 0 || hidden % 64) return fail("route: hidden must be a positive multiple of 64, got %d", hidden);
  if (n_experts < 1 || n_experts > 512) return fail("route: n_experts must be in [1, 512], got %d", n_experts);
  if (top_k < 1 || top_k > n_experts || top_k > 32)
    return fail("route: top_k must be in [1, min(n_experts, 32)], got %d", top_k);
  if (score_mode < 0 || score_mode > 2) return fail("route: unknown score_mode %d", score_mode);
  if (T == 0) return 0;
  if (!x || !router_w || !topk_idx || !topk_w) return fail("route: x, router_w, topk_idx and topk_w must be non-NULL");
  if (!aligned16(x) || !aligned16(router_w)) return fail("route: x and router_w must be 16-byte aligned");
  uint16_t *logits = logits_out;
  if (!logits) {
    if (!workspace || workspace_bytes < (size_t)T * n_experts * 2)
      return fail("route: workspace too small (need %zu bytes)", (size_t)T * n_experts * 2);
    logits = static_cast<uint16_t *>(workspace);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  // with room for them behind the logits, the byte planes of the integer route (same bits, see mi_moe_router_logits)
  const size_t lbytes = logits_out ? 0 : align_up((size_t)T * n_experts * 2);
  void *planes = workspace ? static_cast<char *>(workspace) + lbytes : nullptr;
  const bool roomy = workspace && router_logits_i8_applies(T, hidden, n_experts) &&
                     workspace_bytes >= lbytes + router_logits_i8_bytes(T, hidden, n_experts) + 256;
  if (roomy && router_tile_applies(T, hidden, n_experts, top_k)) {
    MI_HIP(launch_router_tile(x, router_w, router_bias, T, hidden, n_experts, top_k, score_mode, logits, topk_idx, topk_w,
                              planes, st));
    return 0;
  }
  if (roomy) MI_HIP(launch_router_logits_i8(x, router_w, router_bias, T, hidden, n_experts, logits, planes, st));
  else MI_HIP(launch_router_logits(x, router_w, router_bias, T, hidden, n_experts, logits, st));
  MI_HIP(launch_router_select(logits, T, n_experts, top_k, score_mode, topk_idx, topk_w, st));
  return 0;
} MI_CATCH("route")

int mi_moe_router_logits_workspace_size(int64_t T, int32_t hidden, int32_t n_experts, size_t *bytes) try {
  if (!bytes) return fail("router_logits_workspace_size: bytes is NULL");
  if (T < 0 || hidden <= 0 || n_experts < 1 || n_experts > 512) return fail("router_logits_workspace_size: bad arguments");
  *bytes = router_logits_i8_applies(T, hidden, n_experts) ? router_logits_i8_bytes(T, hidden, n_experts) + 256 : 256;
  return 0;
} MI_CATCH("router_logits_workspace_size")

int mi_moe_router_logits(const uint16_t *x, const uint16_t *router_w, const float *router_bias, int64_t T,
                         int32_t hidden, int32_t n_experts, uint16_t *logits, void *workspace,
                         size_t workspace_bytes, void *stream) try {
  if (T < 0) return fail("router_logits: negative token count");
  if (hidden <= 0 || hidden % 64) return fail("router_logits: hidden must be a positive multiple of 64, got %d", hidden);
  if (n_experts < 1 || n_experts > 512) return fail("router_logits: n_experts must be in [1, 512], got %d", n_experts);
  if (T == 0) return 0;
  if (!x || !router_w || !logits) return fail("router_logits: x, router_w and logits must be non-NULL");
  if (!aligned16(x) || !aligned16(router_w)) return fail("router_logits: x and router_w must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (router_logits_i8_applies(T, hidden, n_experts)) {
    const size_t need = router_logits_i8_bytes(T, hidden, n_experts) + 256;
    if (!workspace || workspace_bytes < need) return fail("router_logits: workspace too small (need %zu bytes)", need);
    MI_HIP(launch_router_logits_i8(x, router_w, router_bias, T, hidden, n_experts, logits, workspace, st));
  } else {
    MI_HIP(launch_router_logits(x, router_w, router_bias, T, hidden, n_experts, logits, st));
  }
  return 0;
} MI_CATCH("router_logits")

int mi_moe_dispatch_workspace_size(int32_t n_experts, int64_t P, size_t *bytes) try {
  if (!bytes) return fail("dispatch_workspace_size: bytes is NULL");
  if (n_experts < 1 || n_experts > 512 || P < 0) return fail("dispatch_workspace_size: bad arguments");
  // scratch + counts/offsets/active/n_active stand-ins for outputs the caller leaves NULL
  *bytes = align_up(dispatch_workspace_bytes(n_experts, P)) + 256;
  return 0;
} MI_CATCH("dispatch_workspace_size")

int mi_moe_dispatch(const uint32_t *expert_of_pair, int64_t P, int32_t n_experts, uint32_t *counts,
                    uint32_t *offsets, uint32_t *perm, uint32_t *inv_perm, void *workspace,
                    size_t workspace_bytes, void *stream) try {
  if (P < 0 || P > (int64_t)1 << 30) return fail("dispatch: pair count out of range");
  if (n_experts < 1 || n_experts > 512) return fail("dispatch: n_experts must be in [1, 512], got %d", n_experts);
  if (!perm) return fail("dispatch: perm must be non-NULL");
  if (P > 0 && !expert_of_pair) return fail("dispatch: expert_of_pair is NULL");
  size_t need = 0;
  mi_moe_dispatch_workspace_size(n_experts, P, &need);
  // (512 bytes were all that up to 4096 pairs needed before the two-launch form took those from 2049 on: one block does without)
  const size_t least = align_up(dispatch_workspace_least(n_experts, P)) + 256;
  if (!workspace || workspace_bytes < least) return fail("dispatch: workspace too small (need %zu bytes)", need);
  Carver cv(workspace);
  void *scratch = workspace_bytes < need ? nullptr : cv.take<char>(dispatch_workspace_bytes(n_experts, P));
  hipStream_t st = static_cast<hipStream_t>(stream);
  MI_HIP(launch_dispatch(expert_of_pair, P, n_experts, 1, counts, offsets, perm, inv_perm, nullptr, nullptr,
                         nullptr, 0, 0, ShortTiles{}, PrepareArgs{}, scratch, st));
  return 0;
} MI_CATCH("dispatch")

int mi_moe_gather_qmm_workspace_size(int32_t n_experts, int64_t n_idx, int32_t M, size_t *bytes) try {
  if (!bytes) return fail("gather_qmm_workspace_size: bytes is NULL");
  if (n_experts < 1 || n_experts > 512 || n_idx < 0 || M < 1) return fail("gather_qmm_workspace_size: bad arguments");
  const int64_t rows = n_idx * M;  // perm and the (src, dst) row maps hold one entry per output row
  *bytes = align_up(dispatch_workspace_bytes(n_experts, rows)) + 2 * align_up((size_t)(n_experts + 1) * 4) +
           align_up((size_t)n_experts * 64) + 3 * align_up((size_t)rows * 4) + 256;
  return 0;
} MI_CATCH("gather_qmm_workspace_size")

// which products the tuned kernels take; everything else goes to the plain ones
static bool tuned_shape(int32_t dtype, int32_t transpose, int32_t group_size, int32_t bits, int32_t N, int32_t K) {
  return dtype == MI_MOE_DTYPE_BF16 && transpose && group_size == 64 && (bits == 4 || bits == 8) && K % 64 == 0 &&
         (bits != 4 || K % 128 == 0) && N % 16 == 0;
}

static int check_qmm_shape(const char *who, int32_t dtype, int32_t transpose, int32_t group_size, int32_t bits,
                           int32_t N, int32_t K) {
  if (dtype != MI_MOE_DTYPE_BF16 && dtype != MI_MOE_DTYPE_F16 && dtype != MI_MOE_DTYPE_F32)
    return fail("%s: dtype must be MI_MOE_DTYPE_BF16, _F16 or _F32, got %d", who, dtype);
  if (bits != 2 && bits != 4 && bits != 8) return fail("%s: bits must be 2, 4 or 8, got %d", who, bits);
  if (group_size != 32 && group_size != 64 && group_size != 128)
    return fail("%s: group_size must be 32, 64 or 128, got %d", who, group_size);
  if (K <= 0 || N <= 0) return fail("%s: N and K must be positive, got %d, %d", who, N, K);
  // the quantised axis: K with transpose = true (w [N, K*bits/32]), N otherwise (w [K, N*bits/32])
  const int32_t q_axis = transpose ? K : N;
  if (q_axis % group_size)
    return fail("%s: %s (%d) must be a multiple of group_size (%d)", who, transpose ? "K" : "N", q_axis, group_size);
  return 0;
}

static int gather_qmm_impl(const void *x, const uint32_t *w, const void *scales, const void *biases,
                           const uint32_t *lhs_indices, const uint32_t *rhs_indices, int64_t n_idx, int64_t x_batch,
                           int32_t M, int32_t N, int32_t K, int32_t n_experts, int32_t transpose, int32_t group_size,
                           int32_t bits, int32_t dtype, void *y, void *workspace, size_t workspace_bytes,
                           void *stream) {
  if (check_qmm_shape("gather_qmm", dtype, transpose, group_size, bits, N, K)) return 1;
  if (M < 1) return fail("gather_qmm: M must be positive, got %d", M);
  if (n_experts < 1) return fail("gather_qmm: n_experts must be positive, got %d", n_experts);
  if (n_idx < 0 || n_idx * M > (int64_t)1 << 30) return fail("gather_qmm: index count out of range");
  if (n_idx == 0) return 0;
  if (!x || !w || !scales || !biases || !y) return fail("gather_qmm: x, w, scales, biases and y must be non-NULL");
  if (!rhs_indices) return fail("gather_qmm: rhs_indices is required");
  // x_batch = matrices in x (0 = not told).  Without lhs_indices index j reads x[j], so there must be n_idx of them;
  // with lhs_indices the kernels clamp an index beyond x_batch - 1 (and an expert index beyond n_experts - 1) instead
  // of following it: the rows it belongs to are then meaningless, but no memory outside the operands is read.
  if (x_batch < 0 || x_batch > (int64_t)UINT32_MAX) return fail("gather_qmm: x_batch out of range");
  if (!lhs_indices && x_batch > 0 && n_idx > x_batch)
    return fail("gather_qmm: %lld indices without lhs_indices need as many matrices in x, got %lld", (long long)n_idx,
                (long long)x_batch);
  const uint32_t n_lhs = (uint32_t)x_batch;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (!tuned_shape(dtype, transpose, group_size, bits, N, K) || n_experts > 512) {  // the plain kernels, no workspace
    MI_HIP(launch_qmm_plain(x, w, scales, biases, lhs_indices, rhs_indices, nullptr, nullptr, n_lhs, (uint32_t)n_experts,
                            n_idx * M, M, N, K, group_size, bits, transpose != 0, dtype, y, st));
    return 0;
  }
  if (!aligned16(x) || !aligned16(w) || !aligned16(scales) || !aligned16(biases) || !aligned16(y))
    return fail("gather_qmm: pointers must be 16-byte aligned");
  const int64_t rows = n_idx * M;
  size_t need = 0;
  mi_moe_gather_qmm_workspace_size(n_experts, n_idx, M, &need);
  const size_t full = dispatch_workspace_bytes(n_experts, rows), little = dispatch_workspace_least(n_experts, rows);
  const size_t least = need - align_up(full) + align_up(little);  // (as in mi_moe_dispatch)
  if (!workspace || workspace_bytes < least) return fail("gather_qmm: workspace too small (need %zu bytes)", need);
  Carver cv(workspace);
  void *scratch = cv.take<char>(workspace_bytes < need ? little : full);
  if (workspace_bytes < need) scratch = nullptr;
  uint32_t *counts = cv.take<uint32_t>(n_experts + 1);
  uint32_t *offsets = cv.take<uint32_t>(n_experts + 1);
  uint32_t *work = cv.take<uint32_t>((size_t)n_experts * 16);
  uint32_t *perm = cv.take<uint32_t>((size_t)rows);
  uint32_t *src_rows = cv.take<uint32_t>((size_t)rows);
  uint32_t *dst_rows = cv.take<uint32_t>((size_t)rows);
  MI_HIP(launch_dispatch(rhs_indices, n_idx, n_experts, 1, counts, offsets, perm, nullptr, nullptr, work,
                         nullptr, 0, 0, ShortTiles{}, PrepareArgs{}, scratch, st));
  MI_HIP(launch_row_maps(perm, lhs_indices, n_lhs, offsets, n_idx, M, n_experts, src_rows, dst_rows, work, st));
  GroupedArgs a{};
  a.x = static_cast<const uint16_t *>(x);
  a.src_rows = src_rows;
  a.dst_rows = dst_rows;
  a.work = work;
  a.max_active = (int)(n_idx < n_experts ? n_idx : n_experts);
  a.w0 = w; a.s0 = static_cast<const uint16_t *>(scales); a.b0 = static_cast<const uint16_t *>(biases);
  a.y = static_cast<uint16_t *>(y);
  a.N = N;
  a.K = K;
  a.bits = bits;
  a.total_rows = rows;
  a.max_rows_per_expert = rows;
  MI_HIP(launch_grouped_qmm(a, false, st));
  return 0;
}

int mi_moe_gather_qmm(const uint16_t *x, const uint32_t *w, const uint16_t *scales,
                      const uint16_t *biases, const uint32_t *lhs_indices, const uint32_t *rhs_indices,
                      int64_t n_idx, int64_t x_batch, int32_t M, int32_t N, int32_t K, int32_t n_experts,
                      int32_t transpose, int32_t group_size, int32_t bits, int32_t sorted_indices,
                      uint16_t *y, void *workspace, size_t workspace_bytes, void *stream) try {
  (void)sorted_indices;  // a hint in MLX; the segments are rebuilt here either way
  return gather_qmm_impl(x, w, scales, biases, lhs_indices, rhs_indices, n_idx, x_batch, M, N, K, n_experts, transpose,
                         group_size, bits, MI_MOE_DTYPE_BF16, y, workspace, workspace_bytes, stream);
} MI_CATCH("gather_qmm")

int mi_moe_gather_qmm_typed(const void *x, const uint32_t *w, const void *scales, const void *biases,
                            const uint32_t *lhs_indices, const uint32_t *rhs_indices, int64_t n_idx,
                            int64_t x_batch, int32_t M, int32_t N, int32_t K, int32_t n_experts,
                            int32_t transpose, int32_t group_size, int32_t bits, int32_t sorted_indices,
                            int32_t dtype, void *y, void *workspace, size_t workspace_bytes, void *stream) try {
  (void)sorted_indices;
  return gather_qmm_impl(x, w, scales, biases, lhs_indices, rhs_indices, n_idx, x_batch, M, N, K, n_experts, transpose,
                         group_size, bits, dtype, y, workspace, workspace_bytes, stream);
} MI_CATCH("gather_qmm_typed")

static size_t qmm_dense_bytes(int64_t M, int32_t K, int32_t bits, size_t *mt_words) {
  const size_t ntiles = (size_t)((M + kBigTileM - 1) / kBigTileM);
  *mt_words = tile_list_words((int)ntiles, 1);
  size_t b = 256 + 256 + 64 + *mt_words * 4 + 256;  // alignment of the base, the record, the tile lists
  if (bits == 4 && M >= tiled_avg_rows(bits)) b += (size_t)M * K * 2 + 256;
  return b;
}

static size_t codes_bytes(int64_t M, int32_t K, int32_t group_size, int32_t bits) {
  return 256 + align_up(codes_copy_bytes(bits, M, K)) + align_up(codes_sums_bytes(M, K, group_size));
}

int mi_moe_quantized_matmul_workspace_size(int64_t M, int32_t K, int32_t bits, size_t *bytes) try {
  if (!bytes) return fail("quantized_matmul_workspace_size: bytes is NULL");
  if (M < 0 || K <= 0 || M * (int64_t)K > (int64_t)1 << 40) return fail("quantized_matmul_workspace_size: bad sizes");
  size_t mt = 0;
  const size_t tuned = qmm_dense_bytes(M, K, bits, &mt), codes = codes_bytes(M, K, 32, bits);
  *bytes = tuned > codes ? tuned : codes;  // (the group size is not known here: the largest need)
  return 0;
} MI_CATCH("quantized_matmul_workspace_size")

// What the products on raw codes take: transposed weights, bf16 or f16 (see qmm_codes.hip for f32), any group.  Their descriptors
// hold a 32-bit size of one matrix, and both kernels read scales a word or more at a time: an even number of them, so that no
// word reaches behind the tensor (groups of 128 only: K / 128 and N both odd).
static bool codes_shape(int32_t dtype, int32_t transpose, int32_t group_size, int32_t bits, int32_t N, int32_t K) {
  return transpose && dtype != MI_MOE_DTYPE_F32 && bits != 2 && K % 128 == 0 && (int64_t)N * K * bits / 8 < (int64_t)1 << 31 && (int64_t)N * K < (int64_t)1 << 33 &&
         (int64_t)N * (K / group_size) % 2 == 0;
}

// Which transposed dense products take the kernel of a few rows (nothing to prepare, one launch).  Measured, us of the kernels
// (few rows / the one it stands against):
//   4096 x 4096, 16 rows of 4-bit codes 18.3 (f16), 20.7 (bf16, groups of 32) / tiles on raw codes 19.8, 26.8;
//   of 8-bit codes 26.7, 27.4 / 23.5, 24.8.  One row of 4-bit codes is still the plain kernel's: 7.5 / 6.7 (f16), unless the tuned bf16 shapes apply (no plain kernel there).
//   More rows of short 4-bit ones: 4096 x 2048 at 20 / 32 rows 14.0, 18.0 / tiles 17.9, 18.1; 4096 x 4096 23.9, 31.6 / 21.7, 21.9;
//   1024 x 1024 8.9, 11.0 / 15.5, 15.6.
//   bf16, groups of 64 / streaming kernel and its record's launch: 4-bit 4096 x 2048 at 1 / 8 / 16 rows 5.4, 7.9, 10.5 /
//   7.9, 9.5, 13.5, 4096 x 4096 7.0, 12.3, 17.6 / 10.4, 12.6, 20.2; 8-bit 2048 x 4096 at 1 / 2 / 4 / 8 / 16 rows 8.6, 9.3, 10.9,
//   14.1, 20.8 / 10.1, 10.2, 10.7, 13.6, 17.7, 4096 x 1024 4.7, 4.8, 5.4, 6.1, 7.5 / 7.4, 7.7, 8.1, 8.9, 10.6.
// (Before the codes were centred.  The kernel of a few rows now: 4096 x 4096, 16 rows of 4-bit codes 17.1, 17.3; 4096 x 2048 f16 at 20 / 32 rows
//   13.2, 17.3; 1024 x 1024 8.8, 11.0; bf16, groups of 64 4-bit 4096 x 2048 4.4, 7.1, 9.6, 4096 x 4096 5.8, 11.1, 16.3; 8-bit 4096 x 1024 4.1, 4.3,
//   4.7, 5.4, 6.8; tiles on raw codes 4096 x 4096 f16 at 20 / 32 rows 16.7, 16.9.)
static bool dense_takes_rows(bool tuned, int32_t bits, int64_t M, int32_t K) {
  if (tuned && bits == 8) return M <= kRowsMost && M * K <= (int64_t)1 << 14;
  if (M == 1 && !tuned && bits == 4) return false;
  if (M <= (bits == 4 ? kRowsMost : 12)) return true;
  return bits == 4 && M <= 2 * kRowsMost && M * K <= (int64_t)1 << 16;
}

// bf16, groups of 64: whether the 256 x 256 tiles with dequantised weights are faster than the 64 x 128 (or smaller) tiles
// on raw codes.  The larger tiles pay once their launch fills the chip.  Their time is close to 55 + 0.37 per tile (up to
// 256 tiles, K = 4096), that of the others to 15 + 0.113 per 64 x 128 tile; both go with K, so the line is the same for
// every K.  Measured, 256 x 256 / raw codes, us of the call, 4-bit: 4096 x 4096 at 64 / 128 / 512 / 1024 / 1280 / 2048 / 8192 rows
// 59.2, 61.5, 66.8, 79.1, 80.3, 104, 279 / 22.6, 24.2, 41.4, 66.4, 90.9, 124, 466; 14336 x 4096 at 256 / 512 / 2048 rows 80.4, 103,
// 248 / 65.2, 113, 406; 8-bit 2048 x 4096 at 64 / 1024 / 2048 / 4096 rows 56.9, 61.9, 72.6, 98.9 / 22.7, 39.8, 64.9, 129.
// (Before the codes were centred.  On raw codes, us of the kernels, now: 4096 x 4096 at 64 / 128 / 512 / 1024 rows 18.3, 20.0, 38.8, 64.7;
// 14336 x 4096 at 256 rows 58.2; 8-bit 2048 x 4096 at 64 / 1024 / 2048 rows 20.3, 40.3, 66.4.)
static bool dense_takes_large_tiles(int64_t M, int32_t N) {
  const int64_t large = (M + 255) / 256 * ((N + 255) / 256), small = (M + 63) / 64 * ((N + 127) / 128);
  return 10 * small > 33 * large + 3540;
}

// linear_bias: [N] added with a rounding of its own, or nullptr
static int quantized_matmul_impl(const void *x, const uint32_t *w, const void *scales, const void *biases,
                                 const void *linear_bias, int64_t M, int32_t N, int32_t K, int32_t transpose, int32_t group_size,
                                 int32_t bits, int32_t dtype, void *y, void *workspace, size_t workspace_bytes,
                                 void *stream) {
  if (check_qmm_shape("quantized_matmul", dtype, transpose, group_size, bits, N, K)) return 1;
  if (M < 0 || M > (int64_t)1 << 30) return fail("quantized_matmul: row count out of range");
  if (M == 0) return 0;
  if (!x || !w || !scales || !biases || !y) return fail("quantized_matmul: x, w, scales, biases and y must be non-NULL");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool tuned = tuned_shape(dtype, transpose, group_size, bits, N, K), codes = codes_shape(dtype, transpose, group_size, bits, N, K);
  size_t mt_words = 0;
  if (tuned) {
    if (!aligned16(x) || !aligned16(w) || !aligned16(scales) || !aligned16(biases) || !aligned16(y))
      return fail("quantized_matmul: pointers must be 16-byte aligned");
    const size_t need = qmm_dense_bytes(M, K, bits, &mt_words);
    if (!workspace || workspace_bytes < need) return fail("quantized_matmul: workspace too small (need %zu bytes)", need);
  }
  const bool one_plain = M == 1 && !tuned && bits == 4;
  if (codes && dense_takes_rows(tuned, bits, M, K) && aligned16(x) && aligned16(w) && aligned16(scales) && aligned16(biases)) {
    RowsArgs a{};
    a.x = x;
    a.w0 = w; a.s0 = scales; a.b0 = biases;
    a.bias = linear_bias;
    a.y = y;
    a.N = N;
    a.K = K;
    a.M = M;
    if (qmm_rows_applies(a, group_size, bits, dtype, false)) {
      MI_HIP(launch_qmm_rows(a, group_size, bits, dtype, false, st));
      return 0;
    }
  }
  const bool streamed = tuned && bits == 8 && M < tiled_avg_rows(bits);  // (see dense_takes_rows)
  const bool large_tiles = tuned && codes && !streamed && dense_takes_large_tiles(M, N);
  // (x and w are read and y is written 16 bytes at a time, scales and biases by words)
  if (codes && !one_plain && !streamed && !large_tiles && M * K * 4 < (int64_t)1 << 31 && workspace && workspace_bytes >= codes_bytes(M, K, group_size, bits) && aligned16(x) && aligned16(w) && aligned16(y) &&
      ((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 3u) == 0) {
    Carver cv(workspace);
    const size_t copy_bytes = codes_copy_bytes(bits, M, K);
    uint16_t *copy = copy_bytes ? reinterpret_cast<uint16_t *>(cv.take<char>(copy_bytes)) : nullptr;
    uint16_t *sums = reinterpret_cast<uint16_t *>(cv.take<char>(codes_sums_bytes(M, K, group_size)));
    MI_HIP(launch_prepare_rows(x, M, K, group_size, dtype, false, copy, sums, st));
    CodesArgs a{};
    a.x = copy ? copy : x;
    a.x_rows = M;
    a.sums = sums;
    a.w0 = w; a.s0 = scales; a.b0 = biases;
    a.bias = linear_bias;
    a.y = y;
    a.N = N;
    a.K = K;
    a.M = M;
    MI_HIP(launch_qmm_codes_dense(a, group_size, bits, dtype, st));
    return 0;
  }
  if (!transpose && aligned16(x) && aligned16(w) && aligned16(y)) {
    ColsArgs a{};
    a.x = x;
    a.w = w;
    a.s = scales; a.b = biases;
    a.y = y;
    a.N = N;
    a.K = K;
    a.M = M;
    if (qmm_cols_applies(a, bits, dtype)) {
      MI_HIP(launch_qmm_cols(a, group_size, bits, dtype, st));
      return 0;
    }
  }
  if (!tuned) {  // the plain kernels, no workspace
    MI_HIP(launch_qmm_plain(x, w, scales, biases, nullptr, nullptr, nullptr, nullptr, 0u, 1u, M, 1, N, K, group_size, bits,
                            transpose != 0, dtype, y, st));
    if (linear_bias) MI_HIP(launch_add_row_bias(y, linear_bias, M, N, dtype, st));
    return 0;
  }
  Carver cv(workspace);
  uint32_t *work = cv.take<uint32_t>(16);
  uint32_t *mtiles = cv.take<uint32_t>(mt_words);
  // one segment of M rows: the tiled kernel from the batch threshold on (fewer rows: streaming passes).  Where the 256-row
  // tiles fill the chip the rows behind the last whole tile are one more of them, in the same launch (in a class of their
  // own, one launch after the other: 1800 x 4096 x 4096 140 us; 2048 rows 104)
  const bool big = M >= tiled_avg_rows(bits) && (K / 64) % 2 == 0;
  const uint16_t *xb = static_cast<const uint16_t *>(x);
  uint16_t *xperm = (bits == 4 && big) ? cv.take<uint16_t>((size_t)M * K) : nullptr;
  const int cap256 = (int)((M + kBigTileM - 1) / kBigTileM);
  MI_HIP(launch_dense_records(M, big ? tiled_avg_rows(bits) : 0, large_tiles, work, mtiles, cap256, st));
  if (xperm) MI_HIP(launch_pair_rows(xb, M, K, xperm, st));
  GroupedArgs a{};
  a.x = xb;
  a.x_perm = bits == 4 ? xperm : xb;
  a.work = work;
  a.max_active = 1;
  a.mtiles = big ? mtiles : nullptr;
  a.max_mtiles = big ? cap256 : 0;
  a.tile_cap_e = big ? 1 : 0;
  a.w0 = w; a.s0 = static_cast<const uint16_t *>(scales); a.b0 = static_cast<const uint16_t *>(biases);
  a.y = static_cast<uint16_t *>(y);
  a.N = N;
  a.K = K;
  a.bits = bits;
  a.total_rows = M;
  a.max_rows_per_expert = M;
  if (large_tiles) MI_HIP(launch_large_qmm_class(a, false, 0, st));
  else MI_HIP(launch_grouped_qmm(a, false, st));
  if (linear_bias) MI_HIP(launch_add_row_bias(y, linear_bias, M, N, dtype, st));
  return 0;
}

int mi_moe_quantized_matmul(const uint16_t *x, const uint32_t *w, const uint16_t *scales,
                            const uint16_t *biases, int64_t M, int32_t N, int32_t K, int32_t transpose,
                            int32_t group_size, int32_t bits, uint16_t *y, void *workspace,
                            size_t workspace_bytes, void *stream) try {
  return quantized_matmul_impl(x, w, scales, biases, nullptr, M, N, K, transpose, group_size, bits, MI_MOE_DTYPE_BF16, y,
                               workspace, workspace_bytes, stream);
} MI_CATCH("quantized_matmul")

int mi_moe_quantized_matmul_typed(const void *x, const uint32_t *w, const void *scales, const void *biases,
                                  int64_t M, int32_t N, int32_t K, int32_t transpose, int32_t group_size,
                                  int32_t bits, int32_t dtype, void *y, void *workspace, size_t workspace_bytes,
                                  void *stream) try {
  return quantized_matmul_impl(x, w, scales, biases, nullptr, M, N, K, transpose, group_size, bits, dtype, y, workspace,
                               workspace_bytes, stream);
} MI_CATCH("quantized_matmul_typed")

int mi_moe_quantized_linear_typed(const void *x, const uint32_t *w, const void *scales, const void *biases,
                                  const void *linear_bias, int64_t M, int32_t N, int32_t K, int32_t group_size,
                                  int32_t bits, int32_t dtype, void *y, void *workspace, size_t workspace_bytes,
                                  void *stream) try {
  return quantized_matmul_impl(x, w, scales, biases, linear_bias, M, N, K, 1, group_size, bits, dtype, y, workspace,
                               workspace_bytes, stream);
} MI_CATCH("quantized_linear_typed")

int mi_moe_swiglu(const uint16_t *gate, const uint16_t *up, int64_t n, uint16_t *out, void *stream) try {
  if (n < 0) return fail("swiglu: negative element count");
  if (n == 0) return 0;
  if (!gate || !up || !out) return fail("swiglu: gate, up and out must be non-NULL");
  MI_HIP(launch_swiglu(gate, up, n, out, static_cast<hipStream_t>(stream)));
  return 0;
} MI_CATCH("swiglu")

int mi_moe_stream_probe(const void *buf, size_t bytes, uint32_t *sink, void *stream) try {
  if (bytes == 0) return 0;
  if (bytes % 32768) return fail("stream_probe: bytes must be a multiple of 32768, got %zu", bytes);
  if (bytes > ((size_t)1 << 34)) return fail("stream_probe: at most 16 GiB, got %zu", bytes);
  if (!buf || !sink) return fail("stream_probe: buf and sink must be non-NULL");
  if (reinterpret_cast<uintptr_t>(buf) % 16) return fail("stream_probe: buf must be 16-byte aligned");
  MI_HIP(launch_stream_probe(buf, bytes, sink, static_cast<hipStream_t>(stream)));
  return 0;
} MI_CATCH("stream_probe")

int mi_moe_combine(const uint16_t *y, const uint16_t *scores, const uint32_t *inv_perm, int64_t T,
                   int32_t top_k, int32_t hidden, uint16_t *out, void *stream) try {
  if (T < 0) return fail("combine: negative token count");
  if (top_k < 1) return fail("combine: top_k must be positive, got %d", top_k);
  if (hidden <= 0 || hidden % 8) return fail("combine: hidden must be a positive multiple of 8, got %d", hidden);
  if (T == 0) return 0;
  if (!y || !scores || !out) return fail("combine: y, scores and out must be non-NULL");
  if (!aligned16(y) || !aligned16(out)) return fail("combine: y and out must be 16-byte aligned");
  MI_HIP(launch_combine(y, scores, inv_perm, T, top_k, hidden, nullptr, out, static_cast<hipStream_t>(stream)));
  return 0;
} MI_CATCH("combine")

static int check_quant_args(const char *who, int64_t rows, int64_t cols, int32_t group_size, int32_t bits) {
  if (bits != 2 && bits != 4 && bits != 8) return fail("%s: bits must be 2, 4 or 8, got %d", who, bits);
  if (group_size != 32 && group_size != 64 && group_size != 128)
    return fail("%s: group_size must be 32, 64 or 128, got %d", who, group_size);
  if (rows < 0 || cols < 0) return fail("%s: negative shape", who);
  if (cols % group_size) return fail("%s: columns (%lld) must be divisible by group_size (%d)", who, (long long)cols, group_size);
  return 0;
}

static int check_dtype(const char *who, int32_t dtype) {
  if (dtype != MI_MOE_DTYPE_BF16 && dtype != MI_MOE_DTYPE_F16 && dtype != MI_MOE_DTYPE_F32)
    return fail("%s: dtype must be MI_MOE_DTYPE_BF16, _F16 or _F32, got %d", who, dtype);
  return 0;
}

int mi_moe_quantize_typed(const float *w, int64_t rows, int64_t cols, int32_t group_size, int32_t bits,
                          int32_t dtype, uint32_t *q, void *scales, void *biases, void *stream) try {
  if (check_quant_args("quantize", rows, cols, group_size, bits) || check_dtype("quantize", dtype)) return 1;
  if (rows * cols == 0) return 0;
  if (!w || !q || !scales || !biases) return fail("quantize: w, q, scales and biases must be non-NULL");
  MI_HIP(launch_quantize(w, rows, cols, group_size, bits, q, scales, biases, dtype, static_cast<hipStream_t>(stream)));
  return 0;
} MI_CATCH("quantize_typed")

int mi_moe_quantize(const float *w, int64_t rows, int64_t cols, int32_t group_size, int32_t bits,
                    uint32_t *q, uint16_t *scales, uint16_t *biases, void *stream) try {
  return mi_moe_quantize_typed(w, rows, cols, group_size, bits, MI_MOE_DTYPE_BF16, q, scales, biases, stream);
} MI_CATCH("quantize")

int mi_moe_dequantize_typed(const uint32_t *q, const void *scales, const void *biases, int64_t rows,
                            int64_t cols, int32_t group_size, int32_t bits, int32_t dtype, float *w_hat,
                            void *stream) try {
  if (check_quant_args("dequantize", rows, cols, group_size, bits) || check_dtype("dequantize", dtype)) return 1;
  if (rows * cols == 0) return 0;
  if (!q || !scales || !biases || !w_hat) return fail("dequantize: q, scales, biases and w_hat must be non-NULL");
  MI_HIP(launch_dequantize(q, scales, biases, rows, cols, group_size, bits, w_hat, dtype, false, static_cast<hipStream_t>(stream)));
  return 0;
} MI_CATCH("dequantize_typed")

int mi_moe_dequantize_native(const uint32_t *q, const void *scales, const void *biases, int64_t rows,
                             int64_t cols, int32_t group_size, int32_t bits, int32_t dtype, void *w_hat,
                             void *stream) try {
  if (check_quant_args("dequantize", rows, cols, group_size, bits) || check_dtype("dequantize", dtype)) return 1;
  if (rows * cols == 0) return 0;
  if (!q || !scales || !biases || !w_hat) return fail("dequantize: q, scales, biases and w_hat must be non-NULL");
  MI_HIP(launch_dequantize(q, scales, biases, rows, cols, group_size, bits, w_hat, dtype, true, static_cast<hipStream_t>(stream)));
  return 0;
} MI_CATCH("dequantize_native")

int mi_moe_dequantize(const uint32_t *q, const uint16_t *scales, const uint16_t *biases, int64_t rows,
                      int64_t cols, int32_t group_size, int32_t bits, float *w_hat, void *stream) try {
  return mi_moe_dequantize_typed(q, scales, biases, rows, cols, group_size, bits, MI_MOE_DTYPE_BF16, w_hat, stream);
} MI_CATCH("dequantize")

// ------------------------------------------------------------------ introspection (no counterpart in the reference)

int32_t mi_moe_debug_kernel_count(void) {
  int32_t n = 0;
  for (const KernelSlot *s = kernel_slots(); s; s = s->next) ++n;
  return n;
}

const char *mi_moe_debug_kernel_name(int32_t index) {
  int32_t i = 0;
  for (KernelSlot *s = kernel_slots(); s; s = s->next, ++i)
    if (i == index) return s->name;
  return nullptr;
}

int64_t mi_moe_debug_kernel_launches(int32_t index) {
  int32_t i = 0;
  for (KernelSlot *s = kernel_slots(); s; s = s->next, ++i)
    if (i == index) return (int64_t)__atomic_load_n(&s->launches, __ATOMIC_RELAXED);
  return -1;
}

namespace {
// nothing is launched while one of these lives on the calling thread: launch_kernel writes to `plan` instead
struct PlanScope {
  LaunchPlan plan;
  PlanScope(char *out, size_t cap) : plan{out, cap} {
    if (out && cap) out[0] = 0;
    g_launch_plan = &plan;
  }
  ~PlanScope() { g_launch_plan = nullptr; }
};
}  // namespace

int mi_moe_debug_plan_grouped(int32_t N, int32_t K, int32_t bits, int32_t glu, int64_t total_rows, int32_t max_active,
                              int64_t max_rows_per_expert, int64_t max_streamed_rows, int32_t tile_lists,
                              int32_t paired_out, char *out, size_t cap) try {
  if (bits != 4 && bits != 8) return fail("debug_plan_grouped: the tuned kernels take 4- or 8-bit codes, got %d", bits);
  if (N <= 0 || K <= 0 || K % 64 || (bits == 4 && K % 128) || N % 16)
    return fail("debug_plan_grouped: N must be a multiple of 16, K of 64 (4-bit: 128), got %d, %d", N, K);
  if (total_rows < 0 || max_active < 0 || max_rows_per_expert < 0 || max_streamed_rows < 0) return fail("debug_plan_grouped: negative count");
  static const uint32_t dummy[4] = {0, 0, 0, 0};  // never read: nothing is launched
  GroupedArgs a{};
  a.x = a.x_perm = reinterpret_cast<const uint16_t *>(dummy);
  a.work = dummy;
  a.w0 = a.w1 = dummy;
  a.N = N; a.K = K; a.bits = bits;
  a.total_rows = total_rows;
  a.max_active = max_active;
  a.max_rows_per_expert = max_rows_per_expert;
  a.max_streamed_rows = max_streamed_rows;
  a.y_paired = paired_out != 0;
  if (tile_lists) {
    a.mtiles = dummy;
    a.max_mtiles = (int)(total_rows / kBigTileM + max_active);
    a.tile_cap_e = max_active;
  }
  PlanScope scope(out, cap);
  MI_HIP(launch_grouped_qmm(a, glu != 0, nullptr));
  return 0;
} MI_CATCH("debug_plan_grouped")

int mi_moe_debug_plan_forward(const mi_moe_config *cfg, int64_t T, char *out, size_t cap) try {
  if (check_config(cfg)) return 1;
  if (T < 1 || T * cfg->top_k > (int64_t)1 << 30) return fail("debug_plan_forward: token count out of range");
  if (plain_config(*cfg)) {
    if (out && cap) out[0] = 0;
    return 0;  // products on raw codes or plain ones: none of the listed kernels
  }
  const ForwardWs f = carve_forward(*cfg, T, reinterpret_cast<void *>(uintptr_t{256}), true);
  if (f.mid) {
    if (out && cap) out[0] = 0;
    return 0;  // (neither are the short tiles)
  }
  mi_moe_weights w{};
  GroupedArgs a{}, d{};
  grouped_args(*cfg, w, f, reinterpret_cast<const uint16_t *>(uintptr_t{256}), T, a, d);
  PlanScope scope(out, cap);
  MI_HIP(launch_grouped_qmm(a, true, nullptr));
  MI_HIP(launch_grouped_qmm(d, false, nullptr));
  return 0;
} MI_CATCH("debug_plan_forward")

int mi_moe_debug_tile_rule(const mi_moe_config *cfg, int64_t T, int32_t *tiled, int32_t *tile_min_rows) try {
  if (check_config(cfg)) return 1;
  if (T < 0 || T * cfg->top_k > (int64_t)1 << 30) return fail("debug_tile_rule: token count out of range");
  const ForwardWs f = carve_forward(*cfg, T, nullptr, true);
  if (tiled) *tiled = f.mid ? 2 : f.pieces && cfg->bits == 4 ? 3 : f.tiled ? 1 : 0;
  if (tile_min_rows) *tile_min_rows = f.mid ? 1 : f.tmr;
  return 0;
} MI_CATCH("debug_tile_rule")

int32_t mi_moe_debug_side_streams_created(void) { return g_side_streams_created.load(); }

}  // extern "C"
