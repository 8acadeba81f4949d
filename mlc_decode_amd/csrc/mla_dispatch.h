// mla_dispatch.h -- which decodes the wide kernel takes, and what bounds a sequence's pages (host code,
// no HIP: the CPU tests compile these rules by themselves).
//
// The wide kernel (PV split by output dims) beats the one-ring kernel where a segment is long enough
// to repay its start and end: a second ring to fill, P^T through LDS, rows staged through LDS on the
// way out.  Both sides of each line are main + combine kernel, us, one-ring -> wide, 256 CUs.
#pragma once
#include <stdint.h>

namespace mla {

// The most pages a sequence of a contiguous cache can have: a batch stride's worth of tokens where the
// sequences lie one after another.  A batch stride of less than a page of tokens belongs to another
// order (token-major, or one sequence, whose batch stride is never used) and bounds nothing.
inline int64_t contiguous_pages_bound(int64_t stride_batch, int64_t stride_tok) {
  const int64_t page = 64 * stride_tok;
  return page > 0 && stride_batch >= page ? (stride_batch + page - 1) / page : INT64_MAX;
}

// 65 .. 127 rows leave row tiles of a workgroup empty; with one-page sequences on up to half of the
// CUs nothing makes up for it (top 64: 32 sequences x 72 heads 23.2 -> 24.3, 64 x 100 heads 25.4 ->
// 26.7; but 8 x 72 22.8 -> 20.8, 132 x 100 28.1 -> 27.7, and two pages: 64 x 72 28.4 -> 26.9).
inline bool wide_pads_one_page(int rows, int batch, int pages, int cus) {
  return rows < 128 && pages == 1 && batch >= 16 && 2 * batch <= cus;
}

// Several query tokens whose heads do not fill whole workgroups: the rows of a one-split sequence are
// not one run of the output, and each is placed by itself.  One-page sequences on up to a fifth of the
// CUs lose by it (fp8, 38 sequences x 32 tokens: 64 heads x 2 22.9 -> 24.6, 40 x 4 23.4 -> 24.2; 16 x 64
// tokens, 72 x 2 24.9 -> 25.6; but 8 sequences 26.1 -> 25.4, 64 27.0 -> 26.9, and two pages: 38 x 128
// tokens, 64 x 2 31.5 -> 28.0; one token: 16 x 160 heads 24.9 -> 23.1).
inline bool wide_breaks_one_page(int rows, int heads, int batch, int pages, int cus) {
  return rows > heads && heads % 128 != 0 && pages == 1 && batch >= 16 && 5 * batch <= cus;
}

// Sparse decode over a 16-bit pool, more than 32 rows.  Up to 64 rows: four pages per segment (every
// part or sequence has one at least), or 4/3 pages per segment where the schedule fills the chip (64
// sequences x 64 heads, top 512: 27.2 -> 25.2, top 256 22.1 -> 22.2; 132 x 40, top 256: 28.6 -> 26.0,
// top 128 19.9 -> 20.8), or lists of 32 pages there (8 x 64, top 2048: 23.9 -> 19.7; top 1536 21.6 ->
// 23.0), or so few pages that the chip is idle: up to 16 without padding rows (1 x 64, top 64 12.5 ->
// 11.8, 4 x 64, top 256 14.5 -> 14.0, 32 x 64, top 64 16.6 -> 17.8), with them only those of one sequence
// of four pages or more (1 x 48, top 512 13.7 -> 13.4; top 64 11.5 -> 12.1, 2 x 48, top 512 13.6 -> 13.8,
// 1 x 33 12.5 -> 12.7).
// The wide form also multiplies a page id by a 32-bit page stride, which the C ABI does not bound for an
// index list; the one-ring kernel does so in 64 bits.
inline bool wide_takes_sparse(int rows, int batch, int topk, int num_parts, int cus, int64_t kv_stride_page,
                              int64_t kv_rope_stride_page) {
  constexpr int64_t kLimit = int64_t(1) << 32;
  if (kv_stride_page >= kLimit || kv_rope_stride_page >= kLimit) return false;
  const int pages = (topk + 63) / 64;
  if (rows > 64) return !wide_pads_one_page(rows, batch, pages, cus);
  const int64_t total = (int64_t)batch * pages;
  if (total >= 4 * (int64_t)(num_parts > batch ? num_parts : batch)) return true;
  if (total <= 16 && (rows == 64 || (batch == 1 && pages >= 4 && rows >= 40))) return true;
  return num_parts >= cus && (3 * total >= 4 * ((int64_t)num_parts + batch) || (total >= num_parts && pages >= 32));
}

// Paged decode over the fp8 cache, more than 32 rows.  The lengths are on the device: the block
// table's width is what the host knows of them, an upper bound.  Up to 64 rows: four pages per segment
// where the parts do not fill the chip (one sequence x 40 heads of 8192 tokens in 8 splits 70.1 ->
// 61.0, of 512 in 2 26.2 -> 25.6, in 4 19.0 -> 19.9), two without padding rows (64 heads: of 512 in 4
// 20.6 -> 20.1, in 8 17.3 -> 17.4), else six, or 15/8 with sequences of eight pages
// (64 sequences x 64 heads x 1024 tokens: 32.3 -> 31.6, x 512 25.1 -> 25.4; 132 x 512 41.9 -> 38.6,
// x 256 29.0 -> 30.7; 16 x 1024 24.1 -> 27.0).  The wide form forms a lane's scale offset (three block
// strides) in 32 bits.
inline bool wide_takes_fp8(int rows, int heads, int batch, int table_width, int num_parts, int cus,
                           int64_t scale_stride_blk) {
  if (scale_stride_blk >= (int64_t(1) << 28)) return false;
  if (rows > 64)
    return !wide_pads_one_page(rows, batch, table_width, cus) && !wide_breaks_one_page(rows, heads, batch, table_width, cus);
  const int64_t total = (int64_t)batch * table_width;
  const int64_t segments = num_parts > batch ? num_parts : batch;
  if (total >= (num_parts >= cus ? 6 : rows == 64 ? 2 : 4) * segments) return true;
  return num_parts >= cus && table_width >= 8 && 8 * total >= 15 * ((int64_t)num_parts + batch);
}

}  // namespace mla
