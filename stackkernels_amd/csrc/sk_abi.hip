// extern "C" entry points of libsk_attn.so (declared in include/sk_attn.h).
//
// This layer validates arguments, fills the kernel parameter blocks, applies
// the gfx950 split table for decode, and launches on the caller's stream.  It
// never allocates device memory and never synchronises the host.
#include <stdarg.h>
#include <stdio.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "sk_attn.h"
#include "sk_kernels.h"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  snprintf(g_err, sizeof(g_err), "%s: %s", what, hipGetErrorString(e));
  return (int)e;
}

int elem_bytes(int dtype) { return dtype == SK_F32 ? 4 : 2; }

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// Common shape checks; messages follow the reference's
// validate_attention_layout (src/stackkernels/_opt/memory/layout.py:19-39).
int check_dims(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D) {
  if (dtype != SK_F32 && dtype != SK_F16 && dtype != SK_BF16)
    return fail(SK_EUNSUPPORTED, "unsupported dtype code %d", dtype);
  if (B < 0 || Hq < 0 || Hkv <= 0 || Sq < 0 || Sk < 0 || D <= 0)
    return fail(SK_EINVAL, "invalid sizes B=%d Hq=%d Hkv=%d Sq=%d Sk=%d D=%d", B, Hq, Hkv, Sq, Sk, D);
  if (Hq % Hkv != 0)
    return fail(SK_EINVAL, "Query heads (%d) must be divisible by KV heads (%d) for GQA/MQA", Hq, Hkv);
  if (sk::padded_head_dim(D) == 0)
    return fail(SK_EUNSUPPORTED, "head dim %d unsupported: need a multiple of 8 in [8, 256]", D);
  return SK_OK;
}

int check_strides(int dtype, const char* name, const int64_t* st) {
  if (!st) return fail(SK_EINVAL, "%s strides pointer is NULL", name);
  const int64_t unit = dtype == SK_F32 ? 4 : 8;  // 16 bytes in elements
  for (int i = 0; i < 3; ++i)
    if (st[i] < 0 || st[i] % unit != 0)
      return fail(SK_EINVAL, "%s stride[%d]=%lld must be a non-negative multiple of %lld elements",
                  name, i, (long long)st[i], (long long)unit);
  return SK_OK;
}

int check_ptr(const char* name, const void* p) {
  if (!p) return fail(SK_EINVAL, "%s pointer is NULL", name);
  if (!aligned16(p)) return fail(SK_EINVAL, "%s pointer is not 16-byte aligned", name);
  return SK_OK;
}

// gfx950 decode split table.  A split is one workgroup per (batch, KV head);
// the table sizes the split count to the workgroups the chip holds at once,
// counted as eight waves per CU (16 query heads per wave: 1, 2 or 4 waves per
// workgroup):
// * groups of up to 16 heads (one-wave workgroups): one round with a
//   uniform cache length (every split the same size; C4: 4 splits, 1.7%
//   faster than two rounds), about two rounds with per-row lengths and over
//   paged pools (per_row), whose rows spread their keys over their splits so
//   a row shorter than the longest leaves a one-round grid uneven (8
//   splits: 6.9% and 7.7% faster than 4 at the C4 shape with lengths U[1, Sk]).
//   A uniform round is not overfilled: counts round down (368 rows and heads,
//   S_k = 4,000 132.9 us at 6 splits, 120.7 at 5; 1,200, S_k = 1,000 114.5 at
//   2, 98.2 at 1); with per-row lengths the one round rounds up (720, S_k <=
//   1,500 59.3 us at 3 splits, 64.1 at 2);
// * head dims above 128, groups of up to 16: four workgroups fit on a CU, so
//   a uniform round is 1,024 (180, S_k = 5,357 209 us at 6 splits, 157 at 5;
//   above 1,024 units two splits, 219 -> 191 us at 1,200; one whole round
//   against two and three, 64 units, S_k = 16,384: 174, 191 and 205 us with
//   16-head groups, 168, 176 and 186 with 4; 16 units, S_k = 32,768: 94, 112
//   and 120), and per-row lengths
//   take two such rounds that fit (368, S_k <= 976 53.4 us at 2 splits, 42.1 at
//   5, 47.3 at 6; 800, S_k <= 1,500 121 at 2, 130 at 3), two splits above
//   1,024 units (1,120, S_k <= 1,572 179 us whole, 155 at 2, 163 at 4; 147
//   shapes up to 2,047 units 1% below three or four splits on average);
// * 32- and 64-head groups: exactly one round, so no split waits for a second
//   round; a 64-head group writes 32 KB of partials per split, so fewer,
//   longer splits also keep that traffic small (C5: 64 splits; 32 and 128
//   splits measured 15% and 10% slower).
// A split keeps at least 256 keys, 128 with 64 to 384 (batch, KV head) units
// of up to 16 heads (360 units, S_k <= 500, D = 128: 28.0 us whole, 20.9 at 3
// splits; 800 units, S_k <= 700: 45.0 at 2, 47.9 at 3).  Small calls (at most
// 1,024 query heads in all, whose partials cost the combine little) split
// further, because a split's tiles follow one another:
// * up to 32 heads a group, to 64 keys while that gives at most 512 workgroups
//   and to one 32-key tile while at most 256.  Microseconds of both kernels
//   (graph replays), H_q = 32, H_kv = 8, D = 128 bf16, 256 keys a split -> so: B
//   = 1, S_k = 1,000 19.2 -> 8.4 (32 splits), S_k = 4,096 16.2 -> 10.8 (64); B
//   = 16, S_k = 1,000 22.4 -> 19.3 (7).  Past those limits more splits lose: B =
//   1, S_k = 32,768 31 us at 128, 36 at 256; 64 x 64 heads, S_k = 500 16 us
//   whole, 23 at 6;
// * above 32, to 128 keys while at most 256 workgroups of the 64-key tiles up to
//   D = 128 (16 units, S_k = 3,356 19.6 us at 13 splits, 19.2 at 16, 21.2 at
//   21), and there from three splits on (2 units, S_k = 263 8.2 us whole, 10.1
//   at 2), or 512 above (15 units, S_k = 6,286 17% faster with 33 than with 22);
// * above 16, to at most 64 splits, whose partials are read by one workgroup
//   per head: 64 heads, 2 units, S_k = 27,491 19.7 us at 107 splits of 256
//   keys, 22.5 at 215 of 128; 32 heads, 1 unit, S_k = 34,585 22.8 and 28.4.
// Caches below 192 keys stay whole, below 256 at head dims up to 64 and, up to
// 128, in groups above 16 (16 units, S_k = 211, D = 64 7.6 us whole, 8.4 at 7).
// Up to D = 128 per-row lengths take their second round only where the longest
// row gives each split 512 keys, 352 up to 384 units (B = 32, U[1, 4,096], 256
// keys: 54.6 us with 16 splits, 53.1 with 8; 720 units, U[1, 1,500], 300 keys:
// 64.6 with 5, 59.3 with 3; 368 units, U[1, 4,000], 363 keys: 57.4 with 11,
// 64.6 with 6; 800 units, U[1, 3,000], 600 keys: 113.6 with 5, 118.8 with 3).
// Groups of one or two heads write few partials, and take it from 256 keys on
// and shorter rounds that fit 256 (14 x 32 heads, U[1, 4,467], D = 96 53.5 us
// with 5, 49.4 with 10; 9 x 12, U[1, 10,680] 54.8 with 19, 51.6 with 38; 16 x
// 8, U[1, 5,263] 38.8 with 15, 37.1 with 20).  Over 436 shapes of 90 to 1,300
// units (S_k 800 to 16,384) that is 3.2% below two rounds of 256 keys for all.
// The count is capped at 1024 (the combine kernel's LDS weight array).
int plan_splits(int B, int Hq, int Hkv, int Sk, int D, bool per_row) {
  if (B <= 0 || Hkv <= 0) return 1;
  const int group = Hq / Hkv;
  if (Sk < (D <= 64 || (D <= 128 && group > 16) ? 256 : 192)) return 1;
  const int waves = group <= 16 ? 1 : group <= 32 ? 2 : 4;
  const int64_t slots = 256LL * 8 / waves;
  const int64_t units = (int64_t)B * Hkv;
  int64_t splits = (slots + units - 1) / units;
  if (group <= 16 && per_row) {
    const int64_t two = 2 * slots / units;
    if (D > 128) {
      if (units <= slots / 2) splits = slots / units;
    } else if (group <= 2 && units <= slots / 2) {
      splits = std::max(splits, std::min<int64_t>((2 * slots + units - 1) / units, Sk / 256));
    } else if (Sk >= two * (units <= 384 ? 352 : 512)) {
      splits = std::max(splits, two);
    }
  } else if (group <= 16) {
    if (D <= 128) splits = slots / units;
    else if (units <= slots / 2) splits = slots / 2 / units;
  }
  int64_t most = Sk / (group <= 16 && units >= 64 && units <= 384 ? 128 : 256);
  if ((int64_t)B * Hq <= 1024 && (group <= 32 || D > 128 || Sk >= 384)) {
    const int fits = group > 32 && D <= 128 ? 256 : 512;
    int64_t fine = std::min<int64_t>(fits / units, Sk / (group > 32 ? 128 : 64));
    if (group <= 32) fine = std::max(fine, std::min<int64_t>(256 / units, (Sk + 31) / 32));
    most = std::max(most, group > 16 ? std::min<int64_t>(fine, 64) : fine);
  }
  splits = std::min(splits, most);
  return (int)std::max<int64_t>(1, std::min<int64_t>(splits, 1024));
}

int keys_per_split_for(int Sk, int splits) {
  int kps = (Sk + splits - 1) / splits;
  kps = (kps + 31) / 32 * 32;
  return std::max(kps, 32);
}

// Head-dim columns of a split's partials: the kernel's padded head dim (the
// fp32 kernel is compiled for 64, 128 and 256).
size_t decode_dpad(int dtype, int D) {
  const int dp = sk::padded_head_dim(D);
  return (size_t)(dtype == SK_F32 && dp == 96 ? 128 : dp);
}

size_t decode_ws_bytes(int dtype, int B, int Hq, int D, int splits) {
  // (One fp32 split: the LSE of the fp32 forward that serves groups above 64.)
  if (splits <= 1) return dtype == SK_F32 ? (size_t)B * Hq * sizeof(float) : 0;
  const size_t dpad = decode_dpad(dtype, D);
  return (size_t)B * Hq * splits * (dpad + 1) * sizeof(float);
}

// RoPE arguments of the *_rope entry points -> r.  `tokens` is the number of
// consecutive positions each batch row uses from its base (1 for decode, T
// for the cache append, Sq for the forward).  With one base for the whole
// batch (rope_pos NULL) the positions [rope_start, rope_start + tokens) must
// lie in the table, as the reference's table slice
// cos[start_pos : start_pos + seq_len] requires
// (src/stackkernels/_reference/torch/rope.py:49-50).
int make_rope(const void* cos, const void* sin, int rope_dtype, int rope_rows,
              int64_t rope_stride, const int32_t* rope_pos, int rope_start, int D, int tokens,
              sk::RopeParams* r) {
  if (!cos || !sin) return fail(SK_EINVAL, "rope cos/sin pointer is NULL");
  if (rope_dtype != SK_F32 && rope_dtype != SK_F16 && rope_dtype != SK_BF16)
    return fail(SK_EUNSUPPORTED, "unsupported rope table dtype code %d", rope_dtype);
  if (D % 16 != 0)
    return fail(SK_EUNSUPPORTED, "RoPE needs a head dim that is a multiple of 16, got %d", D);
  if (rope_rows <= 0 || rope_stride < D)
    return fail(SK_EINVAL, "rope table of %d rows with row stride %lld for head dim %d", rope_rows,
                (long long)rope_stride, D);
  if (!aligned16(cos) || !aligned16(sin) || (rope_stride * elem_bytes(rope_dtype)) % 16 != 0)
    return fail(SK_EINVAL, "rope tables must be 16-byte aligned with a row stride that is a "
                "multiple of 16 bytes");
  if (!rope_pos && tokens > 0 &&
      (rope_start < 0 || (int64_t)rope_start + tokens > (int64_t)rope_rows))
    return fail(SK_EINVAL, "positions [%d, %lld) lie outside the rope table of %d rows", rope_start,
                (long long)rope_start + tokens, rope_rows);
  r->cos = cos, r->sin = sin;
  r->stride = rope_stride;
  r->rows = rope_rows;
  r->dtype = rope_dtype;
  r->pos_b = rope_pos;
  r->start = rope_start;
  return SK_OK;
}

// Backward scratch: delta and lse * log2(e) (fp32 per query row, each array
// rounded up to 256 bytes), then, for the five-GEMM backward, the dS tiles of
// one chunk of (batch, KV head) pairs.
size_t bwd_rows_bytes(int B, int Hq, int Sq) {
  const size_t rows = (size_t)B * Hq * Sq;
  return 2 * ((rows * sizeof(float) + 255) / 256 * 256);
}

// Pairs per chunk of the five-GEMM backward when at most `budget` bytes of
// dS tiles fit (0: the seven-GEMM backward runs).  The chunks are as even as
// the budget allows: ceil(pairs / chunks) with the fewest chunks that fit.
int64_t bwd_chunk_pairs(int64_t pairs, size_t pair_bytes, size_t budget) {
  if (pairs <= 0 || pair_bytes == 0 || budget < pair_bytes) return 0;
  const int64_t fit = std::min<int64_t>(pairs, (int64_t)(budget / pair_bytes));
  const int64_t chunks = (pairs + fit - 1) / fit;
  return (pairs + chunks - 1) / chunks;
}

// Bytes sk_attn_bwd_workspace reports: the row statistics plus one chunk of
// dS tiles under SK_BWD_DS_CAP_BYTES.
size_t bwd_ws_bytes(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D, bool causal) {
  const size_t pair = sk::bwd_ds_pair_bytes(dtype, Hq, Hkv, Sq, Sk, D, causal);
  const int64_t chunk = bwd_chunk_pairs((int64_t)B * Hkv, pair, (size_t)SK_BWD_DS_CAP_BYTES);
  return bwd_rows_bytes(B, Hq, Sq) + (size_t)chunk * pair;
}

// Splits of the backward's kernels (kv_iters .. dq_chunks of p), and the
// offset and bytes of their partial sums in the workspace (0: the shape runs
// unsplit, or its pairs in several chunks).
struct BwdParts {
  size_t offset = 0, bytes = 0;
  sk::BwdParams p{};
};
BwdParts bwd_parts(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D, bool causal) {
  BwdParts r;
  if (dtype == SK_F32)
    sk::bwd_f32_split(B, Hq, Hkv, Sq, Sk, D, causal, &r.p);
  else
    sk::bwd_dkv_split(dtype, B, Hq, Hkv, Sq, Sk, D, causal, &r.p.kv_iters, &r.p.kv_chunks);
  const size_t pair = sk::bwd_ds_pair_bytes(dtype, Hq, Hkv, Sq, Sk, D, causal);
  const int64_t pairs = (int64_t)B * Hkv;
  if ((r.p.kv_iters <= 0 && r.p.dq_iters <= 0) ||
      (pair > 0 && bwd_chunk_pairs(pairs, pair, (size_t)SK_BWD_DS_CAP_BYTES) != pairs))
    return BwdParts{};
  r.offset = (bwd_ws_bytes(dtype, B, Hq, Hkv, Sq, Sk, D, causal) + 255) / 256 * 256;
  if (r.p.kv_iters > 0) r.bytes += (size_t)2 * r.p.kv_chunks * pairs * Sk * D * sizeof(float);
  if (r.p.dq_iters > 0) r.bytes += (size_t)r.p.dq_chunks * B * Hq * Sq * D * sizeof(float);
  return r;
}

}  // namespace

extern "C" {

int sk_abi_version(void) { return SK_ABI_VERSION; }

const char* sk_last_error(void) { return g_err; }

}  // extern "C"

// Sizes and work split of the forward: query blocks per (b, h) and, under
// the causal mask, whether blocks j and n_mblocks-1-j are paired in one
// workgroup (when that still leaves enough workgroups: fwd_pair_min).
static int fwd_shape(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D, int is_causal,
                     sk::FwdParams* p) {
  p->B = B, p->Hq = Hq, p->Hkv = Hkv, p->Sq = Sq, p->Sk = Sk, p->D = D, p->group = Hq / Hkv;
  const int rows = dtype == SK_F32 ? sk::fwd_f32_rows_per_block(D, Sq)
                                   : sk::fwd_rows_per_block(dtype, D, (int64_t)B * Hq, Sq, Sk, is_causal != 0);
  p->n_mblocks = (Sq + rows - 1) / rows;
  if ((int64_t)p->n_mblocks * B * Hq > 0x7fffffffLL)
    return fail(SK_EINVAL, "grid too large: %lld workgroups", (long long)p->n_mblocks * B * Hq);
  p->pair_items = dtype != SK_F32 && is_causal && p->n_mblocks >= 2 &&
                  (int64_t)((p->n_mblocks + 1) / 2) * B * Hq >=
                      sk::fwd_pair_min(dtype, D, (int64_t)B * Hq, Sq, Sk, is_causal != 0);
  p->n_items = p->pair_items ? (p->n_mblocks + 1) / 2 : p->n_mblocks;
  p->n_splits = 1;
  return SK_OK;
}

// |sm_scale| as the kernels multiply by it.  A zero scale (every visible key
// weighs the same) runs as 1e-30, which vanishes next to 1 for any ordinary
// score but keeps a masked score, or a running maximum before its first key,
// at -inf, where 0 * -inf would be NaN.
static float softmax_scale(float sm_scale) { return std::max(std::fabs(sm_scale), 1e-30f); }

// Bytes of the split forward's partials (per split and query row, D fp32
// values and an LSE), 0 where it runs without.
static size_t fwd_ws_bytes(int B, int Hq, int Sq, int D, const sk::FwdSplit& f) {
  return f.on() ? (size_t)f.splits * B * Hq * Sq * (D + 1) * sizeof(float) : 0;
}

// Makes p the split forward f: one query block per workgroup and split
// (pairing evens out the causal triangle on full grids only), partials at part.
static void fwd_apply_split(int dtype, const sk::FwdSplit& f, void* part, sk::FwdParams* p) {
  p->pair_items = 0;
  p->pack_heads = f.pack;
  if (dtype != SK_F32) p->n_mblocks = sk::fwd_split_blocks((int64_t)f.pack * p->Sq);
  p->n_items = p->n_mblocks;
  p->n_splits = f.splits;
  p->split_keys = sk::fwd_split_keys(p->Sk, f.splits);
  p->part_o = (float*)part;
  p->part_lse = p->part_o + (size_t)f.splits * p->B * p->Hq * p->Sq * p->D;
}

// Split count and keys per split of a decode call (num_splits 0: the gfx950
// table's pick; for fp32 one split, and always one for fp32 groups above 64).
static int decode_splits(int dtype, int B, int Hq, int Hkv, int Sk, int D, bool per_row, int num_splits,
                         int* splits, int* kps) {
  if (dtype == SK_F32 && (num_splits == 0 || Hq / Hkv > 64)) num_splits = 1;
  if (num_splits == 0) num_splits = plan_splits(B, Hq, Hkv, Sk, D, per_row);
  if (num_splits < 1 || num_splits > 1024)
    return fail(SK_EINVAL, "num_splits=%d outside [1, 1024]", num_splits);
  *kps = keys_per_split_for(Sk, num_splits);
  if (Sk > 0) num_splits = std::min(num_splits, (Sk + *kps - 1) / *kps);
  *splits = num_splits;
  return SK_OK;
}

// sk_attn_fwd, sk_attn_fwd_rope (no workspace: one split) and sk_attn_fwd_ws.
static int fwd_impl(int dtype, const void* q, const void* k, const void* v, void* o, float* lse,
                    void* workspace, size_t workspace_bytes, int num_splits,
                    int B, int Hq, int Hkv, int Sq, int Sk, int D, const int64_t* q_strides,
                    const int64_t* k_strides, const int64_t* v_strides,
                    const int64_t* o_strides, int is_causal, const sk::RopeParams& rope,
                    float sm_scale, void* stream) {
  int rc = check_dims(dtype, B, Hq, Hkv, Sq, Sk, D);
  if (rc) return rc;
  if ((rc = check_strides(dtype, "q", q_strides)) || (rc = check_strides(dtype, "k", k_strides)) ||
      (rc = check_strides(dtype, "v", v_strides)) || (rc = check_strides(dtype, "o", o_strides)))
    return rc;
  if ((int64_t)B * Hq * Sq == 0) return SK_OK;
  if ((rc = check_ptr("q", q)) || (rc = check_ptr("o", o)) || (rc = check_ptr("lse", lse)))
    return rc;
  if (Sk > 0 && ((rc = check_ptr("k", k)) || (rc = check_ptr("v", v)))) return rc;
  if (workspace_bytes > 0 && (rc = check_ptr("workspace", workspace))) return rc;

  sk::FwdParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = o;
  p.lse = lse;
  p.q_sb = q_strides[0], p.q_sh = q_strides[1], p.q_ss = q_strides[2];
  p.k_sb = k_strides[0], p.k_sh = k_strides[1], p.k_ss = k_strides[2];
  p.v_sb = v_strides[0], p.v_sh = v_strides[1], p.v_ss = v_strides[2];
  p.o_sb = o_strides[0], p.o_sh = o_strides[1], p.o_ss = o_strides[2];
  p.scale = softmax_scale(sm_scale);
  p.scale_log2 = p.scale * 1.4426950408889634f;
  const bool neg = sm_scale < 0.f;
  if ((rc = fwd_shape(dtype, B, Hq, Hkv, Sq, Sk, D, is_causal, &p))) return rc;
  p.rope = rope;
  sk::FwdSplit f;
  if (num_splits == 0) {
    f = sk::fwd_key_splits(dtype, D, B, Hq, Hkv, Sq, Sk, is_causal != 0);
    // (Packed heads' rows are addressed from the first one's in 31 bits.)
    if (((int64_t)(f.pack - 1) * q_strides[1] + (int64_t)Sq * q_strides[2] + D) * 2 >= 0x7fffffffLL)
      f.pack = 1;
    if (fwd_ws_bytes(B, Hq, Sq, D, f) > workspace_bytes) f = sk::FwdSplit{};
  } else if (num_splits > 1 && (dtype != SK_F32 || sk::fwd_f32_rows_per_block(D, Sq) == 256)) {
    const int keys = sk::fwd_split_keys(Sk, num_splits);  // (else the fp32 vector kernel: unsplit)
    f.splits = keys > 0 ? (Sk + keys - 1) / keys : 1;
    const size_t need = fwd_ws_bytes(B, Hq, Sq, D, f);
    if (need > workspace_bytes)
      return fail(SK_EWORKSPACE, "workspace of %zu bytes given, %zu needed", workspace_bytes, need);
  }
  p.pack_heads = 1;
  if (f.on()) {
    fwd_apply_split(dtype, f, workspace, &p);
    if ((int64_t)p.n_items * B * Hq * f.splits > 0x7fffffffLL)
      return fail(SK_EINVAL, "grid too large");
  }
  hipStream_t s = (hipStream_t)stream;
  hipError_t e;
  if (dtype == SK_F32) {
    p.q_sign = neg ? 1u : 0u;
    e = sk::launch_fwd_f32(p, is_causal != 0, s);
  } else {
    p.q_sign = neg ? 0x80008000u : 0u;
    e = sk::launch_fwd_mfma(dtype, p, is_causal != 0, s);
  }
  if (e == hipSuccess && p.part_o) e = sk::launch_fwd_combine(dtype, p, s);
  if (e != hipSuccess) return hip_fail(e, "sk_attn_fwd launch");
  return SK_OK;
}

extern "C" {

int sk_attn_fwd(int dtype, const void* q, const void* k, const void* v, void* o, float* lse,
                int B, int Hq, int Hkv, int Sq, int Sk, int D, const int64_t* q_strides,
                const int64_t* k_strides, const int64_t* v_strides, const int64_t* o_strides,
                int is_causal, float sm_scale, void* stream) {
  g_err[0] = 0;
  return fwd_impl(dtype, q, k, v, o, lse, nullptr, 0, 1, B, Hq, Hkv, Sq, Sk, D, q_strides,
                  k_strides, v_strides, o_strides, is_causal, sk::RopeParams{}, sm_scale, stream);
}

int sk_attn_fwd_workspace(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D, int is_causal,
                          size_t* bytes) {
  g_err[0] = 0;
  int rc = check_dims(dtype, B, Hq, Hkv, Sq, Sk, D);
  if (rc) return rc;
  if (!bytes) return fail(SK_EINVAL, "bytes pointer is NULL");
  *bytes = fwd_ws_bytes(B, Hq, Sq, D,
                        sk::fwd_key_splits(dtype, D, B, Hq, Hkv, Sq, Sk, is_causal != 0));
  return SK_OK;
}

int sk_attn_fwd_ws(int dtype, const void* q, const void* k, const void* v, void* o, float* lse,
                   void* workspace, size_t workspace_bytes, int num_splits, int B, int Hq,
                   int Hkv, int Sq, int Sk, int D, const int64_t* q_strides,
                   const int64_t* k_strides, const int64_t* v_strides, const int64_t* o_strides,
                   int is_causal, const void* rope_cos, const void* rope_sin, int rope_dtype,
                   int rope_rows, int64_t rope_stride, const int32_t* rope_pos, int rope_start,
                   float sm_scale, void* stream) {
  g_err[0] = 0;
  if (num_splits < 0 || num_splits > 1024)
    return fail(SK_EINVAL, "num_splits=%d outside [0, 1024]", num_splits);
  sk::RopeParams r{};
  if (rope_cos || rope_sin) {
    const int rc = make_rope(rope_cos, rope_sin, rope_dtype, rope_rows, rope_stride, rope_pos,
                             rope_start, D, (int64_t)B * Hq > 0 ? Sq : 0, &r);
    if (rc) return rc;
  }
  return fwd_impl(dtype, q, k, v, o, lse, workspace, workspace_bytes, num_splits, B, Hq, Hkv, Sq,
                  Sk, D, q_strides, k_strides, v_strides, o_strides, is_causal, r, sm_scale,
                  stream);
}

int sk_attn_fwd_rope(int dtype, const void* q, const void* k, const void* v, void* o, float* lse,
                     int B, int Hq, int Hkv, int Sq, int Sk, int D, const int64_t* q_strides,
                     const int64_t* k_strides, const int64_t* v_strides,
                     const int64_t* o_strides, int is_causal, const void* rope_cos,
                     const void* rope_sin, int rope_dtype, int rope_rows, int64_t rope_stride,
                     const int32_t* rope_pos, int rope_start, float sm_scale, void* stream) {
  g_err[0] = 0;
  sk::RopeParams r{};
  const int rc = make_rope(rope_cos, rope_sin, rope_dtype, rope_rows, rope_stride, rope_pos,
                           rope_start, D, (int64_t)B * Hq > 0 ? Sq : 0, &r);
  if (rc) return rc;
  return fwd_impl(dtype, q, k, v, o, lse, nullptr, 0, 1, B, Hq, Hkv, Sq, Sk, D, q_strides,
                  k_strides, v_strides, o_strides, is_causal, r, sm_scale, stream);
}

int sk_attn_bwd_workspace(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D, int is_causal,
                          size_t* bytes) {
  g_err[0] = 0;
  int rc = check_dims(dtype, B, Hq, Hkv, Sq, Sk, D);
  if (rc) return rc;
  if (!bytes) return fail(SK_EINVAL, "bytes pointer is NULL");
  *bytes = bwd_ws_bytes(dtype, B, Hq, Hkv, Sq, Sk, D, is_causal != 0);
  return SK_OK;
}

int sk_attn_bwd_workspace_best(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D,
                               int is_causal, size_t* bytes) {
  const int rc = sk_attn_bwd_workspace(dtype, B, Hq, Hkv, Sq, Sk, D, is_causal, bytes);
  if (rc) return rc;
  const BwdParts parts = bwd_parts(dtype, B, Hq, Hkv, Sq, Sk, D, is_causal != 0);
  if (parts.bytes > 0) *bytes = parts.offset + parts.bytes;
  return SK_OK;
}

int sk_attn_bwd_workspace_min(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D,
                              int is_causal, size_t* bytes) {
  g_err[0] = 0;
  (void)is_causal;
  int rc = check_dims(dtype, B, Hq, Hkv, Sq, Sk, D);
  if (rc) return rc;
  if (!bytes) return fail(SK_EINVAL, "bytes pointer is NULL");
  *bytes = bwd_rows_bytes(B, Hq, Sq);
  return SK_OK;
}

int sk_attn_bwd(int dtype, const void* dout, const void* q, const void* k, const void* v,
                const void* o, const float* lse, void* dq, void* dk, void* dv, void* workspace,
                size_t workspace_bytes, int B, int Hq, int Hkv, int Sq, int Sk, int D,
                int is_causal, float sm_scale, void* stream) {
  g_err[0] = 0;
  int rc = check_dims(dtype, B, Hq, Hkv, Sq, Sk, D);
  if (rc) return rc;
  if ((int64_t)B * Hq * Sq == 0 && (int64_t)B * Hkv * Sk == 0) return SK_OK;
  const size_t need = bwd_rows_bytes(B, Hq, Sq);
  if (need > 0 && (!workspace || workspace_bytes < need))
    return fail(SK_EWORKSPACE, "workspace of %zu bytes given, at least %zu needed",
                workspace_bytes, need);
  if ((int64_t)B * Hq * Sq > 0 &&
      ((rc = check_ptr("dout", dout)) || (rc = check_ptr("q", q)) || (rc = check_ptr("o", o)) ||
       (rc = check_ptr("lse", lse)) || (rc = check_ptr("dq", dq))))
    return rc;
  if ((int64_t)B * Hkv * Sk > 0 && ((rc = check_ptr("k", k)) || (rc = check_ptr("v", v)) ||
                                    (rc = check_ptr("dk", dk)) || (rc = check_ptr("dv", dv))))
    return rc;
  if (need > 0 && (rc = check_ptr("workspace", workspace))) return rc;

  sk::BwdParams p{};
  p.dout = dout, p.q = q, p.k = k, p.v = v, p.o = o, p.lse = lse;
  p.dq = dq, p.dk = dk, p.dv = dv;
  const size_t rows = (size_t)B * Hq * Sq;
  const size_t rows_bytes = (rows * sizeof(float) + 255) / 256 * 256;
  p.delta = (float*)workspace;
  p.lse_log2 = (float*)((char*)workspace + rows_bytes);
  p.dq_acc = nullptr;
  // The five-GEMM backward where its dS tiles for at least one (batch, KV
  // head) pair fit the workspace past the row statistics (at most
  // SK_BWD_DS_CAP_BYTES of it used); else the seven-GEMM backward.
  const size_t pair_bytes = sk::bwd_ds_pair_bytes(dtype, Hq, Hkv, Sq, Sk, D, is_causal != 0);
  const size_t ds_budget =
      std::min<size_t>(workspace_bytes - std::min(workspace_bytes, need), (size_t)SK_BWD_DS_CAP_BYTES);
  const int64_t chunk = bwd_chunk_pairs((int64_t)B * Hkv, pair_bytes, ds_budget);
  p.ds = chunk > 0 ? (char*)workspace + need : nullptr;
  p.n_pairs = (int)chunk;
  p.bk0 = 0;
  // Split kernels where the workspace holds their partial sums as well.
  const BwdParts parts = bwd_parts(dtype, B, Hq, Hkv, Sq, Sk, D, is_causal != 0);
  if (parts.bytes > 0 && workspace_bytes >= parts.offset + parts.bytes) {
    p.kv_iters = parts.p.kv_iters, p.kv_chunks = parts.p.kv_chunks;
    p.dq_iters = parts.p.dq_iters, p.dq_chunks = parts.p.dq_chunks;
    float* part = (float*)((char*)workspace + parts.offset);
    if (p.kv_iters > 0) {
      const size_t n = (size_t)p.kv_chunks * B * Hkv * Sk * D;
      p.part_dk = part, p.part_dv = part + n;
      part += 2 * n;
    }
    p.part_dq = part;
  }
  p.ds_nqt = (Sq + 31) / 32;
  p.ds_c = sk::ds_causal_c(Sq, Sk);
  p.ds_head_tiles = sk::ds_head_tiles((Sk + 127) / 128, p.ds_nqt, p.ds_c, is_causal != 0);
  p.B = B, p.Hq = Hq, p.Hkv = Hkv, p.Sq = Sq, p.Sk = Sk, p.D = D, p.group = Hq / Hkv;
  p.scale = sm_scale;
  p.scale_log2 = sm_scale * 1.4426950408889634f;
  p.abs_scale_log2 = softmax_scale(sm_scale) * 1.4426950408889634f;
  p.op_sign = sm_scale < 0.f ? 0x80008000u : 0u;
  hipStream_t s = (hipStream_t)stream;
  hipError_t e = hipSuccess;
  if (rows > 0) e = sk::launch_bwd_prep(dtype, p, s);
  if (e != hipSuccess) return hip_fail(e, "sk_attn_bwd preprocess launch");
  if (dtype == SK_F32)
    e = sk::launch_bwd_f32(p, is_causal != 0, s);
  else
    e = sk::launch_bwd_mfma(dtype, p, is_causal != 0, s);
  if (e != hipSuccess) return hip_fail(e, "sk_attn_bwd launch");
  return SK_OK;
}

static int decode_plan_impl(int dtype, int B, int Hq, int Hkv, int Sk, int D, bool per_row,
                            int* num_splits, size_t* workspace_bytes) {
  int rc = check_dims(dtype, B, Hq, Hkv, 1, Sk, D);
  if (rc) return rc;
  if (!num_splits || !workspace_bytes) return fail(SK_EINVAL, "output pointer is NULL");
  int splits = dtype == SK_F32 && Hq / Hkv > 64 ? 1 : plan_splits(B, Hq, Hkv, Sk, D, per_row);
  if (splits > 1) splits = (Sk + keys_per_split_for(Sk, splits) - 1) / keys_per_split_for(Sk, splits);
  *num_splits = splits;
  *workspace_bytes = decode_ws_bytes(dtype, B, Hq, D, splits);
  return SK_OK;
}

int sk_decode_plan(int dtype, int B, int Hq, int Hkv, int Sk, int D, int* num_splits,
                   size_t* workspace_bytes) {
  g_err[0] = 0;
  return decode_plan_impl(dtype, B, Hq, Hkv, Sk, D, false, num_splits, workspace_bytes);
}

int sk_decode_plan_varlen(int dtype, int B, int Hq, int Hkv, int Sk, int D, int* num_splits,
                          size_t* workspace_bytes) {
  g_err[0] = 0;
  return decode_plan_impl(dtype, B, Hq, Hkv, Sk, D, true, num_splits, workspace_bytes);
}

int sk_decode_workspace(int dtype, int B, int Hq, int Hkv, int Sk, int D, int num_splits,
                        size_t* workspace_bytes) {
  g_err[0] = 0;
  int rc = check_dims(dtype, B, Hq, Hkv, 1, Sk, D);
  if (rc) return rc;
  if (!workspace_bytes) return fail(SK_EINVAL, "output pointer is NULL");
  if (num_splits < 1 || num_splits > 1024)
    return fail(SK_EINVAL, "num_splits=%d outside [1, 1024]", num_splits);
  *workspace_bytes = decode_ws_bytes(dtype, B, Hq, D, num_splits);
  return SK_OK;
}

}  // extern "C"

// Paged cache of the decode entry points (block_table null: contiguous).
struct PagedCache {
  const int32_t* block_table = nullptr;
  int page_size = 0, max_pages = 0, num_pages = 0;
};

// Paged-pool arguments of sk_decode_paged / sk_decode_paged_rope -> pc.
static int paged_args(int B, int num_pages, int page_size, int max_pages,
                      const int32_t* block_table, const int32_t* cache_seqlens, PagedCache* pc) {
  if (page_size <= 0 || page_size % 32 != 0)
    return fail(SK_EINVAL, "page_size=%d must be a positive multiple of 32", page_size);
  if (num_pages < 0 || max_pages < 0)
    return fail(SK_EINVAL, "invalid num_pages=%d max_pages=%d", num_pages, max_pages);
  if ((int64_t)max_pages * page_size > 0x7fffffffLL)
    return fail(SK_EINVAL, "max_pages * page_size overflows int");
  if (B > 0 && max_pages > 0 && (!block_table || !cache_seqlens))
    return fail(SK_EINVAL, "block_table and cache_seqlens are required");
  if (max_pages > 0 && num_pages == 0) return fail(SK_EINVAL, "empty page pool");
  pc->block_table = block_table;
  pc->page_size = page_size, pc->max_pages = max_pages, pc->num_pages = num_pages;
  return SK_OK;
}

// sk_decode, sk_decode_varlen and sk_decode_paged: seqlens is null (every row
// sees all Sk keys) or a device array of B per-row key counts; pc describes a
// paged cache (then Sk = max_pages * page_size).
static int decode_impl(int dtype, const void* q, const void* k, const void* v, void* o,
                       void* workspace, size_t workspace_bytes, int num_splits, int B, int Hq,
                       int Hkv, int Sk, int D, const int64_t* q_strides, const int64_t* k_strides,
                       const int64_t* v_strides, const int64_t* o_strides,
                       const int32_t* seqlens, const PagedCache& pc,
                       const sk::RopeParams& rope, float sm_scale, void* stream) {
  int rc = check_dims(dtype, B, Hq, Hkv, 1, Sk, D);
  if (rc) return rc;
  if ((rc = check_strides(dtype, "q", q_strides)) || (rc = check_strides(dtype, "k", k_strides)) ||
      (rc = check_strides(dtype, "v", v_strides)) || (rc = check_strides(dtype, "o", o_strides)))
    return rc;
  if ((int64_t)B * Hq == 0) return SK_OK;
  if ((rc = check_ptr("q", q)) || (rc = check_ptr("o", o))) return rc;
  if (Sk > 0 && ((rc = check_ptr("k", k)) || (rc = check_ptr("v", v)))) return rc;
  if (Hq / Hkv > 64 && dtype != SK_F32)
    return fail(SK_EUNSUPPORTED, "decode supports up to 64 query heads per KV head, got %d", Hq / Hkv);

  int kps = 0;
  if ((rc = decode_splits(dtype, B, Hq, Hkv, Sk, D, seqlens != nullptr, num_splits, &num_splits,
                          &kps)))
    return rc;
  size_t need = decode_ws_bytes(dtype, B, Hq, D, num_splits);
  if (dtype == SK_F32 && num_splits > 1 && workspace_bytes < need) {
    // (fp32 ran unsplit whatever the count: a caller's scratch of that size still serves.)
    num_splits = 1;
    kps = keys_per_split_for(Sk, 1);
    need = decode_ws_bytes(dtype, B, Hq, D, 1);
  }
  if (need > 0 && (!workspace || workspace_bytes < need))
    return fail(SK_EWORKSPACE, "workspace of %zu bytes given, %zu needed", workspace_bytes, need);
  if (need > 0 && (rc = check_ptr("workspace", workspace))) return rc;
  hipStream_t s = (hipStream_t)stream;

  if (dtype == SK_F32 && Hq / Hkv > 64) {
    // The fp32 forward with one query row (reference:
    // src/stackkernels/torch/attention.py:154 computes it the same way).
    sk::FwdParams p{};
    p.q = q, p.k = k, p.v = v, p.o = o, p.lse = (float*)workspace;
    p.q_sb = q_strides[0], p.q_sh = q_strides[1], p.q_ss = q_strides[2];
    p.k_sb = k_strides[0], p.k_sh = k_strides[1], p.k_ss = k_strides[2];
    p.v_sb = v_strides[0], p.v_sh = v_strides[1], p.v_ss = v_strides[2];
    p.o_sb = o_strides[0], p.o_sh = o_strides[1], p.o_ss = o_strides[2];
    p.B = B, p.Hq = Hq, p.Hkv = Hkv, p.Sq = 1, p.Sk = Sk, p.D = D, p.group = Hq / Hkv;
    p.scale = softmax_scale(sm_scale);
    p.scale_log2 = p.scale * 1.4426950408889634f;
    p.q_sign = sm_scale < 0.f ? 1u : 0u;
    p.n_mblocks = 1;
    p.seqlens = seqlens;
    p.block_table = pc.block_table;
    p.page_size = pc.page_size, p.max_pages = pc.max_pages, p.num_pages = pc.num_pages;
    p.rope = rope;
    hipError_t e = sk::launch_fwd_f32(p, false, s);
    if (e != hipSuccess) return hip_fail(e, "sk_decode launch");
    return SK_OK;
  }

  sk::DecParams p{};
  p.q = q, p.k = k, p.v = v, p.o = o;
  p.q_sb = q_strides[0], p.q_sh = q_strides[1];
  p.k_sb = k_strides[0], p.k_sh = k_strides[1], p.k_ss = k_strides[2];
  p.v_sb = v_strides[0], p.v_sh = v_strides[1], p.v_ss = v_strides[2];
  p.o_sb = o_strides[0], p.o_sh = o_strides[1];
  p.B = B, p.Hq = Hq, p.Hkv = Hkv, p.Sk = Sk, p.D = D, p.group = Hq / Hkv;
  p.num_splits = num_splits;
  p.keys_per_split = kps;
  p.dpad = (int)decode_dpad(dtype, D);
  p.scale = softmax_scale(sm_scale);
  p.scale_log2 = p.scale * 1.4426950408889634f;
  p.q_sign = sm_scale < 0.f ? 0x80008000u : 0u;
  p.seqlens = seqlens;
  p.longest_first = seqlens != nullptr && B <= 256;
  p.block_table = pc.block_table;
  p.page_size = pc.page_size, p.max_pages = pc.max_pages, p.num_pages = pc.num_pages;
  p.rope = rope;
  if (num_splits > 1) {
    p.part_o = (float*)workspace;
    p.part_lse = p.part_o + (size_t)B * Hq * num_splits * p.dpad;
  }
  hipError_t e = sk::launch_decode_mfma(dtype, p, s);
  if (e != hipSuccess) return hip_fail(e, "sk_decode split launch");
  if (num_splits > 1) {
    e = sk::launch_decode_combine(dtype, p, s);
    if (e != hipSuccess) return hip_fail(e, "sk_decode combine launch");
  }
  return SK_OK;
}

extern "C" {

int sk_decode(int dtype, const void* q, const void* k, const void* v, void* o, void* workspace,
              size_t workspace_bytes, int num_splits, int B, int Hq, int Hkv, int Sk, int D,
              const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
              const int64_t* o_strides, float sm_scale, void* stream) {
  g_err[0] = 0;
  return decode_impl(dtype, q, k, v, o, workspace, workspace_bytes, num_splits, B, Hq, Hkv, Sk, D,
                     q_strides, k_strides, v_strides, o_strides, nullptr, PagedCache{},
                     sk::RopeParams{}, sm_scale, stream);
}

}  // extern "C"

// Library-held scratch of sk_decode_noalloc: SK_NOALLOC_SCRATCH_BYTES of
// device memory, one copy on every GPU the library runs on, held until the
// process ends.  On the host the array's name is a stand-in, not a device
// address, so host code never passes it to a kernel or a copy: each device's
// address comes from hipGetSymbolAddress, taken once per device with that
// device current, and kept in g_scratch_ptr.  Every sk_decode_noalloc call on
// a GPU shares that GPU's copy; nothing in it must start at zero (each split
// writes its whole partial before the combine reads it), but calls that
// overlap on one GPU race.
static __device__ __align__(256) uint8_t scratch[SK_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices];

// Device address of the scratch copy on the device of stream s.
int scratch_address(hipStream_t s, void** out) {
  hipDevice_t dev = -1;
  hipError_t e = hipStreamGetDevice(s, &dev);
  if (e != hipSuccess) return hip_fail(e, "sk_decode_noalloc: device of the stream");
  if (dev < 0 || dev >= kMaxScratchDevices)
    return fail(SK_EINVAL, "sk_decode_noalloc: device %d outside [0, %d)", dev, kMaxScratchDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    int cur = -1;
    if ((e = hipGetDevice(&cur)) != hipSuccess) return hip_fail(e, "sk_decode_noalloc: hipGetDevice");
    if (cur != dev && (e = hipSetDevice(dev)) != hipSuccess)
      return hip_fail(e, "sk_decode_noalloc: hipSetDevice");
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (cur != dev) (void)hipSetDevice(cur);
    if (e != hipSuccess) return hip_fail(e, "sk_decode_noalloc: hipGetSymbolAddress(scratch)");
    if (!ptr) return fail(SK_EINVAL, "sk_decode_noalloc: no scratch address on device %d", dev);
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return SK_OK;
}

}  // namespace

extern "C" {

int sk_decode_noalloc(int dtype, const void* q, const void* k, const void* v, void* o,
                      int num_splits, int B, int Hq, int Hkv, int Sk, int D,
                      const int64_t* q_strides, const int64_t* k_strides,
                      const int64_t* v_strides, const int64_t* o_strides, float sm_scale,
                      void* stream) {
  g_err[0] = 0;
  int rc = check_dims(dtype, B, Hq, Hkv, 1, Sk, D);
  if (rc) return rc;
  constexpr size_t kBytes = SK_NOALLOC_SCRATCH_BYTES;
  if (num_splits == 0 && dtype != SK_F32 && (int64_t)B * Hq > 0) {
    // the table's split count, lowered until the partials fit the scratch
    const size_t per_split = (size_t)B * Hq * (sk::padded_head_dim(D) + 1) * sizeof(float);
    const int64_t fit = std::max<int64_t>(1, (int64_t)(kBytes / per_split));
    num_splits = (int)std::min<int64_t>(plan_splits(B, Hq, Hkv, Sk, D, false), fit);
  }
  int splits = 0, kps = 0;
  if ((rc = decode_splits(dtype, B, Hq, Hkv, Sk, D, false, num_splits, &splits, &kps))) return rc;
  size_t need = decode_ws_bytes(dtype, B, Hq, D, splits);
  if (dtype == SK_F32 && need > kBytes) splits = 1, need = decode_ws_bytes(dtype, B, Hq, D, 1);
  if (need > kBytes)
    return fail(SK_EWORKSPACE,
                "sk_decode_noalloc: %d split(s) need %zu bytes of scratch, more than the "
                "library's %zu-byte static scratch (pass fewer splits, or use sk_decode)",
                splits, need, kBytes);
  void* ws = nullptr;
  if (need > 0 && (rc = scratch_address((hipStream_t)stream, &ws))) return rc;
  return decode_impl(dtype, q, k, v, o, ws, kBytes, splits, B, Hq, Hkv, Sk, D, q_strides,
                     k_strides, v_strides, o_strides, nullptr, PagedCache{}, sk::RopeParams{},
                     sm_scale, stream);
}

}  // extern "C"

// sk_kv_cache_update (page_size 0: S_cache rows per batch row) and
// sk_kv_cache_update_paged (S_cache = num_pages * page_size pool slots).
static int cache_update_impl(int dtype, const void* k, const void* v, void* k_cache,
                             void* v_cache, const int64_t* slots, int B, int Hkv, int T,
                             int64_t S_cache, int page_size, int D, const int64_t* k_strides,
                             const int64_t* v_strides, const int64_t* kc_strides,
                             const int64_t* vc_strides, const sk::RopeParams& rope,
                             void* stream) {
  if (dtype != SK_F32 && dtype != SK_F16 && dtype != SK_BF16)
    return fail(SK_EUNSUPPORTED, "unsupported dtype code %d", dtype);
  if (B < 0 || Hkv <= 0 || T < 0 || S_cache < 0 || D <= 0)
    return fail(SK_EINVAL, "invalid sizes B=%d Hkv=%d T=%d S_cache=%lld D=%d", B, Hkv, T,
                (long long)S_cache, D);
  const int64_t* sts[4] = {k_strides, v_strides, kc_strides, vc_strides};
  const char* names[4] = {"k", "v", "k_cache", "v_cache"};
  for (int i = 0; i < 4; ++i) {
    if (!sts[i]) return fail(SK_EINVAL, "%s strides pointer is NULL", names[i]);
    for (int j = 0; j < 3; ++j)
      if (sts[i][j] < 0)
        return fail(SK_EINVAL, "%s stride[%d]=%lld must be non-negative", names[i], j,
                    (long long)sts[i][j]);
  }
  if ((int64_t)B * T == 0) return SK_OK;
  const void* ptrs[5] = {k, v, k_cache, v_cache, slots};
  const char* pnames[5] = {"k", "v", "k_cache", "v_cache", "slot_indices"};
  for (int i = 0; i < 5; ++i)
    if (!ptrs[i]) return fail(SK_EINVAL, "%s pointer is NULL", pnames[i]);
  sk::CacheParams p{};
  p.k = k, p.v = v, p.kc = k_cache, p.vc = v_cache, p.slots = slots;
  p.k_sb = k_strides[0], p.k_sh = k_strides[1], p.k_ss = k_strides[2];
  p.v_sb = v_strides[0], p.v_sh = v_strides[1], p.v_ss = v_strides[2];
  p.kc_sb = kc_strides[0], p.kc_sh = kc_strides[1], p.kc_ss = kc_strides[2];
  p.vc_sb = vc_strides[0], p.vc_sh = vc_strides[1], p.vc_ss = vc_strides[2];
  p.B = B, p.Hkv = Hkv, p.T = T, p.S = S_cache;
  p.page_size = page_size;
  p.esize = elem_bytes(dtype);
  p.row_bytes = D * p.esize;
  p.dtype = dtype;
  p.D = D;
  p.rope = rope;
  if (rope.cos) {
    // The rotating kernel moves aligned 16-byte chunks.
    const void* rp[4] = {k, v, k_cache, v_cache};
    for (int i = 0; i < 4; ++i)
      if (!aligned16(rp[i])) return fail(SK_EINVAL, "%s pointer is not 16-byte aligned", names[i]);
    for (int i = 0; i < 4; ++i)
      for (int j = 0; j < 3; ++j)
        if ((sts[i][j] * p.esize) % 16 != 0)
          return fail(SK_EINVAL, "%s stride[%d]=%lld is not a multiple of 16 bytes", names[i], j,
                      (long long)sts[i][j]);
  }
  hipError_t e = sk::launch_kv_cache_update(p, (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, "sk_kv_cache_update launch");
  return SK_OK;
}

extern "C" {

int sk_kv_cache_update(int dtype, const void* k, const void* v, void* k_cache, void* v_cache,
                       const int64_t* slots, int B, int Hkv, int T, int S_cache, int D,
                       const int64_t* k_strides, const int64_t* v_strides,
                       const int64_t* kc_strides, const int64_t* vc_strides, void* stream) {
  g_err[0] = 0;
  return cache_update_impl(dtype, k, v, k_cache, v_cache, slots, B, Hkv, T, S_cache, 0, D,
                           k_strides, v_strides, kc_strides, vc_strides, sk::RopeParams{},
                           stream);
}

int sk_kv_cache_update_paged(int dtype, const void* k, const void* v, void* k_pool,
                             void* v_pool, const int64_t* slot_mapping, int B, int Hkv, int T,
                             int num_pages, int page_size, int D, const int64_t* k_strides,
                             const int64_t* v_strides, const int64_t* kp_strides,
                             const int64_t* vp_strides, void* stream) {
  g_err[0] = 0;
  if (page_size <= 0 || num_pages < 0)
    return fail(SK_EINVAL, "invalid page_size=%d num_pages=%d", page_size, num_pages);
  return cache_update_impl(dtype, k, v, k_pool, v_pool, slot_mapping, B, Hkv, T,
                           (int64_t)num_pages * page_size, page_size, D, k_strides, v_strides,
                           kp_strides, vp_strides, sk::RopeParams{}, stream);
}

int sk_decode_varlen(int dtype, const void* q, const void* k, const void* v, void* o,
                     void* workspace, size_t workspace_bytes, int num_splits, int B, int Hq,
                     int Hkv, int Sk, int D, const int64_t* q_strides, const int64_t* k_strides,
                     const int64_t* v_strides, const int64_t* o_strides,
                     const int32_t* cache_seqlens, float sm_scale, void* stream) {
  g_err[0] = 0;
  if (B > 0 && !cache_seqlens) return fail(SK_EINVAL, "cache_seqlens is null");
  return decode_impl(dtype, q, k, v, o, workspace, workspace_bytes, num_splits, B, Hq, Hkv, Sk, D,
                     q_strides, k_strides, v_strides, o_strides, cache_seqlens, PagedCache{},
                     sk::RopeParams{}, sm_scale, stream);
}

int sk_decode_paged(int dtype, const void* q, const void* k_pool, const void* v_pool, void* o,
                    void* workspace, size_t workspace_bytes, int num_splits, int B, int Hq,
                    int Hkv, int num_pages, int page_size, int max_pages, int D,
                    const int64_t* q_strides, const int64_t* kp_strides,
                    const int64_t* vp_strides, const int64_t* o_strides,
                    const int32_t* block_table, const int32_t* cache_seqlens, float sm_scale,
                    void* stream) {
  g_err[0] = 0;
  PagedCache pc;
  const int rc = paged_args(B, num_pages, page_size, max_pages, block_table, cache_seqlens, &pc);
  if (rc) return rc;
  return decode_impl(dtype, q, k_pool, v_pool, o, workspace, workspace_bytes, num_splits, B, Hq,
                     Hkv, max_pages * page_size, D, q_strides, kp_strides, vp_strides, o_strides,
                     cache_seqlens, pc, sk::RopeParams{}, sm_scale, stream);
}

int sk_decode_rope(int dtype, const void* q, const void* k, const void* v, void* o,
                   void* workspace, size_t workspace_bytes, int num_splits, int B, int Hq,
                   int Hkv, int Sk, int D, const int64_t* q_strides, const int64_t* k_strides,
                   const int64_t* v_strides, const int64_t* o_strides,
                   const int32_t* cache_seqlens, const void* rope_cos, const void* rope_sin,
                   int rope_dtype, int rope_rows, int64_t rope_stride, const int32_t* rope_pos,
                   int rope_start, float sm_scale, void* stream) {
  g_err[0] = 0;
  sk::RopeParams r{};
  const int rc = make_rope(rope_cos, rope_sin, rope_dtype, rope_rows, rope_stride, rope_pos,
                           rope_start, D, B > 0 ? 1 : 0, &r);
  if (rc) return rc;
  return decode_impl(dtype, q, k, v, o, workspace, workspace_bytes, num_splits, B, Hq, Hkv, Sk, D,
                     q_strides, k_strides, v_strides, o_strides, cache_seqlens, PagedCache{}, r,
                     sm_scale, stream);
}

int sk_decode_paged_rope(int dtype, const void* q, const void* k_pool, const void* v_pool,
                         void* o, void* workspace, size_t workspace_bytes, int num_splits, int B,
                         int Hq, int Hkv, int num_pages, int page_size, int max_pages, int D,
                         const int64_t* q_strides, const int64_t* kp_strides,
                         const int64_t* vp_strides, const int64_t* o_strides,
                         const int32_t* block_table, const int32_t* cache_seqlens,
                         const void* rope_cos, const void* rope_sin, int rope_dtype,
                         int rope_rows, int64_t rope_stride, const int32_t* rope_pos,
                         int rope_start, float sm_scale, void* stream) {
  g_err[0] = 0;
  PagedCache pc;
  int rc = paged_args(B, num_pages, page_size, max_pages, block_table, cache_seqlens, &pc);
  if (rc) return rc;
  sk::RopeParams r{};
  rc = make_rope(rope_cos, rope_sin, rope_dtype, rope_rows, rope_stride, rope_pos, rope_start, D,
                 B > 0 ? 1 : 0, &r);
  if (rc) return rc;
  return decode_impl(dtype, q, k_pool, v_pool, o, workspace, workspace_bytes, num_splits, B, Hq,
                     Hkv, max_pages * page_size, D, q_strides, kp_strides, vp_strides, o_strides,
                     cache_seqlens, pc, r, sm_scale, stream);
}

int sk_kv_cache_update_rope(int dtype, const void* k, const void* v, void* k_cache, void* v_cache,
                            const int64_t* slots, int B, int Hkv, int T, int S_cache, int D,
                            const int64_t* k_strides, const int64_t* v_strides,
                            const int64_t* kc_strides, const int64_t* vc_strides,
                            const void* rope_cos, const void* rope_sin, int rope_dtype,
                            int rope_rows, int64_t rope_stride, const int32_t* rope_pos,
                            int rope_start, void* stream) {
  g_err[0] = 0;
  sk::RopeParams r{};
  const int rc = make_rope(rope_cos, rope_sin, rope_dtype, rope_rows, rope_stride, rope_pos,
                           rope_start, D, B > 0 ? T : 0, &r);
  if (rc) return rc;
  return cache_update_impl(dtype, k, v, k_cache, v_cache, slots, B, Hkv, T, S_cache, 0, D,
                           k_strides, v_strides, kc_strides, vc_strides, r, stream);
}

int sk_kv_cache_update_paged_rope(int dtype, const void* k, const void* v, void* k_pool,
                                  void* v_pool, const int64_t* slot_mapping, int B, int Hkv,
                                  int T, int num_pages, int page_size, int D,
                                  const int64_t* k_strides, const int64_t* v_strides,
                                  const int64_t* kp_strides, const int64_t* vp_strides,
                                  const void* rope_cos, const void* rope_sin, int rope_dtype,
                                  int rope_rows, int64_t rope_stride, const int32_t* rope_pos,
                                  int rope_start, void* stream) {
  g_err[0] = 0;
  if (page_size <= 0 || num_pages < 0)
    return fail(SK_EINVAL, "invalid page_size=%d num_pages=%d", page_size, num_pages);
  sk::RopeParams r{};
  const int rc = make_rope(rope_cos, rope_sin, rope_dtype, rope_rows, rope_stride, rope_pos,
                           rope_start, D, B > 0 ? T : 0, &r);
  if (rc) return rc;
  return cache_update_impl(dtype, k, v, k_pool, v_pool, slot_mapping, B, Hkv, T,
                           (int64_t)num_pages * page_size, page_size, D, k_strides, v_strides,
                           kp_strides, vp_strides, r, stream);
}

int sk_rope_rotate(int dtype, const void* x, void* out, int B, int H, int S, int D,
                   const int64_t* x_strides, const int64_t* out_strides, const void* rope_cos,
                   const void* rope_sin, int rope_dtype, int rope_rows, int64_t rope_stride,
                   const int32_t* rope_pos, int rope_start, int inverse, void* stream) {
  g_err[0] = 0;
  int rc = check_dims(dtype, B, H, 1, S, 0, D);
  if (rc) return rc;
  if ((rc = check_strides(dtype, "x", x_strides)) || (rc = check_strides(dtype, "out", out_strides)))
    return rc;
  sk::RopeParams r{};
  const int64_t rows = (int64_t)B * H * S;
  if ((rc = make_rope(rope_cos, rope_sin, rope_dtype, rope_rows, rope_stride, rope_pos,
                      rope_start, D, rows > 0 ? S : 0, &r)))
    return rc;
  if (rows == 0) return SK_OK;
  if ((rc = check_ptr("x", x)) || (rc = check_ptr("out", out))) return rc;
  {
    // out's rows must not overlap one another (else the writes race): sorted
    // by stride, each dimension of extent > 1 must step past the rows of the
    // dimensions below it.
    int64_t ext[3] = {B, H, S}, st[3] = {out_strides[0], out_strides[1], out_strides[2]};
    for (int i = 0; i < 3; ++i)
      for (int j = i + 1; j < 3; ++j)
        if (st[j] < st[i]) std::swap(st[i], st[j]), std::swap(ext[i], ext[j]);
    int64_t span = D;  // elements the dimensions below cover
    for (int i = 0; i < 3; ++i) {
      if (ext[i] <= 1) continue;
      if (st[i] < span) return fail(SK_EINVAL, "out strides make rows overlap");
      span = st[i] * ext[i];
    }
  }
  if (x == out && (x_strides[0] != out_strides[0] || x_strides[1] != out_strides[1] ||
                   x_strides[2] != out_strides[2]))
    return fail(SK_EINVAL, "in place (out == x) needs out's strides to equal x's");
  if (x != out) {
    // In place or disjoint: a partial overlap would let one row's write
    // reach another row's unread input.
    const int64_t es = elem_bytes(dtype);
    const int64_t span_x = ((int64_t)(B - 1) * x_strides[0] + (int64_t)(H - 1) * x_strides[1] +
                            (int64_t)(S - 1) * x_strides[2] + D) * es;
    const int64_t span_o = ((int64_t)(B - 1) * out_strides[0] + (int64_t)(H - 1) * out_strides[1] +
                            (int64_t)(S - 1) * out_strides[2] + D) * es;
    const uintptr_t xa = (uintptr_t)x, oa = (uintptr_t)out;
    if (xa < oa + (uintptr_t)span_o && oa < xa + (uintptr_t)span_x)
      return fail(SK_EINVAL, "out overlaps x without being x");
  }
  sk::RotateParams p{};
  p.x = x, p.out = out;
  p.x_sb = x_strides[0], p.x_sh = x_strides[1], p.x_ss = x_strides[2];
  p.o_sb = out_strides[0], p.o_sh = out_strides[1], p.o_ss = out_strides[2];
  p.B = B, p.H = H, p.S = S, p.D = D;
  p.dtype = dtype;
  p.inverse = inverse != 0;
  p.rope = r;
  const hipError_t e = sk::launch_rope_rotate(p, (hipStream_t)stream);
  if (e != hipSuccess) return hip_fail(e, "sk_rope_rotate launch");
  return SK_OK;
}

}  // extern "C"

// ---------------------------------------------------------------- introspection

static const char* elem_name(int e) {
  return e == SK_BF16 ? "BF16" : e == SK_F16 ? "F16" : e == SK_F32 ? "F32" : "?";
}

extern "C" {

int sk_kernel_config(int op, int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D,
                     int is_causal, int num_splits, int variant, int query_device, int64_t* cfg,
                     char* kernel_name, size_t name_len) {
  g_err[0] = 0;
  if (!cfg) return fail(SK_EINVAL, "cfg pointer is NULL");
  for (int i = 0; i < SK_CFG_LEN; ++i) cfg[i] = 0;
  if (kernel_name && name_len) kernel_name[0] = 0;
  const bool decode = op == SK_OP_DECODE || op == SK_OP_DECODE_COMBINE;
  int rc = check_dims(dtype, B, Hq, Hkv, decode ? 1 : Sq, Sk, D);
  if (rc) return rc;
  if (decode && Hq / Hkv > 64 && dtype != SK_F32)
    return fail(SK_EUNSUPPORTED, "decode supports up to 64 query heads per KV head, got %d", Hq / Hkv);
  // Non-null stand-ins for the optional inputs a variant carries: the plan
  // only tests them for null, and nothing is launched here.
  static const int kStandIn = 0;
  const bool rope = (variant & SK_VARIANT_ROPE) != 0;
  const bool paged = (variant & SK_VARIANT_PAGED) != 0;
  sk::KernelPlan k;
  int64_t splits = 1, kps = 0, paired = 0, chunks = 1, packed = 1, side = 0;
  size_t ws = 0;
  if (op == SK_OP_FWD || op == SK_OP_FWD_COMBINE || (decode && dtype == SK_F32 && Hq / Hkv > 64)) {
    if (op == SK_OP_DECODE_COMBINE) {  // (unsplit: no combine pass)
      cfg[SK_CFG_SPLITS] = 1;
      return SK_OK;
    }
    sk::FwdParams p{};
    if ((rc = fwd_shape(dtype, B, Hq, Hkv, decode ? 1 : Sq, Sk, D, decode ? 0 : is_causal, &p)))
      return rc;
    if (rope) p.rope.cos = &kStandIn;
    if (paged && decode) p.block_table = &kStandIn;
    if (decode) {
      ws = decode_ws_bytes(dtype, B, Hq, D, 1);
    } else {
      // The call with the scratch sk_attn_fwd_workspace reports.
      const sk::FwdSplit f = sk::fwd_key_splits(dtype, D, B, Hq, Hkv, Sq, Sk, is_causal != 0);
      ws = fwd_ws_bytes(B, Hq, Sq, D, f);
      splits = f.splits, packed = f.pack;
      if (f.on()) {
        fwd_apply_split(dtype, f, const_cast<int*>(&kStandIn), &p);
        kps = p.split_keys;
      } else if (op == SK_OP_FWD_COMBINE) {
        cfg[SK_CFG_SPLITS] = 1;
        return SK_OK;
      }
    }
    k = op == SK_OP_FWD_COMBINE ? sk::plan_fwd_combine(dtype, p)
        : dtype == SK_F32       ? sk::plan_fwd_f32(p, !decode && is_causal)
                                : sk::plan_fwd_mfma(dtype, p, is_causal != 0);
    paired = p.pair_items;
  } else if (op == SK_OP_BWD_DKV || op == SK_OP_BWD_DQ || op == SK_OP_BWD_REDUCE) {
    sk::BwdParams p{};
    p.B = B, p.Hq = Hq, p.Hkv = Hkv, p.Sq = Sq, p.Sk = Sk, p.D = D, p.group = Hq / Hkv;
    // The plan of one chunk of pairs at the size sk_attn_bwd_workspace_best reports.
    const int64_t pairs = (int64_t)B * Hkv;
    const int64_t chunk = bwd_chunk_pairs(
        pairs, sk::bwd_ds_pair_bytes(dtype, Hq, Hkv, Sq, Sk, D, is_causal != 0),
        (size_t)SK_BWD_DS_CAP_BYTES);
    if (chunk > 0) {
      p.ds = const_cast<int*>(&kStandIn);
      p.n_pairs = (int)chunk;
      chunks = (pairs + chunk - 1) / chunk;
    }
    const BwdParts parts = bwd_parts(dtype, B, Hq, Hkv, Sq, Sk, D, is_causal != 0);
    ws = parts.bytes > 0 ? parts.offset + parts.bytes
                         : bwd_ws_bytes(dtype, B, Hq, Hkv, Sq, Sk, D, is_causal != 0);
    if (parts.bytes > 0) {
      p.kv_iters = parts.p.kv_iters, p.kv_chunks = parts.p.kv_chunks;
      p.dq_iters = parts.p.dq_iters, p.dq_chunks = parts.p.dq_chunks;
    }
    if (op == SK_OP_BWD_REDUCE && parts.bytes == 0) {
      cfg[SK_CFG_SPLITS] = 1;
      return SK_OK;
    }
    if (op == SK_OP_BWD_DKV && p.kv_iters > 0) splits = p.kv_chunks;
    if (op == SK_OP_BWD_DQ && p.dq_iters > 0) splits = p.dq_chunks;
    if (op == SK_OP_BWD_REDUCE)
      splits = std::max(p.kv_iters > 0 ? p.kv_chunks : 1, p.dq_iters > 0 ? p.dq_chunks : 1);
    if (op == SK_OP_BWD_DQ) side = sk::bwd_forks(dtype, p, is_causal != 0);
    k = op == SK_OP_BWD_DKV  ? sk::plan_bwd_dkv(dtype, p, is_causal != 0)
        : op == SK_OP_BWD_DQ ? sk::plan_bwd_dq(dtype, p, is_causal != 0)
                             : sk::plan_bwd_reduce(dtype, p);
  } else if (decode) {
    int ns = 0, per = 0;
    const bool per_row = (variant & (SK_VARIANT_PAGED | SK_VARIANT_VARLEN)) != 0;
    if ((rc = decode_splits(dtype, B, Hq, Hkv, Sk, D, per_row, num_splits, &ns, &per))) return rc;
    sk::DecParams p{};
    p.B = B, p.Hq = Hq, p.Hkv = Hkv, p.Sk = Sk, p.D = D, p.group = Hq / Hkv;
    p.num_splits = ns, p.keys_per_split = per, p.dpad = (int)decode_dpad(dtype, D);
    if (rope) p.rope.cos = &kStandIn;
    if (paged) p.block_table = &kStandIn;
    splits = ns, kps = per;
    ws = decode_ws_bytes(dtype, B, Hq, D, ns);
    if (op == SK_OP_DECODE_COMBINE && ns <= 1) {  // one split writes O directly
      cfg[SK_CFG_SPLITS] = splits;
      return SK_OK;
    }
    k = op == SK_OP_DECODE ? sk::plan_decode_mfma(dtype, p) : sk::plan_decode_combine(dtype, p);
  } else {
    return fail(SK_EINVAL, "unknown op %d", op);
  }
  if (!k.fn) return fail(SK_EUNSUPPORTED, "no kernel for op %d with these arguments", op);
  cfg[SK_CFG_GRID] = (int64_t)k.grid.x * k.grid.y * k.grid.z / (op == SK_OP_FWD ? splits : 1);
  cfg[SK_CFG_THREADS] = (int64_t)k.block.x * k.block.y * k.block.z;
  cfg[SK_CFG_BLOCK_M] = k.block_m;
  cfg[SK_CFG_BLOCK_N] = k.block_n;
  cfg[SK_CFG_STAGES] = k.stages;
  cfg[SK_CFG_HEAD_DIM] = k.head_dim;
  cfg[SK_CFG_SPLITS] = splits;
  cfg[SK_CFG_PAIRED] = paired;
  cfg[SK_CFG_WORKSPACE] = (int64_t)ws;
  cfg[SK_CFG_KEYS_PER_SPLIT] = kps;
  cfg[SK_CFG_CHUNKS] = chunks;
  cfg[SK_CFG_SIDE_STREAM] = side;
  cfg[SK_CFG_PACKED_HEADS] = packed;
  cfg[SK_CFG_LDS_BYTES] = cfg[SK_CFG_VGPRS] = cfg[SK_CFG_WG_PER_CU] = -1;
  if (kernel_name && name_len)
    snprintf(kernel_name, name_len, "%s<%s, D=%d, BM=%d, BN=%d, stages=%d, causal=%d, paged=%d, rope=%d>",
             k.kernel, elem_name(k.elem), k.head_dim, k.block_m, k.block_n, k.stages, (int)k.causal,
             (int)k.paged, (int)k.rope);
  if (query_device) {
    hipFuncAttributes a{};
    hipError_t e = hipFuncGetAttributes(&a, k.fn);
    if (e != hipSuccess) return hip_fail(e, "sk_kernel_config attributes");
    int per_cu = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k.fn, (int)cfg[SK_CFG_THREADS], 0);
    if (e != hipSuccess) return hip_fail(e, "sk_kernel_config occupancy");
    cfg[SK_CFG_LDS_BYTES] = (int64_t)a.sharedSizeBytes;
    cfg[SK_CFG_VGPRS] = a.numRegs;
    cfg[SK_CFG_WG_PER_CU] = per_cu;
  }
  return SK_OK;
}

}  // extern "C"
