// grouped_plan.h -- which kernels a grouped call (T > 1) runs on.  Host code
// only, no HIP: the choice depends on sizes alone.
//
// Token pairs (16x16x128 MFMA, items of up to 4 rows) for T <= 4, token octets
// (32x32x64 MFMA, items of up to 8 rows) above that, and the stacked kernels
// (items of up to 32 or 64 rows) where an expert's rows fill several octets or
// the chip has octets to spare.
#pragma once

#define MOE_PLAN_PAIR_TOKENS 4
#define MOE_PLAN_ROWS 32   // rows of a stacked item
#define MOE_PLAN_ROWS2 64  // where two token tiles share the weights

struct grouped_plan {
  bool octets;    // T > 4
  bool stacked;   // octets, but on the stacked kernels
  bool in_order;  // stacked: sums block by block in f32 (else in f64)
  int item_rows;
};

static inline grouped_plan plan_grouped(int T, int k, int E, int H, int F, bool shared) {
  grouped_plan p;
  const long P = (long)T * k;
  p.octets = T > MOE_PLAN_PAIR_TOKENS;
  // the stacked kernels add their block sums one by one in f32 on the shapes
  // that always did (results keep their bits).  The others' results came from
  // the octet kernels, which err less (their separate digit planes round less
  // often), so their sums are in f64: 300 tokens on a 5120 x 1536 layer 571 ->
  // 458 us, rows 4.9e-8 -> 3.6e-8 from 64 bits (f32 group sums 405 us, 7.2e-8)
  p.in_order = (H == 128 * 56 || H == 128 * 48 || H == 128 * 32 || H == 128 * 16) &&
               (F == 128 * 8 || F == 128 * 12 || F == 128 * 16 || F == 128 * 24);
  // A stacked workgroup reads an expert's weights once for up to 32 rows, but
  // it has twice the rows of weights of an octet workgroup, all of K instead
  // of half of it, and the same work however few rows its item holds.  So it
  // wants at least a round of octet workgroups to replace (two per CU, 512;
  // below that the chip is not full and the shorter workgroup wins), and rows:
  // 8 per expert with f64 sums (two vector instructions per MFMA value), 5 with
  // f32 sums (one).  us per layer, cold weights, uniform routing, octets /
  // stacked:
  //   5120 x 1536, 8 experts, 2, 8, 16, 32 rows each   33/57  44/58  49/61  70/65
  //   2048 x 768, 32 experts, 2, 8, 16, 32 rows        28/35  39/43  49/44  70/58
  //   6400 x 2560, 128 experts, 2, 4, 8, 16 rows       512/575  572/646  734/696  1098/749
  //   7168 x 2048 (f32), 8 experts, 2, 8, 16 rows      43/64  63/65  78/64
  //   7168 x 2048 (f32), 128 experts, 2, 4, 8 rows     415/427  496/487  632/532
  // Large calls run stacked at fewer rows too, since skewed routing, which the
  // host does not see, gains more there than even routing loses: f32 from 1536
  // workgroups on (2048 x 3072, 233 experts, 4.5 rows, Zipf 249/141; 2048 x
  // 2048, 229 experts, 2.6 rows, uniform 235/258), f64 from 3000 and 4 rows on
  // (random shapes at 4-6 rows: Zipf 22-24% faster, uniform 7-12% slower; at
  // 2-4 rows, or with 1536-3000 workgroups, the two sides cancel or lose).  The
  // workgroups are counted for uniform routing, in the launch with fewer.
  const int gu = F / 64, dn = H / 128;  // octet workgroups per item: k_gate_up_o, k_down_o
  const long n8 = (P / 8 + E / 2 + (shared ? T / 8 : 0)) * (gu < dn ? gu : dn);
  const bool worth = p.in_order ? n8 >= 512 && (P >= 5L * E || n8 >= 1536)
                                : n8 >= 640 && (P >= 8L * E || (P >= 4L * E && n8 >= 3000));
  p.stacked = p.octets && P >= 2L * E && worth;
  // Two token tiles per weight pair (items of up to 64 rows): a weight is read
  // and duplicated once for both, 2048 tokens on the V3 layer 2308 -> 2134 us,
  // but the workgroups are half as many and run twice as long.  So only where
  // 64-row items still make two rounds of workgroups (512 a round) in the launch
  // that has fewer, from 4 pairs per expert on (below that the shared expert's
  // items are the only large ones: 64 tokens on the V3 layer 241 -> 259 us).  us
  // per layer, 32-row / 64-row items, 32 and 64 rows per expert:
  //   7168 x 2048, 8 experts 78/92  104/111; 32 experts 232/221  333/360; 128 experts 762/718  1214/1094
  //   2048 x 1024, 8 experts 34/44  35/48; 32 experts 54/65  75/76; 128 experts 148/152  219/221
  //   4096 x 1536, 32 experts 114/112  166/176; 128 experts 361/350  561/524
  // The f64 sums leave no registers for two tiles.
  const long items64 = (P / 64 > E ? P / 64 : E) + (shared ? T / 64 : 0);
  const int gu2 = F / 128, dn2 = H / 256;  // stacked workgroups per item
  const bool two = p.in_order && P >= 4L * E && items64 * (gu2 < dn2 ? gu2 : dn2) >= 1024;
  p.item_rows = !p.octets ? 4 : !p.stacked ? 8 : two ? MOE_PLAN_ROWS2 : MOE_PLAN_ROWS;
  return p;
}
