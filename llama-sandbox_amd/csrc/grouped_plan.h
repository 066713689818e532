// grouped_plan.h -- which kernels a grouped call (T > 1) runs on.  Host code
// only, no HIP: the choice depends on sizes alone.
//
// Token pairs (16x16x128 MFMA, items of up to 4 rows) for T <= 4, token octets
// (32x32x64 MFMA, items of up to 8 rows) above that, and the stacked kernels
// (items of up to 32 or 64 rows) for calls that fill the chip.
#pragma once

#define MOE_PLAN_PAIR_TOKENS 4
#define MOE_PLAN_ROWS 32   // rows of a stacked item
#define MOE_PLAN_ROWS2 64  // where two token tiles share the weights

struct grouped_plan {
  bool octets;    // T > 4
  bool stacked;   // octets, but on the stacked kernels
  bool in_order;  // stacked: sums block by block in f32 (else in f64)
  bool octet_f64;  // octets with sums in f64 (else in f32)
  int item_rows;
};

static inline grouped_plan plan_grouped(int T, int k, int E, int H, int F, bool shared) {
  grouped_plan p;
  const long P = (long)T * k;
  p.octets = T > MOE_PLAN_PAIR_TOKENS;
  // Order of the stacked kernels' block sums: one by one in f32 on the shapes
  // that they first ran on (results keep their bits), in f64 on all others,
  // which came from the octet kernels.  Those err less than f32 in order (their
  // separate digit planes round less often), so f32 would lose precision there:
  // rms of output rows from 64 bits, f32 / octets / f64, 0.9-1.3e-7 / 4.1-5.8e-8
  // / 3.6e-8.  And f64 everywhere costs the first shapes more than these kernels
  // gained them over their e4m3 form: V3 layer, 64 and 512 tokens Zipf, 512 and
  // 2048 uniform, e4m3 / f32 / f64: 241/227/253, 835/689/907, 1214/1143/1308,
  // 2868/2196/3174 us.
  p.in_order = (H == 128 * 56 || H == 128 * 48 || H == 128 * 32 || H == 128 * 16) &&
               (F == 128 * 8 || F == 128 * 12 || F == 128 * 16 || F == 128 * 24);
  // A stacked workgroup reads an expert's weights once for up to 32 rows, but
  // it has twice the rows of weights of an octet workgroup and all of K instead
  // of half of it.  Where the octets do not fill the chip (two workgroups per
  // CU are 512), the shorter workgroup wins, whatever the rows.  The octets'
  // workgroups are counted for uniform routing, in the launch that has fewer.
  // us per layer, cold weights, uniform, octets / stacked, and their count:
  //   5120 x 1536, 8 experts, 2, 16, 32 rows each   33/46  49/61  70/65 (144, 480, 864)
  //   5120 x 1536, 32 experts, 2, 4, 8 rows         81/88  96/99  116/109 (624, 864, 1344)
  //   6400 x 2560, 128 experts, 2, 4, 8 rows        512/493  572/539  734/601
  // With f32 sums the line lies lower (calls keep the bits that they had):
  //   7168 x 2048, 8 experts, 2, 8, 16 rows         42/65  62/59  78/64 (192, 384, 640)
  //   2048 x 1024, 8 experts, 8, 16, 32 rows        22/30  28/32  36/34 (192, 320, 576)
  const int gu = F / 64, dn = H / 128;  // octet workgroups per item: k_gate_up_o, k_down_o
  const long n8 = (P / 8 + E / 2 + (shared ? T / 8 : 0)) * (gu < dn ? gu : dn);
  p.stacked = p.octets && P >= 2L * E && n8 >= (p.in_order ? 300 : 512);
  // Shapes that sum in f64 do so on octets too, from 2 pairs per expert on: the
  // same rows, bit for bit, as in a larger call.  It costs 3-6% (8 tokens on 5120
  // x 1536, 8 experts 33.2 -> 34.7 us; 32 tokens on 32 experts 95.6 -> 97.9 us;
  // 2048 x 768, 8-12%).
  p.octet_f64 = p.octets && !p.stacked && !p.in_order && P >= 2L * E;
  // Two token tiles per weight pair (items of up to 64 rows): a weight is read
  // and duplicated once for both, but the workgroups are half as many and run
  // twice as long.  So only where 64-row items still make one and a half rounds
  // of workgroups (512 a round) in the launch that has fewer -- or 400, where
  // the average expert has 32-64 rows, one item instead of two --, from 4 pairs
  // per expert on (below that the shared expert's items are the only large
  // ones).  us per layer, 32-row / 64-row items, and their workgroups:
  //   7168 x 2048, 8 experts, 32, 64 rows each      78/92  103/107 (128, 192)
  //   7168 x 2048, 32 experts, 16, 32, 64 rows      170/175  230/209  323/340 (544, 576, 640)
  //   7168 x 2048, 128 experts, 32, 64 rows         748/718  1186/1082 (2176, 2304)
  //   2048 x 1024, 32 experts, 8, 32, 64 rows       45/54  54/65  75/74 (264, 288, 320)
  //   7168 x 1536, 63 experts, 43 rows              466/371 (924)
  // (fitted to 350 random shapes: in the mean 1.0% over the better of the two).
  // The f64 sums leave no registers for two tiles.
  const long items64 = (P / 64 > E ? P / 64 : E) + (shared ? T / 64 : 0);
  const int gu2 = F / 128, dn2 = H / 256;  // stacked workgroups per item
  const long n64 = items64 * (gu2 < dn2 ? gu2 : dn2);
  const bool two = p.in_order && P >= 4L * E && n64 >= (P >= 32L * E && P < 64L * E ? 400 : 768);
  p.item_rows = !p.octets ? 4 : !p.stacked ? 8 : two ? MOE_PLAN_ROWS2 : MOE_PLAN_ROWS;
  return p;
}
