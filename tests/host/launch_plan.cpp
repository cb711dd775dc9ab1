// Prints the launch plan of every problem on standard input, one per line: B N Sq Sk D tri ->
// forward key groups and slices, dQ key groups, dK/dV key groups per wave and slices (on 256 CUs, room for every slice), and
// whether the forward's walks are long enough for its pipelined loop.
#include <cstdint>
#include <cstdio>

#include "../../acctransformer_amd/csrc/fa_index_math.hpp"

int main() {
  int B, N, Sq, Sk, D, tri;
  while (scanf("%d %d %d %d %d %d", &B, &N, &Sq, &Sk, &D, &tri) == 6) {
    const acct::FwdPlan f = acct::fwd_plan(B, N, Sq, Sk, D, false, tri, true, 256, Sk, tri);
    const acct::DkdvPlan d = acct::dkdv_plan(B, N, Sq, Sk, D, tri, SIZE_MAX);
    printf("%d %d %d %d %d %d\n", f.kg, f.kv_split, acct::dq_key_groups(B, N, Sq, Sk, D, tri), d.ngk, d.q_split,
           (int)acct::pipelined_pays(Sq, Sk, tri));
  }
}
