// Prints host evaluations of functions that the kernels and their launches share.
#include "operator_plan.hpp"
#include "stencil_kernels.hpp"
#include "vector_kernels.hpp"

#include <iostream>
#include <limits>
#include <string>
#include <utility>

namespace
{
  ppf::GridDesc
  lattice(int n0, int n1, int n2)
  {
    ppf::GridDesc g {};
    g.nodes[0] = n0;
    g.nodes[1] = n1;
    g.nodes[2] = n2;
    return g;
  }

  /// Whether a transfer launch between the lattices is refused, restriction then prolongation.
  std::string
  refused(const ppf::GridDesc &gc, const ppf::GridDesc &gf)
  {
    std::string r;
    for (const ppf::GridDesc *out : {&gc, &gf})
      try
        {
          (void) ppf::transfer_grid(*out, gc, gf, 1);
          r += "0";
        }
      catch (const ppf::Error &)
        {
          r += "1";
        }
    return r;
  }

  /// Taps of weight zero whose position no tap of the same output has with another weight, and
  /// positions outside the lattice that is read.
  template <int taps>
  void
  count(const int (&pos)[taps], const double (&w)[taps], int n, int &stray, int &outside)
  {
    for (int k = 0; k < taps; ++k)
      {
        bool counts = false;
        for (int m = 0; m < taps; ++m)
          counts = counts || (pos[m] == pos[k] && w[m] != 0.0);
        stray += !counts;
        outside += pos[k] < 0 || pos[k] >= n;
      }
  }

  template <int degree>
  void
  transfer_taps()
  {
    int stray[2] = {}, outside[2] = {};
    for (int periodic = 0; periodic < 2; ++periodic)
      for (int cells = 1; cells <= 5; ++cells) // of the coarse lattice
        {
          const int nc = degree * cells + !periodic, nf = 2 * degree * cells + !periodic;
          for (int J = 0; J < nc; ++J)
            {
              int    pos[ppf::restrict_taps<degree>];
              double w[ppf::restrict_taps<degree>];
              ppf::restrict_axis<degree>(J, nf, periodic, pos, w);
              count(pos, w, nf, stray[0], outside[0]);
            }
          for (int I = 0; I < nf; ++I)
            {
              int    pos[degree + 1];
              double w[degree + 1];
              ppf::prolong_axis<degree>(I, nc, periodic, pos, w);
              count(pos, w, nc, stray[1], outside[1]);
            }
        }
    std::cout << "taps_q" << degree << ": " << stray[0] << " " << outside[0] << " " << stray[1]
              << " " << outside[1] << "\n";
  }
} // namespace

int
main()
{
  // CG's end flag as the launches with scalars 5, 6 and 7 find it when 6 ends the iteration
  std::cout << "turn_open: " << ppf::cg_ended_before(0, 5) << ppf::cg_ended_before(0, 6) << "\n"
            << "turn_racing: " << ppf::cg_ended_before(6, 6) << "\n"
            << "turn_after: " << ppf::cg_ended_before(6, 7) << "\n"
            << "turn_last_tag: " << ppf::cg_ended_before(0x7fffffff, 1)
            << ppf::cg_ended_before(0x7fffffff, 0x7fffffffu) << "\n";

  // fine planes of just under 2^31 nodes, of 2^31 (the coarse one a quarter), and of
  // 2^33 whose number no 32-bit product holds; more planes than a grid's second extent
  std::cout << "transfer_fits: " << refused(lattice(23170, 23170, 1), lattice(46339, 46339, 1))
            << "\n"
            << "transfer_fine_plane: "
            << refused(lattice(32768, 16385, 1), lattice(65536, 32769, 1))
            << refused(lattice(46341, 46340, 1), lattice(92681, 92679, 1)) << "\n"
            << "transfer_planes: " << refused(lattice(2, 2, 40000), lattice(3, 3, 79999)) << "\n";
  // comparisons: in agreement, apart, zero with zero, nothing with something, not finite
  std::cout << "check: ";
  const double inf = std::numeric_limits<double>::infinity();
  for (auto [worst, scale] : {std::pair {1e-13, 2.0}, {1e-3, 2.0}, {0.0, 0.0}, {1e-30, 0.0},
                              {inf, 2.0}, {inf, 0.0}})
    std::cout << int(ppf::check_plan(worst, scale, 1e-11));
  std::cout << "\ncheck_again: ";
  for (unsigned int n : {1u, 2u, 3u, 4u, 20u, 4000000000u})
    std::cout << ppf::applications_until_check(n) << " ";
  std::cout << "\n";
  // plans derived anew: split, coupled and generic before, each followed by each
  std::cout << "keeps_check: ";
  for (int before = 0; before < 3; ++before)
    for (int now = 0; now < 3; ++now)
      {
        ppf::SplitPlan p, q;
        p.eligible = before == 0;
        p.coupled  = before == 1;
        q.eligible = now == 0;
        q.coupled  = now == 1;
        std::cout << ppf::keeps_check(p, q);
      }
  std::cout << "\n";
  std::cout << "limits_auto: " << ppf::column_limit(2, -1, false) << " "
            << ppf::column_limit(3, -1, false) << " " << ppf::node_limit(-1) << "\n"
            << "limits_tiles: " << ppf::column_limit(2, -1, true) << " "
            << ppf::column_limit(3, -1, true) << "\n"
            << "limits_given: " << ppf::column_limit(3, 0, true) << " "
            << ppf::column_limit(3, 7, false) << " " << ppf::node_limit(7) << "\n";
  transfer_taps<1>();
  transfer_taps<2>();
}
