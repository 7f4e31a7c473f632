// Scalar state of a COCG iteration: how the sums of an apply and of an update advance it
// (shared by the finishing kernels, vector.hip, and the one-launch iteration, iter.hip).
#pragma once
#include "common.hpp"

namespace mx {

// alpha (and the fused form's beta) from p^T A p and q^T q; tot = {mu re, im, qtq re, im}
// ({., ., ||A g||^2, .} for a rescue step)
__device__ __forceinline__ void fin_apply_state(SysState* st, int& f, const double (&tot)[4], bool fused) {
  if (f & SF_MR) {
    // rescue step along the hashed direction p = g: alpha = ||r|| / ||A g|| makes the
    // new residual r - alpha A g generic (r^T r no longer ~ 0); beta = 0 restarts
    // COCG from that residual.
    const double qq = tot[2];
    const cplx<double> alpha{sqrt(st->rnorm2 / qq), 0.0};
    if (!(qq > 0.0) || !finite(alpha.re)) f |= SF_BREAKDOWN | SF_PAUSE | SF_LIMIT;   // A g = 0
    else {
      st->alpha = alpha;
      if (fused) {   // beta = 0 restarts the fused recurrence (classic: k_pupdate does);
        st->beta = cplx<double>{0.0, 0.0};   // the step is taken, so the next apply is
        f &= ~(SF_RESTART | SF_MR);           // an ordinary one
        st->xc1 = alpha;                      // x_lo += alpha g now (a replacement has
        st->xc2 = cplx<double>{0.0, 0.0};     // just flushed any deferred term)
        f &= ~SF_XSKIP;
      }
    }
  } else {
    const cplx<double> mu{tot[0], tot[1]}, qtq{tot[2], tot[3]};
    st->mu = mu;
    const cplx<double> rho = st->rho;
    const cplx<double> alpha = cdiv(rho, mu);
    if (!(norm2(mu) > 0.0) || !finite(alpha.re) || !finite(alpha.im)) {
      // p^T A p vanished (or overflowed): replace the residual, then rescue with a
      // step along a hashed direction and restart from p = r
      f |= SF_BREAKDOWN | SF_PAUSE | SF_RESTART | SF_MR;
      if (!finite(mu.re) || !finite(mu.im)) f |= SF_NAN | SF_LIMIT;
    } else {
      if (fused) {   // predicted rho' = alpha^2 q^T q - rho; beta = rho' / rho
        cplx<double> beta = cdiv(alpha * alpha * qtq, rho) - cplx<double>{1.0, 0.0};
        if (!finite(beta.re) || !finite(beta.im)) beta = cplx<double>{0.0, 0.0};
        st->beta = beta;
        // Deferred solution update: x_lo needs alpha p of every pass, but only at a
        // replacement.  A pass may leave x_lo alone when the next one can recover that
        // term: the pass forms p' = r' + beta p, so alpha p = (alpha / beta) (p' - r').
        // The next pass then adds both terms at once, x_lo += (xa + alpha') p' - xa r'
        // (xa = alpha / beta), and x_lo is read and written every other pass.  A pending
        // term is flushed by k_accum before a replacement changes p and r.
        if (f & SF_XPEND) {
          st->xc1 = st->xa + alpha;
          st->xc2 = cplx<double>{-st->xa.re, -st->xa.im};
          f &= ~(SF_XPEND | SF_XSKIP);
        } else if (norm2(beta) >= kDeferBeta2) {
          st->xa = cdiv(alpha, beta);
          f |= SF_XSKIP | SF_XPEND;
        } else {
          st->xc1 = alpha;
          st->xc2 = cplx<double>{0.0, 0.0};
          f &= ~SF_XSKIP;
        }
      }
      st->alpha = alpha;
      f &= ~SF_RESTART;
    }
  }
  if (!(f & SF_PAUSE)) f |= SF_UPD_PENDING;   // the update runs next
}

// rho = r^T r, ||r||^2 of the updated residual and the checks; tot = {rho re, im, ||r||^2}
__device__ __forceinline__ void fin_update_state(SysState* st, int& f, const double (&tot)[3], bool fused) {
  const cplx<double> rho{tot[0], tot[1]};
  const double rn2 = tot[2];
  f &= ~(SF_SAVE | SF_UPD_PENDING);   // any saved best iterate was stored by k_save_best before this
  const bool rescued = (f & SF_MR) != 0;
  f &= ~SF_MR;       // a rescue step (if that was one) is done
  if (!fused) {      // classic: beta from the exact rho'; a rescue step restarts
    if (rescued) st->beta = cplx<double>{0.0, 0.0};
    else if (norm2(st->rho) > 0.0) st->beta = cdiv(rho, st->rho);
    else {           // rho breakdown: restart from the replaced residual
      f |= SF_BREAKDOWN | SF_PAUSE | SF_RESTART;
      st->beta = cplx<double>{0.0, 0.0};
    }
  }
  // r^T r ~ 0 with r != 0: the next step is a rescue step along a hashed direction.
  // The fused form has already built p from r, so it pauses for a replacement, after
  // which k_pupdate writes the rescue direction.
  if (norm2(rho) <= kRhoBreakdown * kRhoBreakdown * rn2 * rn2 && rn2 > 0.0)
    f |= SF_MR | SF_RESTART | (fused ? SF_PAUSE : 0);
  st->rho_old = st->rho;
  st->rho = rho;
  st->rnorm2 = rn2;
  if (rn2 > st->rmax2) st->rmax2 = rn2;
  st->iters += 1;
  st->since += 1;
  if (!finite(rn2) || !finite(rho.re) || !finite(rho.im)) {
    f |= SF_NAN | SF_PAUSE | SF_LIMIT;
  } else if (rn2 <= st->stop2 || rn2 <= st->delta2 * st->rmax2 ||
             (st->refresh_iters > 0 && st->since >= st->refresh_iters)) {
    f |= SF_PAUSE;
  }
  if (st->iters >= st->maxiter) f |= SF_PAUSE | SF_LIMIT;
}

}  // namespace mx
