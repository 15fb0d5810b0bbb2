// Host side of the fused x pass at a run-time x length: plan and kernel choice
// (the kernels of each workgroup size and mask mode are compiled apart).

#include "mr_xbd_rt.hpp"

bool mr_rt_len_make(const mr_fft_len<float> &fx, mr_rt_len *f)
{
    if (fx.nst > MR_RT_MAXST || fx.n > MR_RT_EPT * 1024) return false;
    f->n = fx.n;
    f->nst = fx.nst;
    int Ns = 1;
    for (int s = 0; s < fx.nst; ++s) {
        f->radix[s] = fx.radix[s];
        f->m[s] = fx.n / fx.radix[s];
        f->md[s] = mr_d24_make((unsigned)f->m[s]);
        f->nd[s] = mr_d24_make((unsigned)Ns);
        Ns *= fx.radix[s];
    }
    return true;
}

mr_xbd_rt_fn mr_xbd_rt_512(int L);
mr_xbd_rt_fn mr_xbd_rt_512m(int L);
mr_xbd_rt_fn mr_xbd_rt_1024(int L);
mr_xbd_rt_fn mr_xbd_rt_1024m(int L);

mr_xbd_rt_fn mr_xbd_rt_pick(int L, bool masked, int nt)
{
    if (nt == 512) return masked ? mr_xbd_rt_512m(L) : mr_xbd_rt_512(L);
    return masked ? mr_xbd_rt_1024m(L) : mr_xbd_rt_1024(L);
}
