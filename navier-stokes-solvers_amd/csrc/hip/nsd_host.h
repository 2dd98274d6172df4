/* nsd_host.h -- one step on host arrays (internal to the library). */
#ifndef NSD_HOST_H
#define NSD_HOST_H

#include "ns_device.h"

#ifdef __cplusplus
extern "C" {
#endif

/* A solver's host arrays (ns_spectral_solver.h's layouts).  omega_hat, sfd_hat
 * (NULL: none), t and dt are read and written, the others written. */
typedef struct {
    double *omega_hat, *sfd_hat, *psi_hat, *u_hat, *v_hat;
    double *u, *v, *omega;
    double t, dt;
    int status;
} NsdHostFields;

/* 1 if the context's arrays fit its pinned buffer (allocated on the first call) */
int nsd_host_step_fits(NsdContext *ctx);
/* nsd_state_upload, nsd_sfd_upload, nsd_set_time, one step of fixed dt, nsd_get_time
 * and, unless the status is not 0, nsd_state_download, nsd_state_derived and
 * nsd_sfd_download, with one wait for the device.  Contexts for which
 * nsd_host_step_fits is 1. */
int nsd_host_step(NsdContext *ctx, NsdHostFields *f);

#ifdef __cplusplus
}
#endif
#endif /* NSD_HOST_H */
