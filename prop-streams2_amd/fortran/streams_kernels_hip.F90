! streams_kernels_hip.F90 -- generated by gen_interfaces.py from include/streams_hip.h; do not edit.
!
! Fortran drop-in for the reference's CUDA-Fortran kernel module (streams_kernels_gpu,
! src/multideal/kernels_gpu.F90): same routine names and argument order, device arrays as
! type(c_ptr) handles (hipMalloc'd by the caller), N_S from the preprocessor as in
! index_define.h.  Each wrapper calls the gfx950 library libstreams_hip.so and stops with the
! routine's name on a nonzero status.
#ifndef N_S
#define N_S 9
#endif
module streams_kernels_hip
  use, intrinsic :: iso_c_binding
  implicit none
  private :: check
  interface
    integer(c_int) function streams_species_supported(list, cap) &
        bind(C, name="streams_species_supported")
      import :: c_int, c_double, c_ptr
      type(c_ptr), value :: list
      integer(c_int), value :: cap
    end function streams_species_supported
    integer(c_int) function streams_eval_aux(n_s, nx, ny, nz, ng, nv, nv_aux, istart, iend, jstart, &
        jend, kstart, kend, w, w_aux, p0, t_min_tab, dt_tab, r_univ, rgas, cv_coeff, cp_coeff, &
        nsetcv, trange, indx_cp_l, indx_cp_r, tol_iter_nr, stream, mw, mwinv, visc_species, &
        lambda_species, diffbin_species, num_t_tab, n_eoi, aw_eoi, nainsp, beta0, coeff_eoi) &
        bind(C, name="streams_eval_aux")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: istart
      integer(c_int), value :: iend
      integer(c_int), value :: jstart
      integer(c_int), value :: jend
      integer(c_int), value :: kstart
      integer(c_int), value :: kend
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      real(c_double), value :: p0
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      real(c_double), value :: r_univ
      type(c_ptr), value :: rgas
      type(c_ptr), value :: cv_coeff
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      real(c_double), value :: tol_iter_nr
      type(c_ptr), value :: stream
      type(c_ptr), value :: mw
      type(c_ptr), value :: mwinv
      type(c_ptr), value :: visc_species
      type(c_ptr), value :: lambda_species
      type(c_ptr), value :: diffbin_species
      integer(c_int), value :: num_t_tab
      integer(c_int), value :: n_eoi
      type(c_ptr), value :: aw_eoi
      type(c_ptr), value :: nainsp
      type(c_ptr), value :: beta0
      type(c_ptr), value :: coeff_eoi
    end function streams_eval_aux
    integer(c_int) function streams_eval_aux2(n_s, nx, ny, nz, ng, nv_aux, visc_order, w_aux, &
        coeff_deriv1, dcsidx, detady, dzitdz, eps_sensor, sensor_type, stream) &
        bind(C, name="streams_eval_aux2")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv_aux
      integer(c_int), value :: visc_order
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      real(c_double), value :: eps_sensor
      integer(c_int), value :: sensor_type
      type(c_ptr), value :: stream
    end function streams_eval_aux2
    integer(c_int) function streams_eval_velaux(n_s, nx, ny, nz, ng, nv, nv_aux, w, w_aux, stream) &
        bind(C, name="streams_eval_velaux")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: stream
    end function streams_eval_velaux
    integer(c_int) function streams_les_wale_mut(n_s, nx, ny, nz, ng, nv_aux, ep_order, w_aux, &
        coeff_deriv1, dcsidx, detady, dzitdz, les_c_wale, eps_sensor, sensor_type, stream) &
        bind(C, name="streams_les_wale_mut")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv_aux
      integer(c_int), value :: ep_order
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      real(c_double), value :: les_c_wale
      real(c_double), value :: eps_sensor
      integer(c_int), value :: sensor_type
      type(c_ptr), value :: stream
    end function streams_les_wale_mut
    integer(c_int) function streams_eval_aux_les(n_s, nx, ny, nz, ng, nv, nv_aux, w, w_aux, p0, &
        t_min_tab, dt_tab, r_univ, rgas, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, &
        tol_iter_nr, mw, mwinv, visc_species, lambda_species, diffbin_species, num_t_tab, les_pr, &
        les_sc, stream) &
        bind(C, name="streams_eval_aux_les")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      real(c_double), value :: p0
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      real(c_double), value :: r_univ
      type(c_ptr), value :: rgas
      type(c_ptr), value :: cv_coeff
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      real(c_double), value :: tol_iter_nr
      type(c_ptr), value :: mw
      type(c_ptr), value :: mwinv
      type(c_ptr), value :: visc_species
      type(c_ptr), value :: lambda_species
      type(c_ptr), value :: diffbin_species
      integer(c_int), value :: num_t_tab
      real(c_double), value :: les_pr
      real(c_double), value :: les_sc
      type(c_ptr), value :: stream
    end function streams_eval_aux_les
    integer(c_int) function streams_eval_chem_aux(n_s, nx, ny, nz, nv_aux, ng, nreactions, w_aux, &
        mw, arr_a, arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, p_coeffs, &
        kc_tab, num_t_tab, t_min_tab, dt_tab, r_univ, dcsidx, detady, dzitdz, h298, enable_pasr, &
        les_c_yoshi, les_c_mix, les_c_eps, stream) &
        bind(C, name="streams_eval_chem_aux")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv_aux
      integer(c_int), value :: ng
      integer(c_int), value :: nreactions
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: mw
      type(c_ptr), value :: arr_a
      type(c_ptr), value :: arr_b
      type(c_ptr), value :: arr_ea
      type(c_ptr), value :: tb_eff
      type(c_ptr), value :: falloff_coeffs
      type(c_ptr), value :: reac_ty
      type(c_ptr), value :: isrev
      type(c_ptr), value :: r_coeffs
      type(c_ptr), value :: p_coeffs
      type(c_ptr), value :: kc_tab
      integer(c_int), value :: num_t_tab
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      real(c_double), value :: r_univ
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      type(c_ptr), value :: h298
      integer(c_int), value :: enable_pasr
      real(c_double), value :: les_c_yoshi
      real(c_double), value :: les_c_mix
      real(c_double), value :: les_c_eps
      type(c_ptr), value :: stream
    end function streams_eval_chem_aux
    integer(c_int) function streams_bcextr_var(nx, ny, nz, ng, w_var, stream) &
        bind(C, name="streams_bcextr_var")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      type(c_ptr), value :: w_var
      type(c_ptr), value :: stream
    end function streams_bcextr_var
    integer(c_int) function streams_bcswap(nx, ny, nz, ng, nv, w, periodic, stream) &
        bind(C, name="streams_bcswap")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      type(c_ptr), value :: w
      type(c_ptr), value :: periodic
      type(c_ptr), value :: stream
    end function streams_bcswap
    integer(c_int) function streams_bcextr(ilat, nx, ny, nz, ng, nv, w, stream) &
        bind(C, name="streams_bcextr")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: ilat
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      type(c_ptr), value :: w
      type(c_ptr), value :: stream
    end function streams_bcextr
    integer(c_int) function streams_bcwall_ad(n_s, ilat, nx, ny, nz, ng, w, stream) &
        bind(C, name="streams_bcwall_ad")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: ilat
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      type(c_ptr), value :: w
      type(c_ptr), value :: stream
    end function streams_bcwall_ad
    integer(c_int) function streams_bc_nr_lat(dir, start_or_end, nr_type, n_s, nx, ny, nz, ng, nv, &
        w_aux, w, fl, metric, indx_cp_l, indx_cp_r, rgas, cv_coeff, cp_coeff, nsetcv, trange, winf, &
        stream) &
        bind(C, name="streams_bc_nr_lat")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: dir
      integer(c_int), value :: start_or_end
      integer(c_int), value :: nr_type
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: w
      type(c_ptr), value :: fl
      type(c_ptr), value :: metric
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: rgas
      type(c_ptr), value :: cv_coeff
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      type(c_ptr), value :: winf
      type(c_ptr), value :: stream
    end function streams_bc_nr_lat
    integer(c_int) function streams_euler_x(n_s, nv, nv_aux, nx, ny, nz, ng, istart_face, &
        iend_face, lmax_base, nkeep, rgas, w_aux, coeff_deriv1, dcsidx, fhat, force_zero_flux_min, &
        force_zero_flux_max, weno_scheme, weno_version, sensor_threshold, weno_size, cv_coeff, &
        cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, &
        flux_splitting, eul_imin, eul_imax, fl, stream) &
        bind(C, name="streams_euler_x")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: istart_face
      integer(c_int), value :: iend_face
      integer(c_int), value :: lmax_base
      integer(c_int), value :: nkeep
      type(c_ptr), value :: rgas
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: fhat
      integer(c_int), value :: force_zero_flux_min
      integer(c_int), value :: force_zero_flux_max
      integer(c_int), value :: weno_scheme
      integer(c_int), value :: weno_version
      real(c_double), value :: sensor_threshold
      integer(c_int), value :: weno_size
      type(c_ptr), value :: cv_coeff
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: ep_ord_change
      real(c_double), value :: tol_iter_nr
      real(c_double), value :: rho0
      real(c_double), value :: u0
      integer(c_int), value :: flux_splitting
      integer(c_int), value :: eul_imin
      integer(c_int), value :: eul_imax
      type(c_ptr), value :: fl
      type(c_ptr), value :: stream
    end function streams_euler_x
    integer(c_int) function streams_euler_y(n_s, nv, nv_aux, nx, ny, nz, ng, eul_jmin, eul_jmax, &
        lmax_base, nkeep, rgas, w_aux, fl, coeff_deriv1, detady, fhat, force_zero_flux_min, &
        force_zero_flux_max, weno_scheme, weno_version, sensor_threshold, weno_size, cv_coeff, &
        cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, &
        flux_splitting, stream) &
        bind(C, name="streams_euler_y")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: eul_jmin
      integer(c_int), value :: eul_jmax
      integer(c_int), value :: lmax_base
      integer(c_int), value :: nkeep
      type(c_ptr), value :: rgas
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: detady
      type(c_ptr), value :: fhat
      integer(c_int), value :: force_zero_flux_min
      integer(c_int), value :: force_zero_flux_max
      integer(c_int), value :: weno_scheme
      integer(c_int), value :: weno_version
      real(c_double), value :: sensor_threshold
      integer(c_int), value :: weno_size
      type(c_ptr), value :: cv_coeff
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: ep_ord_change
      real(c_double), value :: tol_iter_nr
      real(c_double), value :: rho0
      real(c_double), value :: u0
      integer(c_int), value :: flux_splitting
      type(c_ptr), value :: stream
    end function streams_euler_y
    integer(c_int) function streams_euler_z(n_s, nv, nv_aux, nx, ny, nz, ng, eul_kmin, eul_kmax, &
        lmax_base, nkeep, rgas, w_aux, fl, coeff_deriv1, dzitdz, fhat, force_zero_flux_min, &
        force_zero_flux_max, weno_scheme, weno_version, sensor_threshold, weno_size, cv_coeff, &
        cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, &
        flux_splitting, stream) &
        bind(C, name="streams_euler_z")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: eul_kmin
      integer(c_int), value :: eul_kmax
      integer(c_int), value :: lmax_base
      integer(c_int), value :: nkeep
      type(c_ptr), value :: rgas
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: dzitdz
      type(c_ptr), value :: fhat
      integer(c_int), value :: force_zero_flux_min
      integer(c_int), value :: force_zero_flux_max
      integer(c_int), value :: weno_scheme
      integer(c_int), value :: weno_version
      real(c_double), value :: sensor_threshold
      integer(c_int), value :: weno_size
      type(c_ptr), value :: cv_coeff
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: ep_ord_change
      real(c_double), value :: tol_iter_nr
      real(c_double), value :: rho0
      real(c_double), value :: u0
      integer(c_int), value :: flux_splitting
      type(c_ptr), value :: stream
    end function streams_euler_z
    integer(c_int) function streams_visflx_x(n_s, nx, ny, nz, nv, nv_aux, ng, x, w_aux, fl, fhat, &
        indx_cp_l, indx_cp_r, cp_coeff, nsetcv, trange, rgas, r_univ, stream) &
        bind(C, name="streams_visflx_x")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: ng
      type(c_ptr), value :: x
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: fhat
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      type(c_ptr), value :: rgas
      real(c_double), value :: r_univ
      type(c_ptr), value :: stream
    end function streams_visflx_x
    integer(c_int) function streams_visflx_y(n_s, nx, ny, nz, nv, nv_aux, ng, y, w_aux, fl, fhat, &
        indx_cp_l, indx_cp_r, cp_coeff, nsetcv, trange, rgas, r_univ, stream) &
        bind(C, name="streams_visflx_y")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: ng
      type(c_ptr), value :: y
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: fhat
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      type(c_ptr), value :: rgas
      real(c_double), value :: r_univ
      type(c_ptr), value :: stream
    end function streams_visflx_y
    integer(c_int) function streams_visflx_z(n_s, nx, ny, nz, nv, nv_aux, ng, z, w_aux, fl, fhat, &
        indx_cp_l, indx_cp_r, cp_coeff, nsetcv, trange, rgas, r_univ, stream) &
        bind(C, name="streams_visflx_z")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: ng
      type(c_ptr), value :: z
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: fhat
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      type(c_ptr), value :: rgas
      real(c_double), value :: r_univ
      type(c_ptr), value :: stream
    end function streams_visflx_z
    integer(c_int) function streams_visflx_reduced(n_s, nx, ny, nz, ng, nv_aux, visc_order, w_aux, &
        fl, coeff_deriv1, dcsidx, detady, dzitdz, stream) &
        bind(C, name="streams_visflx_reduced")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv_aux
      integer(c_int), value :: visc_order
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      type(c_ptr), value :: stream
    end function streams_visflx_reduced
    integer(c_int) function streams_visflx(n_s, nx, ny, nz, ng, nv_aux, visc_order, w_aux, fl, &
        coeff_deriv1, coeff_deriv2, dcsidx, detady, dzitdz, dcsidxs, detadys, dzitdzs, dcsidx2, &
        detady2, dzitdz2, stream) &
        bind(C, name="streams_visflx")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv_aux
      integer(c_int), value :: visc_order
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: coeff_deriv2
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      type(c_ptr), value :: dcsidxs
      type(c_ptr), value :: detadys
      type(c_ptr), value :: dzitdzs
      type(c_ptr), value :: dcsidx2
      type(c_ptr), value :: detady2
      type(c_ptr), value :: dzitdz2
      type(c_ptr), value :: stream
    end function streams_visflx
    integer(c_int) function streams_compute_chemistry(n_s, nx, ny, nz, nv, nv_aux, ng, nreactions, &
        w, w_aux, fl, mw, arr_a, arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, &
        p_coeffs, kc_tab, num_t_tab, t_min_tab, dt_tab, r_univ, indx_cp_l, indx_cp_r, cv_coeff, &
        nsetcv, trange, tol_iter_nr, stream) &
        bind(C, name="streams_compute_chemistry")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: ng
      integer(c_int), value :: nreactions
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: mw
      type(c_ptr), value :: arr_a
      type(c_ptr), value :: arr_b
      type(c_ptr), value :: arr_ea
      type(c_ptr), value :: tb_eff
      type(c_ptr), value :: falloff_coeffs
      type(c_ptr), value :: reac_ty
      type(c_ptr), value :: isrev
      type(c_ptr), value :: r_coeffs
      type(c_ptr), value :: p_coeffs
      type(c_ptr), value :: kc_tab
      integer(c_int), value :: num_t_tab
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      real(c_double), value :: r_univ
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: cv_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      real(c_double), value :: tol_iter_nr
      type(c_ptr), value :: stream
    end function streams_compute_chemistry
    integer(c_int) function streams_rosenbrock(n_s, nv, nv_aux, nx, ny, nz, ng, w, w_aux, fl, mw, &
        nreactions, arr_a, arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, &
        p_coeffs, kc_tab, num_t_tab, t_min_tab, dt_tab, r_univ, tol_iter_nr, cv_coeff, nsetcv, &
        trange, indx_cp_l, indx_cp_r, dttry, time_start, time_end, maxsteps, maxtry, tol, &
        simpler_splitting, enable_pasr, les_c_yoshi, les_c_mix, les_c_eps, dcsidx, detady, dzitdz, &
        stream) &
        bind(C, name="streams_rosenbrock")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: mw
      integer(c_int), value :: nreactions
      type(c_ptr), value :: arr_a
      type(c_ptr), value :: arr_b
      type(c_ptr), value :: arr_ea
      type(c_ptr), value :: tb_eff
      type(c_ptr), value :: falloff_coeffs
      type(c_ptr), value :: reac_ty
      type(c_ptr), value :: isrev
      type(c_ptr), value :: r_coeffs
      type(c_ptr), value :: p_coeffs
      type(c_ptr), value :: kc_tab
      integer(c_int), value :: num_t_tab
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      real(c_double), value :: r_univ
      real(c_double), value :: tol_iter_nr
      type(c_ptr), value :: cv_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      real(c_double), value :: dttry
      real(c_double), value :: time_start
      real(c_double), value :: time_end
      integer(c_int), value :: maxsteps
      integer(c_int), value :: maxtry
      real(c_double), value :: tol
      integer(c_int), value :: simpler_splitting
      integer(c_int), value :: enable_pasr
      real(c_double), value :: les_c_yoshi
      real(c_double), value :: les_c_mix
      real(c_double), value :: les_c_eps
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      type(c_ptr), value :: stream
    end function streams_rosenbrock
    integer(c_int) function streams_rosenbrock_krylov(n_s, nv, nv_aux, nx, ny, nz, ng, w, w_aux, &
        fl, mw, nreactions, arr_a, arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, &
        p_coeffs, kc_tab, num_t_tab, t_min_tab, dt_tab, r_univ, tol_iter_nr, cv_coeff, nsetcv, &
        trange, indx_cp_l, indx_cp_r, dttry, time_start, time_end, simpler_splitting, fl_sav, &
        maxsteps, enable_pasr, les_c_yoshi, les_c_mix, les_c_eps, dcsidx, detady, dzitdz, stream) &
        bind(C, name="streams_rosenbrock_krylov")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: mw
      integer(c_int), value :: nreactions
      type(c_ptr), value :: arr_a
      type(c_ptr), value :: arr_b
      type(c_ptr), value :: arr_ea
      type(c_ptr), value :: tb_eff
      type(c_ptr), value :: falloff_coeffs
      type(c_ptr), value :: reac_ty
      type(c_ptr), value :: isrev
      type(c_ptr), value :: r_coeffs
      type(c_ptr), value :: p_coeffs
      type(c_ptr), value :: kc_tab
      integer(c_int), value :: num_t_tab
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      real(c_double), value :: r_univ
      real(c_double), value :: tol_iter_nr
      type(c_ptr), value :: cv_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      real(c_double), value :: dttry
      real(c_double), value :: time_start
      real(c_double), value :: time_end
      integer(c_int), value :: simpler_splitting
      type(c_ptr), value :: fl_sav
      integer(c_int), value :: maxsteps
      integer(c_int), value :: enable_pasr
      real(c_double), value :: les_c_yoshi
      real(c_double), value :: les_c_mix
      real(c_double), value :: les_c_eps
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      type(c_ptr), value :: stream
    end function streams_rosenbrock_krylov
    integer(c_int) function streams_init_flux(nx, ny, nz, nv, fl, fln, rhodt, stream) &
        bind(C, name="streams_init_flux")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv
      type(c_ptr), value :: fl
      type(c_ptr), value :: fln
      real(c_double), value :: rhodt
      type(c_ptr), value :: stream
    end function streams_init_flux
    integer(c_int) function streams_update_flux(nx, ny, nz, nv, fl, fln, gamdt, stream) &
        bind(C, name="streams_update_flux")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv
      type(c_ptr), value :: fl
      type(c_ptr), value :: fln
      real(c_double), value :: gamdt
      type(c_ptr), value :: stream
    end function streams_update_flux
    integer(c_int) function streams_init_flux_simpler(nx, ny, nz, nv, fl, fln, fl_sav, rhodt, &
        stream) &
        bind(C, name="streams_init_flux_simpler")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv
      type(c_ptr), value :: fl
      type(c_ptr), value :: fln
      type(c_ptr), value :: fl_sav
      real(c_double), value :: rhodt
      type(c_ptr), value :: stream
    end function streams_init_flux_simpler
    integer(c_int) function streams_sav_flx(nx, ny, nz, nv, fl, fl_sav, stream) &
        bind(C, name="streams_sav_flx")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv
      type(c_ptr), value :: fl
      type(c_ptr), value :: fl_sav
      type(c_ptr), value :: stream
    end function streams_sav_flx
    integer(c_int) function streams_update_simpler_flux(nx, ny, nz, nv, fl, fln, fl_sav, gamdt, &
        stream) &
        bind(C, name="streams_update_simpler_flux")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: nv
      type(c_ptr), value :: fl
      type(c_ptr), value :: fln
      type(c_ptr), value :: fl_sav
      real(c_double), value :: gamdt
      type(c_ptr), value :: stream
    end function streams_update_simpler_flux
    integer(c_int) function streams_update_field(nx, ny, nz, ng, nv, w, fln, fluid_mask, stream) &
        bind(C, name="streams_update_field")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      type(c_ptr), value :: w
      type(c_ptr), value :: fln
      type(c_ptr), value :: fluid_mask
      type(c_ptr), value :: stream
    end function streams_update_field
    integer(c_int) function streams_compute_dt(n_s, nx, ny, nz, ng, nv, nv_aux, dcsidx, detady, &
        dzitdz, dcsidxs, detadys, dzitdzs, w, w_aux, dtmax9, indx_cp_l, indx_cp_r, cp_coeff, &
        nsetcv, trange, fluid_mask, stream) &
        bind(C, name="streams_compute_dt")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      type(c_ptr), value :: dcsidxs
      type(c_ptr), value :: detadys
      type(c_ptr), value :: dzitdzs
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: dtmax9
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      type(c_ptr), value :: fluid_mask
      type(c_ptr), value :: stream
    end function streams_compute_dt
    integer(c_int) function streams_compute_dt_noalloc(n_s, nx, ny, nz, ng, nv, nv_aux, dcsidx, &
        detady, dzitdz, dcsidxs, detadys, dzitdzs, w, w_aux, dtmax9, indx_cp_l, indx_cp_r, &
        cp_coeff, nsetcv, trange, fluid_mask, stream) &
        bind(C, name="streams_compute_dt_noalloc")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      integer(c_int), value :: nv_aux
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      type(c_ptr), value :: dcsidxs
      type(c_ptr), value :: detadys
      type(c_ptr), value :: dzitdzs
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: dtmax9
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      type(c_ptr), value :: fluid_mask
      type(c_ptr), value :: stream
    end function streams_compute_dt_noalloc
    integer(c_int) function streams_copy_cpu_gpu(nx, ny, nz, ng, nv, w_host, w_gpu, stream) &
        bind(C, name="streams_copy_cpu_gpu")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      type(c_ptr), value :: w_host
      type(c_ptr), value :: w_gpu
      type(c_ptr), value :: stream
    end function streams_copy_cpu_gpu
    integer(c_int) function streams_copy_gpu_cpu(nx, ny, nz, ng, nv, w_gpu, w_host, stream) &
        bind(C, name="streams_copy_gpu_cpu")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      type(c_ptr), value :: w_gpu
      type(c_ptr), value :: w_host
      type(c_ptr), value :: stream
    end function streams_copy_gpu_cpu
    integer(c_int) function streams_field_interior(nx, ny, nz, ng, nv, w_gpu, dense, to_dense, &
        stream) &
        bind(C, name="streams_field_interior")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      type(c_ptr), value :: w_gpu
      type(c_ptr), value :: dense
      integer(c_int), value :: to_dense
      type(c_ptr), value :: stream
    end function streams_field_interior
    integer(c_int) function streams_compute_residual(nx, ny, nz, ng, nv, fln, dt, residual_rhou, &
        fluid_mask, stream) &
        bind(C, name="streams_compute_residual")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      type(c_ptr), value :: fln
      real(c_double), value :: dt
      type(c_ptr), value :: residual_rhou
      type(c_ptr), value :: fluid_mask
      type(c_ptr), value :: stream
    end function streams_compute_residual
    integer(c_int) function streams_compute_rho_t_p_minmax(n_s, nx, ny, nz, ng, nv_aux, w_aux, &
        rhomin, rhomax, tmin, tmax, pmin, pmax, fluid_mask, stream) &
        bind(C, name="streams_compute_rho_t_p_minmax")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv_aux
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: rhomin
      type(c_ptr), value :: rhomax
      type(c_ptr), value :: tmin
      type(c_ptr), value :: tmax
      type(c_ptr), value :: pmin
      type(c_ptr), value :: pmax
      type(c_ptr), value :: fluid_mask
      type(c_ptr), value :: stream
    end function streams_compute_rho_t_p_minmax
    integer(c_int) function streams_find_boom(nx, ny, nz, ng, nv, fln, dt, fluid_mask, ncoords1, &
        ncoords3, nboom, first_ijk, stream) &
        bind(C, name="streams_find_boom")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv
      type(c_ptr), value :: fln
      real(c_double), value :: dt
      type(c_ptr), value :: fluid_mask
      integer(c_int), value :: ncoords1
      integer(c_int), value :: ncoords3
      type(c_ptr), value :: nboom
      type(c_ptr), value :: first_ijk
      type(c_ptr), value :: stream
    end function streams_find_boom
    integer(c_int) function streams_rhs_sweep(dir, n_s, nv_aux, nx, ny, nz, ng, lmax_base, nkeep, &
        rgas, w_aux, coeff_deriv1, metric, coord, fhat, force_zero_flux_min, force_zero_flux_max, &
        weno_scheme, weno_version, sensor_threshold, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, &
        indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, flux_splitting, visc, r_univ, init, rhodt, &
        fl, fln, stream) &
        bind(C, name="streams_rhs_sweep")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: dir
      integer(c_int), value :: n_s
      integer(c_int), value :: nv_aux
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: lmax_base
      integer(c_int), value :: nkeep
      type(c_ptr), value :: rgas
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: metric
      type(c_ptr), value :: coord
      type(c_ptr), value :: fhat
      integer(c_int), value :: force_zero_flux_min
      integer(c_int), value :: force_zero_flux_max
      integer(c_int), value :: weno_scheme
      integer(c_int), value :: weno_version
      real(c_double), value :: sensor_threshold
      type(c_ptr), value :: cv_coeff
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      type(c_ptr), value :: ep_ord_change
      real(c_double), value :: tol_iter_nr
      real(c_double), value :: rho0
      real(c_double), value :: u0
      integer(c_int), value :: flux_splitting
      integer(c_int), value :: visc
      real(c_double), value :: r_univ
      integer(c_int), value :: init
      real(c_double), value :: rhodt
      type(c_ptr), value :: fl
      type(c_ptr), value :: fln
      type(c_ptr), value :: stream
    end function streams_rhs_sweep
    integer(c_int) function streams_kinetics_pack(n_s, nreactions, arr_a, arr_b, arr_ea, tb_eff, &
        falloff_coeffs, reac_ty, isrev, r_coeffs, p_coeffs, mw, out, cap) &
        bind(C, name="streams_kinetics_pack")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nreactions
      type(c_ptr), value :: arr_a
      type(c_ptr), value :: arr_b
      type(c_ptr), value :: arr_ea
      type(c_ptr), value :: tb_eff
      type(c_ptr), value :: falloff_coeffs
      type(c_ptr), value :: reac_ty
      type(c_ptr), value :: isrev
      type(c_ptr), value :: r_coeffs
      type(c_ptr), value :: p_coeffs
      type(c_ptr), value :: mw
      type(c_ptr), value :: out
      integer(c_int), value :: cap
    end function streams_kinetics_pack
    integer(c_int) function streams_rhs_finish(n_s, nx, ny, nz, ng, nv_aux, visc_order, w, w_aux, &
        fl, fln, coeff_deriv1, dcsidx, detady, dzitdz, reduced, chem, nreactions, mw, kin_pack, &
        kc_tab, num_t_tab, t_min_tab, dt_tab, r_univ, gamdt, fluid_mask, stream) &
        bind(C, name="streams_rhs_finish")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv_aux
      integer(c_int), value :: visc_order
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: fln
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      integer(c_int), value :: reduced
      integer(c_int), value :: chem
      integer(c_int), value :: nreactions
      type(c_ptr), value :: mw
      type(c_ptr), value :: kin_pack
      type(c_ptr), value :: kc_tab
      integer(c_int), value :: num_t_tab
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      real(c_double), value :: r_univ
      real(c_double), value :: gamdt
      type(c_ptr), value :: fluid_mask
      type(c_ptr), value :: stream
    end function streams_rhs_finish
    integer(c_int) function streams_rhs_finish_next(n_s, nx, ny, nz, ng, nv_aux, visc_order, w, &
        w_aux, fl, fln, coeff_deriv1, dcsidx, detady, dzitdz, reduced, chem, nreactions, mw, &
        kin_pack, kc_tab, num_t_tab, t_min_tab, dt_tab, r_univ, gamdt, rhodt_next, fluid_mask, &
        stream) &
        bind(C, name="streams_rhs_finish_next")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv_aux
      integer(c_int), value :: visc_order
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: fln
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      integer(c_int), value :: reduced
      integer(c_int), value :: chem
      integer(c_int), value :: nreactions
      type(c_ptr), value :: mw
      type(c_ptr), value :: kin_pack
      type(c_ptr), value :: kc_tab
      integer(c_int), value :: num_t_tab
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      real(c_double), value :: r_univ
      real(c_double), value :: gamdt
      real(c_double), value :: rhodt_next
      type(c_ptr), value :: fluid_mask
      type(c_ptr), value :: stream
    end function streams_rhs_finish_next
    integer(c_int) function streams_rhs_cells(n_s, nx, ny, nz, ng, nv_aux, lmax_base, w, w_aux, fl, &
        fln, coeff_deriv1, dcsidx, detady, dzitdz, x, y, z, cp_coeff, nsetcv, trange, indx_cp_l, &
        indx_cp_r, r_univ, chem, nreactions, mw, kin_pack, kc_tab, num_t_tab, t_min_tab, dt_tab, &
        init, rhodt, gamdt, fold, rhodt_next, fluid_mask, stream) &
        bind(C, name="streams_rhs_cells")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nx
      integer(c_int), value :: ny
      integer(c_int), value :: nz
      integer(c_int), value :: ng
      integer(c_int), value :: nv_aux
      integer(c_int), value :: lmax_base
      type(c_ptr), value :: w
      type(c_ptr), value :: w_aux
      type(c_ptr), value :: fl
      type(c_ptr), value :: fln
      type(c_ptr), value :: coeff_deriv1
      type(c_ptr), value :: dcsidx
      type(c_ptr), value :: detady
      type(c_ptr), value :: dzitdz
      type(c_ptr), value :: x
      type(c_ptr), value :: y
      type(c_ptr), value :: z
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      real(c_double), value :: r_univ
      integer(c_int), value :: chem
      integer(c_int), value :: nreactions
      type(c_ptr), value :: mw
      type(c_ptr), value :: kin_pack
      type(c_ptr), value :: kc_tab
      integer(c_int), value :: num_t_tab
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      integer(c_int), value :: init
      real(c_double), value :: rhodt
      real(c_double), value :: gamdt
      integer(c_int), value :: fold
      real(c_double), value :: rhodt_next
      type(c_ptr), value :: fluid_mask
      type(c_ptr), value :: stream
    end function streams_rhs_cells
    integer(c_int) function streams_reactor_batch(n_s, nbatch, w, tguess, dttry, time_end, &
        pressure, mw, rgas, cp_coeff, nreactions, kin_pack, kc_tab, num_t_tab, t_min_tab, dt_tab, &
        r_univ, tol_iter_nr, cv_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, maxsteps, maxtry, tol, &
        nacc, nrej, t_done, dt_next, work, wg_per_cu, mixed, stream) &
        bind(C, name="streams_reactor_batch")
      import :: c_int, c_double, c_ptr
      integer(c_int), value :: n_s
      integer(c_int), value :: nbatch
      type(c_ptr), value :: w
      type(c_ptr), value :: tguess
      type(c_ptr), value :: dttry
      type(c_ptr), value :: time_end
      type(c_ptr), value :: pressure
      type(c_ptr), value :: mw
      type(c_ptr), value :: rgas
      type(c_ptr), value :: cp_coeff
      integer(c_int), value :: nreactions
      type(c_ptr), value :: kin_pack
      type(c_ptr), value :: kc_tab
      integer(c_int), value :: num_t_tab
      real(c_double), value :: t_min_tab
      real(c_double), value :: dt_tab
      real(c_double), value :: r_univ
      real(c_double), value :: tol_iter_nr
      type(c_ptr), value :: cv_coeff
      integer(c_int), value :: nsetcv
      type(c_ptr), value :: trange
      integer(c_int), value :: indx_cp_l
      integer(c_int), value :: indx_cp_r
      integer(c_int), value :: maxsteps
      integer(c_int), value :: maxtry
      real(c_double), value :: tol
      type(c_ptr), value :: nacc
      type(c_ptr), value :: nrej
      type(c_ptr), value :: t_done
      type(c_ptr), value :: dt_next
      type(c_ptr), value :: work
      integer(c_int), value :: wg_per_cu
      integer(c_int), value :: mixed
      type(c_ptr), value :: stream
    end function streams_reactor_batch
  end interface
contains
  subroutine check(rc, what)
    integer(c_int), intent(in) :: rc
    character(len=*), intent(in) :: what
    if (rc /= 0) then
      write(*, '(a,a,a,i0)') 'streams_kernels_hip: ', what, ' returned ', rc
      error stop 1
    end if
  end subroutine check
  subroutine eval_aux_cuf(nx, ny, nz, ng, nv, nv_aux, istart, iend, jstart, jend, kstart, kend, w, &
      w_aux, p0, t_min_tab, dt_tab, r_univ, rgas, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, &
      indx_cp_r, tol_iter_nr, stream, mw, mwinv, visc_species, lambda_species, diffbin_species, &
      num_t_tab, n_eoi, aw_eoi, nainsp, beta0, coeff_eoi)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: istart
    integer(c_int), value :: iend
    integer(c_int), value :: jstart
    integer(c_int), value :: jend
    integer(c_int), value :: kstart
    integer(c_int), value :: kend
    type(c_ptr), value :: w
    type(c_ptr), value :: w_aux
    real(c_double), value :: p0
    real(c_double), value :: t_min_tab
    real(c_double), value :: dt_tab
    real(c_double), value :: r_univ
    type(c_ptr), value :: rgas
    type(c_ptr), value :: cv_coeff
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    real(c_double), value :: tol_iter_nr
    type(c_ptr), value :: stream
    type(c_ptr), value :: mw
    type(c_ptr), value :: mwinv
    type(c_ptr), value :: visc_species
    type(c_ptr), value :: lambda_species
    type(c_ptr), value :: diffbin_species
    integer(c_int), value :: num_t_tab
    integer(c_int), value :: n_eoi
    type(c_ptr), value :: aw_eoi
    type(c_ptr), value :: nainsp
    type(c_ptr), value :: beta0
    type(c_ptr), value :: coeff_eoi
    call check(streams_eval_aux(N_S, nx, ny, nz, ng, nv, nv_aux, istart, iend, jstart, jend, &
        kstart, kend, w, w_aux, p0, t_min_tab, dt_tab, r_univ, rgas, cv_coeff, cp_coeff, nsetcv, &
        trange, indx_cp_l, indx_cp_r, tol_iter_nr, stream, mw, mwinv, visc_species, lambda_species, &
        diffbin_species, num_t_tab, n_eoi, aw_eoi, nainsp, beta0, coeff_eoi), 'eval_aux_cuf')
  end subroutine eval_aux_cuf
  subroutine eval_aux2_cuf(nx, ny, nz, ng, nv_aux, visc_order, w_aux, coeff_deriv1, dcsidx, detady, &
      dzitdz, eps_sensor, sensor_type, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv_aux
    integer(c_int), value :: visc_order
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: coeff_deriv1
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: detady
    type(c_ptr), value :: dzitdz
    real(c_double), value :: eps_sensor
    integer(c_int), value :: sensor_type
    type(c_ptr), value :: stream
    call check(streams_eval_aux2(N_S, nx, ny, nz, ng, nv_aux, visc_order, w_aux, coeff_deriv1, &
        dcsidx, detady, dzitdz, eps_sensor, sensor_type, stream), 'eval_aux2_cuf')
  end subroutine eval_aux2_cuf
  subroutine eval_velaux_cuf(nx, ny, nz, ng, nv, nv_aux, w, w_aux, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    type(c_ptr), value :: w
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: stream
    call check(streams_eval_velaux(N_S, nx, ny, nz, ng, nv, nv_aux, w, w_aux, stream), 'eval_velaux_cuf')
  end subroutine eval_velaux_cuf
  subroutine les_wale_mut_cuf(nx, ny, nz, ng, nv_aux, ep_order, w_aux, coeff_deriv1, dcsidx, &
      detady, dzitdz, les_c_wale, eps_sensor, sensor_type, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv_aux
    integer(c_int), value :: ep_order
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: coeff_deriv1
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: detady
    type(c_ptr), value :: dzitdz
    real(c_double), value :: les_c_wale
    real(c_double), value :: eps_sensor
    integer(c_int), value :: sensor_type
    type(c_ptr), value :: stream
    call check(streams_les_wale_mut(N_S, nx, ny, nz, ng, nv_aux, ep_order, w_aux, coeff_deriv1, &
        dcsidx, detady, dzitdz, les_c_wale, eps_sensor, sensor_type, stream), 'les_wale_mut_cuf')
  end subroutine les_wale_mut_cuf
  subroutine eval_aux_les_cuf(nx, ny, nz, ng, nv, nv_aux, w, w_aux, p0, t_min_tab, dt_tab, r_univ, &
      rgas, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, tol_iter_nr, mw, mwinv, &
      visc_species, lambda_species, diffbin_species, num_t_tab, les_pr, les_sc, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    type(c_ptr), value :: w
    type(c_ptr), value :: w_aux
    real(c_double), value :: p0
    real(c_double), value :: t_min_tab
    real(c_double), value :: dt_tab
    real(c_double), value :: r_univ
    type(c_ptr), value :: rgas
    type(c_ptr), value :: cv_coeff
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    real(c_double), value :: tol_iter_nr
    type(c_ptr), value :: mw
    type(c_ptr), value :: mwinv
    type(c_ptr), value :: visc_species
    type(c_ptr), value :: lambda_species
    type(c_ptr), value :: diffbin_species
    integer(c_int), value :: num_t_tab
    real(c_double), value :: les_pr
    real(c_double), value :: les_sc
    type(c_ptr), value :: stream
    call check(streams_eval_aux_les(N_S, nx, ny, nz, ng, nv, nv_aux, w, w_aux, p0, t_min_tab, &
        dt_tab, r_univ, rgas, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, &
        tol_iter_nr, mw, mwinv, visc_species, lambda_species, diffbin_species, num_t_tab, les_pr, &
        les_sc, stream), 'eval_aux_les_cuf')
  end subroutine eval_aux_les_cuf
  subroutine eval_chem_aux_cuf(nx, ny, nz, nv_aux, ng, nreactions, w_aux, mw, arr_a, arr_b, arr_ea, &
      tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, p_coeffs, kc_tab, num_t_tab, t_min_tab, &
      dt_tab, r_univ, dcsidx, detady, dzitdz, h298, enable_pasr, les_c_yoshi, les_c_mix, les_c_eps, &
      stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv_aux
    integer(c_int), value :: ng
    integer(c_int), value :: nreactions
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: mw
    type(c_ptr), value :: arr_a
    type(c_ptr), value :: arr_b
    type(c_ptr), value :: arr_ea
    type(c_ptr), value :: tb_eff
    type(c_ptr), value :: falloff_coeffs
    type(c_ptr), value :: reac_ty
    type(c_ptr), value :: isrev
    type(c_ptr), value :: r_coeffs
    type(c_ptr), value :: p_coeffs
    type(c_ptr), value :: kc_tab
    integer(c_int), value :: num_t_tab
    real(c_double), value :: t_min_tab
    real(c_double), value :: dt_tab
    real(c_double), value :: r_univ
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: detady
    type(c_ptr), value :: dzitdz
    type(c_ptr), value :: h298
    integer(c_int), value :: enable_pasr
    real(c_double), value :: les_c_yoshi
    real(c_double), value :: les_c_mix
    real(c_double), value :: les_c_eps
    type(c_ptr), value :: stream
    call check(streams_eval_chem_aux(N_S, nx, ny, nz, nv_aux, ng, nreactions, w_aux, mw, arr_a, &
        arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, p_coeffs, kc_tab, &
        num_t_tab, t_min_tab, dt_tab, r_univ, dcsidx, detady, dzitdz, h298, enable_pasr, &
        les_c_yoshi, les_c_mix, les_c_eps, stream), 'eval_chem_aux_cuf')
  end subroutine eval_chem_aux_cuf
  subroutine bcextr_var_cuf(nx, ny, nz, ng, w_var, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    type(c_ptr), value :: w_var
    type(c_ptr), value :: stream
    call check(streams_bcextr_var(nx, ny, nz, ng, w_var, stream), 'bcextr_var_cuf')
  end subroutine bcextr_var_cuf
  subroutine bcswap(nx, ny, nz, ng, nv, w, periodic, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    type(c_ptr), value :: w
    type(c_ptr), value :: periodic
    type(c_ptr), value :: stream
    call check(streams_bcswap(nx, ny, nz, ng, nv, w, periodic, stream), 'bcswap')
  end subroutine bcswap
  subroutine bcextr_cuf(ilat, nx, ny, nz, ng, nv, w, stream)
    integer(c_int), value :: ilat
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    type(c_ptr), value :: w
    type(c_ptr), value :: stream
    call check(streams_bcextr(ilat, nx, ny, nz, ng, nv, w, stream), 'bcextr_cuf')
  end subroutine bcextr_cuf
  subroutine bcwall_ad_cuf(ilat, nx, ny, nz, ng, w, stream)
    integer(c_int), value :: ilat
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    type(c_ptr), value :: w
    type(c_ptr), value :: stream
    call check(streams_bcwall_ad(N_S, ilat, nx, ny, nz, ng, w, stream), 'bcwall_ad_cuf')
  end subroutine bcwall_ad_cuf
  subroutine bc_nr_lat(dir, start_or_end, nr_type, nx, ny, nz, ng, nv, w_aux, w, fl, metric, &
      indx_cp_l, indx_cp_r, rgas, cv_coeff, cp_coeff, nsetcv, trange, winf, stream)
    integer(c_int), value :: dir
    integer(c_int), value :: start_or_end
    integer(c_int), value :: nr_type
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: w
    type(c_ptr), value :: fl
    type(c_ptr), value :: metric
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: rgas
    type(c_ptr), value :: cv_coeff
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    type(c_ptr), value :: winf
    type(c_ptr), value :: stream
    call check(streams_bc_nr_lat(dir, start_or_end, nr_type, N_S, nx, ny, nz, ng, nv, w_aux, w, fl, &
        metric, indx_cp_l, indx_cp_r, rgas, cv_coeff, cp_coeff, nsetcv, trange, winf, stream), 'bc_nr_lat')
  end subroutine bc_nr_lat
  subroutine euler_x(nv, nv_aux, nx, ny, nz, ng, istart_face, iend_face, lmax_base, nkeep, rgas, &
      w_aux, coeff_deriv1, dcsidx, fhat, force_zero_flux_min, force_zero_flux_max, weno_scheme, &
      weno_version, sensor_threshold, weno_size, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, &
      indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, flux_splitting, eul_imin, eul_imax, fl, &
      stream)
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: istart_face
    integer(c_int), value :: iend_face
    integer(c_int), value :: lmax_base
    integer(c_int), value :: nkeep
    type(c_ptr), value :: rgas
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: coeff_deriv1
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: fhat
    integer(c_int), value :: force_zero_flux_min
    integer(c_int), value :: force_zero_flux_max
    integer(c_int), value :: weno_scheme
    integer(c_int), value :: weno_version
    real(c_double), value :: sensor_threshold
    integer(c_int), value :: weno_size
    type(c_ptr), value :: cv_coeff
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: ep_ord_change
    real(c_double), value :: tol_iter_nr
    real(c_double), value :: rho0
    real(c_double), value :: u0
    integer(c_int), value :: flux_splitting
    integer(c_int), value :: eul_imin
    integer(c_int), value :: eul_imax
    type(c_ptr), value :: fl
    type(c_ptr), value :: stream
    call check(streams_euler_x(N_S, nv, nv_aux, nx, ny, nz, ng, istart_face, iend_face, lmax_base, &
        nkeep, rgas, w_aux, coeff_deriv1, dcsidx, fhat, force_zero_flux_min, force_zero_flux_max, &
        weno_scheme, weno_version, sensor_threshold, weno_size, cv_coeff, cp_coeff, nsetcv, trange, &
        indx_cp_l, indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, flux_splitting, eul_imin, &
        eul_imax, fl, stream), 'euler_x')
  end subroutine euler_x
  subroutine euler_y(nv, nv_aux, nx, ny, nz, ng, eul_jmin, eul_jmax, lmax_base, nkeep, rgas, w_aux, &
      fl, coeff_deriv1, detady, fhat, force_zero_flux_min, force_zero_flux_max, weno_scheme, &
      weno_version, sensor_threshold, weno_size, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, &
      indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, flux_splitting, stream)
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: eul_jmin
    integer(c_int), value :: eul_jmax
    integer(c_int), value :: lmax_base
    integer(c_int), value :: nkeep
    type(c_ptr), value :: rgas
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: coeff_deriv1
    type(c_ptr), value :: detady
    type(c_ptr), value :: fhat
    integer(c_int), value :: force_zero_flux_min
    integer(c_int), value :: force_zero_flux_max
    integer(c_int), value :: weno_scheme
    integer(c_int), value :: weno_version
    real(c_double), value :: sensor_threshold
    integer(c_int), value :: weno_size
    type(c_ptr), value :: cv_coeff
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: ep_ord_change
    real(c_double), value :: tol_iter_nr
    real(c_double), value :: rho0
    real(c_double), value :: u0
    integer(c_int), value :: flux_splitting
    type(c_ptr), value :: stream
    call check(streams_euler_y(N_S, nv, nv_aux, nx, ny, nz, ng, eul_jmin, eul_jmax, lmax_base, &
        nkeep, rgas, w_aux, fl, coeff_deriv1, detady, fhat, force_zero_flux_min, &
        force_zero_flux_max, weno_scheme, weno_version, sensor_threshold, weno_size, cv_coeff, &
        cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, &
        flux_splitting, stream), 'euler_y')
  end subroutine euler_y
  subroutine euler_z(nv, nv_aux, nx, ny, nz, ng, eul_kmin, eul_kmax, lmax_base, nkeep, rgas, w_aux, &
      fl, coeff_deriv1, dzitdz, fhat, force_zero_flux_min, force_zero_flux_max, weno_scheme, &
      weno_version, sensor_threshold, weno_size, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, &
      indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, flux_splitting, stream)
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: eul_kmin
    integer(c_int), value :: eul_kmax
    integer(c_int), value :: lmax_base
    integer(c_int), value :: nkeep
    type(c_ptr), value :: rgas
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: coeff_deriv1
    type(c_ptr), value :: dzitdz
    type(c_ptr), value :: fhat
    integer(c_int), value :: force_zero_flux_min
    integer(c_int), value :: force_zero_flux_max
    integer(c_int), value :: weno_scheme
    integer(c_int), value :: weno_version
    real(c_double), value :: sensor_threshold
    integer(c_int), value :: weno_size
    type(c_ptr), value :: cv_coeff
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: ep_ord_change
    real(c_double), value :: tol_iter_nr
    real(c_double), value :: rho0
    real(c_double), value :: u0
    integer(c_int), value :: flux_splitting
    type(c_ptr), value :: stream
    call check(streams_euler_z(N_S, nv, nv_aux, nx, ny, nz, ng, eul_kmin, eul_kmax, lmax_base, &
        nkeep, rgas, w_aux, fl, coeff_deriv1, dzitdz, fhat, force_zero_flux_min, &
        force_zero_flux_max, weno_scheme, weno_version, sensor_threshold, weno_size, cv_coeff, &
        cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, ep_ord_change, tol_iter_nr, rho0, u0, &
        flux_splitting, stream), 'euler_z')
  end subroutine euler_z
  subroutine visflx_x_cuf(nx, ny, nz, nv, nv_aux, ng, x, w_aux, fl, fhat, indx_cp_l, indx_cp_r, &
      cp_coeff, nsetcv, trange, rgas, r_univ, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: ng
    type(c_ptr), value :: x
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: fhat
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    type(c_ptr), value :: rgas
    real(c_double), value :: r_univ
    type(c_ptr), value :: stream
    call check(streams_visflx_x(N_S, nx, ny, nz, nv, nv_aux, ng, x, w_aux, fl, fhat, indx_cp_l, &
        indx_cp_r, cp_coeff, nsetcv, trange, rgas, r_univ, stream), 'visflx_x_cuf')
  end subroutine visflx_x_cuf
  subroutine visflx_y_cuf(nx, ny, nz, nv, nv_aux, ng, y, w_aux, fl, fhat, indx_cp_l, indx_cp_r, &
      cp_coeff, nsetcv, trange, rgas, r_univ, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: ng
    type(c_ptr), value :: y
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: fhat
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    type(c_ptr), value :: rgas
    real(c_double), value :: r_univ
    type(c_ptr), value :: stream
    call check(streams_visflx_y(N_S, nx, ny, nz, nv, nv_aux, ng, y, w_aux, fl, fhat, indx_cp_l, &
        indx_cp_r, cp_coeff, nsetcv, trange, rgas, r_univ, stream), 'visflx_y_cuf')
  end subroutine visflx_y_cuf
  subroutine visflx_z_cuf(nx, ny, nz, nv, nv_aux, ng, z, w_aux, fl, fhat, indx_cp_l, indx_cp_r, &
      cp_coeff, nsetcv, trange, rgas, r_univ, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: ng
    type(c_ptr), value :: z
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: fhat
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    type(c_ptr), value :: rgas
    real(c_double), value :: r_univ
    type(c_ptr), value :: stream
    call check(streams_visflx_z(N_S, nx, ny, nz, nv, nv_aux, ng, z, w_aux, fl, fhat, indx_cp_l, &
        indx_cp_r, cp_coeff, nsetcv, trange, rgas, r_univ, stream), 'visflx_z_cuf')
  end subroutine visflx_z_cuf
  subroutine visflx_reduced_cuf(nx, ny, nz, ng, nv_aux, visc_order, w_aux, fl, coeff_deriv1, &
      dcsidx, detady, dzitdz, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv_aux
    integer(c_int), value :: visc_order
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: coeff_deriv1
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: detady
    type(c_ptr), value :: dzitdz
    type(c_ptr), value :: stream
    call check(streams_visflx_reduced(N_S, nx, ny, nz, ng, nv_aux, visc_order, w_aux, fl, &
        coeff_deriv1, dcsidx, detady, dzitdz, stream), 'visflx_reduced_cuf')
  end subroutine visflx_reduced_cuf
  subroutine visflx_cuf(nx, ny, nz, ng, nv_aux, visc_order, w_aux, fl, coeff_deriv1, coeff_deriv2, &
      dcsidx, detady, dzitdz, dcsidxs, detadys, dzitdzs, dcsidx2, detady2, dzitdz2, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv_aux
    integer(c_int), value :: visc_order
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: coeff_deriv1
    type(c_ptr), value :: coeff_deriv2
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: detady
    type(c_ptr), value :: dzitdz
    type(c_ptr), value :: dcsidxs
    type(c_ptr), value :: detadys
    type(c_ptr), value :: dzitdzs
    type(c_ptr), value :: dcsidx2
    type(c_ptr), value :: detady2
    type(c_ptr), value :: dzitdz2
    type(c_ptr), value :: stream
    call check(streams_visflx(N_S, nx, ny, nz, ng, nv_aux, visc_order, w_aux, fl, coeff_deriv1, &
        coeff_deriv2, dcsidx, detady, dzitdz, dcsidxs, detadys, dzitdzs, dcsidx2, detady2, dzitdz2, &
        stream), 'visflx_cuf')
  end subroutine visflx_cuf
  subroutine compute_chemistry_cuf(nx, ny, nz, nv, nv_aux, ng, nreactions, w, w_aux, fl, mw, arr_a, &
      arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, p_coeffs, kc_tab, num_t_tab, &
      t_min_tab, dt_tab, r_univ, indx_cp_l, indx_cp_r, cv_coeff, nsetcv, trange, tol_iter_nr, &
      stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: ng
    integer(c_int), value :: nreactions
    type(c_ptr), value :: w
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: mw
    type(c_ptr), value :: arr_a
    type(c_ptr), value :: arr_b
    type(c_ptr), value :: arr_ea
    type(c_ptr), value :: tb_eff
    type(c_ptr), value :: falloff_coeffs
    type(c_ptr), value :: reac_ty
    type(c_ptr), value :: isrev
    type(c_ptr), value :: r_coeffs
    type(c_ptr), value :: p_coeffs
    type(c_ptr), value :: kc_tab
    integer(c_int), value :: num_t_tab
    real(c_double), value :: t_min_tab
    real(c_double), value :: dt_tab
    real(c_double), value :: r_univ
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: cv_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    real(c_double), value :: tol_iter_nr
    type(c_ptr), value :: stream
    call check(streams_compute_chemistry(N_S, nx, ny, nz, nv, nv_aux, ng, nreactions, w, w_aux, fl, &
        mw, arr_a, arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, p_coeffs, &
        kc_tab, num_t_tab, t_min_tab, dt_tab, r_univ, indx_cp_l, indx_cp_r, cv_coeff, nsetcv, &
        trange, tol_iter_nr, stream), 'compute_chemistry_cuf')
  end subroutine compute_chemistry_cuf
  subroutine rosenbrock(nv, nv_aux, nx, ny, nz, ng, w, w_aux, fl, mw, nreactions, arr_a, arr_b, &
      arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, p_coeffs, kc_tab, num_t_tab, &
      t_min_tab, dt_tab, r_univ, tol_iter_nr, cv_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, &
      dttry, time_start, time_end, maxsteps, maxtry, tol, simpler_splitting, enable_pasr, &
      les_c_yoshi, les_c_mix, les_c_eps, dcsidx, detady, dzitdz, stream)
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    type(c_ptr), value :: w
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: mw
    integer(c_int), value :: nreactions
    type(c_ptr), value :: arr_a
    type(c_ptr), value :: arr_b
    type(c_ptr), value :: arr_ea
    type(c_ptr), value :: tb_eff
    type(c_ptr), value :: falloff_coeffs
    type(c_ptr), value :: reac_ty
    type(c_ptr), value :: isrev
    type(c_ptr), value :: r_coeffs
    type(c_ptr), value :: p_coeffs
    type(c_ptr), value :: kc_tab
    integer(c_int), value :: num_t_tab
    real(c_double), value :: t_min_tab
    real(c_double), value :: dt_tab
    real(c_double), value :: r_univ
    real(c_double), value :: tol_iter_nr
    type(c_ptr), value :: cv_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    real(c_double), value :: dttry
    real(c_double), value :: time_start
    real(c_double), value :: time_end
    integer(c_int), value :: maxsteps
    integer(c_int), value :: maxtry
    real(c_double), value :: tol
    integer(c_int), value :: simpler_splitting
    integer(c_int), value :: enable_pasr
    real(c_double), value :: les_c_yoshi
    real(c_double), value :: les_c_mix
    real(c_double), value :: les_c_eps
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: detady
    type(c_ptr), value :: dzitdz
    type(c_ptr), value :: stream
    call check(streams_rosenbrock(N_S, nv, nv_aux, nx, ny, nz, ng, w, w_aux, fl, mw, nreactions, &
        arr_a, arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, p_coeffs, kc_tab, &
        num_t_tab, t_min_tab, dt_tab, r_univ, tol_iter_nr, cv_coeff, nsetcv, trange, indx_cp_l, &
        indx_cp_r, dttry, time_start, time_end, maxsteps, maxtry, tol, simpler_splitting, &
        enable_pasr, les_c_yoshi, les_c_mix, les_c_eps, dcsidx, detady, dzitdz, stream), 'rosenbrock')
  end subroutine rosenbrock
  subroutine rosenbrock_krylov(nv, nv_aux, nx, ny, nz, ng, w, w_aux, fl, mw, nreactions, arr_a, &
      arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, p_coeffs, kc_tab, num_t_tab, &
      t_min_tab, dt_tab, r_univ, tol_iter_nr, cv_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, &
      dttry, time_start, time_end, simpler_splitting, fl_sav, maxsteps, enable_pasr, les_c_yoshi, &
      les_c_mix, les_c_eps, dcsidx, detady, dzitdz, stream)
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    type(c_ptr), value :: w
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: mw
    integer(c_int), value :: nreactions
    type(c_ptr), value :: arr_a
    type(c_ptr), value :: arr_b
    type(c_ptr), value :: arr_ea
    type(c_ptr), value :: tb_eff
    type(c_ptr), value :: falloff_coeffs
    type(c_ptr), value :: reac_ty
    type(c_ptr), value :: isrev
    type(c_ptr), value :: r_coeffs
    type(c_ptr), value :: p_coeffs
    type(c_ptr), value :: kc_tab
    integer(c_int), value :: num_t_tab
    real(c_double), value :: t_min_tab
    real(c_double), value :: dt_tab
    real(c_double), value :: r_univ
    real(c_double), value :: tol_iter_nr
    type(c_ptr), value :: cv_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    real(c_double), value :: dttry
    real(c_double), value :: time_start
    real(c_double), value :: time_end
    integer(c_int), value :: simpler_splitting
    type(c_ptr), value :: fl_sav
    integer(c_int), value :: maxsteps
    integer(c_int), value :: enable_pasr
    real(c_double), value :: les_c_yoshi
    real(c_double), value :: les_c_mix
    real(c_double), value :: les_c_eps
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: detady
    type(c_ptr), value :: dzitdz
    type(c_ptr), value :: stream
    call check(streams_rosenbrock_krylov(N_S, nv, nv_aux, nx, ny, nz, ng, w, w_aux, fl, mw, &
        nreactions, arr_a, arr_b, arr_ea, tb_eff, falloff_coeffs, reac_ty, isrev, r_coeffs, &
        p_coeffs, kc_tab, num_t_tab, t_min_tab, dt_tab, r_univ, tol_iter_nr, cv_coeff, nsetcv, &
        trange, indx_cp_l, indx_cp_r, dttry, time_start, time_end, simpler_splitting, fl_sav, &
        maxsteps, enable_pasr, les_c_yoshi, les_c_mix, les_c_eps, dcsidx, detady, dzitdz, stream), 'rosenbrock_krylov')
  end subroutine rosenbrock_krylov
  subroutine init_flux_cuf(nx, ny, nz, nv, fl, fln, rhodt, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv
    type(c_ptr), value :: fl
    type(c_ptr), value :: fln
    real(c_double), value :: rhodt
    type(c_ptr), value :: stream
    call check(streams_init_flux(nx, ny, nz, nv, fl, fln, rhodt, stream), 'init_flux_cuf')
  end subroutine init_flux_cuf
  subroutine update_flux_cuf(nx, ny, nz, nv, fl, fln, gamdt, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv
    type(c_ptr), value :: fl
    type(c_ptr), value :: fln
    real(c_double), value :: gamdt
    type(c_ptr), value :: stream
    call check(streams_update_flux(nx, ny, nz, nv, fl, fln, gamdt, stream), 'update_flux_cuf')
  end subroutine update_flux_cuf
  subroutine init_flux_simpler_cuf(nx, ny, nz, nv, fl, fln, fl_sav, rhodt, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv
    type(c_ptr), value :: fl
    type(c_ptr), value :: fln
    type(c_ptr), value :: fl_sav
    real(c_double), value :: rhodt
    type(c_ptr), value :: stream
    call check(streams_init_flux_simpler(nx, ny, nz, nv, fl, fln, fl_sav, rhodt, stream), 'init_flux_simpler_cuf')
  end subroutine init_flux_simpler_cuf
  subroutine sav_flx_cuf(nx, ny, nz, nv, fl, fl_sav, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv
    type(c_ptr), value :: fl
    type(c_ptr), value :: fl_sav
    type(c_ptr), value :: stream
    call check(streams_sav_flx(nx, ny, nz, nv, fl, fl_sav, stream), 'sav_flx_cuf')
  end subroutine sav_flx_cuf
  subroutine update_simpler_flux_cuf(nx, ny, nz, nv, fl, fln, fl_sav, gamdt, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: nv
    type(c_ptr), value :: fl
    type(c_ptr), value :: fln
    type(c_ptr), value :: fl_sav
    real(c_double), value :: gamdt
    type(c_ptr), value :: stream
    call check(streams_update_simpler_flux(nx, ny, nz, nv, fl, fln, fl_sav, gamdt, stream), 'update_simpler_flux_cuf')
  end subroutine update_simpler_flux_cuf
  subroutine update_field_cuf(nx, ny, nz, ng, nv, w, fln, fluid_mask, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    type(c_ptr), value :: w
    type(c_ptr), value :: fln
    type(c_ptr), value :: fluid_mask
    type(c_ptr), value :: stream
    call check(streams_update_field(nx, ny, nz, ng, nv, w, fln, fluid_mask, stream), 'update_field_cuf')
  end subroutine update_field_cuf
  subroutine compute_dt_cuf(nx, ny, nz, ng, nv, nv_aux, dcsidx, detady, dzitdz, dcsidxs, detadys, &
      dzitdzs, w, w_aux, dtmax9, indx_cp_l, indx_cp_r, cp_coeff, nsetcv, trange, fluid_mask, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    integer(c_int), value :: nv_aux
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: detady
    type(c_ptr), value :: dzitdz
    type(c_ptr), value :: dcsidxs
    type(c_ptr), value :: detadys
    type(c_ptr), value :: dzitdzs
    type(c_ptr), value :: w
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: dtmax9
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    type(c_ptr), value :: fluid_mask
    type(c_ptr), value :: stream
    call check(streams_compute_dt(N_S, nx, ny, nz, ng, nv, nv_aux, dcsidx, detady, dzitdz, dcsidxs, &
        detadys, dzitdzs, w, w_aux, dtmax9, indx_cp_l, indx_cp_r, cp_coeff, nsetcv, trange, &
        fluid_mask, stream), 'compute_dt_cuf')
  end subroutine compute_dt_cuf
  subroutine copy_cpu_gpu(nx, ny, nz, ng, nv, w_host, w_gpu, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    type(c_ptr), value :: w_host
    type(c_ptr), value :: w_gpu
    type(c_ptr), value :: stream
    call check(streams_copy_cpu_gpu(nx, ny, nz, ng, nv, w_host, w_gpu, stream), 'copy_cpu_gpu')
  end subroutine copy_cpu_gpu
  subroutine copy_gpu_cpu(nx, ny, nz, ng, nv, w_gpu, w_host, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    type(c_ptr), value :: w_gpu
    type(c_ptr), value :: w_host
    type(c_ptr), value :: stream
    call check(streams_copy_gpu_cpu(nx, ny, nz, ng, nv, w_gpu, w_host, stream), 'copy_gpu_cpu')
  end subroutine copy_gpu_cpu
  subroutine compute_residual_cuf(nx, ny, nz, ng, nv, fln, dt, residual_rhou, fluid_mask, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    type(c_ptr), value :: fln
    real(c_double), value :: dt
    type(c_ptr), value :: residual_rhou
    type(c_ptr), value :: fluid_mask
    type(c_ptr), value :: stream
    call check(streams_compute_residual(nx, ny, nz, ng, nv, fln, dt, residual_rhou, fluid_mask, &
        stream), 'compute_residual_cuf')
  end subroutine compute_residual_cuf
  subroutine compute_rho_t_p_minmax_cuf(nx, ny, nz, ng, nv_aux, w_aux, rhomin, rhomax, tmin, tmax, &
      pmin, pmax, fluid_mask, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv_aux
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: rhomin
    type(c_ptr), value :: rhomax
    type(c_ptr), value :: tmin
    type(c_ptr), value :: tmax
    type(c_ptr), value :: pmin
    type(c_ptr), value :: pmax
    type(c_ptr), value :: fluid_mask
    type(c_ptr), value :: stream
    call check(streams_compute_rho_t_p_minmax(N_S, nx, ny, nz, ng, nv_aux, w_aux, rhomin, rhomax, &
        tmin, tmax, pmin, pmax, fluid_mask, stream), 'compute_rho_t_p_minmax_cuf')
  end subroutine compute_rho_t_p_minmax_cuf
  subroutine find_boom_cuf(nx, ny, nz, ng, nv, fln, dt, fluid_mask, ncoords1, ncoords3, nboom, &
      first_ijk, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv
    type(c_ptr), value :: fln
    real(c_double), value :: dt
    type(c_ptr), value :: fluid_mask
    integer(c_int), value :: ncoords1
    integer(c_int), value :: ncoords3
    type(c_ptr), value :: nboom
    type(c_ptr), value :: first_ijk
    type(c_ptr), value :: stream
    call check(streams_find_boom(nx, ny, nz, ng, nv, fln, dt, fluid_mask, ncoords1, ncoords3, &
        nboom, first_ijk, stream), 'find_boom_cuf')
  end subroutine find_boom_cuf
  subroutine rhs_sweep(dir, nv_aux, nx, ny, nz, ng, lmax_base, nkeep, rgas, w_aux, coeff_deriv1, &
      metric, coord, fhat, force_zero_flux_min, force_zero_flux_max, weno_scheme, weno_version, &
      sensor_threshold, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, ep_ord_change, &
      tol_iter_nr, rho0, u0, flux_splitting, visc, r_univ, init, rhodt, fl, fln, stream)
    integer(c_int), value :: dir
    integer(c_int), value :: nv_aux
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: lmax_base
    integer(c_int), value :: nkeep
    type(c_ptr), value :: rgas
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: coeff_deriv1
    type(c_ptr), value :: metric
    type(c_ptr), value :: coord
    type(c_ptr), value :: fhat
    integer(c_int), value :: force_zero_flux_min
    integer(c_int), value :: force_zero_flux_max
    integer(c_int), value :: weno_scheme
    integer(c_int), value :: weno_version
    real(c_double), value :: sensor_threshold
    type(c_ptr), value :: cv_coeff
    type(c_ptr), value :: cp_coeff
    integer(c_int), value :: nsetcv
    type(c_ptr), value :: trange
    integer(c_int), value :: indx_cp_l
    integer(c_int), value :: indx_cp_r
    type(c_ptr), value :: ep_ord_change
    real(c_double), value :: tol_iter_nr
    real(c_double), value :: rho0
    real(c_double), value :: u0
    integer(c_int), value :: flux_splitting
    integer(c_int), value :: visc
    real(c_double), value :: r_univ
    integer(c_int), value :: init
    real(c_double), value :: rhodt
    type(c_ptr), value :: fl
    type(c_ptr), value :: fln
    type(c_ptr), value :: stream
    call check(streams_rhs_sweep(dir, N_S, nv_aux, nx, ny, nz, ng, lmax_base, nkeep, rgas, w_aux, &
        coeff_deriv1, metric, coord, fhat, force_zero_flux_min, force_zero_flux_max, weno_scheme, &
        weno_version, sensor_threshold, cv_coeff, cp_coeff, nsetcv, trange, indx_cp_l, indx_cp_r, &
        ep_ord_change, tol_iter_nr, rho0, u0, flux_splitting, visc, r_univ, init, rhodt, fl, fln, &
        stream), 'rhs_sweep')
  end subroutine rhs_sweep
  subroutine rhs_finish(nx, ny, nz, ng, nv_aux, visc_order, w, w_aux, fl, fln, coeff_deriv1, &
      dcsidx, detady, dzitdz, reduced, chem, nreactions, mw, kin_pack, kc_tab, num_t_tab, &
      t_min_tab, dt_tab, r_univ, gamdt, fluid_mask, stream)
    integer(c_int), value :: nx
    integer(c_int), value :: ny
    integer(c_int), value :: nz
    integer(c_int), value :: ng
    integer(c_int), value :: nv_aux
    integer(c_int), value :: visc_order
    type(c_ptr), value :: w
    type(c_ptr), value :: w_aux
    type(c_ptr), value :: fl
    type(c_ptr), value :: fln
    type(c_ptr), value :: coeff_deriv1
    type(c_ptr), value :: dcsidx
    type(c_ptr), value :: detady
    type(c_ptr), value :: dzitdz
    integer(c_int), value :: reduced
    integer(c_int), value :: chem
    integer(c_int), value :: nreactions
    type(c_ptr), value :: mw
    type(c_ptr), value :: kin_pack
    type(c_ptr), value :: kc_tab
    integer(c_int), value :: num_t_tab
    real(c_double), value :: t_min_tab
    real(c_double), value :: dt_tab
    real(c_double), value :: r_univ
    real(c_double), value :: gamdt
    type(c_ptr), value :: fluid_mask
    type(c_ptr), value :: stream
    call check(streams_rhs_finish(N_S, nx, ny, nz, ng, nv_aux, visc_order, w, w_aux, fl, fln, &
        coeff_deriv1, dcsidx, detady, dzitdz, reduced, chem, nreactions, mw, kin_pack, kc_tab, &
        num_t_tab, t_min_tab, dt_tab, r_univ, gamdt, fluid_mask, stream), 'rhs_finish')
  end subroutine rhs_finish
end module streams_kernels_hip
